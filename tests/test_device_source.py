"""Properties of the device code's source that no run on a GPU shows reliably."""
import re

import pytest

from conftest import PKG_DIR

FILES = sorted(p for p in (PKG_DIR / "csrc").iterdir() if p.suffix in (".hip", ".h", ".cpp"))


@pytest.mark.parametrize("path", FILES, ids=lambda p: p.name)
def test_inline_asm_holds_no_vector_instruction(path):
    """The compiler keeps the wait states between an MFMA and a vector write of its SrcC registers for its own
    instructions only, so an inline asm may hold scalar waits and barriers or nothing at all."""
    text = re.sub(r"//[^\n]*", "", path.read_text())
    for m in re.finditer(r"\basm\b(?:\s+volatile)?\s*\(((?:\s*\"(?:[^\"\\]|\\.)*\")+)", text):
        body = "".join(re.findall(r"\"((?:[^\"\\]|\\.)*)\"", m.group(1)))
        for line in re.split(r"\\n|;", body.replace("\\t", " ")):
            assert not line.strip() or line.split()[0] in ("s_waitcnt", "s_barrier"), f"{path.name}: asm({body!r})"
