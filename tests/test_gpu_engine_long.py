"""Forwards above 2560 rows, whose matmuls follow the long-prefill plans (two column tiles per wave, gate_up
with its SiLU epilogue, unsplit projections as f16), against the same tokens as a shorter state and its
continuation, whose matmuls run other plans."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine(sdamd, synth, tmp_path_factory):
    cfg = dict(synth.CONFIG_2B, layer_types=["linear_attention", "full_attention"])
    d = synth.write_model(str(tmp_path_factory.mktemp("long")), cfg, vocab=4096, seed=5)
    eng, _, _ = sdamd.load_decider(d)
    yield eng
    eng.free()


@pytest.mark.parametrize("n", [2561, 2688, 3001, 4096])
def test_long_forward_matches_its_continuation(engine, n):
    """Hidden rows within 2e-2 (the tests' activation bound): the two differ in summation order only."""
    ids = np.random.default_rng(n).integers(0, 4096, n).astype(np.uint32)
    cut = n - 700
    rows = [cut, cut + 1, n - 333, n - 1]
    whole = engine.forward(ids, rows).hidden
    prefix = engine.forward(ids[:cut], [], keep=True).snapshot
    part = engine.forward(ids[cut:], [r - cut for r in rows], cache=prefix).hidden
    err = float(np.abs(whole - part).max())
    assert err < 2e-2, f"n={n}: max |dh| {err}"
