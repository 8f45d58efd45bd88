"""The work that a user of this engine has it do, as cases that can be timed and compared.

Kernel-level cases go through the `op_*` entry points on device buffers; their shapes are the layers of
the 2B hybrid (hidden 2048, intermediate 6144, 16 delta-rule heads of 128, 8 query and 2 key/value heads
of 256, int4 group-32 weights) over the row counts that its calls have: a question of a few tokens, a
batch of questions, a state of hundreds to thousands of tokens.  Whole calls go through `Engine` and
`ask_ids` on the 24-layer 2B with seeded random weights.

`listed()` names the cases, `draw()` gives more of the same ranges, `prepare()` makes what the program
has in hand before the call, `run()` is one call, `work()` what the call cannot do without, `tolerance()`
how far two correct implementations at this precision differ, `exact()` the results in 64 bits by plain
torch.
"""
import importlib.util
import json
import math
import os
import sys
import tempfile

import numpy as np
import torch

# ---- the framework --------------------------------------------------------------------------------


def _pkg():
    """The package of this repository (its folder's name is not a Python identifier)."""
    if "sdamd" not in sys.modules:
        here = os.path.join(os.getcwd(), "strands-decider-rs_amd")
        spec = importlib.util.spec_from_file_location("sdamd", os.path.join(here, "__init__.py"),
                                                      submodule_search_locations=[here])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["sdamd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["sdamd"]


# The matrices of one layer as (N, K): the fused projections that the engine runs and the separate ones.
SHAPES = {
    "in_proj": (8256, 2048),  # delta-rule layer: q | k | v | z | a | b
    "qkv": (5120, 2048),      # attention layer: q and gate, k, v
    "o": (2048, 2048),        # out_proj, o_proj, one q projection, an adapter's proj
    "gate_up": (12288, 2048),
    "down": (2048, 6144),
    "gate": (6144, 2048),
    "kv": (512, 2048),
}
HQ, HK, HD, RD, CTX = 8, 2, 256, 64, 4096
H, DK, DV = 16, 128, 128
VOCAB = 151936
THETA = 1e7


# ---- cases ----------------------------------------------------------------------------------------

def listed():
    return [
        # The projections of an attention layer and its MLP for a question of 8 tokens, in a captured
        # graph: the short rows, where a call is launches and one read of the weights.
        dict(name="layer_m8", op="layer", m=8),
        # One projection for a batch of three 40-token questions.
        dict(name="in_proj_m120", op="matmul", shape="in_proj", m=120),
        # One projection for a 512-token state (the headline workload's prefill).
        dict(name="gate_up_m512", op="matmul", shape="gate_up", m=512),
        # The MLP's second matrix for a long, ragged state: K is three times the hidden size.
        dict(name="down_m1777", op="matmul", shape="down", m=1777),
        # A matrix in one of the other weight formats that a model file may hold (an adapter's
        # projection in int3 with biases, group 64) for a 300-token input.
        dict(name="int3_m300", op="format", shape="o", m=300, bits=3, group=64, asym=True),
        # One gated-delta-net recurrence: a 512-token state from nothing, and a ragged continuation of
        # a state that is already there.
        dict(name="gdn_512", op="gdn", l=512, load=False),
        dict(name="gdn_1900_on", op="gdn", l=1900, load=True),
        # Attention of a batch of questions' rows over a 512-token prefix, and of a long input over itself.
        dict(name="attn_120_on_512", op="attention", l=120, p=512),
        dict(name="attn_2048", op="attention", l=2048, p=0),
        # Whole calls: a 16-token question from a 512-token state's snapshot (the smallest forward, by
        # launches); ask_ids of a 512-token state with three 40-token questions (the headline
        # workload); one forward of a long context and its question.
        dict(name="question_16_on_512", op="question", l=16, p=512),
        dict(name="ask_512_3x40", op="ask", s=512, n=3, q=40),
        dict(name="context_3000", op="context", l=3000),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["layer", "matmul", "matmul", "matmul", "format", "gdn", "gdn", "attention", "attention",
                     "question", "ask", "context"])
    if op == "layer":
        return dict(op=op, m=rng.randint(1, 20))
    if op == "matmul":
        return dict(op=op, shape=rng.choice(sorted(SHAPES)), m=_logint(rng, 21, 2600))
    if op == "format":
        bits, group, asym = rng.choice([2, 3, 4]), rng.choice([32, 64, 128]), rng.random() < 0.5
        if (bits, group, asym) == (4, 32, False):
            asym = True
        return dict(op=op, shape=rng.choice(["o", "kv", "down"]), m=_logint(rng, 1, 600), bits=bits, group=group,
                    asym=asym)
    if op == "gdn":
        return dict(op=op, l=_logint(rng, 65, 3000), load=rng.random() < 0.5)
    if op == "attention":
        p = 0 if rng.random() < 0.4 else _logint(rng, 64, 2048)
        return dict(op=op, l=_logint(rng, 21, min(2600, CTX - p)), p=p)
    if op == "question":
        return dict(op=op, l=rng.randint(2, 64), p=_logint(rng, 64, 2048))
    if op == "ask":
        return dict(op=op, s=_logint(rng, 128, 2048), n=rng.randint(2, 8), q=rng.randint(24, 64))
    return dict(op="context", l=_logint(rng, 65, 3000))


# ---- inputs ---------------------------------------------------------------------------------------

def _gen(seed, salt):
    return torch.Generator("cuda").manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFF)


def _words(g, n, k, bits):
    """Random codes of n x k weights in the model's layout: every bit of every word is a code bit."""
    return torch.randint(-2 ** 31, 2 ** 31, (n, k // 32, bits), generator=g, device="cuda", dtype=torch.int64).to(torch.int32)


def _scales(g, n, groups):
    return torch.empty(n, groups, device="cuda").uniform_(0.005, 0.02, generator=g).half()


def _w4(seed, shape):
    n, k = SHAPES[shape]
    g = _gen(seed, 17 + sorted(SHAPES).index(shape))
    return _words(g, n, k, 4), _scales(g, n, k // 32)


def _rows(seed, salt, m, k):
    return torch.randn(m, k, generator=_gen(seed, salt), device="cuda").half()


LAYER = ["qkv", "o", "gate_up", "down"]


def _gdn_inputs(case, seed):
    """q, k, v as they leave the conv, gates a and b, decay rates and a state of a previous part."""
    g = _gen(seed, 5)
    l = case["l"]
    qkv = torch.randn(l, 2 * H * DK + H * DV, generator=g, device="cuda")
    gates = torch.randn(l, 2 * H, generator=g, device="cuda").half()
    rate = -torch.empty(H, device="cuda").uniform_(0.02, 2.0, generator=g)
    bias = torch.zeros(H, device="cuda")
    state = 0.3 * torch.randn(H, DK, DV, generator=g, device="cuda")
    return qkv, gates, rate, bias, state if case["load"] else torch.zeros_like(state)


_TABLE = None


def _rope():
    """[CTX][RD/2][2] cosines and sines, angles in 64 bits."""
    global _TABLE
    if _TABLE is None:
        t = torch.arange(CTX, dtype=torch.float64)[:, None]
        a = t / THETA ** (torch.arange(0, RD, 2, dtype=torch.float64) / RD)
        _TABLE = torch.stack([a.cos(), a.sin()], -1).float().cuda().contiguous()
    return _TABLE


def _attn_inputs(case, seed):
    """The qkv projection's output, the norm weights, and a cache whose first p rows are filled."""
    g = _gen(seed, 7)
    big = torch.randn(case["l"], 2 * HQ * HD + 2 * HK * HD, generator=g, device="cuda").half()
    qw = 1 + 0.1 * torch.randn(HD, generator=g, device="cuda")
    kw = 1 + 0.1 * torch.randn(HD, generator=g, device="cuda")
    k = torch.randn(HK, CTX, HD, generator=g, device="cuda").half()
    v = torch.randn(HK, CTX, HD, generator=g, device="cuda").half()
    k[:, case["p"]:] = 0
    v[:, case["p"]:] = 0
    return big, qw, kw, k, v


def _block_k(k):
    """[HK][CTX][HD] -> the cache's blocks of 32 rows, [HK][CTX/32][HD/32][32 rows][32 dims]."""
    return k.view(HK, CTX // 32, 32, HD // 32, 32).transpose(2, 3).contiguous()


def _block_v(v):
    """[HK][CTX][HD] -> transposed in blocks of 32 rows, [HK][CTX/32][HD][32 rows]."""
    return v.view(HK, CTX // 32, 32, HD).transpose(2, 3).contiguous()


_MODEL = None
_LOADED = None


def _model_dir():
    """The 2B with seeded random weights, written once."""
    global _MODEL
    if _MODEL is None:
        _pkg()
        import sdamd.synth as synth
        _MODEL = synth.write_model(os.path.join(tempfile.gettempdir(), "sd_cases_2b_%d" % os.getuid()),
                                   synth.CONFIG_2B, vocab=VOCAB, seed=0)
    return _MODEL


def _loaded():
    """The engine and head that the program keeps from its start."""
    global _LOADED
    if _LOADED is None:
        eng, head, _ = _pkg().load_decider(_model_dir())
        _LOADED = (eng, head)
    return _LOADED


def _tokens(seed, salt, n):
    return np.random.default_rng([int(seed), salt]).integers(0, VOCAB, n).astype(np.uint32)


def _spread(n, count):
    """`count` option rows spread over n tokens, before the last one."""
    return sorted({int((i + 1) * (n - 1) / (count + 1)) for i in range(count)})


def _question_ids(case, seed):
    return _tokens(seed, 2, case["l"]), _spread(case["l"], 3) + [case["l"] - 1]


def _ask_ids(case, seed):
    qs = [_tokens(seed, 10 + i, case["q"]) for i in range(case["n"])]
    opts = [_spread(case["q"], 2 + i % 4) for i in range(case["n"])]
    return _tokens(seed, 1, case["s"]), qs, opts


def prepare(case, seed):
    sd, op = _pkg(), case["op"]
    if op == "layer":
        # the layer's weights as they are kept, and the captured graph that a serving loop replays
        m, st = case["m"], {"op": op, "keep": [], "out": []}
        for i, s in enumerate(LAYER):
            n, k = SHAPES[s]
            w, sc = _w4(seed, s)
            a, y = _rows(seed, 40 + i, m, k), torch.zeros(m, n, device="cuda", dtype=torch.float16)
            sd.op_repack_w4(w.data_ptr(), sc.data_ptr(), n, k)
            sd.op_matmul_noalloc(a.data_ptr(), w.data_ptr(), sc.data_ptr(), y.data_ptr(), m, n, k, True)
            st["keep"].append((a, w, sc, n, k))
            st["out"].append(y)
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"]):
            stream = torch.cuda.current_stream().cuda_stream
            for (a, w, sc, n, k), y in zip(st["keep"], st["out"]):
                sd.op_matmul_noalloc(a.data_ptr(), w.data_ptr(), sc.data_ptr(), y.data_ptr(), m, n, k, True, stream)
        return st
    if op == "matmul":
        n, k = SHAPES[case["shape"]]
        w, sc = _w4(seed, case["shape"])
        sd.op_repack_w4(w.data_ptr(), sc.data_ptr(), n, k)
        return {"op": op, "a": _rows(seed, 3, case["m"], k), "w": w, "s": sc, "n": n, "k": k,
                "y": torch.zeros(case["m"], n, device="cuda", dtype=torch.float16)}
    if op == "format":
        n, k = SHAPES[case["shape"]]
        w, sc, bi = _format_weights(case, seed)
        return {"op": op, "a": _rows(seed, 3, case["m"], k), "w": w, "s": sc, "b": bi, "n": n, "k": k,
                "bits": case["bits"], "group": case["group"], "asym": case["asym"],
                "y": torch.zeros(case["m"], n, device="cuda", dtype=torch.float16)}
    if op == "gdn":
        qkv, gates, rate, bias, state = _gdn_inputs(case, seed)
        return {"op": op, "qkv": qkv, "gates": gates, "rate": rate, "bias": bias, "state": state, "load": case["load"],
                "o": torch.zeros(case["l"], H * DV, device="cuda")}
    if op == "attention":
        big, qw, kw, k, v = _attn_inputs(case, seed)
        l = case["l"]
        return {"op": op, "big": big, "qw": qw, "kw": kw, "rope": _rope(), "p": case["p"], "k": _block_k(k),
                "v": _block_v(v), "q": torch.zeros(HQ, l, HD, device="cuda", dtype=torch.float16),
                "out": torch.zeros(l, HQ * HD, device="cuda", dtype=torch.float16)}
    eng, head = _loaded()
    if op == "question":
        ids, rows = _question_ids(case, seed)
        snap = eng.forward(_tokens(seed, 1, case["p"]), [], keep=True).snapshot
        return {"op": op, "eng": eng, "ids": ids, "rows": rows, "snap": snap}
    if op == "ask":
        ids, qs, opts = _ask_ids(case, seed)
        return {"op": op, "eng": eng, "head": head, "ids": ids, "qs": qs, "opts": opts}
    return {"op": op, "eng": eng, "ids": _tokens(seed, 1, case["l"]), "rows": _spread(case["l"], 4) + [case["l"] - 1]}


def _format_weights(case, seed):
    n, k = SHAPES[case["shape"]]
    g = _gen(seed, 31)
    w, sc = _words(g, n, k, case["bits"]), _scales(g, n, k // case["group"])
    bi = None
    if case["asym"]:  # the biases centre the codes, as a quantizer's zero points do
        centre = ((1 << case["bits"]) - 1) / 2
        bi = (-centre * sc.float() * torch.empty(sc.shape, device="cuda").uniform_(0.9, 1.1, generator=g)).half()
    return w, sc, bi


def run(st):
    sd, op = _pkg(), st["op"]
    if op == "layer":
        st["graph"].replay()
        return st["out"]
    if op == "matmul":
        m = st["a"].shape[0]
        sd.op_matmul(st["a"].data_ptr(), st["w"].data_ptr(), st["s"].data_ptr(), st["y"].data_ptr(), m, st["n"], st["k"],
                     m <= 20, -1, True)
        return st["y"]
    if op == "format":
        sd.op_matmul_fmt(st["a"].data_ptr(), st["w"].data_ptr(), st["s"].data_ptr(),
                         st["b"].data_ptr() if st["asym"] else None, st["y"].data_ptr(), st["a"].shape[0], st["n"],
                         st["k"], st["bits"], st["group"], st["asym"])
        return st["y"]
    if op == "gdn":
        sd.op_gdn(st["qkv"].data_ptr(), st["gates"].data_ptr(), 2 * H, 0, H, st["rate"].data_ptr(),
                  st["bias"].data_ptr(), st["qkv"].shape[0], H, DK, DV, st["state"].data_ptr(), st["load"],
                  st["o"].data_ptr())
        return {"o": st["o"], "state": st["state"]}
    if op == "attention":
        sd.op_attention(st["big"].data_ptr(), st["big"].shape[1], st["qw"].data_ptr(), st["kw"].data_ptr(),
                        st["rope"].data_ptr(), st["big"].shape[0], st["p"], HQ, HK, HD, RD, st["q"].data_ptr(),
                        st["k"].data_ptr(), st["v"].data_ptr(), CTX, st["out"].data_ptr())
        return {"out": st["out"], "q": st["q"], "k": st["k"], "v": st["v"]}
    if op == "question":
        return st["eng"].forward(st["ids"], st["rows"], cache=st["snap"]).hidden
    if op == "ask":
        return sd.ask_ids(st["eng"], st["head"], st["ids"], st["qs"], st["opts"], [1.0] * len(st["qs"]))
    return st["eng"].forward(st["ids"], st["rows"]).hidden


# ---- what a call cannot do without ----------------------------------------------------------------

LAYERS_GDN, LAYERS_ATTN = 18, 6
PARAMS = (LAYERS_GDN * (8256 * 2048 + 2048 * 2048) + LAYERS_ATTN * (5120 * 2048 + 2048 * 2048)
          + (LAYERS_GDN + LAYERS_ATTN) * (12288 * 2048 + 2048 * 6144))


def _w4_bytes(n, k):
    return n * k // 2 + n * k // 16


def _attn_flops(l, p):
    return 4 * HQ * HD * (l * p + l * (l + 1) // 2)


def _gdn_flops(l):
    return 7 * H * DK * DV * l


def work(case):
    op = case["op"]
    if op in ("layer", "matmul", "format"):
        m, b, f = case["m"], 0, 0
        for s in LAYER if op == "layer" else [case["shape"]]:
            n, k = SHAPES[s]
            if op == "format":
                b += n * k * case["bits"] // 8 + (4 if case["asym"] else 2) * n * k // case["group"]
            else:
                b += _w4_bytes(n, k)
            b += 2 * m * (n + k)
            f += 2 * m * n * k
        return {"bytes": b, "flops": f}
    if op == "gdn":
        l = case["l"]
        return {"bytes": 4 * l * (2 * H * DK + 2 * H * DV) + 4 * l * H + (2 if case["load"] else 1) * 4 * H * DK * DV,
                "flops": _gdn_flops(l)}
    if op == "attention":
        l, p = case["l"], case["p"]
        return {"bytes": 2 * l * (2 * HQ * HD + 2 * HK * HD) + 2 * 2 * HK * HD * (p + l) + 2 * 2 * l * HQ * HD,
                "flops": _attn_flops(l, p)}
    if op == "question":
        m, attn = case["l"], _attn_flops(case["l"], case["p"])
        kv = case["p"] + m
    elif op == "ask":
        m = case["s"] + case["n"] * case["q"]
        attn, kv = _attn_flops(case["s"], 0) + case["n"] * _attn_flops(case["q"], case["s"]), m
    else:
        m, attn, kv = case["l"], _attn_flops(case["l"], 0), case["l"]
    states = (2 if op == "question" else 1) * LAYERS_GDN * 4 * H * DK * DV
    return {"bytes": PARAMS // 2 + PARAMS // 16 + LAYERS_ATTN * 2 * 2 * HK * HD * kv + states,
            "flops": 2 * m * PARAMS + LAYERS_ATTN * attn + LAYERS_GDN * _gdn_flops(m)}


def tolerance(case):
    # About four times what the outputs were measured to be off from `exact`: one rounding to f16 of the
    # projections (2.1e-4; 2.7e-4 with the weights rounded to f16 as well) and of attention (3.3e-4), the
    # split-f16 products of the chunked delta rule (7e-6), and 24 layers of such roundings (1.5e-3 in the
    # hidden rows, up to 2.4e-3 in a probability).
    return {"layer": {"rel": 8e-4}, "matmul": {"rel": 1.1e-3}, "format": {"rel": 8e-4}, "gdn": {"rel": 3e-5},
            "attention": {"rel": 1.3e-3}, "question": {"rel": 6e-3}, "ask": {"rel": 1e-2},
            "context": {"rel": 6e-3}}[case["op"]]


# ---- 64-bit results by plain torch ----------------------------------------------------------------

def _codes(w, bits):
    """[n][k/32][bits] words -> codes [n][k] in f64 (the model's bit order)."""
    n, kb, _ = w.shape
    w = w.to(torch.int64) & 0xFFFFFFFF
    e = torch.arange(32, device=w.device)
    if bits == 4:
        c = (w[:, :, :, None] >> (4 * torch.arange(8, device=w.device))) & 15
        return c.reshape(n, kb * 32).double()
    c = (w[:, :, :2, None] >> (2 * torch.arange(16, device=w.device))) & 3
    c = c.reshape(n, kb, 32)
    if bits == 3:
        c = c | (((w[:, :, 2:3] >> e) & 1) << 2)
    return c.reshape(n, kb * 32).double()


def _dense(w, s, b, bits, group):
    c, s = _codes(w, bits), s.double().repeat_interleave(group, 1)
    return (c - (1 << (bits - 1))) * s if b is None else c * s + b.double().repeat_interleave(group, 1)


def _delta_rule(q, k, v, a, b, rate, bias, state):
    """Token by token in f64: q, k [l][H][DK], v [l][H][DV], a, b [l][H], state [H][DK][DV] -> o, state."""
    q = q / (q.square().sum(-1, keepdim=True) + 1e-6).sqrt() / math.sqrt(DK)
    k = k / (k.square().sum(-1, keepdim=True) + 1e-6).sqrt()
    decay = (rate * torch.nn.functional.softplus(a + bias)).exp()
    beta = torch.sigmoid(b)
    s, out = state.clone(), torch.empty_like(v)
    for t in range(q.shape[0]):
        s *= decay[t][:, None, None]
        d = (v[t] - (s * k[t][:, :, None]).sum(1)) * beta[t][:, None]
        s += k[t][:, :, None] * d[:, None, :]
        out[t] = (s * q[t][:, :, None]).sum(1)
    return out, s


def _rms(x, w):
    return x / (x.square().mean(-1, keepdim=True) + 1e-6).sqrt() * w


def _rotate(x, first):
    """Rotate-half on the first RD dims of [l][heads][HD], the rows at positions first, first + 1, ..."""
    t = torch.arange(first, first + x.shape[0], device=x.device, dtype=torch.float64)[:, None]
    a = t / THETA ** (torch.arange(0, RD, 2, device=x.device, dtype=torch.float64) / RD)
    c, s = a.cos()[:, None], a.sin()[:, None]
    lo, hi = x[..., :RD // 2], x[..., RD // 2:RD]
    return torch.cat([lo * c - hi * s, hi * c + lo * s, x[..., RD:]], -1)


def _attend(big, qw, kw, k_old, v_old):
    """big [l][...] f64, the old rows [HK][p][HD] -> gated output [l][HQ HD], q, and all rows' k and v."""
    l, p = big.shape[0], k_old.shape[1]
    qg = big[:, :2 * HQ * HD].view(l, HQ, 2, HD)
    kv = big[:, 2 * HQ * HD:2 * HQ * HD + 2 * HK * HD].view(l, 2, HK, HD)
    q = _rotate(_rms(qg[:, :, 0], qw), p).transpose(0, 1)
    k = torch.cat([k_old, _rotate(_rms(kv[:, 0], kw), p).transpose(0, 1)], 1)
    v = torch.cat([v_old, kv[:, 1].transpose(0, 1)], 1)
    hide = torch.arange(p + l, device=big.device)[None] > torch.arange(p, p + l, device=big.device)[:, None]
    out = torch.empty(l, HQ, HD, device=big.device, dtype=torch.float64)
    for h in range(HQ):
        s = (q[h] @ k[h // (HQ // HK)].T / math.sqrt(HD)).masked_fill(hide, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[h // (HQ // HK)]
    return (out * torch.sigmoid(qg[:, :, 1])).reshape(l, HQ * HD), q, k, v


class _Torso:
    """The 2B in f64, from the model directory's own files."""

    def __init__(self, d):
        with open(os.path.join(d, "manifest.json")) as f:
            m = json.load(f)
        self.t, self.kinds = m["tensors"], m["config"]["layer_types"]
        self.data = np.memmap(os.path.join(d, "weights.0.bin"), np.uint8, "r")
        e = m["embed"]
        rows = np.memmap(os.path.join(d, e["rows"]), np.uint8, "r").reshape(e["vocab"], e["row_bytes"])
        self.embed, self.qb = rows, e["parts"][0][1]
        with open(os.path.join(d, "head.safetensors"), "rb") as f:
            raw = f.read()
        n = int.from_bytes(raw[:8], "little")
        self.head = {}
        for name, x in json.loads(raw[8:8 + n]).items():
            a, b = x["data_offsets"]
            v = np.frombuffer(raw, np.float32, (b - a) // 4, 8 + n + a).reshape(x["shape"])
            self.head[name] = torch.from_numpy(v.copy()).cuda().double()

    def raw(self, name, dtype):
        t = self.t[name]
        return torch.from_numpy(self.data[t["offset"]:t["offset"] + t["bytes"]].view(dtype).copy()).cuda()

    def vec(self, name):
        return self.raw(name, np.float32).double()

    def mm(self, x, name):
        t = self.t[name + ".q"]
        n, k = t["N"], t["K"]
        w = _dense(self.raw(name + ".q", np.int32).view(n, k // 32, 4),
                   self.raw(name + ".s", np.float16).view(n, k // 32), None, 4, 32)
        return x @ w.T

    def forward(self, ids, cache=None):
        """Final-normed rows of all tokens, and the cache after them."""
        r = torch.from_numpy(np.ascontiguousarray(self.embed[ids])).cuda()
        x = _dense(r[:, :self.qb].contiguous().view(torch.int32).view(len(ids), -1, 4),
                   r[:, self.qb:].contiguous().view(torch.float16), None, 4, 32)
        new, l = [], len(ids)
        for i, kind in enumerate(self.kinds):
            p = "layers.%d." % i
            h = _rms(x, self.vec(p + "in_norm"))
            if kind == "linear_attention":
                c = 2 * H * DK + H * DV
                big = self.mm(h, p + "in_proj")
                hist, s0 = cache[i] if cache else (torch.zeros(3, c, device="cuda", dtype=torch.float64),
                                                   torch.zeros(H, DK, DV, device="cuda", dtype=torch.float64))
                rows = torch.cat([hist, big[:, :c]])
                w = self.vec(p + "conv").view(c, 4)
                y = torch.nn.functional.silu(sum(rows[j:j + l] * w[:, j] for j in range(4)))
                o, s1 = _delta_rule(y[:, :H * DK].reshape(l, H, DK), y[:, H * DK:2 * H * DK].reshape(l, H, DK),
                                    y[:, 2 * H * DK:].reshape(l, H, DV), big[:, c + H * DV:c + H * DV + H],
                                    big[:, c + H * DV + H:c + H * DV + 2 * H], self.vec(p + "neg_exp_A"),
                                    self.vec(p + "dt_bias"), s0)
                z = big[:, c:c + H * DV].reshape(l, H, DV)
                o = (_rms(o, self.vec(p + "gnorm")) * torch.nn.functional.silu(z)).reshape(l, H * DV)
                y, kept = self.mm(o, p + "out_proj"), (rows[-3:], s1)
            else:
                none = torch.zeros(HK, 0, HD, device="cuda", dtype=torch.float64)
                k0, v0 = cache[i] if cache else (none, none)
                o, _, k1, v1 = _attend(self.mm(h, p + "qkv"), self.vec(p + "q_norm"), self.vec(p + "k_norm"), k0, v0)
                y, kept = self.mm(o, p + "o_proj"), (k1, v1)
            x = x + y
            new.append(kept)
            gu = self.mm(_rms(x, self.vec(p + "post_norm")), p + "gate_up")
            half = gu.shape[1] // 2
            x = x + self.mm(torch.nn.functional.silu(gu[:, :half]) * gu[:, half:], p + "down")
        return _rms(x, self.vec("final_norm")), new

    def probs(self, rows):
        """Option rows and the answer row last -> the options' probabilities at temperature 1."""
        mean = rows.mean(-1, keepdim=True)
        n = (rows - mean) / ((rows - mean).square().mean(-1, keepdim=True) + 1e-5).sqrt()
        n = n * self.head["norm.weight"] + self.head["norm.bias"]
        q = self.head["q.weight"] @ n[-1] + self.head["q.bias"]
        k = n[:-1] @ self.head["k.weight"].T + self.head["k.bias"]
        return torch.softmax(k @ q / math.sqrt(q.numel()), -1).cpu().numpy()


def exact(case, seed):
    op = case["op"]
    if op in ("layer", "matmul"):
        names = LAYER if op == "layer" else [case["shape"]]
        out = []
        for i, s in enumerate(names):
            w, sc = _w4(seed, s)
            a = _rows(seed, 40 + i if op == "layer" else 3, case["m"], SHAPES[s][1])
            out.append(a.double() @ _dense(w, sc, None, 4, 32).T)
        return out if op == "layer" else out[0]
    if op == "format":
        w, sc, bi = _format_weights(case, seed)
        return _rows(seed, 3, case["m"], SHAPES[case["shape"]][1]).double() @ _dense(w, sc, bi, case["bits"], case["group"]).T
    if op == "gdn":
        qkv, gates, rate, bias, state = (t.double() for t in _gdn_inputs(case, seed))
        l = case["l"]
        o, s = _delta_rule(qkv[:, :H * DK].reshape(l, H, DK), qkv[:, H * DK:2 * H * DK].reshape(l, H, DK),
                           qkv[:, 2 * H * DK:].reshape(l, H, DV), gates[:, :H], gates[:, H:], rate, bias, state)
        return {"o": o.reshape(l, H * DV), "state": s}
    if op == "attention":
        big, qw, kw, k, v = (t.double() for t in _attn_inputs(case, seed))
        p, l = case["p"], case["l"]
        out, q, k1, v1 = _attend(big, qw, kw, k[:, :p], v[:, :p])
        k[:, :p + l], v[:, :p + l] = k1, v1
        return {"out": out, "q": q.contiguous(), "k": _block_k(k), "v": _block_v(v)}
    torso = _Torso(_model_dir())
    if op == "question":
        _, cache = torso.forward(_tokens(seed, 1, case["p"]))
        ids, rows = _question_ids(case, seed)
        return torso.forward(ids, cache)[0][rows].contiguous()
    if op == "ask":
        ids, qs, opts = _ask_ids(case, seed)
        _, cache = torso.forward(ids)
        return [torso.probs(torso.forward(q, cache)[0][o + [case["q"] - 1]]) for q, o in zip(qs, opts)]
    rows = _spread(case["l"], 4) + [case["l"] - 1]
    return torso.forward(_tokens(seed, 1, case["l"]))[0][rows].contiguous()
