"""The attention kernel that takes 32 (query, head) rows per workgroup (more than 128 rows, a power of two
of query heads per kv head), against the CPU oracle: edges of its tiles and key blocks, every group size
it takes, both query paths, scores that raise the running maximum block after block, and the group sizes
it leaves to the other kernel."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
I = ctypes.c_int
HD, CTX = 256, 4096


def dev(a):
    a = np.ascontiguousarray(a)
    return torch.from_numpy(a.view(np.uint8).reshape(-1).copy()).cuda()


def check(sdamd, o, seed, hq, hk, L, P, rd=64, gain=1.0, shift=0, own=False):
    """P prefix rows straight in the cache, then L rows; out within 2 f16 ulp + 1e-3 of the oracle (scores,
    softmax and P V in f32 against the oracle's f64 softmax: the bound of the other attention tests).  own: the
    oracle's attention takes the queries and the cache that the GPU prepared, so that only scores, softmax and P V
    differ."""
    from conftest import f16_ulp
    rng = np.random.default_rng(seed)
    qw = (gain * (1 + 0.1 * rng.standard_normal(HD))).astype(np.float32)
    kw = (1 + 0.1 * rng.standard_normal(HD)).astype(np.float32)
    rope = o.rope_table(rd, 1e7)
    stride = 2 * hq * HD + 2 * hk * HD
    big = rng.standard_normal((L, stride)).astype(np.float16)
    oK, oV = np.zeros((hk, CTX, HD), np.uint16), np.zeros((hk, CTX, HD), np.uint16)
    oK[:, :P] = rng.standard_normal((hk, P, HD)).astype(np.float16).view(np.uint16)
    oV[:, :P] = rng.standard_normal((hk, P, HD)).astype(np.float16).view(np.uint16)
    dK = dev(oK.reshape(hk, CTX // 32, 32, HD // 32, 32).transpose(0, 1, 3, 2, 4))
    dV = dev(oV.reshape(hk, CTX // 32, 32, HD).transpose(0, 1, 3, 2))
    if shift:  # the cache starts `shift` bytes past a 16-byte piece
        pad = torch.zeros(shift, dtype=torch.uint8, device="cuda")
        dK, dV = (torch.cat([pad, t])[shift:] for t in (dK, dV))
        assert dK.data_ptr() % 16 == shift and dV.data_ptr() % 16 == shift
    dbig, dqw, dkw, drope = dev(big), dev(qw), dev(kw), dev(rope)
    dQ = torch.zeros(hq * L * HD * 2, dtype=torch.uint8, device="cuda")
    dout = torch.full((L * hq * HD * 2,), 0xFF, dtype=torch.uint8, device="cuda")  # NaN until written
    sdamd.op_attention(dbig.data_ptr(), stride, dqw.data_ptr(), dkw.data_ptr(), drope.data_ptr(), L, P, hq, hk, HD, rd,
                       dQ.data_ptr(), dK.data_ptr(), dV.data_ptr(), CTX, dout.data_ptr())
    torch.cuda.synchronize()
    Q = np.empty((hq, L, HD), np.uint16)
    o.lib().or_qk_prep(o.P(big.view(np.uint16)), I(stride), o.P(qw), o.P(kw), o.P(rope), I(L), I(P), I(CTX), I(hq),
                       I(hk), I(HD), I(rd), o.P(Q), o.P(oK), o.P(oV))
    if own:
        Q = dQ.cpu().numpy().view(np.uint16).reshape(hq, L, HD).copy()
        oK = dK.cpu().numpy().view(np.uint16).reshape(hk, CTX // 32, HD // 32, 32, 32).transpose(0, 1, 3, 2, 4).reshape(hk, CTX, HD).copy()
        oV = dV.cpu().numpy().view(np.uint16).reshape(hk, CTX // 32, HD, 32).transpose(0, 1, 3, 2).reshape(hk, CTX, HD).copy()
    out = np.empty((L, hq * HD), np.uint16)
    o.lib().or_attn(o.P(Q), o.P(oK), o.P(oV), o.P(big.view(np.uint16)), I(stride), I(L), I(P), I(CTX), I(hq), I(hk),
                    I(HD), o.P(out))
    got = dout.cpu().numpy().view(np.float16).reshape(L, hq * HD).astype(np.float32)
    want = o.h2f(out)
    # a large gain on q: the 1-ulp f16 difference of a query (2^-11) moves its scores (up to ~100) by ~0.05,
    # which is a factor e^0.05 between two keys' weights
    extra = 1e-3 if gain == 1.0 else 5e-2
    if own:
        # a score is 256 f32 products and sums, off by about 16 x 2^-24 of the sum of their magnitudes, which moves a
        # weight and the weights' sum by as much relative to itself, and the output by twice that of the values
        q, k, v = (np.abs(o.h2f(x)[:, :P + L]) for x in (Q, oK, oV))
        sums = max(float((q[h] @ k[h // (hq // hk)].T).max()) / 16 for h in range(hq))
        extra = 2 * 16 * 2.0 ** -24 * sums * float(v.max())
        assert extra < 1e-2
    bad = ~(np.abs(got - want) <= 2.0 * f16_ulp(want) + extra)
    assert not bad.any(), (f"L={L} P={P} heads {hq}/{hk}: {int(bad.sum())} outputs off, "
                           f"max {np.abs(got - want).max():.3g}")


@pytest.mark.parametrize("L,P", [(129, 0), (129, 31), (136, 31), (150, 0), (150, 40), (159, 64), (193, 33), (256, 0), (257, 95), (264, 0), (300, 0), (513, 700)])
def test_rows_kernel_edges(sdamd, oracle, L, P):
    """Ragged last tiles (8 queries each), prefixes that end inside a 32-key block, splits of 1, 2 and 4; without a
    prefix the other kernel up to 256 rows."""
    check(sdamd, oracle, L + P, 8, 2, L, P)


@pytest.mark.parametrize("hq,hk", [(2, 2), (4, 2), (8, 1), (16, 1), (6, 2)])
@pytest.mark.parametrize("L,P", [(141, 50), (269, 50)])
def test_rows_kernel_groups(sdamd, oracle, hq, hk, L, P):
    """1, 2, 8 and 16 query heads per kv head (32, 16, 4 and 2 queries per tile); 3 take the other kernel, as 2
    query heads do up to 256 rows."""
    check(sdamd, oracle, 7 * hq + hk, hq, hk, L, P)


@pytest.mark.parametrize("L,P", [(160, 0), (160, 70), (300, 33)])
def test_cache_that_starts_between_16_byte_pieces(sdamd, oracle, L, P):
    """The other kernel takes it, with and without key splits."""
    check(sdamd, oracle, 3 * L + P, 8, 2, L, P, shift=8)


def test_rows_kernel_reads_prepared_queries(sdamd, oracle):
    """rotary_dim 32: the queries come from qk_prep's buffer."""
    check(sdamd, oracle, 5, 8, 2, 170, 40, rd=32)


def test_rows_kernel_raises_its_maximum(sdamd, oracle):
    """Queries scaled by 12: scores of a standard deviation of 12 in the exponent, so the running maximum
    rises by more than the kernel's slack again and again.  From the GPU's own queries (the kernel that reads
    them prepared) the oracle's scores are the same but for the f32 sums."""
    check(sdamd, oracle, 9, 8, 2, 400, 100, gain=12.0)
    check(sdamd, oracle, 9, 8, 2, 400, 100, gain=12.0, rd=32, own=True)
    check(sdamd, oracle, 10, 8, 2, 200, 900, gain=12.0, rd=32, own=True)


def test_a_tile_of_one_query_is_as_fast_as_one_of_two(sdamd):
    """257 and 258 rows have the same tiles and key blocks but for the last tile's one or two queries.  The faster
    of 9 rounds each, in turn; before the rows past the last were kept running it was 1.06 to 1.13."""
    hq, hk, rd, calls = 8, 2, 64, {}
    stride = 2 * hq * HD + 2 * hk * HD
    w, rope = torch.ones(HD, device="cuda"), torch.zeros(CTX, rd // 2, 2, device="cuda")
    for L in (257, 258):
        big, out = torch.randn(L, stride, device="cuda").half(), torch.zeros(L, hq * HD, device="cuda").half()
        K, V, Q = (torch.randn(n, device="cuda").half() for n in (hk * CTX * HD, hk * CTX * HD, hq * L * HD))

        def call(L=L, big=big, out=out, K=K, V=V, Q=Q):
            sdamd.op_attention(big.data_ptr(), stride, w.data_ptr(), w.data_ptr(), rope.data_ptr(), L, 0, hq, hk, HD, rd,
                               Q.data_ptr(), K.data_ptr(), V.data_ptr(), CTX, out.data_ptr(),
                               torch.cuda.current_stream().cuda_stream)
        call()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for _ in range(20):
                call()
        calls[L] = g
    best = dict.fromkeys(calls, float("inf"))
    a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    for _ in range(9):
        for L, g in calls.items():
            g.replay()
            a.record()
            g.replay()
            b.record()
            torch.cuda.synchronize()
            best[L] = min(best[L], a.elapsed_time(b))
    assert best[257] < 1.04 * best[258], best
