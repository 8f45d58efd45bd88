"""Many rows of the formats that keep the model's layout (int2, int3, asymmetric, group above 32), which run
on the kernel that dequantizes a weight once per 32 or 64 rows, against the CPU oracle's f32 dequant."""
import numpy as np
import pytest

from golden import cases as gcases

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def dev(a):
    a = np.ascontiguousarray(a)
    return torch.from_numpy(a.view(np.uint8).reshape(-1).copy()).cuda()


# the first size of the rule (more than 256 workgroups of 16 columns x 32 rows), one row past a tile of 32 and of
# 64, ragged columns, k steps that are no multiple of the ring's four nor of the two parts, one step in all
@pytest.mark.parametrize("M,N,K", [(65, 2048, 512), (97, 1376, 640), (257, 2048, 128), (321, 2000, 896), (700, 200, 384),
                                   (1025, 520, 1152)])
@pytest.mark.parametrize("bits,group,asym", [(4, 64, False), (4, 32, True), (3, 32, False), (3, 128, True), (2, 64, False),
                                             (2, 32, True)])
def test_many_rows(sdamd, oracle, M, N, K, bits, group, asym):
    """Within one f16 ulp of the oracle, plus 2e-5 for the f32 summation order (the bound of the GEMV's own
    tests)."""
    from conftest import f16_ulp
    rng = np.random.default_rng(bits * 1000 + group + M + N + K + asym)
    A = rng.standard_normal((M, K)).astype(np.float16)
    codes = rng.integers(0, 1 << bits, size=(N, K), dtype=np.uint32)
    W = gcases.pack_codes(codes, bits)
    S = rng.uniform(0.005, 0.03, size=N * K // group).astype(np.float16)
    B = rng.uniform(-0.1, 0.1, size=N * K // group).astype(np.float16) if asym else None
    dA, dW, dS, dB = dev(A), dev(W), dev(S), dev(B) if asym else None
    dY = torch.full((M * N * 2,), 0xAB, dtype=torch.uint8, device="cuda")
    sdamd.op_matmul_fmt(dA.data_ptr(), dW.data_ptr(), dS.data_ptr(), dB.data_ptr() if asym else None, dY.data_ptr(),
                        M, N, K, bits, group, asym)
    torch.cuda.synchronize()
    got = dY.cpu().numpy().view(np.float16).reshape(M, N).astype(np.float32)
    want = oracle.h2f(oracle.matmul(A.view(np.uint16), W, S.view(np.uint16), N, K, False, bits=bits, group=group,
                                    asym=asym, Bi=None if B is None else B.view(np.uint16)))
    err = np.abs(got - want)
    assert (err <= 1.01 * f16_ulp(want) + 2e-5).all(), f"max err {err.max()}"


@pytest.mark.parametrize("M,N", [(7, 8256), (8, 8192), (8, 8256), (16, 5120), (16, 8256), (17, 4096), (17, 4112)])
def test_both_sides_of_the_line_at_few_rows(sdamd, oracle, M, N):
    """Up to 16 rows the kernel runs from 8 rows and 513 blocks of 16 columns on, above from 257 on; the GEMV
    takes the others."""
    test_many_rows(sdamd, oracle, M, N, 256, 3, 64, True)


def test_rows_that_start_between_16_byte_pieces(sdamd):
    """A at 8 bytes past a piece (the GEMV takes it): the aligned call's result, but for the f32 summation order."""
    from conftest import f16_ulp
    M, N, K = 80, 2048, 512
    rng = np.random.default_rng(3)
    A = rng.standard_normal((M, K)).astype(np.float16)
    W = gcases.pack_codes(rng.integers(0, 8, size=(N, K), dtype=np.uint32), 3)
    S, B = (rng.uniform(-0.05, 0.05, size=N * K // 64).astype(np.float16) for _ in range(2))
    dA, dW, dS, dB = dev(A), dev(W), dev(S), dev(B)
    dU = torch.zeros(M * K * 2 + 16, dtype=torch.uint8, device="cuda")
    dU[8:8 + M * K * 2] = dA
    got = []
    for a in (dA.data_ptr(), dU.data_ptr() + 8):
        y = torch.zeros(M * N * 2, dtype=torch.uint8, device="cuda")
        sdamd.op_matmul_fmt(a, dW.data_ptr(), dS.data_ptr(), dB.data_ptr(), y.data_ptr(), M, N, K, 3, 64, True)
        torch.cuda.synchronize()
        got.append(y.cpu().numpy().view(np.float16).astype(np.float32))
    assert (np.abs(got[0] - got[1]) <= 1.01 * f16_ulp(got[0]) + 2e-5).all()


def test_rows_past_the_last_are_not_written(sdamd):
    """The output ends at row M (a tile holds 32 or 64)."""
    M, N, K = 65, 2048, 256
    z = torch.zeros(N * K, dtype=torch.uint8, device="cuda")
    y = torch.full(((M + 64) * N * 2,), 0xAB, dtype=torch.uint8, device="cuda")
    a = torch.zeros(M * K * 2, dtype=torch.uint8, device="cuda")
    sdamd.op_matmul_fmt(a.data_ptr(), z.data_ptr(), z.data_ptr(), None, y.data_ptr(), M, N, K, 3, 64, False)
    torch.cuda.synchronize()
    assert (y[:M * N * 2] == 0).all() and (y[M * N * 2:] == 0xAB).all()


@pytest.mark.parametrize("n", [130, 500])
def test_model_of_other_formats_many_rows(sdamd, synth, n, tmp_path):
    """A forward whose projections are all in other formats (partial outputs with k splits among them) against
    the same tokens as a state and its continuation of 20 (the GEMV rows)."""
    fmt = {"in_proj": (3, 64, True), "out_proj": (2, 32, False), "qkv": (4, 64, True), "o_proj": (3, 32, False),
           "gate_up": (4, 128, False), "down": (3, 128, True)}
    cfg = dict(synth.CONFIG_TINY, hidden_size=2048, layer_types=["linear_attention", "full_attention"])
    eng, _, _ = sdamd.load_decider(synth.write_model(str(tmp_path), cfg, vocab=2048, seed=3, mat_fmt=fmt))
    ids = np.random.default_rng(n).integers(0, 2048, n).astype(np.uint32)
    whole = eng.forward(ids, [n - 20, n - 1]).hidden
    prefix = eng.forward(ids[:n - 20], [], keep=True).snapshot
    part = eng.forward(ids[n - 20:], [0, 19], cache=prefix).hidden
    eng.free()
    err = float(np.abs(whole - part).max())
    assert err < 2e-2, err
