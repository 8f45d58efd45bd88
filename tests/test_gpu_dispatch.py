"""The dispatch rules' lines: which launches calls on either side of them make."""
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


ROWS, QUERIES = "32 (query, head) rows per workgroup", "16 queries of a head per workgroup"


@pytest.mark.parametrize("hq,hk,L,P,kernel,ks", [
    (8, 2, 128, 512, QUERIES, 4), (8, 2, 129, 512, ROWS, 4), (8, 2, 200, 512, ROWS, 2), (8, 2, 256, 2048, ROWS, 2),
    (8, 2, 257, 512, ROWS, 1), (16, 2, 250, 512, ROWS, 1),
    (2, 2, 129, 512, QUERIES, 8), (2, 2, 256, 2048, QUERIES, 8), (2, 2, 257, 512, ROWS, 1), (4, 1, 129, 512, ROWS, 4),
    (8, 2, 128, 0, QUERIES, 4), (8, 2, 129, 0, QUERIES, 1), (8, 2, 256, 0, QUERIES, 1), (8, 2, 257, 0, ROWS, 1),
    (16, 1, 256, 0, QUERIES, 1), (32, 8, 129, 0, ROWS, 1), (2, 2, 256, 0, QUERIES, 1), (6, 2, 129, 0, QUERIES, 1),
    (6, 2, 200, 512, QUERIES, 2), (6, 2, 300, 512, QUERIES, 1)])
def test_attention_kernel_and_splits(sdamd, hq, hk, L, P, kernel, ks):
    """Which attention kernel runs, in how many key splits (a combine follows more than one)."""
    from launches import launches
    hd, ctx, stride = 256, 4096, 2 * hq * 256 + 2 * hk * 256
    big, out, q = (torch.zeros(n, device="cuda").half() for n in (L * stride, L * hq * hd, L * hq * hd))
    w, rope = torch.ones(hd, device="cuda"), torch.zeros(ctx, 32, 2, device="cuda")
    k, v = (torch.zeros(hk * ctx * hd, device="cuda").half() for _ in range(2))
    got = launches(sdamd, lambda s: sdamd.op_attention(big.data_ptr(), stride, w.data_ptr(), w.data_ptr(), rope.data_ptr(), L, P, hq,
                                                       hk, hd, 64, q.data_ptr(), k.data_ptr(), v.data_ptr(), ctx, out.data_ptr(), s))
    assert len(got) == (4 if ks > 1 else 3), got  # two integers, the rows' k and v, attention, the combine
    grid = (hk, -(-L * (hq // hk) // 32), ks) if kernel is ROWS else (-(-L // 16), hq, ks)
    assert got[2][0] == grid, got


@pytest.mark.parametrize("M,N,K,rows,columns,threads", [
    (2561, 5120, 2048, 128, 256, 256), (2561, 7168, 2048, 96, 128, 256), (2800, 7168, 2048, 128, 256, 256),  # two column tiles per wave
    (2700, 9216, 512, 96, 128, 256), (2700, 16384, 256, 128, 128, 256), (3200, 4096, 1024, 128, 256, 256),
    (2561, 2048, 2048, 128, 256, 512), (2560, 2048, 2560, 128, 128, 256), (4096, 1280, 4096, 128, 256, 512),  # and k halves
    (4096, 1024, 1024, 128, 128, 256), (2816, 1536, 2048, 128, 128, 256), (2561, 2048, 1024, 128, 128, 256)])
def test_long_prefill_tiles(sdamd, M, N, K, rows, columns, threads):
    """The tile of an int4 matmul above 2560 rows: its grid and workgroup size."""
    from launches import launches
    a, w, s, y = (torch.zeros(n, device="cuda").half() for n in (M * K, N * K // 4, N * K // 32, M * N))
    got = launches(sdamd, lambda st: sdamd.op_matmul(a.data_ptr(), w.data_ptr(), s.data_ptr(), y.data_ptr(), M, N, K, False, -1, True, st))
    assert got == [((-(-N // columns), -(-M // rows), 1), threads)], got


@pytest.mark.parametrize("M,N,K,many", [(7, 8256, 256, False), (8, 8192, 256, False), (8, 8256, 256, True), (16, 5120, 256, False),
                                        (17, 4096, 256, False), (17, 4112, 256, True), (64, 4096, 256, True),
                                        (64, 4096, 128, False), (65, 4096, 128, True), (300, 2048, 192, False)])
def test_other_formats_at_many_rows(sdamd, M, N, K, many):
    """The kernel that dequantizes a weight once per 32 or 64 rows (64 columns per workgroup; 16 for the other)."""
    from launches import launches
    a, w, s, y = (torch.zeros(n, device="cuda").half() for n in (M * K, N * K * 3 // 16, N * K // 32, M * N))
    got = launches(sdamd, lambda st: sdamd.op_matmul_fmt(a.data_ptr(), w.data_ptr(), s.data_ptr(), None, y.data_ptr(), M, N, K, 3, 32,
                                                         False, st))
    assert len(got) == 1 and got[0][0][0] == -(-N // (64 if many else 16)), got


@pytest.mark.parametrize("H,L,load,copied,halves", [(16, 1024, True, True, 2), (16, 1023, True, False, 1), (16, 1024, False, False, 2),
                                                    (17, 1024, True, False, 1), (34, 1100, True, False, 1)])
def test_gdn_copies_its_state_only_for_two_workgroups_per_slice(sdamd, H, L, load, copied, halves):
    """A long continuation starts from a copy of its state where the scan then runs as two workgroups per slice: up
    to 16 heads."""
    from launches import launches
    qkv, gates, o = torch.zeros(L, 3 * H * 128, device="cuda"), torch.zeros(L, 2 * H, device="cuda").half(), torch.zeros(L, H * 128, device="cuda")
    rate, bias, state = torch.full((H,), -1.0, device="cuda"), torch.zeros(H, device="cuda"), torch.zeros(H, 128, 128, device="cuda")
    got = launches(sdamd, lambda s: sdamd.op_gdn(qkv.data_ptr(), gates.data_ptr(), 2 * H, 0, H, rate.data_ptr(), bias.data_ptr(), L, H,
                                                 128, 128, state.data_ptr(), load, o.data_ptr(), s))
    assert len(got) == (3 if copied else 2), got
    assert got[-1][0] == (H, 8, halves), got
