"""The dispatch rules' lines: which launches calls on either side of them make."""
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


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
