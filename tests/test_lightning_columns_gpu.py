"""The chunked form of the linear attention takes 16 or 32 value columns a workgroup, by how many workgroups that makes: a
launch of many sequences (32) gives the bits of one launch a sequence (16), outputs and states."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("H,dk,dv,lens", [(16, 128, 128, [130, 64, 1, 65]), (40, 72, 24, [63, 5, 129, 64, 200]),
                                          (80, 66, 41, [70, 17])])
def test_many_sequences_and_one_at_a_time(H, dk, dv, lens):
    from bitnet_c_amd import ops
    torch.manual_seed(dk + dv)
    B, T = len(lens), sum(lens)
    assert ops.lightning_chunked(dk, dv) and B * H * -(-dv // 16) > 256 >= H * -(-dv // 16)
    x = torch.randn(T, H * (2 * dk + dv), device=DEV)
    decay = torch.rand(H, device=DEV) * 0.2 + 0.8
    state = torch.randn(B + 1, H * dk * dv, device=DEV)
    alone, slots = state.clone(), torch.randperm(B).to(torch.int32)
    tiles, row = [], 0
    for b, n in enumerate(lens):
        tiles.append([b, row, n, 0 if b == 1 else 40])
        row += n
    scan = lambda st, tl: ops.lightning_scan(x, 0, H * dk, 2 * H * dk, decay, st, slots.to(DEV), H, dk, dv,
                                             tiles=torch.tensor(tl, dtype=torch.int32, device=DEV), chain=False)
    together = scan(state, tiles)
    for t in tiles:
        rows = slice(t[1], t[1] + t[2])
        assert torch.equal(scan(alone, [t])[rows], together[rows])
    assert torch.isfinite(together).all() and torch.equal(state, alone)


def test_which_launches_take_32_columns():
    """Those whose rounds over the 256 CUs are then the shorter ones; never where 32 columns save no workgroup."""
    from bitnet_c_amd import ops
    columns = ops._fn("lightning", "bn_lightning_columns")
    assert columns(4, 16, 128, 128) == 32 and columns(1, 32, 128, 128) == 16 and columns(2, 32, 128, 128) == 32
    assert columns(2, 16, 128, 128) == 16 and columns(5, 40, 72, 24) == 32 and columns(2, 65, 128, 48) == 16
    assert all(columns(n, h, 128, dv) == 16 for n in (1, 8, 31) for h in (16, 64) for dv in (1, 16))
    assert columns(31, 64, 64, 128) == 16


# one token of every sequence: the same bits as the walk of a step that holds that token alone.  key widths: one row, the edges of
# the forms' rows; value columns under, at and over a workgroup's 64; sequences at their first token and a padding row
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dk,dv", [(1, 64), (32, 33), (33, 128), (64, 65), (100, 70), (128, 128), (129, 64), (256, 100)])
@pytest.mark.parametrize("silu", [True, False])
def test_decode_step_gives_the_bits_of_the_walk(dtype, dk, dv, silu):
    from bitnet_c_amd import ops
    H, B = 3, 5
    g = torch.Generator().manual_seed(dk + dv)
    x = torch.randn(B, H * (2 * dk + dv) + 3, generator=g).to(dtype).cuda()
    decay = torch.rand(H, generator=g).cuda()
    state = torch.randn(B + 1, H * dk * dv, generator=g).cuda()
    slots, lens = torch.tensor([3, 0, 5, 1, 4], dtype=torch.int32).cuda(), torch.tensor([1, 9, 0, 2, 70], dtype=torch.int32).cuda()
    tiles = torch.tensor([[i, i, 1, int(lens[i]) - 1] for i in (0, 1, 3, 4)], dtype=torch.int32).cuda()
    kw = dict(silu=silu, k_scale=1.0 if silu else 0.25)
    a, b = state.clone(), state.clone()
    got = ops.lightning_scan(x, 0, H * dk, 2 * H * dk, decay, a, slots, H, dk, dv, seq_lens=lens, **kw)
    want = ops.lightning_scan(x, 0, H * dk, 2 * H * dk, decay, b, slots, H, dk, dv, tiles=tiles, chain=True, **kw)
    live = [0, 1, 3, 4]
    assert torch.equal(got[live], want[live]) and torch.equal(a, b)
