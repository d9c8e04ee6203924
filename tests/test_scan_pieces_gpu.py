"""The wkv and min-GRU recurrences over sequences cut into pieces against the plain walk, and the token shift's wide form
against the narrow one."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rand(shape, seed, lo=-1.0, hi=1.0):
    g = torch.Generator().manual_seed(seed)
    return lo + (hi - lo) * torch.rand(shape, generator=g)


def _close(got, want, walks):
    """Both are float32 sums of the same terms; a term passes through at most `walks` roundings of 2^-24 more."""
    scale = want.abs().max()
    return float((got - want).abs().max()) <= walks * 2.0 ** -24 * 4 * float(scale)


# lengths: shorter than a piece, its edges, several pieces, a last piece of one token; a tile of no rows between them; the
# second sequence continues one (position 5)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,d", [(2, 64), (3, 24), (1, 128)])
@pytest.mark.parametrize("lens", [[1, 63], [64, 65], [300, 129], [257, 2]])
def test_wkv_pieces(dtype, H, d, lens):
    from bitnet_c_amd import ops
    T, A, D = sum(lens), H * d, 40
    r, k, v, dd, h = (_rand((T, w), 10 + i).to(dtype).cuda() for i, w in enumerate((A, A, A, A, D)))
    w0, u = _rand((A,), 20, -4.0, 0.0).cuda(), _rand((A,), 21).cuda()
    n = ops.wkv_state_floats(H, d, d)
    dk_pad = n // (H * d)
    state = torch.zeros(4, n + D)
    P = dk_pad // ops.WKV_ROWS_PER_THREAD                 # rows beyond dk stay zero, as the kernel keeps them
    S = _rand((H, ops.WKV_ROWS_PER_THREAD, d, P), 22)
    rows = torch.arange(P)[None, :] * ops.WKV_ROWS_PER_THREAD + torch.arange(ops.WKV_ROWS_PER_THREAD)[:, None]
    S = torch.where((rows < d)[None, :, None, :], S, torch.zeros(()))
    state[2, :n] = S.reshape(-1)
    tiles = torch.tensor([(0, 0, lens[0], 0), (1, 0, 0, 0), (2, lens[0], lens[1], 5)], dtype=torch.int32).cuda()
    slots = torch.tensor([1, 3, 2], dtype=torch.int32).cuda()
    out = {}
    for pieces in (False, True):
        st = state.clone().cuda()
        o = ops.wkv_scan(r, k, v, dd, w0, u, h, st, slots, H, d, d, tiles=tiles, pieces=pieces)
        out[pieces] = o.cpu(), st.cpu()
    assert _close(out[True][0], out[False][0], max(lens) + d) and _close(out[True][1][:, :n], out[False][1][:, :n], max(lens) + 4)
    assert torch.equal(out[True][1][:, n:], out[False][1][:, n:])                    # the last rows
    assert torch.equal(out[True][1][[0, 3]], state[[0, 3]])                          # rows of no sequence


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("W", [64, 100])
@pytest.mark.parametrize("lens", [[1, 63], [64, 65], [300, 129], [257, 2]])
def test_mingru_pieces(dtype, W, lens):
    from bitnet_c_amd import ops
    T = sum(lens)
    zxg = _rand((T, 3 * W), 1, -3.0, 3.0).to(dtype).cuda()
    bz, bx, state = _rand((W,), 2).cuda(), _rand((W,), 3).cuda(), _rand((4, W + 3), 4)
    tiles = torch.tensor([(0, 0, lens[0], 0), (1, 0, 0, 0), (2, lens[0], lens[1], 5)], dtype=torch.int32).cuda()
    slots = torch.tensor([1, 3, 2], dtype=torch.int32).cuda()
    out = {}
    for pieces in (False, True):
        st = state.clone().cuda()
        y = ops.mingru_scan(zxg, bz, bx, st, slots, W, tiles=tiles, pieces=pieces)
        out[pieces] = y.float().cpu(), st.cpu()
    # a state is a chain of one multiply-add a token; bf16 outputs of states that differ by a rounding may fall on
    # neighbouring numbers (2^-8)
    scale = float(out[False][0].abs().max())
    assert float((out[True][0] - out[False][0]).abs().max()) <= (2.0 ** -8 if dtype == torch.bfloat16 else 512 * 2.0 ** -24) * scale
    assert _close(out[True][1][:, :W], out[False][1][:, :W], 512)
    assert torch.equal(out[True][1][:, W:], state[:, W:]) and torch.equal(out[True][1][[0, 3]], state[[0, 3]])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,D", [(1, 8), (5, 2048), (1023, 16), (1027, 2056), (1024, 4096)])
def test_token_shift_wide(dtype, T, D):
    """The 16-byte form against the narrow one, which a state at an odd address goes to: the same bits."""
    from bitnet_c_amd import ops
    h, mu = _rand((T, D), 5).to(dtype).cuda(), _rand((3, D), 6).cuda()
    cut = T // 3
    positions = torch.cat([torch.arange(7, 7 + cut), torch.arange(T - cut - T // 4), torch.full((T // 4,), -1)]).int()[:T]
    seq = torch.cat([torch.zeros(cut), torch.ones(T - cut)]).int()
    slots = torch.tensor([2, 0], dtype=torch.int32).cuda()
    plain = _rand((3, D + 8), 7).cuda()
    odd = torch.zeros(3, D + 9).cuda()
    odd[:, :D] = plain[:, :D]
    a = ops.token_shift(h, mu, plain, positions.cuda(), seq.cuda(), slots)
    b = ops.token_shift(h, mu, odd, positions.cuda(), seq.cuda(), slots)
    assert torch.equal(a, b)


# widths around the narrowest that the wide form takes, and steps around the smallest whose workgroups take four rows
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,D", [(5, 504), (5, 512), (1, 520), (731, 4096), (733, 4096), (367, 4096), (5901, 512)])
def test_token_shift_forms(dtype, T, D):
    test_token_shift_wide(dtype, T, D)


# one token of every sequence: the same bits as the walk of a step that holds that token alone; channels under, at and over a
# workgroup's 64, sequences at their first token and a padding row
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("W,bias", [(1, True), (64, False), (65, True), (2048, True)])
def test_mingru_decode_step(dtype, W, bias):
    from bitnet_c_amd import ops
    g = torch.Generator().manual_seed(W)
    B = 5
    zxg = torch.randn(B, 3 * W + 8, generator=g).to(dtype).cuda()[:, :3 * W]
    bz, bx = (torch.randn(W, generator=g).cuda() if bias else None for _ in range(2))
    state = torch.randn(B + 1, W + 4, generator=g).cuda()
    slots, lens = torch.tensor([3, 0, 5, 1, 4], dtype=torch.int32).cuda(), torch.tensor([1, 9, 0, 2, 70], dtype=torch.int32).cuda()
    a, b = state.clone(), state.clone()
    got = ops.mingru_scan(zxg, bz, bx, a, slots, W, seq_lens=lens)
    tiles = torch.tensor([[i, i, 1, int(lens[i]) - 1] for i in (0, 1, 3, 4)], dtype=torch.int32).cuda()
    want = ops.mingru_scan(zxg, bz, bx, b, slots, W, tiles=tiles)
    live = [0, 1, 3, 4]
    assert torch.equal(got[live], want[live]) and torch.equal(a, b)
