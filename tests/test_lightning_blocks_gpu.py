"""Linear attention in blocks of 64 tokens, one after the other and side by side, against the recurrence in float64: blocks that are not full, key and value
widths that fill no tile, a state that goes on and one that starts, a sequence of no rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _recurrence(q, k, v, decay, S):
    out = []
    for t in range(q.shape[0]):
        S = decay[:, None, None] * S + k[t][:, :, None] * v[t][:, None, :]
        out.append((S * q[t][:, :, None]).sum(1))
    return torch.stack(out), S


@pytest.mark.parametrize("dk,dv", [(64, 64), (128, 128), (8, 20), (72, 40), (104, 150), (48, 300)])
@pytest.mark.parametrize("lens", [(1, 15), (63, 64), (65, 16), (128, 129), (300, 200)])
@pytest.mark.parametrize("silu", [True, False])
def test_blocks(dk, dv, lens, silu):
    from bitnet_c_amd import ops
    H, T = 2, sum(lens)
    g = torch.Generator().manual_seed(T + dk + dv)
    x = torch.randn(T, H * (2 * dk + dv) + 8 - H * dv % 8, generator=g).bfloat16()
    decay = torch.tensor([0.999, 0.3])
    S0 = torch.randn(H, dk, dv, generator=g)
    state = torch.zeros(4, H * dk * dv + 3)
    state[2, :H * dk * dv] = S0.reshape(-1)
    tiles = torch.tensor([(0, 0, lens[0], 0), (1, 0, 0, 0), (2, lens[0], lens[1], 5)], dtype=torch.int32).cuda()
    slots = torch.tensor([1, 3, 2], dtype=torch.int32).cuda()
    scale, got = 0.5, {}
    for pieces in (False, True):
        st = state.clone().cuda()
        o = ops.lightning_scan(x.cuda(), 0, H * dk, 2 * H * dk, decay.cuda(), st, slots, H, dk, dv, tiles=tiles, chain=False, silu=silu, k_scale=scale, pieces=pieces)
        got[pieces] = o.cpu(), st.cpu()
    assert torch.equal(got[False][0], got[True][0]) and torch.equal(got[False][1], got[True][1])
    assert torch.equal(got[True][1][[0, 3]], state[[0, 3]]) and torch.equal(got[True][1][:, H * dk * dv:], state[:, H * dk * dv:])
    act = (lambda z: z * torch.sigmoid(z)) if silu else (lambda z: z)
    q, k, v = (act(x[:, a:a + H * w].double()).reshape(T, H, w) for a, w in ((0, dk), (H * dk, dk), (2 * H * dk, dv)))
    at = 0
    for slot, n, S in ((1, lens[0], torch.zeros(H, dk, dv)), (2, lens[1], S0)):
        want, S = _recurrence(q[at:at + n], k[at:at + n] * scale, v[at:at + n], decay.double(), S.double())
        # a term meets at most one rounding a row and one a token behind it, four of its factors and their activations
        tol = (n + dk + 16) * 2.0 ** -24
        assert float((got[True][0][at:at + n].double() - want.reshape(n, -1)).abs().max()) <= tol * float(want.abs().max())
        assert float((got[True][1][slot, :H * dk * dv].double() - S.reshape(-1)).abs().max()) <= tol * float(S.abs().max())
        at += n


def test_rows_that_are_no_groups_of_eight_go_on_as_before():
    from bitnet_c_amd import ops
    take = ops._fn("lightning", "bn_lightning_blocks_take")
    assert take(1 << 12, 1024, 0, 256, 128, 0) and take(1 << 12, 1024, 8, 256, 8, 0)
    assert not any((take(1 << 12, 1020, 0, 256, 128, 0), take(1 << 12, 1024, 4, 256, 128, 0), take(1 << 12, 1024, 0, 260, 128, 0), take(1 << 12, 1024, 0, 256, 100, 0),
                    take(1 << 12, 1024, 0, 256, 136, 0), take(1 << 12, 1024, 0, 256, 128, 2), take((1 << 12) + 2, 1024, 0, 256, 128, 0)))


@pytest.mark.parametrize("pieces", [False, True])
def test_numbers_that_are_none_reach_no_token_before_them(pieces):
    from bitnet_c_amd import ops
    H, d, T, bad = 1, 128, 150, 70
    g = torch.Generator().manual_seed(3)
    x = torch.randn(T, 3 * d, generator=g).bfloat16().cuda()
    tiles, slots = torch.tensor([(0, 0, T, 0)], dtype=torch.int32).cuda(), torch.zeros(1, dtype=torch.int32).cuda()
    run = lambda: ops.lightning_scan(x, 0, d, 2 * d, torch.tensor([0.9]).cuda(), torch.zeros(1, d * d).cuda(), slots, H, d, d, tiles=tiles, chain=False,
                                     silu=False, pieces=pieces)
    clean = run()
    for col in (5, d + 5, 2 * d + 5):
        kept, x[bad, col] = x[bad, col].clone(), float("inf")
        got = run()
        x[bad, col] = kept
        # the walk of a block with such a value adds it in another order: sums of up to 70 terms and 128 rows
        assert torch.allclose(got[:bad], clean[:bad], rtol=200 * 2.0 ** -24, atol=200 * 2.0 ** -24 * float(clean.abs().max()))
        assert not bool(torch.isfinite(got[bad, 5]))
    assert torch.equal(run(), clean)


@pytest.mark.parametrize("pieces", [False, True])
def test_silu_of_every_number_there_is(pieces):
    """A token whose values are all 2^16 numbers of bf16, infinities and NaN among them, a column each; beside the walk token by token and float64."""
    from bitnet_c_amd import ops
    H, dk, dv = 64, 8, 1024
    v = torch.arange(-2 ** 15, 2 ** 15, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    x = torch.cat([torch.ones(2 * H * dk, dtype=torch.bfloat16), v]).view(1, -1)
    tiles, slots = torch.tensor([(0, 0, 1, 0)], dtype=torch.int32).cuda(), torch.zeros(1, dtype=torch.int32).cuda()
    run = lambda **kw: ops.lightning_scan(x.cuda(), 0, H * dk, 2 * H * dk, torch.full((H,), 0.5).cuda(), torch.zeros(1, H * dk * dv).cuda(), slots, H, dk, dv,
                                          tiles=tiles, silu=True, k_scale=0.125, **kw).cpu().view(-1).double()
    got, chain = run(chain=False, pieces=pieces), run(chain=True)
    one = torch.sigmoid(torch.ones((), dtype=torch.float64))
    want = v.double() * torch.sigmoid(v.double()) * (one * one)         # k . q = 8 (silu 1)^2 / 8
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    for other in (want, chain):
        ok = v.isfinite()
        # a dozen roundings of factors near 1, two of exponents of up to 126; below -87 a value is given as 0
        assert bool(((got - other).abs()[ok] <= 64 * 2.0 ** -24 * other.abs()[ok] + 1.5e-36).all())


def test_which_steps_take_blocks():
    from bitnet_c_amd import ops
    assert ops.lightning_in_blocks((16, 1), 16, 128, 128) and ops.lightning_in_blocks((2048, 64), 16, 128, 128) and not ops.lightning_in_blocks((1984, 64), 16, 128, 128)
    assert ops.lightning_in_pieces(65, 1, 16, 128) and not ops.lightning_in_pieces(64, 1, 16, 128) and not ops.lightning_in_pieces(1024, 4, 16, 128)
    assert ops.lightning_in_pieces(2000, 4, 16, 128) and not ops.lightning_in_pieces(32768, 16, 16, 128)


def test_short_sequences_and_narrow_keys_keep_their_form():
    from bitnet_c_amd import ops
    take, chunks = ops.lightning_takes_blocks, lambda n, *a: bool(ops._fn("lightning", "bn_lightning_prefers_chunks")(n, *a))
    # in the chunked form's place
    assert chunks(1, 16, 128, 128) and chunks(4, 8, 128, 256) and chunks(8, 16, 96, 96)
    assert not take((128, 1), 16, 128, 128) and take((192, 1), 16, 128, 128) and take((16, 1), 32, 64, 64) and not take((16, 1), 32, 16, 64)
    assert take((16, 8), 16, 96, 96) and not take((64, 4), 8, 128, 256) and take((128, 4), 8, 128, 256)
    # in the chain's
    assert not chunks(16, 16, 128, 128) and not chunks(64, 32, 64, 64) and not chunks(8, 64, 32, 32)
    assert take((512, 16), 16, 128, 128) and not take((496, 16), 16, 128, 128) and take((3072, 64), 32, 64, 64) and not take((3008, 64), 32, 64, 64)
    assert take((512, 8), 64, 32, 32) and not take((448, 8), 64, 32, 32) and not take((8192, 16), 64, 32, 32)
    # one block has nothing beside it
    assert not ops.lightning_in_pieces(64, 1, 8, 128) and ops.lightning_in_pieces(65, 1, 8, 128)


@pytest.mark.parametrize("lens,H,dk,dv", [((16,), 4, 64, 64), ((33, 31), 4, 64, 64), ((40,) * 8, 64, 32, 32), ((300, 5), 4, 64, 64)])
def test_the_form_that_is_taken(lens, H, dk, dv):
    """Unasked, the step takes the form that the rule names, bit for bit."""
    from bitnet_c_amd import ops
    T, g = sum(lens), torch.Generator().manual_seed(sum(lens))
    x, decay = torch.randn(T, H * (2 * dk + dv), generator=g).bfloat16().cuda(), torch.linspace(0.5, 0.999, H).cuda()
    at = [sum(lens[:i]) for i in range(len(lens))]
    tiles, slots = torch.tensor([(i, a, n, 0) for i, (a, n) in enumerate(zip(at, lens))], dtype=torch.int32).cuda(), torch.arange(len(lens), dtype=torch.int32).cuda()
    run = lambda **kw: ops.lightning_scan(x, 0, H * dk, 2 * H * dk, decay, torch.zeros(len(lens), H * dk * dv).cuda(), slots, H, dk, dv, tiles=tiles, **kw)
    got, sizes = run(), (T, len(lens))
    if ops.lightning_takes_blocks(sizes, H, dk, dv):
        assert torch.equal(got, run(chain=False))
    elif not ops._fn("lightning", "bn_lightning_prefers_chunks")(len(lens), H, dk, dv):
        assert torch.equal(got, run(chain=True))
    else:                                                 # the chunked form adds up in another order than either
        assert not torch.equal(got, run(chain=False)) and torch.allclose(got, run(chain=True), rtol=1e-3, atol=1e-4)
