"""The wkv recurrence sixteen tokens at a time, whole sequences and pieces, against the recurrence in float64: blocks that are not full, heads and
columns that fill no tile, decays that vanish within a block, and numbers that are none."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _recurrence(r, k, v, d, w0, u, S, H, dk, dv):
    """float64: o [T, H dv] and the state behind them; S [H, dk, dv]."""
    T = r.shape[0]
    r, k, d = (t.double().reshape(T, H, dk) for t in (r, k, d))
    v, u, w0 = v.double().reshape(T, H, dv), u.double().reshape(H, dk, 1), w0.double().reshape(H, dk)
    S, out = S.double(), []
    for t in range(T):
        kv = k[t][:, :, None] * v[t][:, None, :]
        out.append(((S + u * kv) * r[t][:, :, None]).sum(1))
        S = torch.exp(-torch.exp(d[t] + w0))[:, :, None] * S + kv
    return torch.stack(out).reshape(T, H * dv), S


def _place(S, P):
    """[H, dk, dv] in the kernel's order: (row p 16 + ii, column j) at (ii dv + j) P + p."""
    H, dk, dv = S.shape
    full = torch.zeros(H, P * 16, dv)
    full[:, :dk] = S
    return full.reshape(H, P, 16, dv).permute(0, 2, 3, 1).reshape(-1)


CASES = [(2, 64, 64), (1, 128, 128), (3, 36, 20), (1, 100, 128), (2, 64, 60), (1, 40, 72)]      # the last: more columns than the blocks' waves own


@pytest.mark.parametrize("pieces", [False, True])
@pytest.mark.parametrize("H,dk,dv", CASES)
@pytest.mark.parametrize("lens,decay", [((1, 15), 0.0), ((16, 17), 3.0), ((64, 65), -4.0), ((79, 130), -1.0), ((3, 200), 6.0)])
def test_blocks(H, dk, dv, lens, decay, pieces):
    from bitnet_c_amd import ops
    T, D = sum(lens), 40
    g = torch.Generator().manual_seed(T + dk)
    rnd = lambda *s: torch.randn(*s, generator=g)
    wide = rnd(T, 3 * H * dk + 4).bfloat16()                                  # r, k and d as columns of one product
    r, k, d = (wide[:, q * H * dk:(q + 1) * H * dk] for q in range(3))
    v, h = rnd(T, H * dv).bfloat16(), rnd(T, D).bfloat16()
    w0, u = rnd(H * dk) + decay, rnd(H * dk)
    n = ops.wkv_state_floats(H, dk, dv)
    P = n // (H * dv * 16)
    S0 = rnd(H, dk, dv)
    state = torch.zeros(4, n + D)
    state[2, :n] = _place(S0, P)
    tiles = torch.tensor([(0, 0, lens[0], 0), (1, 0, 0, 0), (2, lens[0], lens[1], 5)], dtype=torch.int32).cuda()
    slots = torch.tensor([1, 3, 2], dtype=torch.int32).cuda()
    st, wc = state.clone().cuda(), wide.cuda()
    o = ops.wkv_scan(*(wc[:, q * H * dk:(q + 1) * H * dk] for q in (0, 1)), v.cuda(), wc[:, 2 * H * dk:3 * H * dk], w0.cuda(), u.cuda(), h.cuda(), st,
                     slots, H, dk, dv, tiles=tiles, pieces=pieces).cpu()
    at = 0
    for slot, length, S in ((1, lens[0], torch.zeros(H, dk, dv)), (2, lens[1], S0)):
        rows = slice(at, at + length)
        at += length
        want, S = _recurrence(r[rows], k[rows], v[rows], d[rows], w0, u, S, H, dk, dv)
        # a term of a sum passes through at most one rounding a token behind it and one a row; the sums' terms are about sqrt(dk) times smaller
        # than their largest values, whose scale the bound is taken from
        tol = (length + dk + 8) * 2.0 ** -24
        assert float((o[rows].double() - want).abs().max()) <= tol * float(want.abs().max())
        assert float((st[slot, :n].cpu().double() - _place(S, P).double()).abs().max()) <= tol * float(S.abs().max())
        assert torch.equal(st[slot, n:].cpu(), h[rows][-1].float())
    assert torch.equal(st[[0, 3]].cpu(), state[[0, 3]])


@pytest.mark.parametrize("pieces", [False, True])
@pytest.mark.parametrize("what", ["v", "k", "r"])
def test_numbers_that_are_none_reach_no_token_before_them(what, pieces):
    from bitnet_c_amd import ops
    H, d, T, bad = 1, 64, 100, 70
    g = torch.Generator().manual_seed(3)
    t = {n: torch.randn(T, d, generator=g).bfloat16().cuda() for n in "rkvd"}
    w0, u, h = torch.zeros(d).cuda(), torch.ones(d).cuda(), torch.zeros(T, 8).bfloat16().cuda()
    tiles, slots = torch.tensor([(0, 0, T, 0)], dtype=torch.int32).cuda(), torch.zeros(1, dtype=torch.int32).cuda()
    run = lambda: ops.wkv_scan(t["r"], t["k"], t["v"], t["d"], w0, u, h, torch.zeros(1, ops.wkv_state_floats(H, d, d) + 8).cuda(), slots, H, d, d,
                               tiles=tiles, pieces=pieces)
    clean = run()
    t[what][bad, 5] = float("inf")
    got = run()
    assert torch.equal(got[:bad], clean[:bad]) if what != "v" else torch.allclose(got[:bad], clean[:bad], rtol=1e-5, atol=1e-4)
    if what == "v":                                       # one column, from the token on
        assert torch.equal(torch.cat([got[:, :5], got[:, 6:]], 1)[:64], torch.cat([clean[:, :5], clean[:, 6:]], 1)[:64])
        assert not bool(torch.isfinite(got[bad:, 5]).any()) and bool(torch.isfinite(got[:, :5]).all())
    else:
        assert not bool(torch.isfinite(got[bad]).any())


# the norm and gate behind the recurrence: heads of 1 to 64 lanes, a last workgroup that is not full, gates further apart than they are
# long, and what the form of eight numbers a lane does not take (an odd gate, other head sizes, few numbers)
@pytest.mark.parametrize("T,H,dv,skip,pad", [(4097, 8, 8, 8, 8), (1025, 16, 16, 0, 0), (347, 24, 32, 8, 0), (131, 32, 64, 16, 8), (129, 17, 128, 0, 8),
                                             (70, 15, 256, 8, 0), (37, 14, 512, 8, 8), (131, 32, 64, 3, 5), (300, 10, 96, 0, 0), (127, 32, 64, 0, 0)])
def test_norm_and_gate_of_a_prompt(T, H, dv, skip, pad):
    from bitnet_c_amd import ops
    g = torch.Generator(device="cuda").manual_seed(T + dv)
    o = torch.randn(T, H * dv, generator=g, device="cuda") * torch.logspace(-6, 6, T, device="cuda")[:, None]
    gate = torch.randn(T, skip + H * dv + pad, generator=g, device="cuda").to(torch.bfloat16)[:, skip:skip + H * dv]
    weight = torch.rand(H * dv, generator=g, device="cuda") + 0.5
    o[T // 2, :dv] = 0                                   # a head of zeros; a head with NaN keeps it to itself
    o[T - 1, -1] = float("nan")
    d = o.double().view(T, H, dv)
    for w in (weight, None):
        want = (d / torch.sqrt((d * d).mean(2, keepdim=True) + 1e-6)).view(T, H * dv) * torch.nn.functional.silu(gate.double())
        want = want if w is None else want * w.double()
        got = ops.head_norm_gate(o, gate, w, H, dv, 1e-6)
        assert torch.equal(got.isnan(), want.isnan()) and int(got.isnan().sum()) == dv
        got, want = got.nan_to_num(0.0).double(), want.nan_to_num(0.0)
        assert float((got - want).norm() / want.norm()) < 2.0 ** -8          # one rounding to bf16
        assert bool(((got - want).abs() <= want.abs() * (2.0 ** -8 + 1e-5)).all())
