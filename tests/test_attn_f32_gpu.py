"""The plain float32 attention on the float32 matrix instruction: prompt and decode forms against 64 bits, and against each
other bit for bit (a page's keys are summed by themselves, pages folded into runs, runs folded in order)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
PAGE = 64


def _setup(H, Hkv, hs, lens, seed=0):
    """Pages of a shared pool in a shuffled order, NaN where nothing was written."""
    g = torch.Generator().manual_seed(seed)
    pages = [-(-n // PAGE) for n in lens]
    order = torch.randperm(sum(pages) + 2, generator=g)
    kp = torch.full((sum(pages) + 2, Hkv, PAGE, hs), float("nan"))
    vp = kp.clone()
    bt = torch.full((len(lens), max(pages) + 1), int(order[-1]), dtype=torch.int32)
    keys, values, at = [], [], 0
    for b, n in enumerate(lens):
        k, v = torch.randn(n, Hkv, hs, generator=g), torch.randn(n, Hkv, hs, generator=g)
        for p in range(pages[b]):
            m = min(PAGE, n - p * PAGE)
            bt[b, p] = order[at]
            kp[order[at], :, :m] = k[p * PAGE:p * PAGE + m].transpose(0, 1)
            vp[order[at], :, :m] = v[p * PAGE:p * PAGE + m].transpose(0, 1)
            at += 1
        keys.append(k)
        values.append(v)
    q = [torch.randn(n, H * hs, generator=g) for n in lens]
    return kp.cuda(), vp.cuda(), bt.cuda(), keys, values, q


def _exact(q, k, v, H, Hkv, hs, scale, first):
    """Rows first .. of one sequence in 64 bits."""
    n = k.shape[0]
    q = q[first:].double().view(-1, H, hs).transpose(0, 1)
    k, v = (t.double().transpose(0, 1).repeat_interleave(H // Hkv, dim=0) for t in (k, v))
    s = q @ k.transpose(1, 2).contiguous() * scale
    s = s.masked_fill(torch.arange(n)[None, :] > torch.arange(first, n)[:, None], float("-inf"))
    return (torch.softmax(s, dim=-1) @ v).transpose(0, 1).reshape(n - first, H * hs)


# lengths: one key, the edges of a page and of a run of four pages, several runs; heads: one a group, not a power of two, more
# than a tile of sixteen
@pytest.mark.parametrize("H,Hkv,hs", [(4, 2, 16), (3, 1, 32), (2, 2, 64), (8, 2, 128), (20, 1, 64), (6, 2, 128)])
def test_prompt_and_decode(H, Hkv, hs):
    from bitnet_c_amd import ops
    lens = [1, 63, 64, 65, 255, 256, 257, 700]
    scale = hs ** -0.5
    kp, vp, bt, keys, values, q = _setup(H, Hkv, hs, lens, H * hs)
    # a whole prompt of every sequence, in tiles of both sizes that are taken
    flat = torch.cat(q).cuda()
    outs = []
    for plain in (True, False):
        _, _, qt = ops.attention_row_shape(H, Hkv, False, torch.float32, hs, plain)
        tiles, row = [], 0
        for b, n in enumerate(lens):
            tiles += [(b, row + i, min(qt, n - i), i) for i in range(0, n, qt)]
            row += n
        tiles.append((0, 0, 0, 0))                                       # a tile of no rows
        out = torch.full((sum(lens), H * hs), float("nan")).cuda()
        ops.attention(flat, out, kp, vp, bt, H, Hkv, hs, scale, tiles=torch.tensor(tiles, dtype=torch.int32).cuda(), qt=qt)
        outs.append(out)
    assert torch.equal(outs[0], outs[1])
    exact = [_exact(q[b], keys[b], values[b], H, Hkv, hs, scale, 0) for b in range(len(lens))]
    # a score's chain of hs + 4 links at |q||k| scale, which moves a weight by as much; the values' sums likewise
    worst = 2.0 ** -24 * (hs + 4) * max(float(t.abs().max()) for t in q) * max(float(t.abs().max()) for t in keys) * hs ** 0.5
    tol = (2 * worst + 2.0 ** -24 * 300) * max(float(t.abs().max()) for t in values)
    assert float((outs[0].cpu().double() - torch.cat(exact)).abs().max()) <= tol
    # the last token of every sequence, decoded; one padding row
    last = torch.stack([t[-1] for t in q] + [q[0][0]]).cuda()
    sl = torch.tensor(lens + [0], dtype=torch.int32).cuda()
    table = torch.cat([bt, bt[:1]])
    want = outs[0][torch.tensor(lens).cumsum(0).cuda() - 1]
    n_splits, chunk = ops.decode_splits(len(sl), H, Hkv, table.shape[1] * PAGE, torch.float32)
    got = torch.full((len(sl), H * hs), float("nan")).cuda()
    ops.attention(last, got, kp, vp, table, H, Hkv, hs, scale, seq_lens=sl, n_splits=n_splits, chunk=chunk)
    assert torch.equal(got[:-1], want) and float(got[-1].abs().max()) == 0.0
    # a table of one run (no second kernel), of very many (a workgroup takes several), and the sequences one by one
    got = torch.full((1, H * hs), float("nan")).cuda()
    ops.attention(last[4:5], got, kp, vp, table[4:5, :4].contiguous(), H, Hkv, hs, scale, seq_lens=sl[4:5])
    assert torch.equal(got, want[4:5])
    wide = torch.zeros((1, 20000), dtype=torch.int32).cuda()
    wide[:, :table.shape[1]] = table[7:8]
    got = torch.full((1, H * hs), float("nan")).cuda()
    ops.attention(last[7:8], got, kp, vp, wide, H, Hkv, hs, scale, seq_lens=sl[7:8])
    assert torch.equal(got, want[7:8])


def test_a_key_far_above_the_others_and_rows_before_it():
    """Weights that vanish beside one key: a page folded after a page with a far larger maximum, and the other way round."""
    from bitnet_c_amd import ops
    H, Hkv, hs, n = 2, 1, 64, 600
    kp, vp, bt, keys, values, q = _setup(H, Hkv, hs, [n], 5)
    for at in (10, 400):
        page, row = int(bt[0, at // PAGE]), at % PAGE
        keys[0][at] = q[0][n - 1, :hs] * 40.0
        kp[page, 0, row] = keys[0][at, 0].cuda()
    _, _, qt = ops.attention_row_shape(H, Hkv, False, torch.float32, hs, True)
    tiles = torch.tensor([(0, i, min(qt, n - i), i) for i in range(0, n, qt)], dtype=torch.int32).cuda()
    out = torch.full((n, H * hs), float("nan")).cuda()
    ops.attention(q[0].cuda(), out, kp, vp, bt, H, Hkv, hs, hs ** -0.5, tiles=tiles, qt=qt)
    exact = _exact(q[0], keys[0], values[0], H, Hkv, hs, hs ** -0.5, 0)
    # scores up to 40 |q|^2 / 8: some 400, whose rounding (2^-24 of it, times the chain) moves a weight by some 1e-3
    assert float((out.cpu().double() - exact).abs().max()) <= 400 * 2.0 ** -24 * (hs + 4) * 4


@pytest.mark.parametrize("hs", [16, 128])
def test_keys_that_are_not_numbers(hs):
    """A page of keys (and a run of pages) of nothing but NaN gives NaN to every row that sees it, as one such key among others
    does, and so does a query of NaN: no page is passed over for it."""
    from bitnet_c_amd import ops
    H, Hkv, n = 4, 2, 700
    kp, vp, bt, _, _, q = _setup(H, Hkv, hs, [n], 3)
    q = q[0].cuda()
    q[50, :hs] = float("nan")
    q[699, hs:2 * hs] = float("nan")
    for first, last in ((64, 127), (256, 511), (130, 130)):
        k = kp.clone()
        for p in range(first // PAGE, last // PAGE + 1):
            lo, hi = max(first - p * PAGE, 0), min(last - p * PAGE, PAGE - 1)
            k[int(bt[0, p]), 1, lo:hi + 1] = float("nan")
        want = torch.zeros(n, H, dtype=torch.bool)
        want[50, 0] = want[699, 1] = True
        want[first:, 2:] = True
        for plain in (True, False):
            _, _, qt = ops.attention_row_shape(H, Hkv, False, torch.float32, hs, plain)
            tiles = torch.tensor([(0, i, min(qt, n - i), i) for i in range(0, n, qt)], dtype=torch.int32).cuda()
            out = torch.zeros(n, H * hs).cuda()
            ops.attention(q, out, k, vp, bt, H, Hkv, hs, hs ** -0.5, tiles=tiles, qt=qt)
            assert torch.equal(out.view(n, H, hs).isnan().cpu(), want[:, :, None].expand(n, H, hs))
        rows = [50, 63, 127, 128, 129, 255, 511, 600, 699]
        sl = torch.tensor([r + 1 for r in rows] + [0], dtype=torch.int32).cuda()
        for width in (bt.shape[1], 2 ** 24 // (10 * H * (hs + 2)) + 1):                  # parts of a page, and of a run of pages
            table = torch.zeros((len(sl), width), dtype=torch.int32).cuda()
            table[:, :bt.shape[1]] = bt
            n_splits, chunk = ops.decode_splits(len(sl), H, Hkv, width * PAGE, torch.float32)
            got = torch.zeros(len(sl), H * hs).cuda()
            ops.attention(torch.cat([q[rows], q[50:51]]), got, k, vp, table, H, Hkv, hs, hs ** -0.5, seq_lens=sl, n_splits=n_splits, chunk=chunk)
            assert torch.equal(got[:-1].view(-1, H, hs).isnan().cpu(), want[rows][:, :, None].expand(len(rows), H, hs))
            assert float(got[-1].abs().max()) == 0.0
