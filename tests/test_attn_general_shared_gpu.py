"""The prompt form of the general matrix-core attention stages a block of keys and values once for the heads of a
workgroup (four, two or one of a kv head).  How many share it must not show: heads that share a kv head give the same
bits as the same heads with a copy of that kv head each, and both lie beside a float32 softmax."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _pages(x, table, page, transposed):
    """[T, G, d] into pages of `page` positions named by `table`; what lies behind the last position is NaN."""
    T, G, d = x.shape
    out = torch.full((len(table), G, page, d), float("nan"), dtype=torch.bfloat16)
    for p, t in enumerate(table):
        part = x[p * page:(p + 1) * page]
        out[t, :, :part.shape[0]] = part.transpose(0, 1)
    return (out.transpose(2, 3) if transposed else out).contiguous().to(DEV)


def _expected(q, k, v, lo, scale, window, keep):
    H, G = q.shape[1], k.shape[1]
    k, v = (t.float().repeat_interleave(H // G, 1) for t in (k, v))
    s = torch.einsum("qhd,khd->hqk", q.float(), k) * scale
    i, j = torch.arange(lo, lo + q.shape[0])[:, None], torch.arange(k.shape[0])[None]
    seen = (j <= i) & (((i - j) < window) | (j < keep) if window else True)
    return torch.einsum("hqk,khd->qhd", torch.softmax(s.masked_fill(~seen, -math.inf), -1), v)


@pytest.mark.parametrize("hs,vd", [(32, 32), (64, 128), (96, 64), (128, 128), (160, 64), (192, 192), (256, 96), (256, 256)])
@pytest.mark.parametrize("T,lo,window,keep", [(1, 0, 0, 0), (150, 33, 0, 0), (200, 96, 45, 3), (128, 127, 0, 0)])
def test_heads_that_share_a_block_and_heads_on_their_own_give_the_same_bits(hs, vd, T, lo, window, keep):
    from bitnet_c_amd import ops
    from bitnet_c_amd.cache import PAGE
    torch.manual_seed(hs + vd + T)
    G, group, n, qt = 2, 4, T - lo, ops.GENERAL_PROMPT_TILE
    scale = 1.0 / math.sqrt(hs)
    q, k, v = (torch.randn(s).to(torch.bfloat16) for s in ((n, G * group, hs), (T, G, hs), (T, G, vd)))
    n_pages = -(-T // PAGE)
    table = list(range(n_pages))[::-1]
    tiles = [[0, i, min(qt, n - i), lo + i] for i in range(0, n, qt)] + [[0, 0, 0, 0]]
    tiles = torch.tensor(tiles[::-1], dtype=torch.int32, device=DEV)
    outs = []
    for copies in (1, 2, 4):                             # four, two and one head of a kv head
        kk, vv = k.repeat_interleave(copies, 1), v.repeat_interleave(copies, 1)
        out = torch.full((n, G * group * vd), 7.0, dtype=torch.bfloat16, device=DEV)
        ops.attention_general_prompt(q.reshape(n, -1).to(DEV), out, _pages(kk, table, PAGE, False), _pages(vv, table, PAGE, True),
                                     torch.tensor([table], dtype=torch.int32, device=DEV), G * group, G * copies, hs, vd, scale,
                                     tiles, window=window, keep_first=keep)
        outs.append(out.cpu())
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    want = _expected(q, k, v, lo, scale, window, keep)
    # the weights are rounded to bf16 in numerator and denominator (at most 2^-8 of |v| in all, |v| < 5) and the result once more
    # (2^-9 of itself)
    assert float((outs[0].float().reshape(want.shape) - want).abs().max()) <= 5 * 2.0 ** -8 + 5 * 2.0 ** -9


def test_more_tiles_than_a_launch_has_room_for():
    """A list of over 65,535 tiles, most of no rows (as a list may end in them), with rows in front of and behind that place."""
    from bitnet_c_amd import ops
    from bitnet_c_amd.cache import PAGE
    torch.manual_seed(2)
    H, G, hs, n, qt = 2, 1, 32, 70, ops.GENERAL_PROMPT_TILE
    q, k, v = (torch.randn(n, h, hs).to(torch.bfloat16) for h in (H, G, G))
    table = list(range(-(-n // PAGE)))
    tiles = torch.tensor([[0, i, min(qt, n - i), i] for i in range(0, n, qt)], dtype=torch.int32)
    outs = []
    for places in (range(len(tiles)), [0, 65534, 65535, 65536, 70000]):
        many = torch.zeros(max(places) + 1, 4, dtype=torch.int32)
        many[list(places)] = tiles
        out = torch.full((n, H * hs), 7.0, dtype=torch.bfloat16, device=DEV)
        ops.attention_general_prompt(q.reshape(n, -1).to(DEV), out, _pages(k, table, PAGE, False), _pages(v, table, PAGE, True),
                                     torch.tensor([table], dtype=torch.int32, device=DEV), H, G, hs, hs, 0.2, many.to(DEV))
        outs.append(out)
    assert torch.equal(*outs) and float((outs[0].float().cpu().view(n, H, hs) - _expected(q, k, v, 0, 0.2, 0, 0)).abs().max()) < 0.05
