"""Prompt attention over heads of 128 whose two groups of waves take turns: keys split between the groups, a tile a group (quads, lone pairs, pairs of two
sequences, lone tiles, lists that end in empty tiles or come in any order), and the workgroups of one group, each where the launch chooses it."""
import random

import pytest
import torch

from test_kernels_gpu import _attn_case, _paged, _rand, mfma_close

pytestmark = pytest.mark.gpu

# heads, kv heads, tokens in front and new ones per sequence, window
CASES = [
    (8, 2, [0], [1], 0), (8, 2, [0, 130], [63, 200], 0), (32, 8, [5, 0, 64], [33, 257, 65], 0), (4, 4, [700], [129], 0), (12, 4, [0], [333], 100),      # split
    (32, 8, [0], [1500], 0), (32, 1, [0], [1400], 0),                                              # split, a pair a workgroup
    (64, 64, [0], [1300], 0), (64, 64, [0, 64, 3, 0], [700, 801, 900, 1000], 0), (64, 64, [0, 0], [1024, 1280], 300),      # a tile a group, two turns
    (40, 40, [0, 10, 0, 0], [300, 200, 129, 250], 0), (40, 40, [0, 0, 0, 64, 0], [128] * 4 + [257], 70),                 # a tile a group, a turn a workgroup
    (64, 64, [0, 9, 0, 0, 0, 0, 0], [300, 450, 200, 129, 380, 260, 511], 0),                          # one group
]


@pytest.mark.parametrize("H,Hkv,before,new,window", CASES)
def test_turns(H, Hkv, before, new, window):
    hs, dtype = 128, torch.bfloat16
    ops, qkv, kp, vp, bt, ref, scale = _attn_case(dtype, H, Hkv, hs, before, new, window, 77)
    _, _, qt = ops.attention_row_shape(H, Hkv, False, dtype, hs)
    tiles, r = [], 0
    for s, (p0, n) in enumerate(zip(before, new)):
        tiles += [(s, r + i, min(qt, n - i), p0 + i) for i in range(0, n, qt)]
        r += n
    paired, shuffled = ops.pair_tiles(tiles), list(tiles)
    random.Random(1).shuffle(shuffled)
    for order in (paired, tiles, shuffled, paired + [(0, 0, 0, 0)] * 5):
        out = torch.full((r, H * hs), float("nan"), dtype=dtype).cuda()
        ops.attention(qkv, out, kp, vp, bt, H, Hkv, hs, scale, window=window, tiles=torch.tensor(order, dtype=torch.int32).cuda(), qt=qt)
        assert mfma_close(out.float(), ref)


# each form where its rule begins: PF_* of the kernel's source, then as above; lists in which a pair's place among its sequence's is found over more than 64 and 128 of them
ONE, ONE_PAIRED, SPLIT, SPLIT_PAIRED, EACH, EACH_PAIRED = range(2, 8)
FORMS = [
    (SPLIT, 8, 2, [0, 130], [63, 200], 0), (SPLIT_PAIRED, 32, 8, [0], [1500], 0), (SPLIT_PAIRED, 32, 8, [0], [1100], 740),
    (ONE, 40, 40, [0, 300, 0, 64, 7, 0, 0, 500], [128, 60, 128, 1, 90, 128, 100, 127], 0), (EACH, 40, 40, [0, 10, 0, 70], [130, 200, 256, 129], 0),
    (EACH, 16, 4, [0] * 18, [100] * 17 + [33], 50), (SPLIT_PAIRED, 16, 4, [0] * 16, [200] * 16, 0), (EACH_PAIRED, 40, 40, [5] * 7, [129] * 7, 0), (ONE_PAIRED, 64, 64, [0] * 9, [70] * 9, 0),
    (ONE_PAIRED, 64, 64, [0, 9, 0, 0, 0, 0, 0], [300, 450, 200, 129, 380, 260, 511], 0), (ONE_PAIRED, 64, 64, [0, 64, 3, 0], [700, 801, 900, 1000], 0),
    (EACH, 32, 8, [3], [1200], 512), (EACH, 16, 1, [0], [2100], 700), (EACH_PAIRED, 64, 64, [0], [1921], 0),
    (EACH_PAIRED, 32, 2, [0, 5], [1040, 1036], 0), (EACH_PAIRED, 48, 3, [40], [1393], 0),
]


@pytest.mark.parametrize("form,H,Hkv,before,new,window", FORMS)
def test_forms(form, H, Hkv, before, new, window):
    from bitnet_c_amd import ops
    hs, dtype = 128, torch.bfloat16
    _, gt, qt = ops.attention_row_shape(H, Hkv, False, dtype, hs)
    tiles, r, q, k, v = [], 0, [], [], []
    for s, (p0, n) in enumerate(zip(before, new)):
        tiles += [(s, r + i, min(qt, n - i), p0 + i) for i in range(0, n, qt)]
        r += n
        q.append(_rand((n, H, hs), dtype, 3 * s))
        k.append(_rand((p0 + n, Hkv, hs), dtype, 3 * s + 1))
        v.append(_rand((p0 + n, Hkv, hs), dtype, 3 * s + 2))
    assert ops._fn("attn_mfma", "bn_attn_mfma_prompt_form")(len(tiles), r, len(new), H, Hkv, hs, gt, window) == form
    kp, vp, bt = _paged(k, v, dtype, sum(-(-t.shape[0] // 64) for t in k) + 3, 5)
    refs = []
    for p0, n, qs, ks, vs in zip(before, new, q, k, v):
        at, key = torch.arange(p0, p0 + n).cuda()[:, None], torch.arange(p0 + n).cuda()[None]
        hide = (key > at) | ((key <= at - window) if window else torch.zeros_like(key > at))
        qs, ks, vs = (t.cuda().double() for t in (qs, ks, vs))
        heads = [((qs[:, h] @ ks[:, h * Hkv // H].t()) * hs ** -0.5).masked_fill(hide, float("-inf")).softmax(1) @ vs[:, h * Hkv // H] for h in range(H)]
        refs.append(torch.stack(heads, 1).reshape(n, H * hs))
    qkv = torch.cat([torch.cat(q).reshape(r, H * hs), torch.full((r, 2 * Hkv * hs), float("nan"), dtype=dtype)], 1).cuda()
    kp, vp, bt, ref = kp.cuda(), vp.cuda(), bt.cuda(), torch.cat(refs)
    pairs, shuffled = ops.pair_tiles(tiles), list(tiles)
    random.Random(1).shuffle(shuffled)
    for order in (pairs, shuffled, pairs + [(0, 0, 0, 0)] * 3):
        out = torch.full((r, H * hs), float("nan"), dtype=dtype).cuda()
        ops.attention(qkv, out, kp, vp, bt, H, Hkv, hs, hs ** -0.5, window=window, tiles=torch.tensor(order, dtype=torch.int32).cuda(), qt=qt)
        assert mfma_close(out.float(), ref)


def test_no_window_is_a_wide_one():
    """A window that no walk reaches takes the form that none takes."""
    from bitnet_c_amd import ops
    take = ops._fn("attn_mfma", "bn_attn_mfma_prompt_form")
    for H, Hkv, gt, qt in ((32, 8, 4, 32), (16, 4, 4, 32), (64, 8, 8, 16), (40, 40, 1, 128)):
        for n_seqs, n in ((1, 1200), (1, 2048), (1, 4096), (2, 640), (4, 1000), (8, 1024), (16, 300), (32, 64)):
            args = (n_seqs * -(-n // qt), n_seqs * n, n_seqs, H, Hkv, 128, gt)
            assert take(*args, 0) == take(*args, n) == take(*args, 100000)
    assert take(1, 1, 1, 4, 4, 96, 1, 0) == take(0, 1, 1, 4, 4, 128, 1, 0) == take(1, 1, 0, 4, 4, 128, 1, 0) == -1
