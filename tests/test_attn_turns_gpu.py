"""Prompt attention over heads of 128 whose two groups of waves take turns: keys split between the groups, a tile a group (quads, lone pairs, pairs of two
sequences, lone tiles, lists that end in empty tiles or come in any order), and the workgroups of one group, each where the launch chooses it."""
import random

import pytest
import torch

from test_kernels_gpu import _attn_case, mfma_close

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
