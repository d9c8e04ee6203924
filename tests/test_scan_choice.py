"""Which prompt steps cut their recurrences into pieces: a choice that the eager step of a request and the captured step that
replays it make alike; and the lengths of a captured step's lists of tiles."""
import random

import torch


def _context(n_new, captured=None):
    from bitnet_c_amd.engine.step import StepContext
    rows, seqs = captured or (sum(n_new), len(n_new))
    i32 = torch.zeros(rows, dtype=torch.int32)
    return StepContext(torch.device("cpu"), torch.bfloat16, i32, i32, i32, i32[:0], i32[:0], i32[:0], False, [-1] * seqs,
                       [0] * seqs if captured else n_new, [0] * seqs, captured=captured is not None)


def test_eager_and_captured_steps_have_the_same_sizes():
    from bitnet_c_amd.engine.step import Engine, StepEntry
    rng = random.Random(5)
    shapes = [[n] for n in (2, 16, 17, 193, 200, 255, 256, 257, 513, 2049, 8192)] + [[700] * 3, [256] * 2, [8] * 32, [40] * 200]
    shapes += [[rng.randint(1, 400) for _ in range(rng.randint(1, 20))] for _ in range(50)]
    for n_new in shapes:
        key = Engine._prompt_key([StepEntry(0, [0] * n, [0]) for n in n_new], n_new)
        assert _context(n_new).sizes == _context(n_new, captured=key[:2]).sizes == key[:2]
    assert _context([3] * 300).sizes[1] == 300                   # more sequences than any captured step holds


def test_which_steps_are_cut():
    from bitnet_c_amd import ops
    bf16 = torch.bfloat16
    wkv = lambda sizes, H, d=64, dtype=bf16: ops.wkv_in_pieces(dtype, sizes, H, d, d)
    gru = lambda sizes, W, dtype=bf16: ops.mingru_in_pieces(dtype, sizes, W)
    assert wkv((256, 1), 32) and wkv((2048, 1), 32) and wkv((2048, 2), 32) and wkv((2048, 4), 16) and wkv((8192, 32), 1)
    assert not wkv((2048, 4), 32) and not wkv((512, 2), 32) and not wkv((192, 1), 32) and not wkv((512, 1), 32, 128)
    assert not wkv((256, 32), 2) and not wkv((1024, 64), 1)       # many short sequences: a piece each
    assert gru((256, 1), 2048) and gru((1024, 4), 2048) and gru((4096, 8), 2048) and not gru((2048, 8), 2048) and not gru((192, 1), 64)
    assert not wkv((2048, 1), 32, dtype=torch.float32) and not gru((2048, 1), 2048, torch.float32)
    assert not wkv((1 << 24, 1), 32)                              # scratch beyond its bound


def test_a_captured_step_has_room_for_every_list_of_tiles():
    from bitnet_c_amd import ops
    from bitnet_c_amd.engine.step import _bucket, _most_tiles, _query_tiles, _row_bucket
    rng = random.Random(6)
    shapes = [[n] for n in (1, 2, 15, 16, 17, 63, 64, 65, 256, 8192)] + [[1] * 256, [1] * 12 + [4], [17] * 15 + [1], [65, 1, 63], [64] * 8]
    shapes += [[rng.randint(1, 300) for _ in range(rng.randint(1, 20))] for _ in range(200)]
    for n_new in shapes:
        rows, seqs = _row_bucket(sum(n_new)), _bucket(len(n_new))
        for qt in (1, 4, 16, 32, 48, 64, 128, ops.SEQUENCE_TILE):
            assert len(_query_tiles(n_new, [5] * len(n_new), qt)) <= _most_tiles(rows, seqs, qt)
        assert _most_tiles(rows, seqs, ops.SEQUENCE_TILE) == seqs            # no tile that no sequence can have
