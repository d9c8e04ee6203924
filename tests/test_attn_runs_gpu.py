"""The runs that a decode step's keys are cut in for the general kernel: single pages while the launch leaves few rows of partial sums,
two pages else, where the plan is made and where the kernel follows the longest sequence in device memory alike."""
import pytest
import torch


def _ops():
    from bitnet_c_amd import ops
    return ops


@pytest.mark.parametrize("n_seqs,H,Hkv", [(1, 16, 4), (4, 16, 4), (16, 16, 4), (4, 64, 1), (64, 16, 16), (64, 64, 1)])
@pytest.mark.parametrize("pages", [1, 2, 3, 7, 23, 24, 64, 65, 500])
@pytest.mark.parametrize("window", [0, 100, 5000])
def test_plan(n_seqs, H, Hkv, pages, window):
    ops = _ops()
    n, chunk, follows = ops.general_decode_plan(n_seqs, H, Hkv, pages * ops.PAGE, window)
    most = window + ops.PAGE if window else pages * ops.PAGE
    assert follows == (not window) and 1 <= n <= 64 and chunk % ops.PAGE == 0 and n * chunk >= most
    one = ops.decode_splits(n_seqs, H, Hkv, most, torch.bfloat16, target_wgs=ops.VECTOR_DECODE_TARGET_WGS, min_pages=1)
    two = ops.decode_splits(n_seqs, H, Hkv, most, torch.bfloat16, target_wgs=ops.VECTOR_DECODE_TARGET_WGS)
    assert (n, chunk) == (one if n_seqs * H * one[0] <= ops.GENERAL_PAGE_RUN_ROWS else two)


@pytest.mark.gpu
@pytest.mark.parametrize("n_seqs,H,Hkv,n,pages", [(4, 16, 4, 24, 1), (1, 16, 2, 40, 1), (5, 75, 1, 16, 1), (8, 64, 1, 16, 2), (6, 64, 2, 16, 2)])
def test_runs_that_follow_the_longest_sequence(n_seqs, H, Hkv, n, pages):
    """4 x 16 x 24 and 5 x 75 x 16 rows (6,000, the most): runs of a page; 6 x 64 x 16 (6,144): of two.  The bits of runs of that length."""
    ops, hs = _ops(), 64
    assert (n_seqs * H * n <= ops.GENERAL_PAGE_RUN_ROWS) == (pages == 1)
    g = torch.Generator().manual_seed(n_seqs + H)
    q = torch.randn((n_seqs, H * hs), generator=g).bfloat16().cuda()
    k, v = (torch.randn(s, generator=g).bfloat16().cuda() for s in ((n_seqs * n, Hkv, 64, hs), (n_seqs * n, Hkv, hs, 64)))
    table = torch.arange(n_seqs * n, dtype=torch.int32).reshape(n_seqs, n).cuda()
    lens = torch.tensor([(64 * n, 130, 64, 1, 0, 65, 200, 129)[(i + 1) % 8] for i in range(n_seqs)], dtype=torch.int32).cuda()
    longest = torch.tensor([int(lens.max())], dtype=torch.int32).cuda()
    follows, fixed = (torch.empty((n_seqs, H * hs), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    args = (k, v, table, lens, H, Hkv, hs, hs, hs ** -0.5)
    ops.attention_general_decode(q, follows, *args, n_splits=n, max_len_dev=longest)
    ops.attention_general_decode(q, fixed, *args, n_splits=n, chunk=64 * pages)
    assert torch.equal(follows, fixed)


@pytest.mark.parametrize("n_seqs,H,Hkv,hs,tokens,window,whole", [
    (64, 16, 4, 128, 100, 0, True), (63, 16, 4, 128, 100, 0, False), (32, 32, 8, 128, 130, 0, True), (31, 32, 8, 128, 130, 0, False), (32, 32, 8, 128, 200, 0, False),
    (1, 32, 4, 64, 128, 0, True), (1, 32, 4, 64, 129, 0, False), (1, 32, 4, 96, 128, 0, False), (16, 64, 1, 128, 128, 0, True), (15, 64, 1, 128, 128, 0, False),
    (16, 64, 1, 128, 129, 0, False), (64, 16, 2, 256, 128, 0, False), (128, 16, 2, 256, 128, 0, True), (64, 16, 4, 128, 5000, 64, True), (64, 16, 4, 128, 5000, 65, True),
    (64, 16, 4, 128, 5000, 129, False), (1, 16, 4, 128, 64, 0, True)])
def test_short_sequences_stay_whole(n_seqs, H, Hkv, hs, tokens, window, whole):
    """No merge where longer runs are one: in 256 workgroups and more, and for two pages with heads of 64 or 2,048 rows of partial sums; else the plan."""
    ops = _ops()
    plan = ops.general_decode_plan(n_seqs, H, Hkv, tokens, window)
    got = ops.general_decode_runs(n_seqs, H, Hkv, hs, tokens, window)
    assert (got[0] == 1) == whole and got[2] == plan[2]
    if not whole:
        assert got == plan and plan[0] > 1
