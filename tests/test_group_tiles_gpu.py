"""The rows per tile of matrices that one launch streams together: sixteen where that leaves two rows of tiles for every CU; the products'
bits do not depend on it."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("widths,rows", [([2048] * 4 + [64], [16] * 4 + [None]), ([2048] * 4, [16] * 4), ([2032] + [2048] * 3, [None] * 4),
                                         ([1024] * 4 + [32], [None] * 5), ([8192, 255, 256], [16, None, 16])])
@pytest.mark.parametrize("M", [1, 2, 4, 5, 16])
def test_rows_per_tile_of_a_group(widths, rows, M):
    from bitnet_c_amd import ops
    if ops._compute_units() == 256:
        assert ops.group_tile_rows(widths) == rows
    g = torch.Generator().manual_seed(M + len(widths))
    x = torch.randn((M, 512), generator=g).bfloat16().cuda()
    ws = [(torch.randn((n, 512), generator=g) * 0.05).bfloat16().cuda() for n in widths]
    got = ops.linear_group([(x, w, ops.stream_copy(w, r), None) for w, r in zip(ws, ops.group_tile_rows(widths))])
    own = ops.linear_group([(x, w, ops.stream_copy(w), None) for w in ws])
    assert all(torch.equal(a, b) for a, b in zip(got, own))
