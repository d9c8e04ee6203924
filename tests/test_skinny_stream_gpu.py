"""The products of up to 16 rows over streamed copies whose K is whole chunks of 256: the same bits as the kernels over the
row-major matrix, which sum in the same order."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ops():
    from bitnet_c_amd import ops
    return ops


def _data(M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
    w = (torch.randn(N, K, generator=g) * 0.05).to(torch.bfloat16).cuda()
    return x, w


# rows: the edges of 2, 4, 8 and 16, by which the activations' loads go; K: one chunk, seven (a wave without any), a chunk a
# wave, nine (one wave has two), two a wave, 17 to 25 (two, three and four a wave, even and odd counts in turn), seven a wave;
# columns: one, no multiple of the tile's rows
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("N,K,R", [(1, 256, 16), (40, 1792, 12), (33, 2048, 8), (72, 2304, 16), (30, 4096, 10), (17, 4352, 16),
                                   (24, 6144, 7), (16, 6400, 16), (18, 14336, 16)])
def test_whole_chunks_give_the_bits_of_the_row_major_kernels(M, N, K, R):
    ops = _ops()
    x, w = _data(M, N, K, 100 * M + N)
    sw = ops.stream_copy(w, R)
    for dtype in (torch.bfloat16, torch.float32):
        assert torch.equal(ops.linear(x, w, dtype), ops.linear(x, w, dtype, streamed=sw)), dtype
    for act in ("relu2", "tanh"):
        assert torch.equal(ops.linear_unary(x, w, act), ops.linear_unary(x, w, act, sw)), act
    # rows that lie further apart than they are long, and what lies between them
    wide = torch.full((M, K + 64), float("nan"), dtype=torch.bfloat16, device="cuda")
    wide[:, :K] = x
    assert torch.equal(ops.linear(wide[:, :K], w), ops.linear(wide[:, :K], w, streamed=sw))
    # into the stream, and the product and the gated unit behind the norm that this leaves
    weight = torch.linspace(0.5, 1.5, N, device="cuda")
    streams = [torch.linspace(-1, 1, M * N, device="cuda").view(M, N).contiguous() for _ in range(2)]
    a, b = (ops.linear_into_stream(x, w, s, weight, 1e-5, c) for s, c in zip(streams, (None, sw)))
    assert torch.equal(*streams) and torch.equal(a.scaled, b.scaled)
    assert torch.allclose(a.slots.sum(1), b.slots.sum(1), rtol=1e-5)        # a slot a column tile: R columns or what suits N


@pytest.mark.parametrize("M", [1, 2, 4, 8, 11, 16])
@pytest.mark.parametrize("N,K", [(48, 2048), (16, 4096), (80, 256), (32, 5632), (304, 8192)])
def test_products_behind_a_deferred_norm(M, N, K):
    ops = _ops()
    x, w = _data(M, N, K, M + N)
    small, lift = _data(M, K, 256, M)
    stream = x.float()
    pre = ops.linear_into_stream(small, lift, stream, torch.linspace(0.5, 1.5, K, device="cuda"), 1e-5, ops.stream_copy(lift))
    for R in (16, 12):
        assert torch.equal(ops.linear_prenorm(pre, w), ops.linear_prenorm(pre, w, ops.stream_copy(w, R)))
    for act in ("silu", "relu2"):
        assert torch.equal(ops.linear_swiglu_prenorm(pre, w, act), ops.linear_swiglu_prenorm(pre, w, act, ops.stream_copy(w, 16)))
