"""Products of few rows that form their rows from the residual stream, and products and means that add themselves to it,
against the kernels of their own: the same bits."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu


def _ops():
    from bitnet_c_amd import ops
    return ops


def _same(a, b):
    return torch.equal(a.float().nan_to_num(7.0), b.float().nan_to_num(7.0))


def _rows(M, K, seed):
    g = torch.Generator().manual_seed(seed)
    x = (torch.randn(M, K, generator=g) * torch.logspace(-1, 1, K)).cuda()
    d = torch.randn(M, K, generator=g).bfloat16().cuda()
    w = torch.linspace(0.5, 1.5, K).cuda()
    if M > 3:
        x[1, K // 2], d[1, 3], x[2, 0], d[3, 1] = float("inf"), float("inf"), float("nan"), float("nan")
    return x, d, w, g


# rows: the edges of 2, 4 and 8; K: fewer chunks than waves, threads without a number, a chunk a wave; columns: one, no multiple
# of the tile's rows, tiles of fewer rows
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("N,K,R", [(1, 512, 16), (33, 768, 8), (40, 1024, 12), (30, 1792, 16), (48, 2048, 16)])
def test_products_form_their_rows(M, N, K, R):
    ops = _ops()
    x, d, nw, g = _rows(M, K, M + N + K)
    w = torch.randn(N, K, generator=g).bfloat16().cuda()
    sw = ops.stream_copy(w, R)
    h = ops.add_rmsnorm(x.clone(), None, nw, 1e-5, torch.bfloat16)
    for act in (None, "relu2", "gelu_erf"):
        pre = ops.stream_norm(x, nw, 1e-5, torch.bfloat16)
        assert ops.takes_stream_norm(pre, w, sw) and not ops.takes_stream_norm(pre, w, None)
        want = ops.linear(h, w, streamed=sw) if act is None else ops.linear_unary(h, w, act, sw)
        assert _same(ops.linear_stream_norm(pre, w, sw, activation=act), want), act
    if not ops.can_norm_rows(M, K, torch.bfloat16, ops.ROWS_SUM):
        assert M > 4
        return
    new = x.clone()
    h = ops.add_normed_rmsnorm(new, d, nw, 1e-6, out_dtype=torch.bfloat16, rows_out=True)
    for act in (None, "relu2", "gelu_erf"):
        old = x.clone()
        owner = types.SimpleNamespace(x=old)
        got = ops.linear_stream_norm(ops.stream_sum(owner, d, nw, 1e-6), w, sw, activation=act)
        want = ops.linear(h, w, streamed=sw) if act is None else ops.linear_unary(h, w, act, sw)
        assert _same(got, want) and _same(owner.x, new) and _same(old, x) and owner.x is not old, act
    owner = types.SimpleNamespace(x=x.clone())
    assert _same(ops.stream_sum(owner, d, nw, 1e-6).materialize(), h) and _same(owner.x, new)


# several products of the same rows, as they are or mixed with the rows before them (a token without one, a row that is nobody's)
@pytest.mark.parametrize("M", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("K", [512, 768, 2048])
def test_groups_form_their_rows(M, K):
    ops = _ops()
    x, _, nw, g = _rows(M, K, M + K)
    items = []
    for N, R, act in ((33, 16, None), (40, 8, "tanh"), (1, 12, None)):
        w = torch.randn(N, K, generator=g).bfloat16().cuda()
        items.append((w, ops.stream_copy(w, R), act))
    h = ops.add_rmsnorm(x.clone(), None, nw, 1e-5, torch.bfloat16)
    pre = ops.stream_norm(x, nw, 1e-5, torch.bfloat16)
    for got, want in zip(ops.linear_group_stream_norm(pre, items), ops.linear_group([(h, *i) for i in items])):
        assert _same(got, want)
    if not ops.can_norm_rows(M, K, torch.bfloat16, ops.ROWS_SHIFT):
        assert M > 4
        return
    mu = torch.rand(len(items), K, generator=g).cuda()
    state = torch.randn(M + 2, K + 12, generator=g).cuda()[:, 8:]
    slots = torch.arange(M + 1, 1, -1, dtype=torch.int32).cuda()
    positions = torch.tensor([(5, 0, -1)[m % 3] for m in range(M)], dtype=torch.int32).cuda()
    mixes = ops.token_shift(h, mu, state, positions, torch.arange(M, dtype=torch.int32).cuda(), slots)
    got = ops.linear_group_stream_norm(pre, items, (mu, state, positions, slots))
    assert _same(got[-1], h)
    for a, b in zip(got, ops.linear_group([(m, *i) for m, i in zip(mixes, items)])):
        assert _same(a, b)


@pytest.mark.parametrize("M", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("N,K,R", [(33, 1024, 8), (24, 1792, 16), (40, 2048, 12), (16, 768, 16)])
def test_products_norm_and_gate_their_rows(M, N, K, R):
    ops = _ops()
    o, _, nw, g = _rows(M, K, M + N + K)
    wide = torch.randn(M, K + 16, generator=g).bfloat16().cuda()
    w = torch.randn(N, K, generator=g).bfloat16().cuda()
    for gate in (wide[:, :K], wide[:, 8:K + 8], wide[:, 1:K + 1]):
        for act in ("sigmoid", "silu"):
            want = ops.linear(ops.row_norm_gate(o, gate, nw, 1e-6, act), w)
            assert _same(ops.linear_row_norm_gate(o, gate, nw, 1e-6, act, w, ops.stream_copy(w, R)), want), act


def test_other_sizes_keep_their_kernels():
    ops = _ops()
    for M, K in ((9, 2048), (1, 256), (1, 2304), (1, 2000), (0, 2048)):
        assert not ops.can_norm_rows(M, K, torch.bfloat16)


@pytest.mark.parametrize("M", [1, 2, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("N,K,R", [(1, 256, 16), (33, 2048, 8), (24, 2560, 12), (32, 8192, 16)])
def test_products_add_themselves_rounded(M, N, K, R):
    ops = _ops()
    g = torch.Generator().manual_seed(M + N + K)
    x, w = torch.randn(M, K, generator=g).bfloat16().cuda(), torch.randn(N, K, generator=g).bfloat16().cuda()
    stream = torch.randn(M, N, generator=g).cuda()
    want = stream + ops.linear(x, w, streamed=ops.stream_copy(w, R)).float()
    assert ops.linear_add(x, w, ops.stream_copy(w, R), stream) and torch.equal(stream, want)
    assert not ops.linear_add(x, w, None, stream) and torch.equal(stream, want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,D", [(1, 512), (3, 2048), (2, 2056), (5, 8192)])
def test_mean_of_two_norms_into_the_stream(T, D, dtype):
    ops = _ops()
    g = torch.Generator().manual_seed(T + D)
    a, b = (torch.randn(T, D, generator=g).to(dtype).cuda() for _ in range(2))
    wa, wb = torch.rand(D, generator=g).cuda(), torch.rand(D, generator=g).cuda()
    stream = torch.randn(T, D, generator=g).cuda()
    for second in ((b, wb), (None, None)):
        want = stream + ops.rmsnorm_mean(a, wa, *second, 1e-6).float()
        assert torch.equal(ops.rmsnorm_mean(a, wa, *second, 1e-6, into=stream.clone()), want)
    with pytest.raises(ops.KernelError):
        ops.rmsnorm_mean(a[:, :8].contiguous(), wa[:8].contiguous(), None, None, 1e-6, into=stream[:, :8].contiguous())
