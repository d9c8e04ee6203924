"""Products that share a launch, activations in a product's own kernel, the decode step of wkv with its norm and gate, and the
mean of two normed branches in 16-byte groups: each against the kernels that do the same one by one."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rand(shape, seed, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(shape, generator=g).to(dtype).cuda()


# columns: less than a tile, not a multiple of one, several tile heights; K: under, at and over a wave's chunk of 256, more
# chunks than waves
@pytest.mark.parametrize("M", [1, 5, 16, 17])
@pytest.mark.parametrize("K,Ns,rows", [(64, [16, 8, 33], [16, 8, 12]), (256, [2048, 64], [8, 16]), (264, [100] * 6, [10] * 6),
                                       (2304, [48, 5, 640, 16], [16, 5, 12, 3])])
def test_group_is_the_products_one_by_one(M, K, Ns, rows):
    from bitnet_c_amd import ops
    acts = ["tanh", None, "gelu_erf", None, "silu", "sigmoid"]
    items, want = [], []
    for j, (N, R) in enumerate(zip(Ns, rows)):
        x, w = _rand((M, K), j, torch.bfloat16), _rand((N, K), 50 + j, torch.bfloat16)
        sw = ops.stream_copy(w, R)
        items.append((x, w, sw, acts[j]))
        want.append(ops.linear(x, w, streamed=sw) if acts[j] is None else ops.linear_unary(x, w, acts[j], sw))
    got = ops.linear_group(items)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    items[0] = items[0][:2] + (None,) + items[0][3:]                  # a matrix without a streamed copy: one by one
    assert all(torch.equal(a, b) for a, b in zip(ops.linear_group(items), want))


@pytest.mark.parametrize("activation", ["gelu_erf", "gelu_tanh", "silu", "relu2", "tanh", "sigmoid"])
@pytest.mark.parametrize("M", [1, 16, 17])
def test_activation_in_the_product(activation, M):
    from bitnet_c_amd import ops
    x, w = _rand((M, 320), 1, torch.bfloat16), _rand((72, 320), 2, torch.bfloat16) / 16
    z = (x.double() @ w.double().t()).float()
    want = ops.unary_act(z.clone(), activation).double()
    for sw in (None, ops.stream_copy(w)):
        y = ops.linear_unary(x, w, activation, sw).double()
        # one rounding of the result (2^-9) up to 16 rows, and one of the product before the activation beyond (every activation
        # here moves by at most 2 |z| of what its argument moves by)
        tol = 2.0 ** -8 * want.abs() + 2.0 ** -16 * 320 ** 0.5 + (2.0 ** -8 * 2 * (1 + z.abs()).double() ** 2 if M > 16 else 0.0)
        assert torch.all((y - want).abs() <= tol)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,d", [(2, 64), (3, 24), (1, 128), (5, 8)])
@pytest.mark.parametrize("weighted", [True, False])
def test_wkv_step(dtype, H, d, weighted):
    """Sequences at position 0 and later, a padding row; state, last row and outputs as the scan and the norm leave them."""
    from bitnet_c_amd import ops
    if not ops.wkv_step_supported(d, d):
        pytest.skip("a head of this size does not fit the kernel")
    B, A, D = 4, H * d, 40
    r, k, v, dd, g = (_rand((B, A), 10 + i, dtype) for i in range(5))
    h, w0, u = _rand((B, D), 20, dtype), _rand((A,), 21) - 2.0, _rand((A,), 22)
    weight = _rand((A,), 23) if weighted else None
    n = ops.wkv_state_floats(H, d, d)
    state = torch.zeros(6, n + D).cuda()
    lens, slots = torch.tensor([1, 9, 0, 3], dtype=torch.int32).cuda(), torch.tensor([4, 0, 5, 2], dtype=torch.int32).cuda()
    for i in range(3):                                    # a state that the kernels themselves have made
        ops.wkv_scan(r * (i + 1), k, v, dd, w0, u, h, state, slots, H, d, d, seq_lens=torch.tensor([5, 5, 0, 5], dtype=torch.int32).cuda())
    a, b = state.clone(), state.clone()
    o = ops.wkv_scan(r, k, v, dd, w0, u, h, a, slots, H, d, d, seq_lens=lens)
    want = ops.head_norm_gate(o, g, weight, H, d, 1e-6)
    got = ops.wkv_step(r, k, v, dd, w0, u, h, b, slots, H, d, d, lens, g, weight, 1e-6)
    assert torch.equal(a, b)
    live = [0, 1, 3]
    # (the bits are equal: test_wkv_step_gives_the_bits_of_the_scan_and_the_norm)
    tol = 2.0 ** -7 if dtype == torch.bfloat16 else 1e-6
    assert torch.all((got[live] - want[live]).abs() <= tol * want[live].abs() + 1e-30)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,d", [(3, 64), (2, 24), (2, 65), (1, 128), (1, 1)])
def test_wkv_step_gives_the_bits_of_the_scan_and_the_norm(dtype, H, d):
    """Head widths under, at and over a wave: a decode step's output is the one that a prompt step gives the same position."""
    from bitnet_c_amd import ops
    B, A, D = 7, H * d, 24
    r, k, v, dd, g = (_rand((B, A), 30 + i, dtype) for i in range(5))
    h, w0, u, weight = _rand((B, D), 40, dtype), _rand((A,), 41) - 2.0, _rand((A,), 42), _rand((A,), 43)
    state = torch.zeros(B, ops.wkv_state_floats(H, d, d) + D).cuda()
    slots, lens = torch.randperm(B).to(torch.int32).cuda(), torch.full((B,), 9, dtype=torch.int32).cuda()
    for i in range(2):
        ops.wkv_scan(r * (i + 1), k, v, dd, w0, u, h, state, slots, H, d, d, seq_lens=lens)
    a, b = state.clone(), state.clone()
    want = ops.head_norm_gate(ops.wkv_scan(r, k, v, dd, w0, u, h, a, slots, H, d, d, seq_lens=lens), g, weight, H, d, 1e-6)
    got = ops.wkv_step(r, k, v, dd, w0, u, h, b, slots, H, d, d, lens, g, weight, 1e-6)
    assert torch.equal(got, want) and torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dim", [8, 2048, 2056, 4096, 8192, 2052, 37])
@pytest.mark.parametrize("two", [True, False])
def test_rmsnorm_mean(dtype, dim, two):
    from bitnet_c_amd import ops
    a, b = _rand((3, dim), 1, dtype), _rand((3, dim), 2, dtype) * 5
    wa, wb = _rand((dim,), 3), _rand((dim,), 4)
    unit = lambda t: t.double() / torch.sqrt((t.double() ** 2).mean(-1, keepdim=True) + 1e-5)
    want = 0.5 * (unit(a) * wa.double() + unit(b) * wb.double()) if two else unit(a) * wa.double()
    got = ops.rmsnorm_mean(a, wa, b, wb, 1e-5) if two else ops.rmsnorm_mean(a, wa, None, None, 1e-5)
    # a float32 sum of dim squares and a few products, then the result's own rounding
    tol = (2.0 ** -8 if dtype == torch.bfloat16 else 0.0) + 2.0 ** -24 * (dim ** 0.5 + 8)
    assert float((got.double() - want).abs().max()) <= tol * float(want.abs().max())


@pytest.mark.parametrize("shift", [4, 1])
def test_rmsnorm_mean_weights_at_any_address(shift):
    """Weights at addresses that are multiples of 16 bytes (the wide kernel's) and of 4 (the other's)."""
    from bitnet_c_amd import ops
    dim = 2048
    a, b, wa, wb = _rand((3, dim), 1), _rand((3, dim), 2), _rand((dim,), 3), _rand((dim,), 4)
    want = ops.rmsnorm_mean(a, wa, b, wb, 1e-5)
    moved = []
    for w in (wa, wb):
        v = torch.empty(dim + 8, device="cuda")[shift:shift + dim]
        moved.append(v.copy_(w))
    got = ops.rmsnorm_mean(a, moved[0], b, moved[1], 1e-5)
    assert torch.equal(got, want) or shift == 1
    assert float((got - want).abs().max()) <= 2.0 ** -23 * (dim ** 0.5 + 8) * float(want.abs().max())


# widths: one group of eight, a workgroup's 256 groups and one past them, the most that registers hold (8,192) and beyond, not a
# multiple of eight
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dim", [8, 2048, 2056, 8192, 8200, 36])
@pytest.mark.parametrize("parts", [0, 1, 3])
@pytest.mark.parametrize("form", ["norm", "rows", "sum"])
def test_add_normed_rmsnorm_widths(dtype, dim, parts, form):
    from bitnet_c_amd import ops
    T = 3
    x, wb, w = _rand((T, dim), 1), _rand((dim,), 2), _rand((dim,), 3)
    if parts:
        delta = ops.PartialSums(_rand((parts, T, dim), 4))
        d = delta.slabs.double().sum(0)
    else:
        delta = _rand((T, dim), 4, dtype)
        d = delta.double()
    new = x.double() + d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-6) * wb.double()
    want = new / torch.sqrt((new * new).mean(-1, keepdim=True) + 1e-5) * w.double() if form == "norm" else new
    kw = dict(weight=w, eps=1e-5, out_dtype=dtype) if form == "norm" else dict(out_dtype=dtype, rows_out=True) if form == "rows" else {}
    out = ops.add_normed_rmsnorm(x, delta, wb, 1e-6, **kw)
    # float32 sums of dim squares and a handful of products; the result's own rounding
    tol = 2.0 ** -24 * (dim ** 0.5 + 16)
    assert float((x.double() - new).abs().max()) <= tol * float(new.abs().max())
    if form != "sum":
        tol += 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
        assert float((out.double() - want).abs().max()) <= tol * float(want.abs().max())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("W", [8, 2048, 2056, 8192, 8200, 36])
def test_row_norm_gate_widths(dtype, W):
    from bitnet_c_amd import ops
    T = 3
    o, weight = _rand((T, W), 1), _rand((W,), 2)
    gate = _rand((T, W + 24), 3, dtype)[:, 16:16 + W]
    f = o.double() / torch.sqrt((o.double() ** 2).mean(-1, keepdim=True) + 1e-6)
    want = f * weight.double() * torch.sigmoid(gate.double())
    got = ops.row_norm_gate(o, gate, weight, 1e-6)
    tol = (2.0 ** -8 if dtype == torch.bfloat16 else 0.0) + 2.0 ** -24 * (W ** 0.5 + 16)
    assert float((got.double() - want).abs().max()) <= tol * float(want.abs().max())


@pytest.mark.parametrize("shift", [4, 1])
def test_add_normed_rmsnorm_at_any_address(shift):
    """Rows and weights at addresses that are multiples of 16 and not of 32 bytes, and of 4 (which the wide kernel leaves to the
    other): what rows at the start of an allocation give."""
    from bitnet_c_amd import ops
    T, dim = 3, 2048

    def moved(t):
        buf = torch.empty(t.numel() + 8, dtype=t.dtype, device="cuda")
        v = buf[shift:shift + t.numel()].view(t.shape)
        v.copy_(t)
        assert v.data_ptr() % 32 == shift * t.element_size() % 32
        return v

    x, wb, w, delta = _rand((T, dim), 1), _rand((dim,), 2), _rand((dim,), 3), _rand((T, dim), 4)
    a, b = x.clone(), moved(x)
    out = ops.add_normed_rmsnorm(a, delta, wb, 1e-6, weight=w, eps=1e-5, out_dtype=torch.float32)
    got = ops.add_normed_rmsnorm(b, moved(delta), moved(wb), 1e-6, weight=moved(w), eps=1e-5, out_dtype=torch.float32)
    if shift == 4:
        assert torch.equal(a, b) and torch.equal(out, got)
    tol = 2.0 ** -24 * (dim ** 0.5 + 16)
    assert float((a - b).abs().max()) <= 2 * tol * float(a.abs().max()) and float((out - got).abs().max()) <= 2 * tol * float(out.abs().max())


# the widths below and at which the wide kernels begin
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dim", [504, 512, 1016, 1024])
def test_row_kernels_where_the_wide_ones_begin(dtype, dim):
    test_rmsnorm_mean(dtype, dim, True)
    test_add_normed_rmsnorm_widths(dtype, dim, 0, "norm")
    test_add_normed_rmsnorm_widths(dtype, dim, 3, "rows")
    test_row_norm_gate_widths(dtype, dim)


# the decay's last product inside the step: the same bits as the streaming product's in front of it.  head sizes: one tile of
# channels, two tiles for four waves, more tiles than waves; ranks: one block of 32, as many as a form holds and one fewer
@pytest.mark.parametrize("B", [1, 3, 16])
@pytest.mark.parametrize("H,d,rank", [(2, 16, 32), (3, 32, 64), (4, 64, 64), (2, 64, 96), (1, 96, 128), (2, 128, 224), (1, 64, 256)])
def test_wkv_step_with_the_decay_s_product(B, H, d, rank):
    from bitnet_c_amd import ops
    g = torch.Generator().manual_seed(B + H + d + rank)
    D = 64

    def rand(*shape):
        return torch.randn(*shape, generator=g).bfloat16().cuda()
    r, k, v, gate, h = rand(B, H * d), rand(B, H * d), rand(B, H * d), rand(B, H * d), rand(B, D)
    low, w2 = rand(B, rank + 8)[:, 8:], rand(H * d, rank) * 0.1
    w0, u = torch.rand(H * d, generator=g).cuda() - 3.0, torch.rand(H * d, generator=g).cuda()
    state = torch.randn(B + 2, ops.wkv_state_floats(H, d, d) + D, generator=g).cuda()
    slots, lens = torch.arange(B, 0, -1, dtype=torch.int32).cuda(), torch.tensor([5 - 5 * (i == 1) for i in range(B)], dtype=torch.int32).cuda()
    assert ops.wkv_step_takes_low(low, w2, d, d) and not ops.wkv_step_takes_low(low[:, :rank - 8], w2[:, :rank - 8].contiguous(), d, d)
    a, b = state.clone(), state.clone()
    want = ops.wkv_step(r, k, v, ops.linear(low, w2), w0, u, h, a, slots, H, d, d, lens, gate, None, 1e-6)
    got = ops.wkv_step(r, k, v, None, w0, u, h, b, slots, H, d, d, lens, gate, None, 1e-6, low, w2)
    live = lens > 0
    assert torch.equal(got[live], want[live]) and torch.equal(a, b)
