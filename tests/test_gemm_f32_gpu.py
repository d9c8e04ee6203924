"""The float32 product, every number in three bf16 parts: every form of the kernel against 64 bits, and against each other bit for bit
(the order of summation is a function of K alone).  What the parts keep of the operands is test_f32_parts_gpu.py's."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ops():
    from bitnet_c_amd import ops
    return ops


def _data(M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(M, K, generator=g), torch.randn(N, K, generator=g)


def _bound(x, w):
    """What float32 sums of products can be off by at the most, whatever their order in a chunk: its 128 large part products are added by
    as many roundings, the five kinds of small ones, 2^-8 of them and less, by 640 (two and a half large ones), the chunks' sums by
    K / 128; every one is 2^-24 of a partial sum, which the sum of magnitudes bounds, and the part products that are not formed are
    below one more."""
    K = x.shape[1]
    links = 4 * 32 + -(-K // 128) + 4
    return links * 2.0 ** -24 * (x.abs().double() @ w.abs().double().t())


# rows: the streaming kernel's tiles of 16 and their edges, the tile kernels' 32, 64, 128; columns: not a multiple of 8, 12 or
# 16, one past a tile; K: one 16-byte group, the edges of a block of 16, a step of 32 and a chunk of 128, several chunks,
# more chunks than one round of the streaming kernel's shared memory holds at 64 rows (16)
@pytest.mark.parametrize("M,N,K", [(1, 1, 4), (1, 2048, 12), (2, 17, 16), (15, 3072, 36), (16, 70, 128), (17, 130, 132), (33, 64, 2052),
                                   (64, 65, 2176), (64, 16, 8200)])
def test_forms_agree_up_to_64_rows(M, N, K):
    ops = _ops()
    x, w = _data(M, N, K, 11 * M + N)
    xd, wd = x.cuda(), w.cuda()
    y = ops._f32_product(xd, wd)
    assert torch.all((y.cpu().double() - x.double() @ w.double().t()).abs() <= _bound(x, w))
    for form in (1, 2, 3, 4, 5):
        assert torch.equal(ops._f32_product(xd, wd, form=form), y), form
    assert torch.equal(ops.linear(xd, wd), y)


@pytest.mark.parametrize("M,N,K", [(65, 31, 64), (127, 129, 100), (129, 257, 1000), (300, 2048, 512)])
def test_forms_agree_beyond_64_rows(M, N, K):
    ops = _ops()
    x, w = _data(M, N, K, M)
    xd, wd = x.cuda(), w.cuda()
    y = ops._f32_product(xd, wd)
    assert torch.all((y.cpu().double() - x.double() @ w.double().t()).abs() <= _bound(x, w))
    for form in (2, 3, 4, 5):
        assert torch.equal(ops._f32_product(xd, wd, form=form), y), form
    for m in (1, 17, 64):                                  # a row alone and among others
        assert torch.equal(ops._f32_product(xd[:m].contiguous(), wd), y[:m]), m
    with pytest.raises(ops.KernelError):
        ops._f32_product(xd, wd, form=1)                   # the streaming form ends at 64 rows


@pytest.mark.parametrize("activation", ["silu", "gelu_tanh", "relu2"])
@pytest.mark.parametrize("M,F,K", [(1, 8, 16), (7, 88, 132), (40, 64, 260), (130, 200, 64)])
def test_gated_epilogue(M, F, K, activation):
    ops = _ops()
    x, w = _data(M, 2 * F, K, F)
    xd, wi = x.cuda(), ops.interleave_gate_up(w[:F], w[F:]).cuda()
    want = ops.swiglu(ops._f32_product(xd, wi), True, activation)
    for form in (0, 1, 2, 3, 4, 5) if M <= 64 else (0, 2, 3, 4, 5):
        assert torch.equal(ops._f32_product(xd, wi, True, activation, form), want), form
    assert torch.equal(ops.linear_swiglu(xd, wi, True, activation=activation), want)


# widths that are no multiple of 8: one column, a remainder of each kind, one past whole workgroups of eight
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh", "relu2"])
@pytest.mark.parametrize("M,F,K", [(1, 1, 4), (1, 172, 64), (3, 9, 132), (8, 15, 64), (16, 44, 1156)])
def test_gated_epilogue_of_stacked_rows(M, F, K, activation):
    """All gate rows in front of all up rows: the bits of the product and the gated unit's kernel, with a norm of the rows too."""
    ops = _ops()
    x, w = _data(M, 2 * F, K, F)
    wide = torch.full((2 * F, K + 4), float("nan"), device="cuda")
    wide[:, :K] = w.cuda()
    xd, wd = x.cuda(), wide[:, :K]
    want = ops.swiglu(ops._f32_product(xd, wd), False, activation)
    assert ops.stacked_swiglu(M, wd, False)
    assert torch.equal(ops.linear_swiglu(xd, wd, False, activation=activation), want)
    pre = ops.stream_norm(xd, (torch.arange(K, device="cuda") % 7).float() / 7 + 0.5, 1e-5)
    if ops.takes_stream_norm(pre, wd):
        want = ops.swiglu(ops.linear_stream_norm(pre, wd), False, activation)
        assert torch.equal(ops.linear_stream_norm(pre, wd, None, 2, activation), want)
    assert not ops.stacked_swiglu(17, wd, False) and not ops.stacked_swiglu(M, wd, True)
    with pytest.raises(ops.KernelError):
        ops._f32_product(torch.cat([xd] * 17), wd, 2, activation)


def test_operands_that_are_not_aligned():
    """Activations at any address and stride give the same bits; weights whose rows are not whole 16-byte groups go to the
    tiled kernel, at every row count."""
    ops = _ops()
    x, w = _data(5, 40, 64, 3)
    y = ops.linear(x.cuda(), w.cuda())
    wide = torch.zeros(5, 71).cuda()
    wide[:, 3:67] = x.cuda()
    assert torch.equal(ops.linear(wide[:, 3:67], w.cuda()), y)
    padded = torch.zeros(40, 68).cuda()
    padded[:, :64] = w.cuda()
    assert torch.equal(ops.linear(x.cuda(), padded[:, :64]), y)
    shifted = torch.zeros(40 * 64 + 1).cuda()[1:].view(40, 64)
    shifted.copy_(w)
    assert ops._f32_product(x.cuda(), shifted) is None
    for m in (1, 5):
        got = ops.linear(x[:m].cuda(), shifted)
        assert torch.all((got.cpu().double() - x[:m].double() @ w.double().t()).abs() <= 64 * 2.0 ** -24 * (x[:m].abs().double() @ w.abs().double().t()))


def test_infinities_and_nan_stay_in_their_rows_and_columns():
    ops = _ops()
    x, w = _data(20, 48, 100, 9)
    x[3, 7], x[4, 99], w[5, 0] = float("inf"), float("nan"), float("-inf")
    for form in (1, 2, 3, 4, 5):
        y = ops._f32_product(x.cuda(), w.cuda(), form=form).cpu()
        fine = torch.isfinite(y)
        assert not fine[3].any() and not fine[4].any() and not fine[:, 5].any()
        fine[3], fine[4], fine[:, 5] = True, True, True
        assert fine.all()


# the forms that stage straight into shared memory (K of whole steps of 32): rows and columns at the edges of tiles of 32 and
# 64, one row and one column; K: one step, two, three and four (a chunk), chunks with one, two and three steps behind them,
# fewer and more steps than the four buffers; rows that lie further apart than they are long, NaN between and behind them
@pytest.mark.parametrize("M,N", [(1, 1), (31, 33), (32, 64), (64, 16), (65, 130), (129, 48), (300, 257)])
@pytest.mark.parametrize("K", [32, 64, 96, 128, 160, 192, 224, 256, 1056, 2048])
def test_forms_straight_into_shared_memory(M, N, K):
    ops = _ops()
    x, w = _data(M, N, K, M + 3 * N + K)
    wide, tall = torch.full((M + 1, K + 8), float("nan"), device="cuda"), torch.full((N + 1, K + 4), float("nan"), device="cuda")
    wide[:M, :K], tall[:N, :K] = x.cuda(), w.cuda()
    xd, wd = wide[:M, :K], tall[:N, :K]
    want = ops._f32_product(xd, wd, form=4)
    assert torch.all((want.cpu().double() - x.double() @ w.double().t()).abs() <= _bound(x, w))
    for form in (6, 7, 8, 0):
        assert torch.equal(ops._f32_product(xd, wd, form=form), want), form
    if N % 16 == 0:
        glu = ops._f32_product(xd, wd, True, "silu", form=4)
        for form in (6, 7, 8):
            assert torch.equal(ops._f32_product(xd, wd, True, "silu", form=form), glu), form


def test_forms_of_whole_steps_refuse_other_widths():
    ops = _ops()
    x, w = _data(40, 40, 100, 1)
    for form in (6, 7, 8):
        with pytest.raises(ops.KernelError):
            ops._f32_product(x.cuda(), w.cuda(), form=form)


# rows: the edges of 2, 4, 8 and 16; K: one chunk of 128, fewer chunks than waves, a chunk a wave, one wave with two, two and
# three a wave, five and six a wave; columns: one, no multiple of the tile's rows
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("N,K,R", [(1, 128, 16), (33, 896, 8), (40, 1024, 12), (16, 1152, 16), (30, 2048, 16), (17, 3072, 10), (24, 5632, 8)])
def test_streamed_copies_give_the_same_bits(M, N, K, R):
    ops = _ops()
    x, w = _data(M, N, K, 7 * M + N)
    xd, wd = x.cuda(), w.cuda()
    sw = ops.stream_copy(wd, R)
    assert torch.equal(ops.unstream(sw), wd)
    assert torch.equal(ops.linear(xd, wd, streamed=sw), ops.linear(xd, wd))
    wide = torch.full((M, K + 12), float("nan"), device="cuda")
    wide[:, :K] = xd
    assert torch.equal(ops.linear(wide[:, :K], wd, streamed=sw), ops.linear(xd, wd))
    if R == 16 and N % 16 == 0:
        assert torch.equal(ops.linear_swiglu(xd, wd, True, streamed=sw), ops.linear_swiglu(xd, wd, True))


def test_streamed_copies_whose_sums_do_not_fit_are_not_read():
    """Shared memory holds the sums of 84 chunks at 9 to 16 rows and of 234 at 5 to 8: a longer K is read from the row-major
    matrix."""
    ops = _ops()
    takes = ops._fn("gemm_f32", "bn_gemm_f32_streamed_supports")
    for m, most in ((9, 84), (16, 84), (5, 234), (8, 234)):
        assert takes(m, 16, 128 * most, 128 * most, 16, None) == 1 and takes(m, 16, 128 * (most + 1), 128 * (most + 1), 16, None) == 0
    for K in (84 * 128, 85 * 128, 14336):
        x, w = _data(16, 16, K, 3)
        xd, wd = x.cuda(), w.cuda()
        sw = ops.stream_copy(wd)
        for m in (8, 16):
            assert torch.equal(ops.linear(xd[:m].contiguous(), wd, streamed=sw), ops.linear(xd[:m].contiguous(), wd)), (K, m)


# a norm taken into the product behind it, and a product added into the stream, against the kernels of their own: the same bits.
# rows: the edges of 1, 2, 4 and 8; K: less than a thread's group of four, a chunk's remainder, fewer chunks than waves (the
# row-major kernel), one to four a wave, the widest at 2 rows and at 8; infinite and NaN rows stay their own
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("N,K,R", [(16, 4, 16), (36, 172, 16), (40, 896, 12), (28, 1024, 16), (24, 1152, 8), (16, 2048, 16), (32, 4096, 16)])
def test_products_with_a_norm_and_into_the_stream(M, N, K, R):
    ops = _ops()
    x, w = _data(M, N, K, 5 * M + N)
    xd, wd = x.cuda(), w.cuda()
    nw = torch.linspace(0.5, 1.5, K, device="cuda")
    if M > 3:
        xd[1, K // 2], xd[2, 0] = float("inf"), float("nan")
    copies = [None] + ([ops.stream_copy(wd, R)] if K % ops.F32_STREAM_CHUNK == 0 else [])
    xd = xd * torch.logspace(-1, 1, K, device="cuda") if K > 4 else xd
    if ops.can_norm_rows(M, K, torch.float32):
        h = ops.add_rmsnorm(xd.clone(), None, nw, 1e-5, torch.float32)
        for sw in copies:
            pre = ops.stream_norm(xd, nw, 1e-5)
            assert torch.equal(ops.linear_stream_norm(pre, wd, sw).nan_to_num(7.0), ops.linear(h, wd).nan_to_num(7.0)), sw is None
            if N % 16 == 0 and R == 16:
                assert torch.equal(ops.linear_stream_norm(pre, wd, sw, True).nan_to_num(7.0),
                                   ops.linear_swiglu(h, wd, True).nan_to_num(7.0)), sw is None
    else:
        assert K == 4096 and M > 2
    stream = torch.randn(M, N, device="cuda")
    for sw in copies:
        got = stream.clone()
        out = ops.linear_into_stream(xd, wd, got, torch.ones(N, device="cuda"), 1e-5, sw)
        assert out.stream is got
        assert torch.equal(got.nan_to_num(7.0), (stream + ops.linear(xd, wd)).nan_to_num(7.0)), sw is None


# where a norm stays a kernel of its own because the product reads a streamed copy then; the same bits on every route
@pytest.mark.parametrize("K", [384, 512, 896, 1024])
def test_norms_of_narrow_rows_stay_in_front_of_streamed_products(K, monkeypatch):
    ops = _ops()
    from bitnet_c_amd.parts.linear import Linear
    x, w = _data(3, 32, K, K)
    lin = Linear()
    lin.load(w, None, torch.device("cuda"), torch.float32)
    nw, calls = torch.linspace(0.5, 1.5, K, device="cuda"), []
    inside = ops.linear_stream_norm
    monkeypatch.setattr(ops, "linear_stream_norm", lambda *a, **k: (calls.append(1), inside(*a, **k))[1])
    want = ops.linear(ops.add_rmsnorm(x.cuda(), None, nw, 1e-5, torch.float32), w.cuda())
    for keep in (False, True):
        lin.keep_streamed(keep)
        calls.clear()
        assert torch.equal(lin(ops.stream_norm(x.cuda(), nw, 1e-5)), want)
        assert len(calls) == (0 if keep and 512 <= K < 1024 else 1)


# the forms beyond the tiles' first ones: rows at the edges of 32 and 64, columns one past a tile of 16, 32, 64 and 128; K: one block of 32, a
# chunk's remainder, as many chunks as the groups and waves that take them in turns, one more, and one round of eight more
@pytest.mark.parametrize("M,N", [(17, 1), (33, 65), (64, 129), (65, 33), (129, 300)])
@pytest.mark.parametrize("K", [4, 32, 36, 128, 160, 256, 512, 640, 1028, 1152, 2176])
def test_forms_that_share_out_the_chunks(M, N, K):
    ops = _ops()
    x, w = _data(M, N, K, M + 3 * N + K)
    wide, tall = torch.full((M + 1, K + 8), float("nan"), device="cuda"), torch.full((N + 1, K + 4), float("nan"), device="cuda")
    wide[:M, :K], tall[:N, :K] = x.cuda(), w.cuda()
    xd, wd = wide[:M, :K], tall[:N, :K]
    want = ops._f32_product(xd, wd, form=4)
    assert torch.all((want.cpu().double() - x.double() @ w.double().t()).abs() <= _bound(x, w))
    for form in (1, 5, 9, 10) + ((6, 8, 11, 12) if K % 32 == 0 else ()):
        if form > 1 or M <= 64:
            assert torch.equal(ops._f32_product(xd, wd, form=form), want), form
    if N % 16 == 0:
        glu = ops._f32_product(xd, wd, True, "silu", form=4)
        for form in (9, 10) + ((11, 12) if K % 32 == 0 else ()):
            assert torch.equal(ops._f32_product(xd, wd, True, "silu", form=form), glu), form


@pytest.mark.parametrize("M", [1, 3, 8, 16, 40])
def test_infinite_operands_give_infinite_sums(M):
    """An infinite number has no second part, and the nearest bf16 number of the largest float32 ones is infinite: sums with either
    come out as the float32 operations give them, and the others keep their bits."""
    ops = _ops()
    x, w = _data(M, 48, 256, M)
    w[7] = w[7].abs()
    plain = ops._f32_product(x.cuda(), w.cuda()).cpu()
    x[M // 2, 9], w[3, 200], w[5] = float("inf"), float("-inf"), 0.0
    w[5, 77], x[:, 77] = 0.25, 3.4e38
    want = x.double() @ w.double().t()
    sw = ops.stream_copy(w.cuda())
    runs = [ops._f32_product(x.cuda(), w.cuda(), form=f).cpu() for f in (1, 2, 4, 5, 6, 8, 9, 10, 11, 12)]
    runs += [ops.linear(x.cuda(), w.cuda(), streamed=sw).cpu()]
    for i, y in enumerate(runs):
        assert torch.equal(y.isnan(), want.isnan()), i
        big = want.float().isinf()
        assert torch.equal(y[big & ~want.isnan()], want.float()[big & ~want.isnan()]), i
        assert torch.all((y[:, 5] - 0.25 * 3.4e38).abs()[torch.arange(M) != M // 2] <= 0.25 * 3.4e38 * 2.0 ** -20), i
    x2, w2 = _data(M, 48, 256, M)
    w2[7] = w2[7].abs()
    x2[M // 2, 9] = float("inf")
    for f in (1, 4, 6, 9):
        y = ops._f32_product(x2.cuda(), w2.cuda(), form=f).cpu()
        rest = torch.arange(M) != M // 2
        assert torch.equal(y[rest], plain[rest]) and bool(y[M // 2].isinf().all()) and float(y[M // 2, 7]) == float("inf"), f


# chunks of K on both sides of where the rows' staged parts no longer fit beside the chunks' sums (and the rows are staged as they are),
# and of where neither fits
@pytest.mark.parametrize("M,fits,most", [(1, 1102, 1134), (2, 1102, 1134), (3, 502, 534), (4, 502, 534), (5, 202, 234), (8, 202, 234), (9, 52, 84), (16, 52, 84)])
def test_streamed_copies_of_rows_about_as_long_as_shared_memory_holds(M, fits, most):
    ops = _ops()
    takes = ops._fn("gemm_f32", "bn_gemm_f32_streamed_supports")
    for chunks in (fits, fits + 1, most - 1, most, most + 1):
        K = 128 * chunks
        assert takes(M, 16, K, K, 16, None) == (chunks <= most)
        x, w = _data(M, 16, K, chunks)
        xd, wd = x.cuda(), w.cuda()
        y = ops.linear(xd, wd, streamed=ops.stream_copy(wd))
        assert torch.equal(y, ops.linear(xd, wd)), K
        assert torch.all((y.cpu().double() - x.double() @ w.double().t()).abs() <= _bound(x, w)), K


# the largest numbers, whose nearest bf16 number is infinite, in finite results: rows of every kernel and form, also of normed rows, staged in
# parts (up to 4) and as they are; fewer chunks than waves, one a wave, more
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8, 16, 40, 130])
@pytest.mark.parametrize("K", [256, 1024, 2176])
def test_results_with_the_largest_operands_do_not_depend_on_the_kernel(M, K):
    ops = _ops()
    x, w = _data(M, 48, K, M + K)
    x[:, 5], x[:, 9] = 3.4e38 * x[:, 5].sign(), x[:, 9] * 2.0 ** -100
    w[:, 5], w[7, 9] = w[:, 5] * 2.0 ** -100, -3.395e38
    exact = x.double() @ w.double().t()
    xd, wd = x.cuda(), w.cuda()
    want = ops._f32_product(xd, wd, form=4)
    assert torch.all((want.cpu().double() - exact).abs() <= _bound(x, w))
    for form in (0, 2, 3, 5, 9, 10) + ((6, 7, 8, 11, 12) if K % 32 == 0 else ()) + ((1,) if M <= 64 else ()):
        assert torch.equal(ops._f32_product(xd, wd, form=form), want), form
    if M <= 16:
        assert torch.equal(ops.linear(xd, wd, streamed=ops.stream_copy(wd)), want)
    if ops.can_norm_rows(M, K, torch.float32):
        nw = torch.linspace(0.5, 1.5, K)
        nw[5] = 3.4e38
        xd, nw = _data(M, 48, K, M)[0].sign().cuda(), nw.cuda()              # normed: times 1 / sqrt(1 + eps)
        h = ops.add_rmsnorm(xd.clone(), None, nw, 1e-5, torch.float32)
        assert bool((h[:, 5].abs() > 3.389e38).all())
        wd[7, 9], wd[20, 5] = 1.0, 1.5                                       # an infinite result among the finite ones
        want = ops.linear(h, wd)
        assert bool(want[:, 20].isinf().all()) and int(want.isfinite().sum()) == M * 47
        for sw in (None, ops.stream_copy(wd)):
            assert torch.equal(ops.linear_stream_norm(ops.stream_norm(xd, nw, 1e-5), wd, sw), want), sw is None


# operands whose third, second or first bf16 part is rounded or zero (below 2^-110, 2^-118 and 2^-126), rows of them beside ordinary ones, against
# ordinary and large weights and small weights against ordinary and large rows: float32 products and sums, which keep denormal numbers
@pytest.mark.parametrize("M", [1, 3, 8, 16, 40, 130])
@pytest.mark.parametrize("K", [132, 1024])
@pytest.mark.parametrize("small,large", [(-108, 0), (-112, 0), (-116, 30), (-120, 0), (-122, 45), (-125, 0), (-132, 20), (-133, 45)])
def test_small_operands_keep_their_bits(M, K, small, large):
    ops = _ops()
    x, w = _data(M, 48, K, M + K)
    x[::2] *= 2.0 ** small
    x[1::2, ::3] *= 2.0 ** small
    w[:16] *= 2.0 ** large
    for x, w in ((x, w), (w[:M].contiguous(), torch.cat([x, x, x])[:48].contiguous())):
        exact = x.double() @ w.double().t()
        bound = _bound(x, w) + K * 2.0 ** -149             # every sum is rounded to a multiple of 2^-149 at the least
        xd, wd = x.cuda(), w.cuda()
        want = ops._f32_product(xd, wd, form=4)
        assert torch.all((want.cpu().double() - exact).abs() <= bound)
        for form in (0, 2, 3, 5, 9, 10) + ((6, 7, 8, 11, 12) if K % 32 == 0 else ()) + ((1,) if len(x) <= 64 else ()):
            assert torch.equal(ops._f32_product(xd, wd, form=form), want), form
        if len(w) % 16 == 0:
            for form in (0, 2, 4, 5, 9, 10):
                assert torch.equal(ops._f32_product(xd, wd, True, "silu", form), ops.swiglu(want, True, "silu")), form
            if len(x) <= 16:
                assert torch.equal(ops._f32_product(xd, wd, 2, "silu"), ops.swiglu(want, False, "silu"))
        if len(x) <= 16 and K % 128 == 0:
            assert torch.equal(ops.linear(xd, wd, streamed=ops.stream_copy(wd)), want)
    if ops.can_norm_rows(M, K, torch.float32):
        x, w = _data(M, 48, K, M)
        nw = torch.linspace(0.5, 1.5, K) * 2.0 ** small
        xd, wd, nw = x.cuda(), w.cuda(), nw.cuda()
        h = ops.add_rmsnorm(xd.clone(), None, nw, 1e-5, torch.float32)
        want = ops.linear(h, wd)
        assert torch.all((want.cpu().double() - h.cpu().double() @ w.double().t()).abs() <= _bound(h.cpu(), w) + K * 2.0 ** -149)
        for sw in (None, ops.stream_copy(wd)) if K % 128 == 0 else (None,):
            assert torch.equal(ops.linear_stream_norm(ops.stream_norm(xd, nw, 1e-5), wd, sw), want), sw is None


@pytest.mark.parametrize("F", [4095, 4097, 5461])
def test_wide_stacked_rows_are_normed_in_front(F, monkeypatch):
    """A feed-forward of gate rows in front of up rows takes its norm into the product while the CUs hold all its workgroups; the bits
    are those of the kernels of their own either way."""
    ops = _ops()
    from bitnet_c_amd.parts.ffn import SwiGLU
    part = SwiGLU(64, F)
    x, w = _data(3, 2 * F, 64, F)
    part.load({"w_gate": w[:F], "w_up": w[F:], "w_down": w[:F].t().contiguous()}, torch.device("cuda"), torch.float32)
    nw, calls, inside = torch.linspace(0.5, 1.5, 64, device="cuda"), [], ops.linear_stream_norm
    monkeypatch.setattr(ops, "linear_stream_norm", lambda *a, **k: (calls.append(1), inside(*a, **k))[1])
    got = part.forward(ops.stream_norm(x.cuda(), nw, 1e-5), None)
    assert len(calls) == (2 * F <= 32 * ops._compute_units())
    h = ops.add_rmsnorm(x.cuda(), None, nw, 1e-5, torch.float32)
    want = part.down(ops.swiglu(ops._f32_product(h, w.cuda()), False, "silu"))
    assert torch.equal(got, want)
