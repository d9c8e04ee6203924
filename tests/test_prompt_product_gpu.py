"""The prompt product whose two groups of waves take turns at the matrix cores: whole results, gated units and slabs over ranges of K, at
sizes that fill no tile and at which every tile is the one that is chosen."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ops():
    from bitnet_c_amd import ops
    return ops


def _data(M, N, K, pad=0):
    g = torch.Generator(device="cuda").manual_seed(M * 31 + N * 7 + K)
    x = torch.randn(M, K + pad, generator=g, device="cuda").to(torch.bfloat16)[:, :K]
    w = (torch.randn(N, K, generator=g, device="cuda") * 0.05).to(torch.bfloat16)
    return x, w, x.double() @ w.double().t()


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


# one step, two, an odd and an even number of them; rows and columns: one past a tile, one short of it, sixteen and four past
SHAPES = [(1, 16, 64), (129, 208, 64), (129, 1040, 4096), (193, 4112, 192), (300, 528, 128), (511, 8208, 1088), (700, 8208, 448),
          (1000, 12304, 320), (1025, 16400, 128), (385, 16400, 192), (570, 11216, 2048), (257, 4112, 64)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_products_and_gated_units(M, N, K):
    ops = _ops()
    x, w, ref = _data(M, N, K, 24)                   # rows that lie further apart than they are long
    assert _rel(ops.gemm_mfma(x, w, torch.float32), ref) < 1e-5          # bf16 products are exact in float32: the sums' roundings
    assert _rel(ops.gemm_mfma(x, w), ref) < 2.0 ** -8                    # one rounding to bf16
    if N % 4 == 0:                                   # columns that end inside a tile of 16
        assert _rel(ops.gemm_mfma(x, w[:N - 12], torch.float32), ref[:, :N - 12]) < 1e-5
    v = ref.view(M, N // 16, 2, 8)
    for act, fn in (("silu", torch.nn.functional.silu), ("relu2", lambda t: t.clamp(min=0) ** 2),
                    ("gelu_tanh", lambda t: torch.nn.functional.gelu(t, approximate="tanh"))):
        want = (fn(v[:, :, 0]) * v[:, :, 1]).reshape(M, N // 2)
        got = ops.gemm_mfma(x, w, glu8=True, activation=act)
        assert _rel(got, want) < 2.0 ** -8, act      # the unit is formed in float32 and rounded once
        if M >= ops.PROMPT_ROWS:
            assert torch.equal(ops.linear_swiglu(x, w, True, activation=act), got), act


@pytest.mark.parametrize("act", ["silu", "gelu_tanh", "relu2"])
def test_gates_of_every_finite_number(act):
    """Eight gates a row that are one bf16 number each, beside ups of one: the activation of every finite number."""
    ops = _ops()
    v = torch.arange(2 ** 16, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    v = v[v.isfinite()].view(-1, 8).cuda()
    x = torch.zeros(v.shape[0], 64, dtype=torch.bfloat16, device="cuda")
    x[:, :8], x[:, 8] = v, 1.0
    w = torch.zeros(16, 64, dtype=torch.bfloat16, device="cuda")
    w[torch.arange(8), torch.arange(8)], w[8:, 8] = 1.0, 1.0
    got, z = ops.linear_swiglu(x, w, True, activation=act).double(), v.double()
    y = (2 / torch.pi) ** 0.5 * (z + 0.044715 * z ** 3)
    want = z * torch.sigmoid(z) if act == "silu" else z * torch.sigmoid(2 * y) if act == "gelu_tanh" else z.clamp(min=0) ** 2
    inf = want > 3.39e38                                  # beyond bf16
    assert bool((got[inf] > 3.38e38).all())
    # the rounding to bf16; an exponent of up to 150 is a float32 number; factors below 1.2e-38 are 0
    assert bool(((got - want).abs()[~inf] <= want.abs()[~inf] * (2.0 ** -8 + 150 * 2.0 ** -23) + 4e-36).all())


# slabs: two to six ranges of K, the last one shorter; every range summed alone
@pytest.mark.parametrize("M,N,K", [(129, 264, 8256), (200, 4096, 8192), (257, 4104, 14336), (513, 1032, 4160), (1500, 2056, 8192),
                                   (513, 4104, 14336), (900, 4100, 9024), (300, 520, 64), (130, 136, 8896)])
def test_slabs(M, N, K):
    ops = _ops()
    x, w, ref = _data(M, N, K)
    parts = ops.linear_split_rows(x, w)
    S = parts.slabs.shape[0]
    steps = -(-(K // 64) // S) * 64
    assert 1 <= S <= 6 and (S - 1) * steps < K and _rel(parts.slabs.double().sum(0), ref) < 1e-5
    for s in range(S):
        a, b = s * steps, min(K, (s + 1) * steps)
        assert _rel(parts.slabs[s], x[:, a:b].double() @ w[:, a:b].double().t()) < 1e-5, s
    # into the stream, and normed
    stream = torch.linspace(-1, 1, M * N, device="cuda").view(M, N).contiguous()
    weight = torch.linspace(0.5, 1.5, N, device="cuda")
    want = stream.double() + ref
    h = ops.add_rmsnorm(stream, parts, weight, 1e-5, torch.bfloat16)
    assert _rel(stream, want) < 1e-5
    assert _rel(h, want / torch.sqrt((want * want).mean(1, keepdim=True) + 1e-5) * weight) < 2.0 ** -8


# products in one launch: sizes at which each tile is chosen, with rows and columns that fill none, and a group beside others
@pytest.mark.parametrize("n,M,N,K", [(3, 129, 260, 64), (6, 130, 2052, 192), (2, 1025, 2048, 128), (4, 1000, 1028, 576), (5, 2049, 1540, 64),
                                     (4, 4099, 2564, 128)])
def test_products_side_by_side(n, M, N, K):
    ops = _ops()
    assert ops.group_rows(n, M, N, K)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    xs = torch.randn(n, M, K + 8, generator=g, device="cuda").to(torch.bfloat16)[:, :, :K]        # rows further apart than they are long
    ws = [(torch.randn(N, K, generator=g, device="cuda") * 0.05).to(torch.bfloat16) for _ in range(n)]
    other = (xs[0], ws[0][:16].contiguous(), None, "tanh"), (xs[1], ws[1][:N - 4], None, None)
    items = [(x, w, None, None) for x, w in zip(xs, ws)]
    got = ops.linear_group([items[0], other[0], *items[1:], other[1]])
    beside = [got.pop(1), got.pop()]
    for (x, w, _, _), y, alone in zip(items, got, ops.gemm_items(list(xs), ws)):
        assert torch.equal(y, alone) and _rel(y, x.double() @ w.double().t()) < 2.0 ** -8
    assert _rel(beside[0], torch.tanh(xs[0].double() @ ws[0][:16].double().t())) < 2.0 ** -7
    assert torch.equal(beside[1], ops.linear(xs[1], ws[1][:N - 4]))
    with pytest.raises(ops.KernelError):
        ops.gemm_items([xs[0], xs[1, 1:]], ws[:2])


# an activation on the sums: the same edges, from its least rows on; results that lie nowhere near a whole 16 bytes
@pytest.mark.parametrize("M,N,K", [(256, 2048, 64), (257, 4112, 64), (300, 528, 128), (511, 8204, 1088), (700, 8208, 448), (1025, 16396, 128)])
@pytest.mark.parametrize("act", ["gelu_erf", "relu2"])
def test_activations_on_the_sums(M, N, K, act):
    ops = _ops()
    x, w, ref = _data(M, N, K, 24)
    got = ops.gemm_unary(x, w, act)
    want = torch.nn.functional.gelu(ref) if act == "gelu_erf" else ref.clamp(min=0) ** 2
    assert _rel(got, want) < 2.0 ** -8
    # element by element: the sums' roundings, the rounding to bf16 and 1e-4 of the value where it is as small as 1e-20 (|z| < 9.3)
    assert bool(((got.double() - want).abs() <= want.abs() * (2.0 ** -8 + 1e-4) + 1e-5).all())
    two = ops.unary_act(ops.linear(x, w), act)
    assert _rel(got, want) <= _rel(two, want)            # one rounding instead of two
    assert torch.equal(ops.linear_unary(x, w, act), got if ops.unary_in_product(M, N, K, act) else two)
    x = x.clone()
    x[M - 1, 5], x[M - 2, 7] = float("nan"), 1e9          # NaN stays NaN (as the library's two kernels have it), a large number gives itself or 0
    got, z = ops.gemm_unary(x, w, act), x[M - 2].double() @ w.double().t()
    large = z.clamp(min=0) if act == "gelu_erf" else z.clamp(min=0) ** 2
    assert torch.equal(got[M - 1].isnan(), ops.unary_act(ops.linear(x, w), act)[M - 1].isnan())
    assert _rel(got[M - 2], large) < 2.0 ** -8 and _rel(got[:M - 2], want[:M - 2]) < 2.0 ** -8


# experts whose lists hold more tiles than rows fill: one live tile, numbers of them that are no multiple of the XCDs, every tile live; some experts without rows
@pytest.mark.parametrize("E,D,F,T,used", [(64, 64, 640, 17, 1), (16, 192, 1096, 40, 3), (8, 320, 576, 300, 8), (5, 128, 4168, 700, 2), (2, 576, 2056, 1024, 2)])
def test_experts_whose_lists_are_not_full(E, D, F, T, used):
    ops = _ops()
    g = torch.Generator(device="cuda").manual_seed(E + D + F + T)
    h = torch.randn(T, D, generator=g, device="cuda").to(torch.bfloat16)
    up = (torch.randn(E, F, D, generator=g, device="cuda") / D ** 0.5).to(torch.bfloat16)
    down = (torch.randn(E, D, F, generator=g, device="cuda") / F ** 0.5).to(torch.bfloat16)
    names = torch.randperm(E, generator=torch.Generator().manual_seed(T))[:used].int()
    ids = names[torch.randint(0, used, (T, 1), generator=torch.Generator().manual_seed(D))].cuda()
    ids[:used, 0] = names.cuda()
    wts = torch.rand(T, 1, generator=g, device="cuda") + 0.5
    y = ops.moe_experts_grouped(h, up, down, ids, wts, "relu2", False).slabs[0]
    for e in names.tolist():
        rows = (ids[:, 0] == e).nonzero().view(-1)
        mid = ((h[rows].double() @ up[e].double().t()).clamp(min=0) ** 2).to(torch.bfloat16).double()
        want = wts[rows].double() * (mid @ down[e].double().t())
        off = (y[rows].double() - want).norm(dim=1) / want.norm(dim=1)
        # most rows: float32 sums; a few: a term of the middle whose float32 sum is rounded to the neighbouring bf16 number, 2^-8 of that term
        assert float(off.median()) < 1e-6 and float(off.max()) < 2.0 ** -8


def test_numbers_that_are_none():
    """A row of X or of W that holds NaN or an infinity reaches its own results alone."""
    ops = _ops()
    M, N, K = 260, 528, 192
    x, w, ref = _data(M, N, K)
    x, w = x.clone(), w.clone()
    x[255, 3], x[256, 191], w[17, 64] = float("nan"), float("inf"), float("nan")
    y = ops.gemm_mfma(x, w, torch.float32)
    bad = torch.zeros(M, N, dtype=torch.bool, device="cuda")
    bad[255], bad[256], bad[:, 17] = True, True, True
    assert not bool(y[bad].isfinite().any()) and _rel(y[~bad], ref[~bad]) < 1e-5


def test_what_the_rules_say():
    ops = _ops()
    bf = torch.bfloat16
    assert ops.can_split_rows(129, 4096, 14336, bf) and ops.can_split_rows(2048, 4096, 14336, bf)
    assert not ops.can_split_rows(128, 4096, 14336, bf) and not ops.can_split_rows(2049, 4096, 14336, bf)
    assert not ops.can_split_rows(548, 4096, 4096, bf) and not ops.can_split_rows(548, 4096, 14336 + 32, bf)
    assert not ops.can_split_rows(548, 4096, 14336, torch.float32)
    assert ops.group_rows(4, 129, 2048, 2048) and ops.group_rows(2, 1024, 2048, 2048) and not ops.group_rows(2, 1023, 2048, 2048)
    assert not ops.group_rows(4, 128, 2048, 2048) and not ops.group_rows(4, 8192, 2048, 2048) and not ops.group_rows(7, 512, 512, 512)
    for act, (M, N, K) in (("gelu_erf", (256, 16384, 4096)), ("relu2", (2048, 8192, 2048))):
        assert ops.unary_in_product(M, N, K, act) and not ops.unary_in_product(255, N, K, act) and not ops.unary_in_product(1024, 2048, 2048, act)
        assert not ops.unary_in_product(M, N, K + 32, act) and not ops.unary_in_product(M, N - 2, K, act) and not ops.unary_in_product(M, N, K, "silu")
    assert not ops.group_rows(4, 512, 2048, 2080) and not ops.group_rows(4, 512, 2046, 2048) and not ops.group_rows(1, 2048, 512, 512)
    with pytest.raises(ops.KernelError):
        ops.linear_split_rows(torch.zeros(130, 96, dtype=bf, device="cuda"), torch.zeros(64, 96, dtype=bf, device="cuda"))


def test_slabs_are_left_where_ranges_pay():
    """The rule goes by the plan's ranges on both sides of any K, the shortest as well."""
    ops = _ops()
    for K in (8192, 8256, 8704):
        assert ops.can_split_rows(2048, 2048, K, torch.bfloat16) and ops.can_split_rows(1280, 4096, K, torch.bfloat16)
        assert not ops.can_split_rows(4096, 2048, K, torch.bfloat16) and not ops.can_split_rows(2048, 4096, K, torch.bfloat16)
    for M, N, K in ((2048, 2048, 8192), (3072, 2048, 8192), (3072, 2048, 8256), (4096, 2048, 10240), (2048, 4096, 9216), (2048, 4096, 10240), (1024, 8192, 9216)):
        assert ops.can_split_rows(M, N, K, torch.bfloat16) == (ops._fn("gemm_mfma", "bn_gemm_mfma_splits")(M, N, K) > 1)
    assert not ops.can_split_rows(2048, 2048, 8192 - 64, torch.bfloat16)


def test_few_tiles_of_long_rows_are_no_group():
    ops = _ops()
    for n, M, N, K, take in ((2, 1024, 256, 1024, True), (2, 1024, 256, 1088, False), (2, 2048, 512, 4096, True), (2, 1024, 512, 4096, False), (3, 129, 256, 960, True),
                             (3, 129, 256, 1024, False), (3, 129, 1024, 4096, False), (3, 129, 1280, 4096, True), (4, 129, 256, 8192, True)):
        assert ops.group_rows(n, M, N, K) == take, (n, M, N, K)


@pytest.mark.parametrize("M", [193, 250, 256, 300, 577, 2049])
@pytest.mark.parametrize("act", ["gelu_erf", "relu2"])
def test_an_eager_step_rounds_where_its_replay_does(M, act):
    """The rows of a step are those of the captured step that replays it, which is longer: an activation is taken of rounded numbers in both or in neither."""
    ops = _ops()
    x, w, _ = _data(ops.row_bucket(M), 8192, 1024)
    assert ops.unary_in_product(ops.row_bucket(M), 8192, 1024, act)
    assert torch.equal(ops.linear_unary(x[:M], w, act), ops.linear_unary(x, w, act)[:M])


@pytest.mark.parametrize("M,N,K,split", [(2600, 2048, 8192, False), (2560, 2048, 8192, True), (2100, 3072, 8192, False), (2048, 3072, 8192, True)])
def test_an_eager_step_leaves_slabs_where_its_replay_does(M, N, K, split):
    from bitnet_c_amd.parts.linear import Linear
    ops = _ops()
    x, w, _ = _data(ops.row_bucket(M), N, K)
    lin = Linear()
    lin.load(w, None, "cuda", torch.bfloat16)
    assert isinstance(lin.lazy(x[:M]), ops.PartialSums) == isinstance(lin.lazy(x), ops.PartialSums) == split
