"""The float32 product keeps all 24 bits of its operands, although it multiplies bf16 parts of them: sums of four products, where a part
or a product of parts that is not there shows."""
import pytest
import torch

ALL = [("h", "h"), ("h", "m"), ("m", "h"), ("h", "l"), ("m", "m"), ("l", "h")]


def _data(M, N, K, seed):
    """Positive numbers with full mantissas in four columns (in different chunks where there are several, the last one among them)."""
    g = torch.Generator().manual_seed(seed)
    x, at = torch.zeros(M, K), [0, K // 3, K - 2, K - 1]
    x[:, at] = 0.5 + torch.rand(M, 4, generator=g)
    return x, 0.5 + torch.rand(N, K, generator=g)


def _bound(x, w):
    """Four large part products are added (three roundings, and one as the small ones' sum joins), the small ones, 2^-8 of them, by five
    instructions before; the three that are not formed are below 3 * 2^-26 of a product.  5 * 2^-24 of the sum holds all."""
    return 5 * 2.0 ** -24 * (x.double() @ w.double().t())


def _parts(t):
    h = t.bfloat16().float()
    m = (t - h).bfloat16().float()
    return {"h": h.double(), "m": m.double(), "l": (t - h - m).bfloat16().double()}


def test_a_product_that_is_left_out_breaks_the_bound():
    x, w = _data(40, 48, 132, 5)
    X, W, exact = _parts(x), _parts(w), x.double() @ w.double().t()
    err = lambda terms: ((sum(X[a] @ W[b].t() for a, b in terms) - exact).abs() / _bound(x, w)).max()
    assert err(ALL) < 0.1
    for gone in ALL:
        assert err([t for t in ALL if t != gone]) > 2, gone


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 3, 8, 16, 40, 130])
@pytest.mark.parametrize("K", [4, 132, 1024, 2176])
def test_every_form_keeps_the_operands_bits(M, K):
    from bitnet_c_amd import ops
    x, w = _data(M, 48, K, M + K)
    xd, wd = x.cuda(), w.cuda()
    fits = lambda y, x: bool(torch.all((y.cpu().double() - x.double() @ w.double().t()).abs() <= _bound(x, w)))
    for form in (0, 2, 3, 4, 5, 9, 10) + ((6, 7, 8, 11, 12) if K % 32 == 0 else ()) + ((1,) if M <= 64 else ()):
        assert fits(ops._f32_product(xd, wd, form=form), x), form
    copies = [None] + ([ops.stream_copy(wd)] if K % 128 == 0 else [])
    for sw in copies:
        assert fits(ops.linear(xd, wd, streamed=sw), x)
        if ops.can_norm_rows(M, K, torch.float32):
            nw = torch.linspace(0.5, 1.5, K, device="cuda")
            h = ops.add_rmsnorm(xd.clone(), None, nw, 1e-5, torch.float32).cpu()
            assert fits(ops.linear_stream_norm(ops.stream_norm(xd, nw, 1e-5), wd, sw), h)
    powers = 2.0 ** torch.randint(-3, 4, (48, K), generator=torch.Generator().manual_seed(K)).float()
    one = torch.zeros(M, K)
    one[:, K - 1] = 1 + 2.0 ** -9 + 2.0 ** -18 + 2.0 ** -23          # a part each, times a power of two: exact
    for a, b in ((one, powers), (powers[:M], torch.cat([one, one, one])[:48] if M >= 16 else one)):
        for form in (0, 2, 4, 5, 9):
            assert torch.equal(ops._f32_product(a.cuda().contiguous(), b.cuda().contiguous(), form=form).cpu().double(), a.double() @ b.double().t()), form
