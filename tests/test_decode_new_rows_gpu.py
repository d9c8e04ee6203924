"""The decode attention of the general form that norms, rotates and stores its new rows itself, against qk_norm_store in front of it."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ops():
    from bitnet_c_amd import ops
    return ops


def _freq(dims):
    return (10000.0 ** (-2.0 * torch.arange(dims // 2, dtype=torch.float64) / dims)).to(torch.float32).cuda()


# hs, vd, heads, kv heads, rope_dims, norm, temperature, window, kept first keys, splits, columns behind the heads;
# lengths: a new token alone, at either end of a block of 32 and of a page, in the middle of both, a padding row
LENS = [1, 32, 33, 64, 65, 100, 128, 0, 129, 513, 700]
CASES = [(128, 128, 16, 4, 64, True, 0, 0, 0, 1, 0), (128, 128, 16, 4, 0, False, 16, 0, 0, 4, 0), (128, 128, 8, 8, 128, True, 0, 0, 0, 11, 0),
         (64, 128, 40, 2, 64, True, 7, 0, 0, 3, 0), (96, 64, 6, 2, 64, False, 0, 0, 0, 2, 384), (32, 32, 4, 4, 0, True, 0, 0, 0, 1, 0),
         (256, 256, 18, 1, 192, True, 0, 0, 0, 12, 0), (192, 96, 4, 2, 128, True, 3, 0, 0, 1, 0), (128, 128, 4, 1, 64, True, 0, 100, 0, 1, 512),
         (128, 64, 34, 2, 128, True, 0, 200, 5, 5, 0), (160, 128, 4, 2, 64, True, 0, 0, 0, 2, 0)]


@pytest.mark.parametrize("from_k", [False, True])
@pytest.mark.parametrize("hs,vd,H,G,dims,norm,every,window,keep,splits,more", CASES)
def test_new_rows(hs, vd, H, G, dims, norm, every, window, keep, splits, more, from_k):
    ops = _ops()
    if not ops.attention_general_supported(torch.bfloat16, hs, vd):
        pytest.skip("a head size that the kernel does not have")
    gen = torch.Generator(device="cuda").manual_seed(hs + vd + H + dims)
    B, P = len(LENS), ops.PAGE
    if from_k and hs != vd:
        pytest.skip("values that are the keys are as wide")
    width = H * hs + G * (hs + vd) + more if not from_k else (H + G) * hs + more
    qkv = torch.randn(B, width + 8, generator=gen, device="cuda").to(torch.bfloat16)[:, :width]
    per = -(-max(LENS) // P) + 1
    table = torch.randperm(B * per, generator=gen, device="cuda").to(torch.int32).view(B, per)
    kp = torch.randn(B * per, G, P, hs, generator=gen, device="cuda").to(torch.bfloat16)
    vp = torch.randn(B * per, G, vd, P, generator=gen, device="cuda").to(torch.bfloat16)
    lens = torch.tensor(LENS, dtype=torch.int32, device="cuda")
    for b, n in enumerate(LENS):                          # what lies behind a sequence's keys may be anything
        if n:
            kp[table[b, (n - 1) // P], :, (n - 1) % P:] = float("nan")
            vp[table[b, (n - 1) // P], :, :, (n - 1) % P:] = float("nan")
    weights = [torch.rand(hs, generator=gen, device="cuda") + 0.5 for _ in range(2)] if norm else [None, None]
    inv = _freq(dims) if dims else None
    chunk = -(-(min(window + P, per * P) if window else per * P) // (splits * P)) * P if splits > 1 else 0
    gate = qkv[:, width - H * vd:] if more else None
    args = dict(window=window, keep_first=keep, n_splits=splits, chunk=chunk, gate=gate, sink=bool(keep))
    old, kp2, vp2, want = qkv.clone(), kp.clone(), vp.clone(), torch.empty(B, H * vd, dtype=torch.bfloat16, device="cuda")
    wide = torch.zeros(B, width + 8, dtype=torch.bfloat16, device="cuda")
    wide[:, :width] = old
    rows = wide[:, :width]
    ops.qk_norm_store(rows, lens - 1, H, G, hs, v_dim=vd, q_weight=weights[0], k_weight=weights[1], eps=1e-6, temp_coef=0.3, temp_every=every,
                      seq_index=torch.arange(B, dtype=torch.int32, device="cuda"), block_table=table, k_pages=kp2, v_pages=vp2,
                      v_transposed=True, inv_freq=inv, rope_dims=dims, v_from_k=from_k)
    ops.attention_general_decode(rows, want, kp2, vp2, table, lens, H, G, hs, vd, hs ** -0.5,
                                 **dict(args, gate=rows[:, width - H * vd:] if more else None))
    out = torch.empty_like(want)
    fresh = ops.FreshRows(*weights, 1e-6, inv, dims, 0.3, every, from_k)
    ops.attention_general_decode(qkv, out, kp, vp, table, lens, H, G, hs, vd, hs ** -0.5, fresh=fresh, **args)
    assert torch.equal(qkv, old) and torch.equal(vp.view(torch.int16), vp2.view(torch.int16))      # values as they are; no other place is touched
    same = (kp == kp2) | (kp.isnan() & kp2.isnan())
    moved = ~same                                         # a norm's sum in another order: a key may round to its neighbour
    assert not norm or int(moved.sum()) <= kp.numel() // 1000
    assert norm or bool(same.all())
    assert bool(((kp.double() - kp2.double()).abs()[moved] <= kp2.double().abs()[moved] * 2.0 ** -7).all())
    scale = want.double().norm(dim=1) + 1e-9
    assert bool(((out.double() - want.double()).norm(dim=1) <= scale * 2.0 ** -8).all())           # the result's rounding
    assert bool(out[LENS.index(0)].eq(0).all())


def test_what_is_refused():
    ops = _ops()
    assert ops.takes_fresh_rope(128, 64) and ops.takes_fresh_rope(128, 128) and not ops.takes_fresh_rope(128, 96) and not ops.takes_fresh_rope(32, 64)
    assert not ops.takes_fresh_rope(128, 32) and not ops.takes_fresh_rope(128, 0)
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    run = lambda fresh, width: ops.attention_general_decode(z(1, width), z(1, 512), z(1, 1, 64, 128), z(1, 1, 128, 64), i32([[0]]), i32([1]), 4, 1,
                                                            128, 128, 1.0, fresh=fresh)
    run(ops.FreshRows(), 768)
    for fresh, width in ((ops.FreshRows(), 640), (ops.FreshRows(inv_freq=_freq(32), rope_dims=32), 768),
                         (ops.FreshRows(q_weight=torch.ones(128, device="cuda")), 768), (ops.FreshRows(inv_freq=_freq(64), rope_dims=128), 768)):
        with pytest.raises(ops.KernelError):
            run(fresh, width)


def test_norms_that_lie_anywhere():
    """A layer whose norms are pieces of one tensor, on no 16 bytes, decodes as before: through qk_norm_store."""
    from bitnet_c_amd.cache import PagedCache
    from bitnet_c_amd.parts import MIXERS, PartSpec
    from test_parts_gpu import _ctx
    H, G, hs, hidden, bf = 4, 2, 64, 64, torch.bfloat16
    gen = torch.Generator().manual_seed(3)
    steps = [torch.randn(n, hidden, generator=gen).to(bf).cuda() for n in (70, 1, 1)]
    results, weights = [], None
    for shift in (0, 1):
        att = MIXERS.build(PartSpec.of("attention", hidden=hidden, n_heads=H, n_kv_heads=G, head_dim=hs, scale=hs ** -0.5, position=PartSpec.of("none"),
                                       qk_norm_eps=1e-6))
        weights = weights or {k: torch.randn(v.shape, generator=gen) * 0.2 + (k in ("q_norm", "k_norm")) for k, v in att.tensors().items()}
        norms = torch.zeros(2 * hs + 4, device="cuda")
        tensors = dict(weights, q_norm=norms[shift:shift + hs], k_norm=norms[hs + shift:2 * hs + shift])
        for k in ("q_norm", "k_norm"):
            tensors[k].copy_(weights[k])
        att.load(tensors, "cuda", bf)
        assert att.q_norm.data_ptr() % 16 == 4 * shift
        cache = PagedCache([att.cache_need()], [None], 64 * 8, dtype=bf, device="cuda")
        slot, out = cache.alloc_slot(), []
        for x in steps:
            ctx, tables, longest = _ctx(cache, [slot], [x.shape[0]], bf)
            out.append(att.forward(x, ctx, cache.view(0, tables, longest)))
            cache.commit([slot], [x.shape[0]])
        results.append(torch.cat(out))
    a, b = (r.double() for r in results)
    assert torch.equal(a[:70], b[:70])                    # prompts go one way
    assert float((a - b).norm()) <= 2.0 ** -7 * float(a.norm())        # a norm's sum in another order, then two roundings to bf16
