"""The merge of a decode step's splits: out = sum_s e^(m_s - m) o_s / sum_s e^(m_s - m) l_s from the partial sums that the attention
kernels leave in the caller's room, against the same in 64 bits.  Numbers of splits at the edges of the kernels' forms (up to 4, 8,
16, 32 and 64), sequences that fill them, end in the middle, hold one key, and hold none."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SPLITS = [3, 4, 5, 8, 9, 16, 17, 32, 33, 64]


def _ops():
    from bitnet_c_amd import ops
    return ops


def _step(n, H, Hkv, hs, vd, seed):
    g = torch.Generator().manual_seed(seed)
    lens = torch.tensor([64 * n, 64 * (n // 2) + 5, 1, 0], dtype=torch.int32)
    q = torch.randn((4, H * hs), generator=g).bfloat16().cuda()
    k, v = (torch.randn((4 * n, Hkv, 64 * d), generator=g).bfloat16().cuda() for d in (hs, vd))
    return q, k, v, torch.arange(4 * n, dtype=torch.int32).reshape(4, n).cuda(), lens.cuda()


def _merged(po, ml, rows, n, vd, gate=None, sink=None):
    """(values, what the float32 sums and the bf16 rounding may be off by).  The weights' exponentials are float32 functions of
    differences of numbers up to 2^6 that are exact to 2^-18 then, 2^-17 with the function's own error; the sums of n terms and the
    reciprocal (n + 4) 2^-24; the gate's fast exponential and division 2^-18; the result is rounded to bf16, 2^-8 of it at the most."""
    ml, po = ml.double().cpu().reshape(rows, n, 2), po.double().cpu().reshape(rows, n, vd)
    m = ml[..., 0]
    top = m.amax(1) if sink is None else torch.maximum(m.amax(1), torch.full((rows,), float(sink), dtype=torch.float64))
    w = torch.where(torch.isinf(m), torch.zeros_like(m), torch.exp(m - torch.where(torch.isinf(top), torch.zeros_like(top), top)[:, None]))
    assert m[~torch.isinf(m)].abs().max() < 64
    po = torch.where(w[..., None] > 0, po, torch.zeros_like(po))               # a split without keys may hold anything
    den = (w * torch.where(w > 0, ml[..., 1], torch.zeros_like(m))).sum(1) + (0 if sink is None else torch.exp(sink - top))
    inv = torch.where(den > 0, 1 / den, torch.zeros_like(den))[:, None]
    if gate is not None:
        inv = inv * torch.sigmoid(gate.double().cpu().reshape(rows, vd))
    want, size = (w[..., None] * po).sum(1) * inv, (w[..., None] * po.abs()).sum(1) * inv
    return want, size * (2.0 ** -16 + (n + 4) * 2.0 ** -24) + want.abs() * 2.0 ** -8


@pytest.mark.parametrize("n", SPLITS)
@pytest.mark.parametrize("hs", [64, 128])
def test_merge_of_the_matrix_core_kernel(n, hs):
    ops, H, Hkv = _ops(), 8, 2
    q, k, v, table, lens = _step(n, H, Hkv, hs, hs, n + hs)
    out = torch.full((4, H * hs), float("nan"), dtype=torch.bfloat16, device="cuda")
    room = torch.full((4 * H * n * (hs + 2) + 1,), float("nan"), device="cuda")
    po, ml = room[1:1 + 4 * H * n * hs], room[1 + 4 * H * n * hs:]              # floats at odd addresses are room too
    GT = ops.attention_row_shape(H, Hkv, True)[1]
    rc = ops._fn("attn_mfma", "bn_attn_mfma")(q.data_ptr(), H * hs, out.data_ptr(), H * hs, k.data_ptr(), v.data_ptr(), table.data_ptr(), n,
                                              lens.data_ptr(), None, 4, 4, H, Hkv, hs, GT, 0, 0.1, n, 64, po.data_ptr(), ml.data_ptr(),
                                              None, 0, 0, None, None, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    want, off = _merged(po, ml, 4 * H, n, hs)
    assert torch.all((out.double().cpu().reshape(4 * H, hs) - want).abs() <= off)
    assert not out[3].any()                                                    # no keys: zeros


@pytest.mark.parametrize("n", SPLITS)
@pytest.mark.parametrize("hs,vd,gated,sink", [(64, 32, False, False), (128, 128, True, False), (96, 96, False, True), (192, 256, True, True)])
def test_merge_of_the_general_kernel(n, hs, vd, gated, sink):
    ops, H, Hkv = _ops(), 8, 2
    if not ops.attention_general_supported(torch.bfloat16, hs, vd):
        hs = 256
    q, k, v, table, lens = _step(n, H, Hkv, hs, vd, n + hs + vd)
    out = torch.full((4, H * vd), float("nan"), dtype=torch.bfloat16, device="cuda")
    gate = torch.randn((4, H * vd), device="cuda").bfloat16() if gated else None
    po, ml = (torch.full((4 * H * n, d), float("nan"), device="cuda") for d in (vd, 2))
    rc = ops._fn("attn_mfma_general", "bn_attn_general_decode")(
        q.data_ptr(), H * hs, out.data_ptr(), H * vd, k.data_ptr(), v.data_ptr(), table.data_ptr(), n, lens.data_ptr(), 4, H, Hkv, hs, vd,
        0.1, None, None, int(sink), None, 0, 0, gate.data_ptr() if gated else None, H * vd if gated else 0, n, 64, po.data_ptr(),
        ml.data_ptr(), None, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    want, off = _merged(po, ml, 4 * H, n, vd, gate, 0.0 if sink else None)
    assert torch.all((out.double().cpu().reshape(4 * H, vd) - want).abs() <= off)
