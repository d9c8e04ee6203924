"""C entry points called with the arguments that they have always had, by a caller that brings its own declarations: a new argument in front of the stream
would be read from what such a caller did not pass."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
I, F, P, L = ctypes.c_int, ctypes.c_float, ctypes.c_void_p, ctypes.c_longlong


def _entry(library, name, *args):
    from bitnet_c_amd.csrc import build
    f = getattr(ctypes.CDLL(build.find_built(library) or build.compile_source(library)), name)
    f.restype, f.argtypes = I, list(args)
    return f


def test_general_decode_attention():
    from bitnet_c_amd import ops
    H, G, hs, B = 4, 2, 128, 3
    decode = _entry("attn_mfma_general", "bn_attn_general_decode", P, I, P, I, P, P, P, I, P, I, I, I, I, I, F, P, P, I, P, I, I, P, I, I, I, P, P, P, P)
    gen = torch.Generator(device="cuda").manual_seed(1)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda").to(torch.bfloat16)
    q, kp, vp = rand(B, H * hs), rand(2 * B, G, 64, hs), rand(2 * B, G, hs, 64)
    table, lens = torch.arange(2 * B, dtype=torch.int32, device="cuda").view(B, 2), torch.tensor([5, 0, 100], dtype=torch.int32, device="cuda")
    want, got = torch.empty(B, H * hs, dtype=torch.bfloat16, device="cuda"), torch.full((B, H * hs), 7.0, dtype=torch.bfloat16, device="cuda")
    ops.attention_general_decode(q, want, kp, vp, table, lens, H, G, hs, hs, 0.1)
    stream = torch.cuda.current_stream().cuda_stream
    assert decode(q.data_ptr(), H * hs, got.data_ptr(), H * hs, kp.data_ptr(), vp.data_ptr(), table.data_ptr(), 2, lens.data_ptr(), B, H, G, hs, hs, 0.1,
                  None, None, 0, None, 0, 0, None, 0, 1, 0, None, None, None, stream) == 0
    assert torch.equal(got, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_linear_attention(dtype):
    from bitnet_c_amd import ops
    H, d, B = 2, 64, 3
    scan = _entry("lightning", "bn_lightning_scan", I, P, I, I, I, I, P, P, P, L, P, I, P, P, I, I, I, I, P, I, P, I, P, F, P)
    gen = torch.Generator(device="cuda").manual_seed(2)
    x, decay = torch.randn(B, 3 * H * d, generator=gen, device="cuda").to(dtype), torch.tensor([0.9, 0.5], device="cuda")
    lens, slots = torch.tensor([4, 0, 1], dtype=torch.int32, device="cuda"), torch.arange(B, dtype=torch.int32, device="cuda")
    state = torch.randn(B, H * d * d, generator=gen, device="cuda")
    a, b, got = state.clone(), state.clone(), torch.empty(B, H * d, device="cuda")
    want = ops.lightning_scan(x, 0, H * d, 2 * H * d, decay, a, slots, H, d, d, seq_lens=lens)
    assert scan(ops._code(dtype), x.data_ptr(), 3 * H * d, 0, H * d, 2 * H * d, decay.data_ptr(), got.data_ptr(), b.data_ptr(), H * d * d, None, B, lens.data_ptr(),
                slots.data_ptr(), H, d, d, B, None, 1, None, 0, None, 1.0, torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(a, b) and torch.equal(got[[0, 2]], want[[0, 2]])
