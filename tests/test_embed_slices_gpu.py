"""Embeddings of few rows are cut into slices over several workgroups, those of 512 rows and more are not: the same bits whatever the
number of rows, with unknown tokens and padding rows among them, at widths around a slice's and above what the slices cover at once."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dim", [1, 255, 256, 257, 1000, 2048])
@pytest.mark.parametrize("rows", [1, 3, 200, 511, 512])
def test_rows_in_slices(rows, dim, dtype):
    from bitnet_c_amd import ops
    g = torch.Generator().manual_seed(rows + dim)
    table, places = torch.randn((50, dim), generator=g).to(dtype), torch.randn((40, dim), generator=g).to(dtype)
    tokens = torch.randint(-1, 52, (700,), generator=g, dtype=torch.int32)          # -1, 50, 51: not in the table
    positions = torch.randint(-1, 42, (700,), generator=g, dtype=torch.int32)       # -1: a padding row; 40, 41: no learned place
    freq = torch.rand(((dim + 1) // 2,), generator=g)
    t, p, table, places, freq = tokens.cuda(), positions.cuda(), table.cuda(), places.cuda(), freq.cuda()
    plain = ops.embed_gather(table, t, 1.5)
    known = (tokens >= 0) & (tokens < 50)
    want = table.cpu()[tokens.long().clamp(0, 49)].float() * 1.5 * known[:, None]
    assert torch.equal(plain.cpu(), want)
    whole = [plain, ops.embed_gather_sinusoid(table, t, p, freq, 1.5), ops.embed_gather_learned(table, t, p, places, 1.5)]
    few = [f[:rows].contiguous() for f in (t, p)]
    part = [ops.embed_gather(table, few[0], 1.5), ops.embed_gather_sinusoid(table, *few, freq, 1.5),
            ops.embed_gather_learned(table, *few, places, 1.5)]
    for a, b in zip(part, whole):
        assert torch.equal(a, b[:rows])
