"""The float32 decode attention that rotates the query and the new key and stores the new key and value by itself gives the
bits of the kernel that rotates and stores followed by the plain attention, and leaves the same pages."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("H,Hkv,hs", [(4, 2, 16), (3, 1, 32), (2, 2, 64), (8, 2, 128), (20, 1, 64)])
@pytest.mark.parametrize("rotate,write", [(True, True), (True, False), (False, True)])
def test_rotation_and_store_inside_the_kernel(H, Hkv, hs, rotate, write):
    from bitnet_c_amd import ops
    from bitnet_c_amd.cache import PAGE
    torch.manual_seed(H * hs)
    lens = [1, 16, 17, PAGE, PAGE + 1, 4 * PAGE, 4 * PAGE + 1, 0, 611]         # the new position included; 0: a padding row
    B, width = len(lens), -(-max(lens) // PAGE)
    table = torch.randperm(B * width).to(torch.int32).reshape(B, width).to(DEV)
    pages = [torch.randn(B * width, Hkv, PAGE, hs, device=DEV) for _ in range(2)]
    for b, n in enumerate(lens):                         # what lies behind the keys before the new one may be anything
        for p in range(width):
            hold = max(0, min(PAGE, n - (1 if write else 0) - p * PAGE))
            for t in pages:
                t[int(table[b, p]), :, hold:] = float("nan")
    qkv = torch.randn(B, (H + 2 * Hkv) * hs, device=DEV)
    inv_freq = 1.0 / 10000.0 ** (torch.arange(hs // 2, device=DEV, dtype=torch.float32) * 2 / hs)
    seq_lens = torch.tensor(lens, dtype=torch.int32, device=DEV)
    n_splits, chunk = ops.decode_splits(B, H, Hkv, width * PAGE, torch.float32)
    args = dict(seq_lens=seq_lens, n_splits=n_splits, chunk=chunk, v_transposed=False, blocked=False)
    apart = [t.clone() for t in pages]
    rows, want, got = qkv.clone(), *(torch.full((B, H * hs), 7.0, device=DEV) for _ in range(2))
    ops.rope_kv_write(rows, seq_lens - 1, H, Hkv, hs, inv_freq=inv_freq if rotate else None, rope_dims=hs if rotate else 0,
                      seq_index=torch.arange(B, dtype=torch.int32, device=DEV) if write else None,
                      block_table=table if write else None, k_pages=apart[0] if write else None, v_pages=apart[1] if write else None,
                      v_transposed=False, blocked=False)
    ops.attention(rows, want, *apart, table, H, Hkv, hs, 0.3, **args)
    ops.attention(qkv, got, *pages, table, H, Hkv, hs, 0.3, fused_rotate=inv_freq if rotate else None, fused_write=write, **args)
    assert torch.isfinite(want).all() and torch.equal(got, want)
    for a, b in zip(apart, pages):
        assert torch.equal(a.nan_to_num(9.0), b.nan_to_num(9.0))


@pytest.mark.parametrize("H,Hkv,hs", [(4, 2, 16), (3, 1, 32), (2, 2, 64), (8, 2, 128), (20, 1, 64)])
def test_parts_of_a_page_and_of_a_run_give_the_same_bits(H, Hkv, hs):
    """What decides between them is the room for partial sums (bn_attn_f32_part_pages)."""
    from bitnet_c_amd import ops
    from bitnet_c_amd.cache import PAGE
    torch.manual_seed(hs)
    lens = [1, PAGE, PAGE + 1, 3 * PAGE + 7, 4 * PAGE, 4 * PAGE + 1, 0, 8 * PAGE, 2500]
    B, width = len(lens), -(-max(lens) // PAGE)
    part_pages = ops._fn("attn_f32", "bn_attn_f32_part_pages")
    assert part_pages(B * H, width, hs) == 1 and part_pages(64 * 2 ** 20, width, hs) == 4
    table = torch.randperm(B * width).to(torch.int32).reshape(B, width).to(DEV)
    kp, vp = (torch.randn(B * width, Hkv, PAGE, hs, device=DEV) for _ in range(2))
    q = torch.randn(B, H * hs, device=DEV)
    seq_lens = torch.tensor(lens, dtype=torch.int32, device=DEV)
    one, run = (torch.full((B, H * hs), 7.0, device=DEV) for _ in range(2))
    n_splits, chunk = ops.decode_splits(B, H, Hkv, width * PAGE, torch.float32)
    ops.attention(q, one, kp, vp, table, H, Hkv, hs, 0.3, seq_lens=seq_lens, n_splits=n_splits, chunk=chunk, v_transposed=False, blocked=False)
    parts = -(-width // 4)
    po, pm = torch.empty(B * H * parts, hs, device=DEV), torch.empty(B * H * parts, 2, device=DEV)
    _, GT, _ = ops.attention_row_shape(H, Hkv, True, None, hs)
    rc = ops._fn("attn_f32", "bn_attn_f32")(q.data_ptr(), H * hs, run.data_ptr(), H * hs, kp.data_ptr(), vp.data_ptr(), table.data_ptr(),
                                            width, seq_lens.data_ptr(), None, B, H, Hkv, hs, GT, 0.3, 4, po.data_ptr(), pm.data_ptr(),
                                            None, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and torch.equal(one, run)


@pytest.mark.parametrize("H,Hkv,hs", [(4, 2, 16), (3, 1, 32), (2, 2, 64), (8, 2, 128), (20, 1, 64)])
def test_a_table_much_wider_than_its_sequences(H, Hkv, hs):
    """Most workgroups find no keys, the others take several parts, and the parts are runs of pages where pages would be too
    many: the bits, and the stored keys and values, of a table of the sequences' own width."""
    from bitnet_c_amd import ops
    from bitnet_c_amd.cache import PAGE
    torch.manual_seed(H + hs)
    lens = [1, 64, 65, 0, 256, 257, 4 * PAGE + 63, 1000, 319]
    B, need = len(lens), -(-max(lens) // PAGE)
    inv_freq = 1.0 / 10000.0 ** (torch.arange(hs // 2, device=DEV, dtype=torch.float32) * 2 / hs)
    seq_lens = torch.tensor(lens, dtype=torch.int32, device=DEV)
    own = torch.randperm(B * need).to(torch.int32).reshape(B, need)
    pages = [torch.randn(B * need, Hkv, PAGE, hs, device=DEV) for _ in range(2)]
    qkv = torch.randn(B, (H + 2 * Hkv) * hs, device=DEV)
    part_pages, results = set(), []
    runs = (1 << 24) // (B * H * (hs + 2)) + 1                # pages of a table whose pages' sums would take over 64 MB
    for width in (need, 512, max(runs, 1024)):
        table = torch.zeros((B, width), dtype=torch.int32)
        table[:, :need] = own
        part_pages.add(ops._fn("attn_f32", "bn_attn_f32_part_pages")(B * H, width, hs))
        kp, vp = (t.clone() for t in pages)
        out = torch.full((B, H * hs), 7.0, device=DEV)
        n_splits, chunk = ops.decode_splits(B, H, Hkv, width * PAGE, torch.float32)
        ops.attention(qkv, out, kp, vp, table.to(DEV), H, Hkv, hs, 0.3, seq_lens=seq_lens, n_splits=n_splits, chunk=chunk,
                      v_transposed=False, blocked=False, fused_rotate=inv_freq, fused_write=True)
        results.append((out, kp, vp))
    assert part_pages == {1, 4}
    for got in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(got, results[0]))


@pytest.mark.parametrize("H,Hkv,hs", [(8, 2, 128), (20, 1, 64)])
@pytest.mark.parametrize("B", [9, 7])
def test_the_scratch_of_a_step_is_bounded(H, Hkv, hs, B):
    """Rows whose partial sums would take more than 128 MB are taken in turns over one buffer, to the same bits."""
    from bitnet_c_amd import ops
    from bitnet_c_amd.cache import PAGE
    torch.manual_seed(B)
    limit = 128 << 20
    width = 4 * (limit // (4 * 9 * H * (hs + 2))) * 2 + 3      # nine rows' runs take over twice the limit
    lens = [300, 1, 0, 65, 256, 257, 700, 64, 2][:B]
    need = -(-max(lens) // PAGE)
    table = torch.zeros((B, width), dtype=torch.int32)
    table[:, :need] = torch.randperm(B * need).to(torch.int32).reshape(B, need)
    kp, vp = (torch.randn(B * need, Hkv, PAGE, hs, device=DEV) for _ in range(2))
    qkv = torch.randn(B, (H + 2 * Hkv) * hs, device=DEV)
    seq_lens = torch.tensor(lens, dtype=torch.int32, device=DEV)
    results = []
    for t in (table[:, :need].contiguous().to(DEV), table.to(DEV)):
        a, b = kp.clone(), vp.clone()
        out = torch.full((B, H * hs), 7.0, device=DEV)
        n_splits, chunk = ops.decode_splits(B, H, Hkv, t.shape[1] * PAGE, torch.float32)
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        ops.attention(qkv, out, a, b, t, H, Hkv, hs, 0.3, seq_lens=seq_lens, n_splits=n_splits, chunk=chunk, v_transposed=False,
                      blocked=False, fused_write=True)
        assert torch.cuda.max_memory_allocated() - before <= limit + (1 << 16)
        results.append((out, a, b))
    assert all(torch.equal(x, y) for x, y in zip(*results))
