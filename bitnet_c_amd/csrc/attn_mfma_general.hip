// Prompt attention on the matrix cores for the attention mixer's general form: head sizes that are multiples of 32,
// values of a width of their own (a multiple of 32), a logarithmic distance bias, a sink in the softmax, no rotation
// (the queries and keys arrive encoded).  bf16, 16x16x32 MFMA.  Keys lie in pages with a row per position
// ([page, kv head, BN_PAGE, hs]), values transposed ([page, kv head, vd, BN_PAGE]): both operands of both products are
// then 16 consecutive bytes a lane.  The prompt form lays them out through shared memory, the decode form takes them straight
// from the pages.
//
// A wave owns one tile of up to 16 query tokens of one head and walks the keys 0 .. last query in blocks of 32 (with a
// window w > 0 a query at position i sees the keys i - w + 1 .. i only, and the walk begins at the block of the tile's
// first visible key; with keep_first k > 0 the keys 0 .. k - 1 stay in sight, and the walk begins at block 0 and leaps from
// the block behind the kept keys to the window's first):
//   S^T = K . Q^T      two tiles of 16 keys x 16 queries; tile h holds the block's keys 8 (i / 4) + 4 h + i % 4 in its
//                      row i, so that lane group g ends up with the scores of keys 8 g .. 8 g + 7 of its query column:
//                      what the second product wants from it as its operand, without any exchange
//   s = S scale - a[h] ln(1 + b[h] (i - j)) or S scale - a[h] (i - j), masked above the diagonal; online softmax in base 2, float32
//   O^T += V^T . P^T   vd / 16 tiles; the weights' sums from the matrix cores as well (a tile of ones times P^T), so that
//                      numerator and denominator see the same bf16 weights
// and at the end the sink (one more term of score 0 without a value) joins the sums, then O / l is stored, times
// sigmoid(gate) element by element when the mixer gates its heads' outputs.
//
// Decode form (attn_general_decode_kernel): the 16 columns of a tile are the query heads that share a kv head (the one new
// token of a sequence), so a block of keys and values is loaded once for all of them: a wave owns (sequence, kv head,
// sixteen of its heads, split of the keys) and either stores the result or, with the keys split over gridDim.z, leaves
// unnormalised sums with their maximum and weight sum for attn_general_combine_kernel, which merges the splits in index
// order.  Splits are runs of whole pages; with a window they are counted from the page of the window's first key, and the
// kept first keys are the first split's.
// Every other shape or type is the vector kernel's (attn_rows.hip).
#include "common.h"
#include <math.h>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) float f32x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;

#define AG_LOG2E 1.4426950408889634f

struct GenArgs {
    const bf16* q;            // [T, q_stride]: head h at h * hs, norms and temperature applied
    bf16* out;                // [T, out_stride]: head h at h * vd
    const bf16* k_pages;      // [pages, Hkv, BN_PAGE, hs]
    const bf16* v_pages;      // [pages, Hkv, vd, BN_PAGE]
    const int* block_table;   // [seqs, bt_stride]
    const int* tiles;         // [n, 4]: sequence, first row, rows <= 16, position of the first
    const float* dist_a;      // [H] or null
    const float* dist_b;      // [H], or null: the bias is linear, dist_a[h] (i - j)
    const bf16* gate;         // [T, gate_stride] beside out's columns, or null: out times sigmoid(gate)
    int gate_stride;
    int q_stride, out_stride, bt_stride, H, Hkv;
    float scale;
    int sink;                 // 1: one more term without a value in the softmax's denominator, exp(sink_values[head])
    const float* sink_values; // [H] float32, or null: the term's score is 0
    int window;               // 0: every earlier key; else the last `window` positions, the query's own included
    int keep_first;           // with a window: the first keep_first positions stay visible however far back they are
};

__device__ __forceinline__ bf16x8 ag_ld16(const bf16* p) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(p));
}
// a decode step's cached keys and values; ONCE: non-temporally
template <bool ONCE> __device__ __forceinline__ bf16x8 ag_ld16_cached(const bf16* p) {
    if constexpr (ONCE) return __builtin_bit_cast(bf16x8, bn_load_once(p));
    else return ag_ld16(p);
}

// the largest of a value over the lanes 16, 32 and 48 away (the four lane groups of a column): two half-wave swaps between registers
__device__ __forceinline__ float ag_max_over_groups(float x) {
    const unsigned b = __float_as_uint(x);
    const auto r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    const unsigned c = __float_as_uint(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
    const auto t = __builtin_amdgcn_permlane32_swap(c, c, false, false);
    return fmaxf(__uint_as_float(t[0]), __uint_as_float(t[1]));
}

// a lane's eight scores (keys first .. first + 7) of the query at qpos: scaled, less the distance bias, in the exponent's
// base 2.  bias: 0 none, 1 logarithmic (a ln(1 + b d) log2(e) = a log2(1 + b d)), 2 linear (a d, with log2(e) in a)
__device__ __forceinline__ void ag_scores(float (&s)[8], const f32x4& s0, const f32x4& s1, float scale2, int bias, float ba, float bb,
                                          int qpos, int first) {
#pragma unroll
    for (int e = 0; e < 8; ++e) s[e] = (e < 4 ? s0[e & 3] : s1[e & 3]) * scale2;
    const float dist = (float)(qpos - first);
    if (bias == 2) {
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] = fmaf(-ba, dist - (float)e, s[e]);
    } else if (bias == 1) {
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] -= ba * __log2f(1.0f + bb * (dist - (float)e));
    }
}

// four consecutive outputs of a head and, with a gate, times the sigmoids of the four gate values beside them:
// one 8-byte store
__device__ __forceinline__ void ag_store4(bf16* op, const bf16* gp, float x0, float x1, float x2, float x3) {
    if (gp) {
        const uint2 gw = *reinterpret_cast<const uint2*>(gp);
        x0 /= 1.0f + __expf(-bf16lo_to_f32(gw.x)); x1 /= 1.0f + __expf(-bf16hi_to_f32(gw.x));
        x2 /= 1.0f + __expf(-bf16lo_to_f32(gw.y)); x3 /= 1.0f + __expf(-bf16hi_to_f32(gw.y));
    }
    const bf16 o0 = __float2bfloat16(x0), o1 = __float2bfloat16(x1), o2 = __float2bfloat16(x2), o3 = __float2bfloat16(x3);
    uint2 w;
    w.x = (uint32_t)__builtin_bit_cast(unsigned short, o0) | ((uint32_t)__builtin_bit_cast(unsigned short, o1) << 16);
    w.y = (uint32_t)__builtin_bit_cast(unsigned short, o2) | ((uint32_t)__builtin_bit_cast(unsigned short, o3) << 16);
    *reinterpret_cast<uint2*>(op) = w;
}

// A workgroup is 4, 2 or 1 heads of one kv head (a wave each); they stage a block of keys and values through shared memory, the
// loads of a block under way while the one before is worked on.  What bounds it: first the address unit of the loads (an operand
// straight from the pages is sixteen rows in each sixteen lanes, 64 cycles an instruction instead of 16: a block took 4 x 16 x 64
// cycles a workgroup, whatever ran beside it), now the instructions of a wave's softmax, so a block that is seen whole is not masked,
// sums are rescaled only when a maximum has moved, and two waves a SIMD are asked for where the registers reach, which keeps the sums
// out of the accumulation registers (the vector unit has to copy them).  Workgroups that follow each other are heads of one tile: since
// they go to the XCDs in turn, the tiles of a head (whose keys and values are the same) meet in few of the eight L2s, where tile
// after tile of a head is read by every one of them (16 prompts of 100 tokens, 16 heads on 16: 25 us tile by tile, 13.3 now).  us at
// 2,048 tokens, 16 heads 128 wide with 4 kv heads 228 -> 64, with 16 of them 228 -> 85; 64 wide, 32 heads on 8: 227 -> 55; 16 tokens
// behind 4,000: 219 -> 107.
template <int DC, int DT, int WAVES>     // hs = 32 DC, vd = 16 DT, heads of a workgroup
__global__ __launch_bounds__(WAVES * BN_WAVE, DC + DT <= (WAVES > 1 ? 16 : 14) ? 2 : 1) void attn_general_prompt_kernel(GenArgs a) {
    constexpr int HS = 32 * DC, VD = 16 * DT, THREADS = WAVES * BN_WAVE;
    constexpr int KEYS = 128 * DC, VALUES = 64 * DT;                     // 16-byte pieces of a block of 32 keys, and of its values
    constexpr int KN = (KEYS + THREADS - 1) / THREADS, VN = (VALUES + THREADS - 1) / THREADS;       // a thread's share of them
    constexpr int BUFFERS = WAVES > 1 ? 2 : 1;
    __shared__ __align__(16) u32x4 staged[BUFFERS][KEYS + VALUES];
    const int* tl = a.tiles + 4 * blockIdx.y;
    const int seq = tl[0], row0 = tl[1], n = min(tl[2], 16), pos0 = tl[3];
    const int head = blockIdx.x * WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (n <= 0 || pos0 < 0) return;                      // the whole workgroup
    const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
    const int kvh = head / (a.H / a.Hkv);
    const bool col_ok = i < n;                           // this lane's query column exists
    const int qpos = pos0 + i;
    const int k_hi = pos0 + n;                           // keys of this tile: positions below this

    // Q^T: column i, dimensions 32 c + 8 g .. + 7 (a row that does not exist reads the tile's last one and is never stored)
    bf16x8 qf[DC];
    {
        const bf16* qp = a.q + (size_t)(row0 + min(i, n - 1)) * a.q_stride + (size_t)head * HS + 8 * g;
#pragma unroll
        for (int c = 0; c < DC; ++c) qf[c] = ag_ld16(qp + 32 * c);
    }
    const float scale2 = a.scale * AG_LOG2E;
    const int bias = a.dist_a ? (a.dist_b ? 1 : 2) : 0;
    const float ba = bias ? a.dist_a[head] * (bias == 2 ? AG_LOG2E : 1.0f) : 0.f, bb = bias == 1 ? a.dist_b[head] : 0.f;
    f32x4 acc[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    const bf16x8 ones = __builtin_bit_cast(bf16x8, make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u));

    // A block's pieces as they lie in the pages (the keys one run, of the values 64 bytes a dimension), and where a piece goes:
    // piece 64 (2 c + tile) + 16 g + (i ^ (4 g + c % 4)) is dimensions 32 c + 8 g .. + 7 of row i of key tile `tile`, piece
    // KEYS + 64 t + 16 g + (i ^ 4 g) keys 8 g .. 8 g + 7 of value column 16 t + i.  A wave then reads an operand as 1 KB in a row, and
    // the exclusive or keeps the pieces that a row's threads write in different banks.
    const int* pages = a.block_table + (size_t)seq * a.bt_stride;
    u32x4 kr[KN], vr[VN];
    auto ask = [&](int kb, int page) {
        const size_t at = (size_t)page * a.Hkv + kvh;
        const u32x4* kp = reinterpret_cast<const u32x4*>(a.k_pages + (at * BN_PAGE + kb % BN_PAGE) * HS);
        const bf16* vp = a.v_pages + at * VD * BN_PAGE + kb % BN_PAGE;
#pragma unroll
        for (int u = 0; u < KN; ++u) {
            const int piece = u * THREADS + threadIdx.x;
            if (KEYS % THREADS == 0 || piece < KEYS) kr[u] = kp[piece];
        }
#pragma unroll
        for (int u = 0; u < VN; ++u) {
            const int piece = u * THREADS + threadIdx.x;
            if (VALUES % THREADS == 0 || piece < VALUES) vr[u] = *reinterpret_cast<const u32x4*>(vp + (piece >> 2) * BN_PAGE + 8 * (piece & 3));
        }
    };
    auto put = [&](u32x4* to) {
#pragma unroll
        for (int u = 0; u < KN; ++u) {
            const int piece = u * THREADS + threadIdx.x, r = piece / (4 * DC), q = piece % (4 * DC);
            const int pi = (r >> 3) << 2 | (r & 3), pg = q & 3, pc = q >> 2;
            if (KEYS % THREADS == 0 || piece < KEYS) to[64 * (2 * pc + (r >> 2 & 1)) + 16 * pg + (pi ^ (4 * pg + (pc & 3)))] = kr[u];
        }
#pragma unroll
        for (int u = 0; u < VN; ++u) {
            const int piece = u * THREADS + threadIdx.x, pi = piece >> 2 & 15, pg = piece & 3;
            if (VALUES % THREADS == 0 || piece < VALUES) to[KEYS + 64 * (piece >> 6) + 16 * pg + (pi ^ (4 * pg))] = vr[u];
        }
    };
    const int k_lo = a.window > 0 ? max(0, pos0 - a.window + 1) & ~31 : 0;      // the block of the first key any row sees
    const int q_lo = a.window > 0 ? qpos - a.window : -1;                        // keys at or below this are out of sight
    const int width = a.window > 0 ? a.window : pos0 + 32;                       // (no window: every block is above its edge)
    const int keep = a.window > 0 ? min(a.keep_first, k_hi) : 0;                 // keys below this stay in sight
    auto leap = [&](int kb) { return kb >= keep && kb < k_lo ? k_lo : kb; };     // past what no row of the tile sees
    const int last_block = ((k_hi - 1) / 32) * 32;       // asked for again behind the end: a load without a branch around it
    int kb = leap(0), next = leap(kb + 32), buffer = 0;
    int page = pages[min(next, last_block) / BN_PAGE];   // the page of the block that is asked for next: itself asked for a block before
    ask(kb, pages[kb / BN_PAGE]);
    put(staged[0]);
    ask(min(next, last_block), page);
    page = pages[min(leap(next + 32), last_block) / BN_PAGE];
    __syncthreads();
    for (; kb < k_hi; kb = next, next = leap(next + 32)) {
        const u32x4* block = staged[buffer];
        if (BUFFERS == 2) {                              // the other buffer was read before the barrier behind the last block
            buffer ^= 1;
            put(staged[buffer]);
            ask(min(leap(next + 32), last_block), page);
            page = pages[min(leap(leap(next + 32) + 32), last_block) / BN_PAGE];
        }
        f32x4 st0 = (f32x4){0.f, 0.f, 0.f, 0.f}, st1 = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            const u32x4* kt = block + 128 * c + 16 * g + (i ^ (4 * g + (c & 3)));
            st0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kt[0]), qf[c], st0, 0, 0, 0);
            st1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kt[64]), qf[c], st1, 0, 0, 0);
        }
        // this lane's eight scores: keys kb + 8 g + e, e = 4 h + r
        float s[8];
        ag_scores(s, st0, st1, scale2, bias, ba, bb, qpos, kb + 8 * g);
        // a block that every row sees whole is not masked (a column without a query is never stored)
        float mx = -INFINITY;
        if (kb + 31 <= pos0 && (kb + 31 < keep || kb > pos0 + n - 1 - width)) {
#pragma unroll
            for (int e = 0; e < 8; ++e) mx = fmaxf(mx, s[e]);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int key = kb + 8 * g + e;
                float v = s[e];
                if (!col_ok || key > qpos || key >= k_hi || (key <= q_lo && key >= keep)) v = -INFINITY;
                s[e] = v;
                mx = fmaxf(mx, v);
            }
        }
        mx = ag_max_over_groups(mx);
        const float m_new = fmaxf(m, mx);
        float alpha = 1.f;
        if (m_new == -INFINITY) {
#pragma unroll
            for (int e = 0; e < 8; ++e) s[e] = 0.f;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) s[e] = __builtin_amdgcn_exp2f(s[e] - m_new);
            alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - m_new);
        }
        const bool rescale = __any(alpha != 1.f);        // a factor of 1 for every column changes nothing
        m = m_new;
        const f32x8 pv = {s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7]};
        const bf16x8 pb = __builtin_convertvector(pv, bf16x8);
        const f32x4 lsum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb, (f32x4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        l = fmaf(l, alpha, lsum[0]);
        bf16x8 va[DT];
#pragma unroll
        for (int t = 0; t < DT; ++t) va[t] = __builtin_bit_cast(bf16x8, block[KEYS + 64 * t + 16 * g + (i ^ (4 * g))]);
        // keys past the tile's last position may hold anything in V^T (0 * NaN is NaN): cleared
        if (kb + 32 > k_hi) {
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                uint4 w = __builtin_bit_cast(uint4, va[t]);
                const int first = kb + 8 * g;
                if (first + 0 >= k_hi) w.x &= 0xffff0000u;
                if (first + 1 >= k_hi) w.x &= 0x0000ffffu;
                if (first + 2 >= k_hi) w.y &= 0xffff0000u;
                if (first + 3 >= k_hi) w.y &= 0x0000ffffu;
                if (first + 4 >= k_hi) w.z &= 0xffff0000u;
                if (first + 5 >= k_hi) w.z &= 0x0000ffffu;
                if (first + 6 >= k_hi) w.w &= 0xffff0000u;
                if (first + 7 >= k_hi) w.w &= 0x0000ffffu;
                va[t] = __builtin_bit_cast(bf16x8, w);
            }
        }
        if (rescale) {
#pragma unroll
            for (int t = 0; t < DT; ++t) acc[t] *= alpha;
        }
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[t], pb, acc[t], 0, 0, 0);
        }
        __syncthreads();
        if (BUFFERS == 1) {
            put(staged[0]);
            ask(min(leap(next + 32), last_block), page);
            page = pages[min(leap(leap(next + 32) + 32), last_block) / BN_PAGE];
            __syncthreads();
        }
    }
    // the sink: a term 2^(sv - m') with no value, m' = max(m, sv)
    float fa = 1.f;
    if (a.sink) {
        const float sv = a.sink_values ? a.sink_values[head] * AG_LOG2E : 0.f;       // the sink's score in the exponent's base 2
        const float m2 = fmaxf(m, sv);
        fa = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - m2);
        l = fmaf(l, fa, __builtin_amdgcn_exp2f(sv - m2));
    }
    const float inv = l > 0.f ? fa / l : 0.f;
    if (!col_ok) return;
    // acc[t][r] = O^T[value column 16 t + 4 g + r][query i]: four consecutive columns, one 8-byte store
    bf16* op = a.out + (size_t)(row0 + i) * a.out_stride + (size_t)head * VD + 4 * g;
    const bf16* gp = a.gate ? a.gate + (size_t)(row0 + i) * a.gate_stride + (size_t)head * VD + 4 * g : nullptr;
#pragma unroll
    for (int t = 0; t < DT; ++t)
        ag_store4(op + 16 * t, gp ? gp + 16 * t : nullptr, acc[t][0] * inv, acc[t][1] * inv, acc[t][2] * inv, acc[t][3] * inv);
}

struct GenDecodeArgs {
    const bf16* q;            // [n_seqs, q_stride]: head h at h * hs, row b is sequence b's new token
    bf16* out;                // [n_seqs, out_stride]
    const bf16* k_pages;
    const bf16* v_pages;
    const int* block_table;   // [n_seqs, bt_stride]
    const int* seq_lens;      // [n_seqs] keys in the cache, the new one included; 0: a padding row
    const float* dist_a;
    const float* dist_b;      // null: the bias is linear
    const bf16* gate;         // [n_seqs, gate_stride] or null
    int gate_stride;
    float* part_o;            // [n_seqs H, n_splits, vd]   (n_splits > 1)
    float* part_ml;           // [n_seqs H, n_splits, 2]: maximum (natural exponent) and sum of the weights
    const int* max_len;       // != null: the longest sequence's key count; the keys per split follow from it
    int q_stride, out_stride, bt_stride, H, Hkv, n_splits, chunk, window, keep_first, sink;
    const float* sink_values; // [H] float32, or null (score 0)
    float scale;
    // (NEW: the row of q holds projections, its keys at q + H hs)
    bf16* k_new;              // the pages again, to be written
    bf16* v_new;
    const float* wq;          // [hs] norms of every query and key head; null: none
    const float* wk;
    const float* inv_freq;    // [rope_dims / 2] rotation in split-half pairs; null: none
    int rope_dims, temp_every;
    int min_pages;            // of a run whose length follows max_len
    int v_col;                // the first value's column of the row: behind the keys, or the keys as projected
    float eps, temp_coef;
};

// Keys and values that one wave reads each are read non-temporally (ONCE) while a launch's tables hold no more than this many MB of
// them: a load takes half a line, of a key the next load the other half and of a value the next block's, and what the L2
// does not hold in between is fetched twice.  us over memory that no cache holds, plain / non-temporal: one sequence of 2,000 at 16
// heads over 4 (4 MB) 10.8 / 10.3, four of 2,000 (16 MB) 11.6 / 11.3, 16 of 300 over 8 (20 MB) 13.7 / 13.7, 16 of 1,000 over 4 (33 MB)
// 14.4 / 14.6, 16 of 2,000 (66 MB) 21.1 / 22.6, 16 of 1,000 over 16 (131 MB) 33.8 / 38.4; of 300 keys alone 11.3 / 11.6.  Where
// several waves read them: 64 heads over one, one of 500 10.3 / 11.1, 16 of 2,000 20.9 / 21.7.  (Both loops in one kernel, chosen by
// the length on the device: 0.4 us slower than either.)
#define AG_ONCE_MB 24

// Runs of one page, while a launch leaves no more than this many rows of partial sums (sequences x heads x splits) to merge; else of
// BN_SPLIT_MIN_PAGES.  A wave walks its run block by block and waits for the values of each, so that a page more is 1.5 us more; against
// that stands what the merge reads.  us, runs of two pages and more -> this, keys in front: 16 heads of 128 over 4, one sequence 130 7.4 -> 6.3,
// 300 9.9 -> 6.8, 1,000 9.2 -> 7.6, 2,000 9.8 -> 8.5, four of 300 11.1 -> 7.4, of 800 11.8 -> 8.0, of 1,500 10.5 -> 10.5, 16 of 300 11.8 -> 9.6,
// of 1,000 (4,096 rows) 13.8 -> 14.1, 64 of 200 (4,096) 13.8 -> 13.0; 64 heads over one, 16 of 300 (5,120) 11.2 -> 9.4, four of 1,500 (6,144)
// 9.9 -> 10.4, 16 of 1,000 (16,384) 12.8 -> 15.2, 64 of 200 (16,384) 12.9 -> 14.5; 16 of 256 over 2, four of 800 17.5 -> 10.2. A latent cache, 16 heads over
// one row of 192 with 128 values: one of 300 10.3 -> 6.9, of 2,000 9.6 -> 8.6, 16 of 1,000 (4,096) 11.4 -> 9.6, of 2,000 (8,192) 12.6 -> 13.8.  Inside the
// line up to 5 % is lost where 512 workgroups of two pages become 1,024 (eight of 2,000, 16 over 4, 13.9 -> 14.6) and up to 12 % gained
// (16 of 64 over 16, four of 1,000, 10.9 -> 10.1).  Results differ in rounding: a run's probabilities and sums are taken from its own maximum.  (Logits
// of Sunusun and Fazopel at 2,048 columns over three draws, from 64 bits: 3.70e-3 -> 3.71e-3, 4.54e-3 -> 4.54e-3.)
#define AG_PAGE_RUN_ROWS 6000

// NEW: the new token's row is still as projected.  Every wave norms, rotates and scales its queries, and the waves of the run that holds
// the new position its key, in the registers in which they are multiplied (rotations turn pairs a whole number of 32 dimensions apart, so
// a lane holds both); these put key and value in the place of what their block's loads found there, and one of them writes the pages.
// The arithmetic is qk_norm_store_kernel's but for the order of a norm's sum.  us, that kernel and this without NEW -> this alone (norms,
// 64 rotated dimensions), one sequence of 300 / four of 2,000 / 64 of 2,000 keys: 16 heads of 128 over 4 13.4 -> 11.1, 16.6 -> 14.1, 54.6 ->
// 49.9; 64 of 128 over one 13.7 -> 11.2, 16.3 -> 13.8, 48.0 -> 40.9; 16 of 256 over 2 16.8 -> 13.6, 22.5 -> 18.3, 70.6 -> 63.9; 16 of 64 over 16
// 11.8 -> 9.4, 18.5 -> 15.1, 126 -> 119: faster everywhere.  Bound by latency: everything that waits for no length is asked for in front of
// the length itself, and the pages are written behind the loop (asked for inside branches and written in front of it 2 us more).
template <int DC, int DT, bool ONCE, bool NEW>     // hs = 32 DC, vd = 16 DT
__global__ __launch_bounds__(BN_WAVE) void attn_general_decode_kernel(GenDecodeArgs a) {
    constexpr int HS = 32 * DC, VD = 16 * DT;
    const int seq = blockIdx.x, split = blockIdx.z;
    const int G = a.H / a.Hkv, head_tiles = (G + 15) / 16;
    const int kvh = blockIdx.y / head_tiles, ht = blockIdx.y - kvh * head_tiles;
    const int lane = threadIdx.x, i = lane & 15, g = lane >> 4;
    const bool col_ok = 16 * ht + i < G;                 // this lane's column is a head that exists
    const int head = kvh * G + min(16 * ht + i, G - 1);
    bf16x8 qf[DC], key[DC];                              // (NEW) the new token's key, and its value's column 16 t + i
    bf16 value[DT];
    constexpr int HC = DC / 2 > 0 ? DC / 2 : 1;
    float4 nq[2 * DC], nk[2 * DC], turn[2 * HC];
    const int hc = NEW && a.inv_freq ? a.rope_dims / 64 : 0;            // chunks of 32 between the two of a pair
    if constexpr (NEW) {                                 // all that no length is needed for, before the loads that follow from one another
        const bf16* row = a.q + (size_t)seq * a.q_stride + 8 * g;
        const bf16* vp = a.q + (size_t)seq * a.q_stride + a.v_col + (size_t)kvh * VD + i;
#pragma unroll
        for (int c = 0; c < DC; ++c) { qf[c] = ag_ld16(row + (size_t)head * HS + 32 * c); key[c] = ag_ld16(row + (size_t)(a.H + kvh) * HS + 32 * c); }
#pragma unroll
        for (int t = 0; t < DT; ++t) value[t] = vp[16 * t];
        const float4 one = make_float4(1.f, 1.f, 1.f, 1.f);
#pragma unroll
        for (int c = 0; c < 2 * DC; ++c) { nq[c] = one; nk[c] = one; }
        if (a.wq) {
#pragma unroll
            for (int c = 0; c < 2 * DC; ++c) {
                nq[c] = *reinterpret_cast<const float4*>(a.wq + 32 * (c >> 1) + 8 * g + 4 * (c & 1));
                nk[c] = *reinterpret_cast<const float4*>(a.wk + 32 * (c >> 1) + 8 * g + 4 * (c & 1));
            }
        }
#pragma unroll
        for (int c = 0; c < 2 * HC; ++c)
            if (c < 2 * hc) turn[c] = *reinterpret_cast<const float4*>(a.inv_freq + 32 * (c >> 1) + 8 * g + 4 * (c & 1));
    }
    const int len = a.seq_lens[seq], qpos = len - 1;
    int k_lo = 0, k_hi = 0, keep = 0;                    // this wave's keys: k_lo .. k_hi - 1, and 0 .. keep - 1
    if (len > 0) {
        const int lo = a.window > 0 ? max(0, len - a.window) : 0;
        if (split == 0 && a.window > 0) keep = min(a.keep_first, lo);
        if (a.n_splits > 1) {
            const int chunk = a.max_len ? bn_split_chunk(*a.max_len, a.n_splits, a.min_pages) : a.chunk;
            const int base = a.window > 0 ? (lo / BN_PAGE) * BN_PAGE : 0;
            k_lo = max(lo, base + split * chunk);
            k_hi = min(len, base + (split + 1) * chunk);
        } else {
            k_lo = lo; k_hi = len;
        }
    }
    const size_t prow = ((size_t)seq * a.H + head) * a.n_splits + split;
    if (k_lo >= k_hi) {                                  // no key for this split (or a padding row): zeros and no weight
        if (!col_ok) return;
        if (a.n_splits > 1) {
#pragma unroll
            for (int t = 0; t < DT; ++t)
                *reinterpret_cast<float4*>(a.part_o + prow * VD + 16 * t + 4 * g) = make_float4(0.f, 0.f, 0.f, 0.f);
            if (g == 0) { a.part_ml[2 * prow] = -INFINITY; a.part_ml[2 * prow + 1] = 0.f; }
        } else {
            bf16* op = a.out + (size_t)seq * a.out_stride + (size_t)head * VD + 4 * g;
#pragma unroll
            for (int t = 0; t < DT; ++t) *reinterpret_cast<uint2*>(op + 16 * t) = make_uint2(0u, 0u);
        }
        return;
    }
    if constexpr (!NEW) {
        const bf16* qp = a.q + (size_t)seq * a.q_stride + (size_t)head * HS + 8 * g;
#pragma unroll
        for (int c = 0; c < DC; ++c) qf[c] = ag_ld16(qp + 32 * c);
    }
    const float scale2 = a.scale * AG_LOG2E;
    const int bias = a.dist_a ? (a.dist_b ? 1 : 2) : 0;
    const float ba = bias ? a.dist_a[head] * (bias == 2 ? AG_LOG2E : 1.0f) : 0.f, bb = bias == 1 ? a.dist_b[head] : 0.f;
    f32x4 acc[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    const bf16x8 ones = __builtin_bit_cast(bf16x8, make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u));
    const int krow = 8 * (i >> 2) + (i & 3);
    bf16x8 kn0[DC], kn1[DC];
    auto ask_keys = [&](int kb) {
        const int page = a.block_table[(size_t)seq * a.bt_stride + kb / BN_PAGE];
        const bf16* kbase = a.k_pages + (((size_t)page * a.Hkv + kvh) * BN_PAGE + kb % BN_PAGE + krow) * HS + 8 * g;
#pragma unroll
        for (int c = 0; c < DC; ++c) { kn0[c] = ag_ld16_cached<ONCE>(kbase + 32 * c); kn1[c] = ag_ld16_cached<ONCE>(kbase + 4 * HS + 32 * c); }
    };
    const int first_block = k_lo & ~31, last_block = ((k_hi - 1) / 32) * 32;
    auto leap = [&](int kb) { return kb >= keep && kb < first_block ? first_block : kb; };
    ask_keys(leap(0));
    const int new_block = NEW && k_hi == len ? last_block : -1;
    if constexpr (NEW) {
        float sn[HC][8], cs[HC][8];
#pragma unroll
        for (int c = 0; c < HC; ++c)
            if (c < hc) {
#pragma unroll
                for (int e = 0; e < 8; ++e) bn_sincos((float)qpos * reinterpret_cast<const float*>(&turn[2 * c + (e >> 2)])[e & 3], &sn[c][e], &cs[c][e]);
            }
        auto shape = [&](bf16x8(&f)[DC], const float4(&w)[2 * DC], float factor) {
            float x[DC][8], ss = 0.f;
#pragma unroll
            for (int c = 0; c < DC; ++c)
#pragma unroll
                for (int e = 0; e < 8; ++e) { x[c][e] = (float)f[c][e]; ss = fmaf(x[c][e], x[c][e], ss); }
            if (a.wq) {
                const auto sum = [](float u, float v) { return u + v; };
                ss = bn_pair_far<32>(bn_pair_far<16>(ss, sum), sum);
                const float r = 1.0f / sqrtf(ss / (float)HS + a.eps);
#pragma unroll
                for (int c = 0; c < DC; ++c)
#pragma unroll
                    for (int e = 0; e < 8; ++e) x[c][e] = x[c][e] * r * reinterpret_cast<const float*>(&w[2 * c + (e >> 2)])[e & 3];
            }
#pragma unroll
            for (int h = 1; h <= DC / 2; ++h)
                if (h == hc) {
#pragma unroll
                    for (int c = 0; c < h; ++c)
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            const float u = x[c][e], v = x[c + h][e];
                            x[c][e] = u * cs[c][e] - v * sn[c][e];
                            x[c + h][e] = v * cs[c][e] + u * sn[c][e];
                        }
                }
#pragma unroll
            for (int c = 0; c < DC; ++c) {
                const f32x8 y = {x[c][0] * factor, x[c][1] * factor, x[c][2] * factor, x[c][3] * factor,
                                 x[c][4] * factor, x[c][5] * factor, x[c][6] * factor, x[c][7] * factor};
                f[c] = __builtin_convertvector(y, bf16x8);
            }
        };
        shape(qf, nq, a.temp_every > 0 ? 1.0f + a.temp_coef * logf((float)(len / a.temp_every) + 1.0f) : 1.0f);
        if (new_block >= 0) shape(key, nk, 1.0f);
    }
    for (int kb = leap(0); kb < k_hi; kb = leap(kb + 32)) {
        const int page = a.block_table[(size_t)seq * a.bt_stride + kb / BN_PAGE];
        const bf16* vbase = a.v_pages + (((size_t)page * a.Hkv + kvh) * VD + i) * BN_PAGE + kb % BN_PAGE + 8 * g;
        bf16x8 k0[DC], k1[DC];
#pragma unroll
        for (int c = 0; c < DC; ++c) { k0[c] = kn0[c]; k1[c] = kn1[c]; }
        if (NEW && kb == new_block) {
            const int at = qpos - kb;
#pragma unroll
            for (int c = 0; c < DC; ++c) {
                if (krow == at) k0[c] = key[c];
                if (krow + 4 == at) k1[c] = key[c];
            }
        }
        ask_keys(min(leap(kb + 32), last_block));
        f32x4 st0 = (f32x4){0.f, 0.f, 0.f, 0.f}, st1 = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            st0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0[c], qf[c], st0, 0, 0, 0);
            st1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1[c], qf[c], st1, 0, 0, 0);
        }
        bf16x8 va[DT];
#pragma unroll
        for (int t = 0; t < DT; ++t) va[t] = ag_ld16_cached<ONCE>(vbase + (size_t)t * 16 * BN_PAGE);
        float s[8];
        ag_scores(s, st0, st1, scale2, bias, ba, bb, qpos, kb + 8 * g);
        float mx = -INFINITY;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int key = kb + 8 * g + e;
            float v = s[e];
            if (!col_ok || (key < k_lo && key >= keep) || key >= k_hi) v = -INFINITY;
            s[e] = v;
            mx = fmaxf(mx, v);
        }
        const auto larger = [](float x, float y) { return fmaxf(x, y); };
        mx = bn_pair_far<32>(bn_pair_far<16>(mx, larger), larger);
        const float m_new = fmaxf(m, mx);
        float alpha = 1.f;
        if (m_new == -INFINITY) {
#pragma unroll
            for (int e = 0; e < 8; ++e) s[e] = 0.f;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) s[e] = __builtin_amdgcn_exp2f(s[e] - m_new);
            alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - m_new);
        }
        m = m_new;
        const f32x8 pv = {s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7]};
        const bf16x8 pb = __builtin_convertvector(pv, bf16x8);
        const f32x4 lsum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb, (f32x4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        l = fmaf(l, alpha, lsum[0]);
        if (NEW && kb == new_block) {
            const int at = qpos - kb - 8 * g;
#pragma unroll
            for (int t = 0; t < DT; ++t)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (e == at) va[t][e] = __builtin_bit_cast(__bf16, value[t]);
        }
        // positions past the sequence's end may hold anything in V^T (0 * NaN is NaN): cleared
        if (kb + 32 > k_hi) {
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                uint4 w = __builtin_bit_cast(uint4, va[t]);
                const int first = kb + 8 * g;
                if (first + 0 >= k_hi) w.x &= 0xffff0000u;
                if (first + 1 >= k_hi) w.x &= 0x0000ffffu;
                if (first + 2 >= k_hi) w.y &= 0xffff0000u;
                if (first + 3 >= k_hi) w.y &= 0x0000ffffu;
                if (first + 4 >= k_hi) w.z &= 0xffff0000u;
                if (first + 5 >= k_hi) w.z &= 0x0000ffffu;
                if (first + 6 >= k_hi) w.w &= 0xffff0000u;
                if (first + 7 >= k_hi) w.w &= 0x0000ffffu;
                va[t] = __builtin_bit_cast(bf16x8, w);
            }
        }
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            acc[t] *= alpha;
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[t], pb, acc[t], 0, 0, 0);
        }
    }
    if (NEW && new_block >= 0 && ht == 0) {              // (behind the loop: a load would wait for the stores in front of it)
        const int page = a.block_table[(size_t)seq * a.bt_stride + qpos / BN_PAGE];
        if (i == 0) {
            bf16* dst = a.k_new + (((size_t)page * a.Hkv + kvh) * BN_PAGE + qpos % BN_PAGE) * HS + 8 * g;
#pragma unroll
            for (int c = 0; c < DC; ++c) *reinterpret_cast<bf16x8*>(dst + 32 * c) = key[c];
        }
        if (g == 0) {
            bf16* dst = a.v_new + (((size_t)page * a.Hkv + kvh) * VD + i) * BN_PAGE + qpos % BN_PAGE;
#pragma unroll
            for (int t = 0; t < DT; ++t) dst[(size_t)t * 16 * BN_PAGE] = value[t];
        }
    }
    if (!col_ok) return;
    if (a.n_splits > 1) {                                // sums relative to the maximum m (base 2), for the merge
#pragma unroll
        for (int t = 0; t < DT; ++t)
            *reinterpret_cast<float4*>(a.part_o + prow * VD + 16 * t + 4 * g) = make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]);
        if (g == 0) { a.part_ml[2 * prow] = m * 0.6931471805599453f; a.part_ml[2 * prow + 1] = l; }
        return;
    }
    float fa = 1.f;
    if (a.sink) {
        const float sv = a.sink_values ? a.sink_values[head] * AG_LOG2E : 0.f;       // the sink's score in the exponent's base 2
        const float m2 = fmaxf(m, sv);
        fa = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - m2);
        l = fmaf(l, fa, __builtin_amdgcn_exp2f(sv - m2));
    }
    const float inv = l > 0.f ? fa / l : 0.f;
    bf16* op = a.out + (size_t)seq * a.out_stride + (size_t)head * VD + 4 * g;
    const bf16* gp = a.gate ? a.gate + (size_t)seq * a.gate_stride + (size_t)head * VD + 4 * g : nullptr;
#pragma unroll
    for (int t = 0; t < DT; ++t)
        ag_store4(op + 16 * t, gp ? gp + 16 * t : nullptr, acc[t][0] * inv, acc[t][1] * inv, acc[t][2] * inv, acc[t][3] * inv);
}

// out[row, d] = sum_s e^(m_s - m) o_s[d] / (sum_s e^(m_s - m) l_s [+ e^(-m) for the sink]) [sigmoid(gate)], the splits in index order;
// one wave a (token, head) row: the splits' factors are formed a lane a split, and a lane takes V value columns.  Bound by its
// chain of waits: all S >= n_splits sums (those past n_splits lie past the buffer's end: zeros, and no trip to memory) and the gate are asked
// for beside the factors' maxima, and a factor comes out of its lane with a v_readlane.  A split without keys holds zeros, and its factor is 0.
// us inside a step, a loop over the splits -> this, 64 rows of 7 splits of 128 columns 5.4 -> 4.7; with the attention in front of it, 16 heads of
// 256 over 2, one sequence of 33 / 49 / 56 / 64 splits 14.5 / 15.5 / 15.2 / 16.3 -> 13.0 / 13.8 / 14.1 / 14.4; past the end the last
// split's sums again, that is 15 more trips of a row of 33 splits: 14.9 / 16.2 / 16.4 / 16.9.
#define AG_MAX_SPLITS BN_WAVE
template <int S, int V>
__global__ __launch_bounds__(BN_WAVE) void attn_general_combine_kernel(bf16* __restrict__ out, int out_stride,
                                                                       const float* __restrict__ part_o,
                                                                       const float* __restrict__ part_ml, int H, int vd,
                                                                       int n_splits, int sink,
                                                                       const float* __restrict__ sink_values,
                                                                       const bf16* __restrict__ gate, int gate_stride) {
    typedef __attribute__((ext_vector_type(V))) float Floats;
    typedef __attribute__((ext_vector_type(V))) __bf16 Bf16s;
    const int row = blockIdx.x, tok = row / H, head = row - tok * H, lane = threadIdx.x;
    const int mine_at = min(lane, n_splits - 1), d = min(V * lane, vd - V);              // vd <= 64 V: V columns a lane
    const float* ml = part_ml + ((size_t)row * n_splits + mine_at) * 2;
    const float own_m = ml[0], own_l = ml[1];
    const auto sums = bn_buffer(part_o + (size_t)row * n_splits * vd, n_splits * vd * 4);
    Floats o[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if constexpr (V == 4) o[s] = __builtin_bit_cast(Floats, __builtin_amdgcn_raw_buffer_load_b128(sums, d * 4, s * vd * 4, 0));
        else if constexpr (V == 2) o[s] = __builtin_bit_cast(Floats, __builtin_amdgcn_raw_buffer_load_b64(sums, d * 4, s * vd * 4, 0));
        else o[s] = __builtin_bit_cast(Floats, __builtin_amdgcn_raw_buffer_load_b32(sums, d * 4, s * vd * 4, 0));
    }
    Bf16s gates = {};
    if (gate) gates = *reinterpret_cast<const Bf16s*>(gate + (size_t)tok * gate_stride + (size_t)head * vd + d);
    const float sv = sink && sink_values ? sink_values[head] : 0.f;
    __builtin_amdgcn_sched_barrier(0);                   // all asked for before anything is waited for
    const float mine = lane < n_splits ? own_m : -INFINITY, sum = lane < n_splits ? own_l : 0.f;
    const float m = wave_max(sink ? fmaxf(sv, mine) : mine);
    const float f = m != -INFINITY ? expf(mine - m) : 0.f, share = f * sum;
    auto of = [](float x, int s) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), s)); };
    float den = sink ? expf(sv - m) : 0.f, num[V] = {};
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const float w = of(f, s);                        // 0 past n_splits, and so is the share
        den += of(share, s);
#pragma unroll
        for (int u = 0; u < V; ++u) num[u] = fmaf(w, o[s][u], num[u]);
    }
    if (V * lane >= vd) return;
    const float inv = den > 0.f ? 1.0f / den : 0.f;
    Bf16s r;
#pragma unroll
    for (int u = 0; u < V; ++u) {
        float x = num[u] * inv;
        if (gate) x /= 1.0f + __expf(-(float)gates[u]);
        r[u] = __builtin_bit_cast(__bf16, __float2bfloat16(x));
    }
    *reinterpret_cast<Bf16s*>(out + (size_t)tok * out_stride + (size_t)head * vd + d) = r;
}

static bool ag_size(int x) { return x == 32 || x == 64 || x == 96 || x == 128 || x == 192 || x == 256; }

// 1 if the kernels take these head sizes (keys 32, 64, 96, 128, 160, 192 or 256 wide, values from the same list without 160;
// keys 160 or 192 wide are a latent beside a rotated part: values at least 64 wide)
extern "C" int bn_attn_general_supports(int hs, int vd) {
    if (hs == 160 || hs == 192) return ag_size(vd) && vd >= 64 && vd <= hs ? 1 : 0;
    return ag_size(hs) && ag_size(vd) ? 1 : 0;
}

// Heads of a workgroup: as many as share a kv head, up to four, since they share the staged block: 2,048 tokens, 16 heads on 4 take
// 74 us with four, 83 with two, 109 with one (tile by tile).
static int ag_waves(int group) { return group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1; }

template <int DC>
static int ag_launch_dt(const GenArgs& a, int vd, int n_tiles, hipStream_t s) {
    const int waves = ag_waves(a.H / a.Hkv);
    const dim3 grid(a.H / waves, n_tiles), block(waves * BN_WAVE);
#define AG_CASE(DT)                                                                                   \
    if (waves == 4) hipLaunchKernelGGL((attn_general_prompt_kernel<DC, DT, 4>), grid, block, 0, s, a);       \
    else if (waves == 2) hipLaunchKernelGGL((attn_general_prompt_kernel<DC, DT, 2>), grid, block, 0, s, a);  \
    else hipLaunchKernelGGL((attn_general_prompt_kernel<DC, DT, 1>), grid, block, 0, s, a);                  \
    return bn_launch_status()
    switch (vd / 16) {
        case 2: AG_CASE(2);
        case 4: AG_CASE(4);
        case 6: AG_CASE(6);
        case 8: AG_CASE(8);
        case 12: AG_CASE(12);
        case 16: AG_CASE(16);
    }
#undef AG_CASE
    return BN_ERR_ARG;
}

static int ag_launch(const GenArgs& a, int hs, int vd, int n_tiles, hipStream_t s) {
    switch (hs / 32) {
        case 1: return ag_launch_dt<1>(a, vd, n_tiles, s);
        case 2: return ag_launch_dt<2>(a, vd, n_tiles, s);
        case 3: return ag_launch_dt<3>(a, vd, n_tiles, s);
        case 4: return ag_launch_dt<4>(a, vd, n_tiles, s);
        case 5: return ag_launch_dt<5>(a, vd, n_tiles, s);
        case 6: return ag_launch_dt<6>(a, vd, n_tiles, s);
        case 8: return ag_launch_dt<8>(a, vd, n_tiles, s);
    }
    return BN_ERR_ARG;
}

extern "C" int bn_attn_general_prompt(const void* q, int q_stride, void* out, int out_stride, const void* k_pages,
                                      const void* v_pages, const int* block_table, int bt_stride, const int* tiles, int n_tiles,
                                      int H, int Hkv, int hs, int vd, float scale, const float* dist_a, const float* dist_b,
                                      int sink, const float* sink_values, int window, int keep_first, const void* gate,
                                      int gate_stride, hipStream_t s) {
    if (n_tiles <= 0 || H <= 0 || Hkv <= 0 || H % Hkv || window < 0 || keep_first < 0 || !bn_attn_general_supports(hs, vd)) return BN_ERR_ARG;
    if (!q || !out || !k_pages || !v_pages || !block_table || !tiles || (dist_b && !dist_a)) return BN_ERR_ARG;
    if (q_stride % 8 || out_stride % 4 || (((uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)v_pages) & 15) || ((uintptr_t)out & 7))
        return BN_ERR_ARG;
    if (gate && (gate_stride % 4 || ((uintptr_t)gate & 7))) return BN_ERR_ARG;
    GenArgs a;
    a.gate = (const bf16*)gate; a.gate_stride = gate_stride; a.keep_first = keep_first;
    a.q = (const bf16*)q; a.out = (bf16*)out; a.k_pages = (const bf16*)k_pages; a.v_pages = (const bf16*)v_pages;
    a.block_table = block_table; a.tiles = tiles; a.dist_a = dist_a; a.dist_b = dist_b;
    a.q_stride = q_stride; a.out_stride = out_stride; a.bt_stride = bt_stride; a.H = H; a.Hkv = Hkv;
    a.scale = scale; a.sink = sink ? 1 : 0; a.sink_values = sink ? sink_values : nullptr; a.window = window;
    for (int first = 0; first < n_tiles; first += 65535) {       // a launch's second dimension
        a.tiles = tiles + 4 * (size_t)first;
        if (int rc = ag_launch(a, hs, vd, n_tiles - first < 65535 ? n_tiles - first : 65535, s)) return rc;
    }
    return 0;
}

template <int DC>
static int ag_launch_decode_dt(const GenDecodeArgs& a, int vd, bool once, dim3 grid, hipStream_t s) {
#define AG_CASE(DT)                                                                                                       \
    if (once && a.k_new) hipLaunchKernelGGL((attn_general_decode_kernel<DC, DT, true, true>), grid, dim3(BN_WAVE), 0, s, a);   \
    else if (once) hipLaunchKernelGGL((attn_general_decode_kernel<DC, DT, true, false>), grid, dim3(BN_WAVE), 0, s, a);        \
    else if (a.k_new) hipLaunchKernelGGL((attn_general_decode_kernel<DC, DT, false, true>), grid, dim3(BN_WAVE), 0, s, a);     \
    else hipLaunchKernelGGL((attn_general_decode_kernel<DC, DT, false, false>), grid, dim3(BN_WAVE), 0, s, a);                 \
    return bn_launch_status()
    switch (vd / 16) {
        case 2: AG_CASE(2);
        case 4: AG_CASE(4);
        case 6: AG_CASE(6);
        case 8: AG_CASE(8);
        case 12: AG_CASE(12);
        case 16: AG_CASE(16);
    }
#undef AG_CASE
    return BN_ERR_ARG;
}

struct AgFresh { int v_from_k; const float* wq; const float* wk; float eps; const float* inv_freq; int rope_dims; float temp_coef; int temp_every; };

// Decode form: row b of q is sequence b's new token (seq_lens[b] keys in the cache, 0 for a padding row, whose output is
// zeros).  n_splits > 1: part_o [n_seqs H n_splits, vd] and part_ml [n_seqs H n_splits, 2] float32 work space; the keys per
// split are `chunk` (a multiple of BN_PAGE), or follow the longest sequence's key count in *max_len.
static int ag_decode(const void* q, int q_stride, void* out, int out_stride, const void* k_pages, const void* v_pages, const int* block_table, int bt_stride,
                     const int* seq_lens, int n_seqs, int H, int Hkv, int hs, int vd, float scale, const float* dist_a, const float* dist_b, int sink,
                     const float* sink_values, int window, int keep_first, const void* gate, int gate_stride, int n_splits, int chunk, float* part_o,
                     float* part_ml, const int* max_len, const AgFresh* fresh, hipStream_t s) {
    if (fresh) {
        const AgFresh& f = *fresh;
        if ((((uintptr_t)f.wq | (uintptr_t)f.wk | (uintptr_t)f.inv_freq) & 15) || q_stride < (H + Hkv) * hs + (f.v_from_k ? 0 : Hkv * vd) ||
            (f.v_from_k && vd != hs) || (f.wq == nullptr) != (f.wk == nullptr) || (f.inv_freq && (f.rope_dims <= 0 || f.rope_dims % 64 || f.rope_dims > hs)))
            return BN_ERR_ARG;
    }
    if (n_seqs <= 0 || H <= 0 || Hkv <= 0 || H % Hkv || window < 0 || keep_first < 0 || n_splits < 1 || !bn_attn_general_supports(hs, vd)) return BN_ERR_ARG;
    if (!q || !out || !k_pages || !v_pages || !block_table || !seq_lens || (dist_b && !dist_a)) return BN_ERR_ARG;
    if (q_stride % 8 || out_stride % 4 || (((uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)v_pages) & 15) || ((uintptr_t)out & 7))
        return BN_ERR_ARG;
    if (n_splits > 1 && (!part_o || !part_ml || ((uintptr_t)part_o & 15) || (!max_len && (chunk <= 0 || chunk % BN_PAGE)))) return BN_ERR_ARG;
    const int head_tiles = (H / Hkv + 15) / 16;
    if ((long long)Hkv * head_tiles > 65535 || n_splits > AG_MAX_SPLITS) return BN_ERR_ARG;
    if (gate && (gate_stride % 4 || ((uintptr_t)gate & 7))) return BN_ERR_ARG;
    GenDecodeArgs a;
    a.gate = (const bf16*)gate; a.gate_stride = gate_stride; a.keep_first = keep_first;
    a.q = (const bf16*)q; a.out = (bf16*)out; a.k_pages = (const bf16*)k_pages; a.v_pages = (const bf16*)v_pages;
    a.block_table = block_table; a.seq_lens = seq_lens; a.dist_a = dist_a; a.dist_b = dist_b; a.part_o = part_o; a.part_ml = part_ml;
    a.max_len = n_splits > 1 ? max_len : nullptr;
    a.min_pages = (long long)n_seqs * H * n_splits <= AG_PAGE_RUN_ROWS ? 1 : BN_SPLIT_MIN_PAGES;
    a.q_stride = q_stride; a.out_stride = out_stride; a.bt_stride = bt_stride; a.H = H; a.Hkv = Hkv; a.n_splits = n_splits;
    a.chunk = chunk; a.window = window; a.sink = sink ? 1 : 0; a.sink_values = sink ? sink_values : nullptr; a.scale = scale;
    const AgFresh f = fresh ? *fresh : AgFresh{};
    a.k_new = fresh ? (bf16*)k_pages : nullptr; a.v_new = fresh ? (bf16*)v_pages : nullptr;
    a.v_col = (f.v_from_k ? H : H + Hkv) * hs;
    a.wq = f.wq; a.wk = f.wk; a.eps = f.eps; a.inv_freq = f.inv_freq; a.rope_dims = f.inv_freq ? f.rope_dims : 0;
    a.temp_coef = f.temp_coef; a.temp_every = f.temp_every;
    const dim3 grid(n_seqs, Hkv * head_tiles, n_splits);
    const long long held = (long long)bt_stride * BN_PAGE, seen = (long long)window + keep_first;     // keys a sequence at the most
    const bool once = head_tiles == 1 && (window > 0 && seen < held ? seen : held) * n_seqs * Hkv * (hs + vd) * 2 <= (long long)AG_ONCE_MB << 20;
    int rc = BN_ERR_ARG;
    switch (hs / 32) {
        case 1: rc = ag_launch_decode_dt<1>(a, vd, once, grid, s); break;
        case 2: rc = ag_launch_decode_dt<2>(a, vd, once, grid, s); break;
        case 3: rc = ag_launch_decode_dt<3>(a, vd, once, grid, s); break;
        case 4: rc = ag_launch_decode_dt<4>(a, vd, once, grid, s); break;
        case 5: rc = ag_launch_decode_dt<5>(a, vd, once, grid, s); break;
        case 6: rc = ag_launch_decode_dt<6>(a, vd, once, grid, s); break;
        case 8: rc = ag_launch_decode_dt<8>(a, vd, once, grid, s); break;
    }
    if (rc != 0 || n_splits == 1) return rc;
    auto combine = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(n_seqs * H), dim3(BN_WAVE), 0, s, (bf16*)out, out_stride, part_o, part_ml, H, vd, n_splits,
                           sink ? 1 : 0, sink ? sink_values : nullptr, (const bf16*)gate, gate_stride);
        return bn_launch_status();
    };
    auto wide = [&](auto most) {
        constexpr int S = decltype(most)::value;
        return vd <= 64 ? combine(attn_general_combine_kernel<S, 1>) : vd <= 128 ? combine(attn_general_combine_kernel<S, 2>) :
               combine(attn_general_combine_kernel<S, 4>);
    };
    if (n_splits <= 4) return wide(std::integral_constant<int, 4>());
    if (n_splits <= 8) return wide(std::integral_constant<int, 8>());
    if (n_splits <= 16) return wide(std::integral_constant<int, 16>());
    if (n_splits <= 32) return wide(std::integral_constant<int, 32>());
    if (n_splits <= 48) return wide(std::integral_constant<int, 48>());
    return wide(std::integral_constant<int, AG_MAX_SPLITS>());
}

extern "C" int bn_attn_general_decode(const void* q, int q_stride, void* out, int out_stride, const void* k_pages,
                                      const void* v_pages, const int* block_table, int bt_stride, const int* seq_lens, int n_seqs,
                                      int H, int Hkv, int hs, int vd, float scale, const float* dist_a, const float* dist_b,
                                      int sink, const float* sink_values, int window, int keep_first, const void* gate, int gate_stride,
                                      int n_splits, int chunk, float* part_o, float* part_ml, const int* max_len, hipStream_t s) {
    return ag_decode(q, q_stride, out, out_stride, k_pages, v_pages, block_table, bt_stride, seq_lens, n_seqs, H, Hkv, hs, vd, scale, dist_a, dist_b, sink, sink_values,
                     window, keep_first, gate, gate_stride, n_splits, chunk, part_o, part_ml, max_len, nullptr, s);
}

// The same over rows of projections (queries, keys, values) that the kernel norms (wq, wk [hs] or null), rotates (inv_freq or null: rope_dims a multiple of
// 64, split-half pairs) and scales (temp_every > 0), and whose keys and values (v_from_k: the keys as projected) it writes to the pages.
extern "C" int bn_attn_general_decode_fresh(const void* q, int q_stride, void* out, int out_stride, const void* k_pages,
                                            const void* v_pages, const int* block_table, int bt_stride, const int* seq_lens, int n_seqs,
                                            int H, int Hkv, int hs, int vd, float scale, const float* dist_a, const float* dist_b,
                                            int sink, const float* sink_values, int window, int keep_first, const void* gate, int gate_stride,
                                            int n_splits, int chunk, float* part_o, float* part_ml, const int* max_len, int v_from_k,
                                            const float* wq, const float* wk, float eps, const float* inv_freq, int rope_dims, float temp_coef,
                                            int temp_every, hipStream_t s) {
    const AgFresh f = {v_from_k, wq, wk, eps, inv_freq, rope_dims, temp_coef, temp_every};
    return ag_decode(q, q_stride, out, out_stride, k_pages, v_pages, block_table, bt_stride, seq_lens, n_seqs, H, Hkv, hs, vd, scale, dist_a, dist_b, sink, sink_values,
                     window, keep_first, gate, gate_stride, n_splits, chunk, part_o, part_ml, max_len, &f, s);
}
