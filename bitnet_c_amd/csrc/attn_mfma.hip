// Attention over the paged bf16 cache on the matrix cores (v_mfma_f32_16x16x32_bf16), for
// head sizes 64 and 128, both phases.  Formulas as in attn_rows.hip (reference:
// src/transformer/gqa_scalar.c:61-207, src/transformer/batched_attn_scalar.c:97-245):
// kv head of head h is h / (H/Hkv); score = (q.k) * scale over the keys at positions <= the
// query's (and inside the window); online softmax; out = sum_t p_t V_t.  Scores, maxima,
// sums and the output accumulate in float32; p is rounded to bf16 for the second product.
//
// A wave works on "columns": a column is one (query token, query head) pair of one kv head,
// 16 columns per MFMA tile.  Everything stays in registers:
//   S^T[key, col]  = K[key, :] . Q[col, :]          A = 16 key rows of K,   B = Q^T
//   O^T[dim, col] += V^T[dim, keys] . P^T[keys, col]  A = 16 rows of V^T,   B = P^T
// The S^T tile leaves lane (col, g) with 4 keys per 16-key tile; the key rows fed to the two
// tiles of a 32-key block are permuted (row i of tile sb is key 8*(i/4) + 4*sb + i%4) so
// that each lane group g ends up with the 8 consecutive keys 8g..8g+7, which is exactly what
// the B operand of the second product wants and what 16 bytes of 8 consecutive positions of one
// value dimension hold.  The pages are laid out for exactly these operands ("blocked" pages,
// common.h): a (page, kv head) holds its 64 positions in two blocks of 32, and a block its keys and
// its values tile by tile in the lanes' order, so that the decode form loads an operand tile as 1 KB of
// consecutive bytes and the prompt form fetches a stage as one run.
//
// Prompt form: four waves own 64*NT columns = consecutive query tokens x GT heads;
// the keys and values they walk are staged through shared memory once for all four, or, where two groups of four take turns
// (attn_mfma_turns_kernel, heads of 128), for all eight.
// Decode form: the 16 columns are the heads of one kv group for the sequence's one new token;
// 4 waves take 32-key blocks in turn and merge through shared memory; long contexts are
// also split over gridDim.z and merged by attn_mfma_combine_kernel in a fixed order (two splits: one workgroup
// of 8 waves where that is the faster way, the same sums in the same order).  What a decode workgroup needs
// before its first block (the query, the frequencies, the new key and value, the length, the first block itself) is
// asked for at once, in straight-line code, with the length and the page numbers through the scalar unit: the first
// block of keys is on its way before the length is known (see the kernel), so that a short launch is two trips to
// memory instead of five.  Every entry of a block table must name a page of the pool for that, also the entries
// behind a sequence's last page.
#include "common.h"
#include "attn_mfma.h"
#include <mutex>
#include <type_traits>

#define PROMPT_BUFFERS 3      // staged key blocks of the prompt form in shared memory

static int compute_units() {
    static int n[64] = {0};                 // per device
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (n[dev] == 0) {
        int v = 0;
        n[dev] = (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0) ? v : 256;
    }
    return n[dev];
}
#include <math.h>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

#define LOG2E 1.4426950408889634f
#define LN2 0.6931471805599453f

struct MfmaArgs {
    const bf16* q;            // [n_tokens, q_stride], head h at h*HS, rotated
    bf16* out;                // [n_tokens, out_stride]
    const bf16* k_pages;      // [pages, Hkv, 64 * HS]: keys in the blocked order of common.h
    const bf16* vt_pages;     // [pages, Hkv, HS * 64]: values in the blocked order of common.h
    const int* block_table;   // [n_seqs, bt_stride]
    const int* seq_lens;      // decode: keys in the cache, the new one included; 0 = padding row
    const int* tiles;         // prompt: [n, 4] = seq, first token row, tokens, position of the first
    float* part_o;            // [n_tokens*H, n_splits, HS]
    float* part_ml;           // [n_tokens*H, n_splits, 2]   (max in natural-log units, sum)
    int q_stride, out_stride, bt_stride;
    int H, Hkv, GT;           // GT: heads of a kv group per column tile row (power of two <= 16)
    int window;
    int n_splits, chunk;
    float scale;
    // decode form only.  rotate != 0: q (and the new key) arrive unrotated and are rotated here,
    // angle = position * inv_freq[i], pairs (i, i + HS/2).  write_kv != 0: the workgroup whose keys
    // include the new position stores the new key (rotated) and value into the pages first.
    const float* inv_freq;
    int rotate, write_kv;
    // by_length != null: the sequences ordered by length, longest first.  Workgroups are handed out
    // in that order, every other run of `order_period` sequences backwards: when the launch puts
    // two workgroups on every CU, the ones that share a CU are then a long and a short sequence.
    const int* by_length;
    int order_period;
    // row_ssq != null (decode form with rotate): q, the new key and the new value of row b are what a product made of
    // an RMSNorm's input times the norm's weights, without the norm's factor (a deferred norm).  The factor
    // 1/sqrt(sum of row_ssq[b][0..n_pieces) / ssq_width + eps) multiplies the whole row, so it is applied here: folded
    // into the rotation's cosines and sines for q and the key, a multiplication for the value.
    const float* row_ssq;
    int n_pieces;
    float inv_ssq_width, ssq_eps;
    // max_len != null (decode form, n_splits > 1): the longest sequence's key count lives in device memory and
    // the keys per split follow from it (bn_split_chunk) instead of from `chunk`: a captured launch then adapts
    // its splits to the lengths of every replay.
    const int* max_len;
};

__device__ __forceinline__ bf16x8 ld16(const bf16* p) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(p));
}
// a decode step's cached keys and values; ONCE: non-temporally
template <bool ONCE> __device__ __forceinline__ bf16x8 ld16_cached(const bf16* p) {
    if constexpr (ONCE) return __builtin_bit_cast(bf16x8, bn_load_once(p));
    else return ld16(p);
}
// Combining a value with the ones 16 and 32 lanes away (the four lane groups of a column) without
// going through shared memory: gfx950 swaps 16- and 32-lane halves between two registers.
// The largest of three in one instruction; fmaxf would first bring each operand into canonical form (an instruction
// each), which the scores out of the matrix cores do not need.
__device__ __forceinline__ float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float max_over_lane_groups(float x) {
    const unsigned b = __float_as_uint(x);
    auto r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    const unsigned c = __float_as_uint(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
    auto t = __builtin_amdgcn_permlane32_swap(c, c, false, false);
    return fmaxf(__uint_as_float(t[0]), __uint_as_float(t[1]));
}
typedef __attribute__((ext_vector_type(8))) float f32x8;
// eight floats to eight bf16, round to nearest even (gfx950 converts two a time in hardware)
__device__ __forceinline__ bf16x8 pack8(const float (&s)[8]) {
    const f32x8 v = {s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7]};
    return __builtin_convertvector(v, bf16x8);
}
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    // round to nearest even, as __float2bfloat16 does
    uint32_t ua = __float_as_uint(a), ub = __float_as_uint(b);
    ua += 0x7fffu + ((ua >> 16) & 1u);
    ub += 0x7fffu + ((ub >> 16) & 1u);
    return (ua >> 16) | (ub & 0xffff0000u);
}

// A barrier of the workgroup that orders its shared memory only.  __syncthreads() also waits for everything that the wave
// has asked from global memory; this one leaves such loads in flight (whoever needs their data waits for it there).
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The float32 value of a bf16 bit pattern, widened where this stands and nowhere else: the compiler moves a plain shift
// up to the load of the pattern, and the load's wait with it.
__device__ __forceinline__ float widen_here(unsigned bits) {
    float f;
    asm volatile("v_lshlrev_b32 %0, 16, %1" : "=v"(f) : "v"(bits));
    return f;
}

// A read of p[idx] for an index that is the same in every lane, through the scalar unit (the
// constant address space makes the compiler pick a scalar load).  Only for memory that no kernel
// writes while this one runs (block tables, lengths).
__device__ __forceinline__ int uniform_load(const int* p, size_t idx) {
    typedef const int __attribute__((address_space(4))) * scalar_ptr;
    return reinterpret_cast<scalar_ptr>(reinterpret_cast<uintptr_t>(p))[idx];
}

// Shared memory serves 16 lanes of a 16-byte read at once, from 64 banks of 4 bytes.  The lanes
// that read a staged key block together hold rows 8a + b (+4 for the second tile), a, b in 0..3, and
// all want the same 16-byte chunk: rows are stored without padding and chunk c of row r lives at
// c ^ f(r), with f distinct for those 16 rows over the 256 bytes that the banks span (head size
// 128: a row is 256 bytes, f = 4a + b; head size 64: two rows share 256 bytes, the row's parity is
// one bit already and f = 2a + b/2 supplies the other three).
template <int HS>
__device__ __forceinline__ int k_swizzle(int row) {
    const int a = (row >> 3) & 3, b = row & 3;
    return HS == 128 ? (a << 2 | b) : (a << 1 | b >> 1);
}

// A 16-byte read serves the lanes in four turns of 16: quads of lanes {0, 3, 5, 6}, {1, 2, 4, 7} and
// the same of the upper 32 lanes (measured with a probe kernel and the bank-conflict counter).  In
// the operand layout lane = i + 16 g, so a turn holds two values of g (0 and 1, or 2 and 3) and, for
// the even one, i/4 in {0, 3}, for the odd one i/4 in {1, 2} (the other turn: the other way round).
// The staged V^T block (rows = dimensions, 16-byte chunks of 8 keys) is stored without padding with
// chunk c of row r at c ^ v_swizzle(r): h(i/4) = (-(i/4)) & 3 makes g ^ h distinct over a turn for
// rows that share their position inside 256 bytes; with 64 keys a row (two rows in 256 bytes, the
// row's lowest bit separates them) bit 1 of the row goes into bit 2 of the chunk as well.
template <int KEYS>
__device__ __forceinline__ int v_swizzle(int row) {
    const int h = (-(row >> 2)) & 3;
    return KEYS == 64 ? (h | ((row >> 1) & 1) << 2) : h;
}

// One 32-key block for NT column tiles, operands straight from the pages (the decode form).  kbase/vbase point at
// the block inside its page (blocked pages, common.h: every load below is 1 KB of consecutive bytes).  qpos/lo: per tile, this lane's column's
// position and first visible key (qpos < 0: no such column).  key_hi: keys >= key_hi do not exist (split end /
// length).  All operands are asked for up front: they come from memory, and the latency is paid once.
// The prompt form below has code of its own on purpose: the decode kernel is sensitive to how the compiler lays
// this code out, and changes made for the staged form must not move it.
// The operands of a block of 32 keys from blocked pages: tile row i of key tile 0 is the block's key 8 (i / 4) + i % 4,
// tile 1 four further; lane i + 16 g of value tile t holds dimension 16 t + i of the block's keys 8 g .. 8 g + 7.
template <int HS, bool ONCE>
__device__ __forceinline__ void load_block(const bf16* __restrict__ kbase, const bf16* __restrict__ vbase,
                                           bf16x8 (&ka)[HS / 32][2], bf16x8 (&va)[HS / 16], int lane) {
#pragma unroll
    for (int c = 0; c < HS / 32; ++c) {
        ka[c][0] = ld16_cached<ONCE>(kbase + (2 * c) * 512 + lane * 8);
        ka[c][1] = ld16_cached<ONCE>(kbase + (2 * c + 1) * 512 + lane * 8);
    }
#pragma unroll
    for (int t = 0; t < HS / 16; ++t) va[t] = ld16_cached<ONCE>(vbase + t * 512 + lane * 8);
}

template <int HS, int NT, bool need_mask>
__device__ __forceinline__ void attend_loaded_m(const bf16x8 (&ka)[HS / 32][2], bf16x8 (&va)[HS / 16],
                                               int kb, const bf16x8 (&q)[NT][HS / 32], f32x4 (&acc)[NT][HS / 16],
                                               float (&m)[NT], float (&l)[NT], const int (&qpos)[NT],
                                               const int (&lo)[NT], int key_hi, float scale2, int lane) {
    constexpr int DC = HS / 32, DT = HS / 16;
    const int g = lane >> 4;
    f32x4 st[NT][2];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) { st[nt][0] = (f32x4){0.f, 0.f, 0.f, 0.f}; st[nt][1] = (f32x4){0.f, 0.f, 0.f, 0.f}; }
#pragma unroll
    for (int c = 0; c < DC; ++c) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            st[nt][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[c][0], q[nt][c], st[nt][0], 0, 0, 0);
            st[nt][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[c][1], q[nt][c], st[nt][1], 0, 0, 0);
        }
    }
    // keys that do not exist may hold anything, NaN included: they are cleared in V^T (0 * NaN is NaN)
    const int first = kb + 8 * g;                     // this lane's 8 keys are first .. first+7
    auto clear_missing = [&](bf16x8 x) {
        uint4 v = __builtin_bit_cast(uint4, x);
        if (first + 0 >= key_hi) v.x &= 0xffff0000u;
        if (first + 1 >= key_hi) v.x &= 0x0000ffffu;
        if (first + 2 >= key_hi) v.y &= 0xffff0000u;
        if (first + 3 >= key_hi) v.y &= 0x0000ffffu;
        if (first + 4 >= key_hi) v.z &= 0xffff0000u;
        if (first + 5 >= key_hi) v.z &= 0x0000ffffu;
        if (first + 6 >= key_hi) v.w &= 0xffff0000u;
        if (first + 7 >= key_hi) v.w &= 0x0000ffffu;
        return __builtin_bit_cast(bf16x8, v);
    };
    if (need_mask) {
#pragma unroll
        for (int t = 0; t < DT; ++t) va[t] = clear_missing(va[t]);
    }
    bf16x8 pb[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        // raw scores; the scale (with log2 e folded in) is applied inside the exponent's fma
        float s[8];
#pragma unroll
        for (int sb = 0; sb < 2; ++sb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float v = st[nt][sb][r];
                if (need_mask) {
                    const int key = kb + 8 * g + 4 * sb + r;
                    if (key > qpos[nt] || key < lo[nt] || key >= key_hi) v = -INFINITY;
                }
                s[sb * 4 + r] = v;
            }
        float mx = fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])), fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7])));
        mx = max_over_lane_groups(mx);
        mx *= scale2;                                  // scale2 > 0: the maximum of the scaled scores
        // The reference point of the exponents moves only when the maximum has grown by more than
        // 2^8: until then p = 2^(s - m) may exceed 1 (at most 256), which float32 sums and bf16
        // weights hold as well, and the accumulators need no rescaling.  The result is the same.
        float m_new = m[nt];
        if (mx > m[nt] + 8.0f || m[nt] == -INFINITY) m_new = mx;
        if (m_new == -INFINITY) {
#pragma unroll
            for (int e = 0; e < 8; ++e) s[e] = 0.f;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) s[e] = __builtin_amdgcn_exp2f(fmaf(s[e], scale2, -m_new));
        }
        const bool moved = m_new != m[nt];
        if (__any(moved)) {
            const float alpha = (moved && m[nt] != -INFINITY) ? __builtin_amdgcn_exp2f(m[nt] - m_new) : (moved ? 0.f : 1.f);
            l[nt] *= alpha;
#pragma unroll
            for (int t = 0; t < DT; ++t) acc[nt][t] *= alpha;
        }
        m[nt] = m_new;
        pb[nt] = pack8(s);
    }
    // The sums of the weights come from the matrix cores too: a tile of ones times P gives every lane
    // the sum over the 32 keys for its column (the same bf16 weights that multiply V, so numerator
    // and denominator agree), instead of eight additions and two exchanges between lane groups.
    f32x4 lsum[NT];
    {
        const bf16x8 ones = __builtin_bit_cast(bf16x8, make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u));
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            lsum[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb[nt], (f32x4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < DT; ++t) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            acc[nt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[t], pb[nt], acc[nt][t], 0, 0, 0);
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) l[nt] += lsum[nt][0];
}

// The prompt form runs a block in two halves, so that a wave can have the first product of the next block on the
// matrix cores while its vector units work on the weights of the current one:
//   block_scores:   S^T = K . Q^T of a staged block of 32 keys (two 16-key tiles per column tile), nothing else;
//   block_weights_values: mask, reference point, exponentials, the sums of the weights and O^T += V^T . P^T.
// Operands come from the staged copies in shared memory (swizzled as k_swizzle / v_swizzle say).
// stage: the staged buffer (the same address in every lane); koff[c]: this lane's byte offset of chunk c of its key row
// of tile 0 (k_read_offsets), the row of tile 1 lies 4 rows further.
template <int HS, int NT, int KSTRIDE>
__device__ __forceinline__ void block_scores(const unsigned char* __restrict__ stage, const int (&koff)[HS / 32],
                                             const bf16x8 (&q)[NT][HS / 32], f32x4 (&st)[NT][2]) {
    constexpr int DC = HS / 32;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) { st[nt][0] = (f32x4){0.f, 0.f, 0.f, 0.f}; st[nt][1] = (f32x4){0.f, 0.f, 0.f, 0.f}; }
#pragma unroll
    for (int c = 0; c < DC; ++c) {
        const bf16x8 k0 = ld16(reinterpret_cast<const bf16*>(stage + koff[c]));
        const bf16x8 k1 = ld16(reinterpret_cast<const bf16*>(stage + koff[c] + 4 * KSTRIDE * 2));
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            st[nt][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0, q[nt][c], st[nt][0], 0, 0, 0);
            st[nt][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1, q[nt][c], st[nt][1], 0, 0, 0);
        }
    }
}

// stage as above; voff: this lane's byte offset of its 8 keys of V^T row i (v_read_offset), row t * 16 + i lies t * 16 rows further.
template <int HS, int NT, int VSTRIDE, bool need_mask>
__device__ __forceinline__ void block_weights_values_m(const f32x4 (&st)[NT][2], const unsigned char* __restrict__ stage, int voff,
                                                       int kb, f32x4 (&acc)[NT][HS / 16], float (&m)[NT], float (&l)[NT],
                                                       const int (&qpos)[NT], const int (&lo)[NT], int key_hi, float scale2,
                                                       int lane) {
    constexpr int DT = HS / 16;
    const int g = lane >> 4;
    const int first = kb + 8 * g;                     // this lane's 8 keys are first .. first+7
    // keys that do not exist may hold anything, NaN included: they are cleared in V^T (0 * NaN is NaN)
    auto clear_missing = [&](bf16x8 x) {
        uint4 v = __builtin_bit_cast(uint4, x);
        if (first + 0 >= key_hi) v.x &= 0xffff0000u;
        if (first + 1 >= key_hi) v.x &= 0x0000ffffu;
        if (first + 2 >= key_hi) v.y &= 0xffff0000u;
        if (first + 3 >= key_hi) v.y &= 0x0000ffffu;
        if (first + 4 >= key_hi) v.z &= 0xffff0000u;
        if (first + 5 >= key_hi) v.z &= 0x0000ffffu;
        if (first + 6 >= key_hi) v.w &= 0xffff0000u;
        if (first + 7 >= key_hi) v.w &= 0x0000ffffu;
        return __builtin_bit_cast(bf16x8, v);
    };
    // the first tiles of V^T are asked for now, so that they arrive while the weights are computed; every later
    // tile is asked for when an earlier one has been used
    constexpr int PF = DT < 4 ? DT : 4;
    bf16x8 vpre[PF];
    auto staged_v = [&](int t) { return ld16(reinterpret_cast<const bf16*>(stage + voff + t * 16 * VSTRIDE * 2)); };
#pragma unroll
    for (int t = 0; t < PF; ++t) vpre[t] = staged_v(t);
    bf16x8 pb[NT];
    float s[NT][8];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        // raw scores; the scale (with log2 e folded in) is applied inside the exponent's fma
#pragma unroll
        for (int sb = 0; sb < 2; ++sb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float v = st[nt][sb][r];
                if (need_mask) {
                    const int key = kb + 8 * g + 4 * sb + r;
                    if (key > qpos[nt] || key < lo[nt] || key >= key_hi) v = -INFINITY;
                }
                s[nt][sb * 4 + r] = v;
            }
        // The reference point m of the exponents moves only when some score of the column exceeds it
        // by more than 2^8: until then p = 2^(s - m) may exceed 1 (at most 256), which float32 sums
        // and bf16 weights hold as well, and nothing has to be rescaled.  So the common block only
        // asks whether any lane of the wave sees such a score; the exchange between the four lane
        // groups of a column, the new reference point and the rescaling happen when one does.
        float mx = max3(s[nt][0], s[nt][1], s[nt][2]);
        mx = max3(mx, s[nt][3], s[nt][4]);
        mx = max3(mx, s[nt][5], s[nt][6]);
        mx = max3(mx, s[nt][7], s[nt][7]);
        float m_new = m[nt];
        mx *= scale2;                                  // scale2 > 0: the maximum of the scaled scores
        if (__any(mx > m[nt] + 8.0f)) {                // also true for a column's first visible key (m = -inf)
            mx = max_over_lane_groups(mx);
            if (mx > m[nt] + 8.0f) m_new = mx;
            const bool moved = m_new != m[nt];
            if (__any(moved)) {
                const float alpha = (moved && m[nt] != -INFINITY) ? __builtin_amdgcn_exp2f(m[nt] - m_new) : (moved ? 0.f : 1.f);
                l[nt] *= alpha;
#pragma unroll
                for (int t = 0; t < DT; ++t) acc[nt][t] *= alpha;
            }
        }
        m[nt] = m_new;
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        // a column that has seen no key yet (only behind a mask) has m = -inf and only scores of -inf: 2^(-inf - 0) = 0
        const float ref = (need_mask && m[nt] == -INFINITY) ? 0.f : m[nt];
#pragma unroll
        for (int e = 0; e < 8; ++e) s[nt][e] = __builtin_amdgcn_exp2f(fmaf(s[nt][e], scale2, -ref));
        pb[nt] = pack8(s[nt]);
    }
    // The sums of the weights come from the matrix cores too: a tile of ones times P gives every lane
    // the sum over the 32 keys for its column (the same bf16 weights that multiply V, so numerator
    // and denominator agree), instead of eight additions and two exchanges between lane groups.
    f32x4 lsum[NT];
    {
        const bf16x8 ones = __builtin_bit_cast(bf16x8, make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u));
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            lsum[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb[nt], (f32x4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < DT; ++t) {
        bf16x8 va = vpre[t % PF];
        if (t + PF < DT) vpre[t % PF] = staged_v(t + PF);
        if (need_mask) va = clear_missing(va);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            acc[nt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, pb[nt], acc[nt][t], 0, 0, 0);
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) l[nt] += lsum[nt][0];
}

// The masked form (a block on the causal diagonal, at a window's edge or at the end of the keys) and
// the plain one are separate instantiations: almost every block is plain, and it carries no mask code.
template <int HS, int NT, bool ONCE>
__device__ __forceinline__ void attend_block(const bf16* __restrict__ kbase, const bf16* __restrict__ vbase,
                                             int kb, const bf16x8 (&q)[NT][HS / 32], f32x4 (&acc)[NT][HS / 16],
                                             float (&m)[NT], float (&l)[NT], const int (&qpos)[NT],
                                             const int (&lo)[NT], int key_hi, bool need_mask, float scale2,
                                             int lane) {
    bf16x8 ka[HS / 32][2];
    bf16x8 va[HS / 16];
    load_block<HS, ONCE>(kbase, vbase, ka, va, lane);
    if (need_mask)
        attend_loaded_m<HS, NT, true>(ka, va, kb, q, acc, m, l, qpos, lo, key_hi, scale2, lane);
    else
        attend_loaded_m<HS, NT, false>(ka, va, kb, q, acc, m, l, qpos, lo, key_hi, scale2, lane);
}
template <int HS, int NT, int VSTRIDE>
__device__ __forceinline__ void block_weights_values(const f32x4 (&st)[NT][2], const unsigned char* __restrict__ stage, int voff, int kb,
                                                     f32x4 (&acc)[NT][HS / 16], float (&m)[NT], float (&l)[NT],
                                                     const int (&qpos)[NT], const int (&lo)[NT], int key_hi, bool need_mask,
                                                     float scale2, int lane) {
    if (need_mask) block_weights_values_m<HS, NT, VSTRIDE, true>(st, stage, voff, kb, acc, m, l, qpos, lo, key_hi, scale2, lane);
    else block_weights_values_m<HS, NT, VSTRIDE, false>(st, stage, voff, kb, acc, m, l, qpos, lo, key_hi, scale2, lane);
}

// ---------------------------------------------------------------------------------------
// prompt form
// ---------------------------------------------------------------------------------------
// The waves of a workgroup need the same keys, so a stage of keys is fetched once per workgroup
// into shared memory, three buffers in turn, one barrier per stage: while stage s is multiplied, stage s + 1
// lies ready, stage s + 2 is stored from registers and the loads of stage s + 3 are in flight.  A wave works on
// two stages at once: it issues the first product of stage s + 1 (S^T = K . Q^T), then turns the scores of
// stage s into weights on the vector units while the last of those matrix instructions finish, and then
// multiplies the weights with the values of stage s.  (The compiler keeps the two in separate basic blocks, so
// inside one wave little more than that tail overlaps; most of the overlap of matrix cores and vector units
// comes from the two waves that share a SIMD.  Measured against one stage at a time: 65 -> 61 us at 2,048
// tokens of the 8B shape, 10.9 -> 9.9 ms at 32,768.)  A workgroup has NG groups of 4 waves; all groups hold the
// same query rows and a stage is NG blocks of 32 keys, one for each group, so the chain of blocks
// that a tile of late positions has to walk is NG times shorter; at the end the groups' partial
// results (reference point, sum, accumulators) are merged through shared memory in group order.  NG is 2 for
// launches of one round over the chip and 1 (with two workgroups a CU) for longer ones; the launch code says why.
// (Heads of 128 take this form, with NG = 1, for many short sequences alone.)
//
// A causal tile's work grows with its position, and a launch is as long as its longest workgroup.  A workgroup
// therefore takes two tiles, 2p and 2p + 1 of the list, and the host orders the list so that these are a long and
// a short tile of the same sequence (the first with the last, the second with the last but one, ...): every
// workgroup walks about the same number of key blocks (a prompt of 2,048 tokens: 65 blocks each, half of them
// per wave group, where the last tile alone walks 64), and the workgroups that run at the same time walk the
// keys of one sequence, which its L2 then holds.  Any order gives the same result.  A launch whose tiles all
// fit on the chip at once (paired = 0) gives every workgroup one tile: it is as long as its longest tile either
// way, and a second tile would only add its fixed cost.  The grid is
// one-dimensional with the kv heads running fastest: consecutive workgroups go to consecutive XCDs, so with
// eight kv heads every XCD serves one of them and its keys and values live in one L2 only.
template <int HS, int NT, int NG>
__global__ __launch_bounds__(256 * NG) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_mfma_prompt_kernel(MfmaArgs a, int n_tiles, int paired) {
    constexpr int DC = HS / 32, DT = HS / 16;
    constexpr int KB = 32 * NG;                           // keys per stage
    constexpr int KS = HS, VS = KB;                       // row strides (elements); both blocks swizzled, no padding
    constexpr int KV4 = 32 * HS / 8 / 256;                // uint4 loads per thread for K (and for V^T)
    constexpr int STAGE = (KB * KS + HS * VS) * 2;        // bytes of one buffer
    constexpr int MERGE = NG > 1 ? 4 * 64 * (DT * 4 + 2) * 4 : 0;
    static_assert(PROMPT_BUFFERS * STAGE >= MERGE, "the merge of the wave groups reuses the staging memory");
    extern __shared__ __align__(16) unsigned char smem[];     // prompt_smem_bytes(HS, NG)
    const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) & 3, grp = threadIdx.x >> 8;
    const int n = lane & 15, g = lane >> 4;
    // Where this thread's pieces of a stage come from (bytes from the page's keys of this kv head, and from its
    // V^T rows) and where they go in a staged buffer, and where this lane's operands lie in it: a handful of
    // numbers that depend on the thread alone.  They are made opaque to the compiler, which otherwise works them
    // out again in every stage (some seventy vector instructions of index arithmetic beside thirty-four products).
    static_assert(KV4 == 1 || KV4 == 2, "a thread stages one or two pieces of K and of V^T");
    int k_src[2], v_src[2], k_dst[2], v_dst[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        // A stage is one or two whole blocks of the blocked pages (common.h), and the threads fetch it in the pages' own
        // order, 16 consecutive bytes a thread: piece idx of the keys is lane i + 16 g of tile (c, tile) of block b, which
        // holds dimensions 32 c + 8 g .. + 7 of the block's key 8 (i / 4) + i % 4 + 4 tile; piece idx of the values is lane
        // i + 16 g of tile t of block b: keys 8 g .. 8 g + 7 of dimension 16 t + i.  The staged copies keep their own
        // (swizzled) order, and sixteen neighbouring lanes store the sixteen rows that sixteen lanes later read together.
        const int idx = threadIdx.x + h * 256 * NG;
        const int b = idx / (4 * HS), rem = idx % (4 * HS);
        const int li = rem & 15, lg = (rem >> 4) & 3, tl = rem >> 6;
        k_src[h] = idx * 16;
        const int krow = 32 * b + 8 * (li >> 2) + (li & 3) + 4 * (tl & 1), kchunk = 4 * (tl >> 1) + lg;
        k_dst[h] = (krow * KS + ((kchunk ^ k_swizzle<HS>(krow)) * 8)) * 2;
        const int vrow = 16 * tl + li, vchunk = 4 * b + lg;
        v_src[h] = idx * 16;
        v_dst[h] = (KB * KS + vrow * VS + ((vchunk ^ v_swizzle<KB>(vrow & 15)) * 8)) * 2;
        asm volatile("" : "+v"(k_src[h]), "+v"(v_src[h]), "+v"(k_dst[h]), "+v"(v_dst[h]));
    }
    int k_read[DC], v_read;
    {
        const int krow0 = 32 * grp + 8 * (n >> 2) + (n & 3);          // this group's block, key row of tile 0
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            k_read[c] = (krow0 * KS + (((c * 4 + g) ^ k_swizzle<HS>(krow0)) * 8)) * 2;
            asm volatile("" : "+v"(k_read[c]));
        }
        v_read = (KB * KS + n * VS + (((4 * grp + g) ^ v_swizzle<VS>(n)) * 8)) * 2;
        asm volatile("" : "+v"(v_read));
    }
    const int G = a.H / a.Hkv, GT = a.GT;
    const int n_head_tiles = (G + GT - 1) / GT;
    const int hy = a.Hkv * n_head_tiles;
    const int pair = blockIdx.x / hy, y = blockIdx.x - pair * hy;
    const int kvh = y / n_head_tiles, ht = y - kvh * n_head_tiles;
  for (int turn = 0; turn <= paired; ++turn) {
    const int tile = paired ? 2 * pair + turn : pair;
    if (tile >= n_tiles) break;                           // an odd number of tiles: the last one has no partner
    const int* tl = a.tiles + 4 * tile;
    const int seq = tl[0], tok0 = tl[1], n_tok = tl[2], pos0 = tl[3];
    if (n_tok <= 0) continue;                             // an empty tile (a list padded to a fixed length): the whole workgroup skips it

    bf16x8 q[NT][DC];
    int qpos[NT], lo[NT], head[NT], tok[NT];
    int w_hi = -1, w_lo = 0x7fffffff, all_hi = 0x7fffffff, all_lo = 0;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int c = (wave * NT + nt) * 16 + n;
        const int ti = c / GT, hg = ht * GT + (c - ti * GT);
        const bool ok = ti < n_tok && hg < G;
        head[nt] = kvh * G + hg;
        tok[nt] = tok0 + ti;
        qpos[nt] = ok ? pos0 + ti : -1;
        lo[nt] = (ok && a.window > 0) ? max(0, qpos[nt] + 1 - a.window) : 0;
#pragma unroll
        for (int c2 = 0; c2 < DC; ++c2) {
            uint4 z = make_uint4(0, 0, 0, 0);
            if (ok) z = *reinterpret_cast<const uint4*>(a.q + (size_t)tok[nt] * a.q_stride + (size_t)head[nt] * HS + c2 * 32 + g * 8);
            q[nt][c2] = __builtin_bit_cast(bf16x8, z);
        }
        if (ok) { w_hi = max(w_hi, qpos[nt]); w_lo = min(w_lo, lo[nt]); all_hi = min(all_hi, qpos[nt]); all_lo = max(all_lo, lo[nt]); }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        w_hi = max(w_hi, __shfl_xor(w_hi, o, BN_WAVE));
        w_lo = min(w_lo, __shfl_xor(w_lo, o, BN_WAVE));
        all_hi = min(all_hi, __shfl_xor(all_hi, o, BN_WAVE));
        all_lo = max(all_lo, __shfl_xor(all_lo, o, BN_WAVE));
    }
    f32x4 acc[NT][DT];
    float m[NT], l[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        m[nt] = -INFINITY; l[nt] = 0.f;
#pragma unroll
        for (int t = 0; t < DT; ++t) acc[nt][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    const float scale2 = a.scale * LOG2E;
    // the workgroup's key range: every wave takes part in the staging of all of it
    const int g_hi = pos0 + n_tok - 1;
    const int g_lo = a.window > 0 ? max(0, pos0 + 1 - a.window) : 0;
    const size_t bt_row = (size_t)seq * a.bt_stride;
    // Two stages are in flight: one or two 16-byte pieces of K and of V^T per thread and stage, in named
    // registers (arrays indexed in a loop end up in memory when they have to live across the products).
    struct Stage { uint4 k0, k1, v0, v1; };
    auto fetch = [&](int kb, Stage& st) {                 // a stage never crosses a page: KB divides BN_PAGE
        const int page = uniform_load(a.block_table, bt_row + kb / BN_PAGE);
        const int koff = kb % BN_PAGE;
        // the same addresses in every lane: the first of the stage's blocks of 32 keys in the page's keys of this kv
        // head, and in its values
        const unsigned char* kg = reinterpret_cast<const unsigned char*>(a.k_pages + (((size_t)page * a.Hkv + kvh) * BN_PAGE + koff) * HS);
        const unsigned char* vg = reinterpret_cast<const unsigned char*>(a.vt_pages + (((size_t)page * a.Hkv + kvh) * BN_PAGE + koff) * HS);
        st.k0 = *reinterpret_cast<const uint4*>(kg + (unsigned)k_src[0]);
        st.v0 = *reinterpret_cast<const uint4*>(vg + (unsigned)v_src[0]);
        if (KV4 > 1) {
            st.k1 = *reinterpret_cast<const uint4*>(kg + (unsigned)k_src[1]);
            st.v1 = *reinterpret_cast<const uint4*>(vg + (unsigned)v_src[1]);
        }
    };
    auto stash = [&](int buf, const Stage& st, int zero = 0) {    // zero: 0, in a form the compiler cannot see through
        unsigned char* stage = smem + buf * STAGE + zero;
        *reinterpret_cast<uint4*>(stage + k_dst[0]) = st.k0;
        *reinterpret_cast<uint4*>(stage + v_dst[0]) = st.v0;
        if (KV4 > 1) {
            *reinterpret_cast<uint4*>(stage + k_dst[1]) = st.k1;
            *reinterpret_cast<uint4*>(stage + v_dst[1]) = st.v1;
        }
    };
    // Stage t holds the keys kb0 + t KB ..; its block for this wave group begins at kbb(t).  A wave skips the blocks
    // that none of its columns can see.
    const int kb0 = (g_lo / KB) * KB;
    const int n_stages = (g_hi - kb0) / KB + 1;
    auto kbb = [&](int t) { return kb0 + t * KB + 32 * grp; };
    auto active = [&](int t) { return t < n_stages && w_hi >= 0 && kbb(t) <= w_hi && kbb(t) + 31 >= w_lo; };
    auto scores = [&](int t, f32x4 (&st)[NT][2]) {
        if (active(t)) block_scores<HS, NT, KS>(smem + (t % PROMPT_BUFFERS) * STAGE, k_read, q, st);
    };
    // One stage of the walk.  `cur` holds the scores of stage t (computed a stage ago), `next` takes those of stage
    // t + 1; `have` holds the loads of stage t + 2, `want` takes those of stage t + 3.
    auto step = [&](int t, f32x4 (&cur)[NT][2], f32x4 (&next)[NT][2], Stage& want, const Stage& have) {
        if (t + 3 < n_stages) fetch(kb0 + (t + 3) * KB, want);
        // The scores of the next block go to the matrix cores before the vector units start on the weights of this
        // one.  (Put into one basic block with the exponentials, so that the compiler can interleave them, they cost
        // more registers than a wave has here: 188 spilled.)
        scores(t + 1, next);
        if (active(t)) {
            const bool need_mask = (kbb(t) + 31 > all_hi) || (kbb(t) < all_lo);
            block_weights_values<HS, NT, VS>(cur, smem + (t % PROMPT_BUFFERS) * STAGE, v_read, kbb(t), acc, m, l, qpos, lo, w_hi + 1,
                                             need_mask, scale2, lane);
        }
        // The stores of a later stage must stay behind the products: next to their loads (where the
        // compiler puts them otherwise) they would wait out the memory latency before the block is
        // multiplied, instead of hiding it behind the block.  An empty asm makes the store offset look
        // as if it came out of the last product.
        int after_products = 0;
        asm volatile("" : "+v"(after_products) : "v"(acc[NT - 1][DT - 1][3]));
        if (t + 2 < n_stages) stash((t + 2) % PROMPT_BUFFERS, have, after_products);
        __syncthreads();
    };
    Stage sa = {make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0)}, sb = sa;
    fetch(kb0, sa);
    if (n_stages > 1) fetch(kb0 + KB, sb);
    stash(0, sa);
    if (n_stages > 1) stash(1, sb);
    if (n_stages > 2) fetch(kb0 + 2 * KB, sa);
    __syncthreads();
    f32x4 s_even[NT][2], s_odd[NT][2];
    scores(0, s_even);
    for (int t = 0; t < n_stages; t += 2) {
        step(t, s_even, s_odd, sb, sa);
        if (t + 1 >= n_stages) break;
        step(t + 1, s_odd, s_even, sa, sb);
    }
    if (NG > 1) {
        // the later groups hand their partial results to group 0, one column tile a time; the staging
        // memory is free now (the loop ended with a barrier)
        float* x_s = reinterpret_cast<float*>(smem);      // [wave][slot][lane]
        constexpr int SLOTS = DT * 4 + 2;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            for (int src = 1; src < NG; ++src) {
                float* mine = x_s + ((size_t)wave * SLOTS) * 64 + lane;
                if (grp == src) {
                    mine[0] = m[nt];
                    mine[64] = l[nt];
#pragma unroll
                    for (int t = 0; t < DT; ++t)
#pragma unroll
                        for (int r = 0; r < 4; ++r) mine[(2 + t * 4 + r) * 64] = acc[nt][t][r];
                }
                __syncthreads();
                if (grp == 0) {
                    const float m1 = mine[0], l1 = mine[64];
                    const float M = fmaxf(m[nt], m1);
                    if (M != -INFINITY) {
                        const float a0 = m[nt] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m[nt] - M);
                        const float a1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m1 - M);
                        l[nt] = l[nt] * a0 + l1 * a1;
#pragma unroll
                        for (int t = 0; t < DT; ++t)
#pragma unroll
                            for (int r = 0; r < 4; ++r) acc[nt][t][r] = acc[nt][t][r] * a0 + mine[(2 + t * 4 + r) * 64] * a1;
                        m[nt] = M;
                    }
                }
                __syncthreads();
            }
        }
    }
    if (grp == 0) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            if (qpos[nt] < 0) continue;
            const float inv = l[nt] > 0.f ? 1.0f / l[nt] : 0.f;
            bf16* o = a.out + (size_t)tok[nt] * a.out_stride + (size_t)head[nt] * HS + 4 * g;
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                uint2 w;
                w.x = pack2(acc[nt][t][0] * inv, acc[nt][t][1] * inv);
                w.y = pack2(acc[nt][t][2] * inv, acc[nt][t][3] * inv);
                *reinterpret_cast<uint2*>(o + t * 16) = w;
            }
        }
    }
    __syncthreads();                                      // the staging memory is free for the next tile
  }
}

// ---------------------------------------------------------------------------------------
// prompt form, long walks: two groups of waves take turns
// ---------------------------------------------------------------------------------------
// The weights of a block of 32 keys, as in block_weights_values_m: mask, reference point, exponentials; the rescaling of what has been summed.
template <int HS, int NT, typename READS>
__device__ __forceinline__ void turn_weights(f32x4 (&st)[NT][2], int kb, f32x4 (&acc)[NT][HS / 16], float (&m)[NT], float (&l)[NT],
                                             const int (&qpos)[NT], const int (&lo)[NT], int key_hi, bool need_mask, float scale2, int g, bf16x8 (&pb)[NT],
                                             READS reads) {
    float s[NT][8];
    if (need_mask) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int from = lo[nt] - kb - 8 * g, to = min(qpos[nt] + 1, key_hi) - kb - 8 * g;       // of the lane's eight keys
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float v = st[nt][e / 4][e % 4];
                v = e < from ? -INFINITY : v;
                v = e >= to ? -INFINITY : v;
                st[nt][e / 4][e % 4] = v;
            }
        }
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int e = 0; e < 8; ++e) s[nt][e] = st[nt][e / 4][e % 4];
    float mx[NT];
    bool above = false;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        mx[nt] = max3(s[nt][0], s[nt][1], s[nt][2]);
        mx[nt] = max3(mx[nt], s[nt][3], s[nt][4]);
        mx[nt] = max3(mx[nt], s[nt][5], s[nt][6]);
        mx[nt] = max3(mx[nt], s[nt][7], s[nt][7]) * scale2;
        above = above || mx[nt] > m[nt] + 8.0f;
    }
    if (__any(above)) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            mx[nt] = max_over_lane_groups(mx[nt]);
            const bool moved = mx[nt] > m[nt] + 8.0f;
            const float alpha = moved ? (m[nt] != -INFINITY ? __builtin_amdgcn_exp2f(m[nt] - mx[nt]) : 0.f) : 1.f;
            if (moved) m[nt] = mx[nt];
            l[nt] *= alpha;
#pragma unroll
            for (int t = 0; t < HS / 16; ++t) acc[nt][t] *= alpha;
        }
    }
    // the next slot's reads between the exponentials: shared memory takes one in some thirty cycles from the four waves of a group
    __builtin_amdgcn_sched_barrier(0);
    reads();
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const float ref = m[nt] == -INFINITY ? 0.f : m[nt];
#pragma unroll
        for (int e = 0; e < 8; ++e) s[nt][e] = __builtin_amdgcn_exp2f(fmaf(s[nt][e], scale2, -ref));
        pb[nt] = pack8(s[nt]);
    }
#pragma unroll
    for (int r = 0; r < 12; ++r) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x402, 4, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
}

// Eight waves, two a SIMD, in two groups of four.  A group's block of 32 keys is two turns, the products (scores of its next block, weights times values of this
// one, from registers alone) and the vector work (the next block's weights, and between its exponentials the reads of the operands after that),
// with a barrier behind each; the groups are one turn apart, so that of the two waves of a SIMD one has the matrix cores while the other
// has the vector unit.  (Left alone the two often want the same one, and wait for operands in front of their products.)
// SPLIT: both groups hold a tile's query columns and share its keys, of every 64 the first group the first 32, the other the rest; at the end
// their partial results (reference point, sum, accumulators) are merged through shared memory, each group merging one of two column tiles.  Else a
// group holds a tile of its own and both walk all the keys that either needs, which are fetched once for both: a workgroup takes two
// neighbouring pairs of the list that belong to one sequence, first their long tiles together, then their short ones, or, of the last of an odd
// number of pairs, its two tiles, which are the middle ones (two pairs of a sequence follow each other in the list, see ops.pair_tiles;
// tiles in another order are taken two by two just the same, and those of a pair of two sequences one by one).
// A block's keys and values go from the pages straight to shared memory, in the pages' own order, which is the operands': a wave fetches pieces of
// 1 KB, three turns or more before they are read.  Ring slot u holds block u's values and block u + 1's keys, which are used together.
// Blocks that every column sees whole run in a loop without a comparison.
// What bounds a step (two blocks, 8 products of 16 x 16 x 128 or so a wave and block: 34 matrix instructions of 16 cycles, some 75 vector instructions): 2,240
// cycles of 2 x (544 + 300), since a vector instruction delays its SIMD's matrix instructions (both read the same registers' ports); the two
// barriers take 10 % of it. 4,096 tokens of 32 heads over 8, us: one group a workgroup 167, keys split 148, a tile each 133 (1.03 PFLOP/s); 8,100 tokens 607, 510,
// 474 (1.13).  Tried, over split keys: operands read in
// the products' turn (8,100 tokens 607, from shared memory's latency); conditions instead of numbers for a block's kind (684: they are carried in
// vector registers); variants of a turn with and without masks (798: their accumulators are copied where they meet).
template <int HS, int NT, bool SPLIT>
__global__ __launch_bounds__(512, 2) void attn_mfma_turns_kernel(MfmaArgs a, int n_tiles, int paired) {
    constexpr int DC = HS / 32, DT = HS / 16, BLOCK = 32 * HS * 2, SLOT = 2 * BLOCK;
    constexpr int RING = SPLIT ? 4 : 5, GROUPS = SPLIT ? 2 : 1;          // slots, and the groups that have slots of their own
    constexpr int LOADS = 2 * GROUPS;                    // of a wave for a slot
    static_assert(BLOCK == 8 * 1024 && NT == 2, "eight pieces of keys and of values; a column tile a group to merge");
    static_assert(4 * 64 * DT * 4 * 4 <= 2 * SLOT, "a group's accumulators of a column tile fit a slot of both groups");
    __shared__ __align__(1024) unsigned char r0[GROUPS * SLOT], r1[GROUPS * SLOT], r2[GROUPS * SLOT], r3[GROUPS * SLOT], r4[SPLIT ? 16 : SLOT];
    const int lane = threadIdx.x & 63;
    // a wave's number in its group, and its group: waves w and w + 4 share a SIMD (groups by the SIMD that a wave finds itself on measured the same or 1 to 2 % slower)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3, grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int own = SPLIT ? grp : 0, piece = SPLIT ? wave : 4 * grp + wave;         // among those that share a slot
    const int n = lane & 15, g = lane >> 4;
    const int G = a.H / a.Hkv, GT = a.GT;
    const int n_head_tiles = (G + GT - 1) / GT;
    const int hy = a.Hkv * n_head_tiles;
    const int number = blockIdx.x / hy, y = blockIdx.x - number * hy;
    const int kvh = y / n_head_tiles, ht = y - kvh * n_head_tiles;
    const float scale2 = a.scale * LOG2E;
    // the list's entries of either group in either turn; -1: none
    int entry[2][2] = {{-1, -1}, {-1, -1}}, first_turn = 0;
    if (SPLIT) {
        entry[0][0] = entry[0][1] = paired ? 2 * number : number;
        if (paired && 2 * number + 1 < n_tiles) entry[1][0] = entry[1][1] = 2 * number + 1;
    } else {
        // Every other pair of a sequence is taken along, and its workgroup leaves.  A tile without a partner comes first, then the even pairs, then the odd
        // ones (with a turn a workgroup: all of this for the first turn, then for the second): workgroups go to the shader engines in turn, and those that had
        // only leaving ones would stay idle (8,100 tokens in the list's order: 894 us, so 510).
        const int pairs = n_tiles / 2, slots = (n_tiles + 1) / 2, at = number % slots - n_tiles % 2, even = (pairs + 1) / 2;
        const int j = at < 0 ? pairs : at < even ? 2 * at : 2 * (at - even) + 1;
        first_turn = number / slots;
        auto of = [&](int p, int seq) { return a.tiles[8 * p] == seq && a.tiles[8 * p + 4] == seq && a.tiles[8 * p + 2] > 0 && a.tiles[8 * p + 6] > 0; };
        const int seq = j < pairs ? a.tiles[8 * j] : 0;
        if (j < pairs && of(j, seq)) {
            int before = 0;                               // pairs of the sequence in front of this one
            for (int p = j - 1 - lane;; p -= 64) {
                const unsigned long long no = ~__ballot(p >= 0 && of(max(p, 0), seq));
                if (no) { before += __builtin_ctzll(no); break; }
                before += 64;
            }
            if (before & 1) return;                       // the pair in front of it takes it along
            const bool two = j + 1 < pairs && of(j + 1, seq);
            entry[0][0] = 2 * j;
            entry[0][1] = two ? 2 * j + 2 : 2 * j + 1;
            if (two) { entry[1][0] = 2 * j + 1; entry[1][1] = 2 * j + 3; }
        } else {
            entry[0][0] = 2 * j;
            if (2 * j + 1 < n_tiles) entry[1][0] = 2 * j + 1;
        }
    }
  for (int turn = first_turn; turn <= (paired ? 1 : first_turn); ++turn) {
    const int e0 = turn ? entry[1][0] : entry[0][0], e1 = turn ? entry[1][1] : entry[0][1];
    if (e0 < 0) break;
    const int* t0 = a.tiles + 4 * e0;
    const int* t1 = a.tiles + 4 * max(e1, 0);
    const int n0 = max(t0[2], 0), n1 = e1 < 0 ? 0 : max(t1[2], 0), pos_0 = t0[3], pos_1 = t1[3];
    if (n0 + n1 == 0) continue;                           // empty tiles (a list padded to a fixed length): the whole workgroup skips them
    const int seq = t0[0], tok0 = grp ? t1[1] : t0[1], n_tok = grp ? n1 : n0, pos0 = grp ? pos_1 : pos_0;
    // the positions that the workgroup's tiles begin and end at
    const int pos_first = n0 == 0 ? pos_1 : n1 == 0 ? pos_0 : min(pos_0, pos_1);
    const int pos_last = max(n0 ? pos_0 + n0 - 1 : 0, n1 ? pos_1 + n1 - 1 : 0);

    bf16x8 q[NT][DC];
    int qpos[NT], lo[NT];
    int w_hi = -1, w_lo = 0x7fffffff, all_hi = 0x7fffffff, all_lo = 0;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int c = (wave * NT + nt) * 16 + n;
        const int ti = c / GT, hg = ht * GT + (c - ti * GT);
        const bool ok = ti < n_tok && hg < G;
        qpos[nt] = ok ? pos0 + ti : -1;
        lo[nt] = (ok && a.window > 0) ? max(0, qpos[nt] + 1 - a.window) : 0;
#pragma unroll
        for (int c2 = 0; c2 < DC; ++c2) {
            uint4 z = make_uint4(0, 0, 0, 0);
            if (ok) z = *reinterpret_cast<const uint4*>(a.q + (size_t)(tok0 + ti) * a.q_stride + (size_t)(kvh * G + hg) * HS + c2 * 32 + g * 8);
            q[nt][c2] = __builtin_bit_cast(bf16x8, z);
        }
        if (ok) { w_hi = max(w_hi, qpos[nt]); w_lo = min(w_lo, lo[nt]); all_hi = min(all_hi, qpos[nt]); all_lo = max(all_lo, lo[nt]); }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        w_hi = max(w_hi, __shfl_xor(w_hi, o, BN_WAVE));
        w_lo = min(w_lo, __shfl_xor(w_lo, o, BN_WAVE));
        all_hi = min(all_hi, __shfl_xor(all_hi, o, BN_WAVE));
        all_lo = max(all_lo, __shfl_xor(all_lo, o, BN_WAVE));
    }
    w_hi = __builtin_amdgcn_readfirstlane(w_hi); w_lo = __builtin_amdgcn_readfirstlane(w_lo);
    all_hi = __builtin_amdgcn_readfirstlane(all_hi); all_lo = __builtin_amdgcn_readfirstlane(all_lo);
    f32x4 acc[NT][DT];
    float m[NT], l[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        m[nt] = -INFINITY; l[nt] = 0.f;
#pragma unroll
        for (int t = 0; t < DT; ++t) acc[nt][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    // The workgroup's steps: the same in every wave.  The group's block of step u starts at key first_key + STEP u.
    constexpr int STEP = 32 * GROUPS;
    static_assert(BN_PAGE == 64, "a page is two blocks");
    const int g_lo = a.window > 0 ? max(0, pos_first + 1 - a.window) : 0;
    const int step0 = g_lo / STEP, steps = pos_last / STEP - step0 + 1, last = steps - 1, first_key = step0 * STEP + 32 * own;
    // of its blocks, the ones that some column of the wave sees (first_u .. last_u), the ones whose keys do not all exist for it (from edge_u on) and the ones
    // that some of its columns sees only in part (from part_u on, and below whole_u); numbers, not conditions: every test is a scalar comparison
    auto from = [&](int key) { return key < first_key ? 0 : (key - first_key) / STEP + 1; };           // the first block that starts behind a key
    const int first_u = w_hi < 0 ? steps : from(w_lo - 32), last_u = min(last, from(w_hi) - 1);
    const int edge_u = from(w_hi - 31), part_u = from(all_hi - 31), whole_u = from(all_lo - 1);
    const size_t page_bytes = (size_t)a.Hkv * BN_PAGE * HS * 2, head_bytes = (size_t)kvh * BN_PAGE * HS * 2;
    const unsigned char* k_pool = reinterpret_cast<const unsigned char*>(a.k_pages) + head_bytes;
    const unsigned char* v_pool = reinterpret_cast<const unsigned char*>(a.vt_pages) + head_bytes;
    const int* table = a.block_table + (size_t)seq * a.bt_stride;
    auto page_of = [&](int u) { return uniform_load(table, (unsigned)(step0 + min(u, last)) / (BN_PAGE / STEP)); };    // a step past the last is the last again: read by nobody
    const unsigned mine = (piece * 64 + lane) * 16;
    auto fetch = [&](const unsigned char* page, int u, unsigned char* to) {
        const __amdgpu_buffer_rsrc_t b = bn_buffer(page, BN_PAGE * HS * 2);
        const unsigned half = (SPLIT ? grp : (step0 + min(u, last)) & 1) * BLOCK;
        bn_load_to_lds(b, to + piece * 1024, mine, half);
        if (SPLIT) bn_load_to_lds(b, to + (piece + 4) * 1024, mine, half + 4096);
    };
    bf16x8 kf[DC][2], vf[DT], pb[NT];
    f32x4 st[NT][2];
    const int at = own * SLOT + lane * 16;
    auto read_keys = [&](const unsigned char* from, int c0, int c1) {
#pragma unroll
        for (int c = c0; c < c1; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h) kf[c][h] = *reinterpret_cast<const bf16x8*>(from + at + BLOCK + (2 * c + h) * 1024);
    };
    auto read_values = [&](const unsigned char* from) {
#pragma unroll
        for (int t = 0; t < DT; ++t) vf[t] = *reinterpret_cast<const bf16x8*>(from + at + t * 1024);
    };
    auto scores = [&]() {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) st[nt][0] = st[nt][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < DC; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) st[nt][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[c][h], q[nt][c], st[nt][h], 0, 0, 0);
    };
    auto values = [&](int u, auto edges) {
        if (decltype(edges)::value && u >= edge_u) {      // keys that do not exist may hold anything, NaN included (0 * NaN is NaN)
            const int left = w_hi + 1 - (first_key + STEP * u + 8 * g);        // of the lane's eight keys
            uint32_t there[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) there[e] = left > 2 * e + 1 ? ~0u : left > 2 * e ? 0xffffu : 0u;
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                uint4 x = __builtin_bit_cast(uint4, vf[t]);
                x.x &= there[0]; x.y &= there[1]; x.z &= there[2]; x.w &= there[3];
                vf[t] = __builtin_bit_cast(bf16x8, x);
            }
        }
        f32x4 lsum[NT];
        const bf16x8 ones = __builtin_bit_cast(bf16x8, make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u));
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) lsum[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb[nt], (f32x4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) acc[nt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[t], pb[nt], acc[nt][t], 0, 0, 0);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) l[nt] += lsum[nt][0];
    };
    auto weights = [&](int u, auto edges, auto reads) {
        if (decltype(edges)::value && (u < first_u || u > last_u)) return;
        turn_weights<HS, NT>(st, first_key + STEP * u, acc, m, l, qpos, lo, w_hi + 1, decltype(edges)::value && (u >= part_u || u < whole_u), scale2, g, pb, reads);
    };
    // a turn's end; behind the products LEFT of this wave's loads may still be on their way: the slot that is read next has arrived
    auto end = [&](auto left) {
        __builtin_amdgcn_sched_barrier(0);
        if (decltype(left)::value >= 0) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(decltype(left)::value < 0 ? 0 : decltype(left)::value) : "memory");
        else asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    using std::integral_constant;
    size_t v_at = page_of(0) * page_bytes;                // of the step whose values are asked for next
    int page_k = page_of(1);                              // of the next step's keys
    auto fill = [&](int u, unsigned char* to) {
        const size_t k_at = page_k * page_bytes;
        fetch(v_pool + v_at, u, to + own * SLOT);
        fetch(k_pool + k_at, u + 1, to + own * SLOT + BLOCK);
        v_at = k_at;
    };
    unsigned char* const r_last = SPLIT ? r3 : r4;
    fetch(k_pool + v_at, 0, r_last + own * SLOT + BLOCK);
    fill(0, r0); page_k = page_of(2);
    fill(1, r1); page_k = page_of(3);
    fill(2, r2); page_k = page_of(4);
    if (!SPLIT) { fill(3, r3); page_k = page_of(5); }
    constexpr int AHEAD = RING - 1;                       // slots that are asked for at the start, and then one a step
    end(integral_constant<int, AHEAD * LOADS>());         // the first keys
    if (grp == 1) end(integral_constant<int, (AHEAD - 1) * LOADS>());        // one turn behind
    read_keys(r_last, 0, DC);
    __builtin_amdgcn_s_setprio(1);
    if (first_u <= 0) scores();
    __builtin_amdgcn_s_setprio(0);
    end(integral_constant<int, (AHEAD - 1) * LOADS>());
    read_keys(r0, 0, DC);
    read_values(r0);
    weights(0, std::true_type(), [] {});
    end(integral_constant<int, (AHEAD - 2) * LOADS>());
    // Slot u's turns.  The vector turn reads slot u + 1 and asks for slot u + AHEAD in the place of slot u - 1, whose operands the last products of either group have
    // used up.  Slot u + 1 has arrived: at the barrier in front of that turn a wave that shares it has asked for slots up to u + AHEAD - 1 and
    // may still wait for AHEAD - 2 of them, whether it ends its products there or, one turn apart, its vector work.
    auto step = [&](int u, unsigned char* free, const unsigned char* next, auto edges) {
        __builtin_amdgcn_s_setprio(1);
        if (!decltype(edges)::value || (u + 1 >= first_u && u < last_u)) scores();
        if (!decltype(edges)::value || (u >= first_u && u <= last_u)) values(u, edges);
        __builtin_amdgcn_s_setprio(0);
        end(integral_constant<int, (AHEAD - 2) * LOADS>());
        if (decltype(edges)::value) {
            read_keys(next, 0, DC);
            read_values(next);
            fill(u + AHEAD, free);
            weights(u + 1, edges, [] {});
        } else {
            read_keys(next, 0, 2);
            fill(u + AHEAD, free);
            weights(u + 1, edges, [&] { read_keys(next, 2, DC); read_values(next); });
        }
        page_k = page_of(u + AHEAD + 2);
        end(integral_constant<int, (AHEAD - 2) * LOADS>());
    };
    // steps whose blocks, and the next step's, every column of the workgroup sees whole
    const int clear = a.window > 0 ? 0 : (pos_first + 1) / STEP;
    int u = 0;
    if constexpr (SPLIT) {
        for (; u + RING < clear; u += RING) {
            step(u, r3, r1, std::false_type());
            step(u + 1, r0, r2, std::false_type());
            step(u + 2, r1, r3, std::false_type());
            step(u + 3, r2, r0, std::false_type());
        }
        for (; u < steps; u += RING) {
            step(u, r3, r1, std::true_type());
            if (u + 1 >= steps) break;
            step(u + 1, r0, r2, std::true_type());
            if (u + 2 >= steps) break;
            step(u + 2, r1, r3, std::true_type());
            if (u + 3 >= steps) break;
            step(u + 3, r2, r0, std::true_type());
        }
    } else {
        for (; u + RING < clear; u += RING) {
            step(u, r4, r1, std::false_type());
            step(u + 1, r0, r2, std::false_type());
            step(u + 2, r1, r3, std::false_type());
            step(u + 3, r2, r4, std::false_type());
            step(u + 4, r3, r0, std::false_type());
        }
        for (; u < steps; u += RING) {
            step(u, r4, r1, std::true_type());
            if (u + 1 >= steps) break;
            step(u + 1, r0, r2, std::true_type());
            if (u + 2 >= steps) break;
            step(u + 2, r1, r3, std::true_type());
            if (u + 3 >= steps) break;
            step(u + 3, r2, r4, std::true_type());
            if (u + 4 >= steps) break;
            step(u + 4, r3, r0, std::true_type());
        }
    }
    if (grp == 0) end(integral_constant<int, 0>());
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");       // nothing is on its way: the ring is free
    auto store = [&](int nt, float inv, auto value) {
        const int c = (wave * NT + nt) * 16 + n, ti = c / GT, hg = ht * GT + (c - ti * GT);
        bf16* o = a.out + (size_t)(tok0 + ti) * a.out_stride + (size_t)(kvh * G + hg) * HS + 4 * g;
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            uint2 w;
            w.x = pack2(value(t, 0) * inv, value(t, 1) * inv);
            w.y = pack2(value(t, 2) * inv, value(t, 3) * inv);
            *reinterpret_cast<uint2*>(o + t * 16) = w;
        }
    };
    if constexpr (SPLIT) {                                // the first group finishes column tile 0, the other tile 1
        float* given = reinterpret_cast<float*>(grp ? r1 : r0) + wave * DT * 4 * 64 + lane;
        const float* got = reinterpret_cast<const float*>(grp ? r0 : r1) + wave * DT * 4 * 64 + lane;
        float2* ml = reinterpret_cast<float2*>(r2) + wave * 64 + lane;           // [group][wave][lane]
        auto give = [&](int nt) {
            ml[grp * 256] = make_float2(m[nt], l[nt]);
#pragma unroll
            for (int t = 0; t < DT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) given[(t * 4 + r) * 64] = acc[nt][t][r];
        };
        auto finish = [&](int nt) {
            if (qpos[nt] < 0) return;
            const float2 o2 = ml[(1 - grp) * 256];
            const float m0 = grp ? o2.x : m[nt], m1 = grp ? m[nt] : o2.x, l0 = grp ? o2.y : l[nt], l1 = grp ? l[nt] : o2.y, M = fmaxf(m0, m1);
            const float a0 = m0 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m0 - M), a1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m1 - M);
            const float sum = l0 * a0 + l1 * a1;
            store(nt, sum > 0.f ? 1.0f / sum : 0.f, [&](int t, int r) {
                const float v = got[(t * 4 + r) * 64];
                return (grp ? v : acc[nt][t][r]) * a0 + (grp ? acc[nt][t][r] : v) * a1;
            });
        };
        if (grp == 0) give(1); else give(0);
        lds_barrier();
        if (grp == 0) finish(0); else finish(1);
    } else {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            if (qpos[nt] >= 0) store(nt, l[nt] > 0.f ? 1.0f / l[nt] : 0.f, [&](int t, int r) { return acc[nt][t][r]; });
    }
    lds_barrier();                                        // the ring is free for the next tile
  }
}

// ---------------------------------------------------------------------------------------
// decode form
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ void rotate8(uint4& lo, uint4& hi, const float* __restrict__ cs, const float* __restrict__ sn) {
    // lo/hi: 8 bf16 each, element e of lo pairs with element e of hi; cs/sn: their 8 cos/sin
    uint32_t* pl = reinterpret_cast<uint32_t*>(&lo);
    uint32_t* ph = reinterpret_cast<uint32_t*>(&hi);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float a0 = bf16lo_to_f32(pl[k]), a1 = bf16hi_to_f32(pl[k]);
        const float b0 = bf16lo_to_f32(ph[k]), b1 = bf16hi_to_f32(ph[k]);
        const float c0 = cs[2 * k], c1 = cs[2 * k + 1], s0 = sn[2 * k], s1 = sn[2 * k + 1];
        pl[k] = pack2(a0 * c0 - b0 * s0, a1 * c1 - b1 * s1);
        ph[k] = pack2(a0 * s0 + b0 * c0, a1 * s1 + b1 * c1);
    }
}

// a - b with its own rounding, whatever a was formed by
__device__ __forceinline__ float minus_rounded(float a, float b) {
#pragma clang fp contract(off)
    return a - b;
}

#define AD_WHOLE_PAGES 16             // widest block table of the WHOLE form (attn_mfma_launch)

// WHOLE: a workgroup of eight waves takes both splits of a launch of two for its sequence and kv head, four waves a split, and
// merges them itself, as attn_mfma_combine_kernel would: the same sums in the same order, so that no bit depends on the form.
template <int HS, bool WHOLE, bool ONCE>
__global__ __launch_bounds__(WHOLE ? 512 : 256) void attn_mfma_decode_kernel(MfmaArgs a) {
    constexpr int DC = HS / 32, DT = HS / 16, HALF = HS / 2;
    constexpr int SPLITS = WHOLE ? 2 : 1, THREADS = 256 * SPLITS;
    __shared__ float m_s[4 * SPLITS][16], l_s[4 * SPLITS][16];
    __shared__ float cos_s[HALF], sin_s[HALF];
    extern __shared__ float o_s[];                      // [split, wave of it][dim][GT + 1]: the heads' columns, padded
    const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) & 3;
    const int n = lane & 15, g = lane >> 4;
    const int G = a.H / a.Hkv, GT = a.GT;
    const int n_head_tiles = (G + GT - 1) / GT;
    // kv heads run fastest in the grid: consecutive workgroups go to different XCDs, so every XCD gets
    // a share of every sequence, however unequal their lengths (with the sequences fastest and a
    // batch that is a multiple of 8, a sequence's heads all landed on one XCD)
    const int kvh = blockIdx.x / n_head_tiles, ht = blockIdx.x - kvh * n_head_tiles;
    int seq = blockIdx.y;
    const int split = WHOLE ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : blockIdx.z;      // of these waves
    if (a.by_length) {
        int r = seq;
        if (a.order_period > 0) {
            const int run = r / a.order_period;
            if (run & 1) {
                const int first = run * a.order_period, last = min(first + a.order_period, (int)gridDim.y) - 1;
                r = first + (last - r);
            }
        }
        seq = uniform_load(a.by_length, r);
        if ((unsigned)seq >= gridDim.y) return;          // not a permutation: touch nothing
    }
    // Everything that does not depend on the sequence's length is asked for now, in straight-line code with no lane left
    // out of a load (a lane without a head, a thread without an element asks for a neighbour's and drops it), so that
    // nothing waits for anything but its own data: the query's heads, the frequencies, the new key and value, the sums of
    // squares of a deferred norm.  The length and the pages come through the scalar unit, beside those loads.
    const int hg = ht * GT + n;
    const bool q_lane = n < GT && hg < G;
    const int head = kvh * G + (q_lane ? hg : 0);
    const bf16* row = a.q + (size_t)seq * a.q_stride;
    uint4 z[DC];
#pragma unroll
    for (int c = 0; c < DC; ++c) z[c] = *reinterpret_cast<const uint4*>(row + (size_t)head * HS + c * 32 + g * 8);
    const int tid = threadIdx.x;
    float freq = 0.f, piece = 0.f;
    if (a.rotate) freq = a.inv_freq[tid & (HALF - 1)];
    if (a.row_ssq) piece = a.row_ssq[(size_t)seq * a.n_pieces + min(lane, a.n_pieces - 1)];
    unsigned new_k0 = 0, new_k1 = 0, new_v = 0;          // bf16 bit patterns, widened where they are used
    if (a.write_kv) {        // threads below HALF hold a pair of the key, the HS behind them an element of the value
        const unsigned short* kn = reinterpret_cast<const unsigned short*>(row + (size_t)(a.H + kvh) * HS);
        const unsigned short* vn = reinterpret_cast<const unsigned short*>(row + (size_t)(a.H + a.Hkv + kvh) * HS);
        new_k0 = kn[tid & (HALF - 1)];
        new_k1 = kn[(tid & (HALF - 1)) + HALF];
        new_v = vn[(tid - HALF) & (HS - 1)];
    }
    const int L = uniform_load(a.seq_lens, seq);
    const int chunk = a.max_len ? bn_split_chunk(uniform_load(a.max_len, 0), a.n_splits) : a.chunk;
    // So is the first block of keys that this wave will take, whose place does not depend on the length when no window
    // cuts the keys: its page and its 16 KB are on their way while the rotation is worked out and the new token is
    // stored, instead of after all that.  If the sequence turns out to end before the block, it is dropped unused (every
    // entry of a block table names a page of the pool, also those behind a sequence's last page); if the block holds
    // the new token's position, it is asked for again behind the store.
    // (With a window, or a table that ends before the block, the loads go to the table's first page and are dropped:
    // loads under a branch would make everything behind it wait for all of them.)
    const int kb_first = split * chunk + 32 * __builtin_amdgcn_readfirstlane(wave);
    const bool ahead = a.window == 0 && kb_first / BN_PAGE < a.bt_stride;
    bf16x8 ka0[DC][2];
    bf16x8 va0[DT];
    const int page0 = uniform_load(a.block_table, (size_t)seq * a.bt_stride + (ahead ? kb_first / BN_PAGE : 0));
    const size_t at0 = (((size_t)page0 * a.Hkv + kvh) * BN_PAGE + kb_first % BN_PAGE) * HS;
    const bf16* kbase0 = a.k_pages + at0;
    const bf16* vbase0 = a.vt_pages + at0;
    load_block<HS, ONCE>(kbase0, vbase0, ka0, va0, lane);
    const bool ok = q_lane && L > 0;
    const int lo_key = a.window > 0 ? max(0, L - a.window) : 0;
    const int k_lo = max(lo_key, split * chunk), k_hi = min(L, (split + 1) * chunk);       // [k_lo, k_hi)
    if (!WHOLE && a.n_splits > 1 && k_lo >= k_hi) {
        // A split without keys (a sequence shorter than the launch's longest, a padding row): it leaves "nothing seen"
        // for the merge, which then does not read its sums, and is gone before it asks for anything else.
        if (threadIdx.x < GT && ht * GT + threadIdx.x < G) {
            const size_t prow = ((size_t)seq * a.H + kvh * G + ht * GT + threadIdx.x) * a.n_splits + split;
            a.part_ml[prow * 2] = -INFINITY;
            a.part_ml[prow * 2 + 1] = 0.f;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // what was asked for has arrived before the wave ends
        return;
    }
    float row_scale = 1.0f;
    if (a.row_ssq) {                                     // the same few floats in every lane, added in piece order
        float ss = 0.f;
        for (int p = 0; p < a.n_pieces; ++p)
            ss += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, piece), p));
        row_scale = 1.0f / sqrtf(ss * a.inv_ssq_width + a.ssq_eps);
    }

    if (a.rotate && L > 0) {
        if (tid < HALF) {                                // HALF <= 64: one frequency a thread
            float sv, cv;
            sincosf((float)(L - 1) * freq, &sv, &cv);
            cos_s[tid] = cv * row_scale; sin_s[tid] = sv * row_scale;
        }
        lds_barrier();                                   // the block that is on its way stays on its way
    }
    // the new token's key and value go into the cache before anyone reads them: the workgroup
    // that owns the new position does it (there is one per kv head: write_kv needs n_head_tiles == 1)
    if (a.write_kv && L > 0 && (WHOLE || (L - 1 >= k_lo && L - 1 < k_hi))) {
        const int pos = L - 1;
        // through the scalar unit (the length is the same in every lane), so that it does not queue behind the block
        // that is on its way
        const int page = uniform_load(a.block_table, (size_t)seq * a.bt_stride + __builtin_amdgcn_readfirstlane(pos / BN_PAGE));
        const int off = pos % BN_PAGE;
        bf16* kdst = const_cast<bf16*>(a.k_pages) + ((size_t)page * a.Hkv + kvh) * BN_PAGE * HS;
        bf16* vdst = const_cast<bf16*>(a.vt_pages) + ((size_t)page * a.Hkv + kvh) * BN_PAGE * HS;
        const int t = threadIdx.x;
        if (t < HALF) {
            float k0 = widen_here(new_k0), k1 = widen_here(new_k1);
            if (a.rotate) {
                const float c = cos_s[t], sv = sin_s[t];
                const float r0 = k0 * c - k1 * sv, r1 = k0 * sv + k1 * c;
                k0 = r0; k1 = r1;
            }
            kdst[bn_blocked_k_offset(off, t, HS)] = __float2bfloat16(k0);
            kdst[bn_blocked_k_offset(off, t + HALF, HS)] = __float2bfloat16(k1);
        } else if (t < HALF + HS) {
            const int d = t - HALF;
            reinterpret_cast<unsigned short*>(vdst)[bn_blocked_v_offset(off, d, HS)] =
                a.row_ssq ? __builtin_bit_cast(unsigned short, __float2bfloat16(widen_here(new_v) * row_scale))
                          : (unsigned short)new_v;
        }
        // only this workgroup reads what it has just stored: a fence of workgroup scope is enough
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        __syncthreads();
    }

    bf16x8 q[1][DC];
    {
        if (!q_lane) {
#pragma unroll
            for (int c = 0; c < DC; ++c) z[c] = make_uint4(0, 0, 0, 0);
        }
        if (a.rotate && L > 0) {
#pragma unroll
            for (int c = 0; c < DC / 2; ++c)      // chunk c holds pair indices c*32 + g*8 .. +7, its partners are in chunk c + DC/2
                rotate8(z[c], z[c + DC / 2], cos_s + c * 32 + g * 8, sin_s + c * 32 + g * 8);
        }
#pragma unroll
        for (int c = 0; c < DC; ++c) q[0][c] = __builtin_bit_cast(bf16x8, z[c]);
    }
    int qpos[1] = {ok ? L - 1 : -1};
    int lo[1] = {lo_key};

    const float scale2 = a.scale * LOG2E;
    const size_t bt_row = (size_t)seq * a.bt_stride;
    const int os = GT + 1;
    f32x4 acc[1][DT];
    float m[1] = {-INFINITY}, l[1] = {0.f};
#pragma unroll
    for (int t = 0; t < DT; ++t) acc[0][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    if (k_lo < k_hi) {
        // (Keeping the next block's operands in a second set of registers while the current block is multiplied was
        // measured and gained nothing: the CU's other waves already cover a wave's wait for its loads.)
        // The waves take the blocks of 32 keys in turn, so that neighbouring waves ask for the two halves of a page at
        // the same time (a wave that takes whole pages by itself was measured 10 to 20 % slower, and so was splitting
        // the sequences of a large batch: the order by length with unsplit sequences keeps the CUs busiest).
        int kb = (k_lo / 32) * 32 + 32 * wave;
        if (ahead && kb == kb_first && kb < k_hi) {        // the block that was asked for at the start
            if (a.write_kv && L - 1 >= kb && L - 1 < kb + 32) load_block<HS, ONCE>(kbase0, vbase0, ka0, va0, lane);
            if ((kb + 32 > k_hi) || (kb < k_lo))
                attend_loaded_m<HS, 1, true>(ka0, va0, kb, q, acc, m, l, qpos, lo, k_hi, scale2, lane);
            else
                attend_loaded_m<HS, 1, false>(ka0, va0, kb, q, acc, m, l, qpos, lo, k_hi, scale2, lane);
            kb += 128;
        }
        for (; kb < k_hi; kb += 128) {
            // the page index is the same for the whole wave: read through the scalar unit, so that it
            // does not queue behind the vector loads
            const int page = uniform_load(a.block_table, bt_row + __builtin_amdgcn_readfirstlane(kb / BN_PAGE));
            const int koff = kb % BN_PAGE;                 // 0 or 32: the page's first or second block
            const bf16* kbase = a.k_pages + (((size_t)page * a.Hkv + kvh) * BN_PAGE + koff) * HS;
            const bf16* vbase = a.vt_pages + (((size_t)page * a.Hkv + kvh) * BN_PAGE + koff) * HS;
            const bool need_mask = (kb + 32 > k_hi) || (kb < k_lo);
            attend_block<HS, 1, ONCE>(kbase, vbase, kb, q, acc, m, l, qpos, lo, k_hi, need_mask, scale2, lane);
        }
    }
    // every wave's (m, l, O^T) into shared memory
    const int at = (WHOLE ? 4 * split : 0) + wave;
    if (g == 0) { m_s[at][n] = m[0]; l_s[at][n] = l[0]; }
    if (n < GT) {
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) o_s[(at * HS + t * 16 + 4 * g + r) * os + n] = acc[0][t][r];
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < HS * GT; idx += THREADS) {
        const int col = idx / HS, dim = idx - col * HS;      // consecutive threads: consecutive dims
        const int hg2 = ht * GT + col;
        if (hg2 >= G) continue;
        const int hd = kvh * G + hg2;
        // a split's four waves, in wave order
        auto merge = [&](int u, float& M, float& num, float& den) {
            const int at = 4 * u;
            M = fmaxf(fmaxf(m_s[at][col], m_s[at + 1][col]), fmaxf(m_s[at + 2][col], m_s[at + 3][col]));
            num = den = 0.f;
            if (M != -INFINITY) {
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const float e = exp2f(m_s[at + w][col] - M);
                    num = fmaf(e, o_s[((at + w) * HS + dim) * os + col], num);
                    den = fmaf(e, l_s[at + w][col], den);
                }
            }
        };
        bf16* out = a.out + (size_t)seq * a.out_stride + (size_t)hd * HS + dim;
        if constexpr (WHOLE) {                               // then the splits, in split order
            float ms[SPLITS], num[SPLITS], den[SPLITS], top = -INFINITY;
#pragma unroll
            for (int u = 0; u < SPLITS; ++u) {
                float M;
                merge(u, M, num[u], den[u]);
                ms[u] = M == -INFINITY ? -INFINITY : M * LN2;
                top = fmaxf(top, ms[u]);
            }
            float w[SPLITS], o = 0.f, z = 0.f;
            int n_live = 0;
#pragma unroll
            for (int u = 0; u < SPLITS; ++u) {
                w[u] = (top == -INFINITY || ms[u] == -INFINITY) ? 0.f : expf(minus_rounded(ms[u], top));
                if (w[u] != 0.f) n_live = u + 1;
            }
#pragma unroll
            for (int u = 0; u < SPLITS; ++u) {
                if (u >= n_live) break;
                z = fmaf(w[u], den[u], z);
                o = fmaf(w[u], w[u] != 0.f ? num[u] : 0.f, o);
            }
            *out = __float2bfloat16(o * (z > 0.f ? 1.0f / z : 0.f));
        } else {
            float M, num, den;
            merge(0, M, num, den);
            if (a.n_splits == 1) {
                *out = __float2bfloat16(den > 0.f ? num / den : 0.f);
            } else {
                const size_t prow = ((size_t)seq * a.H + hd) * a.n_splits + split;
                a.part_o[prow * HS + dim] = num;
                if (dim == 0) { a.part_ml[prow * 2] = (M == -INFINITY) ? -INFINITY : M * LN2; a.part_ml[prow * 2 + 1] = den; }
            }
        }
    }
}

// out[row, d] = sum_s e^{m_s - m} o_s[d] / sum_s e^{m_s - m} l_s: one wave per row, the weights of all splits computed at once
// (one lane per split), the sums in split order.  A launch of a few hundred waves is bound by its chain of waits, not by its
// bytes: all S >= n_splits sums are asked for beside the weights' maxima (the last split's again past the end, and what a split
// without keys holds is dropped: two trips to memory become one), and a weight comes out of its lane with a v_readlane instead of
// through shared memory's crossbar, whose wait in the sum of the denominators came once a split.
//   us inside a step, before -> this: 32 rows of 32 splits 6.9 -> 4.7, 64 of 3 3.9 -> 3.6, 256 of 4 4.7 -> 4.7 (its sums come from memory).
struct __attribute__((packed, aligned(4))) TwoFloats { float x, y; };      // in one load, also where the caller's room is not on 8 bytes
template <int S, int V>
__global__ __launch_bounds__(64) void attn_mfma_combine_kernel(bf16* __restrict__ out, int out_stride,
                                                               const float* __restrict__ part_o,
                                                               const float* __restrict__ part_ml, int H, int n_splits) {
    constexpr int HS = 64 * V;
    const int row = blockIdx.x, lane = threadIdx.x;
    const int tok = row / H, head = row - tok * H;
    const TwoFloats ml = reinterpret_cast<const TwoFloats*>(part_ml)[(size_t)row * n_splits + min(lane, n_splits - 1)];
    const float* po = part_o + (size_t)row * n_splits * HS + V * lane;
    float v[S][V];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const float* from = po + (size_t)min(s, n_splits - 1) * HS;
        if constexpr (V == 2) {
            const TwoFloats two = *reinterpret_cast<const TwoFloats*>(from);
            v[s][0] = two.x; v[s][1] = two.y;
        } else {
            v[s][0] = *from;
        }
    }
    __builtin_amdgcn_sched_barrier(0);                                     // all asked for before anything is waited for
    const float ms = lane < n_splits ? ml.x : -INFINITY;
    const float M = wave_max(ms);
    const float w = (M == -INFINITY || ms == -INFINITY) ? 0.f : expf(ms - M);
    auto of = [](float x, int s) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), s)); };
    float den = 0.f, num[V] = {};
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const float ws = of(w, s);
        den = fmaf(ws, ws != 0.f ? of(ml.y, s) : 0.f, den);                // (no branch: a load would be moved behind it)
#pragma unroll
        for (int u = 0; u < V; ++u) num[u] = fmaf(ws, ws != 0.f ? v[s][u] : 0.f, num[u]);
    }
    const float inv = den > 0.f ? 1.0f / den : 0.f;
    bf16* o = out + (size_t)tok * out_stride + (size_t)head * HS + V * lane;
    bf16 r[V];
#pragma unroll
    for (int u = 0; u < V; ++u) r[u] = __float2bfloat16(num[u] * inv);
    if constexpr (V == 2) *reinterpret_cast<uint32_t*>(o) = __builtin_bit_cast(uint32_t, r);
    else *o = r[0];
}

// 1 when the matrix-core kernels take this shape
extern "C" int bn_attn_mfma_supports(int hs) { return (hs == BN_MFMA_HEAD_DIM_SMALL || hs == BN_MFMA_HEAD_DIM_LARGE) ? 1 : 0; }

// query tokens per tile of the prompt form, for GT heads per group
extern "C" int bn_attn_mfma_prompt_tokens(int hs, int GT) { return (hs == 64 ? 256 : 128) / GT; }

// Which kernel a prompt's launch takes, by its workgroups alone (the tiles' positions are on the device).  PAIRED: a workgroup takes a pair of the list's
// tiles, a long and a short one.
enum { PF_TWO, PF_TWO_PAIRED, PF_ONE, PF_ONE_PAIRED, PF_SPLIT, PF_SPLIT_PAIRED, PF_EACH, PF_EACH_PAIRED };

static int prompt_form(long long n_tiles, long long n_tokens, long long n_seqs, long long wgs_per_seq, int hs, int window) {
    const long long cus = compute_units(), pairs = (n_tiles + 1) / 2;
    const bool paired = n_tiles * wgs_per_seq > cus;     // more tiles than CUs
    const long long wgs = (paired ? pairs : n_tiles) * wgs_per_seq;
    // Two groups of waves a workgroup (eight waves, one workgroup a CU) halve the chain of blocks that a tile walks,
    // which is what a launch of one round waits for.  A launch of several rounds is faster with one group a
    // workgroup and two workgroups a CU: they share nothing and drift apart, so that one's matrix instructions
    // meet the other's vector work, where the two groups of one workgroup meet at a barrier in every stage and do
    // the same thing at the same time (8 to 16 % at 8,192 tokens and for eight or 64 prompts of 128 to 2,048).
    // It is taken from four rounds on, and from two when its rounds (of two workgroups a CU) are not much emptier
    // than those of the wide form (6,144 tokens of one sequence are three full rounds of the wide form and one and
    // a half of the other: 410 against 445 us).
    const double fill1 = (double)wgs / (double)(((wgs + 2 * cus - 1) / (2 * cus)) * 2 * cus);
    const double fill2 = (double)wgs / (double)(((wgs + cus - 1) / cus) * cus);
    const bool one = wgs >= 4 * cus || (wgs >= 2 * cus && fill1 * 1.1 >= fill2);
    if (hs == 64) return one ? (paired ? PF_ONE_PAIRED : PF_ONE) : (paired ? PF_TWO_PAIRED : PF_TWO);
    // Heads of 128: the two groups take turns, over split keys, where those of 64 walk in step (always as fast or faster), or have a tile each (a CU's keys are
    // fetched once for two).  Over 617 launches (nine shapes of heads and windows; 1 to 64 sequences of 16 to 8,100 tokens, some behind earlier ones)
    // what this rule takes is the older forms' time (one group, or two in step, by the rule above) or less but for three (by 3 to 6 %), 14 % less on average, and
    // 3 % more than the fastest form's.  us, one group / split / a tile each (the older form), 32 heads over 8 unless it says more: one prompt of 1,024 36 / 25 /
    // 37 (30), 2,048 71 / 48 / 64 (59), 2,500 109 / 101 / 86 (128), 4,096 167 / 148 / 133 (167), 5,000 351 / 249 / 291 (329), 8,100 607 / 510 / 474 (607); 64 new tokens behind
    // 4,000 115 / 60 / 108 (83); two of 640, 64 heads over 8, 44 / 49 / 38 (53); sixteen of 640 104 / 125 / 114 (104); eight of 700, 40 heads over 40, 98 / 116 / 119 (98).
    if (!paired) return PF_SPLIT;                        // the chip is not full: as many, short chains as there can be
    const long long tokens = n_tokens / n_seqs;          // new ones of a sequence; how many there are before them is not known here
    const long long a_seq = n_tiles / n_seqs;
    const bool equal = n_tiles % n_seqs == 0, alone = n_tiles < 2 * n_seqs;      // alone: sequences of one tile, nothing for two groups to share
    if (pairs * wgs_per_seq <= cus) {
        // Fewer pairs than CUs.  Short sequences, and narrow windows, whose walks are short as well: a tile each (32 sequences of 64 tokens 19 / 22 / 18, the older form
        // 23; one of 2,048 under a window of 512 47 / 38 / 34, 40), where the workgroups that leave do not crowd the others (the last of an odd number of pairs of
        // every sequence: eight of 200 26 / 22 / 27, behind 2,000 134 / 81 / 125); sequences of one tile: all of them at once, two workgroups a CU (eight of
        // 30 behind 2,000, 40 heads over 40, a pair / split / a tile each / this 124 / 78 / 119 / 74, 98)
        const bool spread = n_seqs == 1 || (equal && (a_seq == 2 || a_seq % 4 == 0)) || (n_tiles + n_seqs) * wgs_per_seq * 2 <= 3 * cus;
        if (tokens < 320 && alone) return PF_ONE;
        return (tokens < 320 || (window > 0 && 3LL * window <= 2 * tokens)) && spread ? PF_EACH : PF_SPLIT_PAIRED;
    }
    // A workgroup with a tile a group takes two pairs of a sequence; the last of an odd number of them, and a pair of two sequences' middle tiles, one by
    // one.  Sequences of one length: that many workgroups, in whole rounds; of several: about the pairs' half (the short ones' fill the rounds).
    double rounds = 0.5 * (double)(pairs * wgs_per_seq) / (double)cus + 0.1;
    if (equal) {
        rounds = (double)((n_seqs * ((a_seq / 2 + 1) / 2) + (a_seq % 2 * n_seqs) / 2) * wgs_per_seq) / (double)cus;
        rounds = rounds <= 4.0 ? std::ceil(rounds) : rounds + 0.35;
    }
    // Short sequences (by their new tokens): a tile each in one round, and of two tiles each, whose workgroups leave nobody out (16 of 200, 40 heads over 40, 52 / 69 / 55,
    // behind 2,000 346 / 286 / 234); else two workgroups a CU (16 of 200, 32 over 8, 29 / 41 / 42)
    if (tokens < 640) return !alone && !one && (rounds <= 1.0 || (equal && a_seq == 2)) ? PF_EACH_PAIRED : PF_ONE_PAIRED;
    if (!one) return rounds <= 1.0 ? PF_EACH_PAIRED : PF_SPLIT_PAIRED;
    // Beside the one group's rounds (of two workgroups a CU; a partial one is dearer than its share) one of these takes the less the longer the walk
    double ones = (double)wgs / (double)(2 * cus);
    if (std::fabs(ones - std::round(ones)) > 0.1) ones += 0.2;
    const double walk = window > 0 && window < tokens ? (double)window : (double)tokens;
    return walk >= 1000.0 && rounds * (0.74 + 200.0 / walk) <= 0.97 * ones ? PF_EACH_PAIRED : PF_ONE_PAIRED;
}

static int attn_mfma_launch(const void* q, int q_stride, void* out, int out_stride, const void* k_pages,
                            const void* vt_pages, const int* block_table, int bt_stride, const int* seq_lens,
                            const int* tiles, int n_tiles, int n_tokens, int H, int Hkv, int hs, int GT,
                            int window, float scale, int n_splits, int chunk, float* part_o, float* part_ml,
                            const float* inv_freq, int rotate, int write_kv, const int* by_length,
                            const int* max_len, const float* row_ssq, int n_pieces, int ssq_width, float ssq_eps, int n_seqs,
                            hipStream_t s) {
    if (!bn_attn_mfma_supports(hs) || n_tiles <= 0 || n_tokens <= 0 || H <= 0 || Hkv <= 0 || H % Hkv) return BN_ERR_ARG;
    if (row_ssq && (tiles || !rotate || n_pieces < 1 || n_pieces > 64 || ssq_width < 1)) return BN_ERR_ARG;   // decode form, rotating
    if (GT <= 0 || GT > 16 || (GT & (GT - 1)) || window < 0 || n_splits < 1 || n_splits > 64) return BN_ERR_ARG;
    if (tiles && n_seqs < 1) return BN_ERR_ARG;
    if (n_splits > 1 && (!part_o || !part_ml || (!max_len && (chunk <= 0 || chunk % BN_PAGE)))) return BN_ERR_ARG;
    if (!tiles && (!seq_lens || bt_stride < 1)) return BN_ERR_ARG;      // the decode form reads a row's first entry unasked
    if (max_len && tiles) return BN_ERR_ARG;                               // decode form only
    if (q_stride % 8 || out_stride % 4 || (((uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)vt_pages) & 15) ||
        ((uintptr_t)out & 7))
        return BN_ERR_ARG;
    const int G = H / Hkv;
    const int n_head_tiles = (G + GT - 1) / GT;
    if ((rotate || write_kv) && tiles) return BN_ERR_ARG;                 // decode form only
    if (rotate && !inv_freq) return BN_ERR_ARG;
    if (write_kv && (n_head_tiles != 1 || q_stride < (H + 2 * Hkv) * hs)) return BN_ERR_ARG;
    MfmaArgs a;
    a.q = (const bf16*)q; a.out = (bf16*)out; a.k_pages = (const bf16*)k_pages; a.vt_pages = (const bf16*)vt_pages;
    a.block_table = block_table; a.seq_lens = seq_lens; a.tiles = tiles; a.part_o = part_o; a.part_ml = part_ml;
    a.q_stride = q_stride; a.out_stride = out_stride; a.bt_stride = bt_stride;
    a.H = H; a.Hkv = Hkv; a.GT = GT; a.window = window; a.scale = scale;
    a.n_splits = n_splits; a.chunk = n_splits > 1 ? chunk : 0x40000000;
    a.inv_freq = inv_freq; a.rotate = rotate; a.write_kv = write_kv;
    a.row_ssq = row_ssq; a.n_pieces = n_pieces; a.inv_ssq_width = row_ssq ? 1.0f / (float)ssq_width : 0.f; a.ssq_eps = ssq_eps;
    a.max_len = n_splits > 1 ? max_len : nullptr;
    // the order matters only when the launch holds more workgroups than CUs and no sequence is split
    const int wgs_per_seq = Hkv * n_head_tiles;
    a.by_length = (!tiles && n_splits == 1 && (long long)n_tiles * wgs_per_seq > compute_units()) ? by_length : nullptr;
    a.order_period = compute_units() / wgs_per_seq;
    if (tiles) {
        const int form = prompt_form(n_tiles, n_tokens, n_seqs, wgs_per_seq, hs, window);
        const long long pairs = (n_tiles + 1LL) / 2;
        const int paired = form == PF_ONE_PAIRED || form == PF_SPLIT_PAIRED || form == PF_TWO_PAIRED || form == PF_EACH_PAIRED;
        const long long wgs = (form == PF_EACH ? 2 * pairs : paired ? pairs : n_tiles) * wgs_per_seq;
        if (wgs > 0x7fffffff) return BN_ERR_ARG;
        auto go = [&](auto kernel, int which, int ng) {
            // three staged blocks of 32 keys a group with their values: up to 96 KB, beyond the default limit of dynamic shared memory
            const size_t smem = (size_t)PROMPT_BUFFERS * (32 * ng * hs + hs * 32 * ng) * 2;
            static bool raised[3] = {false, false, false};
            if (!raised[which]) {
                const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                         hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
                if (e != hipSuccess) return (int)e;
                raised[which] = true;
            }
            hipLaunchKernelGGL(kernel, dim3((unsigned)wgs), dim3(256 * ng), smem, s, a, n_tiles, paired);
            return bn_launch_status();
        };
        if (form == PF_TWO || form == PF_TWO_PAIRED) return go(attn_mfma_prompt_kernel<64, 4, 2>, 0, 2);
        if (form == PF_ONE || form == PF_ONE_PAIRED) return hs == 64 ? go(attn_mfma_prompt_kernel<64, 4, 1>, 1, 1) : go(attn_mfma_prompt_kernel<128, 2, 1>, 2, 1);
        if (form == PF_SPLIT || form == PF_SPLIT_PAIRED)
            hipLaunchKernelGGL((attn_mfma_turns_kernel<128, 2, true>), dim3((unsigned)wgs), dim3(512), 0, s, a, n_tiles, paired);
        else                                             // (half of the workgroups find that another has taken their pair along)
            hipLaunchKernelGGL((attn_mfma_turns_kernel<128, 2, false>), dim3((unsigned)wgs), dim3(512), 0, s, a, n_tiles, paired);
        return bn_launch_status();
    }
    if (n_tiles > 65535) return BN_ERR_ARG;                 // sequences are the grid's y
    // Two splits and no more workgroups than CUs: both in one workgroup, without a launch for the merge (WHOLE).  us, merged by a
    // kernel -> whole: 8B heads, one sequence of 253 keys 9.0 -> 6.2, three of 317 10.2 -> 7.6, 16 of 381 12.2 -> 9.3, of 573 14.3 ->
    // 11.9, of 1,021 19.0 -> 17.5, 31 of 573 19.7 -> 16.2; 16 heads over one row, 128 of 573 17.7 -> 14.4.  Up to 16 pages: with sequences
    // of unequal lengths (16 to 64 a page) and half as many workgroups as CUs 16 pages 16.1 -> 15.8, 20 pages 17.4 -> 17.8, 24 pages 18.9
    // -> 20.1 (a long sequence has one CU, not two).  Three and four splits a workgroup, two after two: 8 pages 9.3 -> 10.2, 9 pages
    // 10.4 -> 10.8, not taken.
    const bool whole = n_splits == 2 && window == 0 && bt_stride <= AD_WHOLE_PAGES && (long long)n_tiles * wgs_per_seq <= compute_units();
    auto go = [&](auto kernel, int which) {
        const size_t smem = (size_t)(whole ? 8 : 4) * hs * (GT + 1) * sizeof(float);
        static bool raised[8] = {false, false, false, false, false, false, false, false};
        if (smem > 48 * 1024 && !raised[which]) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 144 * 1024);
            if (e != hipSuccess) return (int)e;
            raised[which] = true;
        }
        hipLaunchKernelGGL(kernel, dim3(Hkv * n_head_tiles, n_tiles, whole ? 1 : n_splits), dim3(whole ? 512 : 256), smem, s, a);
        return bn_launch_status();
    };
    // Keys that many workgroups read (of more than 64 heads over one kv head) are read plainly, others non-temporally.  us, plain /
    // non-temporal, over memory that no cache holds: 8B heads, one sequence of 2,000 10.6 / 9.7, 16 of 2,000 32.2 / 28.4; 32 heads over one
    // (two workgroups) one of 2,000 12.0 / 11.4, 64 over one 16 of 500 13.6 / 12.9, of 2,000 19.8 / 20.1; 128 over one one of 500 10.6 /
    // 11.6, 16 of 2,000 29.0 / 31.7.
    auto pick = [&](auto w, auto once) {
        constexpr bool W = decltype(w)::value, O = decltype(once)::value;
        return hs == 64 ? go(attn_mfma_decode_kernel<64, W, O>, 2 * W + 4 * O) : go(attn_mfma_decode_kernel<128, W, O>, 1 + 2 * W + 4 * O);
    };
    const bool once = n_head_tiles <= 4;
    if (whole) return once ? pick(std::true_type(), std::true_type()) : pick(std::true_type(), std::false_type());
    const int rc = once ? pick(std::false_type(), std::true_type()) : pick(std::false_type(), std::false_type());
    if (rc != 0 || n_splits == 1) return rc;
    auto combine = [&](auto most) {
        constexpr int S = decltype(most)::value;
        auto kernel = hs == 64 ? attn_mfma_combine_kernel<S, 1> : attn_mfma_combine_kernel<S, 2>;
        hipLaunchKernelGGL(kernel, dim3(n_tokens * H), dim3(64), 0, s, (bf16*)out, out_stride, part_o, part_ml, H, n_splits);
        return bn_launch_status();
    };
    if (n_splits <= 4) return combine(std::integral_constant<int, 4>());
    if (n_splits <= 8) return combine(std::integral_constant<int, 8>());
    if (n_splits <= 16) return combine(std::integral_constant<int, 16>());
    if (n_splits <= 32) return combine(std::integral_constant<int, 32>());
    return combine(std::integral_constant<int, 64>());
}

extern "C" int bn_attn_mfma(const void* q, int q_stride, void* out, int out_stride, const void* k_pages,
                            const void* vt_pages, const int* block_table, int bt_stride, const int* seq_lens,
                            const int* tiles, int n_tiles, int n_tokens, int H, int Hkv, int hs, int GT,
                            int window, float scale, int n_splits, int chunk, float* part_o, float* part_ml,
                            const float* inv_freq, int rotate, int write_kv, const int* by_length,
                            const int* max_len, hipStream_t s) {
    return attn_mfma_launch(q, q_stride, out, out_stride, k_pages, vt_pages, block_table, bt_stride, seq_lens, tiles, n_tiles,
                            n_tokens, H, Hkv, hs, GT, window, scale, n_splits, chunk, part_o, part_ml, inv_freq, rotate,
                            write_kv, by_length, max_len, nullptr, 0, 0, 0.f, 1, s);
}

// the prompt form by a caller who knows how many sequences the tiles are of (above: one): the choice among its kernels asks for it
extern "C" int bn_attn_mfma_prompt(const void* q, int q_stride, void* out, int out_stride, const void* k_pages,
                                   const void* vt_pages, const int* block_table, int bt_stride, const int* tiles, int n_tiles,
                                   int n_tokens, int H, int Hkv, int hs, int GT, int window, float scale, int n_seqs, hipStream_t s) {
    if (!tiles) return BN_ERR_ARG;
    return attn_mfma_launch(q, q_stride, out, out_stride, k_pages, vt_pages, block_table, bt_stride, nullptr, tiles, n_tiles,
                            n_tokens, H, Hkv, hs, GT, window, scale, 1, 0, nullptr, nullptr, nullptr, 0, 0, nullptr, nullptr,
                            nullptr, 0, 0, 0.f, n_seqs, s);
}

// the number of that choice (PF_*)
extern "C" int bn_attn_mfma_prompt_form(int n_tiles, int n_tokens, int n_seqs, int H, int Hkv, int hs, int GT, int window) {
    if (!bn_attn_mfma_supports(hs) || n_tiles < 1 || n_tokens < 1 || n_seqs < 1 || H < 1 || Hkv < 1 || H % Hkv || GT < 1) return -1;
    return prompt_form(n_tiles, n_tokens, n_seqs, (long long)Hkv * ((H / Hkv + GT - 1) / GT), hs, window);
}

// The decode form (tiles none, rotate on) over rows whose RMSNorm was left undone: q, the new key and the new value of
// row b still lack the factor 1/sqrt(sum of row_ssq[b][0..n_pieces) / ssq_width + eps), which is applied here.
extern "C" int bn_attn_mfma_scaled(const void* q, int q_stride, void* out, int out_stride, const void* k_pages,
                                   const void* vt_pages, const int* block_table, int bt_stride, const int* seq_lens,
                                   int n_seqs, int H, int Hkv, int hs, int GT, int window, float scale, int n_splits,
                                   int chunk, float* part_o, float* part_ml, const float* inv_freq, int write_kv,
                                   const int* by_length, const int* max_len, const float* row_ssq, int n_pieces,
                                   int ssq_width, float ssq_eps, hipStream_t s) {
    if (!row_ssq) return BN_ERR_ARG;
    return attn_mfma_launch(q, q_stride, out, out_stride, k_pages, vt_pages, block_table, bt_stride, seq_lens, nullptr, n_seqs,
                            n_seqs, H, Hkv, hs, GT, window, scale, n_splits, chunk, part_o, part_ml, inv_freq, 1, write_kv,
                            by_length, max_len, row_ssq, n_pieces, ssq_width, ssq_eps, n_seqs, s);
}

// ---------------------------------------------------------------------------------------
// decode form for callers that cannot allocate (declared and described in attn_mfma.h)
// ---------------------------------------------------------------------------------------
// The split partials of bn_attn_mfma_decode_static.  In host code this name is a stand-in, not a device
// address: the address on the current GPU comes from hipGetSymbolAddress, once per device, and only that
// pointer is ever handed to a kernel.
static __device__ __align__(256) float scratch[BN_ATTN_STATIC_SCRATCH_FLOATS];

static int static_scratch(float** ptr) {
    static std::mutex lock;
    static float* per_device[64] = {nullptr};         // each GPU holds its own copy of the array at its own address
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= 64) return BN_ERR_ARG;
    std::lock_guard<std::mutex> hold(lock);
    if (per_device[dev] == nullptr) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return (int)e;
        if (p == nullptr) return (int)hipErrorInvalidSymbol;
        per_device[dev] = static_cast<float*>(p);
    }
    *ptr = per_device[dev];
    return 0;
}

extern "C" int bn_attn_mfma_decode_static(const void* q, int q_stride, void* out, int out_stride, const void* k_pages,
                                          const void* vt_pages, const int* block_table, int bt_stride,
                                          const int* seq_lens, int n_seqs, int H, int Hkv, int hs, int GT, int window,
                                          float scale, int n_splits, int chunk, const float* inv_freq, int rotate,
                                          int write_kv, const int* by_length, hipStream_t s) {
    if (!seq_lens || n_seqs <= 0 || H <= 0 || n_splits < 1 || n_splits > 64 || !bn_attn_mfma_supports(hs)) return BN_ERR_ARG;
    float* part_o = nullptr;
    float* part_ml = nullptr;
    if (n_splits > 1) {
        const unsigned long long rows = (unsigned long long)n_seqs * (unsigned)H * (unsigned)n_splits;
        if (rows * (unsigned)(hs + 2) > BN_ATTN_STATIC_SCRATCH_FLOATS) return BN_ERR_SCRATCH;
        float* base = nullptr;
        const int rc = static_scratch(&base);
        if (rc != 0) return rc;
        part_o = base;                                // [rows, hs]
        part_ml = base + rows * (unsigned)hs;         // [rows, 2]
    }
    return bn_attn_mfma(q, q_stride, out, out_stride, k_pages, vt_pages, block_table, bt_stride, seq_lens, nullptr,
                        n_seqs, n_seqs, H, Hkv, hs, GT, window, scale, n_splits, chunk, part_o, part_ml, inv_freq, rotate,
                        write_kv, by_length, nullptr, s);
}
