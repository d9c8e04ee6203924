// Causal attention over a float32 cache on the float32 matrix instruction (v_mfma_f32_16x16x4_f32: float32 products and
// sums): the plain form, pages with a row per position, no window, bias or sink, head sizes 16, 32, 64 and 128.  What has
// any of those, and every other head size, is attn_rows.hip's.
//
// Formulas (reference): kv head of head h is h / (H / Hkv) (src/transformer/gqa_scalar.c:77); score = (q.k) * scale
// (gqa_scalar.c:92-93); only keys at positions <= the query's (gqa_scalar.c:69,80); softmax by max-subtract and exp, out =
// sum_t p_t V_t (gqa_scalar.c:104-119).
//
// A wave owns 16 rows (query tokens x heads that share a kv head) as the columns of its tiles: S^T = K Q^T, and the lane's
// four scores of a tile of 16 keys are, as they lie, the operand of O^T = V^T P^T.
//
// One order of summation, whoever computes a row: a page of 64 keys is summed by itself from nothing (its maximum, its
// exponentials' sum, its values' sum); the pages of a run of 256 positions are folded in order from nothing; the runs are
// folded in order.  The prompt form walks a row's pages and folds as it goes; the decode form gives every page (or, for so many rows
// that the pages' sums would not have the room, every run) a workgroup, and a small kernel folds them: the same bits (float32
// logits do not depend on how a sequence was cut into steps).
//
// The prompt form is bound by the instruction (a page is 8,192 cycles of a SIMD for a wave of 16 rows x 128): a workgroup of 4
// waves shares the staged page, two workgroups a CU stage and multiply in turn.  Eight prompts of 64 to 1,024 tokens, 16
// heads of 128 over 4: 0.31 ms a layer (2.70 in attn_rows.hip).
#include "common.h"
#include <math.h>

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define AF_RUN_PAGES 4
#define AF_PARTS_BYTES (64ll << 20)
#define AF_SCRATCH_BYTES (128ll << 20)
#define AF_GROUPS 2048

struct AfArgs {
    const float* q;           // [n_tokens, q_stride], head h at h * hs, rotated (unless inv_freq says that the kernel does it)
    float* out;               // [n_tokens, out_stride]
    const float* k_pages;     // [n_pages, Hkv, BN_PAGE, hs]
    const float* v_pages;
    const int* block_table;   // [n_seqs, bt_stride]
    const int* seq_lens;      // decode form: keys in the cache, the new one included
    const int* tiles;         // prompt form: [n, 4] = sequence, first token row, tokens, position of the first
    float* part_o;            // [rows at once * H, n_parts, hs] (n_parts > 1)
    float* part_ml;           // [rows at once * H, n_parts, 2]
    int q_stride, out_stride, bt_stride, H, Hkv;
    int GT;                   // heads of a kv group handled together (a power of two <= 16)
    int n_parts, part_pages;  // decode form: parts that the block table can hold, and a part's pages (1 or AF_RUN_PAGES)
    float scale;
    const float* inv_freq;    // decode form: not null: q and the new key are rotated here, angle position * inv_freq[i], pairs (i, i + hs / 2)
    int write;                // decode form: the new key and value (behind q in its row) are stored at position seq_lens - 1
    float* k_new;             // k_pages and v_pages, to write
    float* v_new;
};

// The fold of (m, l, o) into (M, L, O), its operations written out (no contraction left to the compiler): the same parts give
// the same bits wherever they are folded.
__device__ __forceinline__ void af_factors(float M, float m, float& m2, float& fa, float& fb) {
    m2 = fmaxf(M, m);
    fa = expf(M - m2);                            // 0 when nothing was there before (M = -inf)
    fb = expf(m - m2);
}
__device__ __forceinline__ float af_fold(float O, float fa, float o, float fb) { return __fmaf_rn(O, fa, __fmul_rn(o, fb)); }

// How a head's dimensions lie over the tiles of the second product: V values are read VW at a time, tile (h, i) holds the
// dimensions 16 VW h + VW * (row of the tile) + i.
template <int HS> struct AfShape {
    static constexpr int NB = HS / 16;            // 16-byte groups of a key that a lane reads
    static constexpr int VW = HS >= 64 ? 4 : HS / 16;
    static constexpr int NH = HS / (16 * VW);
};

template <int HS> struct AfSums {                 // a lane's sums of its row (replicated over the four lanes that share it but for o)
    float m, l;
    f32x4 o[AfShape<HS>::NH][AfShape<HS>::VW];
    __device__ __forceinline__ void clear() {
        m = -INFINITY; l = 0.f;
#pragma unroll
        for (int h = 0; h < AfShape<HS>::NH; ++h)
#pragma unroll
            for (int i = 0; i < AfShape<HS>::VW; ++i) o[h][i] = 0.f;
    }
    __device__ __forceinline__ void fold(const AfSums& p) {
        if (p.l == 0.f) return;                   // a part of which this row saw no key changes nothing (one whose scores are all NaN does)
        float m2, fa, fb;
        af_factors(m, p.m, m2, fa, fb);
        l = af_fold(l, fa, p.l, fb);
        m = m2;
#pragma unroll
        for (int h = 0; h < AfShape<HS>::NH; ++h)
#pragma unroll
            for (int i = 0; i < AfShape<HS>::VW; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) o[h][i][j] = af_fold(o[h][i][j], fa, p.o[h][i][j], fb);
    }
};

// the larger of, and the sum with, the value of the lane 16 or 32 away
template <int O> __device__ __forceinline__ float af_pair_max(float v) {
    return bn_pair_far<O>(v, [](float a, float b) { return fmaxf(a, b); });
}
template <int O> __device__ __forceinline__ float af_pair_sum(float v) {
    return bn_pair_far<O>(v, [](float a, float b) { return __fadd_rn(a, b); });
}

// One page of keys from nothing.  k(t, b): the lane's 16 bytes of key 16 t + lane % 16, dimensions 16 b + 4 g ..; v(t, e, h):
// its VW values of key 16 t + 4 g + e; last: the last key of the page that the lane's row sees (63: all, < 0: none).
template <int HS, typename KF, typename VF>
__device__ __forceinline__ void af_page(const f32x4 (&q)[HS / 16], float scale, int last, bool masked, KF k, VF v, AfSums<HS>& p) {
    using S = AfShape<HS>;
    const int g = (threadIdx.x & 63) >> 4;
    f32x4 s[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        s[t] = 0.f;
#pragma unroll
        for (int b = 0; b < S::NB; ++b) {
            const f32x4 kf = k(t, b);
#pragma unroll
            for (int e = 0; e < 4; ++e) s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[e], q[b][e], s[t], 0, 0, 0);
        }
    }
    float m = -INFINITY;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            s[t][e] = masked && 16 * t + 4 * g + e > last ? -INFINITY : __fmul_rn(s[t][e], scale);
            m = fmaxf(m, s[t][e]);
        }
    m = af_pair_max<16>(m);
    m = af_pair_max<32>(m);
    const float base = m == -INFINITY ? 0.f : m;  // a row that sees no key of the page: every exponential is 0
    float l = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) { s[t][e] = expf(__fsub_rn(s[t][e], base)); l = __fadd_rn(l, s[t][e]); }
    l = af_pair_sum<16>(l);
    l = af_pair_sum<32>(l);
    p.clear();
    p.m = m; p.l = l;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int h = 0; h < S::NH; ++h) {
                float vf[S::VW];
                v(t, e, h, vf);
#pragma unroll
                for (int i = 0; i < S::VW; ++i) p.o[h][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i], s[t][e], p.o[h][i], 0, 0, 0);
            }
}

template <int VW> __device__ __forceinline__ void af_values(const float* p, float (&v)[VW]) {
    if (VW == 4) { const f32x4 t = *reinterpret_cast<const f32x4*>(p); v[0] = t[0]; v[1 % VW] = t[1]; v[2 % VW] = t[2]; v[3 % VW] = t[3]; }
    else if (VW == 2) { const float2 t = *reinterpret_cast<const float2*>(p); v[0] = t.x; v[1 % VW] = t.y; }
    else v[0] = *p;
}

template <int HS>
__global__ __launch_bounds__(256, 2) void attn_f32_prompt_kernel(AfArgs a) {
    using S = AfShape<HS>;
    constexpr int STRIDE = HS + 4;                // of a staged row: the rows that 16 lanes read together fall on different banks
    __shared__ __align__(16) float ks[BN_PAGE * STRIDE];
    __shared__ __align__(16) float vs[BN_PAGE * STRIDE];
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int GT = a.GT, G = a.H / a.Hkv, per_wave = 16 / GT;
    const int head_tiles = (G + GT - 1) / GT;
    const int kvh = blockIdx.y / head_tiles, ht = blockIdx.y - kvh * head_tiles;
    const int* tl = a.tiles + 4 * blockIdx.x;
    const int seq = tl[0], tok0 = tl[1], n_tok = min(tl[2], 4 * per_wave), pos0 = tl[3];
    if (n_tok <= 0 || pos0 < 0) return;           // a tile of no rows
    const int hi = pos0 + n_tok;
    const int tok = wave * per_wave + r / GT, hg = ht * GT + r % GT, head = kvh * G + hg;
    const bool live = tok < n_tok && hg < G;
    const int qpos = live ? pos0 + tok : -1;
    const int wave_last = pos0 + min(n_tok, (wave + 1) * per_wave) - 1;      // the wave's last query; below: it has none
    const bool wave_live = wave * per_wave < n_tok;
    f32x4 q[S::NB];
#pragma unroll
    for (int b = 0; b < S::NB; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            q[b][e] = live ? a.q[(size_t)(tok0 + tok) * a.q_stride + (size_t)head * HS + 16 * b + 4 * g + e] : 0.f;
    AfSums<HS> run, tot;
    run.clear();
    tot.clear();
    for (int j0 = 0; j0 < hi; j0 += BN_PAGE) {
        const int page = a.block_table[(size_t)seq * a.bt_stride + j0 / BN_PAGE];
        const float* kg = a.k_pages + ((size_t)page * a.Hkv + kvh) * BN_PAGE * HS;
        const float* vg = a.v_pages + ((size_t)page * a.Hkv + kvh) * BN_PAGE * HS;
        constexpr int GROUPS = BN_PAGE * HS / 4 / 256;
        f32x4 kr[GROUPS], vr[GROUPS];
#pragma unroll
        for (int i = 0; i < GROUPS; ++i) {        // rows that are not written yet are staged as zeros
            const int at = 4 * (tid + 256 * i);
            const bool in = j0 + at / HS < hi;
            kr[i] = *reinterpret_cast<const f32x4*>(kg + (in ? at : 0));
            vr[i] = *reinterpret_cast<const f32x4*>(vg + (in ? at : 0));
            if (!in) { kr[i] = 0.f; vr[i] = 0.f; }
        }
        __syncthreads();                          // the page before has been read
#pragma unroll
        for (int i = 0; i < GROUPS; ++i) {
            const int at = 4 * (tid + 256 * i), row = at / HS, d = at % HS;
            *reinterpret_cast<f32x4*>(&ks[row * STRIDE + d]) = kr[i];
            *reinterpret_cast<f32x4*>(&vs[row * STRIDE + d]) = vr[i];
        }
        __syncthreads();
        if (wave_live && j0 <= wave_last) {
            AfSums<HS> p;
            af_page<HS>(q, a.scale, qpos - j0, j0 + BN_PAGE > pos0 + wave * per_wave,
                        [&](int t, int b) { return *reinterpret_cast<const f32x4*>(&ks[(16 * t + r) * STRIDE + 16 * b + 4 * g]); },
                        [&](int t, int e, int h, float (&v)[S::VW]) { af_values<S::VW>(&vs[(16 * t + 4 * g + e) * STRIDE + 16 * S::VW * h + S::VW * r], v); },
                        p);
            run.fold(p);
            if ((j0 / BN_PAGE) % AF_RUN_PAGES == AF_RUN_PAGES - 1) { tot.fold(run); run.clear(); }
        }
    }
    tot.fold(run);
    if (!live) return;
    const float inv = tot.l > 0.f ? 1.0f / tot.l : 0.f;
    float* o = a.out + (size_t)(tok0 + tok) * a.out_stride + (size_t)head * HS;
#pragma unroll
    for (int h = 0; h < S::NH; ++h)
#pragma unroll
        for (int i = 0; i < S::VW; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) o[16 * S::VW * h + S::VW * (4 * g + j) + i] = __fmul_rn(tot.o[h][i][j], inv);
}

// A workgroup of 4 waves takes a part of a sequence's keys, one page or the pages of a run in turn: wave t of it multiplies the keys 16 t .. 16 t + 15 with the
// queries, then, with the page's scores exchanged through shared memory, the weights with a quarter of the value's dimensions.
// Everything of a page is asked for at once, keys as they lie (their operand comes through shared memory: sixteen rows in sixteen
// lanes of a load would cost four times the cycles).  inv_freq: the query and the new key arrive unrotated; write: the workgroup
// that holds the new position stores the new key and value into the pages, and reads them from the token's row itself.  The order
// of every sum is the prompt form's (af_page).  What bounds it is how fast a CU can draw its keys and values (some 25 bytes a
// nanosecond), and, in a table much wider than its sequences, how fast workgroups without keys end: they ask for nothing but a
// length.  us with the fold, 16 heads of 128 over 4, rotation and store inside, in a table of its own width / of 8,192 positions /
// of 131,072 (in brackets: with every workgroup staging its queries first, and the pages of a run in 16 waves of one workgroup):
// one sequence of 200 keys 10.2 / 10.2 / 10.2 (10.1 / 10.2 / 30.3), 64 of 200 23.8 / 31.0 / 31.3 (22.7 / 100 / 100), 64 of 1,000
// 62.7 / 64.9 / 65.1 (65.6 / 154 / 155), eight of 2,000 26.1 / 25.8 / 29.5 (25.6 / 33 / 98).
template <int HS, int PAGES>
__global__ __launch_bounds__(256, PAGES == 1 ? 3 : 2) void attn_f32_decode_kernel(AfArgs a) {
    constexpr int NB = HS / 16, STRIDE = HS + 4, HALF = HS / 2;
    constexpr int VW = HS >= 64 ? HS / 64 : 1;    // tiles of the second product a wave: value dimensions 16 VW part + VW row + tile
    constexpr int PARTS = HS / (16 * VW);         // waves of a page that have any
    constexpr int OWN = HS / 16;                  // the sums that a thread folds: (head, dimension) number tid + 256 o
    __shared__ __align__(16) float ks[4 * 16 * STRIDE];      // every wave's keys; later [16][HS + 1], the page's sums
    __shared__ __align__(16) float sx[4 * 64 * 4];           // the page's scores, as the lanes hold them
    __shared__ __align__(16) float qs[16 * STRIDE];          // the queries
    __shared__ __align__(16) float kn[HS];                   // the new key
    __shared__ float cos_s[HALF], sin_s[HALF];
    __shared__ float sm[16], sl[16];
    float* so = ks;
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int t = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int GT = a.GT, G = a.H / a.Hkv;
    const int head_tiles = (G + GT - 1) / GT;
    const int kvh = blockIdx.y / head_tiles, ht = blockIdx.y - kvh * head_tiles;
    const int tok = blockIdx.x, len = a.seq_lens[tok];
    constexpr int part_keys = PAGES * BN_PAGE;
    const int rows = min(GT, G - ht * GT);
    const float* row = a.q + (size_t)tok * a.q_stride;
    const float* new_v = row + (size_t)(a.H + a.Hkv + kvh) * HS;
    // the queries (rows without a head as zeros) and the new key, a pair of dimensions a thread
    constexpr int PAIRS = (17 * HALF + 255) / 256;
    float x0[PAIRS], x1[PAIRS];
#pragma unroll
    for (int p = 0; p < PAIRS; ++p) {
        const int idx = min(tid + 256 * p, 17 * HALF - 1), h = idx / HALF, i = idx - h * HALF;
        const float* src = row + (size_t)(h == 16 && a.write ? a.H + kvh : kvh * G + ht * GT + min(h, rows - 1)) * HS + i;
        x0[p] = src[0];
        x1[p] = src[HALF];
    }
    // A table is as wide as the longest sequence there can be: most workgroups of a short one have no keys.  The loads above stay in
    // front of this, on their way while the length is waited for.
    asm volatile("" ::: "memory");
    if (blockIdx.z > 0 && (int)blockIdx.z * part_keys >= len) return;
    const float freq = a.inv_freq ? a.inv_freq[tid % HALF] : 0.f;
    // The queries and the new key into shared memory, once the first page's keys and values have been asked for: an angle's sine
    // and cosine are formed by one thread a pair of dimensions (17 heads turn by the same ones), and the barrier between leaves
    // the page on its way.  (One sequence of 200 keys, with the fold: 10.1 -> 9.8 us; eight of 2,000 28.4 -> 28.0.)
    auto turn = [&]() {
        if (a.inv_freq) {
            if (tid < HALF) sincosf((float)(len - 1) * freq, &sin_s[tid], &cos_s[tid]);
            bn_lds_barrier();
        }
#pragma unroll
        for (int p = 0; p < PAIRS; ++p) {
            const int idx = tid + 256 * p, h = idx / HALF, i = idx - h * HALF;
            if (idx >= 17 * HALF || (h == 16 && !a.write)) break;
            if (a.inv_freq) bn_rotate_pair(x0[p], x1[p], cos_s[i], sin_s[i]);
            if (h < 16 && h >= rows) x0[p] = x1[p] = 0.f;
            float* dst = h == 16 ? kn + i : qs + h * STRIDE + i;
            dst[0] = x0[p];
            dst[HALF] = x1[p];
        }
    };
    bool turned = false;
    for (int part = blockIdx.z; part < a.n_parts && (part == 0 || part * part_keys < len); part += gridDim.z) {
        float M[OWN], L[OWN], O[OWN];             // (of more pages than one)
#pragma unroll
        for (int o = 0; o < OWN; ++o) { M[o] = -INFINITY; L[o] = 0.f; O[o] = 0.f; }
#pragma unroll 1
        for (int j0 = part * part_keys; j0 < min((part + 1) * part_keys, len); j0 += BN_PAGE) {
            const int last = min(len - 1 - j0, BN_PAGE - 1);
            const bool newest = a.write && len - 1 - j0 < BN_PAGE;           // the page holds the new position: its row `last`
            f32x4 kr[NB];
            float vf[4][4][VW], nv[VW];
            const size_t at = ((size_t)a.block_table[(size_t)tok * a.bt_stride + j0 / BN_PAGE] * a.Hkv + kvh) * BN_PAGE * HS;
            const f32x4* kg = reinterpret_cast<const f32x4*>(a.k_pages + at + (size_t)16 * t * HS);
#pragma unroll
            for (int i = 0; i < NB; ++i) kr[i] = kg[lane + 64 * i];
            const float* vbase = a.v_pages + at + (4 * g * HS + 16 * VW * t + VW * r);
            if (t < PARTS) {
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int e = 0; e < 4; ++e) af_values<VW>(vbase + (16 * u + e) * HS, vf[u][e]);
                if (newest) af_values<VW>(new_v + 16 * VW * t + VW * r, nv);
            }
            if (!turned) turn();
            turned = true;
            __syncthreads();                      // the queries and the new key are there; the sums of the page before have been read
            float* mine = ks + t * 16 * STRIDE;
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int piece = lane + 64 * i, key = piece / (HS / 4), d = 4 * (piece % (HS / 4));
                if (newest && 16 * t + key == last) kr[i] = *reinterpret_cast<const f32x4*>(kn + d);
                *reinterpret_cast<f32x4*>(mine + key * STRIDE + d) = kr[i];
            }
            if (newest && ht == 0 && t == 0) {    // the new position's rows of the pages, by a wave
                float* kd = a.k_new + at + (size_t)last * HS;
                float* vd = a.v_new + at + (size_t)last * HS;
                for (int d = lane; d < HS; d += 64) { kd[d] = kn[d]; vd[d] = new_v[d]; }
            }
            __builtin_amdgcn_wave_barrier();      // a wave's own keys: its shared-memory operations run in order
            {
                f32x4 s = 0.f;
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const f32x4 kf = *reinterpret_cast<const f32x4*>(mine + r * STRIDE + 16 * b + 4 * g);
                    const f32x4 qf = *reinterpret_cast<const f32x4*>(qs + r * STRIDE + 16 * b + 4 * g);
#pragma unroll
                    for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[e], qf[e], s, 0, 0, 0);
                }
                *reinterpret_cast<f32x4*>(sx + (t * 64 + lane) * 4) = s;
            }
            __syncthreads();
            if (t < PARTS) {
                f32x4 s[4];
                float m = -INFINITY, l = 0.f;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    s[u] = *reinterpret_cast<const f32x4*>(sx + (u * 64 + lane) * 4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        s[u][e] = 16 * u + 4 * g + e > last ? -INFINITY : __fmul_rn(s[u][e], a.scale);
                        m = fmaxf(m, s[u][e]);
                    }
                }
                m = af_pair_max<16>(m);
                m = af_pair_max<32>(m);
                const float base = m == -INFINITY ? 0.f : m;
                f32x4 o[VW];
#pragma unroll
                for (int i = 0; i < VW; ++i) o[i] = 0.f;
                if (last < BN_PAGE - 1 || newest) {       // the new value comes from the token's row; rows behind the last key count as zeros
#pragma unroll
                    for (int u = 0; u < 4; ++u)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int key = 16 * u + 4 * g + e;
#pragma unroll
                            for (int i = 0; i < VW; ++i) vf[u][e][i] = key > last ? 0.f : key == last && newest ? nv[i] : vf[u][e][i];
                        }
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int e = 0; e < 4; ++e) { s[u][e] = expf(__fsub_rn(s[u][e], base)); l = __fadd_rn(l, s[u][e]); }
                l = af_pair_sum<16>(l);
                l = af_pair_sum<32>(l);
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int i = 0; i < VW; ++i) o[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[u][e][i], s[u][e], o[i], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < VW; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) so[r * (HS + 1) + 16 * VW * t + VW * (4 * g + j) + i] = o[i][j];
                if (t == 0 && g == 0) { sm[r] = m; sl[r] = l; }
            }
            __syncthreads();
            if (PAGES > 1)
#pragma unroll
                for (int o = 0; o < OWN; ++o) {
                    const int idx = tid + 256 * o, h = idx / HS, d = idx - h * HS;
                    if (h >= rows) break;
                    const float m = sm[h], l = sl[h];
                    if (l == 0.f) continue;
                    float m2, fa, fb;
                    af_factors(M[o], m, m2, fa, fb);
                    L[o] = af_fold(L[o], fa, l, fb);
                    O[o] = af_fold(O[o], fa, so[h * (HS + 1) + d], fb);
                    M[o] = m2;
                }
            // (the barrier behind the next page's loads stands before its keys are stored over the sums)
        }
        auto put = [&](int idx, float m, float l, float x) {
            const int h = idx / HS, d = idx - h * HS, head = kvh * G + ht * GT + h;
            if (a.n_parts == 1) {
                a.out[(size_t)tok * a.out_stride + (size_t)head * HS + d] = __fmul_rn(x, l > 0.f ? 1.0f / l : 0.f);
            } else {
                const size_t at = ((size_t)tok * a.H + head) * a.n_parts + part;
                a.part_o[at * HS + d] = x;
                if (d == 0) { a.part_ml[2 * at] = m; a.part_ml[2 * at + 1] = l; }
            }
        };
        if (PAGES == 1) {                         // a page alone: folded into nothing it is itself
            const bool none = len <= 0;
            for (int idx = tid; idx < rows * HS; idx += 256) {
                const int h = idx / HS;
                put(idx, none ? -INFINITY : sm[h], none ? 0.f : sl[h], none ? 0.f : so[h * (HS + 1) + idx - h * HS]);
            }
        } else {
#pragma unroll
            for (int o = 0; o < OWN; ++o)
                if (tid + 256 * o < rows * HS) put(tid + 256 * o, M[o], L[o], O[o]);
        }
    }
}

// The parts of a row in order: the per_run parts of a run from nothing (a group of 128 threads a run), then the runs.
__global__ __launch_bounds__(1024) void attn_f32_fold_kernel(AfArgs a, int hs, int per_run) {
    __shared__ float ro[8][128], rm[8], rl[8];
    const int row = blockIdx.x, tok = row / a.H, head = row - tok * a.H, d = threadIdx.x & 127;
    const int group = threadIdx.x >> 7, groups = blockDim.x >> 7;
    const int len = a.seq_lens[tok], runs = (len + AF_RUN_PAGES * BN_PAGE - 1) / (AF_RUN_PAGES * BN_PAGE);
    const int part_keys = AF_RUN_PAGES / per_run * BN_PAGE, parts = (len + part_keys - 1) / part_keys;
    const float* ml = a.part_ml + (size_t)row * a.n_parts * 2;
    const float* po = a.part_o + (size_t)row * a.n_parts * hs + min(d, hs - 1);
    float M = -INFINITY, L = 0.f, O = 0.f;
    for (int r0 = 0; r0 < runs; r0 += groups) {
        if (r0 + group < runs) {
            const int first = (r0 + group) * per_run;
            float m[AF_RUN_PAGES], l[AF_RUN_PAGES], o[AF_RUN_PAGES], RM = -INFINITY, RL = 0.f, RO = 0.f;
#pragma unroll
            for (int i = 0; i < AF_RUN_PAGES; ++i) {
                const int at = min(first + i, parts - 1);
                m[i] = ml[2 * at]; l[i] = ml[2 * at + 1]; o[i] = po[(size_t)at * hs];
            }
#pragma unroll
            for (int i = 0; i < AF_RUN_PAGES; ++i) {
                if (i >= per_run || first + i >= parts || l[i] == 0.f) continue;
                float m2, fa, fb;
                af_factors(RM, m[i], m2, fa, fb);
                RL = af_fold(RL, fa, l[i], fb);
                RO = af_fold(RO, fa, o[i], fb);
                RM = m2;
            }
            ro[group][d] = RO;
            if (d == 0) { rm[group] = RM; rl[group] = RL; }
        }
        __syncthreads();
        for (int i = 0; i < min(groups, runs - r0); ++i) {
            if (rl[i] == 0.f) continue;
            float m2, fa, fb;
            af_factors(M, rm[i], m2, fa, fb);
            L = af_fold(L, fa, rl[i], fb);
            O = af_fold(O, fa, ro[i][d], fb);
            M = m2;
        }
        __syncthreads();
    }
    if (group == 0 && d < hs) a.out[(size_t)tok * a.out_stride + (size_t)head * hs + d] = __fmul_rn(O, L > 0.f ? 1.0f / L : 0.f);
}

// Rows of a decode step that are taken at a time: as many as keep the partial sums (of n_parts parts a row) under
// AF_SCRATCH_BYTES, in turns of equal size; one row's at the least (with four heads a kv head under a hundredth of the keys and
// values that the row's table can hold in this layer).  The turns share one buffer, so a step's scratch does not grow with its
// rows, and a row's sums are the same in any turn.  Tables of 131,072 positions, 32 heads of 128 over 8, 64 / 256 sequences of 200
// keys: 126 / 516 us and 106 / 122 MB; in turns of 64 MB 235 / 991 us, of 256 MB 84 / 300; 64 rows at once 42 us and 520 MB (the
// vector kernel, whose parts are runs of 2,048 positions: 157 / 627 us and 65 / 260 MB).
static int af_rows_at_once(int n_seqs, int H, int n_parts, int hs) {
    if (n_parts <= 1) return n_seqs;
    const long long most = AF_SCRATCH_BYTES / ((long long)H * n_parts * (hs + 2) * 4);
    if (most >= n_seqs) return n_seqs;
    const int turns = most <= 1 ? n_seqs : (int)((n_seqs + most - 1) / most);
    return (n_seqs + turns - 1) / turns;
}

template <int HS>
static int af_launch(const AfArgs& a, int n_tiles, hipStream_t s) {
    const int G = a.H / a.Hkv, heads = a.Hkv * ((G + a.GT - 1) / a.GT);
    if (a.tiles) {
        hipLaunchKernelGGL(attn_f32_prompt_kernel<HS>, dim3(n_tiles, heads), dim3(256), 0, s, a);
        return bn_launch_status();
    }
    const int at_once = af_rows_at_once(n_tiles, a.H, a.n_parts, HS);
    const int per_run = AF_RUN_PAGES / a.part_pages, runs = (a.n_parts + per_run - 1) / per_run;
    for (int first = 0; first < n_tiles; first += at_once) {
        const int n = n_tiles - first < at_once ? n_tiles - first : at_once;
        AfArgs t = a;
        t.q += (size_t)first * a.q_stride;
        t.out += (size_t)first * a.out_stride;
        t.block_table += (size_t)first * a.bt_stride;
        t.seq_lens += first;
        // A workgroup a part up to some AF_GROUPS workgroups, of which a CU holds three of heads 128 wide; a longer table's parts
        // are taken in turn.  us with 8,192 / 2,048 / 768, 16 heads of 128 over 4: 64 sequences of 1,000 keys 67.6 / 62.7 / 54.9,
        // one of 8,000 beside 63 of 200 192 / 206 / 234, one of 100,000 275 / 278 / 269.
        int z = AF_GROUPS / (n * heads);
        z = z < 1 ? 1 : z > a.n_parts ? a.n_parts : z;
        if (a.part_pages == 1) hipLaunchKernelGGL((attn_f32_decode_kernel<HS, 1>), dim3(n, heads, z), dim3(256), 0, s, t);
        else hipLaunchKernelGGL((attn_f32_decode_kernel<HS, AF_RUN_PAGES>), dim3(n, heads, z), dim3(256), 0, s, t);
        if (int rc = bn_launch_status()) return rc;
        if (a.n_parts == 1) continue;
        hipLaunchKernelGGL(attn_f32_fold_kernel, dim3(n * a.H), dim3(128 * (runs < 8 ? runs : 8)), 0, s, t, HS, per_run);
        if (int rc = bn_launch_status()) return rc;
    }
    return 0;
}

extern "C" int bn_attn_f32_supports(int hs) { return hs == 16 || hs == 32 || hs == 64 || hs == 128; }
// Pages of a part of the decode form for a step of this many rows (n_seqs x heads) over tables of bt_stride pages: one, which spreads
// a sequence's keys over the most CUs (one sequence of 200 keys 8.9 us and the fold, a run a workgroup 18.6), while the partial sums
// stay under AF_PARTS_BYTES; then a run, whose sums take a quarter of the room.
extern "C" int bn_attn_f32_part_pages(long long rows, int bt_stride, int hs) {
    return rows * bt_stride * (hs + 2) * 4 <= AF_PARTS_BYTES ? 1 : AF_RUN_PAGES;
}

// Rows whose partial sums, of n_parts parts each, the caller gives room for.
extern "C" int bn_attn_f32_rows(int n_seqs, int H, int n_parts, int hs) { return af_rows_at_once(n_seqs, H, n_parts, hs); }

// tiles: the prompt form, tiles of up to 64 / GT tokens; null: the decode form, n_tiles sequences in parts of
// part_pages pages (1 or a run's), with partial sums of ceil(bt_stride / part_pages) parts a row if that is more than one, for
// bn_attn_f32_rows rows.  Decode form only: inv_freq
// [hs / 2], not null: q and the new key arrive unrotated; write: a row of q is [H + 2 Hkv heads], its new key and value are stored
// into the pages at position seq_lens - 1 (a row of no keys stores nothing).
extern "C" int bn_attn_f32(const void* q, int q_stride, void* out, int out_stride, const void* k_pages, const void* v_pages,
                           const int* block_table, int bt_stride, const int* seq_lens, const int* tiles, int n_tiles, int H, int Hkv,
                           int hs, int GT, float scale, int part_pages, float* part_o, float* part_ml, const float* inv_freq, int write,
                           hipStream_t s) {
    if (n_tiles <= 0 || n_tiles > 65535 * 128 || H <= 0 || Hkv <= 0 || H % Hkv || GT < 1 || GT > 16 || (GT & (GT - 1))) return BN_ERR_ARG;
    if (Hkv * ((H / Hkv + GT - 1) / GT) > 65535 || bt_stride < 1) return BN_ERR_ARG;
    if (tiles && (inv_freq || write)) return BN_ERR_ARG;
    if (write && (q_stride < (H + 2 * Hkv) * hs || q_stride % 2 || ((uintptr_t)q & 7))) return BN_ERR_ARG;
    if (!tiles && part_pages != 1 && part_pages != AF_RUN_PAGES) return BN_ERR_ARG;
    const int n_parts = tiles ? 1 : (bt_stride + part_pages - 1) / part_pages;
    if (!tiles && (!seq_lens || (n_parts > 1 && (!part_o || !part_ml)))) return BN_ERR_ARG;
    AfArgs a = {(const float*)q, (float*)out, (const float*)k_pages, (const float*)v_pages, block_table, seq_lens, tiles, part_o,
                part_ml, q_stride, out_stride, bt_stride, H, Hkv, GT, n_parts, part_pages, scale, inv_freq, write, (float*)k_pages, (float*)v_pages};
    switch (hs) {
        case 16: return af_launch<16>(a, n_tiles, s);
        case 32: return af_launch<32>(a, n_tiles, s);
        case 64: return af_launch<64>(a, n_tiles, s);
        case 128: return af_launch<128>(a, n_tiles, s);
    }
    return BN_ERR_ARG;
}
