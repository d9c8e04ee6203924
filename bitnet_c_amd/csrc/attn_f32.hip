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
// folded in order.  The prompt form walks a row's pages and folds as it goes; the decode form gives every page of a run a
// wave and every run a workgroup, and a small kernel folds the runs: the same bits (float32 logits do not depend on how a
// sequence was cut into steps).
//
// The prompt form is bound by the instruction (a page is 8,192 cycles of a SIMD for a wave of 16 rows x 128): a workgroup of 4
// waves shares the staged page, two workgroups a CU stage and multiply in turn.  Eight prompts of 64 to 1,024 tokens, 16
// heads of 128 over 4: 0.31 ms a layer (2.70 in attn_rows.hip).  The decode form is bound by latency: one page a wave, all its
// 64 KB asked for at once; the same eight sequences 20 us and 4 for the fold (243), one sequence of 200 keys 18 (58).
#include "common.h"
#include <math.h>

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define AF_RUN_PAGES 4

struct AfArgs {
    const float* q;           // [n_tokens, q_stride], head h at h * hs (already rotated)
    float* out;               // [n_tokens, out_stride]
    const float* k_pages;     // [n_pages, Hkv, BN_PAGE, hs]
    const float* v_pages;
    const int* block_table;   // [n_seqs, bt_stride]
    const int* seq_lens;      // decode form: keys in the cache, the new one included
    const int* tiles;         // prompt form: [n, 4] = sequence, first token row, tokens, position of the first
    float* part_o;            // [n_tokens * H, n_runs, hs] (n_runs > 1)
    float* part_ml;           // [n_tokens * H, n_runs, 2]
    int q_stride, out_stride, bt_stride, H, Hkv;
    int GT;                   // heads of a kv group handled together (a power of two <= 16)
    int n_runs;               // runs that the block table can hold
    float scale;
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
        if (p.m == -INFINITY) return;             // a part of which this row saw no key changes nothing
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
    m = fmaxf(m, __shfl_xor(m, 16, BN_WAVE));
    m = fmaxf(m, __shfl_xor(m, 32, BN_WAVE));
    const float base = m == -INFINITY ? 0.f : m;  // a row that sees no key of the page: every exponential is 0
    float l = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) { s[t][e] = expf(__fsub_rn(s[t][e], base)); l = __fadd_rn(l, s[t][e]); }
    l = __fadd_rn(l, __shfl_xor(l, 16, BN_WAVE));
    l = __fadd_rn(l, __shfl_xor(l, 32, BN_WAVE));
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

template <int HS>
__global__ __launch_bounds__(256, 1) void attn_f32_decode_kernel(AfArgs a) {
    using S = AfShape<HS>;
    __shared__ float so[AF_RUN_PAGES][16][HS + 1];
    __shared__ float sm[AF_RUN_PAGES][16], sl[AF_RUN_PAGES][16];
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int GT = a.GT, G = a.H / a.Hkv;
    const int head_tiles = (G + GT - 1) / GT;
    const int kvh = blockIdx.y / head_tiles, ht = blockIdx.y - kvh * head_tiles;
    const int tok = blockIdx.x, len = a.seq_lens[tok];
    const int rows = min(GT, G - ht * GT);
    const bool live = r < rows;
    const float* qp = a.q + (size_t)tok * a.q_stride + (size_t)(kvh * G + ht * GT + (live ? r : 0)) * HS + 4 * g;
    f32x4 q[S::NB];
#pragma unroll
    for (int b = 0; b < S::NB; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) q[b][e] = live ? qp[16 * b + e] : 0.f;
    for (int run = blockIdx.z; run < a.n_runs && (run == 0 || run * AF_RUN_PAGES * BN_PAGE < len); run += gridDim.z) {
        const int j0 = (run * AF_RUN_PAGES + wave) * BN_PAGE;
        AfSums<HS> p;
        p.m = -INFINITY; p.l = 0.f;
        if (j0 < len) {
            const int page = a.block_table[(size_t)tok * a.bt_stride + j0 / BN_PAGE];
            const float* kg = a.k_pages + ((size_t)page * a.Hkv + kvh) * BN_PAGE * HS;
            const float* vg = a.v_pages + ((size_t)page * a.Hkv + kvh) * BN_PAGE * HS;
            const int last = min(len - 1 - j0, BN_PAGE - 1);
            f32x4 kf[4][S::NB];
            float vf[4][4][S::NH][S::VW];
            if (last == BN_PAGE - 1) {            // a whole page: straight-line loads
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int b = 0; b < S::NB; ++b) kf[t][b] = *reinterpret_cast<const f32x4*>(kg + (16 * t + r) * HS + 16 * b + 4 * g);
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int h = 0; h < S::NH; ++h) af_values<S::VW>(vg + (16 * t + 4 * g + e) * HS + 16 * S::VW * h + S::VW * r, vf[t][e][h]);
            } else {                              // rows behind the last key count as zeros
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int b = 0; b < S::NB; ++b) kf[t][b] = *reinterpret_cast<const f32x4*>(kg + min(16 * t + r, last) * HS + 16 * b + 4 * g);
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int h = 0; h < S::NH; ++h) {
                            const int row = 16 * t + 4 * g + e;
                            af_values<S::VW>(vg + min(row, last) * HS + 16 * S::VW * h + S::VW * r, vf[t][e][h]);
#pragma unroll
                            for (int i = 0; i < S::VW; ++i) vf[t][e][h][i] = row <= last ? vf[t][e][h][i] : 0.f;
                        }
            }
            af_page<HS>(q, a.scale, last, last < BN_PAGE - 1, [&](int t, int b) { return kf[t][b]; },
                        [&](int t, int e, int h, float (&v)[S::VW]) {
#pragma unroll
                            for (int i = 0; i < S::VW; ++i) v[i] = vf[t][e][h][i];
                        },
                        p);
#pragma unroll
            for (int h = 0; h < S::NH; ++h)
#pragma unroll
                for (int i = 0; i < S::VW; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) so[wave][r][16 * S::VW * h + S::VW * (4 * g + j) + i] = p.o[h][i][j];
        }
        if (g == 0) { sm[wave][r] = p.m; sl[wave][r] = p.l; }
        __syncthreads();
        for (int idx = tid; idx < rows * HS; idx += 256) {
            const int row = idx / HS, d = idx - row * HS;
            float M = -INFINITY, L = 0.f, O = 0.f;
#pragma unroll
            for (int w = 0; w < AF_RUN_PAGES; ++w) {
                const float m = sm[w][row];
                if (m == -INFINITY) continue;
                float m2, fa, fb;
                af_factors(M, m, m2, fa, fb);
                L = af_fold(L, fa, sl[w][row], fb);
                O = af_fold(O, fa, so[w][row][d], fb);
                M = m2;
            }
            const int head = kvh * G + ht * GT + row;
            if (a.n_runs == 1) {
                a.out[(size_t)tok * a.out_stride + (size_t)head * HS + d] = __fmul_rn(O, L > 0.f ? 1.0f / L : 0.f);
            } else {
                const size_t at = ((size_t)tok * a.H + head) * a.n_runs + run;
                a.part_o[at * HS + d] = O;
                if (d == 0) { a.part_ml[2 * at] = M; a.part_ml[2 * at + 1] = L; }
            }
        }
        __syncthreads();
    }
}

// the runs of a row in order
__global__ __launch_bounds__(128) void attn_f32_fold_kernel(AfArgs a, int hs) {
    const int row = blockIdx.x, tok = row / a.H, head = row - tok * a.H, d = threadIdx.x;
    if (d >= hs) return;
    const int len = a.seq_lens[tok], runs = (len + AF_RUN_PAGES * BN_PAGE - 1) / (AF_RUN_PAGES * BN_PAGE);
    const float* ml = a.part_ml + (size_t)row * a.n_runs * 2;
    const float* po = a.part_o + (size_t)row * a.n_runs * hs + d;
    float M = -INFINITY, L = 0.f, O = 0.f;
    for (int s0 = 0; s0 < runs; s0 += 8) {        // eight runs' sums are asked for at once
        float m[8], l[8], o[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int s = min(s0 + i, runs - 1);
            m[i] = ml[2 * s]; l[i] = ml[2 * s + 1]; o[i] = po[(size_t)s * hs];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (s0 + i >= runs || m[i] == -INFINITY) continue;
            float m2, fa, fb;
            af_factors(M, m[i], m2, fa, fb);
            L = af_fold(L, fa, l[i], fb);
            O = af_fold(O, fa, o[i], fb);
            M = m2;
        }
    }
    a.out[(size_t)tok * a.out_stride + (size_t)head * hs + d] = __fmul_rn(O, L > 0.f ? 1.0f / L : 0.f);
}

template <int HS>
static int af_launch(const AfArgs& a, int n_tiles, hipStream_t s) {
    const int G = a.H / a.Hkv, heads = a.Hkv * ((G + a.GT - 1) / a.GT);
    if (a.tiles) {
        hipLaunchKernelGGL(attn_f32_prompt_kernel<HS>, dim3(n_tiles, heads), dim3(256), 0, s, a);
        return bn_launch_status();
    }
    // a workgroup a run up to some 2,048 workgroups; a longer table's runs are taken in turn
    int z = 2048 / (n_tiles * heads);
    z = z < 1 ? 1 : z > a.n_runs ? a.n_runs : z;
    hipLaunchKernelGGL(attn_f32_decode_kernel<HS>, dim3(n_tiles, heads, z), dim3(256), 0, s, a);
    if (int rc = bn_launch_status()) return rc;
    if (a.n_runs > 1) hipLaunchKernelGGL(attn_f32_fold_kernel, dim3(n_tiles * a.H), dim3(128), 0, s, a, HS);
    return bn_launch_status();
}

extern "C" int bn_attn_f32_supports(int hs) { return hs == 16 || hs == 32 || hs == 64 || hs == 128; }
extern "C" int bn_attn_f32_run_keys(void) { return AF_RUN_PAGES * BN_PAGE; }

// tiles: the prompt form, tiles of up to 64 / GT tokens; null: the decode form, n_tiles sequences, with n_runs > 1 over
// partial sums of n_runs runs a row (the runs that a block table of bt_stride pages can hold)
extern "C" int bn_attn_f32(const void* q, int q_stride, void* out, int out_stride, const void* k_pages, const void* v_pages,
                           const int* block_table, int bt_stride, const int* seq_lens, const int* tiles, int n_tiles, int H, int Hkv,
                           int hs, int GT, float scale, int n_runs, float* part_o, float* part_ml, hipStream_t s) {
    if (n_tiles <= 0 || n_tiles > 65535 * 128 || H <= 0 || Hkv <= 0 || H % Hkv || GT < 1 || GT > 16 || (GT & (GT - 1))) return BN_ERR_ARG;
    if (Hkv * ((H / Hkv + GT - 1) / GT) > 65535 || bt_stride < 1 || n_runs < 1) return BN_ERR_ARG;
    if (!tiles && (!seq_lens || (long long)n_runs * AF_RUN_PAGES < bt_stride || (n_runs > 1 && (!part_o || !part_ml)))) return BN_ERR_ARG;
    AfArgs a = {(const float*)q, (float*)out, (const float*)k_pages, (const float*)v_pages, block_table, seq_lens, tiles, part_o,
                part_ml, q_stride, out_stride, bt_stride, H, Hkv, GT, n_runs, scale};
    switch (hs) {
        case 16: return af_launch<16>(a, n_tiles, s);
        case 32: return af_launch<32>(a, n_tiles, s);
        case 64: return af_launch<64>(a, n_tiles, s);
        case 128: return af_launch<128>(a, n_tiles, s);
    }
    return BN_ERR_ARG;
}
