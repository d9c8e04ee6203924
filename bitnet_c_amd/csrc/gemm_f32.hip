// C[M, N] = A[M, K] . W[N, K]^T in true float32 on the float32 matrix instruction (v_mfma_f32_16x16x4_f32: float32
// products and float32 sums, no reduced-precision mode), the matrix product of the float32 path.  W is row-major
// [out, in] as the reference keeps it (src/model.c:157-158); out[row] = sum_col W[row, col] x[col]
// (src/quant/f32_scalar.c:4-32).
//
// One order of summation, a function of K alone, whatever M, N, the kernel and its tiles are, so that a row's result does
// not depend on what else is in the batch: K is cut in chunks of 128; a chunk is summed from nothing by 32 instructions, the
// one of (block j of 16 columns, e) taking columns 16 j + 4 g + e (g = 0..3, the instruction's four); the chunks' sums are
// added in order.  The cut is what lets a product of few rows spread one output's K over the waves of a workgroup (and it
// keeps the rounding error at that of a sum of 128 and of K / 128 terms).
//
// gemm_f32_streamed_kernel, up to 16 rows over a streamed copy of W: see there.
// gemm_f32_stream_kernel, up to 64 rows over W itself: bound by the bytes of W.  A workgroup of 8 waves owns up to 16 columns
// and all of K; a wave takes every eighth chunk, asks for its whole 8 KB of W (and the rows' 128 columns of A) at once and
// leaves 16 x 16 sums in shared memory; then a thread an output adds them up in order.  us at one row, 1.5 GB of weights in
// turn, and at 6.5 TB/s: 11,264 x 2,048 24 (14), 2,048 x 5,632 19.5 (7), 32,000 x 2,048 52 (40), 28,672 x 4,096 103 (72); the
// vector kernel that walked K in one chain (gemm_tiled.hip) took 325 on the average of a layer's products, whatever the rows
// up to 16.  Its loads of W are plain: two of them take the halves of a line, and non-temporal ones were slower (11,264 x 2,048
// at 8 rows 25 -> 26 us, 32,000 x 2,048 59 -> 65).
// gemm_f32_dma_kernel, more rows, K of whole steps of 32: bound by the instruction (157 TFLOP/s on this chip, 32 cycles each on
// a SIMD).  5,136 x 11,264 x 2,048 1.72 ms (138 TFLOP/s), 5,136 x 2,048 x 5,632 0.91 ms (131), 5,136 x 2,048 x 2,048 0.35 ms (124;
// the last round's empty CUs).
// gemm_f32_tile_kernel, other K: the same products staged through registers (117, 109 and 106 TFLOP/s there).
#include "common.h"
#include <type_traits>

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define GF_CHUNK 128                 // columns of K whose products are summed from nothing
#define GF_BLOCKS (GF_CHUNK / 16)
#define GF_WAVES 8                   // waves of a workgroup of the streaming kernel
#define GF_SUMS_KB 64                // shared memory for a round of chunk sums

struct GfArgs {
    const float* x;
    const float* w;
    float* y;
    int M, N, K;                     // N: rows of W
    int ldx, ldw, ldy;
    int cols;                        // columns a workgroup of the streaming kernel owns (<= 16)
    int glu;                         // rows of W are gate and up rows in turns of 8; y[M, N / 2] = act(gate) * up
    int act;
    int add;                         // y += the product (kernels of up to 16 rows, no glu)
    const float* norm_w;             // rows of x are normed on their way in: x * scale * norm_w; null: as they are
    float eps;
};

struct gf_true { static constexpr bool value = true; };
struct gf_false { static constexpr bool value = false; };

__device__ __forceinline__ f32x4 gf_load(const float* p, bool ok) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (ok) v = *reinterpret_cast<const f32x4*>(p);
    return v;
}

// A norm in front of a product of few rows: every workgroup sums the squares of the rows itself, while its first weights are on
// their way, instead of a kernel of its own that the product would wait for (4.4 us a launch; the rows come from the L2).  The
// sums, their order and the factor are add_rmsnorm_row_kernel's (elementwise.hip): 256 threads take a row in groups of four, a
// wave's sums are added as a butterfly, the four waves' in order; here the halves of the workgroup take every other row.
// NR: rows a half takes; NV: groups a thread and row.  parts: [2 NR][4], a wave's sum of a row.
//   us in a decode step of Llama, 2,048 columns, one row: norm 4.4 + 11,264 x 2,048 16.4 -> 16.7, norm 4.4 + 3,072 x 2,048 6.9 -> 6.9;
//   whole calls, prompt of 199 and 16 steps 14.3 -> 13.7 ms, eight prompts and 8 steps 55.3 -> 54.8.  Up to 8 rows: beyond that a
//   workgroup reads more of the rows than of its weights, and the rows' registers are not there (GF_NORM_LOADS).
__device__ __forceinline__ float gf_norm_scale(const GfArgs& a, const float* parts, int row) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) ss += parts[row * 4 + i];
    return 1.0f / sqrtf(ss / (float)a.K + a.eps);
}
template <int NR, int NV> struct GfNorm {
    f32x4 v[NR][NV], w[NV];
    __device__ __forceinline__ void load(const GfArgs& a, int tid) {
        const int t = tid & 255, half = __builtin_amdgcn_readfirstlane(tid >> 8);
#pragma unroll
        for (int i = 0; i < NR; ++i)
#pragma unroll
            for (int k = 0; k < NV; ++k)
                v[i][k] = *reinterpret_cast<const f32x4*>(a.x + (size_t)min(half + 2 * i, a.M - 1) * a.ldx + min((k * 256 + t) * 4, a.K - 4));
#pragma unroll
        for (int k = 0; k < NV; ++k) w[k] = *reinterpret_cast<const f32x4*>(a.norm_w + min((k * 256 + t) * 4, a.K - 4));
    }
    __device__ __forceinline__ void sum(const GfArgs& a, int tid, float* parts) {
        const int t = tid & 255, half = __builtin_amdgcn_readfirstlane(tid >> 8), wave = (tid >> 6) & 3;
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            float ss = 0.f;
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                const float s = bn_add_squares(ss, v[i][k], k);
                if ((k * 256 + t) * 4 < a.K) ss = s;
            }
            ss = wave_sum(ss);
            if ((tid & 63) == 0) parts[(half + 2 * i) * 4 + wave] = ss;
        }
    }
    // the normed rows to shared memory, row_bytes apart (behind a barrier after sum)
    __device__ __forceinline__ void store(const GfArgs& a, int tid, const float* parts, unsigned char* rows, int row_bytes) {
        const int t = tid & 255, half = __builtin_amdgcn_readfirstlane(tid >> 8);
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const float scale = gf_norm_scale(a, parts, half + 2 * i);
#pragma unroll
            for (int k = 0; k < NV; ++k)
                if ((k * 256 + t) * 4 < a.K) *reinterpret_cast<f32x4*>(rows + (half + 2 * i) * row_bytes + (k * 256 + t) * 16) = v[i][k] * scale * w[k];
        }
    }
};
#define GF_NORM_LOADS 10             // (NR + 1) * NV at the most: what registers hold beside the first weights in flight

// MT row tiles of 16 share a wave's registers of W.  NR, NV: as GfNorm's; NR 0: no norm.
template <int MT, int NR = 0, int NV = 1>
__global__ __launch_bounds__(64 * GF_WAVES, 4) void gemm_f32_stream_kernel(GfArgs a) {
    constexpr int ROUND = GF_SUMS_KB / MT;                       // chunks whose sums shared memory holds at a time
    constexpr int THREADS = 64 * GF_WAVES;
    __shared__ float sums[ROUND * MT * 256];                     // [chunk][row tile][row][column]
    float scale = 1.f;                                           // of row r
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * a.cols;
    // lanes without a column or a row read their neighbour's (no other bytes, and no load under a branch); what they form is
    // not stored
    const float* wp = a.w + (size_t)min(n0 + min(r, a.cols - 1), a.N - 1) * a.ldw + 4 * g;
    const float* xp[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) xp[t] = a.x + (size_t)min(16 * t + r, a.M - 1) * a.ldx + 4 * g;
    const int n_chunks = (a.K + GF_CHUNK - 1) / GF_CHUNK;
    // the outputs that this thread adds up
    constexpr int OWN = (MT * 256 + THREADS - 1) / THREADS;
    float tot[OWN], old[OWN];
#pragma unroll
    for (int o = 0; o < OWN; ++o) tot[o] = old[o] = 0.f;
    if (a.add && MT == 1 && tid < 256) {                         // asked for before the weights
        const int m = tid >> 4, n = n0 + (tid & 15);
        if (m < a.M && n < a.N) old[0] = a.y[(size_t)m * a.ldy + n];
    }
    if constexpr (NR > 0) {
        GfNorm<NR, NV> norm;
        norm.load(a, tid);
        norm.sum(a, tid, sums);                                  // where the chunks' sums come later
        bn_lds_barrier();
        scale = gf_norm_scale(a, sums, min(r, a.M - 1));
        bn_lds_barrier();
    }

    for (int c0 = 0; c0 < n_chunks; c0 += ROUND) {
        const int c1 = min(n_chunks, c0 + ROUND);
        auto chunk = [&](int c, auto whole) {
            const int k0 = c * GF_CHUNK;
            auto fetch = [&](const float* p, f32x4 (&v)[GF_BLOCKS]) {
#pragma unroll
                for (int j = 0; j < GF_BLOCKS; ++j)
                    v[j] = gf_load(p + k0 + 16 * j, decltype(whole)::value || k0 + 16 * j + 4 * g < a.K);
            };
            f32x4 wv[GF_BLOCKS];
            fetch(wp, wv);
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                f32x4 xv[GF_BLOCKS], acc = {0.f, 0.f, 0.f, 0.f};
                fetch(xp[t], xv);
                if constexpr (NR > 0) {
                    f32x4 nw[GF_BLOCKS];
                    fetch(a.norm_w + 4 * g, nw);
#pragma unroll
                    for (int j = 0; j < GF_BLOCKS; ++j) xv[j] = xv[j] * scale * nw[j];
                }
#pragma unroll
                for (int j = 0; j < GF_BLOCKS; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[j][e], xv[j][e], acc, 0, 0, 0);
                // lane: columns 4 g .. 4 g + 3 of row r
                *reinterpret_cast<f32x4*>(&sums[((c - c0) * MT + t) * 256 + 16 * r + 4 * g]) = acc;
            }
        };
        for (int c = c0 + wave; c < c1; c += GF_WAVES) {
            if ((c + 1) * GF_CHUNK <= a.K) chunk(c, gf_true());
            else chunk(c, gf_false());
        }
        __syncthreads();
#pragma unroll
        for (int o = 0; o < OWN; ++o) {
            const int idx = tid + o * THREADS;
            if (idx < MT * 256)
                for (int c = 0; c < c1 - c0; ++c) tot[o] += sums[c * MT * 256 + idx];
        }
        if (c1 < n_chunks) __syncthreads();
    }
    if (a.glu) __syncthreads();
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
        const int idx = tid + o * THREADS;
        if (idx >= MT * 256) continue;
        const int m = idx >> 4, c = idx & 15;
        if (a.glu) sums[idx] = tot[o];
        else if (m < a.M && c < a.cols && n0 + c < a.N) a.y[(size_t)m * a.ldy + n0 + c] = a.add ? old[o] + tot[o] : tot[o];
    }
    if (!a.glu) return;
    __syncthreads();
    for (int idx = tid; idx < MT * 128; idx += THREADS) {
        const int m = idx >> 3, n = idx & 7;
        if (m < a.M) a.y[(size_t)m * a.ldy + n0 / 2 + n] = bn_gate_act(sums[m * 16 + n], a.act) * sums[m * 16 + 8 + n];
    }
}

// ---------------------------------------------------------------------------------------
// The product of up to 16 rows over a streamed copy of W (common.h) whose K is whole chunks.  Bound by the bytes of W: over
// the row-major matrix a load takes 64 bytes of each of 16 rows, half of a cache line, and waits under a test; here it takes
// a tile, 1 KB in a run, non-temporally, in straight-line code with two chunks (16 KB) a wave in flight, and the activations
// go through the wave's own shared memory, so that one row costs one load a chunk instead of eight.  The same sums in the
// same order as the kernels around it (a chunk by itself, the chunks in order): the same bits.  XR: activation loads a lane
// and chunk, for up to 2 XR rows.
//   us at 1 / 8 rows with cold weights in a graph of such launches, row-major -> streamed: 3,072 x 2,048 8.4 / 10.1 -> 7.2 /
//   7.6, 2,048 x 2,048 7.9 / 8.0 -> 6.0 / 6.8, 11,264 x 2,048 23.2 / 26.5 -> 17.6 / 18.7, 2,048 x 5,632 19.3 / 19.7 -> 11.6 /
//   13.1, 32,000 x 2,048 55.6 / 66.4 -> 43.2 / 44.4, 28,672 x 4,096 96 / 117 -> 76.5 / 75.5, 4,096 x 14,336 57 / 63 -> 41 / 42.
//   (16 instructions of 32 cycles stand for 4 KB of eight columns: up to 2,048 columns the matrix unit has half the time.)
#define GF_XROW (GF_CHUNK * 4 + 16)  // bytes between the rows of a wave's staged activations

// NV > 0: behind a norm (GfNorm<XR, NV>; every wave has a chunk).  The normed rows are staged once, all of them, by the threads
// that summed their squares, and the waves read their chunks from there.
template <int XR, int NV = 0>
__global__ __launch_bounds__(64 * GF_WAVES, XR == 8 ? 2 : 4) void gemm_f32_streamed_kernel(GfArgs a, int k_tiles) {
    constexpr int ROWS = 2 * XR;
    constexpr bool NORM = NV > 0;
    extern __shared__ __align__(16) unsigned char smem[];
    const int row_bytes = NORM ? a.K * 4 + 16 : GF_XROW;
    float* sums = reinterpret_cast<float*>(smem + (NORM ? 1 : GF_WAVES) * ROWS * row_bytes);     // [chunk][row][column]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const unsigned tile = a.cols * (BN_STREAM_TILE_COLS_F32 * 4);
    const auto wb = bn_buffer(reinterpret_cast<const char*>(a.w) + (size_t)blockIdx.x * k_tiles * tile, k_tiles * tile);
    const auto xb = bn_buffer(a.x, ((a.M - 1) * a.ldx + a.K) * 4);
    const unsigned w_at = (g * a.cols + min(r, a.cols - 1)) * 16;
    unsigned x_at[XR];
#pragma unroll
    for (int i = 0; i < XR; ++i) x_at[i] = (min(2 * i + (lane >> 5), a.M - 1) * a.ldx + (lane & 31) * 4) * 4;
    unsigned char* xs = smem + (NORM ? 0 : wave * ROWS * GF_XROW);
    unsigned char* park_at = xs + (lane >> 5) * GF_XROW + (lane & 31) * 16;
    const unsigned char* read_at = xs + min(r, a.M - 1) * row_bytes + g * 16;
    f32x4 x[XR];
    auto load_x = [&](int c) {
        if (NORM) return;
#pragma unroll
        for (int i = 0; i < XR; ++i) x[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(xb, x_at[i], c * (GF_CHUNK * 4), 0));
    };
    auto load_w = [&](f32x4 (&w)[GF_BLOCKS], int c) {
        unsigned at = (unsigned)c * GF_BLOCKS * tile;
#pragma unroll
        for (int j = 0; j < GF_BLOCKS; ++j, at += tile)
            w[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(wb, w_at, at, BN_BUFFER_NT));
        __builtin_amdgcn_sched_barrier(0);
    };
    auto park = [&]() {
        if (NORM) return;
#pragma unroll
        for (int i = 0; i < XR; ++i) *reinterpret_cast<f32x4*>(park_at + 2 * i * GF_XROW) = x[i];
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](const f32x4 (&w)[GF_BLOCKS], int c) {
        const unsigned char* from = read_at + (NORM ? c * (GF_CHUNK * 4) : 0);
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int h = 0; h < GF_BLOCKS; h += 4) {
            f32x4 v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = *reinterpret_cast<const f32x4*>(from + (h + j) * 64);
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[h + j][e], v[j][e], acc, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (r < ROWS) *reinterpret_cast<f32x4*>(sums + ((size_t)c * ROWS + r) * 16 + 4 * g) = acc;   // columns 4 g .. 4 g + 3 of row r
        __builtin_amdgcn_wave_barrier();
    };
    const int n_chunks = a.K / GF_CHUNK;
    const int n = (n_chunks - wave + GF_WAVES - 1) / GF_WAVES;               // chunks of this wave: wave, wave + 8, ..
    constexpr int D = GF_WAVES;
    // what the results are added to: an empty buffer, of which a load gives zero and reads nothing, where they are not
    const int om = tid >> 4, on = blockIdx.x * a.cols + (tid & 15);
    const auto yb = bn_buffer(a.y, a.add ? ((a.M - 1) * a.ldy + a.N) * 4 : 0);
    const float old = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(yb, (min(om, a.M - 1) * a.ldy + min(on, a.N - 1)) * 4, 0, 0));
    GfNorm<XR, NORM ? NV : 1> norm;
    if (NORM) norm.load(a, tid);
    auto stage = [&] {                                                       // once a wave, behind its first loads of W
        if (!NORM) return;
        norm.sum(a, tid, sums);                                              // where the chunks' sums come later
        bn_lds_barrier();
        norm.store(a, tid, sums, smem, row_bytes);
        bn_lds_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    if (n == 1) {
        f32x4 w[GF_BLOCKS];
        load_x(wave);
        load_w(w, wave);
        stage();
        park();
        multiply(w, wave);
    } else if (n > 1) {
        int c = wave, left = n;
        f32x4 p[GF_BLOCKS], q[GF_BLOCKS];
        load_x(c);
        load_w(p, c);
        stage();                                                             // (the rows' registers are the second chunk's)
        load_w(q, c + D);
#pragma unroll 1
        for (; left > 3; left -= 2, c += 2 * D) {
            park();
            load_x(c + D);
            multiply(p, c);
            load_w(p, c + 2 * D);
            park();
            load_x(c + 2 * D);
            multiply(q, c + D);
            load_w(q, c + 3 * D);
        }
        park();
        load_x(c + D);
        multiply(p, c);
        if (left == 2) {
            park();
            multiply(q, c + D);
        } else {
            load_w(p, c + 2 * D);
            park();
            load_x(c + 2 * D);
            multiply(q, c + D);
            park();
            multiply(p, c + 2 * D);
        }
    }
    bn_lds_barrier();
    if (tid >= ROWS * 16) return;
    float tot = 0.f;
#pragma unroll 8
    for (int c = 0; c < n_chunks; ++c) tot += sums[(size_t)c * (ROWS * 16) + tid];
    const int m = tid >> 4, col = tid & 15, n0 = blockIdx.x * a.cols;
    if (a.glu) {                                                             // columns 0..7 of the tile are gates, 8..15 their ups
        const float up = bn_lane_xor<8>(tot);
        if (m < a.M && col < 8) a.y[(size_t)m * a.ldy + n0 / 2 + col] = bn_gate_act(tot, a.act) * up;
    } else if (m < a.M && col < a.cols && n0 + col < a.N) {
        a.y[(size_t)m * a.ldy + n0 + col] = a.add ? old + tot : tot;
    }
}

#define GF_BK 32
#define GF_STRIDE (GF_BK + 4)        // of a staged row: 16-byte reads of the lanes' rows fall on different banks

// orders shared memory alone: loads from memory stay in flight across it
__device__ __forceinline__ void gf_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// A workgroup of 4 waves (2 x 2) owns BM rows of A and BN rows of W; a wave (BM / 2) x (BN / 2).
template <int BM, int BN>
__global__ __launch_bounds__(256, 2) void gemm_f32_tile_kernel(GfArgs a, int m_tiles, int n_tiles) {
    constexpr int MT = BM / 32, NT = BN / 32;                    // 16 x 16 tiles of a wave
    constexpr int XL = BM * GF_BK / 4 / 256, WL = BN * GF_BK / 4 / 256;      // 16-byte loads a thread and step
    __shared__ float xs[2][BM * GF_STRIDE];
    __shared__ float ws[2][BN * GF_STRIDE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    // consecutive workgroups go to consecutive XCDs: give each XCD a run of tiles, and walk a run in bands of 8 row tiles, so
    // that what runs on an XCD together shares its operands in that L2
    int id = blockIdx.x;
    const int total = m_tiles * n_tiles;
    {
        const int per = total / 8, rest = total % 8, xcd = id % 8, at = id / 8;
        id = xcd * per + min(xcd, rest) + at;
    }
    const int band = id / (8 * n_tiles), in_band = id - band * 8 * n_tiles;
    const int band_rows = min(8, m_tiles - band * 8);
    const int m0 = (band * 8 + in_band % band_rows) * BM, n0 = (in_band / band_rows) * BN;
    const int wm = (wave & 1) * (BM / 2), wn = (wave >> 1) * (BN / 2);

    f32x4 acc[NT][MT], tot[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) { acc[i][j] = 0.f; tot[i][j] = 0.f; }

    // staging: thread -> (row tid / 8 + 32 i, 16-byte group tid % 8); rows past the matrix read its last row and are not stored.
    // Offsets are 32 bits wide against the tile's own (uniform) address.
    const int sr = tid >> 3, sc = 4 * (tid & 7);
    const float* xbase = a.x + (size_t)m0 * a.ldx;
    const float* wbase = a.w + (size_t)n0 * a.ldw;
    uint32_t xo[XL], wo[WL];
#pragma unroll
    for (int i = 0; i < XL; ++i) xo[i] = (uint32_t)min(sr + 32 * i, a.M - 1 - m0) * (uint32_t)a.ldx;
#pragma unroll
    for (int i = 0; i < WL; ++i) wo[i] = (uint32_t)min(sr + 32 * i, a.N - 1 - n0) * (uint32_t)a.ldw;
    f32x4 xr[XL], wr[WL];
    // loads are in straight line (one under a branch would be waited for at once); groups past K read the row's last one
    // and become zeros when they are stored
    auto load = [&](int k0) {
        const uint32_t k = min(k0 + sc, a.K - 4);
#pragma unroll
        for (int i = 0; i < XL; ++i) xr[i] = *reinterpret_cast<const f32x4*>(xbase + (xo[i] + k));
#pragma unroll
        for (int i = 0; i < WL; ++i) wr[i] = *reinterpret_cast<const f32x4*>(wbase + (wo[i] + k));
    };
    auto store = [&](int b, int k0) {
        if (k0 + GF_BK > a.K && k0 + sc >= a.K) {
#pragma unroll
            for (int i = 0; i < XL; ++i) xr[i] = 0.f;
#pragma unroll
            for (int i = 0; i < WL; ++i) wr[i] = 0.f;
        }
#pragma unroll
        for (int i = 0; i < XL; ++i) *reinterpret_cast<f32x4*>(&xs[b][(sr + 32 * i) * GF_STRIDE + sc]) = xr[i];
#pragma unroll
        for (int i = 0; i < WL; ++i) *reinterpret_cast<f32x4*>(&ws[b][(sr + 32 * i) * GF_STRIDE + sc]) = wr[i];
    };
    f32x4 wv[2][NT], xv[2][MT];                                  // operands of the two blocks of a step
    auto read = [&](int b, int blk) {
#pragma unroll
        for (int i = 0; i < NT; ++i) wv[blk][i] = *reinterpret_cast<const f32x4*>(&ws[b][(wn + 16 * i + r) * GF_STRIDE + 16 * blk + 4 * g]);
#pragma unroll
        for (int j = 0; j < MT; ++j) xv[blk][j] = *reinterpret_cast<const f32x4*>(&xs[b][(wm + 16 * j + r) * GF_STRIDE + 16 * blk + 4 * g]);
    };
    auto multiply = [&](int blk, int from, int to) {
#pragma unroll
        for (int e = from; e < to; ++e)
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < MT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[blk][i][e], xv[blk][j][e], acc[i][j], 0, 0, 0);
    };
    // A step multiplies two blocks of 16; every read of shared memory is asked for a block ahead of its products, a tile's
    // stores stand in front of products that do not need them, and its loads a step earlier.  The one barrier of a step lies
    // between its blocks: in front of it every wave has read all of buffer b and stored its part of the other.
    const int steps = (a.K + GF_BK - 1) / GF_BK;
    load(0);
    store(0, 0);
    load(GF_BK);
    gf_barrier();
    read(0, 0);
    for (int s = 0; s < steps; ++s) {
        const int b = s & 1;
        multiply(0, 0, 1);       // first, so that the compiler's wait for block 0's operands meets no younger access
        __builtin_amdgcn_sched_barrier(0);
        read(b, 1);
        store(b ^ 1, (s + 1) * GF_BK);
        load((s + 2) * GF_BK);
        __builtin_amdgcn_sched_barrier(0);
        multiply(0, 1, 4);
        __builtin_amdgcn_sched_barrier(0);
        gf_barrier();
        read(b ^ 1, 0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(1, 0, 4);
        if ((s + 1) % (GF_CHUNK / GF_BK) == 0 || s + 1 == steps) {           // a chunk of K ends
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < MT; ++j) { tot[i][j] += acc[i][j]; acc[i][j] = 0.f; }
        }
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int n = n0 + wn + 16 * i + 4 * g;
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const int m = m0 + wm + 16 * j + r;
            if (a.glu) {                                         // lanes with g < 2 hold gates, the lane 32 further their ups
                f32x4 up;
#pragma unroll
                for (int e = 0; e < 4; ++e) up[e] = __shfl_xor(tot[i][j][e], 32, BN_WAVE);
                if (g < 2 && m < a.M && n < a.N) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        a.y[(size_t)m * a.ldy + (n0 + wn + 16 * i) / 2 + 4 * g + e] = bn_gate_act(tot[i][j][e], a.act) * up[e];
                }
            } else if (m < a.M) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < a.N) a.y[(size_t)m * a.ldy + n + e] = tot[i][j][e];
            }
        }
    }
}

// Tiles for K of whole steps (K % 32 == 0).  Float32 matrix instructions and vector instructions share the SIMD's
// multipliers, so what the loop above spends on staging (addresses, tests, registers on their way to shared memory: one vector
// instruction for every matrix instruction) it takes from the products.  Here memory goes straight into shared memory
// (buffer loads with an LDS destination: a lane's offset is a constant, the step's lies in a scalar register), rows past the
// matrix lie past the buffer's end, and a chunk's first product starts from a constant zero.  A staged row is 128 bytes, chunk
// c of 16 bytes of row r at c ^ (r / 2 % 8), which keeps the sixteen lanes that shared memory serves together on different banks.
// NB buffers, NB - 1 steps ahead: two where a CU holds several workgroups, four where a launch gives it one or two, whose
// steps would each wait for memory.
template <int BM, int BN, int NB>
__global__ __launch_bounds__(256, 2) void gemm_f32_dma_kernel(GfArgs a, int m_tiles, int n_tiles) {
    constexpr int MT = BM / 32, NT = BN / 32;                    // 16 x 16 tiles of a wave
    constexpr int XI = BM / 32, WI = BN / 32;                    // staging loads of a wave and step, 8 rows each
    // buffers of their own names: the compiler then knows which loads a read of shared memory has to wait for
    __shared__ __align__(1024) unsigned char b0[(BM + BN) * 128], b1[(BM + BN) * 128];
    __shared__ __align__(1024) unsigned char b2[NB == 4 ? (BM + BN) * 128 : 16], b3[NB == 4 ? (BM + BN) * 128 : 16];
    static_assert(NB == 2 || NB == 4, "a chunk is four steps");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    int id = blockIdx.x;                                         // as in gemm_f32_tile_kernel
    const int total = m_tiles * n_tiles;
    {
        const int per = total / 8, rest = total % 8, xcd = id % 8, at = id / 8;
        id = xcd * per + min(xcd, rest) + at;
    }
    const int band = id / (8 * n_tiles), in_band = id - band * 8 * n_tiles;
    const int band_rows = min(8, m_tiles - band * 8);
    const int m0 = (band * 8 + in_band % band_rows) * BM, n0 = (in_band / band_rows) * BN;
    const int wm = (wave & 1) * (BM / 2), wn = (wave >> 1) * (BN / 2);

    f32x4 acc[NT][MT], tot[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) tot[i][j] = 0.f;

    const auto xb = bn_buffer(a.x + (size_t)m0 * a.ldx, ((min(BM, a.M - m0) - 1) * a.ldx + a.K) * 4);
    const auto wb = bn_buffer(a.w + (size_t)n0 * a.ldw, ((min(BN, a.N - n0) - 1) * a.ldw + a.K) * 4);
    // load i of a wave: rows 32 i + 8 wave .. + 7, a lane the 16 bytes at slot lane % 8 of row lane / 8
    const int sr = 8 * wave + (lane >> 3), sc = ((lane & 7) ^ ((sr >> 1) & 7)) * 16;
    unsigned xo[XI], wo[WI];
#pragma unroll
    for (int i = 0; i < XI; ++i) xo[i] = (sr + 32 * i) * a.ldx * 4 + sc;
#pragma unroll
    for (int i = 0; i < WI; ++i) wo[i] = (sr + 32 * i) * a.ldw * 4 + sc;
    auto stage = [&](unsigned char* to, int s) {                 // A's rows, then W's
#pragma unroll
        for (int i = 0; i < XI; ++i) bn_load_to_lds(xb, to + (32 * i + 8 * wave) * 128, xo[i], s * (GF_BK * 4));
#pragma unroll
        for (int i = 0; i < WI; ++i) bn_load_to_lds(wb, to + (BM + 32 * i + 8 * wave) * 128, wo[i], s * (GF_BK * 4));
    };
    // block b of a row: chunk 4 b + g, at (4 b + g) ^ (row / 2 % 8) (a tile's rows begin at multiples of 16)
    const int at0 = r * 128 + ((g ^ (r >> 1)) << 4), at1 = r * 128 + (((4 + g) ^ (r >> 1)) << 4);
    f32x4 wv[2][NT], xv[2][MT];
    auto read = [&](const unsigned char* from, int b) {
        const int at = b ? at1 : at0;
#pragma unroll
        for (int i = 0; i < NT; ++i) wv[b][i] = *reinterpret_cast<const f32x4*>(from + (BM + wn + 16 * i) * 128 + at);
#pragma unroll
        for (int j = 0; j < MT; ++j) xv[b][j] = *reinterpret_cast<const f32x4*>(from + (wm + 16 * j) * 128 + at);
    };
    auto multiply = [&](int b, auto first) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < MT; ++j) {
                    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[b][i][e], xv[b][j][e], decltype(first)::value && e == 0 ? zero : acc[i][j], 0, 0, 0);
                }
    };
    const int steps = a.K / GF_BK;
    // A step asks for the rows of NB - 1 steps on, into the buffer that the step before it has left, and multiplies its own;
    // past its barrier the next step's rows are there.  (The last steps ask for the last rows again, into buffers that nobody
    // reads any more.)
    constexpr int AHEAD = (NB - 2) * (XI + WI);                  // loads that may still be on their way behind a step
    auto arrived = [&]() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(AHEAD) : "memory"); };
    auto step = [&](const unsigned char* now, unsigned char* next, int s, auto first) {
        stage(next, min(s + NB - 1, steps - 1));
        __builtin_amdgcn_sched_barrier(0);
        read(now, 0);
        read(now, 1);
        multiply(0, first);
        multiply(1, gf_false());
        arrived();
    };
    auto fold = [&]() {
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int j = 0; j < MT; ++j) tot[i][j] += acc[i][j];
    };
    // step k of a chunk, k = 0..3
    auto step0 = [&](int s) { step(b0, NB == 2 ? b1 : b3, s, gf_true()); };
    auto step1 = [&](int s) { step(b1, b0, s, gf_false()); };
    auto step2 = [&](int s) { step(NB == 2 ? b0 : b2, b1, s, gf_false()); };
    auto step3 = [&](int s) { step(NB == 2 ? b1 : b3, NB == 2 ? b0 : b2, s, gf_false()); };
    stage(b0, 0);
    if (NB == 4) {
        stage(b1, min(1, steps - 1));
        stage(b2, min(2, steps - 1));
    }
    arrived();
    int s = 0;
#pragma unroll 1
    for (; s + 4 <= steps; s += 4) {
        step0(s);
        step1(s + 1);
        step2(s + 2);
        step3(s + 3);
        fold();
    }
    if (s < steps) {
        step0(s);
        if (s + 1 < steps) step1(s + 1);
        if (s + 2 < steps) step2(s + 2);
        fold();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");             // nothing is on its way into shared memory when the wave ends
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int n = n0 + wn + 16 * i + 4 * g;
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const int m = m0 + wm + 16 * j + r;
            if (a.glu) {                                         // lanes with g < 2 hold gates, the lane 32 further their ups
                f32x4 up;
#pragma unroll
                for (int e = 0; e < 4; ++e) up[e] = __shfl_xor(tot[i][j][e], 32, BN_WAVE);
                if (g < 2 && m < a.M && n < a.N) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        a.y[(size_t)m * a.ldy + (n0 + wn + 16 * i) / 2 + 4 * g + e] = bn_gate_act(tot[i][j][e], a.act) * up[e];
                }
            } else if (m < a.M) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < a.N) a.y[(size_t)m * a.ldy + n + e] = tot[i][j][e];
            }
        }
    }
}

// go(NR, NV) as integral constants for a norm of M rows of K numbers
static int gf_norm_rows(int M) { return M <= 2 ? 1 : M <= 4 ? 2 : 4; }
static bool gf_norm_ok(int M, int K, const float* norm_w) {
    return M >= 1 && M <= 8 && K >= 4 && K % 4 == 0 && K <= 4096 && ((K <= 2048 ? 2 : 4) * (gf_norm_rows(M) + 1)) <= GF_NORM_LOADS &&
           ((uintptr_t)norm_w & 15) == 0;
}
template <typename F> static int gf_norm_pick(int M, int K, F go) {
    using std::integral_constant;
    const int nr = gf_norm_rows(M);
#define GF_PICK(NR_, NV_) return go(integral_constant<int, NR_>(), integral_constant<int, NV_>())
    if (nr == 1 && K > 2048) GF_PICK(1, 4);
    if (nr == 1) GF_PICK(1, 2);
    if (nr == 2) GF_PICK(2, 2);
    GF_PICK(4, 2);
#undef GF_PICK
}

template <int MT, int NR = 0, int NV = 1>
static int gf_launch_stream(const GfArgs& a, hipStream_t s) {
    hipLaunchKernelGGL((gemm_f32_stream_kernel<MT, NR, NV>), dim3((a.N + a.cols - 1) / a.cols), dim3(64 * GF_WAVES), 0, s, a);
    return bn_launch_status();
}

template <int BM, int BN>
static int gf_launch_tile(const GfArgs& a, hipStream_t s) {
    const int mt = (a.M + BM - 1) / BM, nt = (a.N + BN - 1) / BN;
    hipLaunchKernelGGL((gemm_f32_tile_kernel<BM, BN>), dim3(mt * nt), dim3(256), 0, s, a, mt, nt);
    return bn_launch_status();
}

template <int BM, int BN, int NB>
static int gf_launch_dma(const GfArgs& a, hipStream_t s) {
    const int mt = (a.M + BM - 1) / BM, nt = (a.N + BN - 1) / BN;
    if (a.K % GF_BK) return BN_ERR_ARG;
    hipLaunchKernelGGL((gemm_f32_dma_kernel<BM, BN, NB>), dim3(mt * nt), dim3(256), 0, s, a, mt, nt);
    return bn_launch_status();
}

#define GF_CUS 256

// Columns a workgroup of the streaming kernel owns: 16, or fewer where the busiest CU then has at least an eighth fewer.  us at one
// row, 1.5 GB of weights in turn: 2,048 x 5,632 in 16 / 8 20.2 / 19.5, 6,144 x 4,096 in 16 / 12 25.0 / 24.6, 3,072 x 2,048 8.8 / 8.9;
// where the even split gains nothing fewer columns only read the rows more often: 32,000 x 2,048 in 16 / 12 51 / 60.
static int gf_stream_cols(int N) {
    int best = 16, cost = 1 << 30;
    for (int c : {16, 12, 8}) {
        const long long tiles = (N + c - 1) / c, busiest = (tiles + GF_CUS - 1) / GF_CUS * c;
        if (busiest * 8 <= (long long)cost * 7) { best = c; cost = (int)busiest; }
    }
    return best;
}

// The tile kernels' form with the least time for the busiest CU.  Whole steps (K % 32 == 0): a launch's first tile on a CU costs
// more than the ones beside it, ns a step of 32 columns of K with n tiles a CU 200 + 478 n of 64 x 64, 150 + 255 n of 32 x 64, 130
// + 130 n of 32 x 32 (fitted at 2,048 columns, n = 1 to 222, within 5 %).  us at 199 rows, these three: 3,072 x 2,048 45 / 41 / 33,
// 2,048 x 5,632 109 / 64 / 58, 11,264 x 2,048 110 / 91 / 93; at 5,136 rows 11,264 x 2,048 1,722 / 1,811 / 1,860; the kernel that
// stages through registers took 54, 82, 126 and 2,025.  Other K, that kernel: the longer of one tile's own chain of steps and of
// all its tiles' instructions, 128 x 128 2,400 and 2,090 a tile, 64 x 128 1,360 and 1,060, 64 x 64 790 and 520, 32 x 64 520 and 290.
static int gf_tile_form(int M, int N, int K) {
    static const int bm[7] = {128, 64, 64, 32, 64, 32, 32}, bn[7] = {128, 128, 64, 64, 64, 64, 32};
    static const int alone[4] = {2400, 1360, 790, 520}, many[7] = {2090, 1060, 520, 290, 478, 255, 130}, first[3] = {200, 150, 130};
    const bool whole = K % GF_BK == 0;
    int best = 0;
    long long cost = -1;
    for (int i = whole ? 4 : 0; i < (whole ? 7 : 4); ++i) {
        const long long tiles = (long long)((M + bm[i] - 1) / bm[i]) * ((N + bn[i] - 1) / bn[i]);
        const long long per_cu = (tiles + GF_CUS - 1) / GF_CUS, t = per_cu * many[i];
        const long long c = whole ? t + first[i - 4] : t > alone[i] ? t : alone[i];
        if (cost < 0 || c < cost) { best = i; cost = c; }
    }
    return 2 + best;
}

// what the kernels need of the operands: rows of whole 16-byte groups at 16-byte addresses; offsets inside a tile's rows are
// 32 bits wide
extern "C" int bn_gemm_f32_supports(int N, int K, int ldw, const void* w) {
    return N > 0 && K > 0 && K % 4 == 0 && ldw % 4 == 0 && ldw >= K && ldw <= (1 << 22) && ((uintptr_t)w & 15) == 0;
}

// form 0: by the sizes; 1: streaming; 2 .. 5: tiles of 128 x 128, 64 x 128, 64 x 64, 32 x 64; 6 .. 8, for whole steps: tiles of
// 64 x 64, 32 x 64, 32 x 32 straight into shared memory (every form gives the same bits).
// Streaming up to 16 rows.  Whole steps: up to 32 while a CU has one tile of 16 columns, since every workgroup of it reads all
// rows (us at 17 / 32 rows, streaming against tiles of 32 x 32: 2,048 x 2,048 13.6 / 14.9 against 17, 2,048 x 5,632 28 / 33 against
// 38, 4,096 x 14,336 83 / 93 against 106, 11,264 x 2,048 34 / 40 against 26 / 29; at 33 rows 2,048 x 2,048 19.8 against 17.5).  Other K:
// up to 64 while the rows' 16-row tiles times the column tiles of a CU stay few (at 64 rows, against tiles through registers,
// 2,048 x 5,632 54 / 82, 11,264 x 2,048 60 / 54, 28,672 x 4,096 255 / 164; at 20 rows 6,144 x 4,096 43 / 61, 32,000 x 2,048 86 / 54).
//
// norm_w (form 0): the rows of x are normed on their way in, bn_gemm_f32_norm_supports says of which sizes.  add (form 0, up to 16
// rows, no glu): y += the product.
extern "C" int bn_gemm_f32(const void* x, const void* w, void* y, int M, int N, int K, int ldx, int ldw, int ldy, int glu, int act,
                           int form, const float* norm_w, float eps, int add, hipStream_t s) {
    if (M <= 0 || !bn_gemm_f32_supports(N, K, ldw, w) || ldx % 4 || ldx < K || ldx > (1 << 22) || ((uintptr_t)x & 15)) return BN_ERR_ARG;
    if (ldy < (glu ? N / 2 : N) || (glu && N % 16) || act < 0 || act >= BN_ACT_KINDS) return BN_ERR_ARG;
    if ((long long)((M + 31) / 32) * ((N + 63) / 64) > 0x7fffffffLL) return BN_ERR_ARG;
    if (((norm_w || add) && form) || (norm_w && !gf_norm_ok(M, K, norm_w)) || (add && (glu || M > 16))) return BN_ERR_ARG;
    GfArgs a = {(const float*)x, (const float*)w, (float*)y, M, N, K, ldx, ldw, ldy, 16, glu ? 1 : 0, act, add ? 1 : 0, norm_w, eps};
    if (norm_w) {
        a.cols = glu ? 16 : gf_stream_cols(N);
        return gf_norm_pick(M, K, [&](auto nr, auto nv) { return gf_launch_stream<1, decltype(nr)::value, decltype(nv)::value>(a, s); });
    }
    const int mt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
    if (form == 0) {
        const bool streams = K % GF_BK == 0 ? M <= 32 && N <= 16 * GF_CUS : M <= 64 && (long long)mt * N <= 6LL * 16 * GF_CUS;
        form = M <= 16 || streams ? 1 : gf_tile_form(M, N, K);
    }
    switch (form) {
        case 1:
            if (M > 64) return BN_ERR_ARG;
            a.cols = glu ? 16 : gf_stream_cols(N);
            return mt == 1 ? gf_launch_stream<1>(a, s) : mt == 2 ? gf_launch_stream<2>(a, s) : gf_launch_stream<4>(a, s);
        case 2: return gf_launch_tile<128, 128>(a, s);
        case 3: return gf_launch_tile<64, 128>(a, s);
        case 4: return gf_launch_tile<64, 64>(a, s);
        case 5: return gf_launch_tile<32, 64>(a, s);
        case 6: return gf_launch_dma<64, 64, 2>(a, s);
        case 7: return gf_launch_dma<32, 64, 4>(a, s);
        case 8: return gf_launch_dma<32, 32, 4>(a, s);
    }
    return BN_ERR_ARG;
}

// Columns a workgroup of the streaming kernels owns: the rows per tile that a streamed copy of W is best made with.
extern "C" int bn_gemm_f32_stream_cols(int N) { return N < 1 ? 0 : gf_stream_cols(N); }

#define GF_STREAMED_SMEM (150 * 1024)
static int gf_streamed_xr(int M) { return M <= 2 ? 1 : M <= 4 ? 2 : M <= 8 ? 4 : 8; }
static size_t gf_streamed_smem(int M, int K, bool norm) {                    // the staged activations, a sum a chunk, row and column
    const size_t rows = 2 * gf_streamed_xr(M);
    return (norm ? rows * (K * 4 + 16) : GF_WAVES * rows * GF_XROW) + (size_t)(K / GF_CHUNK) * rows * 64;
}

// 1 if the products of up to 16 rows take a norm of such rows with them
extern "C" int bn_gemm_f32_norm_supports(int M, int K) { return gf_norm_ok(M, K, nullptr); }

// 1 if the kernel over a streamed copy takes the product: up to 16 rows, whole chunks whose sums fit into shared memory
// (every K up to 10,752 at 9 to 16 rows, 29,952 at 5 to 8), rows of activations that are whole 16-byte groups.
extern "C" int bn_gemm_f32_streamed_supports(int M, int N, int K, int ldx, int tile_rows, const void* x) {
    return M >= 1 && M <= 16 && N >= 1 && K >= GF_CHUNK && K % GF_CHUNK == 0 && gf_streamed_smem(M, K, false) <= GF_STREAMED_SMEM && ldx >= K &&
           ldx % 4 == 0 && ldx <= 1 << 22 && tile_rows >= 1 && tile_rows <= BN_STREAM_TILE_ROWS && ((uintptr_t)x & 15) == 0;
}

// As bn_gemm_f32 over W's streamed copy (common.h) with that many rows a tile (16 with glu).
extern "C" int bn_gemm_f32_streamed(const void* x, const void* tiles, void* y, int M, int N, int K, int ldx, int tile_rows, int ldy,
                                    int glu, int act, const float* norm_w, float eps, int add, hipStream_t s) {
    if (!bn_gemm_f32_streamed_supports(M, N, K, ldx, tile_rows, x) || !tiles || !y || ((uintptr_t)tiles & 15)) return BN_ERR_ARG;
    if (ldy < (glu ? N / 2 : N) || (glu && (N % 16 || tile_rows != 16)) || act < 0 || act >= BN_ACT_KINDS) return BN_ERR_ARG;
    if ((norm_w && (!gf_norm_ok(M, K, norm_w) || K < GF_WAVES * GF_CHUNK)) || (add && (glu || (long long)M * ldy > 1 << 29))) return BN_ERR_ARG;
    GfArgs a = {(const float*)x, (const float*)tiles, (float*)y, M, N, K, ldx, 0, ldy, tile_rows, glu ? 1 : 0, act, add ? 1 : 0, norm_w, eps};
    auto go = [&](auto kernel) {
        const size_t smem = gf_streamed_smem(M, K, norm_w != nullptr);
        if (smem > 64 * 1024) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            if (e != hipSuccess) return (int)e;
        }
        hipLaunchKernelGGL(kernel, dim3((N + tile_rows - 1) / tile_rows), dim3(64 * GF_WAVES), smem, s, a, K / BN_STREAM_TILE_COLS_F32);
        return bn_launch_status();
    };
    if (norm_w)
        return gf_norm_pick(M, K, [&](auto nr, auto nv) { return go(gemm_f32_streamed_kernel<decltype(nr)::value, decltype(nv)::value>); });
    switch (gf_streamed_xr(M)) {
        case 1: return go(gemm_f32_streamed_kernel<1>);
        case 2: return go(gemm_f32_streamed_kernel<2>);
        case 4: return go(gemm_f32_streamed_kernel<4>);
        default: return go(gemm_f32_streamed_kernel<8>);
    }
}
