// C[M, N] = A[M, K] . W[N, K]^T in float32 on the bf16 matrix instruction (v_mfma_f32_16x16x32_bf16: exact products, float32 sums), the
// matrix product of the float32 path.  W is row-major [out, in] as the reference keeps it (src/model.c:157-158); out[row] = sum_col
// W[row, col] x[col] (src/quant/f32_scalar.c:4-32).
//
// A float32 number is the sum of three bf16 numbers (gf_split: 3 x 8 bits, nothing is lost above 7.7e-34), a product of two nine products of
// those; six are formed, and the three left out, the second parts times the third and the third times themselves, are at most 2^-24
// of the product, of either sign.  The float32 instruction is the slower way to the same sum by 2.7: it takes 256 cycles for 16 x 16 x 32
// on a SIMD, six of these 96.  Fewer links in a chain of sums (six of 32 products in place of 32 of four a chunk) round less: error against
// 64 bits over the largest of a row's sums (2-norms), float32 instruction -> this: 1,000 x 2,048 x 2,048 normal numbers 2.17e-7 -> 1.73e-7,
// 16 x 2,048 x 5,632 2.36e-7 -> 2.05e-7, all positive 7.32e-8 -> 6.84e-8, 64 x 256 x 14,336 2.81e-7 -> 2.58e-7, rows with a few columns a
// hundred times the others 2.10e-7 -> 1.71e-7.  Smaller
// operands, infinite ones and what is no number: see gf_again.
//
// One order of summation, a function of K alone, whatever M, N, the kernel and its tiles are, so that a row's result does
// not depend on what else is in the batch: K is cut in chunks of 128; a chunk is summed from nothing, its four blocks of 32 columns one
// after the other, a block by six instructions, the largest product last (gf_term); lane group g takes columns 4 g .. 4 g + 3 of
// both halves of a block.  The chunks' sums are added in order.  The cut is what lets a product of few rows spread one output's K over the
// waves of a workgroup (and it keeps the rounding error at that of a sum of 128 and of K / 128 terms).
//
// gemm_f32_streamed_kernel, up to 16 rows over a streamed copy of W: see there.
// gemm_f32_stream_kernel, up to 16 rows over W itself: bound by the bytes of W.  A workgroup of 8 waves owns up to 16 columns
// and all of K; a wave takes every eighth chunk, asks for its whole 8 KB of W (and the rows' 128 columns of A) at once and
// leaves 16 x 16 sums in shared memory; then a thread an output adds them up in order.  us at one row, 1.5 GB of weights in
// turn, and at 6.5 TB/s: 11,264 x 2,048 24 (14), 2,048 x 5,632 19.5 (7), 32,000 x 2,048 52 (40), 28,672 x 4,096 103 (72); the
// vector kernel that walked K in one chain (gemm_tiled.hip) took 325 on the average of a layer's products, whatever the rows
// up to 16.  Its loads of W are plain: two of them take the halves of a line, and non-temporal ones were slower (11,264 x 2,048
// at 8 rows 25 -> 26 us, 32,000 x 2,048 59 -> 65).
// gemm_f32_chunks_kernel, more rows and few tiles; gemm_f32_tile_kernel, more: bound by the vector instructions that split the operands
// beside the matrix instruction, at many rows by both and the clock that power leaves them.  us, float32 instruction -> this, 11,264 x 2,048 /
// 2,048 x 5,632 / 3,072 x 2,048 / 2,048 x 2,048: 5,736 rows 1,905 -> 1,242 (213 TFLOP/s) / 980 -> 630 / 526 -> 389 / 370 -> 242; 512 rows 178 ->
// 137 / 95 -> 84 / 53 -> 50 / 38 -> 35; 256 rows 98 -> 82 / 55 -> 54 / 31 -> 35 / 22 -> 24; 199 rows 84 -> 80 / 53 -> 53 / 30 -> 35 / 22 -> 24; 144 rows
// 62 -> 77 / 52 -> 52 / 22 -> 25 / 21 -> 23; 128 rows 55 -> 53 / 37 -> 37 / 22 -> 25 / 16 -> 17; 64 rows 31 -> 38 / 36 -> 23 / 16 -> 18 / 16 -> 11; 33
// rows 33 -> 37 / 38 -> 22 / 16 -> 17 / 16 -> 11; 17 rows 24 -> 26 / 27 -> 21 / 12 -> 10 / 11 -> 10.  So at 33 to 320 rows a layer's first products can
// be slower (up to a quarter), and a layer of 130 to 170 rows is by a tenth: their tiles of 64 rows and more are half empty, and smaller ones
// split their operands too often.
#include "common.h"
#include <type_traits>

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define GF_CHUNK 128                 // columns of K whose products are summed from nothing
#define GF_BLOCKS (GF_CHUNK / 16)
#define GF_WAVES 8                   // waves of a workgroup of the streaming kernel
#define GF_ROUND 64                  // chunks whose sums the streaming kernel's shared memory holds at a time

struct GfArgs {
    const float* x;
    const float* w;
    float* y;
    int M, N, K;                     // N: rows of W
    int ldx, ldw, ldy;
    int cols;                        // columns a workgroup of the streaming kernel owns (<= 16)
    int glu;                         // y[M, N / 2] = act(gate) * up: 1, rows of W are gate and up rows in turns of 8; 2, all gate rows, then all
                                     // up rows (gemm_f32_stream_kernel alone)
    int act;
    int add;                         // y += the product (kernels of up to 16 rows, no glu)
    const float* norm_w;             // rows of x are normed on their way in: x * scale * norm_w; null: as they are
    float eps;
};

// A float32 number as three bf16 numbers, nearest first: what each leaves is exact, and the three hold all 24 bits.
typedef __bf16 gf_b8 __attribute__((ext_vector_type(8)));
struct GfSplit { gf_b8 h, m, l; };
// (Written out, since a vector's conversion back and forth costs a conversion more a number.)
__device__ __forceinline__ uint32_t gf_pair(float a, float b) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{a, b}, b2));
}
// x less one of two bf16 numbers (exact: v_dot2_f32_bf16 with -1 at its place and 0 at the other's, one instruction instead of a shift
// and a subtraction).  The factors come from registers: as an inline constant, -1 would be the float32 number's bits.
__device__ __forceinline__ float gf_less(float x, uint32_t two, uint32_t minus_one) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    asm("" : "+s"(minus_one));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, two), __builtin_bit_cast(b2, minus_one), x, false);
}
template <bool DOT = true> __device__ __forceinline__ void gf_split_pair(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
    h = gf_pair(a, b);
    if constexpr (DOT) {
        a = gf_less(a, h, 0x0000bf80u);
        b = gf_less(b, h, 0xbf800000u);
        m = gf_pair(a, b);
        l = gf_pair(gf_less(a, m, 0x0000bf80u), gf_less(b, m, 0xbf800000u));
    } else {
        a -= bf16lo_to_f32(h);
        b -= bf16hi_to_f32(h);
        m = gf_pair(a, b);
        l = gf_pair(a - bf16lo_to_f32(m), b - bf16hi_to_f32(m));
    }
}
template <bool DOT = true> __device__ __forceinline__ GfSplit gf_split(const f32x4& lo, const f32x4& hi) {
    uint4 h, m, l;
    gf_split_pair<DOT>(lo[0], lo[1], h.x, m.x, l.x);
    gf_split_pair<DOT>(lo[2], lo[3], h.y, m.y, l.y);
    gf_split_pair<DOT>(hi[0], hi[1], h.z, m.z, l.z);
    gf_split_pair<DOT>(hi[2], hi[3], h.w, m.w, l.w);
    return GfSplit{__builtin_bit_cast(gf_b8, h), __builtin_bit_cast(gf_b8, m), __builtin_bit_cast(gf_b8, l)};
}
// Product t of the six, the large one last.  The order of the small ones makes no difference against 64 bits (1.74e-7 of the result at K =
// 2,048 either way); it decides single roundings, and with them by how much ill-conditioned rows differ between a prompt in one step and the
// same in portions: the logits of a mixture of experts behind linear attention (100 tokens, 21 draws of its weights), the largest difference over
// their root mean square, float32 instruction 1.05e-5 on the mean and 2.32e-5 at the most, this order 0.95e-5 and 2.88e-5; in the draw that a
// test bounds by 2e-5 1.46e-5, 1.98e-5, with the third parts first 2.03e-5.  (From 64 bits whole and in portions 1.32e-5 and 1.39e-5 on the
// mean, this 1.12e-5 and 1.10e-5.)
template <int T> __device__ __forceinline__ f32x4 gf_term(const GfSplit& w, const GfSplit& x, const f32x4& acc) {
    const gf_b8 a = T == 0 || T == 2 ? w.m : T == 4 ? w.l : w.h, b = T == 0 || T == 1 ? x.m : T == 3 ? x.l : x.h;
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
}
__device__ __forceinline__ f32x4 gf_products(const GfSplit& w, const GfSplit& x, f32x4 acc) {
    acc = gf_term<0>(w, x, acc);
    acc = gf_term<1>(w, x, acc);
    acc = gf_term<2>(w, x, acc);
    acc = gf_term<3>(w, x, acc);
    acc = gf_term<4>(w, x, acc);
    return gf_term<5>(w, x, acc);
}
// An infinite operand's second and third part are no numbers (nor is the nearest bf16 number of one above 3.389e38 finite), and a part
// below 2^-133 is rounded, so that an operand below 2^-110 loses bits (2^-134 at the most, also below 2^-126: the instructions keep denormal
// numbers).  Results that are not finite, or so small that this could be seen, are formed again by the float32 instruction, from the
// operands as they are and in one order whatever the kernel: a chunk of 128 columns from nothing, 16 at a time, the chunks' sums in order.
// At or above GF_SMALL what is lost is below 2^-24 of the result while the numbers that the lost bits are multiplied by sum up to less than
// 2^50.  (Zero is kept: a row of zeros is none of these.  A sum whose operands all are below 2^-134 comes out as zero.)
#define GF_SMALL 0x1p-60f
__device__ __forceinline__ bool gf_stands(float v) { return (v == 0.f) | ((fabsf(v) >= GF_SMALL) & (fabsf(v) < INFINITY)); }
__device__ __forceinline__ bool gf_stands(const f32x4& v) { return gf_stands(v[0]) & gf_stands(v[1]) & gf_stands(v[2]) & gf_stands(v[3]); }
// w(k), x(k): a lane's four columns of the sixteen from k on, of its row
template <typename W, typename X> __device__ __forceinline__ f32x4 gf_again(int K, W w, X x) {
    f32x4 all = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int k0 = 0; k0 < K; k0 += GF_CHUNK) {
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int k = k0; k < min(k0 + GF_CHUNK, K); k += 16) {
            const f32x4 wv = w(k), xv = x(k);
#pragma unroll
            for (int e = 0; e < 4; ++e) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[e], xv[e], sum, 0, 0, 0);
        }
        all += sum;
    }
    return all;
}
// of a tile of sums as the instruction leaves them (lane r + 16 g: columns 4 g .. 4 g + 3 of row r) the one of this lane's row and column
__device__ __forceinline__ float gf_of_tile(const f32x4& tile, int row, int col) {
    float v = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float s = __shfl(tile[e], (row & 15) + 4 * (col & 12), BN_WAVE);
        v = (col & 3) == e ? s : v;
    }
    return v;
}

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
// Four numbers of a row of x, from column c, to shared memory: as they are, or as their parts, 32 columns' first, second and third ones
// behind each other (64 bytes each) in the order of the matrix instruction's lanes (column 16 h + 4 g + e at 8 g + 4 h + e)
__device__ __forceinline__ int gf_part_at(int c) { return (c >> 5) * 192 + (c >> 2 & 3) * 16 + (c >> 4 & 1) * 8; }
template <bool PARTS> __device__ __forceinline__ void gf_store_row(unsigned char* row, int c, const f32x4& v) {
    if constexpr (PARTS) {
        uint2 h, m, l;
        gf_split_pair(v[0], v[1], h.x, m.x, l.x);
        gf_split_pair(v[2], v[3], h.y, m.y, l.y);
        unsigned char* at = row + gf_part_at(c);
        *reinterpret_cast<uint2*>(at) = h;
        *reinterpret_cast<uint2*>(at + 64) = m;
        *reinterpret_cast<uint2*>(at + 128) = l;
    } else {
        *reinterpret_cast<f32x4*>(row + c * 4) = v;
    }
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
    template <bool PARTS> __device__ __forceinline__ void store(const GfArgs& a, int tid, const float* parts, unsigned char* rows, int row_bytes) {
        const int t = tid & 255, half = __builtin_amdgcn_readfirstlane(tid >> 8);
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const float scale = gf_norm_scale(a, parts, half + 2 * i);
#pragma unroll
            for (int k = 0; k < NV; ++k)
                if ((k * 256 + t) * 4 < a.K) gf_store_row<PARTS>(rows + (half + 2 * i) * row_bytes, (k * 256 + t) * 4, v[i][k] * scale * w[k]);
        }
    }
};
#define GF_NORM_LOADS 10             // (NR + 1) * NV at the most: what registers hold beside the first weights in flight

// NR, NV: as GfNorm's; NR 0: no norm.
template <int NR = 0, int NV = 1>
__global__ __launch_bounds__(64 * GF_WAVES, 4) void gemm_f32_stream_kernel(GfArgs a) {
    __shared__ float sums[GF_ROUND * 256];                       // [chunk][row][column]
    float scale = 1.f;                                           // of row r
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * a.cols;
    // lanes without a column or a row read their neighbour's (no other bytes, and no load under a branch); what they form is
    // not stored
    const int wrow = a.glu == 2 ? min(n0 / 2 + (r & 7), a.N / 2 - 1) + (r >> 3) * (a.N / 2) : min(n0 + min(r, a.cols - 1), a.N - 1);
    const float* wp = a.w + (size_t)wrow * a.ldw + 4 * g;
    const float* xp = a.x + (size_t)min(r, a.M - 1) * a.ldx + 4 * g;
    const int n_chunks = (a.K + GF_CHUNK - 1) / GF_CHUNK;
    // the output that this thread adds up
    const int m = tid >> 4, col = tid & 15, n = n0 + col;
    const bool mine = tid < 256 && m < a.M && col < a.cols && n < a.N;
    float tot = 0.f, old = 0.f;
    if (a.add && mine) old = a.y[(size_t)m * a.ldy + n];         // asked for before the weights
    if constexpr (NR > 0) {
        GfNorm<NR, NV> norm;
        norm.load(a, tid);
        norm.sum(a, tid, sums);                                  // where the chunks' sums come later
        bn_lds_barrier();
        scale = gf_norm_scale(a, sums, min(r, a.M - 1));
        bn_lds_barrier();
    }

    for (int c0 = 0; c0 < n_chunks; c0 += GF_ROUND) {
        const int c1 = min(n_chunks, c0 + GF_ROUND);
        auto chunk = [&](int c, auto whole) {
            const int k0 = c * GF_CHUNK;
            auto fetch = [&](const float* p, f32x4 (&v)[GF_BLOCKS]) {
#pragma unroll
                for (int j = 0; j < GF_BLOCKS; ++j)
                    v[j] = gf_load(p + k0 + 16 * j, decltype(whole)::value || k0 + 16 * j + 4 * g < a.K);
            };
            f32x4 wv[GF_BLOCKS], xv[GF_BLOCKS], acc = {0.f, 0.f, 0.f, 0.f};
            fetch(wp, wv);
            fetch(xp, xv);
            if constexpr (NR > 0) {
                f32x4 nw[GF_BLOCKS];
                fetch(a.norm_w + 4 * g, nw);
#pragma unroll
                for (int j = 0; j < GF_BLOCKS; ++j) xv[j] = xv[j] * scale * nw[j];
            }
#pragma unroll
            for (int j = 0; j < GF_BLOCKS; j += 2) acc = gf_products(gf_split(wv[j], wv[j + 1]), gf_split(xv[j], xv[j + 1]), acc);
            // lane: columns 4 g .. 4 g + 3 of row r
            *reinterpret_cast<f32x4*>(&sums[(c - c0) * 256 + 16 * r + 4 * g]) = acc;
        };
        for (int c = c0 + wave; c < c1; c += GF_WAVES) {
            if ((c + 1) * GF_CHUNK <= a.K) chunk(c, gf_true());
            else chunk(c, gf_false());
        }
        __syncthreads();
        if (tid < 256)
            for (int c = 0; c < c1 - c0; ++c) tot += sums[c * 256 + tid];
        if (c1 < n_chunks) __syncthreads();
    }
    if (tid < 256 && __builtin_expect(__any(!gf_stands(tot)), 0)) {          // see gf_again
        const f32x4 again = gf_again(a.K, [&](int k) { return gf_load(wp + k, k + 4 * g < a.K); }, [&](int k) {
            const f32x4 v = gf_load(xp + k, k + 4 * g < a.K);
            if constexpr (NR > 0) return v * scale * gf_load(a.norm_w + 4 * g + k, k + 4 * g < a.K);
            return v;
        });
        const float own = gf_of_tile(again, m, col);
        tot = gf_stands(tot) ? tot : own;
    }
    if (!a.glu) {
        if (mine) a.y[(size_t)m * a.ldy + n] = a.add ? old + tot : tot;
        return;
    }
    __syncthreads();
    if (tid < 256) sums[tid] = tot;
    __syncthreads();
    if (tid < 128 && tid / 8 < a.M && n0 / 2 + tid % 8 < a.N / 2)
        a.y[(size_t)(tid / 8) * a.ldy + n0 / 2 + tid % 8] = bn_gate_act(sums[tid / 8 * 16 + tid % 8], a.act) * sums[tid / 8 * 16 + 8 + tid % 8];
}

// ---------------------------------------------------------------------------------------
// The product of up to 16 rows over a streamed copy of W (common.h) whose K is whole chunks.  Bound by the bytes of W: over
// the row-major matrix a load takes 64 bytes of each of 16 rows, half of a cache line, and waits under a test; here it takes
// a tile, 1 KB in a run, non-temporally, in straight-line code, and the activations go through the wave's own shared memory, so that
// one row costs one load a chunk instead of eight, and are split there once instead of once a wave.  The same sums in the
// same order as the kernels around it (a chunk by itself, the chunks in order): the same bits.  XR: activation loads a lane
// and chunk, for up to 2 XR rows.  PARTS: staged rows lie there in parts (gf_streamed_parts).
//   us at 1 / 4 / 8 / 16 rows with cold weights in a graph of such launches, float32 instruction with two chunks a wave in flight -> this:
//   3,072 x 2,048 7.1 / 6.7 / 7.0 / 7.8 -> 6.6 / 6.3 / 6.8 / 7.7, 2,048 x 2,048 6.3 / 6.7 / 6.4 / 6.9 -> 5.9 / 6.5 / 6.1 / 7.1, 11,264 x 2,048
//   17.6 / 17.6 / 18.5 / 23.0 -> 16.6 / 16.6 / 17.9 / 22.3, 2,048 x 5,632 12.8 / 14.3 / 13.4 / 15.4 -> 12.0 / 14.0 / 13.3 / 15.5, 32,000 x 2,048
//   42.3 / 42.9 / 43.7 / 55.4 -> 41.7 / 41.6 / 42.4 / 54.6.  Half a chunk of W is
//   loaded and multiplied at a time, the two halves in turn: whole chunks take 118 registers and more instead of 78, and from 5 rows on
//   they spill.  Behind a norm of up to 4 rows, whose registers are gone by then, whole chunks are faster: 3,072 x 2,048 6.5 against 6.9.
// bytes between staged rows of n activations, as they are or in parts
__host__ __device__ constexpr int gf_row_bytes(int n, bool parts) { return n * (parts ? 6 : 4) + 16; }

// NV > 0: behind a norm (GfNorm<XR, NV>; every wave has a chunk).  The normed rows are staged once, all of them, by the threads
// that summed their squares, and the waves read their chunks from there.
template <int XR, bool PARTS, int NV = 0>
__global__ __launch_bounds__(64 * GF_WAVES, XR == 8 ? 2 : 4) void gemm_f32_streamed_kernel(GfArgs a, int k_tiles) {
    constexpr int ROWS = 2 * XR;
    constexpr bool NORM = NV > 0;
    // blocks of W that are loaded and multiplied together: half a chunk, or all of it
    constexpr bool HALVES = !NORM || XR >= 4 || NV > 2;
    constexpr int UNIT = HALVES ? GF_BLOCKS / 2 : GF_BLOCKS;
    extern __shared__ __align__(16) unsigned char smem[];
    const int row_bytes = gf_row_bytes(NORM ? a.K : GF_CHUNK, PARTS);
    float* parts = reinterpret_cast<float*>(smem + (NORM ? 1 : GF_WAVES) * ROWS * row_bytes);    // of the rows' squares
    float* sums = parts + (NORM ? ROWS * 4 : 0);                             // [chunk][row][column]
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
    unsigned char* xs = smem + (NORM ? 0 : wave * ROWS * row_bytes);
    unsigned char* park_at = xs + (lane >> 5) * row_bytes;
    const unsigned char* read_at = xs + min(r, a.M - 1) * row_bytes + g * 16;
    f32x4 x[XR];
    auto load_x = [&](int c) {
        if (NORM) return;
#pragma unroll
        for (int i = 0; i < XR; ++i) x[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(xb, x_at[i], c * (GF_CHUNK * 4), 0));
    };
    auto load_w = [&](f32x4 (&w)[UNIT], int c, int h = 0) {                   // chunk c, from its block 4 h on
        unsigned at = (c * GF_BLOCKS + 4 * h) * tile;
#pragma unroll
        for (int j = 0; j < UNIT; ++j, at += tile)
            w[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(wb, w_at, at, BN_BUFFER_NT));
        __builtin_amdgcn_sched_barrier(0);
    };
    auto park = [&]() {
        if (NORM) return;
#pragma unroll
        for (int i = 0; i < XR; ++i) gf_store_row<PARTS>(park_at + 2 * i * row_bytes, (lane & 31) * 4, x[i]);
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    f32x4 acc;
    auto multiply = [&](const f32x4 (&w)[UNIT], int c, int h = 0) {
        const unsigned char* from = read_at + (NORM ? c * (GF_CHUNK * (PARTS ? 6 : 4)) : 0);
        auto rows = [&](int q) {                                             // block q's of x
            if constexpr (PARTS) {
                const unsigned char* at = from + q * 192;
                return GfSplit{*reinterpret_cast<const gf_b8*>(at), *reinterpret_cast<const gf_b8*>(at + 64), *reinterpret_cast<const gf_b8*>(at + 128)};
            } else {
                return gf_split(*reinterpret_cast<const f32x4*>(from + q * 128), *reinterpret_cast<const f32x4*>(from + q * 128 + 64));
            }
        };
        if (h == 0) acc = 0.f;
#pragma unroll
        for (int q = 0; q < UNIT / 2; ++q) {
            const GfSplit v = rows(2 * h + q);
            acc = gf_products(gf_split(w[2 * q], w[2 * q + 1]), v, acc);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (HALVES && h == 0) return;
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
        norm.sum(a, tid, parts);
        bn_lds_barrier();
        norm.template store<PARTS>(a, tid, parts, smem, row_bytes);
        bn_lds_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (HALVES) {
        if (n > 0) {
            f32x4 p[UNIT], q[UNIT];
            int c = wave;
            load_x(c);
            load_w(p, c, 0);
            stage();
            load_w(q, c, 1);
#pragma unroll 1
            for (int left = n; left > 1; --left, c += D) {
                park();
                load_x(c + D);
                multiply(p, c, 0);
                load_w(p, c + D, 0);
                multiply(q, c, 1);
                load_w(q, c + D, 1);
            }
            park();
            multiply(p, c, 0);
            multiply(q, c, 1);
        }
    } else if (n == 1) {
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
    if (tid >= (ROWS > 4 ? ROWS * 16 : BN_WAVE)) return;                     // (whole waves stay)
    float tot = 0.f;
#pragma unroll 8
    for (int c = 0; c < n_chunks; ++c) tot += sums[(size_t)c * (ROWS * 16) + tid % (ROWS * 16)];
    const int m = tid >> 4, col = tid & 15, n0 = blockIdx.x * a.cols;
    if (__builtin_expect(__any(!gf_stands(tot)), 0)) {                       // see gf_again
        int own_lane = lane;
        asm volatile("" : "+v"(own_lane));                                   // (nothing of this is formed ahead and kept)
        const int row = min(own_lane & 15, a.M - 1), g4 = own_lane >> 4 << 2;
        const float* from = a.w + (size_t)blockIdx.x * k_tiles * (tile / 4) + g4 * a.cols + min(own_lane & 15, a.cols - 1) * 4;
        const float* x_from = a.x + (size_t)row * a.ldx + g4;
        const f32x4 again = gf_again(a.K, [&](int k) { return *reinterpret_cast<const f32x4*>(from + k / 16 * (tile / 4)); }, [&](int k) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(x_from + k);
            if constexpr (NORM) return v * gf_norm_scale(a, parts, row) * *reinterpret_cast<const f32x4*>(a.norm_w + g4 + k);
            return v;
        });
        const float own = gf_of_tile(again, m, col);
        tot = gf_stands(tot) ? tot : own;
    }
    if (a.glu) {                                                             // columns 0..7 of the tile are gates, 8..15 their ups
        const float up = bn_lane_xor<8>(tot);
        if (m < a.M && col < 8) a.y[(size_t)m * a.ldy + n0 / 2 + col] = bn_gate_act(tot, a.act) * up;
    } else if (m < a.M && col < a.cols && n0 + col < a.N) {
        a.y[(size_t)m * a.ldy + n0 + col] = a.add ? old + tot : tot;
    }
}

#define GF_BK 32

// consecutive workgroups go to consecutive XCDs: each XCD gets a run of tiles
__device__ __forceinline__ int gf_run_of_xcd(int id, int total) {
    const int per = total / 8, rest = total % 8, xcd = id % 8;
    return xcd * per + min(xcd, rest) + id / 8;
}
// More than 16 rows and few tiles.  A workgroup owns 16 MT rows and 16 NT columns, its waves take K's chunks in turns, as the streaming
// kernels': no wave waits for another inside a chunk, every one brings its operands itself (memory to shared memory, two blocks of 32
// columns on their way) and splits them between the products of the block before.  Bound by those vector instructions: 17.7 us for 128 rows
// of 2,048 x 2,048 where the tiles below, whose waves wait for each other every block, take 22 and more; what it costs is that an
// operand is split by every workgroup that needs it, so large products are the tiles'.
template <int MT, int NT, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void gemm_f32_chunks_kernel(GfArgs a, int m_tiles, int n_tiles) {
    constexpr int THREADS = 64 * WAVES, ROWS = 16 * MT, COLS = 16 * NT, STRIDE = COLS + 4, OUT = ROWS * COLS / THREADS, FRAGS = MT + NT;
    static_assert(OUT * THREADS == ROWS * COLS, "every thread adds up as many outputs");
    // rows of a block as they come from memory, a wave's own
    __shared__ __align__(1024) unsigned char s0[WAVES * FRAGS * 2048], s1[WAVES * FRAGS * 2048];
    __shared__ float sums[WAVES][ROWS * STRIDE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int id = gf_run_of_xcd(blockIdx.x, m_tiles * n_tiles);
    const int m0 = id % m_tiles * ROWS, n0 = id / m_tiles * COLS;
    const auto xb = bn_buffer(a.x + (size_t)m0 * a.ldx, ((min(ROWS, a.M - m0) - 1) * a.ldx + a.K) * 4);
    const auto wb = bn_buffer(a.w + (size_t)n0 * a.ldw, ((min(COLS, a.N - n0) - 1) * a.ldw + a.K) * 4);
    // a load is eight rows; chunk c of 16 bytes of row r lies at c ^ (r / 2 % 8)
    unsigned xo[2], wo[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int row = 8 * i + (lane >> 3), c = 4 * ((lane & 7) ^ ((row >> 1) & 7));
        xo[i] = (row * a.ldx + c) * 4;
        wo[i] = (row * a.ldw + c) * 4;
    }
    const int blocks = (a.K + GF_BK - 1) / GF_BK, n_chunks = (a.K + GF_CHUNK - 1) / GF_CHUNK;
    auto place = [&](int b) { return ((b >> 2) * WAVES + wave) * 4 + (b & 3); };         // block b of this wave, the waves take chunks in turns
    auto load = [&](unsigned char* to, int b) {
        const unsigned k = min(place(b), blocks - 1) * (GF_BK * 4);
#pragma unroll
        for (int f = 0; f < FRAGS; ++f)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                bn_load_to_lds(f < MT ? xb : wb, to + (wave * FRAGS + f) * 2048 + h * 1024, f < MT ? xo[h] : wo[h],
                               k + (f < MT ? 64 * f * a.ldx : 64 * (f - MT) * a.ldw));
    };
    const int at0 = r * 128 + ((g ^ (r >> 1)) << 4), at1 = r * 128 + (((4 + g) ^ (r >> 1)) << 4);
    f32x4 raw[FRAGS][2], acc[NT][MT];
    auto read = [&]() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };            // rows that new ones may take the place of
    auto get = [&](const unsigned char* from) {                  // (the younger block may be on its way)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * FRAGS) : "memory");
#pragma unroll
        for (int f = 0; f < FRAGS; ++f) {
            raw[f][0] = *reinterpret_cast<const f32x4*>(from + (wave * FRAGS + f) * 2048 + at0);
            raw[f][1] = *reinterpret_cast<const f32x4*>(from + (wave * FRAGS + f) * 2048 + at1);
        }
    };
    GfSplit op[2][FRAGS];
    // columns past K (another row's) are zeros
    auto clear = [&](int b) {
        const int k = place(b) * GF_BK + 4 * g;
        if (k - 4 * g + GF_BK <= a.K) return;
#pragma unroll
        for (int f = 0; f < FRAGS; ++f) {
            if (k >= a.K) raw[f][0] = 0.f;
            if (k + 16 >= a.K) raw[f][1] = 0.f;
        }
    };
    // the products of a block, and between them the parts of the next one's operands
    auto turn = [&](int c, auto u_) {
        constexpr int u = decltype(u_)::value;
        unsigned char* next = u & 1 ? s0 : s1;
        const int b = c + u + 1;
        get(next);
        clear(b);
        __builtin_amdgcn_sched_barrier(0);
        auto term = [&](auto t_) {
            constexpr int t = decltype(t_)::value;
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < MT; ++j)
                    acc[i][j] = gf_term<t>(op[u & 1][MT + i], op[u & 1][j], u == 0 && t == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[i][j]);
#pragma unroll
            for (int f = 0; f < FRAGS; ++f)
                if (f * 6 / FRAGS == t) op[(u + 1) & 1][f] = gf_split(raw[f][0], raw[f][1]);
            __builtin_amdgcn_sched_barrier(0);
        };
        term(std::integral_constant<int, 0>());
        term(std::integral_constant<int, 1>());
        term(std::integral_constant<int, 2>());
        term(std::integral_constant<int, 3>());
        term(std::integral_constant<int, 4>());
        term(std::integral_constant<int, 5>());
        read();
        load(next, b + 2);
        __builtin_amdgcn_sched_barrier(0);                       // (the wait counts loads in this order)
    };
    float tot[OUT];
#pragma unroll
    for (int o = 0; o < OUT; ++o) tot[o] = 0.f;
    load(s0, 0);
    __builtin_amdgcn_sched_barrier(0);
    load(s1, 1);
    __builtin_amdgcn_sched_barrier(0);
    get(s0);
    clear(0);
#pragma unroll
    for (int f = 0; f < FRAGS; ++f) op[0][f] = gf_split(raw[f][0], raw[f][1]);
    __builtin_amdgcn_sched_barrier(0);
    read();
    load(s0, 2);
    __builtin_amdgcn_sched_barrier(0);
    using std::integral_constant;
    for (int c0 = 0; c0 < n_chunks; c0 += WAVES) {               // (a wave without a chunk forms the sums of zeros, which nobody adds)
        const int c = c0 / WAVES * 4;
        turn(c, integral_constant<int, 0>());
        turn(c, integral_constant<int, 1>());
        turn(c, integral_constant<int, 2>());
        turn(c, integral_constant<int, 3>());
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int j = 0; j < MT; ++j) *reinterpret_cast<f32x4*>(&sums[wave][(16 * j + r) * STRIDE + 16 * i + 4 * g]) = acc[i][j];
        bn_lds_barrier();
#pragma unroll
        for (int o = 0; o < OUT; ++o) {
            const int idx = tid + o * THREADS, p = idx / COLS * STRIDE + idx % COLS;
#pragma unroll
            for (int w = 0; w < WAVES; ++w)
                if (c0 + w < n_chunks) tot[o] += sums[w][p];
        }
        bn_lds_barrier();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");             // nothing is on its way into shared memory when the wave ends
#pragma unroll
    for (int o = 0; o < OUT; ++o) {
        if (__builtin_expect(!__any(!gf_stands(tot[o])), 1)) continue;       // see gf_again
        const int idx = tid + o * THREADS, m = idx / COLS, n = idx % COLS, j = __builtin_amdgcn_readfirstlane(m / 16);
        const float* xp = a.x + (size_t)min(m0 + 16 * j + r, a.M - 1) * a.ldx + 4 * g;
#pragma unroll 1
        for (int i = 0; i < NT; ++i) {                           // (a wave's outputs lie in one row of tiles)
            const float* wp = a.w + (size_t)min(n0 + 16 * i + r, a.N - 1) * a.ldw + 4 * g;
            const f32x4 again = gf_again(a.K, [&](int k) { return gf_load(wp + k, k + 4 * g < a.K); }, [&](int k) { return gf_load(xp + k, k + 4 * g < a.K); });
            const float own = gf_of_tile(again, m, n);
            tot[o] = n / 16 != i || gf_stands(tot[o]) ? tot[o] : own;
        }
    }
    if (a.glu) {
#pragma unroll
        for (int o = 0; o < OUT; ++o) {
            const int idx = tid + o * THREADS;
            sums[0][idx / COLS * STRIDE + idx % COLS] = tot[o];
        }
        bn_lds_barrier();
        for (int idx = tid; idx < ROWS * COLS / 2; idx += THREADS) {
            const int m = idx / (COLS / 2), n = idx % (COLS / 2);
            const float* p = &sums[0][m * STRIDE + n / 8 * 16 + n % 8];
            if (m0 + m < a.M && n0 / 2 + n < a.N / 2) a.y[(size_t)(m0 + m) * a.ldy + n0 / 2 + n] = bn_gate_act(p[0], a.act) * p[8];
        }
        return;
    }
#pragma unroll
    for (int o = 0; o < OUT; ++o) {
        const int idx = tid + o * THREADS, m = m0 + idx / COLS, n = n0 + idx % COLS;
        if (m < a.M && n < a.N) a.y[(size_t)m * a.ldy + n] = tot[o];
    }
}

// A workgroup owns BM rows of A and 64 NW rows of W; a wave all of the former and 16 NW of the latter.  The rows of A are split once a
// workgroup and lie in shared memory in parts (two stages); W's are the wave's own, split where they are used: straight to registers, or
// through shared memory by loads of whole lines, which is faster for 128 x 128 (5,736 rows of 11,264 x 2,048 1,217 us against 1,259) and
// narrow tiles (1,602 against 1,609, 199 rows with K in two 33 against 36) and slower for 64 x 128 (1,398 against 1,317).  KG groups of
// four waves take the chunks of K in turns where a launch has a tile a CU, and hand their sums to the first.  WHOLE: K is whole blocks of 32.
// The large tile is bound by the matrix and the vector unit together: the instruction is busy half of the time, one group's splitting
// another half, and the clock at 2.1 GHz (the same with loads of W in another order, deeper rings, and pairs of row tiles at a time).
// v_dot2 in gf_split takes 44 -> 28 instructions for eight numbers and stands in the matrix unit's way: small tiles take it (199 rows 55 ->
// 53 us), large ones do not (1,218 against 1,325).
template <int BM, int NW, int KG, bool WHOLE>
__global__ __launch_bounds__(256 * KG, 2) void gemm_f32_tile_kernel(GfArgs a, int m_tiles, int n_tiles) {
    constexpr int BN = 64 * NW, MT = BM / 16, PLANE = BM * 64, STAGE = 3 * PLANE;
    constexpr int XL = (BM * 4 + 255) / 256;                     // staged items a thread and block
    constexpr int JG = NW == 1 ? 2 : 1, GROUPS = MT / JG;        // row tiles whose products are formed together: chains of six wait for each other
    constexpr bool DIRECT = NW == 2 && BM < 128, DOT = NW == 1;              // W's rows straight to registers; gf_split's form
    __shared__ __align__(1024) unsigned char b0[KG * STAGE], b1[KG * STAGE];
    constexpr int OWN = DIRECT ? 16 : KG * 4 * NW * 2048;        // W's rows, a wave's own
    __shared__ __align__(1024) unsigned char w0[OWN], w1[OWN];
    __shared__ f32x4 handed[KG > 1 ? (KG - 1) * NW * MT * 256 : 1];
    const int tid = threadIdx.x & 255, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kg = KG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
    const int r = lane & 15, g = lane >> 4;
    // an XCD walks its run in bands of 8 row tiles, so that what runs on it together shares its operands in that L2
    const int id = gf_run_of_xcd(blockIdx.x, m_tiles * n_tiles);
    const int band = id / (8 * n_tiles), in_band = id - band * 8 * n_tiles;
    const int band_rows = min(8, m_tiles - band * 8);
    const int m0 = (band * 8 + in_band % band_rows) * BM, n0 = (in_band / band_rows) * BN + wave * 16 * NW;

    f32x4 acc[NW][MT], tot[NW][MT];
#pragma unroll
    for (int i = 0; i < NW; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) tot[i][j] = 0.f;

    // What lies past the matrices lies past the buffers' ends (or is another row's, and cleared).  x: item i of a thread is row tid / 4 +
    // 64 i, columns 4 sg .. + 3 of both blocks of 16; neighbouring lanes ask for neighbouring 16 bytes.  W through shared memory: load i of
    // a wave is rows 8 i .. + 7, whose chunk c of 16 bytes lies at c ^ (row / 2 % 8).
    const int sr = tid >> 2, sg = tid & 3;
    const bool stages = BM >= 64 || tid < 4 * BM;
    const auto xb = bn_buffer(a.x + (size_t)m0 * a.ldx, ((min(BM, a.M - m0) - 1) * a.ldx + a.K) * 4);
    const int nb = min(n0, a.N - 1);                             // (a wave without columns)
    const auto wb = bn_buffer(a.w + (size_t)nb * a.ldw, ((min(16 * NW, a.N - nb) - 1) * a.ldw + a.K) * 4);
    unsigned xo[XL], wo[2 * NW];
#pragma unroll
    for (int i = 0; i < XL; ++i) xo[i] = ((sr + 64 * i) * a.ldx + 4 * sg) * 4;
#pragma unroll
    for (int i = 0; i < 2 * NW; ++i) {
        const int row = DIRECT ? 16 * (i / 2) + r : 8 * i + (lane >> 3);
        wo[i] = (row * a.ldw + (DIRECT ? 16 * (i % 2) + 4 * g : 4 * ((lane & 7) ^ ((row >> 1) & 7)))) * 4;
    }
    const int blocks = (a.K + GF_BK - 1) / GF_BK;
    f32x4 xr[XL][2], wr[NW][2];
    // block b of this group of waves: the groups take the chunks in turns
    auto place = [&](int b) { return KG == 1 ? b : ((b >> 2) * KG + kg) * 4 + (b & 3); };
    auto offset = [&](int b) { return min(place(b), blocks - 1) * (GF_BK * 4); };
    auto load_x = [&](int i, int b) {
#pragma unroll
        for (int h = 0; h < 2; ++h) xr[i][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(xb, xo[i] + 64 * h, offset(b), 0));
    };
    auto load_w = [&](unsigned char* to, int i, int b) {         // rows 16 i .. + 15
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if constexpr (DIRECT) wr[i][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(wb, wo[2 * i + h], offset(b), 0));
            else bn_load_to_lds(wb, to + ((kg * 4 + wave) * NW + i) * 2048 + h * 1024, wo[2 * i + h], offset(b));
        }
    };
    // columns past K (another row's, or none) are zeros
    auto clear = [&](int b) {
        if (WHOLE && KG == 1) return;
        const int k = place(b) * GF_BK + 4 * sg;
        if (k - 4 * sg + GF_BK <= a.K) return;
#pragma unroll
        for (int i = 0; i < XL; ++i) {
            if (k >= a.K) xr[i][0] = 0.f;
            if (k + 16 >= a.K) xr[i][1] = 0.f;
        }
    };
    const int at0 = r * 128 + ((g ^ (r >> 1)) << 4), at1 = r * 128 + (((4 + g) ^ (r >> 1)) << 4);
    auto get_w = [&](const unsigned char* from, int i, int b) {
        const unsigned char* q = from + (DIRECT ? 0 : ((kg * 4 + wave) * NW + i) * 2048);
        f32x4 lo = DIRECT ? wr[i][0] : *reinterpret_cast<const f32x4*>(q + at0), hi = DIRECT ? wr[i][1] : *reinterpret_cast<const f32x4*>(q + at1);
        if (!WHOLE) {
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
            lo = place(b) * GF_BK + 4 * g < a.K ? lo : zero;
            hi = place(b) * GF_BK + 4 * g + 16 < a.K ? hi : zero;
        }
        return gf_split<DOT>(lo, hi);
    };
    // A staged block of 16 rows x 32 columns is 1 KB a part, lane r + 16 g's 16 bytes at 256 g + 16 (r ^ 4 (-g % 4)): no bank conflicts
    // where the sixteen lanes that shared memory serves together are of one row group or of two, nor among the writers' 4 x 4.
    const int put_at = kg * STAGE + (sr >> 4) * 1024 + sg * 256 + ((sr & 15) ^ (4 * (-sg & 3))) * 16;
    const int get_at = kg * STAGE + g * 256 + (r ^ (4 * (-g & 3))) * 16;
    auto put = [&](unsigned char* to, int i) {
        if (!stages) return;
        const GfSplit p = gf_split<DOT>(xr[i][0], xr[i][1]);
        unsigned char* q = to + put_at + i * 4096;
        *reinterpret_cast<gf_b8*>(q) = p.h;
        *reinterpret_cast<gf_b8*>(q + PLANE) = p.m;
        *reinterpret_cast<gf_b8*>(q + 2 * PLANE) = p.l;
    };
    auto get = [&](GfSplit (&to)[JG], const unsigned char* stage, int group) {
#pragma unroll
        for (int j = 0; j < JG; ++j) {
            const unsigned char* q = stage + get_at + (group * JG + j) * 1024;
            to[j] = GfSplit{*reinterpret_cast<const gf_b8*>(q), *reinterpret_cast<const gf_b8*>(q + PLANE), *reinterpret_cast<const gf_b8*>(q + 2 * PLANE)};
        }
    };
    // loads into shared memory of two blocks are on their way at a time: the older one's have arrived (whatever else was asked for since)
    auto arrived = [&]() {
        if (!DIRECT) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NW) : "memory");
    };
    // A block: its products group by group, and between them what the next block waits for, the parts of W's rows and rows of x into the
    // other stage.  The stages change hands in front of the last group, whose operands are in registers by then.
    GfSplit ws[2][NW], xs[2][JG];
    constexpr int PIECES = XL + NW, SPREAD = GROUPS > 1 ? GROUPS - 1 : 1;
    auto turn = [&](int c, auto u_) {
        constexpr int u = decltype(u_)::value;
        const unsigned char* now = u & 1 ? b1 : b0;
        unsigned char *next = u & 1 ? b0 : b1, *wn = u & 1 ? w0 : w1;
        const int b = c + u + 1;                                 // the block that is prepared
        clear(b);
        arrived();
#pragma unroll
        for (int q = 0; q < GROUPS; ++q) {
            constexpr bool one = GROUPS == 1;
            const int at = u * GROUPS + q;                       // groups take turns at the two sets of operands
            if (q == GROUPS - 1 && !one) {
                __builtin_amdgcn_sched_barrier(0);
                bn_lds_barrier();
            }
            if (!one) get(xs[(at + 1) & 1], q == GROUPS - 1 ? next : now, q == GROUPS - 1 ? 0 : q + 1);
#pragma unroll
            for (int p = 0; p < PIECES; ++p) {
                if (p * SPREAD / PIECES != q) continue;
                if (p < NW) {
                    ws[(u + 1) & 1][p] = get_w(wn, p, b);
                    if (DIRECT) load_w(wn, p, b + 1);
                } else {
                    put(next, p - NW);
                    load_x(p - NW, b + 1);
                }
            }
            if (one) {
                bn_lds_barrier();
                get(xs[(at + 1) & 1], next, 0);
            }
            auto term = [&](auto t) {
#pragma unroll
                for (int j = 0; j < JG; ++j)
#pragma unroll
                    for (int i = 0; i < NW; ++i)
                        acc[i][q * JG + j] = gf_term<decltype(t)::value>(ws[u & 1][i], xs[at & 1][j], u == 0 && decltype(t)::value == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[i][q * JG + j]);
            };
            term(std::integral_constant<int, 0>());
            term(std::integral_constant<int, 1>());
            term(std::integral_constant<int, 2>());
            term(std::integral_constant<int, 3>());
            term(std::integral_constant<int, 4>());
            term(std::integral_constant<int, 5>());
            __builtin_amdgcn_sched_barrier(0);
        }
        if (!DIRECT) {                                           // the block's rows of W were read in front of the barrier
#pragma unroll
            for (int i = 0; i < NW; ++i) load_w(wn, i, b + 2);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // the sums of a chunk (of the groups' chunks, in their order) join the totals, which the first group keeps
    auto fold = [&]() {
        if (KG > 1) {
            if (kg > 0) {
#pragma unroll
                for (int i = 0; i < NW; ++i)
#pragma unroll
                    for (int j = 0; j < MT; ++j) handed[(((kg - 1) * NW + i) * MT + j) * 256 + tid] = acc[i][j];
            }
            bn_lds_barrier();                                    // (the next chunks' blocks hold the barrier behind the reads)
        }
        if (KG > 1 && kg > 0) return;
#pragma unroll
        for (int i = 0; i < NW; ++i)
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                tot[i][j] += acc[i][j];
#pragma unroll
                for (int k = 1; k < KG; ++k) tot[i][j] += handed[(((k - 1) * NW + i) * MT + j) * 256 + tid];
            }
    };
#pragma unroll
    for (int i = 0; i < NW; ++i) load_w(w0, i, 0);
#pragma unroll
    for (int i = 0; i < XL; ++i) load_x(i, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (!DIRECT) {
#pragma unroll
        for (int i = 0; i < NW; ++i) load_w(w1, i, 1);
        __builtin_amdgcn_sched_barrier(0);
    }
    clear(0);
    arrived();
#pragma unroll
    for (int i = 0; i < NW; ++i) ws[0][i] = get_w(w0, i, 0);
#pragma unroll
    for (int i = 0; i < XL; ++i) put(b0, i);
    __builtin_amdgcn_sched_barrier(0);
    bn_lds_barrier();                                            // (w0 has been read as well)
#pragma unroll
    for (int i = 0; i < XL; ++i) load_x(i, 1);
#pragma unroll
    for (int i = 0; i < NW; ++i) load_w(w0, i, DIRECT ? 1 : 2);
    __builtin_amdgcn_sched_barrier(0);
    get(xs[0], b0, 0);
    using std::integral_constant;
    const int mine = KG > 1 ? (blocks + 4 * KG - 1) / (4 * KG) * 4 : blocks;             // several groups: whole chunks, past K of zeros
    int c = 0;
#pragma unroll 1
    for (; c + 4 <= mine; c += 4) {
        turn(c, integral_constant<int, 0>());
        turn(c, integral_constant<int, 1>());
        turn(c, integral_constant<int, 2>());
        turn(c, integral_constant<int, 3>());
        fold();
    }
    if (KG == 1 && c < mine) {
        turn(c, integral_constant<int, 0>());
        if (c + 1 < mine) turn(c, integral_constant<int, 1>());
        if (c + 2 < mine) turn(c, integral_constant<int, 2>());
        fold();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");             // nothing is on its way into shared memory when a wave ends
    if (kg > 0) return;
    bool fine = true;
#pragma unroll
    for (int i = 0; i < NW; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) fine = fine && gf_stands(tot[i][j]);
    if (__builtin_expect(__any(!fine), 0)) {                     // see gf_again
#pragma unroll
        for (int i = 0; i < NW; ++i)
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                const float* wp = a.w + (size_t)min(n0 + 16 * i + r, a.N - 1) * a.ldw + 4 * g;
                const float* xp = a.x + (size_t)min(m0 + 16 * j + r, a.M - 1) * a.ldx + 4 * g;
                const f32x4 again = gf_again(a.K, [&](int k) { return gf_load(wp + k, k + 4 * g < a.K); }, [&](int k) { return gf_load(xp + k, k + 4 * g < a.K); });
#pragma unroll
                for (int e = 0; e < 4; ++e) tot[i][j][e] = gf_stands(tot[i][j][e]) ? tot[i][j][e] : again[e];
            }
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        const int n = n0 + 16 * i + 4 * g;
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const int m = m0 + 16 * j + r;
            if (a.glu) {                                         // lanes with g < 2 hold gates, the lane 32 further their ups
                f32x4 up;
#pragma unroll
                for (int e = 0; e < 4; ++e) up[e] = __shfl_xor(tot[i][j][e], 32, BN_WAVE);
                if (g < 2 && m < a.M && n < a.N) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        a.y[(size_t)m * a.ldy + (n0 + 16 * i) / 2 + 4 * g + e] = bn_gate_act(tot[i][j][e], a.act) * up[e];
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

template <int NR = 0, int NV = 1>
static int gf_launch_stream(const GfArgs& a, hipStream_t s) {
    hipLaunchKernelGGL((gemm_f32_stream_kernel<NR, NV>), dim3((a.N + a.cols - 1) / a.cols), dim3(64 * GF_WAVES), 0, s, a);
    return bn_launch_status();
}

template <int MT, int NT, int WAVES>
static int gf_launch_chunks(const GfArgs& a, hipStream_t s) {
    const int mt = (a.M + 16 * MT - 1) / (16 * MT), nt = (a.N + 16 * NT - 1) / (16 * NT);
    hipLaunchKernelGGL((gemm_f32_chunks_kernel<MT, NT, WAVES>), dim3(mt * nt), dim3(64 * WAVES), 0, s, a, mt, nt);
    return bn_launch_status();
}

template <int BM, int NW, int KG, bool WHOLE>
static int gf_launch_tile(const GfArgs& a, hipStream_t s) {
    const int mt = (a.M + BM - 1) / BM, nt = (a.N + 64 * NW - 1) / (64 * NW);
    if (WHOLE && a.K % GF_BK) return BN_ERR_ARG;
    hipLaunchKernelGGL((gemm_f32_tile_kernel<BM, NW, KG, WHOLE>), dim3(mt * nt), dim3(256 * KG), 0, s, a, mt, nt);
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

// The form of a product of more than 16 rows with the least time for the busiest CU: ns a block of 32 columns of K with n tiles a CU, first
// + many n (fitted at 1,024 to 14,336 columns, n = 1 to 248: of 415 sizes, 17 to 5,736 rows of twelve matrices, what it takes is 0.4 % behind the
// fastest form on the mean and 6 to 13 % at 68 to 128 rows of 28,672 x 4,096, the worst).  A launch that gives a CU one tile or two takes a tile's K
// apart over more waves, many tiles a CU take the large ones, which split and stage their operands least.  us, 128 x 128 / 64 x 128 / its K
// in two / 64 x 64 / its K in two / 32 x 64 in four / 32 x 32 chunks / 32 x 16 chunks: 5,736 rows of 11,264 x 2,048 1,217 / 1,317 / 1,545 /
// 1,602 / 2,006 / 2,410 / 3,745 / 4,423; 1,000 of 2,048 x 5,632 220 / 146 / 131 / 156 / 175 / 203 / 290 / 415; 199 of 3,072 x 2,048 89 / 55 / 48 /
// 40 / 36 / 42 / 45 / 48; 128 of 2,048 x 2,048 85 / 52 / 45 / 39 / 33 / 22 / 18 / 20; 64 of 2,048 x 5,632 220 / 125 / 116 / 98 / 83 / 50 / 42 / 24; 144 of 11,264 x
// 2,048 97 / 82 / 94 / 77 / 96 / 89 / 98 / 107.
static int gf_tile_form(int M, int N, int K) {
    static const int form[8] = {6, 7, 8, 11, 12, 5, 9, 10}, bm[8] = {128, 64, 64, 64, 64, 32, 32, 32}, bn[8] = {128, 128, 128, 64, 64, 64, 32, 16};
    static const int first[8] = {300, 170, 0, 190, 45, 10, 25, 30}, many[8] = {1190, 670, 770, 375, 505, 330, 238, 135};
    static const int other[8] = {2, 3, 3, 4, 4, 5, 9, 10};       // the forms for K that is no whole blocks
    const bool whole = K % GF_BK == 0;
    int best = 0;
    long long cost = -1;
    for (int i = 0; i < 8; ++i) {
        if (!whole && (i == 2 || i == 4)) continue;
        const long long tiles = (long long)((M + bm[i] - 1) / bm[i]) * ((N + bn[i] - 1) / bn[i]);
        const long long c = first[i] + (tiles + GF_CUS - 1) / GF_CUS * many[i];
        if (cost < 0 || c < cost) { best = i; cost = c; }
    }
    return whole ? form[best] : other[best];
}

// what the kernels need of the operands: rows of whole 16-byte groups at 16-byte addresses; offsets inside a tile's rows are
// 32 bits wide
extern "C" int bn_gemm_f32_supports(int N, int K, int ldw, const void* w) {
    return N > 0 && K > 0 && K % 4 == 0 && ldw % 4 == 0 && ldw >= K && ldw <= (1 << 22) && ((uintptr_t)w & 15) == 0;
}

// form 0: by the sizes; 1: streaming up to 16 rows, beyond (up to 64) chunks of 32 x 16; 2 .. 5: tiles of 128 x 128, 64 x 128, 64 x 64, 32 x 64;
// 9, 10: chunks of 32 x 32, 32 x 16; for whole blocks of K 6, 7, 8: 128 x 128, 64 x 128, the same with K in two, 11, 12: 64 x 64, with K in two
// (every form gives the same bits).
//
// norm_w (form 0): the rows of x are normed on their way in, bn_gemm_f32_norm_supports says of which sizes.  add (form 0, up to 16
// rows, no glu): y += the product.
extern "C" int bn_gemm_f32(const void* x, const void* w, void* y, int M, int N, int K, int ldx, int ldw, int ldy, int glu, int act,
                           int form, const float* norm_w, float eps, int add, hipStream_t s) {
    if (M <= 0 || !bn_gemm_f32_supports(N, K, ldw, w) || ldx % 4 || ldx < K || ldx > (1 << 22) || ((uintptr_t)x & 15)) return BN_ERR_ARG;
    if (ldy < (glu ? N / 2 : N) || (glu && (glu == 2 ? N % 2 || M > 16 || form > 1 : N % 16)) || act < 0 || act >= BN_ACT_KINDS) return BN_ERR_ARG;
    if ((long long)((M + 31) / 32) * ((N + 15) / 16) > 0x7fffffffLL) return BN_ERR_ARG;
    if (((norm_w || add) && form) || (norm_w && !gf_norm_ok(M, K, norm_w)) || (add && (glu || M > 16))) return BN_ERR_ARG;
    GfArgs a = {(const float*)x, (const float*)w, (float*)y, M, N, K, ldx, ldw, ldy, 16, glu == 2 ? 2 : glu ? 1 : 0, act, add ? 1 : 0, norm_w, eps};
    if (norm_w) {
        a.cols = glu ? 16 : gf_stream_cols(N);
        return gf_norm_pick(M, K, [&](auto nr, auto nv) { return gf_launch_stream<decltype(nr)::value, decltype(nv)::value>(a, s); });
    }
    if (form == 0) form = M <= 16 ? 1 : gf_tile_form(M, N, K);
    switch (form) {
        case 1:
            if (M > 64) return BN_ERR_ARG;
            if (M > 16) return gf_launch_chunks<2, 1, 8>(a, s);
            a.cols = glu ? 16 : gf_stream_cols(N);
            return gf_launch_stream<>(a, s);
        case 2: return gf_launch_tile<128, 2, 1, false>(a, s);
        case 3: return gf_launch_tile<64, 2, 1, false>(a, s);
        case 4: return gf_launch_tile<64, 1, 1, false>(a, s);
        case 5: return gf_launch_tile<32, 1, 4, false>(a, s);
        case 6: return gf_launch_tile<128, 2, 1, true>(a, s);
        case 7: return gf_launch_tile<64, 2, 1, true>(a, s);
        case 8: return gf_launch_tile<64, 2, 2, true>(a, s);
        case 9: return gf_launch_chunks<2, 2, 4>(a, s);
        case 10: return gf_launch_chunks<2, 1, 8>(a, s);
        case 11: return gf_launch_tile<64, 1, 1, true>(a, s);
        case 12: return gf_launch_tile<64, 1, 2, true>(a, s);
    }
    return BN_ERR_ARG;
}

// Columns a workgroup of the streaming kernels owns: the rows per tile that a streamed copy of W is best made with.
extern "C" int bn_gemm_f32_stream_cols(int N) { return N < 1 ? 0 : gf_stream_cols(N); }

#define GF_STREAMED_SMEM (150 * 1024)
static int gf_streamed_xr(int M) { return M <= 2 ? 1 : M <= 4 ? 2 : M <= 8 ? 4 : 8; }
// the staged activations, the parts of their squares, a sum a chunk, row and column
static size_t gf_streamed_smem(int M, int K, bool norm, bool parts) {
    const size_t rows = 2 * gf_streamed_xr(M);
    return (norm ? rows * (gf_row_bytes(K, parts) + 16) : GF_WAVES * rows * gf_row_bytes(GF_CHUNK, parts)) + (size_t)(K / GF_CHUNK) * rows * 64;
}
// Whether staged rows lie there in parts, split once instead of once a wave: where they fit, and unless a CU then holds one workgroup
// instead of two (eight normed rows).
static bool gf_streamed_parts(int M, int K, bool norm) { return (!norm || M <= 4) && gf_streamed_smem(M, K, norm, true) <= GF_STREAMED_SMEM; }

// 1 if the products of up to 16 rows take a norm of such rows with them
extern "C" int bn_gemm_f32_norm_supports(int M, int K) { return gf_norm_ok(M, K, nullptr); }

// 1 if the kernel over a streamed copy takes the product: up to 16 rows, whole chunks whose sums fit into shared memory
// (every K up to 10,752 at 9 to 16 rows, 29,952 at 5 to 8, 68,352 at 3 and 4, 145,152 at 1 and 2), rows of activations that are whole 16-byte groups.
extern "C" int bn_gemm_f32_streamed_supports(int M, int N, int K, int ldx, int tile_rows, const void* x) {
    return M >= 1 && M <= 16 && N >= 1 && K >= GF_CHUNK && K % GF_CHUNK == 0 && gf_streamed_smem(M, K, false, false) <= GF_STREAMED_SMEM && ldx >= K &&
           ldx % 4 == 0 && ldx <= 1 << 22 && tile_rows >= 1 && tile_rows <= BN_STREAM_TILE_ROWS && ((uintptr_t)x & 15) == 0;
}

// As bn_gemm_f32 over W's streamed copy (common.h) with that many rows a tile (16 with glu).
extern "C" int bn_gemm_f32_streamed(const void* x, const void* tiles, void* y, int M, int N, int K, int ldx, int tile_rows, int ldy,
                                    int glu, int act, const float* norm_w, float eps, int add, hipStream_t s) {
    if (!bn_gemm_f32_streamed_supports(M, N, K, ldx, tile_rows, x) || !tiles || !y || ((uintptr_t)tiles & 15)) return BN_ERR_ARG;
    if (ldy < (glu ? N / 2 : N) || (glu && (N % 16 || tile_rows != 16)) || act < 0 || act >= BN_ACT_KINDS) return BN_ERR_ARG;
    if ((norm_w && (!gf_norm_ok(M, K, norm_w) || K < GF_WAVES * GF_CHUNK)) || (add && (glu || (long long)M * ldy > 1 << 29))) return BN_ERR_ARG;
    GfArgs a = {(const float*)x, (const float*)tiles, (float*)y, M, N, K, ldx, 0, ldy, tile_rows, glu ? 1 : 0, act, add ? 1 : 0, norm_w, eps};
    const bool parts = gf_streamed_parts(M, K, norm_w != nullptr);
    auto go = [&](auto kernel) {
        const size_t smem = gf_streamed_smem(M, K, norm_w != nullptr, parts);
        if (smem > 64 * 1024) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            if (e != hipSuccess) return (int)e;
        }
        hipLaunchKernelGGL(kernel, dim3((N + tile_rows - 1) / tile_rows), dim3(64 * GF_WAVES), smem, s, a, K / BN_STREAM_TILE_COLS_F32);
        return bn_launch_status();
    };
    if (norm_w)
        return gf_norm_pick(M, K, [&](auto nr, auto nv) {
            return parts ? go(gemm_f32_streamed_kernel<decltype(nr)::value, true, decltype(nv)::value>) : go(gemm_f32_streamed_kernel<decltype(nr)::value, false, decltype(nv)::value>);
        });
    switch (gf_streamed_xr(M)) {
        case 1: return parts ? go(gemm_f32_streamed_kernel<1, true>) : go(gemm_f32_streamed_kernel<1, false>);
        case 2: return parts ? go(gemm_f32_streamed_kernel<2, true>) : go(gemm_f32_streamed_kernel<2, false>);
        case 4: return parts ? go(gemm_f32_streamed_kernel<4, true>) : go(gemm_f32_streamed_kernel<4, false>);
        default: return parts ? go(gemm_f32_streamed_kernel<8, true>) : go(gemm_f32_streamed_kernel<8, false>);
    }
}
