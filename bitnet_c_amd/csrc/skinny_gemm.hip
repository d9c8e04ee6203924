// Decode-phase matrix product for bf16: Y[M, N] = X[M, K] . W[N, K]^T with M <= 64 rows
// of activations, on the matrix cores (v_mfma_f32_16x16x32_bf16).  The weights are
// streamed once from HBM with 16-byte loads, four lanes covering 64 contiguous bytes of
// one weight row per load and a wave 512 bytes of 16 rows per 256-element K chunk; K is split over the waves of a workgroup and
// the partial sums are added through shared memory in wave order, so the result does
// not depend on timing.  It plays the part of the reference's matvec kernels
// (src/gpu_cuda.cu:3976-4010, one warp per output row) and of its stacked gate/up
// matvec followed by the activation (src/gpu_cuda.cu:4176, :8971), written for 64-wide
// waves and MFMA instead.
//
// DUAL: W holds two row blocks (gate rows n, up rows up_off + n); the epilogue writes
// act(gate) * up, act one of the kinds of bn_gate_act (silu(g) = g / (1 + exp(-g)) for this
// architecture, src/transformer/cpu_backend.c:385-391).
// Neither: Y is the product, or with act BN_ACT_RELU2 the square of its positive part.
// GLU8: the same product with gate and up rows interleaved in blocks of 8 (rows 16t..16t+7 are
// gate rows 8t..8t+7, rows 16t+8..16t+15 the up rows of the same columns): every 16-row tile holds
// both halves of 8 result columns, so the plain kernel does it with half the loads in flight.
//
// The activations: all workgroups read the same X, and a load in the operand layout (one row per
// lane, 64 bytes of it per load) costs a full load instruction however few rows there are.  With
// up to 16 rows (XS) a wave therefore fetches its K chunk of X with dense loads (32 lanes x 16 bytes
// a row), parks it in a region of shared memory of its own (no workgroup barrier) and reads the
// operand fragments from there; the vector memory pipe is left to the weights.
//
// TILED: W is the streamed copy of the matrix (common.h: tiles of up to 16 rows x 32 columns in the lanes' order); a
// load of a wave is then one tile, up to 1 KB of consecutive bytes, ldw the number of tiles along K, and a workgroup
// owns the columns of one row of tiles.  Measured against
// the row-major matrix at 8 rows of an 8B shape: QKV 14.3 -> 13.2 us, output projection 10.7 -> 9.3, gate/up 49.5 ->
// 43.9, down 28.0 -> 24.0.
//
// Needs K % 8 == 0 and 16-byte aligned rows; other shapes go to the tiled kernel.
#include "common.h"
#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

#define SK_CHUNK 256          // K elements per wave iteration

__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

#define SK_XROW 528           // bytes between rows of a wave's staged X chunk (512 + 16: conflict-free 16-byte reads)

#define SK_STREAM_WAVES 8     // waves of a workgroup over a streamed copy of whole chunks

#define SK_ACT_UNARY 16       // act: this plus one of BN_UNARY_*: an activation of one argument on every result

// The result of a product without a gate under its activation: none, a square of the positive part (the gate kind
// BN_ACT_RELU2), or any activation of one argument (UNARY: kept out of the other instantiations, whose registers it would cost).
template <bool UNARY> __device__ __forceinline__ float sk_result(float v, int act) {
    if (UNARY) return act >= SK_ACT_UNARY ? bn_unary_act(v, act - SK_ACT_UNARY) : v;
    const float p = fmaxf(v, 0.f);
    return act == BN_ACT_RELU2 ? p * p : v;
}

// bx: the workgroup's number among those of its product
template <int MT, bool DUAL, typename TO, bool GLU8, bool XS, bool TILED, bool UNARY>
__device__ __forceinline__ void skinny_gemm_body(const bf16* __restrict__ X, const bf16* __restrict__ W, TO* __restrict__ Y, int M, int N,
                                                 int K, int ldx, int ldw, int ldy, int up_off, int act, int bx) {
    constexpr int NA = DUAL ? 2 * MT : MT;            // accumulator tiles per wave
    extern __shared__ __align__(16) float red[];      // [n_waves][NA][64][4]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);      // a scalar
    const int n_waves = blockDim.x >> 6;
    const int i = lane & 15, g = lane >> 4;
    const int CW = TILED ? up_off : 16;               // columns a workgroup owns; TILED: up_off carries the copy's rows per tile
    const int n0 = bx * CW;
    const int n = min(n0 + i, N - 1);                 // clamp: rows past N are computed and dropped
    const int TS = CW * BN_STREAM_TILE_COLS;          // elements of a tile
    // tiled: the row of tiles is the same for all lanes (a base in scalar registers), the lane adds its 16 bytes' place
    const bf16* wrow = TILED ? W + (size_t)bx * ldw * TS : W + (size_t)n * ldw;
    const unsigned lane_at = (g * CW + i) * 8;
    const bf16* urow = DUAL ? W + (size_t)(up_off + n) * ldw : nullptr;

    f32x4 acc[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a) acc[a] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // XS: this wave's staging region, after the partial sums
    unsigned char* xs = reinterpret_cast<unsigned char*>(red + (size_t)n_waves * NA * 256) + (size_t)wave * M * SK_XROW;

    for (int kc = wave * SK_CHUNK; kc < K; kc += n_waves * SK_CHUNK) {
        const int kb = kc + g * 8;                    // lane group g: 8 elements of every 32 (64 contiguous bytes per row and load)
        uint4 wv[8], uv[8];
        uint4 xd[8];
        if (XS) {                                     // issued before the weights: loads return in order
            const int xk = kc + (lane & 31) * 8;
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const int row = 2 * r + (lane >> 5);
                if (2 * r < M)
                    xd[r] = (row < M && xk < K) ? *reinterpret_cast<const uint4*>(X + (size_t)row * ldx + xk)
                                                : make_uint4(0, 0, 0, 0);
            }
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int k = kb + j * 32;
            if (TILED)          // tile kc / 32 + j of this block of rows; its columns past K hold zeros
                wv[j] = (i < CW && kc + j * 32 < K) ? bn_load_once(wrow + (size_t)((kc >> 5) + j) * TS + lane_at)
                                                    : make_uint4(0, 0, 0, 0);
            else
                wv[j] = (k < K) ? *reinterpret_cast<const uint4*>(wrow + k) : make_uint4(0, 0, 0, 0);
            if (DUAL) uv[j] = (k < K) ? *reinterpret_cast<const uint4*>(urow + k) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int m = mt * 16 + i;
            const bf16* xrow = X + (size_t)m * ldx;
            uint4 xv[8];
            if (XS) {
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    const int row = 2 * r + (lane >> 5);
                    if (2 * r < M && row < M)
                        *reinterpret_cast<uint4*>(xs + row * SK_XROW + (lane & 31) * 16) = xd[r];
                }
                __builtin_amdgcn_wave_barrier();      // one wave: its shared-memory operations run in order
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    xv[j] = (m < M) ? *reinterpret_cast<const uint4*>(xs + m * SK_XROW + j * 64 + g * 16)
                                    : make_uint4(0, 0, 0, 0);
                __builtin_amdgcn_wave_barrier();
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int k = kb + j * 32;
                    xv[j] = (m < M && k < K) ? *reinterpret_cast<const uint4*>(xrow + k) : make_uint4(0, 0, 0, 0);
                }
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(xv[j]), as_bf16x8(wv[j]), acc[mt], 0, 0, 0);
                if (DUAL)
                    acc[MT + mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(xv[j]), as_bf16x8(uv[j]),
                                                                          acc[MT + mt], 0, 0, 0);
            }
        }
    }
    // partial sums of every wave -> shared memory
#pragma unroll
    for (int a = 0; a < NA; ++a)
        *reinterpret_cast<f32x4*>(red + (((size_t)wave * NA + a) * 64 + lane) * 4) = acc[a];
    __syncthreads();
    // thread (l, r): C row 4*(l/16)+r of each tile, column l%16; sums over waves in wave order
    for (int idx = threadIdx.x; idx < MT * 256; idx += blockDim.x) {
        const int mt = idx >> 8, rem = idx & 255;
        const int l = rem & 63, r = rem >> 6;
        float v = 0.f, u = 0.f;
        for (int w = 0; w < n_waves; ++w) {
            v += red[(((size_t)w * NA + mt) * 64 + l) * 4 + r];
            if (DUAL) u += red[(((size_t)w * NA + MT + mt) * 64 + l) * 4 + r];
        }
        const int m = mt * 16 + 4 * (l >> 4) + r;
        const int nn = (l & 15) < CW ? n0 + (l & 15) : N;          // a column past the workgroup's own is nobody's
        if (GLU8) {
            // columns 0..7 of the tile are gates, 8..15 the ups of the same result columns
            const float up = bn_lane_xor<8>(v);
            if ((l & 8) == 0 && m < M && nn < N)
                Y[(size_t)m * ldy + (n0 >> 1) + (l & 7)] = from_f32<TO>(bn_gate_act(v, act) * up);
        } else if (m < M && nn < N) {
            const float y = DUAL ? bn_gate_act(v, act) * u : sk_result<UNARY>(v, act);
            Y[(size_t)m * ldy + nn] = from_f32<TO>(y);
        }
    }
}

template <int MT, bool DUAL, typename TO, bool GLU8 = false, bool XS = false, bool TILED = false, bool UNARY = false>
__global__ __launch_bounds__((DUAL && MT >= 3) ? 512 : 1024) void skinny_gemm_kernel(const bf16* __restrict__ X, const bf16* __restrict__ W,
                                                           TO* __restrict__ Y, int M, int N, int K, int ldx,
                                                           int ldw, int ldy, int up_off, int act) {
    skinny_gemm_body<MT, DUAL, TO, GLU8, XS, TILED, UNARY>(X, W, Y, M, N, K, ldx, ldw, ldy, up_off, act, blockIdx.x);
}

// Several products of up to 16 rows over streamed copies that do not depend on each other, as one launch: a launch that waits
// for the one before it costs some 4.5 us whatever it does, and five products of 2,048 x 2,048 take 4.5 to 6 each.  The
// workgroups of product j are the numbers from first[j] on.
#define SK_GROUP 6
struct SkinnyGroup {
    const bf16* x[SK_GROUP];
    const bf16* w[SK_GROUP];
    bf16* y[SK_GROUP];
    int n[SK_GROUP], ldx[SK_GROUP], rows[SK_GROUP], act[SK_GROUP], first[SK_GROUP];      // rows: of a tile of the copy
    int count;
};

__global__ __launch_bounds__(512) void skinny_group_kernel(SkinnyGroup p, int M, int K, int k_tiles) {
    int j = 0;
    while (j + 1 < p.count && (int)blockIdx.x >= p.first[j + 1]) ++j;
    skinny_gemm_body<1, false, bf16, false, true, true, true>(p.x[j], p.w[j], p.y[j], M, p.n[j], K, p.ldx[j], k_tiles, p.n[j], p.rows[j],
                                                              p.act[j], (int)blockIdx.x - p.first[j]);
}

// ---------------------------------------------------------------------------------------
// The same product for up to 16 rows with the neighbouring norm folded in, so that a decode layer
// needs no kernel for its two norms:
//   RES: the product is a part's output.  The epilogue adds it to the float32 residual stream in
//        place (its 16 columns), writes a bf16 copy of the new stream multiplied by the next norm's
//        weights, and the sum of the squares of its 16 columns of every row into a slot of its own.
//   PRE: the activations are such a copy.  1/sqrt(mean(x^2) + eps) (src/transformer/rmsnorm_scalar.c:4-13)
//        multiplies a whole row of the result, so it is applied in the epilogue: every wave fetches the
//        slots of two rows before its K loop and adds them up behind it (lane-strided sums, a tree over
//        the lanes: a fixed order); the staged activations need no work at all.  (Asked for later, before
//        the wave's last chunk, the same loads cost three times as much.)
// GLU8 as above.  bf16 result (RES: no result of its own).
#define SK_SLOT_LOADS 8       // slots per row and lane: at most 512 column tiles (a stream of 8,192 columns)

struct SkinnyFused {
    const float* slots_in;    // [M, n_slots] sums of squares, PRE
    int n_slots;
    float inv_width, eps;     // 1 / columns of the stream, the norm's eps, PRE
    float* resid;             // [M, ld_resid] float32 stream, RES
    bf16* resid_bf16;         // [M, ld_rb] its bf16 copy times next_weight, RES
    const float* next_weight; // [N] weights of the norm that reads the copy, RES
    float* slots_out;         // [M, gridDim.x], RES
    int ld_resid, ld_rb;
};

template <bool GLU8, bool PRE, bool RES, int SL, bool TILED>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 4)))
void skinny_gemm_fused_kernel(const bf16* __restrict__ X, const bf16* __restrict__ W, bf16* __restrict__ Y, int M, int N,
                              int K, int ldx, int ldw, int ldy, int tile_cols, int act, SkinnyFused f) {
    constexpr int NW = 8;                              // always eight waves: wave w owns rows w and w + 8 of the norm
    extern __shared__ __align__(16) float red[];       // [NW][64][4], then 16 row scales, then the staging
    // the wave's number as a scalar: what depends on it alone (its chunks of K, a tile's address) stays in scalar registers
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 15, g = lane >> 4;
    // A workgroup owns tile_cols <= 16 columns (the rest of its MFMA tile is not loaded and not stored): the
    // host picks the width that spreads the column tiles evenly over the CUs.
    const int n0 = blockIdx.x * tile_cols;
    const bool col = i < tile_cols;
    const int n = min(n0 + i, N - 1);
    // tiled: tile_cols is the copy's rows per tile and the workgroup's rows are one row of tiles
    const int TS = tile_cols * BN_STREAM_TILE_COLS;
    // (the row of tiles is the same for all lanes, a base in scalar registers; the lane adds its 16 bytes' place)
    const bf16* wrow = TILED ? W + (size_t)blockIdx.x * ldw * TS : W + (size_t)n * ldw;
    const unsigned lane_at = (g * tile_cols + i) * 8;
    float* scale_s = red + NW * 256;
    unsigned char* xs = reinterpret_cast<unsigned char*>(red + NW * 256 + 16) + (size_t)wave * M * SK_XROW;

    f32x4 acc = (f32x4){0.f, 0.f, 0.f, 0.f};
    auto fetch = [&](int kc, uint4* wv, uint4* xd) {
        const int kb = kc + g * 8;
        const int xk = kc + (lane & 31) * 8;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const int row = 2 * r + (lane >> 5);
            if (2 * r < M)
                xd[r] = (row < M && xk < K) ? *reinterpret_cast<const uint4*>(X + (size_t)row * ldx + xk) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int k = kb + j * 32;
            if (TILED)
                wv[j] = (col && kc + j * 32 < K) ? bn_load_once(wrow + (size_t)((kc >> 5) + j) * TS + lane_at)
                                                 : make_uint4(0, 0, 0, 0);
            else
                wv[j] = (col && k < K) ? *reinterpret_cast<const uint4*>(wrow + k) : make_uint4(0, 0, 0, 0);
        }
    };
    auto multiply = [&](const uint4* wv, const uint4* xd) {
        uint4 xv[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const int row = 2 * r + (lane >> 5);
            if (2 * r < M && row < M) *reinterpret_cast<uint4*>(xs + row * SK_XROW + (lane & 31) * 16) = xd[r];
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < 8; ++j)
            xv[j] = (i < M) ? *reinterpret_cast<const uint4*>(xs + i * SK_XROW + j * 64 + g * 16) : make_uint4(0, 0, 0, 0);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < 8; ++j)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(xv[j]), as_bf16x8(wv[j]), acc, 0, 0, 0);
    };
    auto step = [&](int kc) {
        uint4 wv[8], xd[8];
        fetch(kc, wv, xd);
        multiply(wv, xd);
    };
    // the slots of the norm are asked for first: they arrive while the wave waits for its first weights
    float sv[2][SL];                                   // PRE: this lane's slots of rows wave and wave + 8
    if (PRE) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int m = wave + NW * h;
#pragma unroll
            for (int j = 0; j < SL; ++j) {
                const int t = lane + 64 * j;
                sv[h][j] = (m < M && t < f.n_slots) ? f.slots_in[(size_t)m * f.n_slots + t] : 0.f;
            }
        }
    }
    for (int kc = wave * SK_CHUNK; kc < K; kc += NW * SK_CHUNK) step(kc);
    if (PRE) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float v = 0.f;
#pragma unroll
            for (int j = 0; j < SL; ++j) v += sv[h][j];
            v = wave_sum(v);
            if (lane == 0 && wave + NW * h < 16) scale_s[wave + NW * h] = 1.0f / sqrtf(v * f.inv_width + f.eps);
        }
    }
    *reinterpret_cast<f32x4*>(red + ((size_t)wave * 64 + lane) * 4) = acc;
    __syncthreads();
    // waves 0..3: thread (l, r = wave): C row 4*(l/16)+r, column l%16; sums over waves in wave order
    if (wave < 4) {
        const int l = lane, r = wave;
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) v += red[((size_t)w * 64 + l) * 4 + r];
        const int m = 4 * (l >> 4) + r;
        const int nn = n0 + (l & 15);
        const bool mine = (l & 15) < tile_cols && nn < N;                 // a column this workgroup owns
        if (PRE) v *= scale_s[m];
        if (GLU8) {
            const float up = bn_lane_xor<8>(v);
            if ((l & 8) == 0 && m < M && nn < N)                          // GLU8: tile_cols is 16
                Y[(size_t)m * ldy + (n0 >> 1) + (l & 7)] = __float2bfloat16(bn_gate_act(v, act) * up);
        } else if (RES) {
            float xn = 0.f;
            if (m < M && mine) {
                xn = f.resid[(size_t)m * f.ld_resid + nn] + v;
                f.resid[(size_t)m * f.ld_resid + nn] = xn;
                f.resid_bf16[(size_t)m * f.ld_rb + nn] = __float2bfloat16(xn * f.next_weight[nn]);
            }
            float sq = xn * xn;                                   // the tile's columns of row m: lanes 16 (l / 16) + 0..15
            sq += bn_lane_xor<1>(sq);
            sq += bn_lane_xor<2>(sq);
            sq += bn_lane_xor<4>(sq);
            sq += bn_lane_xor<8>(sq);
            if ((l & 15) == 0 && m < M) f.slots_out[(size_t)m * gridDim.x + blockIdx.x] = sq;
        } else if (m < M && mine) {
            Y[(size_t)m * ldy + nn] = __float2bfloat16(v);
        }
    }
}

// ---------------------------------------------------------------------------------------
// The products of up to 16 rows over a streamed copy whose K is whole chunks (K % 256 == 0), which is every decode product of
// ordinary widths.  Bound by the bytes of W, and at widths of 2,048 by what happens once a launch: the same sums in the same
// order as the kernels above (wave w takes chunks w, w + 8, ..; the waves' sums are added in wave order: the same bits), in
// straight-line code.  Nothing is predicated (a lane without a row or a column reads its neighbour's and drops what it forms;
// a load under a branch makes the compiler wait for every load in flight), the number of activation loads is a template
// argument, a wave has two chunks of weights in flight (16 KB; one where K <= 2,048 gives it no second, so that three
// workgroups fit on a CU), and what the epilogue needs of memory is asked for before the weights.
//   us with cold weights in a graph of such launches, 1 / 8 rows, the kernels above -> these: 2,048 columns of the stream
//   QKV 5.7 / 6.2 -> 4.1 / 4.5, output 5.1 / 5.3 -> 3.7 / 4.0, gate/up (5,632) 12.3 / 13.1 -> 9.9 / 11.0, down 8.1 / 8.9 ->
//   6.5 / 7.3; 8B QKV 12.2 / 13.4 -> 10.3 / 11.5, output 9.4 / 10.0 -> 7.7 / 8.3, gate/up 43.9 / 44.9 -> 38.5 / 40.4, down
//   24.0 / 24.7 -> 21.1 / 22.0 (a plain read of the same bytes with a dependent launch: 4.0, 3.1, 8.3, 5.2; 8.9, 6.5, 35.8,
//   18.4).  At 9 to 16 rows the activations' registers leave room for one workgroup of two chunks a wave on a CU (8B QKV 15.5
//   -> 14.1, gate/up 48.0 -> 43.7).
#define SK_STAGED_ROW(k) ((k) * 2 + 16)      // bytes between staged rows of k numbers

template <int XR, bool ONE, bool STAGED = false>
struct SkStream {
    // XR: activation loads a lane and chunk, for up to 2 XR rows; ONE: a wave has one chunk at most; STAGED (with ONE): the rows
    // lie in shared memory, SK_STAGED_ROW(K) bytes apart, when run's `between` returns
    __amdgpu_buffer_rsrc_t wb, xb;
    unsigned tile, w_at;
    unsigned x_at[XR];
    unsigned char *park_at, *read_at;
    bf16x8 x[XR];
    f32x4 acc;

    // (the scheduling barriers keep the loads of a chunk where they are written: moved up over the products before them they
    // need registers that are not there)
    __device__ __forceinline__ void load_x(int c) {
        if (STAGED) return;
#pragma unroll
        for (int r = 0; r < XR; ++r) x[r] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(xb, x_at[r], c * (SK_CHUNK * 2), 0));
    }
    __device__ __forceinline__ void load_w(bf16x8 (&w)[8], int c) {
        unsigned at = (unsigned)c * 8 * tile;
#pragma unroll
        for (int j = 0; j < 8; ++j, at += tile)
            w[j] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(wb, w_at, at, BN_BUFFER_NT));
        __builtin_amdgcn_sched_barrier(0);
    }
    // the chunk's activations into the wave's own region of shared memory (a wave's operations on it run in order)
    __device__ __forceinline__ void park() {
        if (STAGED) return;
#pragma unroll
        for (int r = 0; r < XR; ++r) *reinterpret_cast<bf16x8*>(park_at + 2 * r * SK_XROW) = x[r];
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_sched_barrier(0);
    }
    __device__ __forceinline__ void multiply(const bf16x8 (&w)[8]) {
#pragma unroll
        for (int h = 0; h < 8; h += 4) {
            bf16x8 v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = *reinterpret_cast<const bf16x8*>(read_at + (h + j) * 64);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[j], w[h + j], acc, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_wave_barrier();
    }
    // this wave's share of X . W^T for row of tiles bx; `between` runs once the first weights have been asked for
    template <typename F>
    __device__ __forceinline__ void run(const bf16* X, const bf16* W, int M, int n_chunks, int ldx, int k_tiles, int rows, int bx,
                                        unsigned char* xs, int lane, int wave, F between) {
        const int i = lane & 15, g = lane >> 4;
        tile = rows * (BN_STREAM_TILE_COLS * 2);
        wb = bn_buffer(reinterpret_cast<const char*>(W) + (size_t)bx * k_tiles * tile, k_tiles * tile);
        xb = bn_buffer(X, ((M - 1) * ldx + n_chunks * SK_CHUNK) * 2);
        w_at = (g * rows + min(i, rows - 1)) * 16;
#pragma unroll
        for (int r = 0; r < XR; ++r) x_at[r] = (min(2 * r + (lane >> 5), M - 1) * ldx + (lane & 31) * 8) * 2;
        xs += (size_t)wave * 2 * XR * SK_XROW;
        park_at = xs + (lane >> 5) * SK_XROW + (lane & 31) * 16;
        read_at = xs + min(i, M - 1) * SK_XROW + g * 16;
        if (STAGED) read_at = xs - (size_t)wave * 2 * XR * SK_XROW + min(i, M - 1) * SK_STAGED_ROW(n_chunks * SK_CHUNK) + wave * (SK_CHUNK * 2) + g * 16;
        acc = (f32x4){0.f, 0.f, 0.f, 0.f};
        const int n = (n_chunks - wave + SK_STREAM_WAVES - 1) / SK_STREAM_WAVES;       // chunks of this wave
        if (ONE || n <= 1) {
            if (n == 1) {
                bf16x8 w[8];
                load_x(wave);
                load_w(w, wave);
                between();
                park();
                multiply(w);
            } else {
                between();
            }
            return;
        }
        constexpr int D = SK_STREAM_WAVES;
        int c = wave, left = n;
        bf16x8 a[8], b[8];
        load_x(c);
        load_w(a, c);
        load_w(b, c + D);
        between();
#pragma unroll 1
        for (; left > 3; left -= 2, c += 2 * D) {
            park();
            load_x(c + D);
            multiply(a);
            load_w(a, c + 2 * D);
            park();
            load_x(c + 2 * D);
            multiply(b);
            load_w(b, c + 3 * D);
        }
        park();
        load_x(c + D);
        multiply(a);
        if (left == 2) {
            park();
            multiply(b);
            return;
        }
        load_w(a, c + 2 * D);
        park();
        load_x(c + 2 * D);
        multiply(b);
        park();
        multiply(a);
    }
};

// the waves' sums -> shared memory; then waves 0..3: thread (l, r = wave) holds row 4 (l / 16) + r, column l % 16 of the product
__device__ __forceinline__ float sk_stream_total(float* red, const f32x4& acc, int lane, int wave) {
    *reinterpret_cast<f32x4*>(red + (wave * 64 + lane) * 4) = acc;
    bn_lds_barrier();
    float v = 0.f;
    if (wave < 4) {
#pragma unroll
        for (int w = 0; w < SK_STREAM_WAVES; ++w) v += red[(w * 64 + lane) * 4 + wave];
    }
    return v;
}

#define SK_STREAM_RED (SK_STREAM_WAVES * 256 + 16)       // floats: the waves' sums, the norm's row factors

template <int XR, bool ONE, typename TO, bool UNARY>
__device__ __forceinline__ void sk_stream_plain(const bf16* X, const bf16* W, TO* Y, int M, int N, int n_chunks, int ldx, int k_tiles,
                                                int ldy, int rows, int act, int bx) {
    extern __shared__ __align__(16) float red[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    SkStream<XR, ONE> s;
    s.run(X, W, M, n_chunks, ldx, k_tiles, rows, bx, reinterpret_cast<unsigned char*>(red + SK_STREAM_RED), lane, wave, [] {});
    const float v = sk_stream_total(red, s.acc, lane, wave);
    if (wave >= 4) return;
    const int m = 4 * (lane >> 4) + wave, n = bx * rows + (lane & 15);
    if (m < M && (lane & 15) < rows && n < N) Y[(size_t)m * ldy + n] = from_f32<TO>(sk_result<UNARY>(v, act));
}

template <int XR, bool ONE, typename TO, bool UNARY>
__global__ __launch_bounds__(64 * SK_STREAM_WAVES, (ONE && XR <= 4) ? 6 : XR == 8 ? 2 : 4)
void skinny_stream_kernel(const bf16* __restrict__ X, const bf16* __restrict__ W, TO* __restrict__ Y, int M, int N, int n_chunks, int ldx,
                          int k_tiles, int ldy, int rows, int act) {
    sk_stream_plain<XR, ONE, TO, UNARY>(X, W, Y, M, N, n_chunks, ldx, k_tiles, ldy, rows, act, blockIdx.x);
}

template <int XR, bool ONE>
__global__ __launch_bounds__(64 * SK_STREAM_WAVES, (ONE && XR <= 4) ? 6 : XR == 8 ? 2 : 4)
void skinny_stream_group_kernel(SkinnyGroup p, int M, int n_chunks, int k_tiles) {
    int j = 0;
    while (j + 1 < p.count && (int)blockIdx.x >= p.first[j + 1]) ++j;
    sk_stream_plain<XR, ONE, bf16, true>(p.x[j], p.w[j], p.y[j], M, p.n[j], n_chunks, p.ldx[j], k_tiles, p.n[j], p.rows[j], p.act[j],
                                         (int)blockIdx.x - p.first[j]);
}

// the forms of skinny_gemm_fused_kernel: a gated unit behind a norm, a product behind a norm, a product into the stream
#define SK_FUSED_GLU 0
#define SK_FUSED_PRE 1
#define SK_FUSED_RES 2
#define SK_FUSED_ADD 3               // into the stream as a bf16 output would be added: rounded first, and nothing left for a norm
template <int XR, bool ONE, int FORM, int SL>
__global__ __launch_bounds__(64 * SK_STREAM_WAVES, (ONE && XR <= 4) ? 6 : XR == 8 ? 2 : 4)
void skinny_stream_fused_kernel(const bf16* __restrict__ X, const bf16* __restrict__ W, bf16* __restrict__ Y, int M, int N, int n_chunks,
                                int ldx, int k_tiles, int ldy, int rows, int act, SkinnyFused f) {
    constexpr bool PRE = FORM == SK_FUSED_GLU || FORM == SK_FUSED_PRE;
    constexpr int H = XR <= 4 ? 1 : 2;                // rows of the norm that a wave adds up: wave, and wave + 8
    extern __shared__ __align__(16) float red[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float* scale_s = red + SK_STREAM_WAVES * 256;
    const int n0 = blockIdx.x * rows, at = lane & 15;
    const int m = 4 * (lane >> 4) + (wave & 3), n = n0 + at;
    float sv[H][SL];
    if (PRE) {
#pragma unroll
        for (int h = 0; h < H; ++h) {
            const unsigned row = (unsigned)min(wave + SK_STREAM_WAVES * h, M - 1) * f.n_slots;
#pragma unroll
            for (int j = 0; j < SL; ++j) sv[h][j] = f.slots_in[row + min(lane + 64 * j, f.n_slots - 1)];
        }
    }
    float old = 0.f, next_w = 0.f;
    if (!PRE) {
        const int nc = min(n, N - 1);
        old = f.resid[(size_t)min(m, M - 1) * f.ld_resid + nc];
        if (FORM == SK_FUSED_RES) next_w = f.next_weight[nc];
    }
    SkStream<XR, ONE> s;
    s.run(X, W, M, n_chunks, ldx, k_tiles, rows, blockIdx.x, reinterpret_cast<unsigned char*>(red + SK_STREAM_RED), lane, wave, [&] {
        if (PRE) {
#pragma unroll
            for (int h = 0; h < H; ++h) {
                float v = 0.f;
#pragma unroll
                for (int j = 0; j < SL; ++j) v += lane + 64 * j < f.n_slots ? sv[h][j] : 0.f;
                v = 1.0f / sqrtf(wave_sum(v) * f.inv_width + f.eps);
                if (lane == 0) scale_s[wave + SK_STREAM_WAVES * h] = v;
            }
        }
    });
    float v = sk_stream_total(red, s.acc, lane, wave);
    if (wave >= 4) return;
    const bool mine = m < M && at < rows && n < N;
    if (PRE) v *= scale_s[m];                         // rows past M: whatever lies there, not stored
    if (FORM == SK_FUSED_GLU) {
        const float up = bn_lane_xor<8>(v);           // columns 0..7 of the tile are gates, 8..15 the ups of the same results
        if (mine && (lane & 8) == 0) Y[(size_t)m * ldy + (n0 >> 1) + (lane & 7)] = __float2bfloat16(bn_gate_act(v, act) * up);
    } else if (FORM == SK_FUSED_PRE) {
        if (mine) Y[(size_t)m * ldy + n] = __float2bfloat16(v);
    } else if (FORM == SK_FUSED_ADD) {
        if (mine) f.resid[(size_t)m * f.ld_resid + n] = old + to_f32(__float2bfloat16(v));
    } else {
        float xn = 0.f;
        if (mine) {
            xn = old + v;
            f.resid[(size_t)m * f.ld_resid + n] = xn;
            f.resid_bf16[(size_t)m * f.ld_rb + n] = __float2bfloat16(xn * next_w);
        }
        float sq = xn * xn;                           // the tile's columns of row m: lanes 16 (l / 16) + 0..15
        sq += bn_lane_xor<1>(sq);
        sq += bn_lane_xor<2>(sq);
        sq += bn_lane_xor<4>(sq);
        sq += bn_lane_xor<8>(sq);
        if (at == 0 && m < M) f.slots_out[(size_t)m * gridDim.x + blockIdx.x] = sq;
    }
}

// A product whose rows the residual stream still has to give: every workgroup forms them itself while its weights are on their
// way, instead of a kernel of one workgroup a row that the product would wait for (3.4 us a launch; the rows come from the L2).
// The operations and their order are those of the kernels in whose place this runs (elementwise.hip), so are the bits; here
// the halves of the workgroup take every other row, eight numbers a thread.
#define SK_ROWS_NORM 0               // x w / rms(x): add_rmsnorm_row_kernel
#define SK_ROWS_SUM 1                // x + w d / rms(d), the new stream: add_normed_rmsnorm_wide_kernel
#define SK_ROWS_SHIFT 2              // h + (h' - h) mu for h the normed row and h' the one before it: that, then token_shift_wide_kernel
#define SK_ROWS_GATE 3               // x w act(gate) / rms(x): row_norm_gate_wide_kernel (lightning.hip)
struct SkinnyRows {
    const float* x;                  // [M, K] the stream (GATE: any rows)
    const bf16* delta;               // [M, K] SUM; GATE: the gates, rows ld_gate apart
    int ld_gate, gate_act;           // GATE: BN_UNARY_*
    const float* w;                  // [K]
    float* x_new;                    // [M, K] SUM: where the first workgroup writes the new stream (the others may still read x)
    int K;
    float eps;
    // SHIFT, row m one token of a sequence of its own: the mixes' weights (of this product), the sequences' state rows, whose
    // first K numbers are h', the tokens' positions (0: h' is zeros; below: a row that is nobody's), and [M, K] for h
    const float* mu;
    const float* state;
    long long state_stride;
    const int* positions;
    const int* slot_ids;
    bf16* h;
};

template <int NR, int MODE> struct SkRowStage {
    float4 x[NR][2], w[2], before[NR][2], mu[2];
    uint4 d[NR];
    int t, half, pos[NR];
    __device__ __forceinline__ int at(int k) const { return MODE == SK_ROWS_SUM || MODE == SK_ROWS_GATE ? t * 8 + k * 4 : (k * 256 + t) * 4; }
    __device__ __forceinline__ void load(const SkinnyRows& p, int M) {
        t = threadIdx.x & 255;
        half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const size_t row = (size_t)min(half + 2 * i, M - 1) * p.K;
            if (MODE == SK_ROWS_SUM) d[i] = *reinterpret_cast<const uint4*>(p.delta + row + min(t * 8, p.K - 8));
            if (MODE == SK_ROWS_GATE)
                d[i] = *reinterpret_cast<const uint4*>(p.delta + (size_t)min(half + 2 * i, M - 1) * p.ld_gate + min(t * 8, p.K - 8));
#pragma unroll
            for (int k = 0; k < 2; ++k) x[i][k] = *reinterpret_cast<const float4*>(p.x + row + min(at(k), p.K - 4));
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) w[k] = *reinterpret_cast<const float4*>(p.w + min(at(k), p.K - 4));
        if (MODE == SK_ROWS_SHIFT) {
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                const int row = min(half + 2 * i, M - 1);
                pos[i] = p.positions[row];
                const float* from = p.state + (size_t)p.slot_ids[row] * p.state_stride;
#pragma unroll
                for (int k = 0; k < 2; ++k) before[i][k] = *reinterpret_cast<const float4*>(from + min(at(k), p.K - 4));
            }
#pragma unroll
            for (int k = 0; k < 2; ++k) mu[k] = *reinterpret_cast<const float4*>(p.mu + min(at(k), p.K - 4));
        }
    }
    // parts: [2 NR][4] floats; rows: the staged rows.  Two barriers; behind the second the rows are there.
    __device__ __forceinline__ void stage(const SkinnyRows& p, int M, float* parts, unsigned char* rows) {
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            float ss = 0.f;
            if (MODE == SK_ROWS_GATE) {
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    ss = __builtin_fmaf(x[i][k].y, x[i][k].y, __builtin_fmaf(x[i][k].x, x[i][k].x, ss));
                    ss = __builtin_fmaf(x[i][k].w, x[i][k].w, __builtin_fmaf(x[i][k].z, x[i][k].z, ss));
                }
                if (at(0) >= p.K) ss = 0.f;
            } else if (MODE != SK_ROWS_SUM) {
#pragma unroll
                for (int k = 0; k < 2; ++k) ss = at(k) < p.K ? bn_add_squares(ss, x[i][k], k) : ss;
            } else {
                const uint32_t two[4] = {d[i].x, d[i].y, d[i].z, d[i].w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float lo = bf16lo_to_f32(two[e]), hi = bf16hi_to_f32(two[e]);
                    ss = __builtin_fmaf(hi, hi, __builtin_fmaf(lo, lo, ss));
                }
                if (at(0) >= p.K) ss = 0.f;
            }
            ss = wave_sum(ss);
            if ((threadIdx.x & 63) == 0) parts[(half + 2 * i) * 4 + ((threadIdx.x >> 6) & 3)] = ss;
        }
        bn_lds_barrier();
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int row = half + 2 * i;
            float ss = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j) ss += parts[row * 4 + j];
            const float f = 1.0f / sqrtf(ss / (float)p.K + p.eps);
            const uint32_t two[4] = {d[i].x, d[i].y, d[i].z, d[i].w};
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                if (at(k) >= p.K) continue;
                float4 v;
                if (MODE != SK_ROWS_SUM) {
                    v = make_float4(x[i][k].x * f * w[k].x, x[i][k].y * f * w[k].y, x[i][k].z * f * w[k].z, x[i][k].w * f * w[k].w);
                    if (MODE == SK_ROWS_GATE) {
                        v.x *= bn_unary_act(bf16lo_to_f32(two[2 * k]), p.gate_act);
                        v.y *= bn_unary_act(bf16hi_to_f32(two[2 * k]), p.gate_act);
                        v.z *= bn_unary_act(bf16lo_to_f32(two[2 * k + 1]), p.gate_act);
                        v.w *= bn_unary_act(bf16hi_to_f32(two[2 * k + 1]), p.gate_act);
                    }
                } else {
                    v.x = __builtin_fmaf(bf16lo_to_f32(two[2 * k]) * f, w[k].x, x[i][k].x);
                    v.y = __builtin_fmaf(bf16hi_to_f32(two[2 * k]) * f, w[k].y, x[i][k].y);
                    v.z = __builtin_fmaf(bf16lo_to_f32(two[2 * k + 1]) * f, w[k].z, x[i][k].z);
                    v.w = __builtin_fmaf(bf16hi_to_f32(two[2 * k + 1]) * f, w[k].w, x[i][k].w);
                    if (blockIdx.x == 0 && row < M) *reinterpret_cast<float4*>(p.x_new + (size_t)row * p.K + at(k)) = v;
                }
                bf16 o[4] = {from_f32<bf16>(v.x), from_f32<bf16>(v.y), from_f32<bf16>(v.z), from_f32<bf16>(v.w)};
                if (MODE == SK_ROWS_SHIFT) {
                    if (blockIdx.x == 0 && row < M) *reinterpret_cast<uint2*>(p.h + (size_t)row * p.K + at(k)) = *reinterpret_cast<const uint2*>(o);
                    const float b4[4] = {before[i][k].x, before[i][k].y, before[i][k].z, before[i][k].w}, m4[4] = {mu[k].x, mu[k].y, mu[k].z, mu[k].w};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float c = to_f32(o[e]), gap = (pos[i] > 0 ? b4[e] : 0.f) - c;
                        o[e] = from_f32<bf16>(pos[i] >= 0 ? fmaf(gap, m4[e], c) : 0.f);
                    }
                }
                *reinterpret_cast<uint2*>(rows + row * SK_STAGED_ROW(p.K) + at(k) * 2) = *reinterpret_cast<const uint2*>(o);
            }
        }
        bn_lds_barrier();
    }
};

template <int XR, int MODE, bool UNARY>
__global__ __launch_bounds__(64 * SK_STREAM_WAVES, 4)
void skinny_stream_rows_kernel(SkinnyRows p, const bf16* __restrict__ W, bf16* __restrict__ Y, int M, int N, int n_chunks, int k_tiles,
                               int rows, int act) {
    extern __shared__ __align__(16) float red[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    unsigned char* staged = reinterpret_cast<unsigned char*>(red + SK_STREAM_RED);
    SkRowStage<XR, MODE> st;
    st.load(p, M);
    SkStream<XR, true, true> s;
    s.run(nullptr, W, M, n_chunks, 0, k_tiles, rows, blockIdx.x, staged, lane, wave, [&] { st.stage(p, M, red, staged); });
    const float v = sk_stream_total(red, s.acc, lane, wave);
    if (wave >= 4) return;
    const int m = 4 * (lane >> 4) + wave, n = blockIdx.x * rows + (lane & 15);
    if (m < M && (lane & 15) < rows && n < N) Y[(size_t)m * N + n] = __float2bfloat16(sk_result<UNARY>(v, act));
}

// Several such products of the same rows in one launch; SHIFT: product j's mixes have the weights mu + j K.
template <int XR, int MODE>
__global__ __launch_bounds__(64 * SK_STREAM_WAVES, 4)
void skinny_stream_rows_group_kernel(SkinnyGroup g, SkinnyRows p, int M, int n_chunks, int k_tiles) {
    extern __shared__ __align__(16) float red[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    unsigned char* staged = reinterpret_cast<unsigned char*>(red + SK_STREAM_RED);
    int j = 0;
    while (j + 1 < g.count && (int)blockIdx.x >= g.first[j + 1]) ++j;
    if (MODE == SK_ROWS_SHIFT) p.mu += (size_t)j * p.K;
    const int rows = g.rows[j], bx = (int)blockIdx.x - g.first[j];
    SkRowStage<XR, MODE> st;
    st.load(p, M);
    SkStream<XR, true, true> s;
    s.run(nullptr, g.w[j], M, n_chunks, 0, k_tiles, rows, bx, staged, lane, wave, [&] { st.stage(p, M, red, staged); });
    const float v = sk_stream_total(red, s.acc, lane, wave);
    if (wave >= 4) return;
    const int m = 4 * (lane >> 4) + wave, n = bx * rows + (lane & 15);
    if (m < M && (lane & 15) < rows && n < g.n[j]) g.y[j][(size_t)m * g.n[j] + n] = __float2bfloat16(sk_result<true>(v, g.act[j]));
}

// whole chunks only; offsets inside a row of tiles and inside the activations are 32 bits wide
static bool sk_stream_ok(int M, int K, int ldx) {
    return M <= 16 && K % SK_CHUNK == 0 && K <= 1 << 24 && (long long)M * ldx <= 1 << 29;
}

// go(XR, ONE) as integral constants for M rows and K columns
template <typename F> static int sk_stream_pick(int M, int K, F go) {
    using std::integral_constant;
    const bool one = K <= SK_CHUNK * SK_STREAM_WAVES;
#define SK_PICK(XR_) return one ? go(integral_constant<int, XR_>(), integral_constant<bool, true>()) \
                                : go(integral_constant<int, XR_>(), integral_constant<bool, false>())
    if (M <= 2) SK_PICK(1);
    if (M <= 4) SK_PICK(2);
    if (M <= 8) SK_PICK(4);
    SK_PICK(8);
#undef SK_PICK
}

template <typename KERNEL, typename... ARGS>
static int sk_stream_launch(KERNEL kernel, int xr, unsigned groups, hipStream_t s, ARGS... args) {
    const size_t smem = SK_STREAM_RED * sizeof(float) + (size_t)SK_STREAM_WAVES * 2 * xr * SK_XROW;
    if (smem > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL(kernel, dim3(groups), dim3(64 * SK_STREAM_WAVES), smem, s, args...);
    return bn_launch_status();
}

extern "C" int bn_skinny_gemm_supports(int M, int N, int K, int ldx, int ldw);

// 1 if products form M rows of K numbers themselves (mode: SK_ROWS_*): whole chunks, one a wave at the most, and from 512 numbers on,
// gated ones from 1,024 (narrower rows are normed by other kernels, in other orders).  Up to the rows where that is the faster way: us
// at 1 / 2 / 4 / 8 rows of 2,048 numbers, two kernels -> one: normed rows x 8,192 9.7 / 10.1 / 10.1 / 10.6 -> 7.6 / 7.5 / 8.0 / 9.5; the new
// stream's x 8,192 9.3 / 9.4 / 9.9 / 10.2 -> 7.4 / 7.5 / 8.6 / 10.9; gated x 2,048 7.0 / 7.1 / 7.1 / 7.9 -> 5.0 / 5.0 / 7.4 / 11.4; five mixes x 4 x
// 2,048 and 64, three kernels -> one, 13.6 / 13.9 / 14.2 / 15.5 -> 11.1 / 11.0 / 13.6 / 19.6.
// Narrower rows gain more (a workgroup forms less and the launches cost the same): of 512 numbers, normed x 2,048 at 1 / 4 / 8 rows 4.6 /
// 4.8 / 4.9 -> 2.9 / 3.8 / 4.5, the new stream's at 1 / 4 4.5 / 4.8 -> 3.0 / 3.8, five mixes 7.6 / 8.3 -> 4.2 / 5.3; of 1,024, gated at 1 / 2
// 5.8 / 5.9 -> 4.1 / 4.2.
extern "C" int bn_skinny_rows_supports(int M, int K, int mode) {
    const int most = mode == SK_ROWS_NORM ? 8 : mode == SK_ROWS_SUM || mode == SK_ROWS_SHIFT ? 4 : mode == SK_ROWS_GATE ? 2 : 0;
    return M >= 1 && M <= most && K % SK_CHUNK == 0 && K >= (mode == SK_ROWS_GATE ? 4 : 2) * SK_CHUNK && K <= SK_CHUNK * SK_STREAM_WAVES;
}

// Y[M, N] (bf16, contiguous) = act(rows . W^T) over W's streamed copy (k_tiles tiles along K, tile_rows rows a tile) for rows
// that are formed on the way: delta null, the rows of x normed with weights w; else x + w delta / rms(delta), which x_new gets too
// (other memory than x).  All contiguous and 16-byte aligned.  act: 0, BN_ACT_RELU2, or SK_ACT_UNARY plus one of BN_UNARY_*.
extern "C" int bn_skinny_rows(const float* x, const void* delta, const float* w, float eps, float* x_new, const void* tiles, void* Y, int M,
                              int N, int K, int k_tiles, int tile_rows, int act, hipStream_t s) {
    if (!bn_skinny_rows_supports(M, K, delta ? SK_ROWS_SUM : SK_ROWS_NORM) || N < 1 || k_tiles != K / BN_STREAM_TILE_COLS || tile_rows < 1 || tile_rows > BN_STREAM_TILE_ROWS ||
        !x || !w || !tiles || !Y || !delta != !x_new || x == x_new) return BN_ERR_ARG;
    if (((uintptr_t)x | (uintptr_t)delta | (uintptr_t)w | (uintptr_t)x_new | (uintptr_t)tiles) & 15) return BN_ERR_ARG;
    if (act != 0 && act != BN_ACT_RELU2 && (act < SK_ACT_UNARY || act >= SK_ACT_UNARY + BN_UNARY_KINDS)) return BN_ERR_ARG;
    SkinnyRows p = {};
    p.x = x; p.delta = (const bf16*)delta; p.w = w; p.x_new = x_new; p.K = K; p.eps = eps;
    return sk_stream_pick(M, K, [&](auto xr, auto) {
        constexpr int XR = decltype(xr)::value < 4 ? decltype(xr)::value : 4, FEW = XR < 2 ? XR : 2;
        auto go = [&](auto kernel) {
            const size_t smem = SK_STREAM_RED * sizeof(float) + (size_t)2 * XR * SK_STAGED_ROW(K);
            hipLaunchKernelGGL(kernel, dim3((N + tile_rows - 1) / tile_rows), dim3(64 * SK_STREAM_WAVES), smem, s, p, (const bf16*)tiles,
                               (bf16*)Y, M, N, K / SK_CHUNK, k_tiles, tile_rows, act);
            return bn_launch_status();
        };
        if (delta) return act >= SK_ACT_UNARY ? go(skinny_stream_rows_kernel<FEW, SK_ROWS_SUM, true>) : go(skinny_stream_rows_kernel<FEW, SK_ROWS_SUM, false>);
        return act >= SK_ACT_UNARY ? go(skinny_stream_rows_kernel<XR, SK_ROWS_NORM, true>) : go(skinny_stream_rows_kernel<XR, SK_ROWS_NORM, false>);
    });
}

// Y[M, N] (bf16, contiguous) = rows . W^T, the rows x w act(gate) / rms(x): x [M, K] float32 contiguous, gate bf16 with row stride
// ld_gate, act one of BN_UNARY_*; W's streamed copy as above.
extern "C" int bn_skinny_gated_rows(const float* x, const void* gate, int ld_gate, int act, const float* w, float eps, const void* tiles, void* Y,
                                    int M, int N, int K, int k_tiles, int tile_rows, hipStream_t s) {
    if (!bn_skinny_rows_supports(M, K, SK_ROWS_GATE) || N < 1 || k_tiles != K / BN_STREAM_TILE_COLS || tile_rows < 1 || tile_rows > BN_STREAM_TILE_ROWS ||
        !x || !gate || !w || !tiles || !Y || ld_gate < K || ld_gate % 8 || act < 0 || act >= BN_UNARY_KINDS) return BN_ERR_ARG;
    if (((uintptr_t)x | (uintptr_t)gate | (uintptr_t)w | (uintptr_t)tiles) & 15) return BN_ERR_ARG;
    SkinnyRows p = {};
    p.x = x; p.delta = (const bf16*)gate; p.ld_gate = ld_gate; p.gate_act = act; p.w = w; p.K = K; p.eps = eps;
    const size_t smem = SK_STREAM_RED * sizeof(float) + (size_t)2 * SK_STAGED_ROW(K);
    hipLaunchKernelGGL((skinny_stream_rows_kernel<1, SK_ROWS_GATE, false>), dim3((N + tile_rows - 1) / tile_rows), dim3(64 * SK_STREAM_WAVES),
                       smem, s, p, (const bf16*)tiles, (bf16*)Y, M, N, K / SK_CHUNK, k_tiles, tile_rows, 0);
    return bn_launch_status();
}

// resid [M, N] (float32, row stride ld_resid) += X . W^T over W's streamed copy, every result rounded to bf16 first; whole chunks.
extern "C" int bn_skinny_add(const void* X, const void* tiles, int M, int N, int K, int ldx, int k_tiles, int tile_rows, float* resid,
                             int ld_resid, hipStream_t s) {
    if (!bn_skinny_gemm_supports(M, N, K, ldx, 8) || ldx < K || !sk_stream_ok(M, K, ldx) || k_tiles != K / BN_STREAM_TILE_COLS ||
        tile_rows < 1 || tile_rows > BN_STREAM_TILE_ROWS || !resid || ld_resid < N || (((uintptr_t)X | (uintptr_t)tiles) & 15))
        return BN_ERR_ARG;
    SkinnyFused f = {};
    f.resid = resid; f.ld_resid = ld_resid;
    return sk_stream_pick(M, K, [&](auto xr, auto one) {
        constexpr int XR = decltype(xr)::value;
        return sk_stream_launch(skinny_stream_fused_kernel<XR, decltype(one)::value, SK_FUSED_ADD, 1>, XR, (unsigned)((N + tile_rows - 1) / tile_rows),
                                s, (const bf16*)X, (const bf16*)tiles, (bf16*)nullptr, M, N, K / SK_CHUNK, ldx, k_tiles, 0, tile_rows, 0, f);
    });
}

static bool sk_tiled_ok(int K, int ldw) { return ldw == (K + BN_STREAM_TILE_COLS - 1) / BN_STREAM_TILE_COLS; }

static int sk_compute_units() {
    static int cus = 0;
    if (!cus) {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0) cus = v;
        else cus = 256;
    }
    return cus;
}

// Columns per workgroup of the fused kernel for a product of N columns (not GLU8): 16, or fewer when that spreads
// the column tiles so much more evenly over the CUs that the busiest CU has at least 15 % fewer columns
// (6,144 columns: 384 tiles of 16 are one and a half rounds over 256 CUs, 512 tiles of 12 are two even ones).
// A CU pulls its bytes no faster when others idle, so the busiest CU's columns are the kernel's time.
static int sk_fused_tile_cols(int N) {
    const int cus = sk_compute_units();
    auto busiest = [&](int tc) { const int tiles = (N + tc - 1) / tc; return (long long)((tiles + cus - 1) / cus) * tc; };
    int pick = 16;
    long long best = busiest(16);
    for (int tc = 14; tc >= 8; tc -= 2) {
        const int tiles = (N + tc - 1) / tc;
        if (tiles > 64 * SK_SLOT_LOADS) continue;                 // a consumer adds up at most that many slots
        const long long c = busiest(tc);
        if (c * 100 <= best * 85 && c < busiest(pick)) pick = tc;
    }
    return pick;
}

// Columns per workgroup that the fused kernel picks for a product of N columns over a row-major W: the rows per tile
// that a streamed copy of W is best made with.
extern "C" int bn_skinny_gemm_fused_tile_cols(int N) { return N < 1 ? 0 : sk_fused_tile_cols(N); }

// Column tiles (= slots per row that a RES call writes) of the fused kernel for N columns; over a streamed copy of W
// (tile_rows > 0) they are its rows of tiles.
extern "C" int bn_skinny_gemm_fused_tiles(int N, int tile_rows) {
    if (N < 1 || tile_rows < 0 || tile_rows > BN_STREAM_TILE_ROWS) return 0;
    const int tc = tile_rows ? tile_rows : sk_fused_tile_cols(N);
    return (N + tc - 1) / tc;
}

// X, W, Y as bn_skinny_gemm with a bf16 result and M <= 16; glu8 as dual == 2 there, act the gate's activation.
// slots_in != null (PRE): X is a stream's bf16 copy as a RES call leaves it, slots_in [M, n_slots] its rows'
// sums of squares in parts, stream_width its number of columns; the result's rows are scaled by
// 1/sqrt(sum / stream_width + eps).
// resid != null (RES): the product is added to resid [M, N] in place; resid_bf16 [M, N] becomes the new stream
// times next_weight [N], slots_out [M, bn_skinny_gemm_fused_tiles(N)] the sums of squares of its column tiles
// (glu8 == 0, no Y).
// tile_rows > 0: W is the streamed copy (common.h) of the matrix (of its 2N interleaved rows with glu8, then with 16 rows
// a tile) with that many rows a tile and ldw its tiles along K; a RES call then writes a slot per row of tiles.
extern "C" int bn_skinny_gemm_fused(const void* X, const void* W, void* Y, int M, int N, int K, int ldx, int ldw, int ldy,
                                    int glu8, int act, const float* slots_in, int n_slots, int stream_width, float eps,
                                    float* resid, int ld_resid, void* resid_bf16, int ld_rb, const float* next_weight,
                                    float* slots_out, int tile_rows, hipStream_t s) {
    const bool tiled = tile_rows != 0;
    if (!bn_skinny_gemm_supports(M, N, K, ldx, tiled ? 8 : ldw) || M > 16 || act < 0 || act >= BN_ACT_KINDS) return BN_ERR_ARG;
    if (tiled && (!sk_tiled_ok(K, ldw) || tile_rows < 1 || tile_rows > BN_STREAM_TILE_ROWS || (glu8 && tile_rows != 16)))
        return BN_ERR_ARG;
    if (((uintptr_t)X | (uintptr_t)W) & 15) return BN_ERR_ARG;
    const bool pre = slots_in != nullptr, res = resid != nullptr;
    if (!pre && !res) return BN_ERR_ARG;
    if (pre && (n_slots < 1 || n_slots > 64 * SK_SLOT_LOADS || stream_width < 1)) return BN_ERR_ARG;
    if (res && (glu8 || !resid_bf16 || !next_weight || !slots_out || ld_resid < N || ld_rb < N)) return BN_ERR_ARG;
    if (!res && (!Y || ldy < N)) return BN_ERR_ARG;
    if (glu8) {
        if (N % 8) return BN_ERR_ARG;
        N *= 2;
    }
    SkinnyFused f;
    f.slots_in = slots_in; f.n_slots = n_slots; f.inv_width = pre ? 1.0f / (float)stream_width : 0.f; f.eps = eps;
    f.resid = resid; f.resid_bf16 = (bf16*)resid_bf16; f.next_weight = next_weight; f.slots_out = slots_out;
    f.ld_resid = ld_resid; f.ld_rb = ld_rb;
    const bool few = n_slots <= 256;                  // four slot loads per row and lane are enough
    if (glu8 && !pre) return BN_ERR_ARG;
    if (tiled && sk_stream_ok(M, K, ldx) && !(pre && res))
        return sk_stream_pick(M, K, [&](auto xr, auto one) {
            constexpr int XR = decltype(xr)::value;
            constexpr bool ONE = decltype(one)::value;
            auto go = [&](auto kernel) {
                return sk_stream_launch(kernel, XR, (unsigned)((N + tile_rows - 1) / tile_rows), s, (const bf16*)X, (const bf16*)W, (bf16*)Y,
                                        M, N, K / SK_CHUNK, ldx, ldw, ldy, tile_rows, act, f);
            };
            if (glu8) return few ? go(skinny_stream_fused_kernel<XR, ONE, SK_FUSED_GLU, 4>) : go(skinny_stream_fused_kernel<XR, ONE, SK_FUSED_GLU, 8>);
            if (pre) return few ? go(skinny_stream_fused_kernel<XR, ONE, SK_FUSED_PRE, 4>) : go(skinny_stream_fused_kernel<XR, ONE, SK_FUSED_PRE, 8>);
            return go(skinny_stream_fused_kernel<XR, ONE, SK_FUSED_RES, 1>);
        });
    const size_t smem = (size_t)(8 * 256 + 16) * sizeof(float) + (size_t)8 * M * SK_XROW;
    const int tile_cols = tiled ? tile_rows : (glu8 ? 16 : sk_fused_tile_cols(N));
    const dim3 grid((N + tile_cols - 1) / tile_cols), block(8 * 64);
    auto go = [&](auto kernel) {
        if (smem > 64 * 1024) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            if (e != hipSuccess) return (int)e;
        }
        hipLaunchKernelGGL(kernel, grid, block, smem, s, (const bf16*)X, (const bf16*)W, (bf16*)Y, M, N, K, ldx, ldw, ldy,
                           tile_cols, act, f);
        return bn_launch_status();
    };
#define SK_FUSED(T)                                                                                                      \
    do {                                                                                                                 \
        if (glu8) return few ? go(skinny_gemm_fused_kernel<true, true, false, 4, T>)                                     \
                             : go(skinny_gemm_fused_kernel<true, true, false, 8, T>);                                    \
        if (pre && res) return few ? go(skinny_gemm_fused_kernel<false, true, true, 4, T>)                               \
                                   : go(skinny_gemm_fused_kernel<false, true, true, 8, T>);                              \
        if (pre) return few ? go(skinny_gemm_fused_kernel<false, true, false, 4, T>)                                     \
                            : go(skinny_gemm_fused_kernel<false, true, false, 8, T>);                                    \
        return go(skinny_gemm_fused_kernel<false, false, true, 4, T>);                                                   \
    } while (0)
    if (tiled) SK_FUSED(true);
    SK_FUSED(false);
#undef SK_FUSED
}

template <int MT, bool DUAL, typename TO, bool GLU8 = false, bool TILED = false, bool UNARY = false>
static int launch(const void* X, const void* W, void* Y, int M, int N, int K, int ldx, int ldw, int ldy,
                  int up_off, int act, int n_waves, hipStream_t s) {
    constexpr int NA = DUAL ? 2 * MT : MT;
    constexpr bool XS = MT == 1 && !DUAL;          // the two-block form has no registers to spare for it
    const size_t smem = (size_t)n_waves * NA * 64 * 4 * sizeof(float) + (XS ? (size_t)n_waves * M * SK_XROW : 0);
    auto kernel = skinny_gemm_kernel<MT, DUAL, TO, GLU8, XS, TILED, UNARY>;
    if (smem > 64 * 1024) {                           // beyond the default limit of dynamic shared memory
        static bool raised = false;                   // per instantiation
        if (!raised) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            if (e != hipSuccess) return (int)e;
            raised = true;
        }
    }
    const int cols = TILED ? up_off : 16;             // columns a workgroup owns
    hipLaunchKernelGGL(kernel, dim3((N + cols - 1) / cols), dim3(n_waves * 64), smem, s,
                       (const bf16*)X, (const bf16*)W, (TO*)Y, M, N, K, ldx, ldw, ldy, up_off, act);
    return bn_launch_status();
}

template <typename TO>
static int launch_glu8(int MT, const void* X, const void* W, void* Y, int M, int N, int K, int ldx, int ldw,
                       int ldy, int act, int n_waves, hipStream_t s) {
    switch (MT) {
        case 1: return launch<1, false, TO, true>(X, W, Y, M, N, K, ldx, ldw, ldy, 0, act, n_waves, s);
        case 2: return launch<2, false, TO, true>(X, W, Y, M, N, K, ldx, ldw, ldy, 0, act, n_waves, s);
        case 3: return launch<3, false, TO, true>(X, W, Y, M, N, K, ldx, ldw, ldy, 0, act, n_waves, s);
        case 4: return launch<4, false, TO, true>(X, W, Y, M, N, K, ldx, ldw, ldy, 0, act, n_waves, s);
    }
    return BN_ERR_ARG;
}

template <bool DUAL, typename TO>
static int launch_mt(int MT, const void* X, const void* W, void* Y, int M, int N, int K, int ldx, int ldw,
                     int ldy, int up_off, int act, int n_waves, hipStream_t s) {
    switch (MT) {
        case 1: return launch<1, DUAL, TO>(X, W, Y, M, N, K, ldx, ldw, ldy, up_off, act, n_waves, s);
        case 2: return launch<2, DUAL, TO>(X, W, Y, M, N, K, ldx, ldw, ldy, up_off, act, n_waves, s);
        case 3: return launch<3, DUAL, TO>(X, W, Y, M, N, K, ldx, ldw, ldy, up_off, act, n_waves, s);
        case 4: return launch<4, DUAL, TO>(X, W, Y, M, N, K, ldx, ldw, ldy, up_off, act, n_waves, s);
    }
    return BN_ERR_ARG;
}

// 1 if the kernel takes the shape, 0 if the caller must use the tiled kernel.
extern "C" int bn_skinny_gemm_supports(int M, int N, int K, int ldx, int ldw) {
    return (M >= 1 && M <= 64 && N >= 1 && K >= 8 && K % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0) ? 1 : 0;
}

// out_dtype: type of Y (bf16 or float32).  dual == 1: N is the width of the result and W has
// the gate rows at [0, N) and the up rows at [up_off, up_off + N).  dual == 2: W has 2N rows, gate
// and up interleaved in blocks of 8 (N a multiple of 8); the result has N columns.  act: the gate's activation
// (BN_ACT_*) when dual != 0; with dual == 0 BN_ACT_RELU2 squares the positive part of every result (a feed-forward without
// a gate), SK_ACT_UNARY + one of BN_UNARY_* puts every result under that activation (bf16 results of up to 16 rows) and any
// other value leaves the product as it is.
// tile_rows > 0: W is the streamed copy (common.h) with that many rows a tile and ldw its tiles along K; up to 16 rows,
// dual == 0.
extern "C" int bn_skinny_gemm(int out_dtype, const void* X, const void* W, void* Y, int M, int N, int K,
                              int ldx, int ldw, int ldy, int dual, int up_off, int act, int tile_rows, hipStream_t s) {
    const bool tiled = tile_rows != 0, unary = act >= SK_ACT_UNARY;
    if (!bn_skinny_gemm_supports(M, N, K, ldx, tiled ? 8 : ldw) || ldy < N || act < 0) return BN_ERR_ARG;
    if (unary ? act >= SK_ACT_UNARY + BN_UNARY_KINDS || dual || M > 16 || out_dtype != BN_DT_BF16 : act >= BN_ACT_KINDS) return BN_ERR_ARG;
    if (((uintptr_t)X | (uintptr_t)W) & 15) return BN_ERR_ARG;
    if (tiled) {
        if (dual || M > 16 || !sk_tiled_ok(K, ldw) || tile_rows < 1 || tile_rows > BN_STREAM_TILE_ROWS) return BN_ERR_ARG;
        if (sk_stream_ok(M, K, ldx) && (out_dtype == BN_DT_BF16 || out_dtype == BN_DT_F32))
            return sk_stream_pick(M, K, [&](auto xr, auto one) {
                constexpr int XR = decltype(xr)::value;
                constexpr bool ONE = decltype(one)::value;
                const unsigned groups = (unsigned)((N + tile_rows - 1) / tile_rows);
                auto go = [&](auto kernel, auto* y) {
                    return sk_stream_launch(kernel, XR, groups, s, (const bf16*)X, (const bf16*)W, y, M, N, K / SK_CHUNK, ldx, ldw, ldy,
                                            tile_rows, act);
                };
                if (unary) return go(skinny_stream_kernel<XR, ONE, bf16, true>, (bf16*)Y);
                if (out_dtype == BN_DT_BF16) return go(skinny_stream_kernel<XR, ONE, bf16, false>, (bf16*)Y);
                return go(skinny_stream_kernel<XR, ONE, float, false>, (float*)Y);
            });
        int n_waves = 8;                           // as the row-major form with staged activations
        const int k_chunks = (K + SK_CHUNK - 1) / SK_CHUNK;
        while (n_waves > 1 && n_waves / 2 >= k_chunks) n_waves >>= 1;
        // the kernel's up_off carries the rows per tile; its grid is one workgroup per row of tiles
        if (unary)
            return launch<1, false, bf16, false, true, true>(X, W, Y, M, N, K, ldx, ldw, ldy, tile_rows, act, n_waves, s);
        if (out_dtype == BN_DT_BF16)
            return launch<1, false, bf16, false, true>(X, W, Y, M, N, K, ldx, ldw, ldy, tile_rows, act, n_waves, s);
        if (out_dtype == BN_DT_F32)
            return launch<1, false, float, false, true>(X, W, Y, M, N, K, ldx, ldw, ldy, tile_rows, act, n_waves, s);
        return BN_ERR_DTYPE;
    }
    if (dual == 2) {
        if (N % 8) return BN_ERR_ARG;
        N *= 2;                                   // rows of W; the kernel halves the column index itself
    }
    const int MT = (M + 15) / 16;
    const int NA = dual == 1 ? 2 * MT : MT;
    // waves per workgroup: enough loads in flight when there are few column tiles, bounded by
    // the K chunks there are and by 48 KB of shared memory for the partial sums
    const int tiles = (N + 15) / 16;
    int n_waves = tiles >= 2048 ? 4 : (tiles >= 1024 ? 8 : 16);
    if (MT == 1 && dual != 1) n_waves = 8;        // staged activations: measured best at every size (several workgroups per CU)
    const int k_chunks = (K + SK_CHUNK - 1) / SK_CHUNK;
    while (n_waves > 1 && n_waves / 2 >= k_chunks) n_waves >>= 1;
    while (n_waves > 1 && n_waves * NA > 48) n_waves >>= 1;
    if (dual == 1 && MT >= 3 && n_waves > 8) n_waves = 8;      // that variant is built for 512 threads
    if (unary) return launch<1, false, bf16, false, false, true>(X, W, Y, M, N, K, ldx, ldw, ldy, 0, act, n_waves, s);
    if (dual == 2) {
        if (out_dtype == BN_DT_BF16) return launch_glu8<bf16>(MT, X, W, Y, M, N, K, ldx, ldw, ldy, act, n_waves, s);
        if (out_dtype == BN_DT_F32) return launch_glu8<float>(MT, X, W, Y, M, N, K, ldx, ldw, ldy, act, n_waves, s);
        return BN_ERR_DTYPE;
    }
    if (out_dtype == BN_DT_BF16)
        return dual ? launch_mt<true, bf16>(MT, X, W, Y, M, N, K, ldx, ldw, ldy, up_off, act, n_waves, s)
                    : launch_mt<false, bf16>(MT, X, W, Y, M, N, K, ldx, ldw, ldy, up_off, act, n_waves, s);
    if (out_dtype == BN_DT_F32)
        return dual ? launch_mt<true, float>(MT, X, W, Y, M, N, K, ldx, ldw, ldy, up_off, act, n_waves, s)
                    : launch_mt<false, float>(MT, X, W, Y, M, N, K, ldx, ldw, ldy, up_off, act, n_waves, s);
    return BN_ERR_DTYPE;
}

// Up to SK_GROUP products of the same M <= 16 rows and K over streamed copies, bf16 results, in one launch.  Arrays of `count`:
// X, W, Y addresses, N columns, ldx, the copies' rows per tile, and the activation of the results (a BN_UNARY_* or -1).  The
// results are contiguous [M, N].
extern "C" int bn_skinny_group(int count, const void* const* X, const void* const* W, void* const* Y, const int* N, const int* ldx,
                               const int* tile_rows, const int* unary, int M, int K, int k_tiles, hipStream_t s) {
    if (count < 1 || count > SK_GROUP || M < 1 || M > 16 || !sk_tiled_ok(K, k_tiles)) return BN_ERR_ARG;
    SkinnyGroup p;
    p.count = count;
    int groups = 0;
    bool whole = true;
    for (int j = 0; j < count; ++j) {
        if (!bn_skinny_gemm_supports(M, N[j], K, ldx[j], 8) || ldx[j] < K || tile_rows[j] < 1 || tile_rows[j] > BN_STREAM_TILE_ROWS ||
            unary[j] < -1 || unary[j] >= BN_UNARY_KINDS || (((uintptr_t)X[j] | (uintptr_t)W[j]) & 15) || !Y[j])
            return BN_ERR_ARG;
        p.x[j] = (const bf16*)X[j]; p.w[j] = (const bf16*)W[j]; p.y[j] = (bf16*)Y[j];
        p.n[j] = N[j]; p.ldx[j] = ldx[j]; p.rows[j] = tile_rows[j]; p.act[j] = unary[j] < 0 ? 0 : SK_ACT_UNARY + unary[j];
        p.first[j] = groups;
        groups += (N[j] + tile_rows[j] - 1) / tile_rows[j];
        whole = whole && sk_stream_ok(M, K, ldx[j]);
    }
    if (whole)
        return sk_stream_pick(M, K, [&](auto xr, auto one) {
            return sk_stream_launch(skinny_stream_group_kernel<decltype(xr)::value, decltype(one)::value>, decltype(xr)::value,
                                    (unsigned)groups, s, p, M, K / SK_CHUNK, k_tiles);
        });
    int n_waves = 8;
    const int k_chunks = (K + SK_CHUNK - 1) / SK_CHUNK;
    while (n_waves > 1 && n_waves / 2 >= k_chunks) n_waves >>= 1;
    const size_t smem = (size_t)n_waves * 256 * sizeof(float) + (size_t)n_waves * M * SK_XROW;
    if (smem > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(skinny_group_kernel),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL(skinny_group_kernel, dim3(groups), dim3(n_waves * 64), smem, s, p, M, K, k_tiles);
    return bn_launch_status();
}

// The same for products of rows that are formed on the way (bn_skinny_rows' norm of the rows of x [M, K] with weights w).  mu null:
// of these rows; else of their mixes with the rows before them, product j's with weights mu + j K (SkinnyRows), and h [M, K] (bf16)
// gets the normed rows.  All contiguous and 16-byte aligned, state_stride a multiple of 4.
extern "C" int bn_skinny_rows_group(const float* x, const float* w, float eps, const float* mu, const float* state, long long state_stride,
                                    const int* positions, const int* slot_ids, void* h, int count, const void* const* W, void* const* Y,
                                    const int* N, const int* tile_rows, const int* unary, int M, int K, int k_tiles, hipStream_t s) {
    if (count < 1 || count > SK_GROUP || !bn_skinny_rows_supports(M, K, mu ? SK_ROWS_SHIFT : SK_ROWS_NORM) || k_tiles != K / BN_STREAM_TILE_COLS || !x || !w) return BN_ERR_ARG;
    if (mu && (!state || !positions || !slot_ids || !h || state_stride < K || state_stride % 4)) return BN_ERR_ARG;
    if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)mu | (uintptr_t)(mu ? state : nullptr) | (uintptr_t)(mu ? h : nullptr)) & 15) return BN_ERR_ARG;
    SkinnyGroup g = {};
    g.count = count;
    int groups = 0;
    for (int j = 0; j < count; ++j) {
        if (N[j] < 1 || tile_rows[j] < 1 || tile_rows[j] > BN_STREAM_TILE_ROWS || unary[j] < -1 || unary[j] >= BN_UNARY_KINDS || !W[j] ||
            ((uintptr_t)W[j] & 15) || !Y[j])
            return BN_ERR_ARG;
        g.w[j] = (const bf16*)W[j]; g.y[j] = (bf16*)Y[j];
        g.n[j] = N[j]; g.rows[j] = tile_rows[j]; g.act[j] = unary[j] < 0 ? 0 : SK_ACT_UNARY + unary[j];
        g.first[j] = groups;
        groups += (N[j] + tile_rows[j] - 1) / tile_rows[j];
    }
    SkinnyRows p = {};
    p.x = x; p.w = w; p.K = K; p.eps = eps;
    p.mu = mu; p.state = state; p.state_stride = state_stride; p.positions = positions; p.slot_ids = slot_ids; p.h = (bf16*)h;
    return sk_stream_pick(M, K, [&](auto xr, auto) {
        constexpr int XR = decltype(xr)::value < 4 ? decltype(xr)::value : 4, FEW = XR < 2 ? XR : 2;
        auto go = [&](auto kernel) {
            const size_t smem = SK_STREAM_RED * sizeof(float) + (size_t)2 * XR * SK_STAGED_ROW(K);
            hipLaunchKernelGGL(kernel, dim3(groups), dim3(64 * SK_STREAM_WAVES), smem, s, g, p, M, K / SK_CHUNK, k_tiles);
            return bn_launch_status();
        };
        return mu ? go(skinny_stream_rows_group_kernel<FEW, SK_ROWS_SHIFT>) : go(skinny_stream_rows_group_kernel<XR, SK_ROWS_NORM>);
    });
}
