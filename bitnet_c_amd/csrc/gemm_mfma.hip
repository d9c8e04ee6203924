// Prompt-phase matrix product for bf16 on the matrix cores: Y[M, N] = X[M, K] . W[N, K]^T for many
// rows of activations, with float32 accumulation and a bf16 or float32 result.  It has the place of
// the reference's batched products (src/gpu_cuda.cu:11571 hands them to a
// library; its own tiled kernels are src/gpu_cuda.cu:4012-4170), written for 64-wide waves and
// v_mfma_f32_16x16x32_bf16.  Two kernels: gemm_turns_kernel (below) where K is whole steps of 64 and rows
// of Y whole groups of four, which is what a model's prompt has; gemm_mfma_kernel for everything else:
//
// A workgroup of eight waves (2 x 4, two waves on every SIMD so that one multiplies while the other
// waits for shared memory) owns a tile of 256 rows of X by BN (256, 192 or 128) rows of W and
// walks K in steps of 64.  Both operands are K-contiguous, so a lane's MFMA operand is 16
// contiguous bytes of one row.  A step's two tiles are fetched with 16-byte loads (eight threads
// cover the 128 bytes of a row) into registers while earlier steps are multiplied, then parked
// in the other half of shared memory: one barrier a step.  The narrower tiles have registers for
// a second set of loads and fetch two steps ahead.  The loop's body has no branch (rows past the
// end are clamped, a K tail is peeled off), and scheduling barriers keep the loads ahead of the
// products and the stores behind them: left alone, the compiler moves the loads down to their
// stores and every step waits out the memory latency.  A wave raises its priority while it
// multiplies, so that the matrix instructions of one wave are not held up by the loads and
// stores that the other wave of its SIMD issues (+3 to 6 %).  Rows are stored without padding and
// their 16-byte chunks swizzled (chunk c of row r at c ^ swizzle(r)) so that the sixteen lanes
// which shared memory serves together never meet in a bank.
//
// W is the A operand and X the B operand of the instruction: a lane then holds four consecutive
// columns n of one row m of the result, which it stores as one 8- or 16-byte word.  With gate and
// up rows interleaved in blocks of 8 (GLU8, see skinny_gemm.hip) the two halves of eight result
// columns sit in lanes 32 apart of the same tile, and the epilogue writes silu(gate) * up
// (src/transformer/cpu_backend.c:385-391) instead of the product.
//
// Workgroups are numbered so that the eight XCDs (consecutive workgroup ids go to consecutive
// XCDs, each with an L2 of its own) each take a band of W and run through all row tiles of X for
// it: a tile of W comes from HBM once.
//
// Grouped form (a mixture of experts): W is a stack of matrices and the rows of X are ordered by the matrix they meet.  A
// list in device memory cuts the rows into tiles of up to 256 rows of one matrix each (matrix, first row, rows); the grid
// is laid out for the most tiles there can be and a workgroup whose tile is not in the list leaves.  A row's result may
// go to another row of Y (row_map), be scaled (row_scale) and pass an activation of one argument first.
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

#define GM_BM 256             // rows of X per workgroup
#define GM_BK 64              // K elements per step: a tile row is 128 bytes, 8 chunks of 16 bytes
#define GM_XCDS 8
#ifndef GM_WGM
#define GM_WGM 2              // waves of a workgroup along the rows of X ...
#endif
#ifndef GM_WGN
#define GM_WGN 4              // ... and along the rows of W
#endif
#define GM_THREADS (64 * GM_WGM * GM_WGN)

__device__ __forceinline__ bf16x8 gm_as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

#define GM_MAX_ITEMS 6

struct GmGroups {
    const int* tiles;         // [n][3]: matrix of the stack, first row of X, rows (<= GM_BM); null: one product over all rows
    const int* n_tiles;       // [1]: tiles in the list
    const int* row_map;       // [rows of X]: the row of Y that takes row m's result; null: m
    const float* row_scale;   // [rows of X]: a factor on row m's result; null: none
    long long w_stride;       // elements from one matrix of the stack to the next
    int unary;                // BN_UNARY_* applied to the result before anything else; < 0: none
    const bf16* x[GM_MAX_ITEMS];            // (GM_ITEMS: X, W and Y of each product)
    const bf16* w[GM_MAX_ITEMS];
    bf16* y[GM_MAX_ITEMS];
};

// Shared memory serves a 16-byte read in four turns of 16 lanes; in the operand layout
// (lane = i + 16 g reads chunk c0 + g of row i) a turn holds two values of g and, for each, two
// values of i / 4.  Two 128-byte rows share the 256 bytes that the banks span: the row's lowest
// bit separates them, bit 1 goes into bit 2 of the chunk, and (-(i / 4)) & 3 makes g ^ h distinct
// over a turn.
__device__ __forceinline__ int gm_swizzle(int row) {
    return ((-(row >> 2)) & 3) | (((row >> 1) & 1) << 2);
}

// A 16 x 16 tile of the result: lane (i, g) holds columns 4 g .. 4 g + 3, counted from n, of row m.  vec: rows of Y are aligned so that
// the four go out as one word.
template <bool GLU8, typename TO>
__device__ __forceinline__ void gm_store(TO* __restrict__ Y, f32x4 v, int m, int n, int M, int N, int ldy, int vec, int act, int g, const GmGroups& grp) {
    auto store4 = [&](TO* dst, int valid) {
        if (vec && valid >= 4) {
            if (sizeof(TO) == 4) {
                *reinterpret_cast<f32x4*>(dst) = v;
            } else {
                uint2 p;
                p.x = (uint32_t)__builtin_bit_cast(uint16_t, __float2bfloat16(v[0])) |
                      ((uint32_t)__builtin_bit_cast(uint16_t, __float2bfloat16(v[1])) << 16);
                p.y = (uint32_t)__builtin_bit_cast(uint16_t, __float2bfloat16(v[2])) |
                      ((uint32_t)__builtin_bit_cast(uint16_t, __float2bfloat16(v[3])) << 16);
                *reinterpret_cast<uint2*>(dst) = p;
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (r < valid) dst[r] = from_f32<TO>(v[r]);
        }
    };
    if (GLU8) {
        // rows 16t..16t+7 of W are gates, 16t+8..16t+15 the ups of the same result columns:
        // lanes with g >= 2 hold the ups of what lanes g - 2 hold the gates of
        f32x4 up;
#pragma unroll
        for (int r = 0; r < 4; ++r) up[r] = __shfl_xor(v[r], 32, BN_WAVE);
        if (g < 2 && m < M) {
            const int f = (n >> 1) + 4 * g;           // result column of v[0]
#pragma unroll
            // silu(g) * u with the hardware's exp2 and reciprocal (an ulp each, far below the result's
            // rounding): expf and a division cost 25 vector instructions a value, a tenth of this kernel's time
            for (int r = 0; r < 4; ++r)
                v[r] = (act == BN_ACT_SILU ? v[r] * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.44269504f * v[r]))
                                           : bn_gate_act(v[r], act)) * up[r];
            store4(Y + (size_t)m * ldy + f, (N >> 1) - f);
        }
    } else if (m < M) {
        if (grp.unary >= 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = bn_unary_act(v[r], grp.unary);
        }
        if (grp.row_scale) v *= grp.row_scale[m];
        const size_t mo = grp.row_map ? (size_t)grp.row_map[m] : (size_t)m;
        store4(Y + mo * ldy + n + 4 * g, N - n - 4 * g);
    }
}

template <int BN, bool GLU8, typename TO>
__global__ __launch_bounds__(GM_THREADS) void gemm_mfma_kernel(const bf16* __restrict__ X, const bf16* __restrict__ W,
                                                               TO* __restrict__ Y, int M, int N, int K, int ldx, int ldw,
                                                               int ldy, int tiles_m, int tiles_n, int vec, int act, GmGroups grp) {
    constexpr int WM = GM_BM / GM_WGM, WN = BN / GM_WGN;      // a wave's part of the tile
    constexpr int MT = WM / 16, NT = WN / 16;         // 16 x 16 result tiles of a wave: MT x NT
    constexpr int PASS = GM_THREADS / 8;              // rows staged by one pass of the workgroup
    constexpr int XL = GM_BM / PASS, WL = BN / PASS;  // staging loads per thread and step
    extern __shared__ __align__(16) unsigned char smem[];     // [2][(GM_BM + BN) rows][128 bytes]
    constexpr int STAGE = (GM_BM + BN) * 128;

    // workgroup -> tile: XCD x takes the column tiles x, x + 8, ...; inside an XCD the row tiles run fastest
    const int xcd = blockIdx.x % GM_XCDS, local = blockIdx.x / GM_XCDS;
    const int tn = xcd + GM_XCDS * (local / tiles_m), tm = local % tiles_m;
    if (tn >= tiles_n) return;                        // the grid is padded to a multiple of 8 column tiles
    int m0 = tm * GM_BM;
    const int n0 = tn * BN;
    if (grp.tiles) {                                  // the tile's rows end where its matrix's rows end
        if (tm >= grp.n_tiles[0]) return;
        const int* tl = grp.tiles + 3 * tm;
        W += (size_t)tl[0] * grp.w_stride;
        m0 = tl[1];
        M = tl[1] + tl[2];
    }

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int i = lane & 15, g = lane >> 4;
    const int wm = (wave / GM_WGN) * WM, wn = (wave % GM_WGN) * WN;
    const int srow = t >> 3, schunk = t & 7;          // staging: 8 threads a row

    f32x4 acc[NT][MT];
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int b = 0; b < MT; ++b) acc[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};

    struct Regs { uint4 x[XL]; uint4 w[WL]; };
    // rows past the end are clamped (their results are dropped), so that a full step's loads carry no predicate
    const bf16* xbase = X + (size_t)min(m0 + srow, M - 1) * ldx + schunk * 8;
    const bf16* wbase = W + (size_t)min(n0 + srow, N - 1) * ldw + schunk * 8;
    const int xrows_left = M - 1 - (m0 + srow), wrows_left = N - 1 - (n0 + srow);
    auto fetch_full = [&](Regs& r, int k0) {
#pragma unroll
        for (int j = 0; j < XL; ++j)
            r.x[j] = *reinterpret_cast<const uint4*>(xbase + (size_t)max(0, min(PASS * j, xrows_left)) * ldx + k0);
#pragma unroll
        for (int j = 0; j < WL; ++j)
            r.w[j] = *reinterpret_cast<const uint4*>(wbase + (size_t)max(0, min(PASS * j, wrows_left)) * ldw + k0);
    };
    auto fetch_tail = [&](Regs& r, int k0) {
        const bool in = k0 + schunk * 8 < K;
#pragma unroll
        for (int j = 0; j < XL; ++j)
            r.x[j] = in ? *reinterpret_cast<const uint4*>(xbase + (size_t)max(0, min(PASS * j, xrows_left)) * ldx + k0) : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < WL; ++j)
            r.w[j] = in ? *reinterpret_cast<const uint4*>(wbase + (size_t)max(0, min(PASS * j, wrows_left)) * ldw + k0) : make_uint4(0, 0, 0, 0);
    };
    auto park = [&](const Regs& r, int buf) {
        unsigned char* xs = smem + (size_t)buf * STAGE;
        unsigned char* ws = xs + GM_BM * 128;
#pragma unroll
        for (int j = 0; j < XL; ++j) {
            const int row = srow + PASS * j;
            *reinterpret_cast<uint4*>(xs + row * 128 + ((schunk ^ gm_swizzle(row & 15)) << 4)) = r.x[j];
        }
#pragma unroll
        for (int j = 0; j < WL; ++j) {
            const int row = srow + PASS * j;
            *reinterpret_cast<uint4*>(ws + row * 128 + ((schunk ^ gm_swizzle(row & 15)) << 4)) = r.w[j];
        }
    };
    const int swz = gm_swizzle(i);
    auto multiply = [&](int buf) {
        const unsigned char* xs = smem + (size_t)buf * STAGE;
        const unsigned char* ws = xs + GM_BM * 128;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int coff = ((kk * 4 + g) ^ swz) << 4;
            uint4 xf[MT], wf[NT];
#pragma unroll
            for (int b = 0; b < MT; ++b) xf[b] = *reinterpret_cast<const uint4*>(xs + (wm + b * 16 + i) * 128 + coff);
#pragma unroll
            for (int a = 0; a < NT; ++a) wf[a] = *reinterpret_cast<const uint4*>(ws + (wn + a * 16 + i) * 128 + coff);
#pragma unroll
            for (int a = 0; a < NT; ++a)
#pragma unroll
                for (int b = 0; b < MT; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gm_as_bf16x8(wf[a]), gm_as_bf16x8(xf[b]), acc[a][b], 0, 0, 0);
        }
    };

    const int n_steps = (K + GM_BK - 1) / GM_BK;
    const int full = K / GM_BK;                       // steps that need no K guard
    constexpr bool TWO = BN < 256;                    // a second set of staging registers: loads two steps ahead
    Regs r0, r1;
    int s = 0;
    if (TWO) {
        fetch_tail(r0, 0);
        if (n_steps > 1) fetch_tail(r1, GM_BK);
        park(r0, 0);
        __syncthreads();
        // even s: buffer 0 holds step s, r1 step s + 1 (on its way), r0 is free
        for (; s + 3 < full; s += 2) {
            fetch_full(r0, (s + 2) * GM_BK);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(1);
            multiply(0);
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
            park(r1, 1);
            __syncthreads();
            fetch_full(r1, (s + 3) * GM_BK);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(1);
            multiply(1);
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
            park(r0, 0);
            __syncthreads();
        }
        // the rest one step ahead: the step on its way is parked first, then r0 alone carries on
        if (s < n_steps) {
            __builtin_amdgcn_s_setprio(1);
            multiply(0);
            __builtin_amdgcn_s_setprio(0);
            if (s + 1 < n_steps) park(r1, 1);
            __syncthreads();
            ++s;
        }
        for (; s < n_steps; ++s) {
            const bool more = s + 1 < n_steps;
            if (more) fetch_tail(r0, (s + 1) * GM_BK);
            __builtin_amdgcn_s_setprio(1);
            multiply(s & 1);
            __builtin_amdgcn_s_setprio(0);
            if (more) park(r0, (s + 1) & 1);
            __syncthreads();
        }
    } else {
        if (full > 0) fetch_full(r0, 0); else fetch_tail(r0, 0);
        park(r0, 0);
        __syncthreads();
        for (; s + 1 < full; ++s) {                   // the next step is a full one: no branch in the body
            fetch_full(r0, (s + 1) * GM_BK);
            __builtin_amdgcn_sched_barrier(0);        // the loads stay ahead of the products ...
            __builtin_amdgcn_s_setprio(1);
            multiply(s & 1);
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);        // ... and the stores of their data behind them
            park(r0, (s + 1) & 1);
            __syncthreads();
        }
        for (; s < n_steps; ++s) {
            const bool more = s + 1 < n_steps;
            if (more) fetch_tail(r0, (s + 1) * GM_BK);
            __builtin_amdgcn_s_setprio(1);
            multiply(s & 1);
            __builtin_amdgcn_s_setprio(0);
            if (more) park(r0, (s + 1) & 1);
            __syncthreads();
        }
    }

#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int b = 0; b < MT; ++b) gm_store<GLU8>(Y, acc[a][b], m0 + wm + b * 16 + i, n0 + wn + a * 16, M, N, ldy, vec, act, g, grp);
}

// ---------------------------------------------------------------------------------------
// The same product where K is whole steps of 64 (every ordinary width).  What bounds it is the matrix cores' power: at 8,192 rows the
// chip runs this kernel a fifth faster over zeros than over numbers, and so it does the library's.
//
// Eight waves (2 x 4), two on every SIMD, in two groups: waves 0 .. 3 own the upper half of the tile's rows of X, waves 4 .. 7 the lower
// one, half a turn behind (one barrier more in front of their loop, one less behind it).  A step is two turns of a group: it reads
// operands from shared memory while the other group multiplies, then multiplies while the other reads, a barrier between; so the
// matrix cores of a SIMD have one wave's products at a time and never wait for shared memory.  The tile's rows of X are taken in two
// parts (first and second half of each group's), W's in two as well: turn I reads X's first part and both of W's and multiplies
// these, turn II reads X's second part in their place and multiplies it with W's parts that are still in registers.
//
// Loads go from memory straight into shared memory (16 bytes a lane; the swizzle of gm_swizzle lies in the address that a lane asks
// for), into buffers of their own names for every part of the even and the odd steps, so that the compiler knows which loads a read of
// shared memory waits for.  A part's buffer is asked for again, for the step after the next, as soon as both groups have read it, a
// step and a half before it is needed: X's first part and W's two in turn II of the step that read them, X's second part in turn I of
// the next.  The waits are counts of a wave's own later loads; the barrier behind them makes them everybody's.
//   us, registers and one barrier a step (above) -> this, 256 x 256: 4,096 x 4,096 at 4,096 rows 139 -> 101, 28,672 x 4,096 at 2,048 /
//   8,192 rows 479 / 1,892 -> 378 / 1,357, 4,096 x 14,336 at 8,192 870 -> 643 (1.50 PFLOP/s; the library 607).  Four waves of 128 x 128
//   over a ring of four stages of 32 took 1,569 at 28,672 x 4,096 x 8,192, the 32x32x16 instruction 1,459.
//
// splits > 1: K is cut into that many ranges of steps_per steps, Y holds a slab of float32 sums for each.
// Workgroups: XCD x takes a run of the tiles, a run is walked in bands of GM_BAND row tiles, the band's rows fastest, so that the
// workgroups which an XCD runs at a time share rows of X and of W in its L2.
#define GM_BAND 4
// EPI: what becomes of the sums.  Each has kernels of its own: a choice between them at run time makes the epilogue too long for the
// instruction cache (28,672 x 4,096 with its gated unit at 2,048 rows 366 us, with every activation in one kernel 395).
#define GM_STORE 0                    // stored (TO)
#define GM_SILU 1                     // silu(gate) * up
#define GM_GATED_GELU 2               // gelu(gate) * up, the tanh form
#define GM_GROUPED 3                  // the grouped form's
#define GM_ITEMS 4                    // stored, of several products of the same sizes (in the ranges' place)
#define GM_GELU_ERF 5                 // gelu(sum), the exact one
#define GM_RELU2 6                    // max(sum, 0)^2
#define GM_GATED_RELU2 7              // max(gate, 0)^2 * up

// z (1 + erf(z / sqrt 2)) / 2 in 17 instructions (erff's alone are 40, with a branch), by the known form erfc(x) = t exp(-x^2 + p(t)), t = 1 / (1 + c x), with a
// polynomial of its own (below): with x = |z| / sqrt 2 and t = 1 / (1 + 0.46 x),
// erfc(x) / 2 = t 2^(p(t) - x^2 / ln 2), p the polynomial of degree 7 that interpolates log2(exp(x^2) erfc(x) / (2 t)) at the Chebyshev
// points of x in [0, 7] (2.6e-7 off at most).  In float32 within 8e-7 of the value above -2, within 2e-5 of it at -13, where 1 + erff is 0.
__device__ __forceinline__ float gm_gelu_erf(float z) {
    const float x = fabsf(z) * 0.70710678f, t = __builtin_amdgcn_rcpf(fmaf(0.46f, x, 1.0f));
    float p = -0.303036511f;
    p = fmaf(p, t, 1.38259172f);
    p = fmaf(p, t, -2.27948308f);
    p = fmaf(p, t, 1.45173085f);
    p = fmaf(p, t, -0.451854527f);
    p = fmaf(p, t, 0.723021328f);
    p = fmaf(p, t, 1.4218868f);
    p = fmaf(p, t, -2.94485712f);
    const float h = t * __builtin_amdgcn_exp2f(fmaf(x * x, -1.44269504f, p));
    return z * (z < 0.f ? h : 1.0f - h);
}

// The gated units' activations, with the hardware's exp2 and reciprocal (an ulp each): z / (1 + exp(-z)), and z (1 + tanh(y)) / 2 with
// y = sqrt(2 / pi) (z + 0.044715 z^3) as z / (1 + exp(-2 y)), which is the same and has no difference of numbers near 1 in it.  (One kernel for both and
// relu2 with the library's functions: 16,384 x 2,048 at 129 / 2,048 / 8,192 rows with gelu 26 / 143 / 549 us, with relu2 23 / 132 / 511; the library's product
// and the unit's kernel 26 / 118 / 479 and 25 / 117 / 462; this 25 / 109 / 422 and 25 / 106 / 407.)
template <int EPI> __device__ __forceinline__ float gm_gate(float z) {
    if (EPI == GM_SILU) return z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.44269504f * z));
    if (EPI == GM_GATED_GELU) return z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-z * fmaf(0.10294324f, z * z, 2.3022082f)));
    const float p = fmaxf(z, 0.f);
    return p * p;
}

template <int BM, int BN, int EPI, typename TO>
__global__ __launch_bounds__(512, 2) void gemm_turns_kernel(const bf16* __restrict__ X, const bf16* __restrict__ W, TO* __restrict__ Y, int M,
                                                            int N, int K, int ldx, int ldw, int ldy, int tiles_m, int tiles_n, int splits,
                                                            int steps_per, GmGroups grp) {
    constexpr int WM = BM / 2, WN = BN / 4;              // a wave's part of the tile, taken in quarters of (16 MH) x (16 NH)
    constexpr int MH = WM / 32, NH = WN / 32;
    constexpr int XL = (BM / 2 + 63) / 64, WL = BN / 128;        // loads of a wave for a part: 8 rows each
    constexpr int XP = BM / 2 % 64 / 8;                  // waves that take the last of X's (0: all)
    static_assert(BM % 64 == 0 && BN % 128 == 0, "whole 16 x 16 tiles in a quarter");
    __shared__ __align__(1024) unsigned char xa0[BM / 2 * 128], xa1[BM / 2 * 128], xb0[BM / 2 * 128], xb1[BM / 2 * 128];
    __shared__ __align__(1024) unsigned char wa0[BN / 2 * 128], wa1[BN / 2 * 128], wb0[BN / 2 * 128], wb1[BN / 2 * 128];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 15, g = lane >> 4;
    const int wr = wave >> 2, wc = wave & 3;

    // The experts' list holds its tiles in front, and the runs are cut from those: cut from all that the grid is for, the last XCDs' would be empty
    // (both products and what stands around them, us, in gemm_mfma_kernel / runs of all / of those with the width that is now taken, 16 experts of 5,632 x 2,048, two a token: 17 tokens
    // 210 / 236 / 189, 512 239 / 290 / 220, 1,000 277 / 392 / 265, 4,096 723 / 673 / 612; 64 gated ones of 1,536 x 4,096, six a token: 64 tokens 673 / 649 /
    // 529, 2,048 862 / 989 / 755)
    if (EPI == GM_GROUPED) tiles_m = grp.n_tiles[0];
    const int mn = tiles_m * tiles_n, total = mn * splits;
    const int xcd = blockIdx.x % GM_XCDS, local = blockIdx.x / GM_XCDS;
    if (EPI == GM_GROUPED && local >= total / GM_XCDS + (xcd < total % GM_XCDS)) return;
    int id = xcd * (total / GM_XCDS) + min(xcd, total % GM_XCDS) + local;
    const int sp = id / mn;
    id -= sp * mn;
    const int band = id / (GM_BAND * tiles_n), in = id - band * GM_BAND * tiles_n, high = min(GM_BAND, tiles_m - band * GM_BAND);
    const int tm = band * GM_BAND + in % high, n0 = in / high * BN;
    int m0 = tm * BM;
    if (EPI == GM_GROUPED) {                             // the tile's rows end where its matrix's rows end
        const int* tl = grp.tiles + 3 * tm;
        W += (size_t)tl[0] * grp.w_stride;
        m0 = tl[1];
        M = tl[1] + tl[2];
    }
    if constexpr (EPI == GM_ITEMS) { X = grp.x[sp]; W = grp.w[sp]; Y = grp.y[sp]; }
    const int k0 = EPI == GM_ITEMS ? 0 : sp * steps_per, steps = EPI == GM_ITEMS ? K / GM_BK : min(steps_per, K / GM_BK - k0);
    const int rows = min(BM, M - m0), cols = min(BN, N - n0);
    const __amdgpu_buffer_rsrc_t xbuf = bn_buffer(X + (size_t)m0 * ldx, ((rows - 1) * ldx + K) * 2);
    const __amdgpu_buffer_rsrc_t wbuf = bn_buffer(W + (size_t)n0 * ldw, ((cols - 1) * ldw + K) * 2);
    // load j of part p: rows 64 j + 8 wave + lane / 8 of the part, which holds WM / 2 rows of each group (WN / 2 of each column of waves);
    // rows past the end are the last one again
    unsigned xo[2][XL], wo[2][WL];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
#pragma unroll
        for (int j = 0; j < XL; ++j) {
            const int r = 64 * j + 8 * wave + (lane >> 3), R = r / (WM / 2) * WM + p * (WM / 2) + r % (WM / 2);
            xo[p][j] = min(R, rows - 1) * ldx * 2 + (((lane & 7) ^ gm_swizzle(r & 15)) << 4);
        }
#pragma unroll
        for (int j = 0; j < WL; ++j) {
            const int r = 64 * j + 8 * wave + (lane >> 3), R = r / (WN / 2) * WN + p * (WN / 2) + r % (WN / 2);
            wo[p][j] = min(R, cols - 1) * ldw * 2 + (((lane & 7) ^ gm_swizzle(r & 15)) << 4);
        }
    }
    // a step past the last is the last one again: read by nobody
    auto load_x = [&](unsigned char* to, int p, int s) {
#pragma unroll
        for (int j = 0; j < XL; ++j)
            if (XP == 0 || j < XL - 1 || wave < XP) bn_load_to_lds(xbuf, to + (8 * j + wave) * 1024, xo[p][j], (k0 + min(s, steps - 1)) * (GM_BK * 2));
    };
    auto load_w = [&](unsigned char* to, int p, int s) {
#pragma unroll
        for (int j = 0; j < WL; ++j) bn_load_to_lds(wbuf, to + (8 * j + wave) * 1024, wo[p][j], (k0 + min(s, steps - 1)) * (GM_BK * 2));
    };
    const int c0 = (g ^ gm_swizzle(i)) << 4, c1 = ((4 + g) ^ gm_swizzle(i)) << 4;
    bf16x8 xf[MH][2], w0[NH][2], w1[NH][2];
    auto read_x = [&](const unsigned char* from) {
        const unsigned char* b = from + (wr * (WM / 2) + i) * 128;
#pragma unroll
        for (int a = 0; a < MH; ++a) {
            xf[a][0] = *reinterpret_cast<const bf16x8*>(b + a * 2048 + c0);
            xf[a][1] = *reinterpret_cast<const bf16x8*>(b + a * 2048 + c1);
        }
    };
    auto read_w = [&](const unsigned char* from, bf16x8 (&w)[NH][2]) {
        const unsigned char* b = from + (wc * (WN / 2) + i) * 128;
#pragma unroll
        for (int a = 0; a < NH; ++a) {
            w[a][0] = *reinterpret_cast<const bf16x8*>(b + a * 2048 + c0);
            w[a][1] = *reinterpret_cast<const bf16x8*>(b + a * 2048 + c1);
        }
    };
    f32x4 acc[2][2][NH][MH];                             // [part of X][part of W]
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v)
#pragma unroll
            for (int a = 0; a < NH; ++a)
#pragma unroll
                for (int b = 0; b < MH; ++b) acc[u][v][a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](f32x4 (&c)[NH][MH], const bf16x8 (&w)[NH][2]) {
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int a = 0; a < NH; ++a)
#pragma unroll
                for (int b = 0; b < MH; ++b) c[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[a][kk], xf[b][kk], c[a][b], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
    };
    // What the next turn reads has arrived when no more of this wave's loads are on their way than it has asked for since: in either
    // turn X's two parts and W's two.  This turn's operands are in registers as well: their buffers may be asked for again.
    auto arrived = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        if (XP == 0 || wave < XP) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * XL + 2 * WL) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * XL - 2 + 2 * WL) : "memory");
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto turn = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto step = [&](int s, unsigned char* x0, unsigned char* x1, unsigned char* v0, unsigned char* v1, unsigned char* other_x1) {
        read_x(x0); read_w(v0, w0); read_w(v1, w1); load_x(other_x1, 1, s + 1);
        arrived(); multiply(acc[0][0], w0); multiply(acc[0][1], w1); turn();
        read_x(x1); load_x(x0, 0, s + 2); load_w(v0, 0, s + 2); load_w(v1, 1, s + 2);
        arrived(); multiply(acc[1][1], w1); multiply(acc[1][0], w0); turn();
    };
    load_x(xa0, 0, 0); load_w(wa0, 0, 0); load_w(wa1, 1, 0); load_x(xa1, 1, 0);
    load_x(xb0, 0, 1); load_w(wb0, 0, 1); load_w(wb1, 1, 1);
    arrived();
    if (wr == 1) turn();
    int s = 0;
    for (; s + 1 < steps; s += 2) {
        step(s, xa0, xa1, wa0, wa1, xb1);
        step(s + 1, xb0, xb1, wb0, wb1, xa1);
    }
    if (s < steps) step(s, xa0, xa1, wa0, wa1, xb1);
    if (wr == 0) turn();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // nothing is on its way into shared memory when the wave ends

    // lane (i, g) of a 16 x 16 tile holds columns 4 g .. 4 g + 3 of row i; rows of Y are whole groups of four (the host has seen to it)
    auto store = [&](TO* dst, const f32x4& v) {
        if (sizeof(TO) == 4) {
            *reinterpret_cast<f32x4*>(dst) = v;
        } else {
            uint2 p;
            p.x = (uint32_t)__builtin_bit_cast(uint16_t, __float2bfloat16(v[0])) | ((uint32_t)__builtin_bit_cast(uint16_t, __float2bfloat16(v[1])) << 16);
            p.y = (uint32_t)__builtin_bit_cast(uint16_t, __float2bfloat16(v[2])) | ((uint32_t)__builtin_bit_cast(uint16_t, __float2bfloat16(v[3])) << 16);
            *reinterpret_cast<uint2*>(dst) = p;
        }
    };
    if (EPI == GM_STORE) Y += (size_t)sp * M * ldy;
    constexpr bool GATED = EPI == GM_SILU || EPI == GM_GATED_GELU || EPI == GM_GATED_RELU2;
    if constexpr (sizeof(TO) == 2 && !GATED && EPI != GM_GROUPED) {
        // bf16 rows go out through shared memory, which nobody reads any more: a wave's part of the tile is written to a buffer of its
        // own, the 16-byte chunks of a row swizzled, and read back row by row, so that a store writes whole rows of 128 bytes and not 32
        // bytes of sixteen (8,192 x 2,048 at 2,048 / 8,192 rows 65.8 -> 52.6, 244 -> 207 us: rows of Y a power of two apart share a
        // channel of the cache; 16,384 x 4,096 197 -> 189, 781 -> 760; 2,048 x 512 at 129 rows 8.8 -> 7.8.  Gated units, whose rows are
        // half as long, are as fast without).
        constexpr int CH = WN / 8, RB = WN * 2, HALF = WM / 2;               // chunks and bytes of a wave's row
        asm volatile("s_barrier" ::: "memory");          // everybody's loads have arrived
        unsigned char* mine = wave == 0 ? xa0 : wave == 1 ? xa1 : wave == 2 ? xb0 : wave == 3 ? xb1 : wave == 4 ? wa0 : wave == 5 ? wa1 : wave == 6 ? wb0 : wb1;
        auto at = [&](int row, int chunk) { return mine + row * RB + ((chunk ^ (row / (256 / RB) & (CH - 1))) << 4); };
        const bool wide = ldy % 8 == 0 && (reinterpret_cast<uintptr_t>(Y) & 15) == 0;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int b = 0; b < MH; ++b)
#pragma unroll
                for (int v = 0; v < 2; ++v)
#pragma unroll
                    for (int a = 0; a < NH; ++a) {
                        f32x4 c = acc[u][v][a][b];
                        if (EPI == GM_GELU_ERF) {
#pragma unroll
                            for (int r = 0; r < 4; ++r) c[r] = gm_gelu_erf(c[r]);
                        } else if (EPI == GM_RELU2) {
#pragma unroll
                            for (int r = 0; r < 4; ++r) c[r] = bn_unary_act(c[r], BN_UNARY_RELU2);
                        }
                        store(reinterpret_cast<TO*>(at(u * HALF + b * 16 + i, (v * (WN / 2) + a * 16 >> 3) + (g >> 1)) + 8 * (g & 1)), c);
                    }
#pragma unroll
            for (int r0 = 0; r0 < HALF; r0 += 64 / CH) {
                const int row = u * HALF + r0 + lane / CH, m = m0 + wr * WM + row, n = n0 + wc * WN + lane % CH * 8;
                const uint4 p = *reinterpret_cast<const uint4*>(at(row, lane % CH));
                if (m >= M || n >= N) continue;
                TO* dst = Y + (size_t)m * ldy + n;
                if (wide && n + 8 <= N) {
                    *reinterpret_cast<uint4*>(dst) = p;
                } else {
                    *reinterpret_cast<uint2*>(dst) = make_uint2(p.x, p.y);
                    if (n + 8 <= N) *reinterpret_cast<uint2*>(dst + 4) = make_uint2(p.z, p.w);
                }
            }
        }
        return;
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v)
#pragma unroll
            for (int a = 0; a < NH; ++a)
#pragma unroll
                for (int b = 0; b < MH; ++b) {
                    const int m = m0 + wr * WM + u * (WM / 2) + b * 16 + i, n = n0 + wc * WN + v * (WN / 2) + a * 16;
                    f32x4 c = acc[u][v][a][b];
                    if (GATED) {
                        // rows n .. n + 7 of W are gates, n + 8 .. n + 15 the ups of the same columns: the lanes with g >= 2 hold the ups
                        // of what the lanes with g - 2 hold the gates of
                        f32x4 up;
#pragma unroll
                        for (int r = 0; r < 4; ++r) up[r] = __shfl_xor(c[r], 32, BN_WAVE);
#pragma unroll
                        for (int r = 0; r < 4; ++r) c[r] = gm_gate<EPI>(c[r]) * up[r];
                        if (g < 2 && m < M && n < N) store(Y + (size_t)m * ldy + (n >> 1) + 4 * g, c);
                    } else if (m < M && n + 4 * g < N) {
                        size_t mo = m;
                        if (EPI == GM_GROUPED) {
                            if (grp.unary >= 0) {
#pragma unroll
                                for (int r = 0; r < 4; ++r) c[r] = bn_unary_act(c[r], grp.unary);
                            }
                            if (grp.row_scale) c *= grp.row_scale[m];
                            if (grp.row_map) mo = grp.row_map[m];
                        }
                        store(Y + mo * ldy + n + 4 * g, c);
                    }
                }
}

static GmGroups gm_no_groups() {
    GmGroups g;
    g = {};
    g.unary = -1;
    return g;
}

template <int BN, bool GLU8, typename TO>
static int gm_launch(const void* X, const void* W, void* Y, int M, int N, int K, int ldx, int ldw, int ldy, int act,
                     hipStream_t s, GmGroups grp = gm_no_groups(), int max_tiles = 0) {
    auto kernel = gemm_mfma_kernel<BN, GLU8, TO>;
    const size_t smem = (size_t)2 * (GM_BM + BN) * 128;
    static bool raised = false;                       // per instantiation
    if (!raised) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return (int)e;
        raised = true;
    }
    const int tiles_m = grp.tiles ? max_tiles : (M + GM_BM - 1) / GM_BM, tiles_n = (N + BN - 1) / BN;
    const int bands = (tiles_n + GM_XCDS - 1) / GM_XCDS;           // column tiles per XCD
    const long long grid = (long long)bands * GM_XCDS * tiles_m;
    if (grid > 0x7fffffffLL) return BN_ERR_ARG;
    const int vec = (ldy % 4 == 0 && ((uintptr_t)Y % (4 * sizeof(TO))) == 0) ? 1 : 0;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(GM_THREADS), smem, s, (const bf16*)X, (const bf16*)W, (TO*)Y,
                       M, N, K, ldx, ldw, ldy, tiles_m, tiles_n, vec, act, grp);
    return bn_launch_status();
}

static int gm_compute_units() {
    static int cus = 0;
    if (!cus) {
        int dev = 0;
        hipDeviceProp_t p;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess) cus = p.multiProcessorCount;
        if (cus <= 0) cus = 256;
    }
    return cus;
}

// Tiles of the form above and what a step of 64 takes, us: a tile alone on its CU, and two where shared memory leaves room for two (0:
// it does not).  Fitted to 2,600 measurements of 14 matrices at 129 to 8,192 rows, which it meets within 8 % (rms): a round costs
// GM_ROUND more (the first loads, the stores), and a step of a round that fills no CU would take GM_IDLE of it (power, memory).
struct GmTile { int bm, bn; double one, two; };
static const GmTile gm_tiles[] = {{256, 256, 1.46, 0.}, {192, 256, 1.17, 0.}, {128, 256, 0.92, 0.}, {256, 128, 0.91, 0.}, {192, 128, 0.74, 1.38}, {128, 128, 0.61, 1.06}};
#define GM_TILES 6
#define GM_ROUND 7.3
#define GM_IDLE 0.68
#define GM_MAX_SPLITS 6

static double gm_cost(const GmTile& t, long long tiles, int steps, int cus, double start) {
    auto round = [&](double step, double fill) { return start + steps * step * (GM_IDLE + (1. - GM_IDLE) * fill); };
    if (t.two > 0.) {                                    // two a CU run on without rounds
        if (tiles <= cus) return round(t.one, (double)tiles / cus);
        if (tiles <= 2 * cus) return round(t.two, tiles / (2. * cus));
        return 2 * start + steps * t.two * tiles / (2. * cus);
    }
    return tiles / cus * round(t.one, 1.) + (tiles % cus ? round(t.one, (double)(tiles % cus) / cus) : 0.);
}

// The tile and the ranges of K (up to max_splits) that take the least time for M rows, N rows of W and K columns; slabs are written and
// read again at 5 TB/s, and more than two of them cost a launch.  bm: the only height to look at, or 0.  cold: what a round costs besides for
// every 256 of its tiles' columns.
static void gm_plan(int M, int N, int K, int bm, int max_splits, int* tile, int* splits, int items = 1, double cold = 0.) {
    const int cus = gm_compute_units(), steps = K / GM_BK;
    double best = -1.;
    for (int i = 0; i < GM_TILES; ++i) {
        const GmTile& t = gm_tiles[i];
        if (bm && t.bm != bm) continue;
        const long long tiles = (long long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * items;
        for (int s = 1; s <= max_splits; ++s) {
            const int per = (steps + s - 1) / s;
            if ((steps + per - 1) / per != s) continue;
            const double cost = gm_cost(t, tiles * s, per, cus, GM_ROUND + cold * t.bn / 256) + (s > 1 ? s * 8e-6 * M * N / 5. + (s > 2 ? 4. : 0.) : 0.);
            if (best < 0. || cost < best) { best = cost; *tile = i; *splits = s; }
        }
    }
}

// whole steps, 32-bit offsets inside a tile, results in whole groups of four
static bool gm_turns_takes(int N, int K, int ldx, int ldw, int ldy, const void* Y, int size) {
    return K % GM_BK == 0 && ldx <= 1 << 22 && ldw <= 1 << 22 && N % 4 == 0 && ldy % 4 == 0 && (uintptr_t)Y % (4 * size) == 0;
}

template <int BM, int BN, int EPI, typename TO>
static int gm_turns_launch(const void* X, const void* W, void* Y, int M, int N, int K, int ldx, int ldw, int ldy, int splits, hipStream_t s,
                           const GmGroups& grp, int max_tiles) {
    const int tiles_m = EPI == GM_GROUPED ? max_tiles : (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    const long long grid = (long long)tiles_m * tiles_n * splits;
    if (grid > 0x7fffffffLL) return BN_ERR_ARG;
    hipLaunchKernelGGL((gemm_turns_kernel<BM, BN, EPI, TO>), dim3((unsigned)grid), dim3(512), 0, s, (const bf16*)X, (const bf16*)W, (TO*)Y, M, N, K,
                       ldx, ldw, ldy, tiles_m, tiles_n, splits, (K / GM_BK + splits - 1) / splits, grp);
    return bn_launch_status();
}

template <int EPI, typename TO>
static int gm_turns(int tile, const void* X, const void* W, void* Y, int M, int N, int K, int ldx, int ldw, int ldy, int splits,
                    hipStream_t s, const GmGroups& grp, int max_tiles = 0) {
#define GM_TILE(I, BM_, BN_) \
    if (tile == I) return gm_turns_launch<BM_, BN_, EPI, TO>(X, W, Y, M, N, K, ldx, ldw, ldy, splits, s, grp, max_tiles)
    GM_TILE(0, 256, 256);
    GM_TILE(3, 256, 128);
    if constexpr (EPI != GM_GROUPED) {                   // grouped tiles are 256 rows
        GM_TILE(1, 192, 256);
        GM_TILE(2, 128, 256);
        GM_TILE(4, 192, 128);
        GM_TILE(5, 128, 128);
    }
#undef GM_TILE
    return BN_ERR_ARG;
}

static int gm_pick_bn(int M, int N, int cus) {
    const int widths[3] = {256, 192, 128};
    const int weight[3] = {100, 104, 112};            // cost of a result column, relative
    const long long tiles_m = (M + GM_BM - 1) / GM_BM;
    long long best = -1;
    int pick = 128;
    for (int c = 0; c < 3; ++c) {
        const long long wgs = tiles_m * ((N + widths[c] - 1) / widths[c]);
        const long long cost = ((wgs + cus - 1) / cus) * widths[c] * weight[c];
        if (best < 0 || cost < best) { best = cost; pick = widths[c]; }
    }
    return pick;
}

// 1 if the kernel takes the shape.
extern "C" int bn_gemm_mfma_supports(int M, int N, int K, int ldx, int ldw) {
    return (M >= 1 && N >= 1 && K >= 8 && K % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0 && ldx >= K && ldw >= K) ? 1 : 0;
}

// out_dtype: type of Y (bf16 or float32).  glu8 != 0: W has 2N rows, gate and up interleaved in
// blocks of 8 (N a multiple of 8), and Y[M, N] = act(gate) * up, act one of BN_ACT_*.  width: the tile's rows of W
// (256, 192 or 128), or 0 for the one that suits the shape.
extern "C" int bn_gemm_mfma(int out_dtype, const void* X, const void* W, void* Y, int M, int N, int K, int ldx, int ldw,
                            int ldy, int glu8, int act, int width, hipStream_t s) {
    if (!bn_gemm_mfma_supports(M, N, K, ldx, ldw) || ldy < N || act < 0 || act >= BN_ACT_KINDS) return BN_ERR_ARG;
    if (width != 0 && width != 256 && width != 192 && width != 128) return BN_ERR_ARG;
    if (((uintptr_t)X | (uintptr_t)W) & 15) return BN_ERR_ARG;
    if (out_dtype != BN_DT_BF16 && out_dtype != BN_DT_F32) return BN_ERR_DTYPE;
    if (glu8) {
        if (N % 8) return BN_ERR_ARG;
        N *= 2;                                       // rows of W
    }
    const bool f32 = out_dtype == BN_DT_F32;
    if (width != 192 && !(glu8 && f32) && gm_turns_takes(N, K, ldx, ldw, ldy, Y, f32 ? 4 : 2)) {
        int tile = width == 256 ? 0 : 3, splits = 1;
        if (!width) gm_plan(M, N, K, 0, 1, &tile, &splits);
        const GmGroups none = gm_no_groups();
        if (glu8 && act == BN_ACT_SILU) return gm_turns<GM_SILU, bf16>(tile, X, W, Y, M, N, K, ldx, ldw, ldy, 1, s, none);
        if (glu8 && act == BN_ACT_GELU_TANH) return gm_turns<GM_GATED_GELU, bf16>(tile, X, W, Y, M, N, K, ldx, ldw, ldy, 1, s, none);
        if (glu8) return gm_turns<GM_GATED_RELU2, bf16>(tile, X, W, Y, M, N, K, ldx, ldw, ldy, 1, s, none);
        return f32 ? gm_turns<GM_STORE, float>(tile, X, W, Y, M, N, K, ldx, ldw, ldy, 1, s, none)
                   : gm_turns<GM_STORE, bf16>(tile, X, W, Y, M, N, K, ldx, ldw, ldy, 1, s, none);
    }
    // The tile width: the one with the least work on the busiest CU (rounds of workgroups over the
    // CUs times the width), a wider tile counting a little less than its width because it reads
    // less of X per result.
    const int bn = width ? width : gm_pick_bn(M, N, gm_compute_units());
#define GM_GO(BN_, GLU_)                                                                          \
    return f32 ? gm_launch<BN_, GLU_, float>(X, W, Y, M, N, K, ldx, ldw, ldy, act, s)             \
               : gm_launch<BN_, GLU_, bf16>(X, W, Y, M, N, K, ldx, ldw, ldy, act, s)
    if (glu8) {
        if (bn == 256) { GM_GO(256, true); }
        if (bn == 192) { GM_GO(192, true); }
        GM_GO(128, true);
    }
    if (bn == 256) { GM_GO(256, false); }
    if (bn == 192) { GM_GO(192, false); }
    GM_GO(128, false);
#undef GM_GO
}

// Ranges of K into which bn_gemm_mfma_slabs cuts a product (1 to GM_MAX_SPLITS).
extern "C" int bn_gemm_mfma_splits(int M, int N, int K) {
    if (M < 1 || N < 1 || K < GM_BK || K % GM_BK) return 0;
    int tile = 0, splits = 1;
    gm_plan(M, N, K, 0, GM_MAX_SPLITS, &tile, &splits);
    return splits;
}

// Y [splits, M, N] (float32, contiguous): the sums of X . W^T over bn_gemm_mfma_splits(M, N, K) ranges of K; whole steps of K.
extern "C" int bn_gemm_mfma_slabs(const void* X, const void* W, float* Y, int M, int N, int K, int ldx, int ldw, int splits, hipStream_t s) {
    if (!bn_gemm_mfma_supports(M, N, K, ldx, ldw) || !gm_turns_takes(N, K, ldx, ldw, N, Y, 4) || (((uintptr_t)X | (uintptr_t)W) & 15)) return BN_ERR_ARG;
    int tile = 0, plan = 1;
    gm_plan(M, N, K, 0, GM_MAX_SPLITS, &tile, &plan);
    if (plan != splits) return BN_ERR_ARG;
    return gm_turns<GM_STORE, float>(tile, X, W, Y, M, N, K, ldx, ldw, N, splits, s, gm_no_groups());
}

// Y [M, N] (bf16, contiguous) = act(X . W^T) on the float32 sums, act the exact gelu or relu2 (BN_UNARY_*).
extern "C" int bn_gemm_mfma_unary(const void* X, const void* W, void* Y, int M, int N, int K, int ldx, int ldw, int kind, hipStream_t s) {
    if (!bn_gemm_mfma_supports(M, N, K, ldx, ldw) || !gm_turns_takes(N, K, ldx, ldw, N, Y, 2) || (((uintptr_t)X | (uintptr_t)W) & 15)) return BN_ERR_ARG;
    if (kind != BN_UNARY_GELU_ERF && kind != BN_UNARY_RELU2) return BN_ERR_ARG;
    int tile = 0, splits = 1;
    gm_plan(M, N, K, 0, 1, &tile, &splits);
    return kind == BN_UNARY_RELU2 ? gm_turns<GM_RELU2, bf16>(tile, X, W, Y, M, N, K, ldx, ldw, N, 1, s, gm_no_groups())
                                  : gm_turns<GM_GELU_ERF, bf16>(tile, X, W, Y, M, N, K, ldx, ldw, N, 1, s, gm_no_groups());
}

// y[i] [M, N] (bf16, contiguous) = x[i] . w[i]^T for n products of the same sizes, in one launch: rows of x[i] ldx apart, w[i] contiguous.
// A product of 2,048 x 2,048 over 2,048 rows is 128 tiles of 256 x 128 on 256 CUs and 23 us, as long as the other half stands idle; four
// of them side by side are two whole rounds of 256 x 256 tiles' work, 57 us instead of 93 (1.2 PFLOP/s).  The item takes the place of the
// range of K, so that the kernels' loops are the same; the tile is the one that suits all items' tiles together.
extern "C" int bn_gemm_mfma_items(int n, const void* const* x, const void* const* w, void* const* y, int M, int N, int K, int ldx, hipStream_t s) {
    if (n < 1 || n > GM_MAX_ITEMS || !bn_gemm_mfma_supports(M, N, K, ldx, K)) return BN_ERR_ARG;
    GmGroups g = gm_no_groups();
    for (int i = 0; i < n; ++i) {
        if (!x[i] || !w[i] || !y[i] || (((uintptr_t)x[i] | (uintptr_t)w[i]) & 15) || !gm_turns_takes(N, K, ldx, K, N, y[i], 2)) return BN_ERR_ARG;
        g.x[i] = (const bf16*)x[i]; g.w[i] = (const bf16*)w[i]; g.y[i] = (bf16*)y[i];
    }
    int tile = 0, splits = 1;
    gm_plan(M, N, K, 0, 1, &tile, &splits, n);
    return gm_turns<GM_ITEMS, bf16>(tile, nullptr, nullptr, nullptr, M, N, K, ldx, K, N, n, s, g);
}

// The grouped form: X [rows, K] ordered by matrix, W [matrices][N, K] (w_stride elements apart), tiles [max_tiles][3] and
// n_tiles [1] in device memory (tiles of at most 256 rows), Y row row_map[m] (or m) = unary(X[m] . W[matrix]^T) * row_scale[m].
// rows: all rows of X (sizes the tile width).  out_dtype: type of Y.
extern "C" int bn_gemm_mfma_grouped(int out_dtype, const void* X, const void* W, void* Y, const int* tiles, const int* n_tiles,
                                    int max_tiles, const int* row_map, const float* row_scale, long long w_stride, int unary,
                                    int rows, int N, int K, int ldx, int ldw, int ldy, hipStream_t s) {
    if (!bn_gemm_mfma_supports(rows, N, K, ldx, ldw) || ldy < N || max_tiles < 1 || !tiles || !n_tiles || w_stride < 0) return BN_ERR_ARG;
    if (unary >= BN_UNARY_KINDS || (((uintptr_t)X | (uintptr_t)W) & 15) || (w_stride % 8)) return BN_ERR_ARG;
    if (out_dtype != BN_DT_BF16 && out_dtype != BN_DT_F32) return BN_ERR_DTYPE;
    GmGroups g;
    g.tiles = tiles; g.n_tiles = n_tiles; g.row_map = row_map; g.row_scale = row_scale; g.w_stride = w_stride;
    g.unary = unary < 0 ? -1 : unary;
    const bool f32 = out_dtype == BN_DT_F32;
    if (gm_turns_takes(N, K, ldx, ldw, ldy, Y, f32 ? 4 : 2)) {
        // Tiles that hold rows, if the rows are spread evenly over the matrices (a tenth of a tile more makes no other); a tile of an expert's matrix is
        // read from memory and by few others, so that a round starts later.  us, the width by rows / 256 tiles and a round as above -> this, 16 experts of
        // 5,632 x 2,048, two a token: 1,000 tokens 291 -> 265, 1,600 314 -> 287, 2,048 383 -> 398; of 2 x 5,504 x 4,096 200 569 -> 493
        // (with the number of tiles known the width is within 5 % of the better of the two everywhere, so within 16 %).
        const int full = (rows + GM_BM - 1) / GM_BM, matrices = max_tiles - full;
        const int live = matrices < 1 ? full : std::min(max_tiles, matrices * std::max(1, (rows / matrices - GM_BM / 10 + GM_BM - 1) / GM_BM));
        int tile = 0, splits = 1;
        gm_plan(live * GM_BM, N, K, GM_BM, 1, &tile, &splits, 1, 17.);
        return f32 ? gm_turns<GM_GROUPED, float>(tile, X, W, Y, rows, N, K, ldx, ldw, ldy, 1, s, g, max_tiles)
                   : gm_turns<GM_GROUPED, bf16>(tile, X, W, Y, rows, N, K, ldx, ldw, ldy, 1, s, g, max_tiles);
    }
    const int bn = gm_pick_bn(rows, N, gm_compute_units());
#define GM_GO_GROUPED(BN_)                                                                                         \
    return f32 ? gm_launch<BN_, false, float>(X, W, Y, rows, N, K, ldx, ldw, ldy, 0, s, g, max_tiles)          \
               : gm_launch<BN_, false, bf16>(X, W, Y, rows, N, K, ldx, ldw, ldy, 0, s, g, max_tiles)
    if (bn == 256) { GM_GO_GROUPED(256); }
    if (bn == 192) { GM_GO_GROUPED(192); }
    GM_GO_GROUPED(128);
#undef GM_GO_GROUPED
}
