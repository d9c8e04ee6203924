// Shared device helpers for the gfx950 kernels of this library.
// Wavefronts are 64 lanes wide; every reduction below assumes that.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

#define BN_WAVE 64
#define BN_PAGE 64            // tokens per cache page; the Python side reads this line (csrc/build.py: header_constant)
// Decode attention splits a sequence's keys over workgroups in runs of at least this many pages: shorter
// runs cost more in merging than they gain in parallelism (measured at batch 1, 8 and 64 of an 8B shape).  The general
// kernel's waves walk a run alone: where few partial sums are left its runs are single pages (AG_PAGE_RUN_ROWS).
#define BN_SPLIT_MIN_PAGES 2
// A float32 cache's keys are summed by attn_rows.hip (what attn_f32.hip, with runs of its own, does not take) in runs of this
// many positions (whole pages, counted from position 0), each run by
// itself and the runs folded in order: a decode step then spreads a long sequence's runs over workgroups and still forms
// every sum in the order in which a prompt step forms it, so that float32 logits do not depend on how a sequence was cut.
#define BN_F32_FOLD_KEYS 2048
#define BN_MAX_HEAD_DIM 256   // the attention kernels take every even head size up to this; the configuration reads this line too
// A latent beside a rotated part is one wide "head" that all query heads share: the vector attention kernel takes key rows
// up to this width, and values up to that one.
#define BN_MAX_LATENT_KEY 576
#define BN_MAX_LATENT_VALUE 512

// The streamed copy of a bf16 weight matrix W[N, K], for the kernels that read W once per call in the operand layout of
// v_mfma_f32_16x16x32_bf16 (lane l = r + 16 g holds columns 8 g .. 8 g + 7 of row r of a 16 x 32 block): tile (a, b) is rows
// R a .. R a + R - 1, columns 32 b .. 32 b + 31, for a number R <= 16 of rows per tile that the copy names (16, or fewer
// where that spreads the tiles more evenly over the CUs); its 32 R elements are stored so that the eight of lane
// r + 16 g (r < R) are the elements 8 (R g + r) .. 8 (R g + r) + 7; tiles in the order [ceil(N / R)][ceil(K / 32)], rows
// past N and columns past K zero.  One load of a wave reads one tile as 64 R consecutive bytes (the lanes r >= R idle).
// A float32 matrix (gemm_f32.hip) is kept the same way in tiles of R rows x 16 columns, four columns to a lane's 16 bytes:
// the elements 4 (R g + r) .. 4 (R g + r) + 3 of a tile are columns 4 g .. 4 g + 3 of its row r.
// The Python side reads these lines too.
#define BN_STREAM_TILE_ROWS 16        // the most rows of a tile
#define BN_STREAM_TILE_COLS 32
#define BN_STREAM_TILE_COLS_F32 16

// Cache pages in the matrix-core attention kernels' own order ("blocked"; bf16, head sizes that are multiples of 32).  A
// page still holds BN_PAGE positions of hs elements for every kv head, keys and values each, but inside a (page, kv head)
// they lie in blocks of 32 positions, and a block in the order in which a wave of the decode kernel loads it: one load
// instruction takes 1 KB of consecutive bytes where pages that hold a row per position (or a row per dimension) give it
// 64 bytes in each of 16 rows.  With position p = 32 b + r inside the page:
//   keys:   the operand of the first product (S^T = K Q^T) is a tile of 16 positions x 32 dimensions, lane i + 16 g holding
//           dimensions 8 g .. 8 g + 7 of tile row i; a block is two such row sets (tile 0: r = 8 (i / 4) + i % 4, tile 1:
//           4 further) for each of hs / 32 dimension chunks c.  Element (p, d = 32 c + 8 g + e) lies at
//           32 hs b + 8 (64 (2 c + tile) + 16 g + i) + e.
//   values: the operand of the second product is a tile of 16 dimensions x 32 positions, lane i + 16 g holding positions
//           8 g .. 8 g + 7 of dimension 16 t + i.  Element (p = 32 b + 8 g + e, d = 16 t + i) lies at
//           32 hs b + 8 (64 t + 16 g + i) + e.
// Eight consecutive dimensions of a key, and eight consecutive positions (from a multiple of 8) of a value's dimension,
// stay 16 consecutive bytes, which is what the writers store at once.
#define BN_KV_BLOCK 32
// the head sizes that the matrix-core attention kernels are built for (the Python side reads these lines)
#define BN_MFMA_HEAD_DIM_SMALL 64
#define BN_MFMA_HEAD_DIM_LARGE 128
__host__ __device__ __forceinline__ int bn_blocked_k_offset(int p, int d, int hs) {
    const int b = p >> 5, r = p & 31;
    const int tile = (r >> 2) & 1, i = ((r >> 3) << 2) | (r & 3);
    return 32 * hs * b + 8 * (64 * (2 * (d >> 5) + tile) + 16 * ((d >> 3) & 3) + i) + (d & 7);
}
__host__ __device__ __forceinline__ int bn_blocked_v_offset(int p, int d, int hs) {
    const int b = p >> 5;
    return 32 * hs * b + 8 * (64 * (d >> 4) + 16 * ((p >> 3) & 3) + (d & 15)) + (p & 7);
}

// error codes returned by the extern "C" entry points (0 = ok, >0 = hipError_t)
#define BN_ERR_ARG   (-1)     // an argument the kernel cannot take (size, alignment)
#define BN_ERR_DTYPE (-2)

#define BN_DT_F32  0
#define BN_DT_BF16 1

typedef __hip_bfloat16 bf16;

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(bf16 v) { return __bfloat162float(v); }
template <typename T> __device__ __forceinline__ T from_f32(float v);
template <> __device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16 from_f32<bf16>(float v) { return __float2bfloat16(v); }

// bf16 bits <-> float without going through the class type (for packed loads)
__device__ __forceinline__ float bf16_bits_to_f32(uint16_t b) {
    return __uint_as_float(((uint32_t)b) << 16);
}
// A rotation of (x0, x1) by an angle, its operations written out: the same bits in every kernel that turns float32 heads.
__device__ __forceinline__ void bn_rotate_pair(float& x0, float& x1, float c, float s) {
    const float y0 = __fmaf_rn(x0, c, -__fmul_rn(x1, s));
    x1 = __fmaf_rn(x0, s, __fmul_rn(x1, c));
    x0 = y0;
}
__device__ __forceinline__ float bf16lo_to_f32(uint32_t two) { return __uint_as_float(two << 16); }
__device__ __forceinline__ float bf16hi_to_f32(uint32_t two) { return __uint_as_float(two & 0xffff0000u); }

// Sixteen bytes that a launch reads once (a streamed copy of weights, the blocked keys and values of a decode step), as a
// non-temporal load: the line takes no other line's place in the L2 for long.  A plain read of cold memory by 256 to 1,792
// workgroups, us without and with it: 8 MB 3.45 / 3.12, 32 MB 6.7 / 6.4, 48 MB 9.3 / 8.8, 112 MB 19.5 / 18.4, 224 MB
// 38.0 / 35.8; no slower where the bytes lie in a cache from the launch before.  Where one load of a wave takes half a line of each
// of 16 rows and another one the other half (row-major weights) plain loads are faster, since the line is asked for twice: us at
// one row, with it / plain, 2,048 x 2,048 5.4 / 4.7, 2,048 x 5,632 10.9 / 9.8, 28,672 x 4,096 45.8 / 41.6, 4,096 x 14,336 26.9 / 25.2
// (4,096 x 4,096 9.3 / 9.4), partial sums of 32 rows 2,048 x 2,048 8.7 / 7.7, 4,096 x 14,336 29.5 / 27.2.
typedef __attribute__((ext_vector_type(4))) uint32_t bn_u32x4;
__device__ __forceinline__ uint4 bn_load_once(const void* p) {
    return __builtin_bit_cast(uint4, __builtin_nontemporal_load(static_cast<const bn_u32x4*>(p)));
}

// A buffer of `bytes` bytes for loads with one 32-bit offset a lane and one in a scalar register: no 64-bit addresses in
// vector registers, and nothing past the buffer's end is read.
#define BN_BUFFER_NT 2                // the loads' cache policy: non-temporal
__device__ __forceinline__ __amdgpu_buffer_rsrc_t bn_buffer(const void* p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00027000);
}

// A load of 16 bytes a lane from a buffer straight into shared memory: lane l's bytes go to lds + 16 l (lds the same in every
// lane).  The wave's count of outstanding loads covers it.
__device__ __forceinline__ void bn_load_to_lds(__amdgpu_buffer_rsrc_t b, void* lds, unsigned lane_offset, unsigned offset) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(b, (__attribute__((address_space(3))) void*)lds, 16, lane_offset, offset, 0, 0);
}

// Reductions over a wave as a butterfly: every lane adds the lane 32, 16, 8, 4, 2 and 1 away, in that order.  The two long
// steps swap halves and rows (v_permlane32_swap, v_permlane16_swap), the short ones are data-parallel-primitive moves inside
// a row of 16; through shared memory's crossbar (__shfl_xor) every step waits some 120 cycles for the one before it, a third
// of a microsecond a sum in kernels that take three (whole calls of Llama, Fazopel and Sunusun at 2,048 columns take 1 to 4 %
// less, block_sum's barriers included).  The same pairs are added either way: the same bits.  All 64 lanes take part.
template <int CTRL> __device__ __forceinline__ float bn_dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
#define BN_DPP_XOR1 0xB1              // quad_perm [1, 0, 3, 2]
#define BN_DPP_XOR2 0x4E              // quad_perm [2, 3, 0, 1]
#define BN_DPP_XOR3 0x1B              // quad_perm [3, 2, 1, 0]
#define BN_DPP_XOR7 0x141             // row_half_mirror
#define BN_DPP_XOR8 0x128             // row_ror:8
// the value of the lane O away (O a power of two below 16)
template <int O> __device__ __forceinline__ float bn_lane_xor(float v) {
    static_assert(O == 1 || O == 2 || O == 4 || O == 8, "inside a row of 16 lanes");
    if constexpr (O == 1) return bn_dpp<BN_DPP_XOR1>(v);
    if constexpr (O == 2) return bn_dpp<BN_DPP_XOR2>(v);
    if constexpr (O == 4) return bn_dpp<BN_DPP_XOR3>(bn_dpp<BN_DPP_XOR7>(v));
    return bn_dpp<BN_DPP_XOR8>(v);
}
// op(v of this lane, v of the lane 32 or 16 away) for an op that does not care which is which
template <int O, typename F> __device__ __forceinline__ float bn_pair_far(float v, F op) {
    static_assert(O == 16 || O == 32, "across rows of 16 lanes");
    const uint32_t b = __builtin_bit_cast(uint32_t, v);
    const auto r = O == 32 ? __builtin_amdgcn_permlane32_swap(b, b, false, false) : __builtin_amdgcn_permlane16_swap(b, b, false, false);
    return op(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
}
template <typename F> __device__ __forceinline__ float bn_wave_reduce(float v, F op) {
    v = bn_pair_far<32>(v, op);
    v = bn_pair_far<16>(v, op);
    v = op(v, bn_lane_xor<8>(v));
    v = op(v, bn_lane_xor<4>(v));
    v = op(v, bn_lane_xor<2>(v));
    return op(v, bn_lane_xor<1>(v));
}
__device__ __forceinline__ float wave_sum(float v) {
    return bn_wave_reduce(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ float wave_max(float v) {
    return bn_wave_reduce(v, [](float a, float b) { return fmaxf(a, b); });
}

// sine and cosine of an angle of any size: the angle less the nearest multiple of 2 pi (2 pi as the sum of two floats, the
// products exact inside the fused operations), then the hardware's functions on what is left, which lies in [-pi, pi]
__device__ __forceinline__ void bn_sincos(float a, float* sn, float* cs) {
    const float k = rintf(a * 0.15915494309189535f);
    float r = fmaf(-k, 6.2831854820251465f, a);
    r = fmaf(-k, -1.7484555e-7f, r);
    *sn = __sinf(r);
    *cs = __cosf(r);
}

// A thread's sum of squares over its groups of four numbers of a row (k: the group's number): one chain, every rounding written
// out, so that kernels which norm the same row form the same bits.
template <typename V> __device__ __forceinline__ float bn_add_squares(float ss, const V& v, int k) {
    ss = k == 0 ? __builtin_fmaf(v.x, v.x, __fmul_rn(v.y, v.y)) : __builtin_fmaf(v.y, v.y, __builtin_fmaf(v.x, v.x, ss));
    return __builtin_fmaf(v.w, v.w, __builtin_fmaf(v.z, v.z, ss));
}

// A barrier that orders shared memory alone: loads and stores of global memory stay in flight across it (__syncthreads waits
// for a row's stores to be acknowledged, a trip to memory).
__device__ __forceinline__ void bn_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Sum over a block of up to 1024 threads; every thread gets the result.
// `scratch` holds at least 16 floats of shared memory.  The order of the additions is
// fixed by the block size alone.  Orders shared memory among the threads, not global memory.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
    const int lane = threadIdx.x & (BN_WAVE - 1), w = threadIdx.x / BN_WAVE;
    const int nw = (blockDim.x + BN_WAVE - 1) / BN_WAVE;
    v = wave_sum(v);
    bn_lds_barrier();
    if (lane == 0) scratch[w] = v;
    bn_lds_barrier();
    float t = 0.f;
    for (int i = 0; i < nw; ++i) t += scratch[i];
    return t;
}
__device__ __forceinline__ float block_max(float v, float* scratch) {
    const int lane = threadIdx.x & (BN_WAVE - 1), w = threadIdx.x / BN_WAVE;
    const int nw = (blockDim.x + BN_WAVE - 1) / BN_WAVE;
    v = wave_max(v);
    bn_lds_barrier();
    if (lane == 0) scratch[w] = v;
    bn_lds_barrier();
    float t = scratch[0];
    for (int i = 1; i < nw; ++i) t = fmaxf(t, scratch[i]);
    return t;
}

// Keys per split of a decode step whose longest sequence holds max_len keys, cut into n_splits runs of whole
// pages: the kernels use it when the length arrives in device memory.  (ops.decode_splits, which makes a plan for a length
// that the host knows, cuts an even number of pages in the same runs while two pages a split are left; an odd one in longer runs.)
__host__ __device__ __forceinline__ int bn_split_chunk(int max_len, int n_splits, int min_pages = BN_SPLIT_MIN_PAGES) {
    const int pages = max_len > 0 ? (max_len + BN_PAGE - 1) / BN_PAGE : 1;
    int per = (pages + n_splits - 1) / n_splits;
    if (per < min_pages) per = min_pages;
    return per * BN_PAGE;
}

// The gate's activation in a gated feed-forward, out = act(gate) * up: the kinds the reference knows
// (src/transformer/cpu_backend.c:343-417).  silu(g) = g / (1 + exp(-g)) with the exact exponential (:356);
// gelu in its tanh form 0.5 g (1 + tanh(0.79788456 g (1 + 0.044715 g^2))) (:27-29; the reference's function also
// returns 0 below -10 and g above 10 and rounds g and the result to half precision, :20-30, which this one does not:
// it is no activation of the architecture built here, and its parity with the reference is not pinned by a test);
// relu2(g) = max(g, 0)^2 (:349-350).  Every kernel that ends in a gated unit takes the kind as an argument.
#define BN_ACT_SILU 0
#define BN_ACT_GELU_TANH 1
#define BN_ACT_RELU2 2
#define BN_ACT_KINDS 3
__device__ __forceinline__ float bn_gate_act(float g, int act) {
    if (act == BN_ACT_SILU) return g / (1.0f + expf(-g));
    if (act == BN_ACT_GELU_TANH) return 0.5f * g * (1.0f + tanhf(0.7978845608028654f * g * (1.0f + 0.044715f * g * g)));
    const float p = fmaxf(g, 0.f);
    return p * p;
}

// Activations of one argument (a feed-forward without a gate; the inner layer of a low-rank projection).
// The Python side reads these lines.
#define BN_UNARY_GELU_ERF 0      // 0.5 z (1 + erf(z / sqrt 2))
#define BN_UNARY_GELU_TANH 1     // the tanh form, as bn_gate_act's
#define BN_UNARY_SILU 2
#define BN_UNARY_RELU2 3
#define BN_UNARY_TANH 4
#define BN_UNARY_SIGMOID 5
#define BN_UNARY_KINDS 6
__device__ __forceinline__ float bn_unary_act(float z, int kind) {
    switch (kind) {
        case BN_UNARY_GELU_ERF: return 0.5f * z * (1.0f + erff(z * 0.7071067811865476f));
        case BN_UNARY_GELU_TANH: return bn_gate_act(z, BN_ACT_GELU_TANH);
        case BN_UNARY_SILU: return bn_gate_act(z, BN_ACT_SILU);
        case BN_UNARY_RELU2: return bn_gate_act(z, BN_ACT_RELU2);
        case BN_UNARY_TANH: return tanhf(z);
        default: return 1.0f / (1.0f + expf(-z));
    }
}

static inline int bn_launch_status() { return (int)hipGetLastError(); }
