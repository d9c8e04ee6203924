// Mixers that carry a state of fixed size from token to token instead of keys and values: the kernels of their
// recurrences, for prompt and decode steps alike.  Every state lives in float32 in the cache's state area, a row per
// sequence slot; a kernel finds a sequence's row through the step's device-side slot ids and its tokens either through
// a list of tiles (one tile a sequence: sequence, first row, rows, position of the first; a tile of no rows is skipped)
// or, tiles == null, as row b = the one new token of sequence b (seq_lens[b] == 0: a padding row, nothing is touched).
// Everything that enters a recurrence is float32: decays, gates, exponentials, the state; the projections that feed
// them arrive in the activations' type.  The order of every sum is a function of the sizes alone.
//
//   token shift   mix_s[t] = h[t] + (h[t-1] - h[t]) * mu_s; h[-1] of a step is the state's copy of the last h, 0 at position 0
//   wkv           o_t = (S + diag(u) k_t v_t^T)^T r_t;  S <- diag(w_t) S + k_t v_t^T;  w_t = exp(-exp(d_t + w0))   per head
//   head norm     y = o / sqrt(mean_head(o^2) + eps) * weight * silu(gate)
//   min-GRU       z = sigmoid(a + bz); c = b + bx; cand = c >= 0 ? c + 1/2 : sigmoid(c); S <- (1 - z) S + z cand; y = S silu(g)
#include "common.h"
#include <math.h>

struct SeqRange { int seq, row0, n, pos0; };

// A barrier of the workgroup that orders its shared memory only.  __syncthreads() also waits for everything that the wave
// has asked from or sent to global memory; this one leaves loads and stores in flight (whoever needs a load's data waits
// for it there), which is what lets a kernel ask for its next tokens before it walks the current ones.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

__device__ __forceinline__ SeqRange seq_range(const int* tiles, const int* seq_lens, int idx) {
    SeqRange r;
    if (tiles) {
        const int* t = tiles + 4 * idx;
        r.seq = t[0]; r.row0 = t[1]; r.n = t[2]; r.pos0 = t[3];
    } else {
        r.seq = idx; r.row0 = idx; r.pos0 = seq_lens[idx] - 1; r.n = r.pos0 >= 0 ? 1 : 0;
    }
    return r;
}

// A step's sequences cut into pieces of `piece` tokens, numbered through sequence after sequence: the first piece of sequence
// `upto`, counting no more sequences than n_tiles.
__device__ __forceinline__ int pieces_before(const int* tiles, int upto, int piece) {
    int n = 0;
    for (int i = 0; i < upto; ++i) n += (max(tiles[4 * i + 2], 0) + piece - 1) / piece;
    return n;
}

// Piece number `at` as a range of its own; n = 0 behind the last one.  last: it is its sequence's last piece.
__device__ __forceinline__ SeqRange piece_range(const int* tiles, int n_tiles, int at, int piece, bool& last) {
    SeqRange r = {0, 0, 0, -1};
    last = false;
    for (int i = 0; i < n_tiles; ++i) {
        const int n = tiles[4 * i + 2], count = (max(n, 0) + piece - 1) / piece;
        if (at < count) {
            r = seq_range(tiles, nullptr, i);
            r.row0 += at * piece;
            r.n = min(piece, n - at * piece);
            last = at == count - 1;
            return r;
        }
        at -= count;
    }
    return r;
}

// ---- token shift ----------------------------------------------------------------------------------------------------
// out[s, t, :] for s < n_mix.  The previous row of the flattened batch is the previous token when it belongs to the same
// sequence; else the sequence's state holds it (zero at position 0).  seq_lens null: the state is read only, and the
// recurrence's kernel stores the step's last h afterwards, when every reader is done.  Else (seq_lens: the sequences'
// lengths behind the step) the workgroup of a sequence's first row, the only reader of the sequence's state, stores the
// step's last row there, each thread the elements that it has read.  TI: the type of h; TO: of the mixes.
template <typename TI, typename TO>
__global__ void token_shift_kernel(TO* __restrict__ out, const TI* __restrict__ h, const float* __restrict__ mu,
                                   float* state, size_t state_stride, const int* __restrict__ positions,
                                   const int* __restrict__ seq_index, const int* __restrict__ slot_ids,
                                   const int* __restrict__ seq_lens, int T_rows, int D, int n_mix) {
    const int t = blockIdx.x;
    const int pos = positions[t], seq = seq_index[t];
    const int before = t > 0 ? t - 1 : 0;
    const int pos_b = positions[before], seq_b = seq_index[before], slot = slot_ids[seq];     // all asked for together
    const TI* cur = h + (size_t)t * D;
    const bool inside = t > 0 && pos > 0 && seq_b == seq && pos_b == pos - 1;
    // both candidates for the previous row are loaded, from places that exist, and one is chosen: a load under a
    // branch would be waited for where it stands, element after element
    const TI* prev_row = h + (size_t)(inside ? t - 1 : t) * D;
    float* prev_state = state + (size_t)slot * state_stride;
    const bool keeps = seq_lens && pos >= 0 && !inside;           // the first row of its sequence in this step
    const int last = keeps ? min(t + max(seq_lens[seq] - 1 - pos, 0), T_rows - 1) : t;
    const TI* last_row = h + (size_t)last * D;
#pragma unroll 4
    for (int e = threadIdx.x; e < D; e += blockDim.x) {
        const float c = to_f32(cur[e]);
        const float pr = to_f32(prev_row[e]), ps = prev_state[e];
        const float p = inside ? pr : (pos > 0 ? ps : 0.f);
        const float d = p - c;
        for (int s = 0; s < n_mix; ++s)
            out[((size_t)s * T_rows + t) * D + e] = from_f32<TO>(pos >= 0 ? fmaf(d, mu[(size_t)s * D + e], c) : 0.f);
        if (keeps) prev_state[e] = to_f32(last_row[e]);
    }
}

// The same for one mix of a float32 stream, four elements a thread (D a multiple of 4, everything 16-byte aligned): what a
// block that mixes its stream with the previous token's runs over a whole prompt step.
template <typename TO>
__global__ __launch_bounds__(256) void token_shift_stream_kernel(TO* __restrict__ out, const float* __restrict__ x,
                                                                 const float* __restrict__ mu, float* state, size_t state_stride,
                                                                 const int* __restrict__ positions, const int* __restrict__ seq_index,
                                                                 const int* __restrict__ slot_ids, const int* __restrict__ seq_lens,
                                                                 int T_rows, int D) {
    const int t = blockIdx.x;
    const int pos = positions[t], seq = seq_index[t];
    const int before = t > 0 ? t - 1 : 0;
    const int pos_b = positions[before], seq_b = seq_index[before], slot = slot_ids[seq];
    const bool inside = t > 0 && pos > 0 && seq_b == seq && pos_b == pos - 1;
    float* st = state + (size_t)slot * state_stride;
    const float* cur = x + (size_t)t * D;
    const float* prev = inside ? cur - D : st;                    // one load for either candidate
    const bool has_prev = pos > 0, keeps = pos >= 0 && !inside;
    const int last = keeps ? min(t + max(seq_lens[seq] - 1 - pos, 0), T_rows - 1) : t;
    const float* last_row = x + (size_t)last * D;
    TO* o = out + (size_t)t * D;
    for (int e = threadIdx.x * 4; e < D; e += 1024) {
        const float4 c = *reinterpret_cast<const float4*>(cur + e), m = *reinterpret_cast<const float4*>(mu + e);
        float4 p = *reinterpret_cast<const float4*>(prev + e);
        if (!has_prev) p = make_float4(0.f, 0.f, 0.f, 0.f);
        float4 r;
        r.x = fmaf(p.x - c.x, m.x, c.x); r.y = fmaf(p.y - c.y, m.y, c.y);
        r.z = fmaf(p.z - c.z, m.z, c.z); r.w = fmaf(p.w - c.w, m.w, c.w);
        if (pos < 0) r = make_float4(0.f, 0.f, 0.f, 0.f);
        if (sizeof(TO) == 2) {
            bf16 b[4] = {from_f32<bf16>(r.x), from_f32<bf16>(r.y), from_f32<bf16>(r.z), from_f32<bf16>(r.w)};
            *reinterpret_cast<uint2*>(o + e) = *reinterpret_cast<const uint2*>(b);
        } else {
            *reinterpret_cast<float4*>(o + e) = r;
        }
        if (keeps) *reinterpret_cast<float4*>(st + e) = *reinterpret_cast<const float4*>(last_row + e);
    }
}

// The mixes of a bf16 or float32 input in 16-byte groups of h (D a multiple of 8, everything 16-byte aligned); the state is read
// only.  Four rows a workgroup in large steps, so that a mix's weights are read once for them.  2,048
// rows x 2,048 columns, five bf16 mixes: 50 MB, 12.7 us (285 with an element a thread and 2-byte stores); one row 3.3 us in a graph of such
// launches (4.4), 6.3 in a decode step's profile.
template <typename T, int TS_ROWS>
__global__ __launch_bounds__(256) void token_shift_wide_kernel(T* __restrict__ out, const T* __restrict__ h, const float* __restrict__ mu,
                                                               const float* __restrict__ state, size_t state_stride,
                                                               const int* __restrict__ positions, const int* __restrict__ seq_index,
                                                               const int* __restrict__ slot_ids, int T_rows, int D, int n_mix) {
    constexpr int EPV = 16 / (int)sizeof(T);
    struct __align__(16) Group { T e[EPV]; };
    const int t0 = blockIdx.x * TS_ROWS, e = (blockIdx.y * 256 + threadIdx.x) * EPV;
    if (e >= D) return;
    float c[TS_ROWS][EPV], d[TS_ROWS][EPV];
    bool any[TS_ROWS];
#pragma unroll
    for (int r = 0; r < TS_ROWS; ++r) {
        const int t = min(t0 + r, T_rows - 1), before = t > 0 ? t - 1 : 0;
        const int pos = positions[t], seq = seq_index[t];
        const bool inside = t > 0 && pos > 0 && seq_index[before] == seq && positions[before] == pos - 1;
        const Group cg = *reinterpret_cast<const Group*>(h + (size_t)t * D + e);
        const Group pg = *reinterpret_cast<const Group*>(h + (size_t)(inside ? t - 1 : t) * D + e);
        const float* ps = state + (size_t)slot_ids[seq] * state_stride + e;      // both candidates are asked for
        float st[EPV];
#pragma unroll
        for (int q = 0; q < EPV; q += 4) *reinterpret_cast<float4*>(st + q) = *reinterpret_cast<const float4*>(ps + q);
        any[r] = pos >= 0;
#pragma unroll
        for (int q = 0; q < EPV; ++q) {
            c[r][q] = to_f32(cg.e[q]);
            d[r][q] = (inside ? to_f32(pg.e[q]) : pos > 0 ? st[q] : 0.f) - c[r][q];
        }
    }
    for (int s = 0; s < n_mix; ++s) {
        float m[EPV];
#pragma unroll
        for (int q = 0; q < EPV; q += 4) *reinterpret_cast<float4*>(m + q) = *reinterpret_cast<const float4*>(mu + (size_t)s * D + e + q);
#pragma unroll
        for (int r = 0; r < TS_ROWS; ++r) {
            if (t0 + r >= T_rows) break;
            Group o;
#pragma unroll
            for (int q = 0; q < EPV; ++q) o.e[q] = from_f32<T>(any[r] ? fmaf(d[r][q], m[q], c[r][q]) : 0.f);
            *reinterpret_cast<Group*>(out + ((size_t)s * T_rows + t0 + r) * D + e) = o;
        }
    }
}

template <typename T>
static void launch_token_shift_wide(T* out, const T* h, const float* mu, const float* state, size_t st, const int* positions,
                                    const int* seq_index, const int* slot_ids, int n_tokens, int D, int n_mix, hipStream_t s) {
    const unsigned y = (unsigned)(D * (int)sizeof(T) / 16 + 255) / 256;
    // Four rows of a workgroup share a mix's weights, which pays once the rows no longer fit what is on its way at a time: us with four /
    // one, bf16, 1,024 x 1,024 6.9 / 5.6, 1,500 x 2,048 11.4 / 11.0, 4,000 x 768 11.1 / 12.4, 2,048 x 2,048 12.7 / 13.2, 4,000 x 4,096 36 /
    // 38; float32 1,024 x 1,024 7.1 / 6.4, 1,024 x 2,048 11.5 / 12.1.
    if ((long long)n_tokens * D * (int)sizeof(T) >= 6000000)
        hipLaunchKernelGGL((token_shift_wide_kernel<T, 4>), dim3((n_tokens + 3) / 4, y), dim3(256), 0, s, out, h, mu, state, st, positions,
                           seq_index, slot_ids, n_tokens, D, n_mix);
    else
        hipLaunchKernelGGL((token_shift_wide_kernel<T, 1>), dim3(n_tokens, y), dim3(256), 0, s, out, h, mu, state, st, positions, seq_index,
                           slot_ids, n_tokens, D, n_mix);
}

// in_dtype: of h; dtype: of the mixes (in_dtype equal to it, or float32).  seq_lens: see above.
extern "C" int bn_token_shift(int in_dtype, int dtype, void* out, const void* h, const float* mu, float* state,
                              long long state_stride, const int* positions, const int* seq_index, const int* slot_ids,
                              const int* seq_lens, int n_tokens, int D, int n_mix, hipStream_t s) {
    if (n_tokens <= 0 || D <= 0 || n_mix <= 0 || !out || !h || !mu || !state || !positions || !seq_index || !slot_ids)
        return BN_ERR_ARG;
    if ((dtype != BN_DT_F32 && dtype != BN_DT_BF16) || (in_dtype != dtype && in_dtype != BN_DT_F32)) return BN_ERR_DTYPE;
    const dim3 grid(n_tokens), block(256);
    const size_t st = (size_t)state_stride;
    // (narrower rows leave most threads of a workgroup of groups idle: us at 64 rows in bf16, wide / not, 256 columns 3.1 / 2.7, 512
    // 3.1 / 3.4; at 1,100 rows of 64 6.6 / 3.1)
    if (in_dtype == dtype && !seq_lens && D >= 512 && D % 8 == 0 && st % 4 == 0 &&
        !(((uintptr_t)out | (uintptr_t)h | (uintptr_t)mu | (uintptr_t)state) & 15)) {
        if (dtype == BN_DT_F32)
            launch_token_shift_wide((float*)out, (const float*)h, mu, state, st, positions, seq_index, slot_ids, n_tokens, D, n_mix, s);
        else
            launch_token_shift_wide((bf16*)out, (const bf16*)h, mu, state, st, positions, seq_index, slot_ids, n_tokens, D, n_mix, s);
    } else if (in_dtype == BN_DT_F32 && seq_lens && n_mix == 1 && D % 4 == 0 && st % 4 == 0 &&
        !(((uintptr_t)out | (uintptr_t)h | (uintptr_t)mu | (uintptr_t)state) & 15)) {
        if (dtype == BN_DT_F32)
            hipLaunchKernelGGL(token_shift_stream_kernel<float>, grid, block, 0, s, (float*)out, (const float*)h, mu, state, st,
                               positions, seq_index, slot_ids, seq_lens, n_tokens, D);
        else
            hipLaunchKernelGGL(token_shift_stream_kernel<bf16>, grid, block, 0, s, (bf16*)out, (const float*)h, mu, state, st,
                               positions, seq_index, slot_ids, seq_lens, n_tokens, D);
    } else if (in_dtype == BN_DT_F32 && dtype == BN_DT_F32)
        hipLaunchKernelGGL((token_shift_kernel<float, float>), grid, block, 0, s, (float*)out, (const float*)h, mu, state, st,
                           positions, seq_index, slot_ids, seq_lens, n_tokens, D, n_mix);
    else if (in_dtype == BN_DT_F32)
        hipLaunchKernelGGL((token_shift_kernel<float, bf16>), grid, block, 0, s, (bf16*)out, (const float*)h, mu, state, st,
                           positions, seq_index, slot_ids, seq_lens, n_tokens, D, n_mix);
    else
        hipLaunchKernelGGL((token_shift_kernel<bf16, bf16>), grid, block, 0, s, (bf16*)out, (const bf16*)h, mu, state, st,
                           positions, seq_index, slot_ids, seq_lens, n_tokens, D, n_mix);
    return bn_launch_status();
}

// ---- the wkv recurrence -----------------------------------------------------------------------------------------------
// A workgroup owns (sequence, head, a block of CB value columns).  Column j of a head's state S[dk, dv] depends on no
// other column, so the columns are spread over threads and workgroups freely (the host picks CB so that a launch fills
// the chip); the dk rows of a column are spread over P threads (P a power of two <= 16, neighbouring lanes), each holding
// WKV_KR consecutive rows in registers, rows p WKV_KR .. p WKV_KR + WKV_KR - 1.  The tokens of a sequence come in chunks
// of TC: r, k, the decay and the block's v are staged in shared memory once a chunk (rows beyond dk zero, which leaves the
// unused registers zero) by waves of the workgroup that do nothing else: while the walking waves run a chunk's tokens
// without a barrier, every thread reading its rows 16 bytes at a time, the staging waves fill the other buffer with the
// next chunk, exponentials of the decay included, so the walk never waits for memory.  A column's sum over the rows is formed in four
// partial sums per thread and a butterfly over the P threads: an order that depends on the head size alone.
#define WKV_KR 16
#define WKV_MAX_DIM 256
#define WKV_MAX_THREADS 256

struct WkvArgs {
    const void* r; const void* k; const void* v; const void* d;     // [T, ld*]: head h at h * dk (v: h * dv)
    int ldr, ldk, ldv, ldd;
    const float* w0;          // [H * dk] added to d before the exponentials
    const float* u;           // [H * dk] the bonus of the current token
    float* o;                 // [T, H * dv] float32
    const void* h;            // [T, D]: the mixer's input, whose last row of every sequence becomes the state's copy
    float* state;             // [slots, state_stride]: S per head in the walkers' order (wkv_state_at), then D values of the last h
    size_t state_stride;
    const int* tiles; const int* seq_lens; const int* slot_ids;
    int H, dk, dv, D, P, CB, TC, walkers;
    int n_tiles;              // (the piece forms)
    float* carry;             // [pieces, H dkp dv]: a piece's own sum, then what the piece starts from
    float* fade;              // [pieces, H dkp]: the product of a piece's decays
    const bf16* low;          // (the step in bf16) [T, ldlow], w2 [H * dk, rank]: d is low . w2^T, formed here (d null)
    const bf16* w2;
    int ldlow, rank;
};

// How a workgroup of the recurrence meets its sequence: the whole of it (WKV_WALK), or, where a step offers too few sequences
// and heads to fill the chip, one piece of WKV_PIECE tokens: every piece's own sum from nothing and the product of its decays
// (WKV_SUMS), a pass that carries the state through the pieces (wkv_carry_kernel), every piece again from its start with
// outputs (WKV_OUTPUTS).  The recurrence is linear in S, so this is the same sum in another order of rounding: not for callers
// whose float32 bits must not depend on how a sequence was cut into steps.
#define WKV_PIECE 64
enum { WKV_WALK = 0, WKV_SUMS = 1, WKV_OUTPUTS = 2 };

// The sum over the P neighbouring lanes that share a column, every lane getting it: a butterfly whose steps of 1 and
// 2 lanes are exchanges inside a group of four and whose steps of 4 and 8 lanes are mirrors of 8 and 16 lanes (after the
// first two steps a group of four holds one value, so a mirror meets the same partner group as an exchange would).
// Data-parallel moves inside a row of 16 lanes: no trip through shared memory.
__device__ __forceinline__ float wkv_lane_sum(float v, int P) {
    if (P >= 2) v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true));     // lanes 1 0 3 2
    if (P >= 4) v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, true));     // lanes 2 3 0 1
    if (P >= 8) v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, true));    // mirror of 8
    if (P >= 16) v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xF, 0xF, true));   // mirror of 16
    return v;
}

// One token of one column: o = sum_i r_i (S_i + u_i k_i v), then S_i <- w_i S_i + k_i v, over this thread's rows; the
// sum in four partial sums and the lanes' butterfly.
__device__ __forceinline__ float wkv_token(const float4 (&r4)[WKV_KR / 4], const float4 (&k4)[WKV_KR / 4],
                                           const float4 (&w4)[WKV_KR / 4], float vj, const float (&ub)[WKV_KR],
                                           float (&S)[WKV_KR], int P) {
    float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q4 = 0; q4 < WKV_KR / 4; ++q4) {
        const float rv[4] = {r4[q4].x, r4[q4].y, r4[q4].z, r4[q4].w}, kv4[4] = {k4[q4].x, k4[q4].y, k4[q4].z, k4[q4].w},
                    wv[4] = {w4[q4].x, w4[q4].y, w4[q4].z, w4[q4].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int ii = q4 * 4 + e;
            const float kv = kv4[e] * vj;
            part[e] = fmaf(rv[e], fmaf(ub[ii], kv, S[ii]), part[e]);
            S[ii] = fmaf(wv[e], S[ii], kv);
        }
    }
    return wkv_lane_sum((part[0] + part[1]) + (part[2] + part[3]), P);
}

template <typename T, int FORM>
__global__ __launch_bounds__(WKV_MAX_THREADS + 128) void wkv_scan_kernel(WkvArgs a) {
    extern __shared__ __align__(16) float smem[];
    bool last_piece = true;
    const SeqRange sr = FORM == WKV_WALK ? seq_range(a.tiles, a.seq_lens, blockIdx.x)
                                         : piece_range(a.tiles, a.n_tiles, blockIdx.x, WKV_PIECE, last_piece);
    if (sr.n <= 0 || sr.pos0 < 0) return;
    const int head = blockIdx.y, cb = blockIdx.z;
    const int P = a.P, dk = a.dk, dv = a.dv, TC = a.TC, CB = a.CB;
    const int dkp = P * WKV_KR;                           // staged rows, zero beyond dk
    const int tid = threadIdx.x, nthreads = blockDim.x;
    const int n_walk = a.walkers;                         // the first n_walk threads walk the tokens, the rest stage them
    const bool walker = tid < n_walk;
    const int p = tid % P, jl = tid / P;
    const int j = cb * CB + jl;                           // a walker's value column
    const bool owns = walker && jl < CB && j < dv;
    const int buf_floats = TC * (3 * dkp + CB);           // one staged chunk: r, k, w as [TC][dkp], then v as [TC][CB]

    // A head's state lies in the order in which the walkers hold it: element (row p WKV_KR + ii, column j) at
    // (ii dv + j) P + p, so that the lanes of a wave, p fastest and then the columns, read and write runs of memory.
    float* S_g = (FORM == WKV_WALK ? a.state + (size_t)a.slot_ids[sr.seq] * a.state_stride : a.carry + (size_t)blockIdx.x * a.H * dkp * dv) +
                 (size_t)head * dkp * dv;
    const bool starts = FORM == WKV_OUTPUTS || (FORM == WKV_WALK && sr.pos0 > 0);
    float S[WKV_KR], ub[WKV_KR], fade[WKV_KR];
#pragma unroll
    for (int ii = 0; ii < WKV_KR; ++ii) {
        const int i = p * WKV_KR + ii;
        S[ii] = (owns && starts) ? S_g[((size_t)ii * dv + j) * P + p] : 0.f;        // rows beyond dk hold zeros
        ub[ii] = (FORM != WKV_SUMS && owns && i < dk) ? a.u[(size_t)head * dk + i] : 0.f;
        fade[ii] = 1.f;
    }

    // the staging threads' work: chunk c0 into buffer b
    auto stage = [&](int c0, int b) {
        float* r_s = smem + (size_t)b * buf_floats;
        float* k_s = r_s + TC * dkp;
        float* w_s = k_s + TC * dkp;
        float* v_s = w_s + TC * dkp;
        const int nc = min(TC, sr.n - c0), lt = tid - n_walk, nl = nthreads - n_walk;
        // eight elements a turn, their loads asked for together (unconditional loads from clamped places: a load
        // under a branch would make the compiler wait for each before the next)
        const int total = nc * dkp;
        for (int base = lt; base < total; base += 8 * nl) {
            float rv[8], kv[8], dv4[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int idx = min(base + q * nl, total - 1);
                const int tt = idx / dkp, i = min(idx - tt * dkp, dk - 1);
                const size_t row = (size_t)(sr.row0 + c0 + tt), c = (size_t)head * dk + i;
                rv[q] = to_f32(reinterpret_cast<const T*>(a.r)[row * a.ldr + c]);
                kv[q] = to_f32(reinterpret_cast<const T*>(a.k)[row * a.ldk + c]);
                dv4[q] = to_f32(reinterpret_cast<const T*>(a.d)[row * a.ldd + c]) + a.w0[c];
            }
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int idx = base + q * nl;
                if (idx < total) {
                    const bool in = idx % dkp < dk;
                    r_s[idx] = in ? rv[q] : 0.f;
                    k_s[idx] = in ? kv[q] : 0.f;
                    w_s[idx] = in ? expf(-expf(dv4[q])) : 0.f;
                }
            }
        }
        const int total_v = nc * CB;
        for (int base = lt; base < total_v; base += 4 * nl) {
            float vv[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int idx = min(base + q * nl, total_v - 1);
                const int tt = idx / CB, col = min(cb * CB + (idx - tt * CB), dv - 1);
                vv[q] = to_f32(reinterpret_cast<const T*>(a.v)[(size_t)(sr.row0 + c0 + tt) * a.ldv + (size_t)head * dv + col]);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int idx = base + q * nl;
                if (idx < total_v) v_s[idx] = cb * CB + idx % CB < dv ? vv[q] : 0.f;
            }
        }
    };

    if (!walker) stage(0, 0);
    lds_barrier();
    int b = 0;
    for (int c0 = 0; c0 < sr.n; c0 += TC, b ^= 1) {
        const int nc = min(TC, sr.n - c0);
        if (!walker) {
            if (c0 + TC < sr.n) stage(c0 + TC, b ^ 1);
        } else if (jl < CB) {
            const float* r_s = smem + (size_t)b * buf_floats;
            const float* k_s = r_s + TC * dkp;
            const float* w_s = k_s + TC * dkp;
            const float* v_s = w_s + TC * dkp;
            // two tokens a turn: both tokens' rows are asked for before the first is used, so the second's way from
            // shared memory is covered by the first's arithmetic
            for (int tt = 0; tt < nc; tt += FORM == WKV_SUMS ? 1 : 2) {
                const bool two = tt + 1 < nc;
                const int t1 = two ? tt + 1 : tt;
                float4 ra[WKV_KR / 4], ka[WKV_KR / 4], wa[WKV_KR / 4], rb[WKV_KR / 4], kb[WKV_KR / 4], wb[WKV_KR / 4];
#pragma unroll
                for (int q4 = 0; q4 < WKV_KR / 4; ++q4) {
                    ra[q4] = reinterpret_cast<const float4*>(r_s + tt * dkp + p * WKV_KR)[q4];
                    ka[q4] = reinterpret_cast<const float4*>(k_s + tt * dkp + p * WKV_KR)[q4];
                    wa[q4] = reinterpret_cast<const float4*>(w_s + tt * dkp + p * WKV_KR)[q4];
                }
                if (FORM == WKV_SUMS) {                   // no outputs: S and the decays' product alone, one token a turn
#pragma unroll
                    for (int ii = 0; ii < WKV_KR; ++ii) {
                        const float ke = reinterpret_cast<const float*>(ka)[ii], we = reinterpret_cast<const float*>(wa)[ii];
                        S[ii] = fmaf(we, S[ii], ke * v_s[tt * CB + jl]);
                        fade[ii] *= we;
                    }
                    continue;
                }
                const float va = v_s[tt * CB + jl];
#pragma unroll
                for (int q4 = 0; q4 < WKV_KR / 4; ++q4) {
                    rb[q4] = reinterpret_cast<const float4*>(r_s + t1 * dkp + p * WKV_KR)[q4];
                    kb[q4] = reinterpret_cast<const float4*>(k_s + t1 * dkp + p * WKV_KR)[q4];
                    wb[q4] = reinterpret_cast<const float4*>(w_s + t1 * dkp + p * WKV_KR)[q4];
                }
                const float vb = v_s[t1 * CB + jl];
                const float acc_a = wkv_token(ra, ka, wa, va, ub, S, P);
                if (p == 0 && owns) a.o[(size_t)(sr.row0 + c0 + tt) * (a.H * dv) + (size_t)head * dv + j] = acc_a;
                if (two) {
                    const float acc_b = wkv_token(rb, kb, wb, vb, ub, S, P);
                    if (p == 0 && owns) a.o[(size_t)(sr.row0 + c0 + t1) * (a.H * dv) + (size_t)head * dv + j] = acc_b;
                }
            }
        }
        lds_barrier();                                    // the chunk has been walked and the next one is staged
    }
    if (FORM != WKV_OUTPUTS) {
#pragma unroll
        for (int ii = 0; ii < WKV_KR; ++ii)
            if (owns) S_g[((size_t)ii * dv + j) * P + p] = S[ii];
    }
    if (FORM == WKV_SUMS) {
        if (owns && jl == 0 && cb == 0) {
            float* f = a.fade + ((size_t)blockIdx.x * a.H + head) * dkp + p * WKV_KR;
#pragma unroll
            for (int ii = 0; ii < WKV_KR; ++ii) f[ii] = fade[ii];
        }
        return;
    }
    if (head == 0 && cb == 0 && last_piece) {             // the step's last h of this sequence, for the next step's shift
        float* hp = a.state + (size_t)a.slot_ids[sr.seq] * a.state_stride + (size_t)a.H * dkp * dv;
        const T* last = reinterpret_cast<const T*>(a.h) + (size_t)(sr.row0 + sr.n - 1) * a.D;
        for (int e = tid; e < a.D; e += nthreads) hp[e] = to_f32(last[e]);
    }
}

// The same recurrence of a bf16 step sixteen tokens at a time on the matrix cores, all numbers float32 (v_mfma_f32_16x16x4f32).
// Over a block of sixteen tokens, W[a, b) the product of the decays of tokens a .. b - 1 in every row i of a head's state:
//     o_t = (r_t W[0, t)) S + sum over s < t of A[t, s] v_s + (sum over i of r_t u k_t) v_t,   A[t, s] = sum over i of r_t W[s + 1, t) k_s
//     S   <- W[0, 16) S + sum over s of (k_s W[s + 1, 16)) v_s^T
// A product of decays exp(-exp(d + w0)) is 2^-(the sum of their rates exp(d + w0) log2 e): one rounding of a number below 1 instead of one a token.
// It is never a quotient: for a pair s < t whose numbers differ first in bit l, the tokens between them split at the token b where t's half of
// that block of 2^(l + 1) begins, W[s + 1, t) = W[s + 1, b) W[b, t), so that A is four matrix products, one a bit, of r_t W[b, t) with
// k_s W[s + 1, b), of which each element is taken from its own pair's bit.  The running sums of rates come from exchanges between the sixteen
// lanes of a row (lane c holds token c).
// A wave owns sixteen rows of the head where it forms A (its share of the sum over i meets the others' in shared memory) and sixteen
// columns of S and o; element (row p 16 + ii, column j) of S lies in register p % 4 of tile p / 4 * 4 + ii / 4, lane (ii % 4, j), which is
// the operand of r S as it stands and sixteen bytes of the state in the walkers' order.  The next two blocks' numbers are asked for
// before this one's are used; one barrier a block.
// A wave's block is some 400 vector instructions, most of them the running sums, the exponentials and what meets them, and 52 matrix
// instructions of 32 cycles, where the walk reads 3 KB of shared memory a wave in every token: a long walk of one sequence is bound by the latency of a
// block (2.3 us, 4.8 in the walk), the pieces by the vector and the matrix units (12 us each of their 33) and by how fast a launch's workgroups
// start.  us, walk -> this, 32 heads of 64 x 64: one sequence of 128 tokens 47 -> 21, 2,048 617 -> 289, in pieces 197 -> 64 (sums 65 -> 19, outputs 95 ->
// 34); sixteen of 512 341 -> 119; 16 heads of 128 x 128: one of 2,048 in pieces 426 -> 88, eight of 512 391 -> 146.  (Pieces of 128 tokens: 73 for one
// sequence of 2,048.)  Error against 64 bits, 2,048 tokens in pieces, walk -> this, by w0 about: -9 6.1e-6 -> 2.5e-7, -6 2.7e-6 -> 2.3e-7, -2 1.5e-7 ->
// 1.3e-7, 0 7.8e-8 -> 8.6e-8 (half a unit in the last place).
#define WKV_BLOCK 16
typedef float wkv_f4 __attribute__((ext_vector_type(4)));

// partner: 2^l lanes away in a row of sixteen, for a value that is the same in every block of 2^l lanes
template <int L> __device__ __forceinline__ float wkv_partner(float v) {
    constexpr int how = L == 0 ? 0xB1 : L == 1 ? 0x4E : L == 2 ? 0x141 : 0x140;
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), how, 0xF, 0xF, true));
}

// A product's result that is next read behind a branch is named here, in front of it: with a short branch between the two, an earlier form of this kernel
// compiled (ROCm 7.2) to a read of the result's last register before it was written.  In the kernels as they are compiled now, on every path, at least the
// 10 wait states that a read behind v_mfma_f32_16x16x4_f32 needs lie in between.
__device__ __forceinline__ void wkv_settle(wkv_f4& x) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float v = x[e];
        asm("" : "+v"(v));
        x[e] = v;
    }
}

template <int P> __device__ __forceinline__ wkv_f4 wkv_shares(const float* at, int apart) {       // the sum of the waves' shares, pair by pair
    if constexpr (P == 1) return *reinterpret_cast<const wkv_f4*>(at);
    else return wkv_shares<P / 2>(at, apart) + wkv_shares<P / 2>(at + P / 2 * apart, apart);
}

__device__ __forceinline__ float wkv_decay(float sum) { return __builtin_amdgcn_exp2f(-sum); }

template <int P, int FORM>
__global__ __launch_bounds__(P * 64, FORM == WKV_WALK ? 2 : 4) void wkv_blocks_kernel(WkvArgs a) {
    constexpr int DKP = P * WKV_KR, ROW = DKP + 4, AROW = WKV_BLOCK + 4;
    __shared__ __align__(16) float r_s[2][WKV_BLOCK * ROW], k_s[2][WKV_BLOCK * ROW], a_s[2][P * WKV_BLOCK * AROW], t_s[2][DKP], own_s[2][P * WKV_BLOCK];
    bool last_piece = true;
    const SeqRange sr = FORM == WKV_WALK ? seq_range(a.tiles, a.seq_lens, blockIdx.x)
                                         : piece_range(a.tiles, a.n_tiles, blockIdx.x, WKV_PIECE, last_piece);
    if (sr.n <= 0 || sr.pos0 < 0) return;
    const int head = blockIdx.y, dk = a.dk, dv = a.dv;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    const int j = w * 16 + c;                             // the lane's column of S and o
    const bool owns = j < dv;
    const int i0 = w * 16 + g * 4;                        // its four rows of r, k and the decay, of token c
    const bool in = i0 < dk;                              // (dk is a multiple of 4)
    const size_t col = (size_t)head * dk + min(i0, dk - 4);

    float* S_g = (FORM == WKV_WALK ? a.state + (size_t)a.slot_ids[sr.seq] * a.state_stride : a.carry + (size_t)blockIdx.x * a.H * DKP * dv) +
                 (size_t)head * DKP * dv;
    const bool starts = FORM == WKV_OUTPUTS || (FORM == WKV_WALK && sr.pos0 > 0);
    wkv_f4 S[P];
#pragma unroll
    for (int m = 0; m < P; ++m)
        S[m] = owns && starts ? *reinterpret_cast<const wkv_f4*>(S_g + ((size_t)((m % 4) * 4 + g) * dv + j) * P + m / 4 * 4) : (wkv_f4)(0.f);
    const float4 off4 = *reinterpret_cast<const float4*>(a.w0 + col), u4 = *reinterpret_cast<const float4*>(a.u + col);
    const float off[4] = {off4.x, off4.y, off4.z, off4.w}, bonus[4] = {u4.x, u4.y, u4.z, u4.w};
    float fade[4] = {0.f, 0.f, 0.f, 0.f};                 // as T below

    struct __align__(8) Four { bf16 e[4]; };
    struct Numbers { Four r, k, d; bf16 v[4]; };
    constexpr int AHEAD = 2;
    Numbers num[AHEAD];
    const bf16* r_g = reinterpret_cast<const bf16*>(a.r) + (size_t)sr.row0 * a.ldr + (size_t)head * dk;      // uniform; a lane's place from there in 32 bits
    const bf16* k_g = reinterpret_cast<const bf16*>(a.k) + (size_t)sr.row0 * a.ldk + (size_t)head * dk;
    const bf16* d_g = reinterpret_cast<const bf16*>(a.d) + (size_t)sr.row0 * a.ldd + (size_t)head * dk;
    const bf16* v_g = reinterpret_cast<const bf16*>(a.v) + (size_t)sr.row0 * a.ldv + (size_t)head * dv;
    float* o_g = a.o + (size_t)sr.row0 * (a.H * dv) + (size_t)head * dv;
    const unsigned ic = min(i0, dk - 4), jc = min(j, dv - 1);
    auto ask = [&](int c0, Numbers& x) {                  // a block's numbers, from places that exist
        const int end = sr.n - 1, at = min(c0, end);
        const unsigned most = end - at, t = min((unsigned)c, most);
        if (FORM != WKV_SUMS) x.r = *reinterpret_cast<const Four*>(r_g + (size_t)at * a.ldr + (__umul24(t, a.ldr) + ic));
        x.k = *reinterpret_cast<const Four*>(k_g + (size_t)at * a.ldk + (__umul24(t, a.ldk) + ic));
        x.d = *reinterpret_cast<const Four*>(d_g + (size_t)at * a.ldd + (__umul24(t, a.ldd) + ic));
#pragma unroll
        for (int q = 0; q < 4; ++q) x.v[q] = (v_g + (size_t)at * a.ldv)[__umul24(min((unsigned)(g * 4 + q), most), a.ldv) + jc];
    };
    // what S does not enter: A's shares, r W and k W in shared memory, the block's v
    auto prepare = [&](int c0, int b, Numbers& x, float (&v)[4]) {
        const int nc = min(WKV_BLOCK, sr.n - c0);
        const bool live = in && c < nc;
        float r[4], k[4], T[4], E[4], F[4];               // T, E, F: -log2 of products of decays
#pragma unroll
        for (int q = 0; q < 4; ++q) {                     // a token behind the last changes nothing: no key, no decay
            r[q] = FORM != WKV_SUMS && live ? to_f32(x.r.e[q]) : 0.f;
            k[q] = live ? to_f32(x.k.e[q]) : 0.f;
            float rate = expf(to_f32(x.d.e[q]) + off[q]) * 1.44269504f;
            asm("" : "+v"(rate));                         // formed by every lane: no branch around it
            T[q] = live ? rate : 0.f;
            v[q] = owns && g * 4 + q < nc ? to_f32(x.v[q]) : 0.f;
            E[q] = F[q] = 0.f;
        }
        ask(c0 + AHEAD * WKV_BLOCK, x);
        wkv_f4 D[4];
#pragma unroll
        for (int l = 0; l < 4; ++l) D[l] = (wkv_f4)(0.f);
        auto level = [&](auto l) {                        // bit l: the pairs' product, then W over blocks of 2^(l + 1)
            constexpr int L = decltype(l)::value;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (FORM != WKV_SUMS)
                    D[L] = __builtin_amdgcn_mfma_f32_16x16x4f32(L ? r[q] * wkv_decay(E[q]) : r[q], L ? k[q] * wkv_decay(F[q]) : k[q], D[L], 0, 0, 0);
                const float o = wkv_partner<L>(T[q]);
                const bool upper = c >> L & 1;
                E[q] += upper ? o : 0.f;
                F[q] += upper ? 0.f : o;
                T[q] += o;
            }
        };
        float own = 0.f;                                  // token c's with itself: every group of lanes holds the sum
        if (FORM != WKV_SUMS) {
            own = fmaf(r[0], bonus[0] * k[0], r[1] * (bonus[1] * k[1])) + fmaf(r[2], bonus[2] * k[2], r[3] * (bonus[3] * k[3]));
            own += __shfl_xor(own, 16);
            own += __shfl_xor(own, 32);
        }
        level(std::integral_constant<int, 0>());
        level(std::integral_constant<int, 1>());
        level(std::integral_constant<int, 2>());
        level(std::integral_constant<int, 3>());
        const int m0 = w / 4 * 4 + g;                     // row w 16 + g 4 + q of the state: tile m0, register w % 4, lanes of group q
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (FORM != WKV_SUMS) r_s[b][c * ROW + q * 4 * P + m0 * 4 + w % 4] = r[q] * wkv_decay(E[q]);
            k_s[b][c * ROW + (q * 4 + w % 4) * P + m0] = k[q] * wkv_decay(F[q]);
            t_s[b][q * 4 * P + m0 * 4 + w % 4] = wkv_decay(T[q]);    // the same from every token's lane
            if (FORM == WKV_SUMS) fade[q] += T[q];
        }
        if (FORM != WKV_SUMS) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {                 // D: column s = c, row t = g 4 + q
                const int t = g * 4 + q, x = t ^ c;
                float d0 = D[0][q], d1 = D[1][q], d2 = D[2][q], d3 = D[3][q];
                asm("" : "+v"(d0), "+v"(d1), "+v"(d2), "+v"(d3));         // read here: chosen from by selects, not by branches
                const float pair = x >= 8 ? d3 : x >= 4 ? d2 : x >= 2 ? d1 : d0;
                a_s[b][(w * WKV_BLOCK + t) * AROW + c] = t > c ? pair : 0.f;
            }
            own_s[b][w * WKV_BLOCK + c] = own;
        }
    };
    // the block's outputs from S and A, and S behind it
    auto advance = [&](int c0, int b, const float (&v)[4], bool last) {
        const int nc = min(WKV_BLOCK, sr.n - c0);
        wkv_f4 o0 = (wkv_f4)(0.f), o1 = (wkv_f4)(0.f), o2 = (wkv_f4)(0.f), own;
        if (FORM != WKV_SUMS) {
#pragma unroll
            for (int m = 0; m < P; ++m) {
                const wkv_f4 rr = *reinterpret_cast<const wkv_f4*>(&r_s[b][c * ROW + g * 4 * P + m * 4]);
#pragma unroll
                for (int q = 0; q < 4; q += 2) {
                    o0 = __builtin_amdgcn_mfma_f32_16x16x4f32(rr[q], S[m][q], o0, 0, 0, 0);
                    o1 = __builtin_amdgcn_mfma_f32_16x16x4f32(rr[q + 1], S[m][q + 1], o1, 0, 0, 0);
                }
            }
            const wkv_f4 am = wkv_shares<P>(&a_s[b][c * AROW + g * 4], WKV_BLOCK * AROW);
#pragma unroll
            for (int q = 0; q < 4; ++q) o2 = __builtin_amdgcn_mfma_f32_16x16x4f32(am[q], v[q], o2, 0, 0, 0);
            own = wkv_shares<P>(&own_s[b][g * 4], WKV_BLOCK);
        }
        o0 += o1;
        wkv_settle(o0);
        wkv_settle(o2);
        if (FORM != WKV_OUTPUTS || !last) {               // (no one asks for what lies behind a piece's end)
#pragma unroll
            for (int m = 0; m < P; ++m) S[m] *= *reinterpret_cast<const wkv_f4*>(&t_s[b][g * 4 * P + m * 4]);
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int m = 0; m < P; m += 4) {
                    const wkv_f4 kk = *reinterpret_cast<const wkv_f4*>(&k_s[b][(g * 4 + q) * ROW + c * P + m]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) S[m + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[e], v[q], S[m + e], 0, 0, 0);
                }
        }
        if (FORM == WKV_SUMS) return;
        const bool fine = fabsf(v[0]) < INFINITY && fabsf(v[1]) < INFINITY && fabsf(v[2]) < INFINITY && fabsf(v[3]) < INFINITY;
        if (!__all(fine)) {                               // an infinity or a NaN must not meet the zeros of the tokens before it
            o2 = (wkv_f4)(0.f);
#pragma unroll 1
            for (int s = 0; s < nc; ++s) {
                const float vs = __shfl(s % 4 == 0 ? v[0] : s % 4 == 1 ? v[1] : s % 4 == 2 ? v[2] : v[3], s / 4 * 16 + c);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float ats = 0.f;
                    for (int p = 0; p < P; ++p) ats += a_s[b][(p * WKV_BLOCK + g * 4 + q) * AROW + s];
                    if (s < g * 4 + q) o2[q] = fmaf(ats, vs, o2[q]);
                }
            }
        }
        o0 += o2;
#pragma unroll
        for (int q = 0; q < 4; ++q) o0[q] = fmaf(own[q], v[q], o0[q]);       // the token's own share last: one rounding of it
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (owns && g * 4 + q < nc) (o_g + (size_t)(c0 + q) * (a.H * dv))[__umul24(g * 4, a.H * dv) + j] = o0[q];
    };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) ask(i * WKV_BLOCK, num[i]);
    float v[2][4];
    prepare(0, 0, num[0], v[0]);
    for (int base = 0; base < sr.n; base += AHEAD * WKV_BLOCK) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int c0 = base + i * WKV_BLOCK;
            if (c0 >= sr.n) break;
            lds_barrier();                                // the block is prepared, and the one before it read
            if (c0 + WKV_BLOCK < sr.n) prepare(c0 + WKV_BLOCK, (i + 1) % 2, num[(i + 1) % AHEAD], v[(i + 1) % 2]);
            advance(c0, i % 2, v[i % 2], c0 + WKV_BLOCK >= sr.n);
        }
    }
#pragma unroll
    for (int m = 0; m < P; ++m) wkv_settle(S[m]);
    if (FORM != WKV_OUTPUTS && owns) {
#pragma unroll
        for (int m = 0; m < P; ++m) *reinterpret_cast<wkv_f4*>(S_g + ((size_t)((m % 4) * 4 + g) * dv + j) * P + m / 4 * 4) = S[m];
    }
    if (FORM == WKV_SUMS) {
        if (c == 0) *reinterpret_cast<float4*>(a.fade + ((size_t)blockIdx.x * a.H + head) * DKP + i0) = make_float4(wkv_decay(fade[0]), wkv_decay(fade[1]), wkv_decay(fade[2]), wkv_decay(fade[3]));
        return;
    }
    if (head == 0 && last_piece) {                        // the step's last h of this sequence, for the next step's shift
        float* hp = a.state + (size_t)a.slot_ids[sr.seq] * a.state_stride + (size_t)a.H * DKP * dv;
        const bf16* last = reinterpret_cast<const bf16*>(a.h) + (size_t)(sr.row0 + sr.n - 1) * a.D;
        for (int e = threadIdx.x; e < a.D; e += P * 64) hp[e] = to_f32(last[e]);
    }
}

template <int FORM> static void wkv_blocks_launch(const WkvArgs& a, int groups, hipStream_t s) {
    if (a.P == 4) hipLaunchKernelGGL((wkv_blocks_kernel<4, FORM>), dim3(groups, a.H), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((wkv_blocks_kernel<8, FORM>), dim3(groups, a.H), dim3(512), 0, s, a);
}

// What wkv_blocks_kernel takes: heads of more than 32 and up to 128 rows whose columns its waves own, read in groups of four bf16 of r, k and d and
// four float32 of the offset, the bonus and a state; rows within 24 bits of their block's first.  Faster than the walk wherever it applies (16 tokens of
// one sequence 15.7 / 15.8 us with the launch, 64 of sixteen sequences 56 / 20); float32 steps stay with the walk, whose bits do not depend on
// how a sequence was cut into steps.
static bool wkv_blocks_take(const WkvArgs& a, bool state_too) {
    const uintptr_t rows = (uintptr_t)a.r | (uintptr_t)a.k | (uintptr_t)a.d, vecs = (uintptr_t)a.w0 | (uintptr_t)a.u | (uintptr_t)a.carry | (uintptr_t)a.fade;
    return (a.P == 4 || a.P == 8) && a.dk % 4 == 0 && (a.ldr | a.ldk | a.ldd | a.ldv | a.H * a.dv) < 1 << 24 && a.dv <= a.P * 16 && ((a.ldr | a.ldk | a.ldd) & 3) == 0 && (rows & 7) == 0 && (vecs & 15) == 0 &&
           (!state_too || (((uintptr_t)a.state & 15) == 0 && a.state_stride % 4 == 0));
}

// A thread an element of a head's state: through the pieces of a sequence S <- fade_p S + S_p, leaving what each piece starts
// from in its place and the last in the slot's state row.  Four pieces' sums are asked for at once.
__global__ __launch_bounds__(256) void wkv_carry_kernel(WkvArgs a) {
    const SeqRange sr = seq_range(a.tiles, a.seq_lens, blockIdx.y);
    if (sr.n <= 0 || sr.pos0 < 0) return;
    const int dkp = a.P * WKV_KR;
    const size_t per_head = (size_t)dkp * a.dv, n = a.H * per_head;
    const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const int head = (int)(e / per_head), at = (int)(e % per_head);
    const int row = at % a.P * WKV_KR + at / (a.dv * a.P);        // element (row p WKV_KR + ii, column j) at (ii dv + j) P + p
    const int pieces = (sr.n + WKV_PIECE - 1) / WKV_PIECE;
    float* st = a.state + (size_t)a.slot_ids[sr.seq] * a.state_stride + e;
    const size_t before = pieces_before(a.tiles, blockIdx.y, WKV_PIECE);
    float* c = a.carry + before * n + e;
    const float* f = a.fade + (before * a.H + head) * dkp + row;
    const size_t fs = (size_t)a.H * dkp;
    float S = sr.pos0 > 0 ? *st : 0.f;
    for (int p0 = 0; p0 < pieces; p0 += 4) {
        float own[4], fd[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int p = min(p0 + q, pieces - 1);
            own[q] = c[(size_t)p * n];
            fd[q] = f[(size_t)p * fs];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (p0 + q < pieces) {
                c[(size_t)(p0 + q) * n] = S;
                S = fmaf(fd[q], S, own[q]);
            }
    }
    *st = S;
}

// The split of a head over threads and workgroups (P, CB, TC, threads).  P follows from the head size alone (it fixes the
// order of a column's sum); CB, the columns of a workgroup, is the largest that still gives the launch `want_wgs`
// workgroups, down to one wave of threads, so that a prompt of one sequence spreads over the chip as a batch does.
static bool wkv_shape(int dk, int dv, int groups, int& P, int& CB, int& TC, int& walkers, int& threads) {
    if (dk < 1 || dv < 1 || dk > WKV_MAX_DIM || dv > WKV_MAX_DIM) return false;
    P = 1;
    while (P * WKV_KR < dk) P <<= 1;                      // <= 16
    const int most = WKV_MAX_THREADS / P, least = BN_WAVE / P;          // columns of a full set of walkers, of one wave
    CB = dv < most ? dv : most;
    while (CB > least && (long long)groups * ((dv + CB - 1) / CB) < 256) CB = (CB + 1) / 2 < least ? least : (CB + 1) / 2;
    walkers = ((CB * P + BN_WAVE - 1) / BN_WAVE) * BN_WAVE;
    threads = walkers + 128;                              // and the staging waves
    TC = 32;                                              // the longest chunk whose two buffers fit beside each other
    while (TC > 4 && (size_t)2 * TC * (3 * P * WKV_KR + CB) * sizeof(float) > 60 * 1024) TC >>= 1;
    return true;
}

extern "C" int bn_wkv_supports(int dk, int dv) {
    int P, CB, TC, wk, th;
    return wkv_shape(dk, dv, 1, P, CB, TC, wk, th) ? 1 : 0;
}

// float32 values of one head's state: dk rounded up to the rows that the walkers hold (a power of two times WKV_KR), times dv
extern "C" int bn_wkv_state_floats(int dk, int dv) {
    int P, CB, TC, wk, th;
    return wkv_shape(dk, dv, 1, P, CB, TC, wk, th) ? P * WKV_KR * dv : 0;
}

extern "C" int bn_wkv_scan(int dtype, const void* r, int ldr, const void* k, int ldk, const void* v, int ldv, const void* d,
                           int ldd, const float* w0, const float* u, float* o, const void* h, float* state,
                           long long state_stride, const int* tiles, int n_tiles, const int* seq_lens, const int* slot_ids,
                           int H, int dk, int dv, int D, int pieces, float* carry, float* fade, hipStream_t s) {
    // pieces: 0, or what the step's sequences can be cut into together (rows carry and fade of as many)
    WkvArgs a;
    int threads;
    if (n_tiles <= 0 || H <= 0 || D <= 0 || pieces < 0 || (pieces > 0 && (!tiles || !carry || !fade || n_tiles > 65535)) ||
        !wkv_shape(dk, dv, (pieces > 0 ? pieces : n_tiles) * H, a.P, a.CB, a.TC, a.walkers, threads))
        return BN_ERR_ARG;
    if (!r || !k || !v || !d || !w0 || !u || !o || !h || !state || !slot_ids || (!tiles && !seq_lens)) return BN_ERR_ARG;
    if (state_stride < (long long)H * a.P * WKV_KR * dv + D) return BN_ERR_ARG;
    a.r = r; a.k = k; a.v = v; a.d = d; a.ldr = ldr; a.ldk = ldk; a.ldv = ldv; a.ldd = ldd;
    a.w0 = w0; a.u = u; a.o = o; a.h = h; a.state = state; a.state_stride = (size_t)state_stride;
    a.tiles = tiles; a.seq_lens = seq_lens; a.slot_ids = slot_ids;
    a.H = H; a.dk = dk; a.dv = dv; a.D = D;
    a.n_tiles = n_tiles; a.carry = carry; a.fade = fade;
    const size_t smem = (size_t)2 * a.TC * (3 * a.P * WKV_KR + a.CB) * sizeof(float);      // two staged chunks
    const dim3 grid(pieces > 0 ? pieces : n_tiles, H, (dv + a.CB - 1) / a.CB), block(threads);
    if (dtype != BN_DT_F32 && dtype != BN_DT_BF16) return BN_ERR_DTYPE;
    const bool f32 = dtype == BN_DT_F32;
    if (pieces == 0) {
        if (!f32 && tiles && wkv_blocks_take(a, true)) wkv_blocks_launch<WKV_WALK>(a, n_tiles, s);
        else if (f32) hipLaunchKernelGGL((wkv_scan_kernel<float, WKV_WALK>), grid, block, smem, s, a);
        else hipLaunchKernelGGL((wkv_scan_kernel<bf16, WKV_WALK>), grid, block, smem, s, a);
        return bn_launch_status();
    }
    const bool blocks = !f32 && wkv_blocks_take(a, false);
    if (blocks) wkv_blocks_launch<WKV_SUMS>(a, pieces, s);
    else if (f32) hipLaunchKernelGGL((wkv_scan_kernel<float, WKV_SUMS>), grid, block, smem, s, a);
    else hipLaunchKernelGGL((wkv_scan_kernel<bf16, WKV_SUMS>), grid, block, smem, s, a);
    if (int rc = bn_launch_status()) return rc;
    const size_t n = (size_t)H * a.P * WKV_KR * dv;
    hipLaunchKernelGGL(wkv_carry_kernel, dim3((unsigned)((n + 255) / 256), n_tiles), dim3(256), 0, s, a);
    if (int rc = bn_launch_status()) return rc;
    if (blocks) wkv_blocks_launch<WKV_OUTPUTS>(a, pieces, s);
    else if (f32) hipLaunchKernelGGL((wkv_scan_kernel<float, WKV_OUTPUTS>), grid, block, smem, s, a);
    else hipLaunchKernelGGL((wkv_scan_kernel<bf16, WKV_OUTPUTS>), grid, block, smem, s, a);
    return bn_launch_status();
}

// ---- per-head RMS of the recurrence's output, its weight and the gate -----------------------------------------------
// one wave per (row, head): y = o / sqrt(mean(o^2) + eps) * weight * silu(gate); weight null: 1
template <typename T>
__global__ __launch_bounds__(BN_WAVE) void head_norm_gate_kernel(T* __restrict__ y, const float* __restrict__ o,
                                                                  const T* __restrict__ gate, int ldg,
                                                                  const float* __restrict__ weight, int H, int dv, float eps) {
    const int t = blockIdx.x, head = blockIdx.y, lane = threadIdx.x;
    const float* ov = o + ((size_t)t * H + head) * dv;
    float ss = 0.f;
    for (int e = lane; e < dv; e += BN_WAVE) ss = fmaf(ov[e], ov[e], ss);
    ss = wave_sum(ss);
    const float f = 1.0f / sqrtf(ss / (float)dv + eps);
    for (int e = lane; e < dv; e += BN_WAVE) {
        const float g = to_f32(gate[(size_t)t * ldg + (size_t)head * dv + e]);
        const float w = weight ? weight[(size_t)head * dv + e] : 1.0f;
        y[((size_t)t * H + head) * dv + e] = from_f32<T>(ov[e] * f * w * bn_unary_act(g, BN_UNARY_SILU));
    }
}

// The same for the rows of a bf16 prompt: a lane holds eight neighbouring numbers of a head (16-byte loads and stores), dv / 8 lanes a
// head.  Bound by memory (5.2 TB/s at 8,192 rows of 32 heads of 64).  us, a wave a head (above: one number a lane at dv = 64, workgroups of
// one wave) -> this at 129 / 512 / 2,048 / 8,192 rows: 32 heads of 64 3.2 -> 2.8, 6.0 -> 3.6, 18.2 -> 8.2, 62.6 -> 30.7; 16 of 128 3.1 -> 3.0, 4.8 ->
// 3.6, 12.3 -> 8.3, 42.9 -> 30.7; 8 of 64 2.5 -> 2.8, 3.2 -> 2.9, 6.0 -> 3.6, 18.3 -> 8.0.  With fewer than HNG_MIN numbers the other is as fast
// or faster by up to 0.6 (16 rows).
#define HNG_WAVES 4
#define HNG_MIN (1 << 18)
__global__ __launch_bounds__(HNG_WAVES* BN_WAVE) void head_norm_gate_rows_kernel(bf16* __restrict__ y, const float* __restrict__ o,
                                                                                 const bf16* __restrict__ gate, int ldg,
                                                                                 const float* __restrict__ weight, size_t n8, int row8, int lanes,
                                                                                 float eps) {
    const size_t at = (size_t)blockIdx.x * (HNG_WAVES * BN_WAVE) + threadIdx.x;
    const bool live = at < n8;                           // (dead lanes are whole heads: n8 is a multiple of lanes)
    const size_t j = live ? at : 0;
    const size_t t = j / row8;
    const int c = (int)(j - t * row8) * 8;
    float v[8], g[8];
    const float4 a0 = reinterpret_cast<const float4*>(o)[2 * j], a1 = reinterpret_cast<const float4*>(o)[2 * j + 1];
    const uint4 b = *reinterpret_cast<const uint4*>(gate + t * (size_t)ldg + c);
    v[0] = a0.x; v[1] = a0.y; v[2] = a0.z; v[3] = a0.w; v[4] = a1.x; v[5] = a1.y; v[6] = a1.z; v[7] = a1.w;
    const uint32_t w[4] = {b.x, b.y, b.z, b.w};
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        g[e] = e & 1 ? bf16hi_to_f32(w[e >> 1]) : bf16lo_to_f32(w[e >> 1]);
        ss = fmaf(v[e], v[e], ss);
    }
    for (int m = 1; m < lanes; m <<= 1) ss += __shfl_xor(ss, m, BN_WAVE);
    if (!live) return;
    const float f = 1.0f / sqrtf(ss / (float)(8 * lanes) + eps);
    float wt[8] = {1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f};
    if (weight) {
        const float4 w0 = *reinterpret_cast<const float4*>(weight + c), w1 = *reinterpret_cast<const float4*>(weight + c + 4);
        wt[0] = w0.x; wt[1] = w0.y; wt[2] = w0.z; wt[3] = w0.w; wt[4] = w1.x; wt[5] = w1.y; wt[6] = w1.z; wt[7] = w1.w;
    }
    uint32_t p[4];
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        const bf16 lo = from_f32<bf16>(v[e] * f * wt[e] * bn_unary_act(g[e], BN_UNARY_SILU));
        const bf16 hi = from_f32<bf16>(v[e + 1] * f * wt[e + 1] * bn_unary_act(g[e + 1], BN_UNARY_SILU));
        p[e >> 1] = (uint32_t)__builtin_bit_cast(uint16_t, lo) | ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
    }
    reinterpret_cast<uint4*>(y)[j] = make_uint4(p[0], p[1], p[2], p[3]);
}

extern "C" int bn_head_norm_gate(int dtype, void* y, const float* o, const void* gate, int ldg, const float* weight,
                                 int n_tokens, int H, int dv, float eps, hipStream_t s) {
    if (n_tokens <= 0 || H <= 0 || dv <= 0 || !y || !o || !gate || ldg < H * dv) return BN_ERR_ARG;
    const dim3 grid(n_tokens, H);
    const int lanes = dv / 8;
    if (dtype == BN_DT_BF16 && (long long)n_tokens * H * dv >= HNG_MIN && dv % 8 == 0 && lanes <= BN_WAVE && (lanes & (lanes - 1)) == 0 && ldg % 8 == 0 &&
        !(((uintptr_t)y | (uintptr_t)o | (uintptr_t)gate | (uintptr_t)weight) & 15)) {
        const size_t n8 = (size_t)n_tokens * H * lanes, wgs = (n8 + HNG_WAVES * BN_WAVE - 1) / (HNG_WAVES * BN_WAVE);
        if (wgs > 0x7fffffff) return BN_ERR_ARG;
        hipLaunchKernelGGL(head_norm_gate_rows_kernel, dim3((unsigned)wgs), dim3(HNG_WAVES * BN_WAVE), 0, s, (bf16*)y, o, (const bf16*)gate, ldg,
                           weight, n8, H * lanes, lanes, eps);
        return bn_launch_status();
    }
    if (dtype == BN_DT_F32)
        hipLaunchKernelGGL(head_norm_gate_kernel<float>, grid, dim3(BN_WAVE), 0, s, (float*)y, o, (const float*)gate, ldg, weight, H, dv, eps);
    else if (dtype == BN_DT_BF16)
        hipLaunchKernelGGL(head_norm_gate_kernel<bf16>, grid, dim3(BN_WAVE), 0, s, (bf16*)y, o, (const bf16*)gate, ldg, weight, H, dv, eps);
    else
        return BN_ERR_DTYPE;
    return bn_launch_status();
}

// ---- a decode step of wkv with its norm and gate -------------------------------------------------------------------------
// One token of every sequence: a workgroup owns a (sequence, head) whole, a thread the rows of a column that the walk gives it
// (P neighbouring lanes a column), so the state's way in and out is one load and one store a number; the columns' sums meet in
// shared memory, where every wave forms the head's mean square as head_norm_gate_kernel does (the same bits as the walk and
// that kernel: a position's output does not depend on the step it came in), and weight and gate follow.  Bound by latency at
// few sequences (a trip to memory for the state, two barriers): one sequence of 32 heads of 64 4.8 us in a graph of such
// launches, 6.9 in a decode step's profile, where the walk and the norm's kernel took 7.8 + 5.0.
// NJ > 0: the decay's last product (low . w2^T, up to 32 NJ columns) is formed here as well, 16 channels a wave on the matrix cores
// in the order of skinny_gemm's kernel (the same bits), instead of in a launch of its own that reads 8 KB a head (3.8 us; this
// kernel 5.0 -> 5.8 with one sequence of 32 heads of 64).
template <typename T, int NJ>
__global__ __launch_bounds__(1024) void wkv_step_kernel(WkvArgs a, T* __restrict__ y, const T* __restrict__ gate, int ldg,
                                                        const float* __restrict__ weight, float eps) {
    __shared__ __align__(16) float r_s[WKV_MAX_DIM], k_s[WKV_MAX_DIM], w_s[WKV_MAX_DIM];
    __shared__ float o_s[WKV_MAX_DIM], d_s[WKV_MAX_DIM];
    const int seq = blockIdx.x, head = blockIdx.y, tid = threadIdx.x;
    const int pos = a.seq_lens[seq] - 1;
    if (pos < 0) return;
    const int P = a.P, dk = a.dk, dv = a.dv, dkp = P * WKV_KR, p = tid % P, j = tid / P;
    const bool owns = j < dv;
    float* S_g = a.state + (size_t)a.slot_ids[seq] * a.state_stride + (size_t)head * dkp * dv;
    float S[WKV_KR], ub[WKV_KR];
    const int jc = owns ? j : 0;                          // loads in straight line; a thread without a column drops what it loads
#pragma unroll
    for (int ii = 0; ii < WKV_KR; ++ii) {
        S[ii] = S_g[((size_t)ii * dv + jc) * P + p];
        ub[ii] = a.u[(size_t)head * dk + min(p * WKV_KR + ii, dk - 1)];
    }
    if constexpr (NJ > 0) {
        typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
        typedef __attribute__((ext_vector_type(4))) float f32x4;
        const int lane = tid & (BN_WAVE - 1), n_waves = blockDim.x / BN_WAVE, i = lane & 15, g = lane >> 4;
        for (int tile = __builtin_amdgcn_readfirstlane(tid / BN_WAVE); 16 * tile < dk; tile += n_waves) {
            const bf16* wr = a.w2 + ((size_t)head * dk + 16 * tile + i) * a.rank + 8 * g;
            const bf16* xr = a.low + (size_t)seq * a.ldlow + 8 * g;
            bf16x8 x[NJ], w[NJ];
#pragma unroll
            for (int q = 0; q < NJ; ++q) {                // past the last 32 columns: those again, not multiplied
                const int c = min(32 * q, a.rank - 32);
                x[q] = *reinterpret_cast<const bf16x8*>(xr + c);
                w[q] = *reinterpret_cast<const bf16x8*>(wr + c);
            }
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < NJ; ++q)
                if (32 * q < a.rank) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[q], w[q], acc, 0, 0, 0);
            if (g == 0) d_s[16 * tile + i] = to_f32(from_f32<bf16>(acc[0]));
        }
        lds_barrier();
    }
    const float vj = to_f32(reinterpret_cast<const T*>(a.v)[(size_t)seq * a.ldv + (size_t)head * dv + jc]);
    const float gj = to_f32(gate[(size_t)seq * ldg + (size_t)head * dv + jc]), wj = weight ? weight[(size_t)head * dv + jc] : 1.0f;
    for (int i = tid; i < dkp; i += blockDim.x) {
        const size_t c = (size_t)head * dk + min(i, dk - 1);
        const float r = to_f32(reinterpret_cast<const T*>(a.r)[(size_t)seq * a.ldr + c]);
        const float k = to_f32(reinterpret_cast<const T*>(a.k)[(size_t)seq * a.ldk + c]);
        const float d = (NJ > 0 ? d_s[min(i, dk - 1)] : to_f32(reinterpret_cast<const T*>(a.d)[(size_t)seq * a.ldd + c])) + a.w0[c];
        r_s[i] = i < dk ? r : 0.f;
        k_s[i] = i < dk ? k : 0.f;
        w_s[i] = i < dk ? expf(-expf(d)) : 0.f;
    }
    if (head == 0) {                                      // the step's h, for the next step's shift
        float* hp = a.state + (size_t)a.slot_ids[seq] * a.state_stride + (size_t)a.H * dkp * dv;
        for (int e = tid; e < a.D; e += blockDim.x) hp[e] = to_f32(reinterpret_cast<const T*>(a.h)[(size_t)seq * a.D + e]);
    }
#pragma unroll
    for (int ii = 0; ii < WKV_KR; ++ii) {
        if (pos == 0 || !owns) S[ii] = 0.f;
        if (p * WKV_KR + ii >= dk) ub[ii] = 0.f;
    }
    lds_barrier();
    float4 rr[WKV_KR / 4], kk[WKV_KR / 4], ww[WKV_KR / 4];
#pragma unroll
    for (int q = 0; q < WKV_KR / 4; ++q) {
        rr[q] = reinterpret_cast<const float4*>(r_s + p * WKV_KR)[q];
        kk[q] = reinterpret_cast<const float4*>(k_s + p * WKV_KR)[q];
        ww[q] = reinterpret_cast<const float4*>(w_s + p * WKV_KR)[q];
    }
    const float o = wkv_token(rr, kk, ww, vj, ub, S, P);
    if (owns && p == 0) o_s[j] = o;
    if (owns) {
#pragma unroll
        for (int ii = 0; ii < WKV_KR; ++ii) S_g[((size_t)ii * dv + j) * P + p] = S[ii];
    }
    lds_barrier();
    float ss = 0.f;
    for (int e = tid & (BN_WAVE - 1); e < dv; e += BN_WAVE) ss = fmaf(o_s[e], o_s[e], ss);
    ss = wave_sum(ss);
    const float f = 1.0f / sqrtf(ss / (float)dv + eps);
    if (owns && p == 0) y[((size_t)seq * a.H + head) * dv + j] = from_f32<T>(o * f * wj * bn_unary_act(gj, BN_UNARY_SILU));
}

// 1 if a head of these sizes fits a workgroup of the kernel above
extern "C" int bn_wkv_step_supports(int dk, int dv) {
    int P, CB, TC, wk, th;
    return wkv_shape(dk, dv, 1, P, CB, TC, wk, th) && P * dv <= 1024 ? 1 : 0;
}

// 1 if the step forms d itself from low [n, rank] and w2 [H dk, rank] (bf16, rows of 16-byte groups at 16-byte addresses)
extern "C" int bn_wkv_step_takes_low(int dk, int dv, int rank) {
    return bn_wkv_step_supports(dk, dv) && dk % 16 == 0 && rank >= 32 && rank <= 256 && rank % 32 == 0;
}

// d null: low [n_seqs, rank] (row stride ldlow) and w2 [H dk, rank] (contiguous) in its place, bf16
extern "C" int bn_wkv_step(int dtype, const void* r, int ldr, const void* k, int ldk, const void* v, int ldv, const void* d, int ldd,
                           const void* low, int ldlow, const void* w2, int rank, const float* w0, const float* u, const void* h, float* state, long long state_stride,
                           const int* seq_lens, const int* slot_ids, int n_seqs, int H, int dk, int dv, int D, void* y,
                           const void* gate, int ldg, const float* weight, float eps, hipStream_t s) {
    WkvArgs a = {};
    int threads;
    if (n_seqs <= 0 || H <= 0 || D <= 0 || !bn_wkv_step_supports(dk, dv) || !wkv_shape(dk, dv, 1, a.P, a.CB, a.TC, a.walkers, threads))
        return BN_ERR_ARG;
    if (!r || !k || !v || !d != (low && w2) || !w0 || !u || !h || !state || !slot_ids || !seq_lens || !y || !gate || ldg < H * dv) return BN_ERR_ARG;
    if (!d && (dtype != BN_DT_BF16 || !bn_wkv_step_takes_low(dk, dv, rank) || ldlow < rank || ldlow % 8 || (((uintptr_t)low | (uintptr_t)w2) & 15)))
        return BN_ERR_ARG;
    if (state_stride < (long long)H * a.P * WKV_KR * dv + D) return BN_ERR_ARG;
    a.r = r; a.k = k; a.v = v; a.d = d; a.ldr = ldr; a.ldk = ldk; a.ldv = ldv; a.ldd = ldd;
    a.w0 = w0; a.u = u; a.h = h; a.state = state; a.state_stride = (size_t)state_stride;
    a.seq_lens = seq_lens; a.slot_ids = slot_ids;
    a.H = H; a.dk = dk; a.dv = dv; a.D = D;
    a.low = (const bf16*)low; a.w2 = (const bf16*)w2; a.ldlow = ldlow; a.rank = rank;
    const dim3 grid(n_seqs, H), block((a.P * dv + BN_WAVE - 1) / BN_WAVE * BN_WAVE);
    auto go = [&](auto kernel, auto* out) {
        hipLaunchKernelGGL(kernel, grid, block, 0, s, a, out, (decltype(out))gate, ldg, weight, eps);
        return bn_launch_status();
    };
    if (dtype == BN_DT_F32) return go(wkv_step_kernel<float, 0>, (float*)y);
    if (dtype != BN_DT_BF16) return BN_ERR_DTYPE;
    if (d) return go(wkv_step_kernel<bf16, 0>, (bf16*)y);
    if (rank <= 64) return go(wkv_step_kernel<bf16, 2>, (bf16*)y);
    return rank <= 128 ? go(wkv_step_kernel<bf16, 4>, (bf16*)y) : go(wkv_step_kernel<bf16, 8>, (bf16*)y);
}

// ---- min-GRU ------------------------------------------------------------------------------------------------------
// zxg [T, ld]: the three projections side by side (update gate at 0, candidate at W, output gate at 2 W), without their
// biases.  A workgroup owns GRU_CH channels of one sequence.  Its tokens come in stages of GRU_TC: all threads load a
// stage (the next one is asked for before the current one is walked), turn it into gate, candidate and silu(g) and
// park those in shared memory; one thread a channel then walks the stage, S <- S + z (cand - S), and leaves S silu(g),
// which all threads store.  The chain of a walked channel is the same operations in the same order whatever the step holds.
#define GRU_CH 64
#define GRU_TC 64
#define GRU_THREADS 256
#define GRU_PER_THREAD (GRU_CH * GRU_TC / GRU_THREADS)

// FORM: the whole sequence, or (long bf16 steps of few sequences) one piece of GRU_TC tokens, as the wkv recurrence is cut, in
// another order of rounding: its own chain from nothing and the product of its (1 - z) (GRU_SUMS), the carry through the pieces (mingru_carry_kernel), the chain
// again from the piece's start with outputs (GRU_OUTPUTS).  One sequence of 2,048 tokens, 2,048 channels: 235 us walked,
// 44 in pieces.
enum { GRU_WALK = 0, GRU_SUMS = 1, GRU_OUTPUTS = 2 };

template <typename T, int FORM>
__global__ __launch_bounds__(GRU_THREADS) void mingru_scan_kernel(T* __restrict__ y, const T* __restrict__ zxg, int ld,
                                                                   const float* __restrict__ bz, const float* __restrict__ bx,
                                                                   float* __restrict__ state, size_t state_stride,
                                                                   const int* __restrict__ tiles, const int* __restrict__ seq_lens,
                                                                   const int* __restrict__ slot_ids, int W, int n_tiles,
                                                                   float* __restrict__ carry, float* __restrict__ fade) {
    __shared__ float z_s[GRU_TC][GRU_CH], c_s[GRU_TC][GRU_CH], g_s[GRU_TC][GRU_CH];
    bool last_piece;
    const SeqRange sr = FORM == GRU_WALK ? seq_range(tiles, seq_lens, blockIdx.x) : piece_range(tiles, n_tiles, blockIdx.x, GRU_TC, last_piece);
    if (sr.n <= 0 || sr.pos0 < 0) return;
    const int tid = threadIdx.x;
    const int cc = tid % GRU_CH, t_first = tid / GRU_CH;            // this thread's channel and its first token of a stage
    const int c = blockIdx.y * GRU_CH + cc;
    const bool has = c < W;
    float* sp = FORM == GRU_WALK ? state + (size_t)slot_ids[sr.seq] * state_stride + c : carry + (size_t)blockIdx.x * W + c;
    float S = (has && tid < GRU_CH && (FORM == GRU_OUTPUTS || (FORM == GRU_WALK && sr.pos0 > 0))) ? *sp : 0.f, kept = 1.f;
    const float biasz = (has && bz) ? bz[c] : 0.f, biasx = (has && bx) ? bx[c] : 0.f;
    const T* in = zxg + (size_t)sr.row0 * ld + (has ? c : 0);
    T* out = y + (size_t)sr.row0 * W + c;
    float zr[GRU_PER_THREAD], cr[GRU_PER_THREAD], gr[GRU_PER_THREAD];
    auto fetch = [&](int t0) {
#pragma unroll
        for (int i = 0; i < GRU_PER_THREAD; ++i) {
            // unconditional loads from clamped places (a load under a branch is waited for where it stands); what a
            // thread without a channel or a token loads is never stored
            const int t = min(t0 + t_first + i * (GRU_THREADS / GRU_CH), sr.n - 1);
            zr[i] = to_f32(in[(size_t)t * ld]);
            cr[i] = to_f32(in[(size_t)t * ld + W]);
            gr[i] = to_f32(in[(size_t)t * ld + 2 * W]);
        }
    };
    fetch(0);
    for (int t0 = 0; t0 < sr.n; t0 += GRU_TC) {
#pragma unroll
        for (int i = 0; i < GRU_PER_THREAD; ++i) {
            const int tt = t_first + i * (GRU_THREADS / GRU_CH);
            const float cp = cr[i] + biasx;
            z_s[tt][cc] = 1.0f / (1.0f + expf(-(zr[i] + biasz)));
            c_s[tt][cc] = cp >= 0.f ? cp + 0.5f : 1.0f / (1.0f + expf(-cp));
            g_s[tt][cc] = bn_unary_act(gr[i], BN_UNARY_SILU);
        }
        lds_barrier();
        if (t0 + GRU_TC < sr.n) fetch(t0 + GRU_TC);
        const int nt = min(GRU_TC, sr.n - t0);
        if (tid < GRU_CH) {
            for (int tt = 0; tt < nt; tt += 8) {                    // eight tokens' values at once, then their chain
                float z8[8], c8[8], g8[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) { z8[i] = z_s[tt + i][cc]; c8[i] = c_s[tt + i][cc]; g8[i] = g_s[tt + i][cc]; }
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    if (tt + i < nt) {
                        S = fmaf(z8[i], c8[i] - S, S);              // (1 - z) S + z cand
                        if (FORM == GRU_SUMS) kept *= 1.f - z8[i];
                        else g_s[tt + i][cc] = S * g8[i];
                    }
                }
            }
        }
        if (FORM == GRU_SUMS) break;                                // a piece is one stage
        lds_barrier();
#pragma unroll
        for (int i = 0; i < GRU_PER_THREAD; ++i) {
            const int tt = t_first + i * (GRU_THREADS / GRU_CH);
            if (has && tt < nt) out[(size_t)(t0 + tt) * W] = from_f32<T>(g_s[tt][cc]);
        }
        lds_barrier();
    }
    if (FORM != GRU_OUTPUTS && has && tid < GRU_CH) {
        *sp = S;
        if (FORM == GRU_SUMS) fade[(size_t)blockIdx.x * W + c] = kept;
    }
}

// a thread a (sequence, channel): S <- kept_p S + S_p through the pieces, leaving what each starts from in its place
__global__ __launch_bounds__(64) void mingru_carry_kernel(float* __restrict__ carry, const float* __restrict__ fade,
                                                          float* __restrict__ state, size_t state_stride, const int* __restrict__ tiles,
                                                          const int* __restrict__ slot_ids, int W) {
    const SeqRange sr = seq_range(tiles, nullptr, blockIdx.y);
    const int c = blockIdx.x * 64 + threadIdx.x;
    if (sr.n <= 0 || sr.pos0 < 0 || c >= W) return;
    const int pieces = (sr.n + GRU_TC - 1) / GRU_TC;
    const size_t at = (size_t)pieces_before(tiles, blockIdx.y, GRU_TC) * W + c;
    float* sp = state + (size_t)slot_ids[sr.seq] * state_stride + c;
    float S = sr.pos0 > 0 ? *sp : 0.f;
    for (int p0 = 0; p0 < pieces; p0 += 8) {
        float own[8], f[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const size_t i = at + (size_t)min(p0 + q, pieces - 1) * W;
            own[q] = carry[i];
            f[q] = fade[i];
        }
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (p0 + q < pieces) {
                carry[at + (size_t)(p0 + q) * W] = S;
                S = fmaf(f[q], S, own[q]);
            }
    }
    *sp = S;
}

// A decode step: a thread a channel, everything it needs asked for at once, where the walk stages its one token through shared
// memory between two barriers (the same operations: the same bits).  us in a decode step, one sequence of 2,048 channels, 6.9 -> 3.5.
template <typename T>
__global__ __launch_bounds__(64) void mingru_step_kernel(T* __restrict__ y, const T* __restrict__ zxg, int ld, const float* __restrict__ bz,
                                                         const float* __restrict__ bx, float* __restrict__ state, size_t state_stride,
                                                         const int* __restrict__ seq_lens, const int* __restrict__ slot_ids, int W) {
    const int seq = blockIdx.y, c = blockIdx.x * 64 + threadIdx.x;
    const int pos = seq_lens[seq] - 1;
    if (pos < 0 || c >= W) return;                        // (a padding row may have no row of zxg)
    const T* in = zxg + (size_t)seq * ld + c;
    const float zr = to_f32(in[0]), cr = to_f32(in[W]), gr = to_f32(in[2 * (size_t)W]);
    const float zb = bz ? bz[c] : 0.f, xb = bx ? bx[c] : 0.f;
    float* sp = state + (size_t)slot_ids[seq] * state_stride + c;
    const float kept = *sp;
    float S = pos > 0 ? kept : 0.f;
    const float cp = cr + xb, z = 1.0f / (1.0f + expf(-(zr + zb)));
    const float cand = cp >= 0.f ? cp + 0.5f : 1.0f / (1.0f + expf(-cp));
    S = fmaf(z, cand - S, S);
    y[(size_t)seq * W + c] = from_f32<T>(S * bn_unary_act(gr, BN_UNARY_SILU));
    *sp = S;
}

extern "C" int bn_mingru_scan(int dtype, void* y, const void* zxg, int ld, const float* bz, const float* bx, float* state,
                              long long state_stride, const int* tiles, int n_tiles, const int* seq_lens,
                              const int* slot_ids, int W, int pieces, float* carry, float* fade, hipStream_t s) {
    if (n_tiles <= 0 || W <= 0 || ld < 3 * W || !y || !zxg || !state || !slot_ids || (!tiles && !seq_lens)) return BN_ERR_ARG;
    if (state_stride < W || pieces < 0 || (pieces > 0 && (!tiles || !carry || !fade || n_tiles > 65535))) return BN_ERR_ARG;
    if (dtype != BN_DT_F32 && dtype != BN_DT_BF16) return BN_ERR_DTYPE;
    const dim3 grid(pieces > 0 ? pieces : n_tiles, (W + GRU_CH - 1) / GRU_CH), block(GRU_THREADS);
    auto launch = [&](auto kernel, auto t) {
        typedef decltype(t) T;
        hipLaunchKernelGGL(kernel, grid, block, 0, s, (T*)y, (const T*)zxg, ld, bz, bx, state, (size_t)state_stride, tiles, seq_lens,
                           slot_ids, W, n_tiles, carry, fade);
    };
    const bool f32 = dtype == BN_DT_F32;
    if (!tiles && n_tiles <= 65535) {
        const dim3 threads((W + 63) / 64, n_tiles);
        if (f32)
            hipLaunchKernelGGL(mingru_step_kernel<float>, threads, dim3(64), 0, s, (float*)y, (const float*)zxg, ld, bz, bx, state,
                               (size_t)state_stride, seq_lens, slot_ids, W);
        else
            hipLaunchKernelGGL(mingru_step_kernel<bf16>, threads, dim3(64), 0, s, (bf16*)y, (const bf16*)zxg, ld, bz, bx, state,
                               (size_t)state_stride, seq_lens, slot_ids, W);
        return bn_launch_status();
    }
    if (pieces == 0) {
        if (f32) launch(mingru_scan_kernel<float, GRU_WALK>, float());
        else launch(mingru_scan_kernel<bf16, GRU_WALK>, bf16());
        return bn_launch_status();
    }
    if (f32) launch(mingru_scan_kernel<float, GRU_SUMS>, float());
    else launch(mingru_scan_kernel<bf16, GRU_SUMS>, bf16());
    if (int rc = bn_launch_status()) return rc;
    hipLaunchKernelGGL(mingru_carry_kernel, dim3((W + 63) / 64, n_tiles), dim3(64), 0, s, carry, fade, state, (size_t)state_stride, tiles,
                       slot_ids, W);
    if (int rc = bn_launch_status()) return rc;
    if (f32) launch(mingru_scan_kernel<float, GRU_OUTPUTS>, float());
    else launch(mingru_scan_kernel<bf16, GRU_OUTPUTS>, bf16());
    return bn_launch_status();
}
