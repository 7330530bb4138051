// gdn_verify.hip -- the gated-delta-rule recurrent verify: q_len[s] tokens of every stream
// through that stream's state of one linear-attention layer, in one launch.
//
// Per token, per group g and state row h (src/core/core_execution.cpp:254-335, the reference's
// GdnOperator::step_token; src/cuda/sixi_kernels.cu:241-281 is its CUDA twin):
//   sk = sum_s S[h][s] k[s]    (times alpha first with SIXI_GDN_DECAY_FIRST, ggml's order)
//   delta = beta * (v[h] - sk);   S[h][s] = alpha S[h][s] + delta k[s];   y[h] = sum_s S[h][s] q[s]
// The reference runs one launch per token and stream with the state in HBM; here the state of a
// (stream, group) is read once and written once (at the snapshot row), and a block of rows runs on
// chip.  Three kernels:
//
// gdn_verify_chunked_kernel (128-dim keys, states of 128 or 64 rows: the model's linear-attention
// layers hold 128 x 128) runs 16 rows at a time in the closed ("WY") form of the delta rule, on the f32 matrix
// cores; its comment below has the algebra and layout.  It is persistent: each work-group runs
// several (stream, group, 64-row half) items and reads half of the next item's state while it
// computes the current one.  Qwen verify batch (32 streams x 16 rows, 48 groups): 52.1-52.8 us
// against 64-65 us for the step by step kernel below; launching one item per work-group it
// measured 63.7 us (every work-group of a CU then loads, computes and stores in step), and without
// the XCD pairing of the two halves of a state 60.5 us.
//
// gdn_scan_kernel (the same shapes, while the work-groups fit the CUs at once: a prompt chunk, or a
// short block of one or a few streams) runs the chunks of a state as a pipeline; its comment has
// the split.
//
// gdn_verify_kernel (64-dim keys) steps token by token on the VALU with the state in registers;
// the decay alpha goes into a scalar factor of the carried state (S = cs * st, below), not into
// every element.  Two work-groups share each (stream, group) when the state has 128 rows, each
// owning half of the rows (the rows update independently; q, k, alpha and beta are staged by
// both).  At 128 x 128 this form took 101 registers (four waves per SIMD) and 62.9 us on the
// Qwen verify batch (the scalar factor took the element update from a multiply and an FMA to one
// FMA: 65.2 -> 62.9 us).
//
// Mapping of gdn_verify_kernel (256 threads): a thread holds R consecutive state rows x C = 16
// consecutive columns; the TPR = K/16 lanes that share the rows form a row group (adjacent lanes),
// whose partial dot products are summed by DPP lane moves (ds_bpermute shuffles measured 94
// against 83 us).  The block's tokens are staged through LDS TC at a time (q, k, v, alpha, beta of
// TC rows); every lane of a row group reads the same q/k columns, so those LDS reads are
// broadcasts.  y leaves from the row group's first lane as R floats.
//
// Roofline: the state dominates the bytes (2 * 4 Hd K per group and stream: read + write); each
// row adds 3 Hd K FMAs, so a block of n rows does 3n/8 FMA per state byte moved -- 6 FMA per byte
// for a 16-row verify block: above the 4.9 FMA per HBM byte of the unpacked FP32 VALU (78.6
// TFLOP/s against 8 TB/s), below the 9.8 of the f32 matrix cores (157.3 TFLOP/s).  Rounding differs from the step by
// step recurrence (sums in another order, the scalar factor, the closed form) at the level of f32
// rounding.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "device_util.hpp"
#include "gdn_internal.hpp"

namespace sixi {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kC = 16;   // state columns per thread
constexpr int kTC = 16;  // tokens staged per pass

// SPLIT work-groups share the HD rows of one (stream, group) state: the delta rule updates
// every row from its own values and the shared k, q, so the rows are independent.
template <int K, int HD, int SPLIT>
struct GdnShape {
    static constexpr int TPR = K / kC;         // lanes per row group
    static constexpr int GROUPS = 256 / TPR;   // row groups per block
    static constexpr int R = HD / SPLIT / GROUPS;  // state rows per thread
    static_assert(R >= 1 && GROUPS * R * SPLIT == HD, "shape");
};

// DPP lane moves (GFX9 encodings): quad_perm [1,0,3,2] and [2,3,0,1], row_half_mirror (lane i of
// each 8-lane half-row reads lane 7 - i)
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}

// Sum over the TPR (4 or 8) adjacent lanes of a row group, the total in every lane of it: two quad
// swaps give each quad its sum, and for 8 lanes the half-row mirror adds the other quad's.
template <int TPR>
__device__ __forceinline__ float group_sum(float v) {
    static_assert(TPR == 4 || TPR == 8, "row groups of 4 or 8 lanes");
    v += dpp<0xB1>(v);
    v += dpp<0x4E>(v);
    if constexpr (TPR == 8) v += dpp<0x141>(v);
    return v;
}

template <int K, int HD, int SPLIT, bool DECAY_FIRST>
__global__ __launch_bounds__(256) void gdn_verify_kernel(GdnArgs a) {
    using Sh = GdnShape<K, HD, SPLIT>;
    constexpr int R = Sh::R, TPR = Sh::TPR;
    constexpr int HR = HD / SPLIT;  // state rows of this work-group
    __shared__ f32x4 lq[kTC][K / 4], lk[kTC][K / 4];
    __shared__ float lv[kTC][HR], la[kTC], lb[kTC];

    const int g = (int)((blockIdx.x / SPLIT) % (unsigned)a.G);
    const int s = (int)((blockIdx.x / SPLIT) / (unsigned)a.G);
    const int hr0 = (int)(blockIdx.x % SPLIT) * HR;  // first state row of the work-group
    const int tid = threadIdx.x;
    const int part = tid % TPR;           // column block: columns part*16 .. part*16+15
    const int rw = (tid / TPR) * R;       // first state row of the thread, in the work-group's rows
    const int row0 = hr0 + rw;            // ... in the state
    int ql = a.q_len ? a.q_len[s] : a.n_rows;
    ql = ql < 0 ? 0 : (ql > a.n_rows ? a.n_rows : ql);
    int snap = a.snap ? a.snap[s] : ql;
    snap = snap < 0 ? 0 : (snap > ql ? ql : snap);

    // The state is carried as S = cs * st: a token's decay multiplies the scalar cs (the same in
    // every lane) instead of every element, and the element update is st += (delta / cs) k^T --
    // one FMA per element instead of a multiply and an FMA.  A token that takes cs outside
    // [2^-30, 2^30] (a gate near 0 or above 1, or not finite) folds it into st first.
    float st[R][kC];
    float cs = 1.0f;
    const char* sin_base = a.s_in + (int64_t)g * a.si_nb2 + (int64_t)s * a.si_nb3 + part * kC * 4;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int u = 0; u < kC / 4; ++u) {
            const f32x4 x = *reinterpret_cast<const f32x4*>(sin_base + (int64_t)(row0 + r) * a.si_nb1 + 16 * u);
#pragma unroll
            for (int e = 0; e < 4; ++e) st[r][4 * u + e] = x[e];
        }
    char* sout_base = a.s_out + (int64_t)g * a.so_nb2 + (int64_t)s * a.so_nb3 + part * kC * 4;
    auto write_state = [&]() {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int u = 0; u < kC / 4; ++u)
                *reinterpret_cast<f32x4*>(sout_base + (int64_t)(row0 + r) * a.so_nb1 + 16 * u) =
                    f32x4{st[r][4 * u], st[r][4 * u + 1], st[r][4 * u + 2], st[r][4 * u + 3]} * cs;
    };
    if (snap == 0) write_state();

    for (int t0 = 0; t0 < ql; t0 += kTC) {
        const int nt = ql - t0 < kTC ? ql - t0 : kTC;
        // stage q, k (K/4 vectors per row), v (HD/4), alpha, beta of rows t0 .. t0+nt-1
        for (int i = tid; i < nt * (K / 4); i += 256) {
            const int t = i / (K / 4), c = i % (K / 4);
            const int64_t off = (int64_t)g * a.q_nb1 + (int64_t)(t0 + t) * a.q_nb2 + (int64_t)s * a.q_nb3 + 16 * c;
            lq[t][c] = *reinterpret_cast<const f32x4*>(a.q + off);
            const int64_t offk = (int64_t)g * a.k_nb1 + (int64_t)(t0 + t) * a.k_nb2 + (int64_t)s * a.k_nb3 + 16 * c;
            lk[t][c] = *reinterpret_cast<const f32x4*>(a.k + offk);
        }
        for (int i = tid; i < nt * (HR / 4); i += 256) {
            const int t = i / (HR / 4), c = i % (HR / 4);
            const f32x4 x = *reinterpret_cast<const f32x4*>(a.v + (int64_t)g * a.v_nb1 + (int64_t)(t0 + t) * a.v_nb2 +
                                                            (int64_t)s * a.v_nb3 + 4 * hr0 + 16 * c);
#pragma unroll
            for (int e = 0; e < 4; ++e) lv[t][4 * c + e] = x[e];
        }
        if (tid < nt) {
            la[tid] = *reinterpret_cast<const float*>(a.alpha + (int64_t)g * a.a_nb0 + (int64_t)(t0 + tid) * a.a_nb1 +
                                                      (int64_t)s * a.a_nb2);
            lb[tid] = *reinterpret_cast<const float*>(a.beta + (int64_t)g * a.b_nb0 + (int64_t)(t0 + tid) * a.b_nb1 +
                                                      (int64_t)s * a.b_nb2);
        }
        __syncthreads();
#pragma unroll 1
        for (int t = 0; t < nt; ++t) {
            float kv[kC], qv[kC];
#pragma unroll
            for (int u = 0; u < kC / 4; ++u) {
                const f32x4 x = lk[t][part * (kC / 4) + u];
#pragma unroll
                for (int e = 0; e < 4; ++e) kv[4 * u + e] = x[e];
            }
            const float al = la[t], be = lb[t];
            // the factor after the token's decay; outside [2^-30, 2^30] (or not finite) the token
            // folds it into st and the factor returns to 1 (the same in every lane)
            const float cn = cs * al;
            const bool fold = !(cn >= 0x1p-30f && cn <= 0x1p30f);
            // S k with the state before the token (decayed first: after it)
            float sk[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float x = 0.0f;
#pragma unroll
                for (int c = 0; c < kC; ++c) x += st[r][c] * kv[c];
                sk[r] = group_sum<TPR>(x) * (DECAY_FIRST ? cn : cs);
            }
            if (fold) {
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int c = 0; c < kC; ++c) st[r][c] *= cn;
            }
            cs = fold ? 1.0f : cn;
            const float bi = be / cs;
            // (q is read once the fold is done: fewer registers live across it)
#pragma unroll
            for (int u = 0; u < kC / 4; ++u) {
                const f32x4 y = lq[t][part * (kC / 4) + u];
#pragma unroll
                for (int e = 0; e < 4; ++e) qv[4 * u + e] = y[e];
            }
            float yo[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float dn = bi * (lv[t][rw + r] - sk[r]);
                float yv = 0.0f;
#pragma unroll
                for (int c = 0; c < kC; ++c) {
                    st[r][c] = fmaf(dn, kv[c], st[r][c]);
                    yv += st[r][c] * qv[c];
                }
                yo[r] = group_sum<TPR>(yv) * cs;
            }
            if (part == 0) {
                char* yp = a.y + (int64_t)g * a.y_nb1 + (int64_t)(t0 + t) * a.y_nb2 + (int64_t)s * a.y_nb3 + row0 * 4;
                if constexpr (R == 4)
                    *reinterpret_cast<f32x4*>(yp) = f32x4{yo[0], yo[1], yo[2], yo[3]};
                else
#pragma unroll
                    for (int r = 0; r < R; ++r) reinterpret_cast<float*>(yp)[r] = yo[r];
            }
            if (t0 + t + 1 == snap) write_state();
        }
        __syncthreads();  // the next pass overwrites the staged rows
    }
}

// ---------------------------------------------------------------------------------------------
// Chunked form on the f32 matrix cores (128-dim keys).  Over a chunk of T = 16 rows the T steps
// of the recurrence are one closed form (the "WY" / "UT" form of the delta rule; every quantity
// below is exact in exact arithmetic, the step by step loop is the definition):
//   A_t = alpha_0 ... alpha_t,   E[t][s] = alpha_{s+1} ... alpha_t (s <= t, 1 at s = t)
//   P = S0 k^T, Z = S0 q^T       (S0 the state before the chunk; P, Z are Hd x T)
//   c_t = A_{t-1} (A_{-1} = 1), or A_t when the decay comes first (ggml's order)
//   L[t][s] = beta_t e(t, s) (k_s . k_t) for s < t, e(t, s) = E[t-1][s] (E[t][s] decay-first)
//   R[h][t] = beta_t (v_t[h] - c_t P[h][t]);  U = R (I + L)^-T  (U[h][t] is token t's delta)
//   y_t[h] = A_t Z[h][t] + sum_{s<=t} U[h][s] E[t][s] (k_s . q_t)
//   S_sigma = A_sigma S0 + sum_{s<=sigma} E[sigma][s] U[:, s] k_s^T
// so a chunk costs the products P and Z (Hd x 128 by 128 x 16 each), one Hd x 16 by 16 x 128
// product per state it writes or carries, k k^T and k q^T (16 x 128 by 128 x 16, shared by the
// work-group) and 16 x 16 work -- the step by step form's 3 Hd K FMAs per row, on the matrix cores
// at twice the unpacked VALU rate.  No gate product spans more than one chunk (the carried state
// is the plain matrix), so the gates' range is that of the step by step recurrence.
//
// Layout: a work-group owns 64 state rows (HD / 64 work-groups per state), wave w rows 16w ..
// 16w+15.  v_mfma_f32_16x16x4f32: lane l supplies A[l%16][l/16] and B[l/16][l%16] and holds
// D[4(l/16) + r][l%16] in register r.  Lane l = 16 gl + lr holds state row lr of its wave, columns
// 16 m + 4 gl + j in register 4 m + j (m = 0..7, j = 0..3): read as eight 16-byte pieces, and at the
// same time the B operand of P^T = k S0^T (k-index 16 m + 4 gl + j at step (m, j)) and the output
// layout of S^T = k^T U'^T whose tile m covers columns 16 m .. 16 m + 15 -- so the state never
// leaves registers between chunks.
constexpr int kCT = 16;    // rows per chunk
constexpr int kCP = 132;   // LDS pitch (floats) of staged k, q rows: 16-byte reads of 8 rows hit distinct banks

__device__ __forceinline__ f32x4 mma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <int HD, bool DECAY_FIRST>
__global__ __launch_bounds__(256) void gdn_verify_chunked_kernel(GdnArgs a, int n_items, int pair) {
    constexpr int K = 128, HR = 64, SPLIT = HD / HR, T = kCT;
    static_assert(HD % HR == 0, "64 state rows per work-group");
    __shared__ __align__(16) float lk[T][kCP], lq[T][kCP];
    __shared__ __align__(16) float lv[T][HR];
    __shared__ __align__(16) float la[T], lb[T];
    __shared__ __align__(16) float lE[T][T];          // E[t][s], 0 for s > t
    __shared__ __align__(16) float lred[4][2][T][T];  // per wave: partial k k^T, k q^T over 32 columns
    __shared__ __align__(16) float lLT[T][T];         // lLT[s][t] = L[t][s]
    __shared__ __align__(16) float lWT[T][T];         // lWT[t][s] = E[t][s] (k_s . q_t)

    const int tid = threadIdx.x;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int gl0 = (tid >> 4) & 3;  // the lane's group: columns 16 m + 4 gl0 .. + 3 of its state row
    // Work item x = 64 rows of one (stream, group) state.  With pair set (two items per state,
    // states a multiple of 8) items x and x + 8 are the two halves of one state: launched
    // round-robin over the 8 XCDs by work-groups b and b + 8, they share the XCD's L2 for the
    // state's q and k rows.
    auto locate = [&](int x, int& g, int& s, int& hr0) {
        int state, half;
        if (pair) {
            state = ((x >> 3) >> 1) * 8 + (x & 7);
            half = (x >> 3) & 1;
        } else {
            state = x / SPLIT;
            half = x % SPLIT;
        }
        g = state % a.G;
        s = state / a.G;
        hr0 = half * HR;
    };
    auto load_state = [&](int x, float (&dst)[32]) {
        int g, s, hr0;
        locate(x, g, s, hr0);
        const char* p = a.s_in + (int64_t)g * a.si_nb2 + (int64_t)s * a.si_nb3 +
                        (int64_t)(hr0 + 16 * wv + (tid & 15)) * a.si_nb1 + 16 * gl0;
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const f32x4 v4 = *reinterpret_cast<const f32x4*>(p + 64 * m);
#pragma unroll
            for (int j = 0; j < 4; ++j) dst[4 * m + j] = v4[j];
        }
    };
    // columns 16 m0 .. 16 m0 + 63 of item x's state rows (registers 4 m0 .. 4 m0 + 15 of st)
    auto load_half = [&](int x, int m0, float* dst) {
        int g, s, hr0;
        locate(x, g, s, hr0);
        const char* p = a.s_in + (int64_t)g * a.si_nb2 + (int64_t)s * a.si_nb3 +
                        (int64_t)(hr0 + 16 * wv + (tid & 15)) * a.si_nb1 + 16 * gl0;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const f32x4 v4 = *reinterpret_cast<const f32x4*>(p + 64 * (m0 + m));
#pragma unroll
            for (int j = 0; j < 4; ++j) dst[4 * m + j] = v4[j];
        }
    };

    // A work-group runs items blockIdx.x, + gridDim.x, ...: the first half of the next item's state
    // (columns 0 .. 63) is read into nst while this item's chunks run, so a work-group's state
    // transfers overlap its own matrix-core work (launched one item per work-group, all of a CU's
    // work-groups load, compute and store in step: 63.7 against 55 us on the verify batch).  The
    // other half is read at the item's start: registers for all of it (148 VGPRs) leave three
    // work-groups per CU, with half of it (125) four fit (54.5 -> 52.8 us).
    float st[32], nst[16];
    load_state(blockIdx.x, st);
    bool first = true;
    for (int x = blockIdx.x; x < n_items; x += gridDim.x) {
        if (!first) load_half(x, 4, st + 16);  // the half not read ahead
        first = false;
        int g, s, hr0;
        locate(x, g, s, hr0);
        const int xn = x + (int)gridDim.x;
        const int h = hr0 + 16 * wv + (tid & 15);  // this lane's state row
        int ql = a.q_len ? a.q_len[s] : a.n_rows;
        ql = ql < 0 ? 0 : (ql > a.n_rows ? a.n_rows : ql);
        int snap = a.snap ? a.snap[s] : ql;
        snap = snap < 0 ? 0 : (snap > ql ? ql : snap);

        char* const sout = a.s_out + (int64_t)g * a.so_nb2 + (int64_t)s * a.so_nb3 + (int64_t)h * a.so_nb1 + 16 * gl0;
        if (snap == 0) {
#pragma unroll
            for (int m = 0; m < 8; ++m)
                *reinterpret_cast<f32x4*>(sout + 64 * m) =
                    f32x4{st[4 * m], st[4 * m + 1], st[4 * m + 2], st[4 * m + 3]};
        }
        if (ql == 0 && xn < n_items) load_half(xn, 0, nst);

        for (int t0 = 0; t0 < ql; t0 += T) {
            const int nt = ql - t0 < T ? ql - t0 : T;
            // the lane's LDS addresses and constants are derived anew in every chunk (an opaque copy
            // of the thread index): hoisted out of the loop they would hold some 60 VGPRs
            int tx;
            asm volatile("v_mov_b32 %0, %1" : "=v"(tx) : "v"(tid));
            const int lr = tx & 15, gl = (tx >> 4) & 3, hw = 16 * wv + lr;
            // stage rows t0 .. t0+nt-1; rows past nt are zero keys, queries and values with gate 1 and
            // beta 0, which leave the state and every other row's result unchanged
            for (int i = tx; i < T * (K / 4); i += 256) {
                const int t = i / (K / 4), c = i % (K / 4);
                f32x4 kx = {0.0f, 0.0f, 0.0f, 0.0f}, qx = kx;
                if (t < nt) {
                    kx = *reinterpret_cast<const f32x4*>(a.k + (int64_t)g * a.k_nb1 + (int64_t)(t0 + t) * a.k_nb2 +
                                                         (int64_t)s * a.k_nb3 + 16 * c);
                    qx = *reinterpret_cast<const f32x4*>(a.q + (int64_t)g * a.q_nb1 + (int64_t)(t0 + t) * a.q_nb2 +
                                                         (int64_t)s * a.q_nb3 + 16 * c);
                }
                *reinterpret_cast<f32x4*>(&lk[t][4 * c]) = kx;
                *reinterpret_cast<f32x4*>(&lq[t][4 * c]) = qx;
            }
            for (int i = tx; i < T * (HR / 4); i += 256) {
                const int t = i / (HR / 4), c = i % (HR / 4);
                f32x4 vx = {0.0f, 0.0f, 0.0f, 0.0f};
                if (t < nt)
                    vx = *reinterpret_cast<const f32x4*>(a.v + (int64_t)g * a.v_nb1 + (int64_t)(t0 + t) * a.v_nb2 +
                                                         (int64_t)s * a.v_nb3 + 4 * hr0 + 16 * c);
                *reinterpret_cast<f32x4*>(&lv[t][4 * c]) = vx;
            }
            if (tx < T) {
                const int64_t ra = (int64_t)g * a.a_nb0 + (int64_t)(t0 + tx) * a.a_nb1 + (int64_t)s * a.a_nb2;
                const int64_t rb = (int64_t)g * a.b_nb0 + (int64_t)(t0 + tx) * a.b_nb1 + (int64_t)s * a.b_nb2;
                la[tx] = tx < nt ? *reinterpret_cast<const float*>(a.alpha + ra) : 1.0f;
                lb[tx] = tx < nt ? *reinterpret_cast<const float*>(a.beta + rb) : 0.0f;
            }
            __syncthreads();
            if (t0 == 0 && xn < n_items) load_half(xn, 0, nst);  // in flight during this item's work

            // E[t][s], one entry per thread, multiplied in row order
            {
                const int et = tx >> 4, es = tx & 15;
                f32x4 a4[T / 4];  // every gate of the chunk (the same address in every lane)
#pragma unroll
                for (int u = 0; u < T / 4; ++u) a4[u] = *reinterpret_cast<const f32x4*>(&la[4 * u]);
                float e = 1.0f;
#pragma unroll
                for (int r = 1; r < T; ++r)
                    if (r > es && r <= et) e *= a4[r / 4][r % 4];
                lE[et][es] = es <= et ? e : 0.0f;
            }
            // P^T = k S0^T and Z^T = q S0^T (lane: P[h][4 gl + j] in register j); wave w also sums
            // k k^T and k q^T over columns 32 w .. 32 w + 31
            f32x4 pt = {0.0f, 0.0f, 0.0f, 0.0f}, zt = pt, gk = pt, gq = pt;
            // (raised wave priority while this wave issues the products: 55.0 -> 53.6-53.9 us on the
            // verify batch; raised around the state's product as well, 54.5 us)
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const f32x4 kx = *reinterpret_cast<const f32x4*>(&lk[lr][16 * m + 4 * gl]);
                const f32x4 qx = *reinterpret_cast<const f32x4*>(&lq[lr][16 * m + 4 * gl]);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    pt = mma4(kx[j], st[4 * m + j], pt);
                    zt = mma4(qx[j], st[4 * m + j], zt);
                }
                if ((m >> 1) == wv) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        gk = mma4(kx[j], kx[j], gk);
                        gq = mma4(kx[j], qx[j], gq);
                    }
                }
            }
            __builtin_amdgcn_s_setprio(0);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                lred[wv][0][4 * gl + r][lr] = gk[r];  // k_{4gl+r} . k_lr, partial
                lred[wv][1][4 * gl + r][lr] = gq[r];  // k_{4gl+r} . q_lr, partial
            }
            __syncthreads();

            // L and W, one entry per thread: row ta, column tb
            {
                const int ta = tx >> 4, tb = tx & 15;
                const float kk = lred[0][0][tb][ta] + lred[1][0][tb][ta] + lred[2][0][tb][ta] + lred[3][0][tb][ta];
                const float kq = lred[0][1][tb][ta] + lred[1][1][tb][ta] + lred[2][1][tb][ta] + lred[3][1][tb][ta];
                float l = 0.0f;
                if (tb < ta) l = lb[ta] * (DECAY_FIRST ? lE[ta][tb] : lE[ta - 1][tb]) * kk;
                lLT[tb][ta] = l;                  // L[ta][tb]
                lWT[ta][tb] = lE[ta][tb] * kq;    // E[ta][tb] (k_tb . q_ta), 0 for tb > ta
            }
            __syncthreads();

            // row lr of M = (I + L)^-1 by back substitution: M[s][t] = [s = t] - sum_{r>t} M[s][r] L[r][t]
            // (row t - 1 of lLT is read while row t is used; the empty asm pins each step in place,
            // else the compiler reads all 36 pieces up front into 144 VGPRs)
            float mr[T];
            mr[T - 1] = lr == T - 1 ? 1.0f : 0.0f;
            f32x4 cur[T / 4], nxt[T / 4];
#pragma unroll
            for (int c = (T - 1) / 4; c < T / 4; ++c) cur[c] = *reinterpret_cast<const f32x4*>(&lLT[T - 2][4 * c]);
#pragma unroll
            for (int t = T - 2; t >= 0; --t) {
                if (t > 0) {
#pragma unroll
                    for (int c = t / 4; c < T / 4; ++c) nxt[c] = *reinterpret_cast<const f32x4*>(&lLT[t - 1][4 * c]);
                }
                float x = lr == t ? 1.0f : 0.0f;
#pragma unroll
                for (int c = (t + 1) / 4; c < T / 4; ++c)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (4 * c + e > t) x = fmaf(-mr[4 * c + e], cur[c][e], x);
                asm volatile("" : "+v"(x) : : "memory");
                mr[t] = x;
#pragma unroll
                for (int c = 0; c < T / 4; ++c) cur[c] = nxt[c];
            }
            // R[h][4 gl + j] and U^T = M R^T (lane: U[h][4 gl + j] in register j)
            const float a0 = la[0];
            f32x4 ut = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int t = 4 * gl + j;
                const float ct = DECAY_FIRST ? lE[t][0] * a0 : (t ? lE[t - 1][0] * a0 : 1.0f);
                const float rv = lb[t] * (lv[t][hw] - ct * pt[j]);
                const float mv = gl == 0 ? mr[j] : gl == 1 ? mr[4 + j] : gl == 2 ? mr[8 + j] : mr[12 + j];
                ut = mma4(mv, rv, ut);
            }
            // y^T = diag(A) Z^T + W^T U^T
            {
                f32x4 yt;
#pragma unroll
                for (int j = 0; j < 4; ++j) yt[j] = lE[4 * gl + j][0] * a0 * zt[j];
                const f32x4 wx = *reinterpret_cast<const f32x4*>(&lWT[lr][4 * gl]);
#pragma unroll
                for (int j = 0; j < 4; ++j) yt = mma4(wx[j], ut[j], yt);
                char* yp = a.y + (int64_t)g * a.y_nb1 + (int64_t)(t0 + 4 * gl) * a.y_nb2 + (int64_t)s * a.y_nb3 + h * 4;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (4 * gl + j < nt) *reinterpret_cast<float*>(yp + (int64_t)j * a.y_nb2) = yt[j];
            }
            // S_sigma = A_sigma S0 + k^T (U E[sigma])^T, tile by tile; written to the snapshot and/or
            // kept as the next chunk's S0
            const bool more = t0 + T < ql;
            const bool snap_here = snap > t0 && snap <= t0 + nt;
            auto advance = [&](int sig, bool write, bool keep) {
                const float as = lE[sig][0] * a0;
                float ub[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) ub[j] = ut[j] * lE[sig][4 * gl + j];
#pragma unroll
                for (int m = 0; m < 8; ++m) {
                    f32x4 acc = f32x4{st[4 * m], st[4 * m + 1], st[4 * m + 2], st[4 * m + 3]} * as;
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc = mma4(lk[4 * gl + j][16 * m + lr], ub[j], acc);
                    if (write) *reinterpret_cast<f32x4*>(sout + 64 * m) = acc;
                    if (keep) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) st[4 * m + j] = acc[j];
                    }
                }
            };
            if (snap_here) advance(snap - 1 - t0, true, more && snap == t0 + T);
            if (more && !(snap_here && snap == t0 + T)) advance(T - 1, false, true);
            if (more) __syncthreads();  // the next chunk overwrites the staged rows
        }
        __syncthreads();  // the next item overwrites the staged rows
#pragma unroll
        for (int i = 0; i < 16; ++i) st[i] = nst[i];
    }
}

// ---------------------------------------------------------------------------------------------
// Long blocks of few streams (a prompt chunk): the chunks of a state are a serial chain, and one
// chain per 64 state rows leaves most of the chip idle.  The chunked kernel above spends 5.8 us per
// chunk there (one stream, 48 groups, 2048 rows: 741 us), of which the matrix cores need 1.6: each
// chunk's loads, Gram products, triangular inverse and state products run one after another.
//
// Here a work-group of eight waves owns 32 state rows (HD / 32 work-groups per state) and runs the
// same algebra as a pipeline over the chunks, an iteration in two halves with a barrier after each:
//   waves 0..3 (consumers) take chunk i: wave = 16 state rows x 64 columns, so P = S0 k^T and
//     Z = S0 q^T are half sums, exchanged through LDS between the halves; then U, y and the state's
//     update, whose operands were read in the first half;
//   waves 4..7 (producers) prepare what does not depend on the state.  Second half: waves 4, 5 hold
//     k (64 columns each) of chunk i + 3 in registers, put it into LDS and sum k k^T, waves 6, 7
//     the same with q and k q^T.  First half: wave 4 makes L and wave 6 makes W of chunk i + 2,
//     wave 7 stages v, the gates and their products E of chunk i + 3, wave 5 inverts I + L of chunk
//     i + 1.  Each issues the global loads of its chunk two iterations ahead.
// Every SIMD holds one consumer and one producer, whose 56 and 16 f32 MFMAs (32 cycles each; wave 5's
// 32, with the inverse) per iteration are its floor: 2816 cycles on the busiest SIMD, 150 us over the 128
// chunks of 2048 rows, which take 307 us (a call; 739 with the chunked kernel).  Before each producer wave had a loop of its own it took 325
// in graph replays, of which the producers switched off left 219 (the consumers' chain P -> exchange
// -> U -> state); the inversion was 35 of it, the staging loads 28, E 27, k k^T and k q^T 24.
constexpr int kScanRows = 32;

struct GdnScanLds {
    float k[3][kCT][kCP], q[3][kCT][kCP];  // chunk c at c % 3
    float v[4][kCT][kScanRows];            // chunk c at c % 4 (E, A, C, B, W alike)
    float E[4][kCT][kCT];                  // E[t][s], 0 for s > t
    float A[4][kCT], C[4][kCT], B[4][kCT]; // A_t, c_t, beta_t
    float W[4][kCT][kCT];                  // W[t][s] = E[t][s] (k_s . q_t)
    float L[2][kCT][kCT], M[2][kCT][kCT];  // chunk c at c % 2; M = (I + L)^-1
    f32x4 P[4][64], Z[2][64];              // half sums of the consumers (Z: of the upper columns)
    f32x4 G[2][64];                        // half sums of the Gram products (upper columns)
};

// Work-group barrier for LDS traffic: global loads stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <int HD, bool DECAY_FIRST>
__global__ __launch_bounds__(512) void gdn_scan_kernel(GdnArgs a, int grouped) {
    constexpr int K = 128, T = kCT, SPLIT = HD / kScanRows;
    static_assert(HD % kScanRows == 0 && K == 2 * 64, "two column halves");
    __shared__ __align__(16) GdnScanLds sh;

    // the work-groups of one state read the same q and k: with `grouped` (states a multiple of 8)
    // they are dealt to one XCD
    const int b = blockIdx.x;
    const int state = grouped ? (b >> 3) / SPLIT * 8 + (b & 7) : b / SPLIT;
    const int hr0 = ((grouped ? b >> 3 : b) % SPLIT) * kScanRows;
    const int g = state % a.G, s = state / a.G;
    int ql = a.q_len ? a.q_len[s] : a.n_rows;
    ql = ql < 0 ? 0 : (ql > a.n_rows ? a.n_rows : ql);
    int snap = a.snap ? a.snap[s] : ql;
    snap = snap < 0 ? 0 : (snap > ql ? ql : snap);
    const int n_chunks = (ql + T - 1) / T;

    const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, lr = lane & 15, gl = lane >> 4;

    if (wv < 4) {
        const int kh = wv & 1;                    // column half
        const int hw = 16 * (wv >> 1) + lr;       // the lane's state row in the work-group
        const int h = hr0 + hw;
        const int64_t col = 256 * kh + 16 * gl;   // bytes
        const char* const sin = a.s_in + (int64_t)g * a.si_nb2 + (int64_t)s * a.si_nb3 + (int64_t)h * a.si_nb1 + col;
        char* const sout = a.s_out + (int64_t)g * a.so_nb2 + (int64_t)s * a.so_nb3 + (int64_t)h * a.so_nb1 + col;
        f32x4 st[4];  // columns 64 kh + 16 m + 4 gl + j in st[m][j]
#pragma unroll
        for (int m = 0; m < 4; ++m) st[m] = *reinterpret_cast<const f32x4*>(sin + 64 * m);
        if (snap == 0) {
#pragma unroll
            for (int m = 0; m < 4; ++m) *reinterpret_cast<f32x4*>(sout + 64 * m) = st[m];
        }
        char* const yb = a.y + (int64_t)g * a.y_nb1 + (int64_t)s * a.y_nb3 + (int64_t)h * 4;
        // rows lr of k and q of the chunk ahead, as P's and Z's A operands
        f32x4 kx[4], qx[4];
        auto read_rows = [&](int c) {
            const int b3 = c % 3;
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                kx[m] = *reinterpret_cast<const f32x4*>(&sh.k[b3][lr][64 * kh + 16 * m + 4 * gl]);
                qx[m] = *reinterpret_cast<const f32x4*>(&sh.q[b3][lr][64 * kh + 16 * m + 4 * gl]);
            }
        };
        for (int i = -3; i < 0; ++i) {
            lds_barrier();
            if (i == -1 && n_chunks > 0) read_rows(0);
            lds_barrier();
        }
        for (int i = 0; i < n_chunks; ++i) {
            const int b3 = i % 3, b4 = i & 3;
            const int t0 = i * T, nt = ql - t0 < T ? ql - t0 : T;
            const bool more = t0 + T < ql;
            const bool snap_here = snap > t0 && snap <= t0 + nt;
            // what the second half needs of the producers' work
            float ka[4][4], vv[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                vv[j] = sh.v[b4][4 * gl + j][hw];
#pragma unroll
                for (int m = 0; m < 4; ++m) ka[m][j] = sh.k[b3][4 * gl + j][64 * kh + 16 * m + lr];
            }
            const f32x4 mx = *reinterpret_cast<const f32x4*>(&sh.M[i & 1][lr][4 * gl]);
            const f32x4 wx = *reinterpret_cast<const f32x4*>(&sh.W[b4][lr][4 * gl]);
            const f32x4 ax = *reinterpret_cast<const f32x4*>(&sh.A[b4][4 * gl]);
            const f32x4 cx = *reinterpret_cast<const f32x4*>(&sh.C[b4][4 * gl]);
            const f32x4 bx = *reinterpret_cast<const f32x4*>(&sh.B[b4][4 * gl]);
            const f32x4 el = *reinterpret_cast<const f32x4*>(&sh.E[b4][T - 1][4 * gl]);
            const float al = sh.A[b4][T - 1];
            f32x4 pt[2], zt[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) pt[u] = zt[u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    pt[m & 1] = mma4(kx[m][j], st[m][j], pt[m & 1]);
                    zt[m & 1] = mma4(qx[m][j], st[m][j], zt[m & 1]);
                }
            f32x4 p = pt[0] + pt[1];
            const f32x4 z = zt[0] + zt[1];
            sh.P[wv][lane] = p;
            if (kh) sh.Z[wv >> 1][lane] = z;
            lds_barrier();
            p += sh.P[wv ^ 1][lane];
            const f32x4 zp = sh.Z[wv >> 1][lane];
            if (more) read_rows(i + 1);
            // U^T = M R^T (lane: U[h][4 gl + j] in register j)
            f32x4 ut = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int j = 0; j < 4; ++j) ut = mma4(mx[j], bx[j] * (vv[j] - cx[j] * p[j]), ut);
            if (snap_here) {
                // S_sigma = A_sigma S0 + k^T (U E[sigma])^T, to the output state
                const int sig = snap - 1 - t0;
                const float as = sh.A[b4][sig];
                const f32x4 ub = ut * *reinterpret_cast<const f32x4*>(&sh.E[b4][sig][4 * gl]);
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    f32x4 acc = st[m] * as;
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc = mma4(ka[m][j], ub[j], acc);
                    *reinterpret_cast<f32x4*>(sout + 64 * m) = acc;
                }
            }
            // the next chunk's S0 (sigma = T - 1; unused after the last chunk) and, between its
            // MFMAs, y^T = diag(A) Z^T + W^T U^T (kept by the lower columns' wave)
            const f32x4 ub = ut * el;
            f32x4 yt = ax * (z + zp);
#pragma unroll
            for (int m = 0; m < 4; ++m) st[m] *= al;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int m = 0; m < 4; ++m) st[m] = mma4(ka[m][j], ub[j], st[m]);
                yt = mma4(wx[j], ut[j], yt);
            }
            if (!kh) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (4 * gl + j < nt) *reinterpret_cast<float*>(yb + (int64_t)(t0 + 4 * gl + j) * a.y_nb2) = yt[j];
            }
            lds_barrier();
        }
        return;
    }

    // ---- producers ---- (one loop for each wave: a common one holds more than the SGPRs)
    auto produce = [&](auto PW) {
        constexpr int pw = decltype(PW)::value, half = pw & 1;
        constexpr bool is_q = pw >= 2;
        const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
        const char* const kb = a.k + (int64_t)g * a.k_nb1 + (int64_t)s * a.k_nb3 + 256 * half + 16 * gl;
        const char* const qb = a.q + (int64_t)g * a.q_nb1 + (int64_t)s * a.q_nb3 + 256 * half + 16 * gl;
        // a chunk in registers: row lr, columns 64 half + 16 m + 4 gl .. + 3 (zeros past the block); in
        // wave 7 also the gates of row lr (1 and 0 past the block) and rows lane / 8, 8 + lane / 8 of v
        struct Chunk {
            f32x4 k[4], q[4], v[2];
            float al, be;
        };
        auto load_rows = [&](int c, Chunk& x) {
            const int t = c * T + lr;
#pragma unroll
            for (int m = 0; m < 4; ++m) x.k[m] = x.q[m] = zero;
            if (t < ql) {
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    x.k[m] = *reinterpret_cast<const f32x4*>(kb + (int64_t)t * a.k_nb2 + 64 * m);
                    if (is_q) x.q[m] = *reinterpret_cast<const f32x4*>(qb + (int64_t)t * a.q_nb2 + 64 * m);
                }
            }
        };
        auto load_gates = [&](int c, Chunk& x) {
            const int t = c * T + lr;
            x.al = 1.0f;
            x.be = 0.0f;
            if (t < ql) {
                x.al = *reinterpret_cast<const float*>(a.alpha + (int64_t)g * a.a_nb0 + (int64_t)t * a.a_nb1 + (int64_t)s * a.a_nb2);
                x.be = *reinterpret_cast<const float*>(a.beta + (int64_t)g * a.b_nb0 + (int64_t)t * a.b_nb1 + (int64_t)s * a.b_nb2);
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int tv = c * T + 8 * u + (lane >> 3);
                x.v[u] = zero;
                if (tv < ql)
                    x.v[u] = *reinterpret_cast<const f32x4*>(a.v + (int64_t)g * a.v_nb1 + (int64_t)tv * a.v_nb2 +
                                                             (int64_t)s * a.v_nb3 + 4 * hr0 + 16 * (lane & 7));
            }
        };
        // M = (I + L)^-1 by blocks: the 4 x 4 diagonal blocks in closed form (D), then twice
        // M <- M - M Lo M with Lo the blocks below the diagonal of the doubled blocks, on the matrix
        // cores (elimination row by row in one wave took 0.6 us of a 2.8 us iteration).  A product's
        // accumulator layout is its B operand's: lane = column lr, rows 4 gl + j.
        auto invert = [&](float (&L)[T][T], float (&M)[T][T]) {
            const int bk = lr >> 2, p = lr & 3;
            const f32x4 l1 = *reinterpret_cast<const f32x4*>(&L[4 * bk + 1][4 * bk]);
            const f32x4 l2 = *reinterpret_cast<const f32x4*>(&L[4 * bk + 2][4 * bk]);
            const f32x4 l3 = *reinterpret_cast<const f32x4*>(&L[4 * bk + 3][4 * bk]);
            const f32x4 lx = *reinterpret_cast<const f32x4*>(&L[lr][4 * gl]);
            const float m10 = -l1[0], m21 = -l2[1], m32 = -l3[2];
            const float m20 = -fmaf(l2[1], m10, l2[0]), m31 = -fmaf(l3[2], m21, l3[1]);
            const float m30 = -fmaf(l3[2], m20, fmaf(l3[1], m10, l3[0]));
            const bool diag = gl == bk;
            f32x4 row = p == 0 ? f32x4{1.0f, 0.0f, 0.0f, 0.0f} : p == 1 ? f32x4{m10, 1.0f, 0.0f, 0.0f}
                      : p == 2 ? f32x4{m20, m21, 1.0f, 0.0f} : f32x4{m30, m31, m32, 1.0f};
            f32x4 col = p == 0 ? f32x4{1.0f, m10, m20, m30} : p == 1 ? f32x4{0.0f, 1.0f, m21, m31}
                      : p == 2 ? f32x4{0.0f, 0.0f, 1.0f, m32} : f32x4{0.0f, 0.0f, 0.0f, 1.0f};
            row = diag ? row : zero;  // D[lr][4 gl + j]
            col = diag ? col : zero;  // D[4 gl + j][lr]
            const f32x4 lo4 = gl + 1 == bk && (bk & 1) ? lx : zero;
            const f32x4 lo8 = gl < 2 && bk >= 2 ? lx : zero;
            f32x4 x = zero, m8 = col;
#pragma unroll
            for (int j = 0; j < 4; ++j) x = mma4(lo4[j], col[j], x);
#pragma unroll
            for (int j = 0; j < 4; ++j) m8 = mma4(-row[j], x[j], m8);
#pragma unroll
            for (int j = 0; j < 4; ++j) M[4 * gl + j][lr] = m8[j];
            x = zero;
#pragma unroll
            for (int j = 0; j < 4; ++j) x = mma4(lo8[j], m8[j], x);
            const f32x4 mrow = *reinterpret_cast<const f32x4*>(&M[lr][4 * gl]);
            f32x4 m16 = m8;
#pragma unroll
            for (int j = 0; j < 4; ++j) m16 = mma4(-mrow[j], x[j], m16);
#pragma unroll
            for (int j = 0; j < 4; ++j) M[4 * gl + j][lr] = m16[j];
        };
        f32x4 gr = zero;  // this wave's Gram product of chunk i + 2, then of chunk i + 3
        // iteration i; x holds chunk i + 3 and takes chunk i + 5
        auto iteration = [&](int i, Chunk& x) {
            if (half == 0 && i + 2 >= 0 && i + 2 < n_chunks) {
                const int b4 = (i + 2) & 3, b2 = i & 1;
                gr += sh.G[is_q][lane];  // k_{4gl+r} . k_lr (or . q_lr)
                if (is_q) {
                    const f32x4 ex = *reinterpret_cast<const f32x4*>(&sh.E[b4][lr][4 * gl]);
                    *reinterpret_cast<f32x4*>(&sh.W[b4][lr][4 * gl]) = ex * gr;  // 0 past the diagonal
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int t = 4 * gl + r;
                        float l = 0.0f;
                        if (lr < t) l = sh.B[b4][t] * (DECAY_FIRST ? sh.E[b4][t][lr] : sh.E[b4][t - 1][lr]) * gr[r];
                        sh.L[b2][t][lr] = l;
                    }
                }
            }
            if (pw == 1 && i + 1 >= 0 && i + 1 < n_chunks) invert(sh.L[(i + 1) & 1], sh.M[(i + 1) & 1]);
            const bool on = i + 3 < n_chunks;
            if (pw == 3 && on) {
                const int b4 = (i + 3) & 3;
#pragma unroll
                for (int u = 0; u < 2; ++u) *reinterpret_cast<f32x4*>(&sh.v[b4][8 * u + (lane >> 3)][4 * (lane & 7)]) = x.v[u];
                // column lr of E, multiplied in row order; this lane's rows 4 gl .. + 3
                float e = 1.0f, ev[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                const int ai = __builtin_bit_cast(int, x.al);
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    const float at = __builtin_bit_cast(float, __builtin_amdgcn_readlane(ai, t));
                    if (t > lr) e *= at;
                    if (gl == t / 4) ev[t % 4] = t >= lr ? e : 0.0f;
                }
                const float a0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(ai, 0));
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int t = 4 * gl + r;
                    sh.E[b4][t][lr] = ev[r];
                    if (lr == 0) {
                        sh.A[b4][t] = ev[r] * a0;
                        if (DECAY_FIRST) sh.C[b4][t] = ev[r] * a0;
                        else if (t + 1 < T) sh.C[b4][t + 1] = ev[r] * a0;
                    }
                }
                if (!DECAY_FIRST && lane == 0) sh.C[b4][0] = 1.0f;
                if (gl == 0) sh.B[b4][lr] = x.be;
                if (i + 5 < n_chunks) load_gates(i + 5, x);
            }
            lds_barrier();
            if (on) {
                const int b3 = (i + 3) % 3;
                f32x4 g2[2] = {zero, zero};
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    *reinterpret_cast<f32x4*>(is_q ? &sh.q[b3][lr][64 * half + 16 * m + 4 * gl]
                                                   : &sh.k[b3][lr][64 * half + 16 * m + 4 * gl]) = is_q ? x.q[m] : x.k[m];
#pragma unroll
                    for (int j = 0; j < 4; ++j) g2[m & 1] = mma4(x.k[m][j], is_q ? x.q[m][j] : x.k[m][j], g2[m & 1]);
                }
                gr = g2[0] + g2[1];
                if (half) sh.G[is_q][lane] = gr;
                if (i + 5 < n_chunks) load_rows(i + 5, x);
            }
            lds_barrier();
        };
        Chunk even, odd;
        load_rows(0, even);
        load_rows(1, odd);
        if (pw == 3) {
            load_gates(0, even);
            load_gates(1, odd);
        }
        for (int i = -3; i < n_chunks; i += 2) {
            iteration(i, even);
            if (i + 1 < n_chunks) iteration(i + 1, odd);
        }
    };
    if (wv == 4) produce(std::integral_constant<int, 0>{});
    else if (wv == 5) produce(std::integral_constant<int, 1>{});
    else if (wv == 6) produce(std::integral_constant<int, 2>{});
    else produce(std::integral_constant<int, 3>{});
}

// Work-groups of the chunked kernel that fit the device at once (each then runs several items).
template <int HD, bool DECAY_FIRST>
int chunked_resident_groups() {
    static int cached = -1;
    if (cached < 0) {
        int dev = 0, cus = 0, per_cu = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, gdn_verify_chunked_kernel<HD, DECAY_FIRST>, 256, 0) ==
                hipSuccess &&
            cus > 0 && per_cu > 0)
            cached = cus * per_cu;
        else
            cached = 0;  // unknown: one item per work-group
    }
    return cached;
}

template <int HD, bool DECAY_FIRST>
hipError_t launch_chunked_df(const GdnArgs& a, hipStream_t stream) {
    const int64_t items = (int64_t)a.S * a.G * (HD / 64);
    if (items > INT32_MAX) return hipErrorInvalidValue;
    const int resident = chunked_resident_groups<HD, DECAY_FIRST>();
    const int64_t groups = resident > 0 && resident < items ? resident : items;
    const int pair = HD == 128 && ((int64_t)a.S * a.G) % 8 == 0;
    hipLaunchKernelGGL((gdn_verify_chunked_kernel<HD, DECAY_FIRST>), dim3((unsigned)groups), dim3(256), 0, stream, a,
                       (int)items, pair);
    return hipGetLastError();
}

template <int HD>
hipError_t launch_scan(const GdnArgs& a, hipStream_t stream) {
    const int64_t groups = (int64_t)a.S * a.G * (HD / kScanRows);
    const int grouped = ((int64_t)a.S * a.G) % 8 == 0;
    if (a.decay_first)
        hipLaunchKernelGGL((gdn_scan_kernel<HD, true>), dim3((unsigned)groups), dim3(512), 0, stream, a, grouped);
    else
        hipLaunchKernelGGL((gdn_scan_kernel<HD, false>), dim3((unsigned)groups), dim3(512), 0, stream, a, grouped);
    return hipGetLastError();
}

template <int HD>
hipError_t launch_chunked(const GdnArgs& a, hipStream_t stream) {
    // While its work-groups fit the CUs at once the scan kernel is the faster one at every length (48
    // groups of 128 rows, one stream, graph replays: 4 rows 9.2 -> 8.0 us, 16 rows 9.4 -> 8.2, 128 rows
    // 40.8 -> 27.5, 2048 rows 674 -> 295); beyond that its eight waves per CU lose to the sixteen of the
    // chunked kernel (chunked against scan: two streams, 16 rows 10.0 against 14.1, 128 rows 45.0 against
    // 51.7; four streams, 128 rows 61.9 against 77.7, 1024 rows 473 each; eight streams, 512 rows 311 against
    // 493).  Long blocks of exactly two streams are the exception that the line leaves out: 512 rows
    // 173 against 158, 2048 rows 748 against 612.
    if ((int64_t)a.S * a.G * (HD / kScanRows) <= device_cu_count()) return launch_scan<HD>(a, stream);
    return a.decay_first ? launch_chunked_df<HD, true>(a, stream) : launch_chunked_df<HD, false>(a, stream);
}

template <int K, int HD, int SPLIT>
hipError_t launch_split(const GdnArgs& a, hipStream_t stream) {
    const dim3 grid((unsigned)((int64_t)a.S * a.G * SPLIT)), block(256);
    if (a.decay_first)
        hipLaunchKernelGGL((gdn_verify_kernel<K, HD, SPLIT, true>), grid, block, 0, stream, a);
    else
        hipLaunchKernelGGL((gdn_verify_kernel<K, HD, SPLIT, false>), grid, block, 0, stream, a);
    return hipGetLastError();
}
template <int K, int HD>
hipError_t launch_shape(const GdnArgs& a, hipStream_t stream) {
    if constexpr (HD / (256 / (K / kC)) >= 2) return launch_split<K, HD, 2>(a, stream);
    else return launch_split<K, HD, 1>(a, stream);
}

}  // namespace

hipError_t launch_gdn_verify(const GdnArgs& a, hipStream_t stream) {
    if ((int64_t)a.S * a.G == 0) return hipSuccess;
    if (a.K == 128 && a.HD == 128) return launch_chunked<128>(a, stream);
    if (a.K == 128 && a.HD == 64) return launch_chunked<64>(a, stream);
    if (a.K == 64 && a.HD == 128) return launch_shape<64, 128>(a, stream);
    if (a.K == 64 && a.HD == 64) return launch_shape<64, 64>(a, stream);
    return hipErrorInvalidValue;
}

}  // namespace sixi
