// Internal declarations shared by the HIP translation units of libgla_hip.so.
// gfx950 (MI355X) only.  Matrices are column-major with explicit leading
// dimensions, exactly the Julia layout the reference works on.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <string>
#include <vector>

#include "gla_hip.h"

namespace gla {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

// Thread-local error text returned by gla_last_error_string().
void set_error(const char *fmt, ...);

#define GLA_HIP_TRY(expr)                                                              \
    do {                                                                               \
        hipError_t _e = (expr);                                                        \
        if (_e != hipSuccess) {                                                        \
            ::gla::set_error("%s:%d %s -> %s", __FILE__, __LINE__, #expr,              \
                             hipGetErrorString(_e));                                   \
            return GLA_ERR_HIP;                                                        \
        }                                                                              \
    } while (0)

#define GLA_LAUNCH_CHECK()                                                             \
    do {                                                                               \
        hipError_t _e = hipGetLastError();                                             \
        if (_e != hipSuccess) {                                                        \
            ::gla::set_error("%s:%d launch failed: %s", __FILE__, __LINE__,            \
                             hipGetErrorString(_e));                                   \
            return GLA_ERR_HIP;                                                        \
        }                                                                              \
    } while (0)

// v from lane K of each 16-lane row to the whole row (DPP row_newbcast:K).
// Every lane reads a valid source, so no "old" value needs setting up; a
// 64-bit value moves in one v_mov_b64_dpp (gfx950 has DPP on 64-bit moves
// for row_newbcast).
template <int K, typename T>
__device__ __forceinline__ T row_bcast(T v)
{
    static_assert(K >= 0 && K < 16, "lane of a 16-lane row");
    return __builtin_amdgcn_update_dpp(v, v, 0x150 + K, 0xF, 0xF, true);
}

// v from the lane DPP control CTRL selects within its row (bound_ctrl off:
// a source outside the row reads 0); 64-bit values move as two halves.
template <int CTRL, typename T>
__device__ __forceinline__ T dppmov(T v)
{
    if constexpr (sizeof(T) == 8) {
        int2 u = __builtin_bit_cast(int2, v);
        u.x = __builtin_amdgcn_update_dpp(0, u.x, CTRL, 0xF, 0xF, false);
        u.y = __builtin_amdgcn_update_dpp(0, u.y, CTRL, 0xF, 0xF, false);
        return __builtin_bit_cast(T, u);
    } else {
        return __builtin_bit_cast(
            T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
    }
}

// Sum over the 16 lanes of each row, the same bits in every lane of the row:
// pairs, quads, half rows, rows (each step adds two equal-order partials).
template <typename T>
__device__ __forceinline__ T row_sum16(T v)
{
    v += dppmov<0xB1>(v);    // quad_perm [1,0,3,2]
    v += dppmov<0x4E>(v);    // quad_perm [2,3,0,1]
    v += dppmov<0x141>(v);   // row_half_mirror
    v += dppmov<0x140>(v);   // row_mirror
    return v;
}

// Sum over the 4 lanes of each quad, the same bits in every lane of it.
template <typename T>
__device__ __forceinline__ T quad_sum(T v)
{
    v += dppmov<0xB1>(v);
    v += dppmov<0x4E>(v);
    return v;
}

// v of lane `src` (wave-uniform) in every lane.
template <typename T>
__device__ __forceinline__ T lane_value(T v, int src)
{
    if constexpr (sizeof(T) == 8) {
        int2 u = __builtin_bit_cast(int2, v);
        u.x = __builtin_amdgcn_readlane(u.x, src);
        u.y = __builtin_amdgcn_readlane(u.y, src);
        return __builtin_bit_cast(T, u);
    } else {
        return __builtin_bit_cast(T, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), src));
    }
}

// Sum over the 64 lanes (all active), the same value in every lane and a
// fixed order: 16-lane row sums by DPP, then the four rows.
template <typename T>
__device__ __forceinline__ T wave_sum_dpp(T v)
{
    v = row_sum16(v);
    return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

// Fused multiply-add in T's own precision.
__device__ __forceinline__ double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// Forward elimination steps of a 16×16 lower-triangular inverse in the
// four-column layout (lane (i, g) holds w[t] = V[i][g + 4t]): for K = 0…14,
// V[i] −= m[K]·V[K] with row K of V broadcast from lane K of each 16-lane
// row; m[K] is this lane's multiplier (zero for i ≤ K), so every step is one
// broadcast and one unconditional FMA per column.
template <int K, typename T>
struct TileInvSteps {
    static __device__ __forceinline__ void run(const T m[16], T w[4])
    {
#pragma unroll
        for (int t = 0; t < 4; ++t) w[t] = fma_t(-m[K], row_bcast<K>(w[t]), w[t]);
        TileInvSteps<K + 1, T>::run(m, w);
    }
};
template <typename T>
struct TileInvSteps<15, T> {   // row 15 has no rows below it
    static __device__ __forceinline__ void run(const T *, T *) {}
};

// The same backward, for an upper-triangular inverse: K = 15…1,
// V[i] −= m[K]·V[K] (m[K] zero for i ≥ K).
template <int K, typename T>
struct TileInvStepsUp {
    static __device__ __forceinline__ void run(const T m[16], T w[4])
    {
#pragma unroll
        for (int t = 0; t < 4; ++t) w[t] = fma_t(-m[K], row_bcast<K>(w[t]), w[t]);
        TileInvStepsUp<K - 1, T>::run(m, w);
    }
};
template <typename T>
struct TileInvStepsUp<0, T> {   // row 0 has no rows above it
    static __device__ __forceinline__ void run(const T *, T *) {}
};

// s = √a and r = 1/√a from the hardware reciprocal square root refined by
// Newton steps (two for FP64, one for FP32) and one correction of s = a·r:
// both within an ulp or two of sqrt(a) and 1/sqrt(a), at a fraction of the
// latency of a correctly rounded square root followed by a division, which
// sit on the serial path of every column.  a = 0 gives s = 0, r = ∞ and a
// negative or NaN a gives NaN, as sqrt and 1/sqrt do.
__device__ __forceinline__ void sqrt_and_rsqrt(double a, double &s, double &r)
{
    double y = __builtin_amdgcn_rsq(a);
    const double h = 0.5 * a;
    double e = __builtin_fma(-h * y, y, 0.5);
    y = __builtin_fma(y, e, y);
    e = __builtin_fma(-h * y, y, 0.5);
    y = __builtin_fma(y, e, y);
    double q = a * y;
    q = __builtin_fma(__builtin_fma(-q, q, a), 0.5 * y, q);
    const bool zero = a == 0.0;
    s = zero ? 0.0 : q;
    r = zero ? __builtin_inf() : y;
}
__device__ __forceinline__ void sqrt_and_rsqrt(float a, float &s, float &r)
{
    float y = __builtin_amdgcn_rsqf(a);
    const float h = 0.5f * a;
    const float e = __builtin_fmaf(-h * y, y, 0.5f);
    y = __builtin_fmaf(y, e, y);
    float q = a * y;
    q = __builtin_fmaf(__builtin_fmaf(-q, q, a), 0.5f * y, q);
    const bool zero = a == 0.0f;
    s = zero ? 0.0f : q;
    r = zero ? __builtin_inff() : y;
}

// 16×16×4 MFMA with one A and one B element per lane; accumulator element r
// of lane l sits at (row(l, r), l % 16) of the 16×16 tile.
template <typename T>
struct PanelMfma;
template <>
struct PanelMfma<double> {
    typedef d4 acc_t;
    static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int l, int r) { return (l >> 4) + 4 * r; }
};
template <>
struct PanelMfma<float> {
    typedef f4 acc_t;
    static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int l, int r) { return 4 * (l >> 4) + r; }
};


// ------------------------------------------------- symmetric tile factor --
// The other half of a lane pair at distance 16 / 32: permlane swaps of v
// with itself.  even(): rows (0, 0, 2, 2) / (01, 01) of v; odd(): rows
// (1, 1, 3, 3) / (23, 23).
template <typename T>
__device__ __forceinline__ void swap16(T v, T &even, T &odd)
{
    if constexpr (sizeof(T) == 8) {
        const uint2 u = __builtin_bit_cast(uint2, v);
        const auto a = __builtin_amdgcn_permlane16_swap(u.x, u.x, false, false);
        const auto b = __builtin_amdgcn_permlane16_swap(u.y, u.y, false, false);
        even = __builtin_bit_cast(T, uint2{a[0], b[0]});
        odd = __builtin_bit_cast(T, uint2{a[1], b[1]});
    } else {
        const unsigned u = __builtin_bit_cast(unsigned, v);
        const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
        even = __builtin_bit_cast(T, (unsigned)a[0]);
        odd = __builtin_bit_cast(T, (unsigned)a[1]);
    }
}
template <typename T>
__device__ __forceinline__ void swap32(T v, T &lo, T &hi)
{
    if constexpr (sizeof(T) == 8) {
        const uint2 u = __builtin_bit_cast(uint2, v);
        const auto a = __builtin_amdgcn_permlane32_swap(u.x, u.x, false, false);
        const auto b = __builtin_amdgcn_permlane32_swap(u.y, u.y, false, false);
        lo = __builtin_bit_cast(T, uint2{a[0], b[0]});
        hi = __builtin_bit_cast(T, uint2{a[1], b[1]});
    } else {
        const unsigned u = __builtin_bit_cast(unsigned, v);
        const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        lo = __builtin_bit_cast(T, (unsigned)a[0]);
        hi = __builtin_bit_cast(T, (unsigned)a[1]);
    }
}

// Lanes below 32 (even rows): a summed over the lane pair at distance 32
// (16); the other lanes: b likewise.
template <typename T>
__device__ __forceinline__ T pair_sum32(T a, T b)
{
    if constexpr (sizeof(T) == 8) {
        const uint2 u = __builtin_bit_cast(uint2, a), v = __builtin_bit_cast(uint2, b);
        const auto x = __builtin_amdgcn_permlane32_swap(u.x, v.x, false, false);
        const auto y = __builtin_amdgcn_permlane32_swap(u.y, v.y, false, false);
        return __builtin_bit_cast(T, uint2{x[0], y[0]}) + __builtin_bit_cast(T, uint2{x[1], y[1]});
    } else {
        const auto x = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a),
                                                        __builtin_bit_cast(unsigned, b), false, false);
        return __builtin_bit_cast(T, (unsigned)x[0]) + __builtin_bit_cast(T, (unsigned)x[1]);
    }
}
template <typename T>
__device__ __forceinline__ T pair_sum16(T a, T b)
{
    if constexpr (sizeof(T) == 8) {
        const uint2 u = __builtin_bit_cast(uint2, a), v = __builtin_bit_cast(uint2, b);
        const auto x = __builtin_amdgcn_permlane16_swap(u.x, v.x, false, false);
        const auto y = __builtin_amdgcn_permlane16_swap(u.y, v.y, false, false);
        return __builtin_bit_cast(T, uint2{x[0], y[0]}) + __builtin_bit_cast(T, uint2{x[1], y[1]});
    } else {
        const auto x = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a),
                                                        __builtin_bit_cast(unsigned, b), false, false);
        return __builtin_bit_cast(T, (unsigned)x[0]) + __builtin_bit_cast(T, (unsigned)x[1]);
    }
}

// 1/a to about an ulp: the hardware estimate (relative error 2^-23 or better)
// and one third-order step (FP64) or Newton step (FP32).  For finite a with a
// finite reciprocal.
__device__ __forceinline__ double recip_step(double a)
{
    const double y = __builtin_amdgcn_rcp(a);
    const double e = __builtin_fma(-a, y, 1.0);
    return __builtin_fma(y, __builtin_fma(e, e, e), y);
}
__device__ __forceinline__ float recip_step(float a)
{
    const float y = __builtin_amdgcn_rcpf(a);
    return __builtin_fmaf(y, __builtin_fmaf(-a, y, 1.0f), y);
}

// 1/√d: the hardware estimate (relative error 2^-23 or better) and, for
// FP64, one third-order step y(1 + e/2 + 3e²/8), e = 1 − d y² (the rest is
// 5e³/16 < 2^-70); FP32 takes one Newton step.  d = 0 gives ∞, d < 0 and
// NaN give NaN: the min keeps e finite where d·y is 0·∞.
__device__ __forceinline__ double rsqrt_step(double d)
{
    const double y = __builtin_amdgcn_rsq(d);
    const double e = __builtin_fmin(__builtin_fma(-(d * y), y, 1.0), 0.5);
    return __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
}
__device__ __forceinline__ float rsqrt_step(float d)
{
    const float y = __builtin_amdgcn_rsqf(d);
    const float e = __builtin_fminf(__builtin_fmaf(-(d * y), y, 1.0f), 0.5f);
    return __builtin_fmaf(y * e, 0.5f, y);
}

// Columns 4S … 4S+3 of the symmetric tile S (accumulator layout, both
// triangles present), column t to c[t] with lane (i, g) holding row i in
// every 16-lane group: by symmetry the columns are rows of the accumulator,
// which sit in one register of the four groups (FP64) or in the four
// registers of one group (FP32).
template <int S>
__device__ __forceinline__ void tile_columns(const d4 &a, double c[4])
{
    double e, o;
    swap16<double>(a[S], e, o);
    swap32<double>(e, c[0], c[2]);
    swap32<double>(o, c[1], c[3]);
}
template <int S>
__device__ __forceinline__ void tile_columns(const f4 &a, float c[4])
{
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        float e, o, lo, hi;
        swap16<float>(a[t], e, o);
        swap32<float>(S & 1 ? o : e, lo, hi);
        c[t] = S & 2 ? hi : lo;
    }
}

// Column C = 4S + t of the factor, in every group: pivot, reciprocal square
// root, scaling, the later columns of the group of four, and step C of the
// inverse's forward elimination V[i] −= (l_i/l_C) V[C] (w[q] holds column
// g + 4q of V, zero above row g + 4q, so columns past C need no step).
template <int C, typename T>
__device__ __forceinline__ void tile_column_step(T c[4], T w[4], T &dsel, T &ysel, int i)
{
    constexpr int t = C & 3;
    const T d = row_bcast<C>(c[t]);
    const T y = rsqrt_step(d);
    const T l = c[t] * y;
    c[t] = l;
    dsel = i == C ? d : dsel;
    ysel = i == C ? y : ysel;
    if constexpr (t < 3) c[t + 1] = fma_t(-l, row_bcast<(C + 1) & 15>(l), c[t + 1]);
    if constexpr (t < 2) c[t + 2] = fma_t(-l, row_bcast<(C + 2) & 15>(l), c[t + 2]);
    if constexpr (t < 1) c[t + 3] = fma_t(-l, row_bcast<(C + 3) & 15>(l), c[t + 3]);
    if constexpr (C < 15) {
        const T m = i > C ? l * y : T(0);
#pragma unroll
        for (int q = 0; q <= C / 4; ++q) w[q] = fma_t(-m, row_bcast<C>(w[q]), w[q]);
    }
}

template <int S, typename T>
__device__ __forceinline__ void tile_four_columns(typename PanelMfma<T>::acc_t &a,
                                                  typename PanelMfma<T>::acc_t &lt, T w[4],
                                                  T &dsel, T &ysel, int i, int g)
{
    T c[4];
    tile_columns<S>(a, c);
    tile_column_step<4 * S, T>(c, w, dsel, ysel, i);
    tile_column_step<4 * S + 1, T>(c, w, dsel, ysel, i);
    tile_column_step<4 * S + 2, T>(c, w, dsel, ysel, i);
    tile_column_step<4 * S + 3, T>(c, w, dsel, ysel, i);
    // element (i, 4S + g): the MFMA operand of the rank-4 update
    const T e = g < 2 ? (g == 0 ? c[0] : c[1]) : (g == 2 ? c[2] : c[3]);
    if constexpr (S < 3) a = PanelMfma<T>::mma(-e, e, a);
    if constexpr (sizeof(T) == 8) {
        lt[S] = e;
    } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) lt[t] = g == S ? c[t] : lt[t];
    }
}

// Factors a symmetric 16×16 tile on one wave.  a: the tile in accumulator
// layout with both triangles (overwritten); on return a holds L transposed
// (lane: row l % 16 at columns row(l, r); entries right of the diagonal are
// meaningless) and w the inverse (w[q] = L⁻¹[i][g + 4q], lane (i, g)).
// Right-looking by four-column groups: within a group column by column as
// cholUnblocked! does (src/cholesky.jl:3-15; the products are (a_ic r)(a_jc
// r), each factor rounded once), then one rank-4 MFMA for the rest of the
// tile.  The inverse's elimination steps fill the pivot chain's latency.
// Returns the mask of the pivots among the first `nvalid` whose square root is
// taken of a negative number.
template <typename T>
__device__ __forceinline__ unsigned tile_factor(typename PanelMfma<T>::acc_t &a, T w[4], int nvalid)
{
    typedef PanelMfma<T> M;
    const int lane = threadIdx.x & 63;
    const int i = lane & 15, g = lane >> 4;
    T dsel = T(1), ysel = T(1);
    typename M::acc_t lt = {T(0), T(0), T(0), T(0)};
#pragma unroll
    for (int q = 0; q < 4; ++q) w[q] = (i == g + 4 * q) ? T(1) : T(0);
    tile_four_columns<0, T>(a, lt, w, dsel, ysel, i, g);
    tile_four_columns<1, T>(a, lt, w, dsel, ysel, i, g);
    tile_four_columns<2, T>(a, lt, w, dsel, ysel, i, g);
    tile_four_columns<3, T>(a, lt, w, dsel, ysel, i, g);
    const unsigned neg = (unsigned)__ballot(dsel < T(0) && i < nvalid) & 0xffffu;
    // the diagonal: √d = d·y corrected once
    T s = dsel * ysel;
    s = fma_t(fma_t(-s, s, dsel), T(0.5) * ysel, s);
    s = dsel == T(0) ? T(0) : s;
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] = M::row(lane, r) == i ? s : lt[r];
#pragma unroll
    for (int q = 0; q < 4; ++q) w[q] *= ysel;
    return neg;
}
// The same; the first such pivot is recorded in *info as gbase + index + 1.
template <typename T>
__device__ __forceinline__ void tile_factor(typename PanelMfma<T>::acc_t &a, T w[4], int nvalid,
                                            int *info, int64_t gbase)
{
    const unsigned neg = tile_factor<T>(a, w, nvalid);
    if (neg != 0 && (threadIdx.x & 63) == 0 && info)
        atomicCAS(info, 0, (int)(gbase + __builtin_ctz(neg) + 1));
}

// Holds a loaded value where it is.  A load from a clamped address whose value
// a select then drops is otherwise turned into a load under a branch, and a
// row of them into round trips one after another: load all, hold all, select.
template <typename T>
__device__ __forceinline__ void hold(T &v)
{
    asm volatile("" : "+v"(v));
}

// Barrier over the workgroup that orders LDS only: outstanding global
// stores stay in flight (__syncthreads waits for them, about a memory round
// trip per barrier).
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// ------------------------------------------------------------------ handle --
// Workspace slots carved out of one device allocation that only grows.
struct Handle {
    int device = 0;
    hipStream_t side = nullptr;       // second stream for look-ahead overlap
    hipEvent_t ev_fork = nullptr;     // main -> side
    hipEvent_t ev_join = nullptr;     // side -> main
    hipEvent_t ev_step[2] = {nullptr, nullptr};
    int *dinfo = nullptr;             // device: first failing pivot (1-based), 0 = ok
    unsigned *dbar = nullptr;         // device: grid-barrier counters
    void *ws = nullptr;               // device workspace
    size_t ws_bytes = 0;
    void *df = nullptr;               // packed tiles of the dataflow Cholesky
    size_t df_bytes = 0;
    bool df_captured = false;         // a graph holds df
    std::vector<void *> df_kept;      // former ones that a graph holds
    int num_cus = 256;
    // Tuning: block width of the look-ahead driver behind cholRecursive!
    // (0: the recursive-halving driver; −1: chosen from n).  Set with
    // gla_set_tuning.
    int64_t chol_block = -1;
    // cholRecursive! factors matrices up to this order in one dataflow launch
    // and the look-ahead driver's block columns likewise (0: neither).
    int64_t chol_df = 8192;
    // Solve the look-ahead Cholesky's panels in one launch each (1) or by the
    // recursive rdiv! (0).
    int chol_psolve = 1;
    // Release the look-ahead Cholesky's side-stream SYRK after the
    // next-block-column update (1) rather than right after the panel solve.
    int chol_syrk_late = 1;
    // Step width of the LDLᵀ driver (128: 128-wide steps; a larger multiple
    // of 128: that width with depth-1 look-ahead).
    int64_t ldlt_block = 512;
    // Block width of the mixed-precision factorisation's look-ahead driver.
    int mixed_block = 512;
    // QR panel kernel: 1 LDS-reduction form, 2 wave-butterfly form.
    int qr_panel = 2;
    // Width of the sub-panels a QR block column is factored in (0: the whole
    // block column in one panel launch; 32 or 64; -1: by the column height).
    int qr_inner = -1;
    // Depth-1 look-ahead in qrBlocked! (trailing update on the side stream).
    int qr_lookahead = 1;
    // Block columns at least this tall are factored by the
    // reconstructed-Householder panel (0: never; -1: any height for block
    // columns at least 32 wide, otherwise by width and height: use_hr).
    int64_t qr_hr = -1;
    // Polls before a device-side wait gives up (a call that synchronises then
    // returns GLA_ERR_TIMEOUT, others leave NaN).
    unsigned spin_limit = 1u << 25;
    // Test setting: every wait of a QR panel, real or complex, is for an arrival
    // that never comes, so each gives up after spin_limit polls.
    int qr_wait_test = 0;
    // CUs kept free of the look-ahead Cholesky's trailing SYRK (0: none;
    // a new handle takes num_cus/8).  When set, the driver runs its chain on
    // `chain` (all CUs) and the SYRK on `masked` (the other CUs), both
    // forked from the caller's stream.
    int side_cu_reserve = 0;
    hipStream_t chain = nullptr;
    hipStream_t masked = nullptr;
};

// Ensure the workspace holds at least `bytes` (grows with hipMalloc, which
// synchronises the device; the first call of a given size pays for it).
int ensure_workspace(Handle *h, size_t bytes);
// The same for the dataflow Cholesky's buffer; false if it cannot be had, or
// would have to grow while stream s is being captured
// (the caller then takes a path without it).
bool ensure_df(Handle *h, hipStream_t s, size_t bytes);
// Whether s is being captured into a graph.
bool capturing(hipStream_t s);

// A launch whose workgroups all wait for each other needs them all on the chip,
// and two such launches that do not fit together could each hold places the
// other waits for.  Each counts a whole CU per workgroup here, dealt out to the
// dies in turn.  resident_begin makes stream s wait, on the device, for the
// oldest such calls of the process until the new one fits beside the rest, and for
// the PanelCalls in flight if it does not fit beside them; resident_end marks
// the new one.  Between the two the caller queues its launches; a lock is
// held meanwhile, so every begin is followed by its end.
// False (nothing held): the stream is being captured, where another stream's
// launch cannot be waited for, or an event failed.
bool resident_begin(Handle *h, hipStream_t s, int64_t workgroups);
int resident_end(Handle *h, hipStream_t s);
// A call that queues panels with grid-wide waits, of up to `workgroups` each, and
// then waits for its stream: such calls run beside one another, but beside
// resident calls only where all fit.  Made before the first launch; queued() after
// the last; destroyed when the stream has been waited for.
struct PanelCall {
    PanelCall(Handle *h, hipStream_t s, int64_t workgroups);
    void queued();
    ~PanelCall();
    PanelCall(const PanelCall &) = delete;
    hipStream_t s;
    int device = -1, weight = 0;
    bool is_queued = false;
    PanelCall *link = nullptr;
};

// ------------------------------------------------------------------ GEMM --
// C = alpha*op(A)*op(B) + beta*C  with op(A) M×K, op(B) K×N.
// mode 0: every element; mode 1: only elements with (row + diag_off) >= col
// ("lower" relative to a diagonal), tiles wholly above it are skipped.
// ta/tb: 'N' or 'T'.  Supported (ta,tb,mode): (N,N,0) (N,T,0) (T,N,0) (N,T,1)
// (N,T,2).  kfrom_row = 1: op(A)(i,k) = 0 for k < i (an upper-triangular
// op(A)), so each tile contracts k from its first row on (no split-K).
template <typename T>
int gemm(hipStream_t s, char ta, char tb, int mode, int64_t M, int64_t N, int64_t K, T alpha,
         const T *A, int64_t lda, const T *B, int64_t ldb, T beta, T *C, int64_t ldc,
         int64_t diag_off = 0, T *ws = nullptr, size_t ws_elems = 0, int kfrom_row = 0);
// Selects the FP64 direct-to-LDS GEMM kernel (0: off).
void set_gemm_dl(int v);
void set_gemm_lds1(int v);
int get_gemm_dl();
int get_gemm_lds1();

// ------------------------------------------------------------- Cholesky --
// Linv: scratch for the 16×16 diagonal-tile inverses (tile_inverse_elems(n)
// elements); null takes it from the handle's workspace.
template <typename T>
int chol_device(Handle *h, hipStream_t s, int64_t n, T *A, int64_t lda, int algo,
                int64_t param, T *Linv = nullptr);

// Dataflow Cholesky (chol_df.hip) of the m×n block column at A (m ≥ n;
// n a multiple of 64 unless m = n), the first n rows its diagonal block: L in
// place, and the 16×16 diagonal-tile inverses in LinvG if given.  Bytes of
// h->df it needs: chol_df_bytes.
size_t chol_df_bytes(int64_t m, int64_t n, size_t esz);
template <typename T>
int chol_df(Handle *h, hipStream_t s, int64_t m, int64_t n, T *A, int64_t lda, int64_t info_base,
            T *LinvG);

// Cholesky building blocks (chol.hip): factor one ≤128 diagonal block in
// place and store the inverses of its 16×16 diagonal tiles; solve rows
// below it (B <- B L⁻ᵀ) with those inverses; inverses of all 16×16 diagonal
// tiles of an n×n lower L; the recursive right-side solve B <- B L⁻ᵀ.
// LDLᴴ (_ldlt_lower!, src/ldlt.jl:16-33) of the nb×nb (nb ≤ 128) block at
// A in one workgroup: D on the diagonal, the unit factor's L below it, and
// the inverses of its unit 16×16 diagonal tiles in LinvG.
template <typename T>
int ldlt_factor_block(hipStream_t s, int nb, T *A, int64_t lda, T *LinvG);
template <typename T>
int chol_factor_block(hipStream_t s, int nb, T *A, int64_t lda, int *info, int64_t info_base,
                      T *LinvG);
// The same for a block classified on the device: flags[0] != 0 — skip;
// flags[1] == 0 — A is within 0.1·√eps of I (Frobenius), factored to
// first order (L = I + strictly-lower(A) + (diag(A) − 1)/2); otherwise the
// full factorisation.
template <typename T>
int chol_factor_block_near_identity(hipStream_t s, int nb, T *A, int64_t lda, int *info,
                                    int64_t info_base, T *LinvG, const int *flags);
// The diagonal-block factorisation of an FP32 block (nb ≤ 128) computed in
// FP64: read and written in FP32, FP32 tile inverses in Linv32.
int chol_factor_block_f32io(hipStream_t s, int nb, float *A, int64_t lda, int *info,
                            int64_t info_base, float *Linv32);
template <typename T>
int chol_solve_block(hipStream_t s, int nb, const T *L, int64_t ldl, const T *LinvG, T *B,
                     int64_t ldb, int64_t nrows);
template <typename T>
int tile_inverses(hipStream_t s, int64_t n, const T *L, int64_t ldl, T *LinvG);
// chol_factor_block for a strided batch, L beside A, with per-matrix info.
template <typename T>
int chol_factor_batched(hipStream_t s, int nb, const T *A, int64_t lda, int64_t sA, T *L,
                        int64_t ldl, int64_t sL, int *info, int64_t batch);
template <typename T>
int trsm_rlt(hipStream_t s, int64_t m, int64_t n, const T *L, int64_t ldl, const T *Linv, T *B,
             int64_t ldb);
size_t tile_inverse_elems(int64_t n);
// Y = M⁻¹ R for a few right-hand sides in one launch (trsv.hip).  M lower
// triangular of order n, element (i, j) at M[i·si + j·sj], one stride ±1
// (a leading stride of 1 is read first); only i ≥ j is read, and with `unit`
// not the diagonal.  R's element (i, k) at R[i·ri + (k mod 16)·rk +
// (k div 16)·rp], divided by div[i·ds] if div is given.  Y: tri_solve_elems
// elements on 16 bytes, rows of 16 per pass (element (i, k) at [(k div 16)·npad·16 + 16 i +
// k mod 16], npad = n rounded up to 128), and a ticket, both set by
// tri_solve_prepare.  If `out` is given, out[i·oi + k·ok] = mul[i·ms]·y (mul
// may be null); if X is, X[i·oi + k·ok] += y.
template <typename T>
struct TriSolve {
    int64_t n;
    const T *M;
    int64_t si, sj;
    int unit, nrhs;
    const T *R;
    int64_t ri, rk, rp;
    const T *div;
    int64_t ds;
    T *Y, *out;
    double *X;
    int64_t oi, ok;
    const T *mul;
    int64_t ms;
    int *ticket, *err;       // *err = 1 if a wait gave up (err may be null)
    unsigned spin_limit;
    int npass;               // set by tri_solve
};
size_t tri_solve_elems(int64_t n, int64_t nrhs);
// cnt elements of Y marked, and the tickets of `solves` launches zeroed.
template <typename T>
int tri_solve_prepare(hipStream_t s, int64_t cnt, T *Y, int *ticket, int solves);
template <typename T>
int tri_solve(hipStream_t s, TriSolve<T> p);
// R (row-major n×16, type T) = B − sym(A) X for the lower-stored FP64 A and
// nrhs ≤ 16 columns of X, B (column-major); Xt: symv_scratch(n) doubles;
// nrm[k] += ‖r_k‖², nrm[16 + k] += ‖x_k‖² (nrm zeroed by the caller).
template <typename T>
int symv_residual(hipStream_t s, int64_t n, const double *A, int64_t lda, const double *X,
                  int64_t ldx, const double *B, int64_t ldb, int nrhs, double *Xt, T *R,
                  double *nrm);
size_t symv_scratch(int64_t n);

// QR building blocks (qr.hip): T of the first k reflectors of F (m×k), and
// A (mA×nA) <- op(Q) A, trans 'N' or 'T', Q from the first b reflectors.
// V (m×n, ld ldv) = the reflectors stored in F with their unit diagonal and
// zeros above.
template <typename T>
int unit_lower_explicit(hipStream_t s, int64_t m, int64_t n, const T *F, int64_t ldf, T *V,
                        int64_t ldv);
size_t qr_tblock_scratch(int64_t m, int64_t k);
size_t qr_apply_scratch(int64_t mA, int64_t nA, int64_t b);
template <typename T>
int qr_tblock_dev(hipStream_t s, int64_t m, int64_t k, const T *F, int64_t ldf, const T *tau,
                  T *Tm, int64_t ldt, T *scratch);
template <typename T>
int qr_apply_dev(hipStream_t s, char trans, int64_t mA, int64_t nA, int64_t b, const T *V,
                 int64_t ldv, const T *Tm, int64_t ldt, T *A, int64_t lda, T *scratch);

// Small helpers used across units.
__global__ void k_set_int(int *p, int v);

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

}  // namespace gla
