// Triangular solves for a few right-hand sides in one launch, and the
// symmetric residual of the mixed-precision refinement.  No counterpart in
// the reference (its Cholesky stops at the factor, src/cholesky.jl:3-55);
// the solve is what `L \ (L' \ b)` would do there.
//
// tri_solve: Y = M⁻¹ R for a lower triangular M given by its first element
// and two strides, so that L, Lᵀ, Uᵀ and U are all read where they lie (a
// backward solve is a lower one with both orders reversed).  128 rows per
// workgroup, 16 per wave, 16 right-hand sides per pass; the passes are
// independent.  Block b streams its tiles M_bj through MFMA as the Y_j
// appear; against its own diagonal block it substitutes tile by tile,
//   y_k = M_kk⁻¹ (r_k − Σ_{l<k} M_kl y_l)
// with M_kk⁻¹ the inverse of a 16×16 tile, formed by its wave before the
// chain reaches it (larger inverses would cost accuracy).  Y is the exchange:
// filled beforehand with a signalling NaN no arithmetic produces, so a value
// is its own arrival mark and one round trip brings it.  Of the block before
// its own a wave takes each tile as it comes, straight into the operand
// layout; all earlier ones come through LDS, a block ahead.
// A workgroup takes its place (b, pass) by a ticket when it starts, and
// waits for smaller b only: whatever else runs on the device, the smallest
// unfinished block is always one that is running.  Waits are bounded; one
// that gives up makes its rows, and so all later ones, NaN.
// Bound: the chain, per block eight substitutions (four MFMAs for the
// inverse, four for the next tile's update, one barrier; FP64 ~700 cycles,
// FP32 ~400) and one exchange (~2.5 µs).  n = 5001, 16 right-hand sides, two
// solves: FP64 473 µs, 5.9 µs a block, FP32 312 µs, 3.9; recursive GEMM-based
// solves on a copied and reversed factor took 3.5 and 2.8 ms.  With every
// wave polling the whole block before its own (eight times the traffic) FP64
// 560 µs.  128 rows, since an exchange per 64 costs more than the longer
// substitution.
// Accuracy: ‖A x − b‖/(‖A‖ ‖x‖) at n = 700…12000 is 0.84…1.0 (FP64) and
// 0.52…0.63 (FP32) of what the recursive form left: sums over 128 columns from
// zero instead of one over half the order.
//
// symv_residual: R = B − A X for symmetric A given by its lower triangle
// (FP64), 16 right-hand sides, with the column sums of squares of R and X
// for the backward error.
#include <algorithm>

#include "gla_coherent.hpp"
#include "gla_internal.hpp"

namespace gla {

namespace {

constexpr int kSB = 128;                  // rows per block
constexpr int kSR = 16;                   // right-hand sides per pass
constexpr int kST = 256;                  // threads per workgroup (residual)

template <typename T>
struct SMfma;
template <>
struct SMfma<double> {
    typedef d4 acc_t;
    static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int l, int r) { return (l >> 4) + 4 * r; }
};
template <>
struct SMfma<float> {
    typedef f4 acc_t;
    static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int l, int r) { return 4 * (l >> 4) + r; }
};

// How M lies in memory: kByRows si = ±1 (a column of M contiguous), kByCols
// sj = 1, kByColsRev sj = −1 (a row of M contiguous: four elements a load).
enum { kByRows, kByCols, kByColsRev };

// The column of a 16×16 tile that lane group lk takes for MFMA q, and its
// inverse: the row of the staged Y at which column k stands.
template <typename T, int MODE>
__device__ __forceinline__ int tile_col(int q, int lk)
{
    if (MODE == kByRows) return 4 * q + lk;
    return sizeof(T) == 8 ? 8 * (q >> 1) + 2 * lk + (q & 1) : 4 * lk + q;
}
template <typename T, int MODE>
__device__ __forceinline__ int staged_row(int k)
{
    if (MODE == kByRows) return k;
    const int kt = k & 15;
    const int p = sizeof(T) == 8 ? (kt & 8) + 4 * (kt & 1) + ((kt >> 1) & 3)
                                 : 4 * (kt & 3) + (kt >> 2);
    return (k & ~15) + p;
}

// Four consecutive elements, aligned as one.
template <bool REV>
__device__ __forceinline__ void load_quad(const float *p, float v[4])
{
    typedef float v4 __attribute__((ext_vector_type(4), aligned(4)));
    const v4 x = *reinterpret_cast<const v4 *>(REV ? p - 3 : p);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = REV ? x[3 - e] : x[e];
}
// (two pairs, eight columns apart)
template <bool REV>
__device__ __forceinline__ void load_quad(const double *p, double v[4])
{
    typedef double v2 __attribute__((ext_vector_type(2), aligned(8)));
    const v2 x = *reinterpret_cast<const v2 *>(REV ? p - 1 : p);
    const v2 y = *reinterpret_cast<const v2 *>(REV ? p - 9 : p + 8);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        v[e] = REV ? x[1 - e] : x[e];
        v[2 + e] = REV ? y[1 - e] : y[e];
    }
}

// This wave's rows (row address pr, lane's row and column group included)
// of the 16 columns at k0.
template <typename T, int MODE>
__device__ __forceinline__ void load_tile(const T *pr, int64_t sj, int64_t k0, T u[4])
{
    if (MODE == kByRows) {
#pragma unroll
        for (int q = 0; q < 4; ++q) u[q] = pr[(k0 + 4 * q) * sj];
    } else {
        load_quad<MODE == kByColsRev>(MODE == kByColsRev ? pr - k0 : pr + k0, u);
    }
}

// Device-coherent loads the compiler may leave in flight.
__device__ __forceinline__ void load_row4(__amdgpu_buffer_rsrc_t y, int off, double v[4])
{
    typedef double d2 __attribute__((ext_vector_type(2)));
    const d2 a = __builtin_bit_cast(d2, __builtin_amdgcn_raw_buffer_load_b128(y, off, 0, 16));
    const d2 b = __builtin_bit_cast(d2, __builtin_amdgcn_raw_buffer_load_b128(y, off + 16, 0, 16));
    v[0] = a[0]; v[1] = a[1]; v[2] = b[0]; v[3] = b[1];
}
__device__ __forceinline__ void load_row4(__amdgpu_buffer_rsrc_t y, int off, float v[4])
{
    const f4 a = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(y, off, 0, 16));
    v[0] = a[0]; v[1] = a[1]; v[2] = a[2]; v[3] = a[3];
}
template <typename T, int MODE>
__global__ __launch_bounds__(512, 2) void tri_solve_kernel(TriSolve<T> p)
{
    typedef SMfma<T> M;
    typedef typename M::acc_t acc_t;
    constexpr int NT = kSB / 16;                    // tiles across a block, and waves
    __shared__ T Ti[NT][16][17];                    // the inverses of the diagonal tiles
    __shared__ __align__(16) T Ys[2][kSB * kSR];    // staged Y_j
    __shared__ T Yd[kSB * kSR];                     // the own block's Y
    __shared__ int place, here[NT];                 // tiles of the block before that are staged
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int lc = lane & 15, lk = lane >> 4;
    if (threadIdx.x == 0) place = atomicAdd(p.ticket, 1);
    if (threadIdx.x < NT) here[threadIdx.x] = 0;
    lds_barrier();
    const int b = place / p.npass, ps = place % p.npass;
    const int64_t n = p.n, r0 = (int64_t)b * kSB, rw = r0 + 16 * w;
    const bool act = rw < n;                        // this wave has rows
    const int nt = (int)std::min<int64_t>(NT, (n - r0 + 15) / 16);
    const int64_t lrow = rw + lc < n ? rw + lc : n - 1;
    const T *pr = p.M + lrow * p.si;                // the lane's row
    if (MODE == kByRows) pr += lk * p.sj;
    else pr += tile_col<T, MODE>(0, lk) * p.sj;
    const int64_t ysize = (n + kSB - 1) / kSB * kSB * kSR;
    T *Y = p.Y + ps * ysize;
    const __amdgpu_buffer_rsrc_t yb =
        __builtin_amdgcn_make_buffer_rsrc(Y, 0, (int)(ysize * sizeof(T)), 0x00027000);

    // the diagonal tile's inverse, a column per lane (each of the four lane
    // groups does the same)
    if (act) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int c = lk + 4 * q;
            const bool in = lc >= c && rw + lc < n;
            const T *pd = p.M + (in ? (rw + lc) * p.si + (rw + c) * p.sj : 0);
            const T v = *pd;
            Ti[w][lc][c] = lc == c && (p.unit || !in) ? T(1) : (in ? v : T(0));
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        T x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            T s = i == lc ? T(1) : T(0);
#pragma unroll
            for (int j = 0; j < i; ++j) s = fma_t(-Ti[w][i][j], x[j], s);
            x[i] = s / Ti[w][i][i];
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
        for (int i = 0; i < 16; ++i) Ti[w][i][lc] = x[i];
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
    T inv[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) inv[q] = Ti[w][lc][M::row(lane, q)];

    // r; the tiles left of the diagonal one, in time for their use
    acc_t tot;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int64_t i = rw + M::row(lane, q);
        const int k = kSR * ps + lc;
        T v = T(0);
        if (i < n && k < p.nrhs) {
            v = p.R[i * p.ri + lc * p.rk + ps * p.rp];
            if (p.div) v = v / p.div[i * p.ds];
        }
        tot[q] = v;
    }
    T dg[NT - 1][4];
    auto load_diag = [&]() {
#pragma unroll
        for (int k = 0; k < NT - 1; ++k)
            if (act && k < w) load_tile<T, MODE>(pr, p.sj, r0 + 16 * k, dg[k]);
    };

    bool lost = false;
    T ua[NT][4], ub[NT][4], yv[4];
    const int goff = (threadIdx.x >> 2) * kSR + 4 * (threadIdx.x & 3);   // in a Y block
    const int srow = staged_row<T, MODE>(threadIdx.x >> 2);
    auto load_block = [&](int j, T (&u)[NT][4]) {
#pragma unroll
        for (int k = 0; k < NT; ++k)
            if (act) load_tile<T, MODE>(pr, p.sj, (int64_t)j * kSB + 16 * k, u[k]);
    };
    auto ask = [&](int j) {
        load_row4(yb, (int)(((int64_t)j * kSB * kSR + goff) * sizeof(T)), yv);
    };
    // tot −= M_bj Y_j with M_bj in use; M_b,j+1 into nxt
    auto link = [&](int j, T (&use)[NT][4], T (&nxt)[NT][4]) {
        for (unsigned spins = 0;; ++spins) {
            const bool miss = is_mark(yv[0]) || is_mark(yv[1]) || is_mark(yv[2]) || is_mark(yv[3]);
            if (!__any(miss) || lost) break;
            if (spins >= p.spin_limit) lost = true;
            __builtin_amdgcn_s_sleep(4);
            asm volatile("" ::: "memory");
            ask(j);
        }
        T *ys = Ys[j & 1];
#pragma unroll
        for (int e = 0; e < 4; ++e) ys[srow * kSR + 4 * (threadIdx.x & 3) + e] = yv[e];
        load_block(j + 1, nxt);
        if (j + 2 < b) ask(j + 1);
        lds_barrier();
        acc_t c = {T(0), T(0), T(0), T(0)};
        if (act) {
#pragma unroll
            for (int k = 0; k < NT; ++k)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    c = M::mma(use[k][q], ys[(16 * k + 4 * q + lk) * kSR + lc], c);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) tot[q] -= c[q];
    };
    acc_t s = {T(0), T(0), T(0), T(0)};
    if (b > 0) {
        int j = 0;
        if (b > 1) ask(0);
        if ((b - 1) & 1) {
            load_block(0, ub);
            link(0, ub, ua);
            j = 1;
        } else {
            load_block(0, ua);
        }
        for (; j < b - 1; j += 2) {
            link(j, ua, ub);
            link(j + 1, ub, ua);
        }
        load_diag();
        // the block before this one: wave k fetches tile k when it comes
        T *ys = Ys[(b - 1) & 1];
        {
            const int row = 16 * w + (lane >> 2);
            for (unsigned spins = 0;; ++spins) {
                asm volatile("" ::: "memory");
                load_row4(yb, (int)((((int64_t)(b - 1) * kSB + row) * kSR + 4 * (lane & 3)) * sizeof(T)),
                          yv);
                const bool miss = is_mark(yv[0]) || is_mark(yv[1]) || is_mark(yv[2]) || is_mark(yv[3]);
                if (!__any(miss) || lost) break;
                if (spins >= p.spin_limit) lost = true;
            }
            const int st = staged_row<T, MODE>(row);
#pragma unroll
            for (int e = 0; e < 4; ++e) ys[st * kSR + 4 * (lane & 3) + e] = yv[e];
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (lane == 0) __hip_atomic_store(&here[w], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        if (act) {
#pragma unroll
            for (int k = 0; k < NT; ++k) {
                while (__hip_atomic_load(&here[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == 0) {}
                asm volatile("" ::: "memory");
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    s = M::mma(ua[k][q], ys[(16 * k + 4 * q + lk) * kSR + lc], s);
            }
        }
    } else {
        load_diag();
    }
    // the diagonal block
    acc_t y = {T(0), T(0), T(0), T(0)};
#pragma unroll
    for (int k = 0; k < NT; ++k) {
        if (k < nt) {
            if (w == k) {
                __builtin_amdgcn_s_setprio(3);
#pragma unroll
                for (int q = 0; q < 4; ++q) y = M::mma(inv[q], tot[q] - s[q], y);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    y[q] = quiet(y[q]);
                    const int i = 16 * w + M::row(lane, q);
                    Yd[staged_row<T, MODE>(i) * kSR + lc] = y[q];
                    store_coherent(Y + (r0 + i) * kSR + lc, (T)y[q]);
                }
                __builtin_amdgcn_s_setprio(0);
            }
            lds_barrier();
            if (k < NT - 1 && act && k < w) {
                if (w == k + 1) __builtin_amdgcn_s_setprio(3);   // the next in the chain
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    s = M::mma(dg[k < NT - 1 ? k : 0][q], Yd[(16 * k + 4 * q + lk) * kSR + lc], s);
            }
        }
    }
    if (lost && p.err && lane == 0) store_coherent(p.err, 1);
    // the caller's result
    const int col = kSR * ps + lc;
    if (act && col < p.nrhs) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t i = rw + M::row(lane, q);
            if (i < n) {
                if (p.out) p.out[i * p.oi + col * p.ok] = p.mul ? p.mul[i * p.ms] * y[q] : (T)y[q];
                if (p.X) p.X[i * p.oi + col * p.ok] += (double)y[q];
            }
        }
    }
}

// Y (the exchange of one or more solves) all marks, their tickets zero.
template <typename T>
__global__ void tri_solve_prepare_kernel(int64_t cnt, T *Y, int *ticket, int solves)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < cnt) reinterpret_cast<typename NaNMark<T>::bits *>(Y)[i] = NaNMark<T>::value;
    if (i < solves) ticket[i] = 0;
}

// ---------------------------------------------------- symmetric residual --
constexpr int kVB = 64;    // rows of a block
// Blocks per rectangle side: the smaller, the more workgroups and the more
// partials a row (2 n/128 of 128 bytes against n/2 of A's elements).  Solve with
// two corrections, 2 -> 4 -> 8 per side: n = 1000 559 -> 672 -> 1146 µs, 8192 4.30 ->
// 4.36 -> 4.78 ms; n = 16384 18.9 ms with 2 and 4, and 4 takes half the workspace.
inline int symv_rb(int64_t n) { return n <= 8192 ? 2 : 4; }

// Symmetric product Y = A X over the lower triangle of A, each element of A
// read once.  Workgroup (I, J), J ≤ I, takes the rectangle of 64×64 blocks
// A_ij with i in rectangle row I, j in rectangle column J (and j ≤ i):
//   y_i += A_ij x_j                 summed into its row partial  Prow[J]
//   y_j += A_ijᵀ x_i   (j < i)      summed into its column partial Pcol[I]
// (diagonal blocks are mirrored from their lower half in LDS).  A row of
// rectangle row R thus has partials Prow[J] for J ≤ R and Pcol[I] for I ≥ R,
// each written by exactly one workgroup; symv_finish_kernel adds them in a
// fixed order, so the result does not depend on scheduling.  The next block
// is loaded into registers while the current one is multiplied.
template <int kRB>
__global__ __launch_bounds__(kST, 2) void symv_rect_kernel(int64_t n, const double *__restrict__ A,
                                                           int64_t lda,
                                                           const double *__restrict__ Xt,
                                                           double *__restrict__ Prow,
                                                           double *__restrict__ Pcol,
                                                           int64_t npad, int NR)
{
    typedef SMfma<double> M;
    constexpr int LDT = kVB + 1;
    __shared__ double Ts[kVB * LDT];           // A_ij column-major: (r, c) at [c·65 + r]
    __shared__ double xi[kVB * kSR], xj[kVB * kSR];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int lc = lane & 15, lk = lane >> 4;
    int rid = blockIdx.x, J = 0;
    while (rid >= NR - J) {
        rid -= NR - J;
        ++J;
    }
    const int I = J + rid;
    const int64_t nb = (n + kVB - 1) / kVB;
    const int64_t i0 = (int64_t)I * kRB, j0 = (int64_t)J * kRB;

    // thread t holds rows lane, columns w + 4u (u < 16) of a block and four
    // elements of its x_i; loads from clamped places, what is out of range
    // dropped when they are staged
    double ra[16], rx[4];
    auto gload = [&](int64_t i, int64_t j) {
        const int64_t row = i * kVB + lane, rc = row < n ? row : n - 1;
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int64_t col = j * kVB + w + 4 * u;
            ra[u] = A[rc + (col < n ? col : n - 1) * lda];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) rx[u] = Xt[i * kVB * kSR + t + kST * u];
    };
    d4 yr[kRB];
#pragma unroll
    for (int b = 0; b < kRB; ++b) yr[b] = d4{0.0, 0.0, 0.0, 0.0};
    gload(i0, j0);
    for (int bj = 0; bj < kRB; ++bj) {
        const int64_t j = j0 + bj;
        if (j >= nb) break;
#pragma unroll
        for (int u = 0; u < 4; ++u) xj[t + kST * u] = Xt[j * kVB * kSR + t + kST * u];
        d4 yc = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int bi = 0; bi < kRB; ++bi) {
            const int64_t i = i0 + bi;
            if (i >= nb || i < j) continue;
#pragma unroll
            for (int u = 0; u < 16; ++u) hold(ra[u]);
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                const bool in = i * kVB + lane < n && j * kVB + w + 4 * u < n;
                Ts[(w + 4 * u) * LDT + lane] = in ? ra[u] : 0.0;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) xi[t + kST * u] = rx[u];
            __syncthreads();
            if (i == j) {
                // upper half of a diagonal block from its lower half
                for (int e = t; e < kVB * kVB; e += kST) {
                    const int r = e % kVB, c = e / kVB;
                    if (r < c) Ts[c * LDT + r] = Ts[r * LDT + c];
                }
                __syncthreads();
            }
            // the next block of the rectangle: (i+1, j), else the first of column j+1
            {
                int64_t ni = i + 1, nj = j;
                if (bi + 1 >= kRB || ni >= nb) {
                    nj = j + 1;
                    ni = nj > i0 ? nj : i0;
                }
                if (nj < j0 + kRB && nj < nb && ni < nb && ni < i0 + kRB) gload(ni, nj);
            }
#pragma unroll
            for (int kq = 0; kq < kVB / 4; ++kq)
                yr[bi] = M::mma(Ts[(4 * kq + lk) * LDT + 16 * w + lc], xj[(4 * kq + lk) * kSR + lc],
                                yr[bi]);
            if (i != j) {
#pragma unroll
                for (int kq = 0; kq < kVB / 4; ++kq)
                    yc = M::mma(Ts[(16 * w + lc) * LDT + 4 * kq + lk], xi[(4 * kq + lk) * kSR + lc],
                                yc);
            }
            __syncthreads();
        }
        double *pc = Pcol + ((int64_t)I * npad + j * kVB + 16 * w) * kSR;
#pragma unroll
        for (int r = 0; r < 4; ++r) pc[M::row(lane, r) * kSR + lc] = yc[r];
    }
#pragma unroll
    for (int bi = 0; bi < kRB; ++bi) {
        const int64_t i = i0 + bi;
        if (i >= nb) break;
        double *pr = Prow + ((int64_t)J * npad + i * kVB + 16 * w) * kSR;
#pragma unroll
        for (int r = 0; r < 4; ++r) pr[M::row(lane, r) * kSR + lc] = yr[bi][r];
    }
}

// R = B − A X with A X = Σ_{J≤R} Prow[J] + Σ_{I≥R} Pcol[I] for the rows of
// rectangle row R, added in that order (type T, row-major n×16);
// nrm[k] += ‖r_k‖², nrm[16+k] += ‖x_k‖² over this workgroup's 64 rows.
template <typename T>
__global__ __launch_bounds__(kST) void symv_finish_kernel(int64_t n, const double *__restrict__ Prow,
                                                          const double *__restrict__ Pcol,
                                                          int64_t npad, int NR, int rb,
                                                          const double *__restrict__ Xt,
                                                          const double *__restrict__ B,
                                                          int64_t ldb, int nrhs, T *__restrict__ R,
                                                          double *nrm)
{
    __shared__ double sr[2 * kST];
    const int64_t r0 = (int64_t)blockIdx.x * kVB;
    const int Rr = (int)(blockIdx.x / rb);
    // every element this thread visits has k = threadIdx.x % 16 (256 is a
    // multiple of 16): accumulate locally, reduce over the 16 threads of each
    // k, one atomic per k and workgroup
    double rs = 0.0, xs = 0.0;
    for (int e = threadIdx.x; e < kVB * kSR; e += kST) {
        const int rl = e / kSR, k = e % kSR;
        const int64_t row = r0 + rl;
        if (row >= n) continue;
        double v = 0.0;
        if (k < nrhs) {
            double ax = 0.0;
            const double *pr = Prow + row * kSR + k, *pc = Pcol + row * kSR + k;
            int q = 0;
            for (; q + 8 <= NR + 1; q += 8) {   // eight in flight
                double p[8];
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    p[u] = q + u <= Rr ? pr[(int64_t)(q + u) * npad * kSR]
                                       : pc[(int64_t)(q + u - 1) * npad * kSR];
#pragma unroll
                for (int u = 0; u < 8; ++u) ax += p[u];
            }
            for (; q < NR + 1; ++q)
                ax += q <= Rr ? pr[(int64_t)q * npad * kSR] : pc[(int64_t)(q - 1) * npad * kSR];
            v = B[row + k * ldb] - ax;
            const double x = Xt[row * kSR + k];
            xs += x * x;
            rs += v * v;
        }
        R[row * kSR + k] = (T)v;
    }
    sr[threadIdx.x] = rs;
    sr[kST + threadIdx.x] = xs;
    __syncthreads();
    if (threadIdx.x < kSR && (int)threadIdx.x < nrhs) {
        double a = 0.0, c = 0.0;
        for (int q = threadIdx.x; q < kST; q += kSR) {
            a += sr[q];
            c += sr[kST + q];
        }
        atomicAdd(nrm + threadIdx.x, a);
        atomicAdd(nrm + kSR + threadIdx.x, c);
    }
}
// Xt (row-major npad×16) = X's first nrhs columns, zero elsewhere.
__global__ void rowmajor16_kernel(int64_t n, int64_t npad, int nrhs, const double *__restrict__ X,
                                  int64_t ldx, double *__restrict__ Xt)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < npad * kSR) {
        const int64_t row = e / kSR;
        const int k = (int)(e % kSR);
        Xt[e] = (k < nrhs && row < n) ? X[row + k * ldx] : 0.0;
    }
}
}  // namespace

size_t tri_solve_elems(int64_t n, int64_t nrhs)
{
    return (size_t)(cdiv(n, kSB) * kSB) * kSR * cdiv(nrhs, kSR);
}

template <typename T>
int tri_solve_prepare(hipStream_t s, int64_t cnt, T *Y, int *ticket, int solves)
{
    hipLaunchKernelGGL((tri_solve_prepare_kernel<T>), dim3((unsigned)cdiv(std::max<int64_t>(cnt, solves), 256)),
                       dim3(256), 0, s, cnt, Y, ticket, solves);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}

template <typename T>
int tri_solve(hipStream_t s, TriSolve<T> p)
{
    if (p.n <= 0 || p.nrhs <= 0) return GLA_OK;
    if (reinterpret_cast<uintptr_t>(p.Y) % 16 != 0) {   // read 16 bytes at a time
        set_error("tri_solve: the exchange is not aligned to 16 bytes");
        return GLA_ERR_UNSUPPORTED;
    }
    p.npass = (int)cdiv(p.nrhs, kSR);
    const dim3 grid((unsigned)(cdiv(p.n, kSB) * p.npass));
    if (p.si == 1 || p.si == -1)
        hipLaunchKernelGGL((tri_solve_kernel<T, kByRows>), grid, dim3(512), 0, s, p);
    else if (p.sj == 1)
        hipLaunchKernelGGL((tri_solve_kernel<T, kByCols>), grid, dim3(512), 0, s, p);
    else
        hipLaunchKernelGGL((tri_solve_kernel<T, kByColsRev>), grid, dim3(512), 0, s, p);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}

// R = B − sym(A) X; Xt scratch: npad×16 FP64 followed by the rectangle
// partials (symv_scratch(n) doubles in all); nrm[32] must be zero on entry.
template <typename T>
int symv_residual(hipStream_t s, int64_t n, const double *A, int64_t lda, const double *X,
                  int64_t ldx, const double *B, int64_t ldb, int nrhs, double *Xt, T *R,
                  double *nrm)
{
    if (n <= 0) return GLA_OK;
    const int64_t nb = cdiv(n, kVB), npad = nb * kVB;
    const int rb = symv_rb(n), NR = (int)cdiv(nb, rb);
    double *Prow = Xt + npad * kSR;
    double *Pcol = Prow + (int64_t)NR * npad * kSR;
    hipLaunchKernelGGL(rowmajor16_kernel, dim3((unsigned)cdiv(npad * kSR, 256)), dim3(256), 0, s,
                       n, npad, nrhs, X, ldx, Xt);
    GLA_LAUNCH_CHECK();
    const dim3 grid((unsigned)(NR * (NR + 1) / 2));
    if (rb == 2)
        hipLaunchKernelGGL(symv_rect_kernel<2>, grid, dim3(kST), 0, s, n, A, lda, Xt, Prow, Pcol,
                           npad, NR);
    else
        hipLaunchKernelGGL(symv_rect_kernel<4>, grid, dim3(kST), 0, s, n, A, lda, Xt, Prow, Pcol,
                           npad, NR);
    GLA_LAUNCH_CHECK();
    hipLaunchKernelGGL((symv_finish_kernel<T>), dim3((unsigned)nb), dim3(kST), 0, s, n, Prow, Pcol,
                       npad, NR, rb, Xt, B, ldb, nrhs, R, nrm);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}

size_t symv_scratch(int64_t n)
{
    const int64_t nb = cdiv(n, kVB), NR = cdiv(nb, symv_rb(n));
    return (size_t)(nb * kVB) * kSR * (1 + 2 * NR);
}

template int tri_solve_prepare<double>(hipStream_t, int64_t, double *, int *, int);
template int tri_solve_prepare<float>(hipStream_t, int64_t, float *, int *, int);
template int tri_solve<double>(hipStream_t, TriSolve<double>);
template int tri_solve<float>(hipStream_t, TriSolve<float>);
template int symv_residual<double>(hipStream_t, int64_t, const double *, int64_t, const double *,
                                   int64_t, const double *, int64_t, int, double *, double *,
                                   double *);
template int symv_residual<float>(hipStream_t, int64_t, const double *, int64_t, const double *,
                                  int64_t, const double *, int64_t, int, double *, float *,
                                  double *);

}  // namespace gla
