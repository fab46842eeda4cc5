// Two-sided Householder reductions (FP64/FP32, real):
//   symtriLower!/symtriUpper!  src/eigenSelfAdjoint.jl:450-564  (A = Q T Qᵀ)
//   bidiagonalize!             src/svd.jl:328-381               (A = Ql B Qrᵀ)
//
// Both produce the reference's reflectors (Julia stdlib reflector!: β =
// −copysign(‖x‖, x₁), v₁ = 1, v = x/(x₁ − β), τ = (x₁ − β)/(−β)) in the
// reference's packing; the per-column rank-2 (or left/right) updates the
// reference applies at once are deferred across a panel of nb columns and
// applied as MFMA GEMMs at the panel's end — the same matrices up to
// rounding.
//
// symtri (lower; upper runs as lower on J A J, J the reversal, which maps
// symtriUpper!'s bottom-up sweep onto symtriLower!'s).  For column c of a
// panel starting at k (j = c − k), with the trailing matrix Ã kept as it
// was at the panel's start and the panel's earlier reflectors in V, W
// (Ã_now = Ã − V Wᵀ − W Vᵀ):
//   tri_col:    a = A[c:n, c] − V W[c,:]ᵀ − W V[c,:]ᵀ (the column brought up
//               to date; a[0] is the diagonal d_c); partial ‖a[1:]‖²;
//   tri_symv:   the reflector's scalars from those partials, then
//               p = Ã[c+1:n, c+1:n] v (the symmetric product from the lower
//               triangle, each 64×64 block read once and used for both
//               A_IJ v_J and A_IJᵀ v_I, partials per block in a fixed
//               order) and Wᵀv, Vᵀv partials;
//   tri_w:      v written into A and V, u = τ (p − V (Wᵀv) − W (Vᵀv)) into
//               W, partial vᵀu;
//   (next tri_col, or tri_wfin at the panel's end): w = u − (τ vᵀu / 2) v,
//               so that Ã_new = Ã_now − v wᵀ − w vᵀ = H Ã_now H.
// Panel end: Ã[k+nb:, k+nb:] −= V Wᵀ + W Vᵀ (two lower-triangle GEMMs).
#include <algorithm>

#include "gla_coherent.hpp"
#include "gla_internal.hpp"

namespace gla {

namespace {

#define GLA_TRY(expr)                  \
    do {                               \
        int _rc = (expr);              \
        if (_rc != GLA_OK) return _rc; \
    } while (0)

constexpr int kTB = 64;       // symmetric-product block
constexpr int kPanel = 32;    // panel width (columns of V, W)

// Scalars of the current column, written by tri_symv's first workgroup.
enum { S_TAU = 0, S_XI = 1, S_BETA = 2, S_UNEXT = 3, S_COUNT = 8 };

constexpr int kRPB = 64;      // rows per workgroup of the row kernels (4 lanes per row)

template <typename T>
__device__ __forceinline__ T wave_sum(T v)
{
    return wave_sum_dpp(v);
}

// Fixed-order sum of part[0..cnt) by one workgroup (every thread gets it).
template <typename T>
__device__ T block_sum_fixed(const T *part, int cnt, T *sh)
{
    T s = T(0);
    for (int i = threadIdx.x; i < cnt; i += blockDim.x) s += part[i];
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    T r = T(0);
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) r += sh[w];
    __syncthreads();
    return r;
}

// The reflector! scalars of column c from ‖a[1:]‖² (partials) and a[1]:
// ξ₁ = a₁ + ν (the divisor of the tail), τ = ξ₁/ν, β = −ν; a zero norm
// leaves the column alone (τ = 0, ξ₁ = 1).
template <typename T>
__device__ __forceinline__ void reflector_scalars(T nrm2, T x1, T &xi, T &tau, T &beta)
{
    const T normu = sqrt(nrm2);
    if (normu == T(0)) {
        xi = T(1);
        tau = T(0);
        beta = x1;
        return;
    }
    const T nu = copysign(normu, x1);
    xi = x1 + nu;
    tau = xi / nu;
    beta = -nu;
}

// Column c brought up to date with the panel's reflectors 0..j−1; before
// that, W[:, j−1] (holding u) becomes w = u − (ξ/2) v for rows ≥ c.  Four
// lanes per row, lane k taking the reflectors l ≡ k (mod 4) (loads from
// clamped indices, all issued at once), summed over the quad.
template <typename T>
__global__ __launch_bounds__(256) void tri_col_kernel(int64_t n, int64_t c, int j, T *A,
                                                      int64_t lda, T *V, T *W, int64_t ldv,
                                                      const T *qpart, int qcnt, const T *scal,
                                                      T *npart)
{
    __shared__ T sh[8];
    __shared__ T wc[kPanel], vc[kPanel];
    const int t = threadIdx.x, k = t & 3;
    const int64_t i = c + (int64_t)blockIdx.x * kRPB + (t >> 2);
    const bool in = i < n;
    const int64_t ic = in ? i : n - 1;
    T wprev_c = T(0), half_xi = T(0);
    if (j > 0) {
        const T vu = block_sum_fixed(qpart, qcnt, sh);
        half_xi = T(0.5) * scal[S_TAU] * vu;              // ξ/2 = τ vᵀu / 2
        wprev_c = scal[S_UNEXT] - half_xi;                // row c: v_c = 1
    }
    if (t < kPanel) {
        wc[t] = t < j ? (t == j - 1 ? wprev_c : W[c + (int64_t)t * ldv]) : T(0);
        vc[t] = t < j ? V[c + (int64_t)t * ldv] : T(0);
    }
    __syncthreads();
    T part = T(0);
    if (j > 0) {
        T wv[kPanel / 4], vv[kPanel / 4];
#pragma unroll
        for (int u = 0; u < kPanel / 4; ++u) {
            const int l = k + 4 * u, lc = l < j ? l : 0;
            wv[u] = W[ic + (int64_t)lc * ldv];
            vv[u] = V[ic + (int64_t)lc * ldv];
        }
#pragma unroll
        for (int u = 0; u < kPanel / 4; ++u) {
            const int l = k + 4 * u;
            T wil = wv[u];
            if (l == j - 1) {
                wil -= half_xi * vv[u];
                if (in) W[i + (int64_t)l * ldv] = wil;
            }
            if (l < j) part += vv[u] * wc[l] + wil * vc[l];
        }
    }
    part = quad_sum(part);
    T a = T(0);
    if (in) {
        a = A[i + c * lda] - part;
        if (k == 0) A[i + c * lda] = a;
    }
    T s = (in && i > c && k == 0) ? a * a : T(0);
    s = wave_sum(s);
    if ((t & 63) == 0) sh[t >> 6] = s;
    __syncthreads();
    if (t == 0) npart[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// After the panel's last column: W[:, j] (u) becomes w for rows ≥ c.
template <typename T>
__global__ void tri_wfin_kernel(int64_t n, int64_t c, int j, T *V, T *W, int64_t ldv,
                                const T *qpart, int qcnt, const T *scal)
{
    __shared__ T sh[8];
    const T vu = block_sum_fixed(qpart, qcnt, sh);
    const T half_xi = T(0.5) * scal[S_TAU] * vu;
    const int64_t i = c + (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) W[i + (int64_t)j * ldv] -= half_xi * V[i + (int64_t)j * ldv];
}

// v_r of row r ≥ r0 = c + 1 from the unscaled column.
template <typename T>
__device__ __forceinline__ T vval(const T *A, int64_t lda, int64_t c, int64_t r, T xi)
{
    return r == c + 1 ? T(1) : A[r + c * lda] / xi;
}

// p = Ã v over the lower-stored trailing block, blocks (I, J), I ≥ J, of
// 64×64; P[s·m + r] is the contribution of the block pairing row block
// r/64 with block s (rows relative to r0).  Diagonal blocks add Wᵀv and
// Vᵀv partials Y1[I·kPanel + l], Y2[I·kPanel + l].
template <typename T>
__global__ __launch_bounds__(256) void tri_symv_kernel(int64_t n, int64_t c, int j, const T *A,
                                                       int64_t lda, const T *V, const T *W,
                                                       int64_t ldv, const T *npart, int ncnt,
                                                       T *P, T *Y1, T *Y2, T *scal, T *tau_out)
{
    __shared__ T sh[8];
    __shared__ T srow[4][kTB];
    const int64_t r0 = c + 1, m = n - r0;
    // block (I, J) from the linear id: row I, J ≤ I
    const int64_t q = blockIdx.x;
    int64_t I = (int64_t)((sqrt(8.0 * (double)q + 1.0) - 1.0) / 2.0);
    while ((I + 1) * (I + 2) / 2 <= q) ++I;
    while (I * (I + 1) / 2 > q) --I;
    const int64_t J = q - I * (I + 1) / 2;
    const T nrm2 = block_sum_fixed(npart, ncnt, sh);
    T xi, tau, beta;
    reflector_scalars(nrm2, A[r0 + c * lda], xi, tau, beta);
    if (q == 0 && threadIdx.x == 0) {
        scal[S_TAU] = tau;
        scal[S_XI] = xi;
        scal[S_BETA] = beta;
        tau_out[c] = tau;
    }
    const int t = threadIdx.x, a = t & 15, b = t >> 4, lane = t & 63, wv = t >> 6;
    // this thread's rows RB + 16u (consecutive lanes read consecutive rows,
    // so each load instruction reads whole cache lines) and columns C0 + u;
    // the loads are unconditional (clamped indices), out-of-range values
    // and the upper part of a diagonal block replaced by zero
    const int64_t RB = r0 + I * kTB + a, C0 = r0 + J * kTB + 4 * b;
    T x[4][4];
    T vr[4], vcv[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int64_t rr = RB + 16 * u, cc = C0 + u;
        vr[u] = rr < n ? vval(A, lda, c, rr, xi) : T(0);
        vcv[u] = cc < n ? vval(A, lda, c, cc, xi) : T(0);
    }
#pragma unroll
    for (int cc = 0; cc < 4; ++cc)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
            const int64_t gi = RB + 16 * rr, gj = C0 + cc;
            const int64_t gic = gi < n ? gi : n - 1, gjc = gj < n ? gj : n - 1;
            const T v = A[gic + gjc * lda];
            x[cc][rr] = (gi < n && gj < n && gi >= gj) ? v : T(0);
        }
    // row sums (A_IJ v_J) and column sums (A_IJᵀ v_I, strictly lower part
    // only on a diagonal block)
    T s[4], qc[4];
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
        T acc = T(0);
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) acc += x[cc][rr] * vcv[cc];
        s[rr] = acc;
    }
#pragma unroll
    for (int cc = 0; cc < 4; ++cc) {
        T acc = T(0);
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
            const bool use = I != J || (RB + 16 * rr > C0 + cc);
            acc += use ? x[cc][rr] * vr[rr] : T(0);
        }
        qc[cc] = acc;
    }
    // s: reduce over b (lane bits 4, 5, then the four waves)
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
        s[rr] += __shfl_xor(s[rr], 16);
        s[rr] += __shfl_xor(s[rr], 32);
    }
    if (lane < 16)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) srow[wv][a + 16 * rr] = s[rr];
    // qc: reduce over a (lane bits 0..3)
#pragma unroll
    for (int cc = 0; cc < 4; ++cc) qc[cc] = row_sum16(qc[cc]);
    __syncthreads();
    if (I == J) {
        // one slot for the diagonal block: row sums plus the transposed part
        __shared__ T scol[kTB];
        if (a == 0)
#pragma unroll
            for (int cc = 0; cc < 4; ++cc) scol[4 * b + cc] = qc[cc];
        __syncthreads();
        if (t < kTB) {
            const int64_t r = I * kTB + t;
            if (r < m) P[J * m + r] = srow[0][t] + srow[1][t] + srow[2][t] + srow[3][t] + scol[t];
        }
        // Wᵀv and Vᵀv over this block's rows: wave wv takes l ≡ wv (mod 4),
        // all loads issued before the sums
        const int64_t gr = r0 + I * kTB + lane;
        const int64_t grc = gr < n ? gr : n - 1;
        const T vg = gr < n ? vval(A, lda, c, gr, xi) : T(0);
        T wl[kPanel / 4], vl[kPanel / 4];
#pragma unroll
        for (int u = 0; u < kPanel / 4; ++u) {
            const int l = wv + 4 * u, lc = l < j ? l : 0;
            wl[u] = W[grc + (int64_t)lc * ldv];
            vl[u] = V[grc + (int64_t)lc * ldv];
        }
#pragma unroll
        for (int u = 0; u < kPanel / 4; ++u) {
            const int l = wv + 4 * u;
            if (l < j) {
                const T y1 = wave_sum(wl[u] * vg);
                const T y2 = wave_sum(vl[u] * vg);
                if (lane == 0) {
                    Y1[I * kPanel + l] = y1;
                    Y2[I * kPanel + l] = y2;
                }
            }
        }
    } else {
        if (t < kTB) {
            const int64_t r = I * kTB + t;
            if (r < m) P[J * m + r] = srow[0][t] + srow[1][t] + srow[2][t] + srow[3][t];
        }
        if (a == 0)
#pragma unroll
            for (int cc = 0; cc < 4; ++cc) {
                const int64_t r = J * kTB + 4 * b + cc;
                if (r < m) P[I * m + r] = qc[cc];
            }
    }
}

// v into A (below the subdiagonal) and V, β on the subdiagonal;
// u = τ (p − V y1 − W y2) into W[:, j]; partial vᵀu.  Four lanes per row:
// lane k sums the block contributions s ≡ k (mod 4) of p and the
// reflectors l ≡ k (mod 4), then the quad sums; y1, y2 (Wᵀv, Vᵀv) are
// summed over the blocks' partials by the whole workgroup, fixed order.
template <typename T>
__global__ __launch_bounds__(256) void tri_w_kernel(int64_t n, int64_t c, int j, T *A, int64_t lda,
                                                    T *V, T *W, int64_t ldv, const T *P, int nbk,
                                                    const T *Y1, const T *Y2, T *scal, T *qpart)
{
    __shared__ T sh[8];
    __shared__ T y1[kPanel], y2[kPanel];
    __shared__ T ys[2][8][kPanel];
    const int t = threadIdx.x, k = t & 3;
    const int64_t r0 = c + 1, m = n - r0;
    const T tau = scal[S_TAU], xi = scal[S_XI], beta = scal[S_BETA];
    {
        const int l = t & (kPanel - 1), pp = t / kPanel;   // 8 parts of the block sums
        T s1 = T(0), s2 = T(0);
        if (l < j)
            for (int I = pp; I < nbk; I += 8) {
                s1 += Y1[I * kPanel + l];
                s2 += Y2[I * kPanel + l];
            }
        ys[0][pp][l] = s1;
        ys[1][pp][l] = s2;
    }
    __syncthreads();
    if (t < kPanel) {
        T s1 = T(0), s2 = T(0);
#pragma unroll
        for (int pp = 0; pp < 8; ++pp) {
            s1 += ys[0][pp][t];
            s2 += ys[1][pp][t];
        }
        y1[t] = s1;
        y2[t] = s2;
    }
    __syncthreads();
    const int64_t r = r0 + (int64_t)blockIdx.x * kRPB + (t >> 2);
    const bool in = r < n;
    const int64_t rc = in ? r : n - 1, rr = rc - r0;
    T p0 = T(0), p1 = T(0);
    int sblk = k;
    for (; sblk + 4 < nbk; sblk += 8) {
        p0 += P[(int64_t)sblk * m + rr];
        p1 += P[(int64_t)(sblk + 4) * m + rr];
    }
    if (sblk < nbk) p0 += P[(int64_t)sblk * m + rr];
    T p = p0 + p1;
    if (j > 0) {
        T wv[kPanel / 4], vv[kPanel / 4];
#pragma unroll
        for (int u = 0; u < kPanel / 4; ++u) {
            const int l = k + 4 * u, lc = l < j ? l : 0;
            vv[u] = V[rc + (int64_t)lc * ldv];
            wv[u] = W[rc + (int64_t)lc * ldv];
        }
#pragma unroll
        for (int u = 0; u < kPanel / 4; ++u) {
            const int l = k + 4 * u;
            if (l < j) p -= vv[u] * y1[l] + wv[u] * y2[l];
        }
    }
    p = quad_sum(p);
    T vu = T(0);
    if (in && k == 0) {
        const T v = r == r0 ? T(1) : A[r + c * lda] / xi;
        const T u = tau * p;
        W[r + (int64_t)j * ldv] = u;
        V[r + (int64_t)j * ldv] = v;
        A[r + c * lda] = r == r0 ? beta : v;
        if (r == r0) scal[S_UNEXT] = u;
        vu = v * u;
    }
    vu = wave_sum(vu);
    if ((t & 63) == 0) sh[t >> 6] = vu;
    __syncthreads();
    if (t == 0) qpart[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// ---- symtriLower! with the matrix in registers ----
// One launch for orders up to 2048.  Workgroup g of P = ⌈n/8⌉ holds the eight
// rows g + P k of the full symmetric matrix; thread 2g' + f of every workgroup
// holds the four columns g' + P (4f + u).  Every workgroup keeps the current
// column x and the vectors v, p, w of the whole order, spread over its threads
// like the columns.  Per column c:
//   the workgroup that holds row c + 1 publishes it (by symmetry the column
//   c + 1 as it stands);  the reflector's scalars from x, v;  p = Ã v for the
//   own rows (both triangles are held, so a row's sum is complete), published;
//   all workgroups gather p and the row;  w = τ p − (τ² vᵀp / 2) v;  the next
//   column x = Ã[:, c+1] − v w[c+1] − w v[c+1] in every workgroup alike, and
//   Ã −= v wᵀ + w vᵀ on the own rows (src/eigenSelfAdjoint.jl:466-491).
// So one exchange per column, and nothing but two vectors moves, in the order
// [g][k] in which a workgroup writes one line and a thread reads 32 bytes.
// Each column has an exchange region of its own, filled beforehand with a
// signalling-NaN pattern no arithmetic produces: a value is its own arrival
// mark.  All workgroups must be resident: such launches, and the QR panels,
// which wait within a launch too, run beside one another only where all fit
// (resident_begin).  Two workgroups fit on a CU, but none beside a panel's.  A
// wait that gives up makes the result NaN.
// Bound: latency.  n = 2048 FP64: 10.4 ms, 5.1 µs a column (3.2 at n = 512),
// about half of it the exchange; the three launches per column of the
// deferred form took 38 ms.  With p and the row in index order (eight
// scattered loads a thread, every one polled) 16.8 ms.
// Accuracy: over 224 matrices of order 17…80 the error against a __float128
// evaluation is 0.62 of the FP64 oracle's (0.63 the deferred form; 0.76 with
// the two products of the update subtracted one after the other).
constexpr int kTRRows = 8;           // rows per workgroup
constexpr int kTRMax = 2048;         // largest order: 256 workgroups of 512 threads

template <typename T>
__global__ void mark_kernel(int64_t cnt, T *p)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    typedef typename NaNMark<T>::bits B;
    if (i < cnt) reinterpret_cast<B *>(p)[i] = NaNMark<T>::value;
}

// Sums of v[0…7] over the wave: the lanes with l % 8 = 0 hold the total of
// v[4·bit5 + 2·bit4 + bit3].
template <typename T>
__device__ __forceinline__ T wave_rows8(const T v[8])
{
    const bool b3 = threadIdx.x & 8;
    T u[4], w[2];
#pragma unroll
    for (int k = 0; k < 4; ++k) u[k] = pair_sum32<T>(v[k], v[k + 4]);
#pragma unroll
    for (int k = 0; k < 2; ++k) w[k] = pair_sum16<T>(u[k], u[k + 2]);
    T z = (b3 ? w[1] : w[0]) + dppmov<0x128>(b3 ? w[0] : w[1]);   // row_ror:8
    z += dppmov<0xB1>(z);
    z += dppmov<0x4E>(z);
    z += dppmov<0x141>(z);
    return z;
}

// Four consecutive values, device-coherent.
__device__ __forceinline__ void store4_coherent(double *p, const double v[4])
{
    typedef double d2 __attribute__((ext_vector_type(2)));
    const d2 a = {v[0], v[1]}, b = {v[2], v[3]};
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\t"
                 "global_store_dwordx4 %0, %2, off offset:16 sc1\n\ts_nop 1" ::"v"(p), "v"(a), "v"(b)
                 : "memory");
}
__device__ __forceinline__ void store4_coherent(float *p, const float v[4])
{
    const f4 a = {v[0], v[1], v[2], v[3]};
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(a) : "memory");
}
__device__ __forceinline__ void load4_coherent(const double *p, double v[4])
{
    typedef double d2 __attribute__((ext_vector_type(2)));
    d2 a, b;
    asm volatile("global_load_dwordx4 %0, %2, off sc1\n\t"
                 "global_load_dwordx4 %1, %2, off offset:16 sc1\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(a), "=&v"(b)
                 : "v"(p)
                 : "memory");
    v[0] = a[0]; v[1] = a[1]; v[2] = b[0]; v[3] = b[1];
}
__device__ __forceinline__ void load4_coherent(const float *p, float v[4])
{
    f4 a;
    asm volatile("global_load_dwordx4 %0, %1, off sc1\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(a)
                 : "v"(p)
                 : "memory");
    v[0] = a[0]; v[1] = a[1]; v[2] = a[2]; v[3] = a[3];
}
// The same from two places, in one round trip.
__device__ __forceinline__ void load4x2_coherent(const double *p, const double *q, double v[4],
                                                 double w[4])
{
    typedef double d2 __attribute__((ext_vector_type(2)));
    d2 a, b, c, d;
    asm volatile("global_load_dwordx4 %0, %4, off sc1\n\t"
                 "global_load_dwordx4 %1, %4, off offset:16 sc1\n\t"
                 "global_load_dwordx4 %2, %5, off sc1\n\t"
                 "global_load_dwordx4 %3, %5, off offset:16 sc1\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(a), "=&v"(b), "=&v"(c), "=&v"(d)
                 : "v"(p), "v"(q)
                 : "memory");
    v[0] = a[0]; v[1] = a[1]; v[2] = b[0]; v[3] = b[1];
    w[0] = c[0]; w[1] = c[1]; w[2] = d[0]; w[3] = d[1];
}
__device__ __forceinline__ void load4x2_coherent(const float *p, const float *q, float v[4],
                                                 float w[4])
{
    f4 a, b;
    asm volatile("global_load_dwordx4 %0, %2, off sc1\n\t"
                 "global_load_dwordx4 %1, %3, off sc1\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(a), "=&v"(b)
                 : "v"(p), "v"(q)
                 : "memory");
    v[0] = a[0]; v[1] = a[1]; v[2] = a[2]; v[3] = a[3];
    w[0] = b[0]; w[1] = b[1]; w[2] = b[2]; w[3] = b[3];
}

template <typename T>
struct TriResP {
    T *A;
    int64_t lda;
    int n;
    T *tau;
    T *xch;              // [n columns][2][P][8]
    unsigned spin_limit;
};

template <typename T>
__global__ __launch_bounds__(512, 4) void tri_resident_kernel(TriResP<T> q)
{
    constexpr int R = kTRRows, U = 4;
    __shared__ T nred[8], vred[8], red[8][R], prow[R], vrow[R], x1s, p1s;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6, nw = blockDim.x >> 6;
    const int g = blockIdx.x, P = gridDim.x, n = q.n;
    const int64_t lda = q.lda;
    // this thread's columns i0 + P u; threads past 2P hold none
    const int gi = t >> 1, f = t & 1;
    const bool act = gi < P;
    const int i0 = act ? gi + 4 * P * f : n;
    const int eo = act ? gi * R + 4 * f : 0;          // its place in an exchanged vector

    T a[R][U], x[U];
#pragma unroll
    for (int k = 0; k < R; ++k)
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int r = g + P * k, i = i0 + P * u;
            const bool in = r < n && i < n;
            const int hi = r > i ? r : i, lo = r > i ? i : r;
            const T v = q.A[in ? hi + (int64_t)lo * lda : 0];
            a[k][u] = in ? quiet(v) : T(0);
        }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int i = i0 + P * u;
        const T v = q.A[i < n ? i : 0];
        x[u] = i < n ? v : T(0);
    }
    bool lost = false;
    int gc = 0, kc = 0;                               // c = gc + P kc
    for (int c = 0; c < n - 2; ++c) {
        T *pc = q.xch + (int64_t)c * 2 * P * R, *yc = pc + P * R;
        const int c1 = c + 1;
        const int g1 = gc + 1 < P ? gc + 1 : 0, k1 = gc + 1 < P ? kc : kc + 1;   // c + 1
        // row c + 1, by the workgroup that holds it
        if (g1 == g && act) {
            T y[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                y[u] = a[0][u];
#pragma unroll
                for (int k = 1; k < R; ++k) y[u] = k == k1 ? T(a[k][u]) : T(y[u]);
            }
            store4_coherent(yc + eo, y);
        }
        // ‖x[c+1:]‖² and x[c+1]
        T sq = T(0);
#pragma unroll
        for (int u = 0; u < U; ++u) sq = i0 + P * u > c ? fma_t(x[u], x[u], sq) : sq;
        sq = wave_sum(sq);
        if (lane == 0) nred[wv] = sq;
        const bool own1 = t == 2 * g1 + (k1 >> 2);
        if (own1) x1s = (k1 & 2) ? ((k1 & 1) ? x[3] : x[2]) : ((k1 & 1) ? x[1] : x[0]);
        lds_barrier();
        T nrm2 = T(0);
        for (int w = 0; w < nw; ++w) nrm2 += nred[w];
        const T nrm = sqrt(nrm2);
        const T x1 = x1s;
        const bool live = nrm != T(0);
        const T nu = copysign(nrm, x1), xi = x1 + nu;
        const T tau = live ? xi / nu : T(0);
        const T rxi = live ? T(1) / xi : T(1);
        T v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + P * u;
            v[u] = i > c1 ? x[u] * rxi : (i == c1 ? T(1) : T(0));
        }
        if (gi == g)
#pragma unroll
            for (int u = 0; u < U; ++u) vrow[4 * f + u] = v[u];
        // p for the own rows
        T s[R];
#pragma unroll
        for (int k = 0; k < R; ++k) {
            T acc = T(0);
#pragma unroll
            for (int u = 0; u < U; ++u) acc = fma_t(a[k][u], v[u], acc);
            s[k] = acc;
        }
        const T z = wave_rows8<T>(s);
        if ((lane & 7) == 0) red[wv][4 * (lane >> 5) + 2 * ((lane >> 4) & 1) + ((lane >> 3) & 1)] = z;
        lds_barrier();
        if (wv == 0 && lane < R) {
            typedef typename NaNMark<T>::bits B;
            T p = T(0);
            for (int w = 0; w < nw; ++w) p += red[w][lane];
            // rows at or before column c: nobody uses them, but their place
            // must not keep the mark
            const int r = g + P * lane;
            p = r > c && r < n ? p : T(0);
            store_coherent(reinterpret_cast<B *>(pc + g * R + lane), __builtin_bit_cast(B, p));
            prow[lane] = p;
        }
        // gather p and row c + 1
        T p[U], y[U];
        {
            auto marked = [](const T (&m)[U]) {
                return is_mark(m[0]) || is_mark(m[1]) || is_mark(m[2]) || is_mark(m[3]);
            };
            unsigned spins = 0;
            load4x2_coherent(pc + eo, yc + eo, p, y);
            while (!lost && __any(marked(p))) {
                load4_coherent(pc + eo, p);
                if (++spins > q.spin_limit) lost = true;
            }
            while (!lost && __any(marked(y))) {
                load4_coherent(yc + eo, y);
                if (++spins > q.spin_limit) lost = true;
            }
        }
        T vp = T(0);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + P * u;
            const bool in = i > c && i < n;
            p[u] = in ? p[u] : T(0);
            y[u] = in ? y[u] : T(0);
            vp = fma_t(v[u], p[u], vp);
        }
        vp = wave_sum(vp);
        if (lane == 0) vred[wv] = vp;
        if (own1) p1s = (k1 & 2) ? ((k1 & 1) ? p[3] : p[2]) : ((k1 & 1) ? p[1] : p[0]);
        lds_barrier();
        // column c: the diagonal, β, v.  Only now: the waves of this workgroup
        // have between them gathered every row, so every workgroup has loaded
        // its part of A
        if (gc == g) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = i0 + P * u;
                if (i >= c && i < n)
                    q.A[i + c * lda] = i == c || !live ? x[u] : (i == c1 ? -nu : v[u]);
            }
            if (t == 0) q.tau[c] = tau;
        }
        vp = T(0);
        for (int w = 0; w < nw; ++w) vp += vred[w];
        const T gam = T(0.5) * tau * (tau * vp);
        const T w1 = tau * p1s - gam;
        T w[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            w[u] = tau * p[u] - gam * v[u];
            x[u] = y[u] - fma_t(v[u], w1, w[u]);
        }
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const T vk = vrow[k], wk = tau * prow[k] - gam * vk;
            // both products first: one rounding at the element's own magnitude
#pragma unroll
            for (int u = 0; u < U; ++u) a[k][u] -= fma_t(wk, v[u], vk * w[u]);
        }
        gc = g1;
        kc = k1;
    }
    // the last 2×2 block
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int i = i0 + P * u;
        if (g == 0 && i >= n - 2 && i < n) q.A[i + (int64_t)(n - 2) * lda] = x[u];
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (g + P * k == n - 1 && i == n - 1) q.A[(n - 1) * (lda + 1)] = a[k][u];
    }
}

// Orders the resident kernel takes.
inline bool tri_resident_fits(int64_t n, int num_cus)
{
    return n >= 3 && n <= kTRMax && cdiv(n, kTRRows) <= num_cus;
}

// symtriLower! by the resident kernel; *done = false (and nothing queued) if
// it cannot run here (resident_begin).
template <typename T>
int tri_resident(Handle *h, hipStream_t s, int64_t n, T *A, int64_t lda, T *tau, T *xch, bool *done)
{
    const int64_t P = cdiv(n, kTRRows);
    *done = resident_begin(h, s, P);
    if (!*done) return GLA_OK;
    const int64_t cnt = n * 2 * P * kTRRows;
    hipLaunchKernelGGL((mark_kernel<T>), dim3((unsigned)cdiv(cnt, 256)), dim3(256), 0, s, cnt, xch);
    const TriResP<T> q{A, lda, (int)n, tau, xch, h->spin_limit};
    hipLaunchKernelGGL((tri_resident_kernel<T>), dim3((unsigned)P), dim3((unsigned)cdiv(2 * P, 64) * 64),
                       0, s, q);
    const int rc = resident_end(h, s);
    GLA_LAUNCH_CHECK();
    return rc;
}

// A[i, j] <-> A[n−1−i, n−1−j] over the whole matrix (J A J in place).
template <typename T>
__global__ void reverse_kernel(int64_t n, T *A, int64_t lda)
{
    const int64_t i = (int64_t)blockIdx.x * 16 + threadIdx.x;
    const int64_t j = (int64_t)blockIdx.y * 16 + threadIdx.y;
    if (i >= n || j >= n) return;
    const int64_t i2 = n - 1 - i, j2 = n - 1 - j;
    // each pair once: the element with the smaller column-major index swaps
    if (i + j * n < i2 + j2 * n) {
        const T a = A[i + j * lda];
        A[i + j * lda] = A[i2 + j2 * lda];
        A[i2 + j2 * lda] = a;
    }
}

template <typename T>
__global__ void zero_kernel(int64_t cnt, T *p)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < cnt) p[i] = T(0);
}


// ------------------------------------------------------ bidiagonalize! ----
// Tall case (m ≥ n), panel [k, k+w), column i = k + j.  The trailing block
// Ã keeps its panel-start values wherever a GEMV reads it (the column and
// row brought up to date lie outside those regions); V, X (m rows) and
// Y, U (n rows) hold the panel's left vectors, A u products, Aᵀ v products
// and right vectors: A_now = Ã − V Yᵀ − X Uᵀ.
enum { B_LTAU = 0, B_LXI = 1, B_LBETA = 2, B_RTAU = 3, B_RXI = 4, B_RBETA = 5 };

// ‖A[i:m, i]‖² partials (the panel's first column, nothing to apply).
template <typename T>
__global__ void bd_col0_kernel(int64_t m, int64_t i, const T *A, int64_t lda, T *npart)
{
    __shared__ T sh[8];
    const int64_t r = i + (int64_t)blockIdx.x * 256 + threadIdx.x;
    T a = r < m ? A[r + i * lda] : T(0);
    T sq = wave_sum(a * a);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = sq;
    __syncthreads();
    if (threadIdx.x == 0) npart[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
}

// Left reflector scalars of column i, then P[rb·C + c'] = Σ over the 64-row
// block rb of Ã[r, i+1+c'] v_r (Ãᵀ v), and on cb = 0 blocks the partials
// Cv1[rb·kPanel + l] = Σ V[r,l] v_r, Cv2 = Σ X[r,l] v_r (l < j).
template <typename T>
__global__ __launch_bounds__(256) void bd_gemvt_kernel(int64_t m, int64_t n, int64_t i, int j,
                                                       const T *A, int64_t lda, const T *V,
                                                       const T *X, int64_t ldm,
                                                       const T *npart, int ncnt, int64_t ncb,
                                                       T *P, T *Cv1, T *Cv2, T *scal, T *taul)
{
    __shared__ T sh[8];
    const T nrm2 = block_sum_fixed(npart, ncnt, sh);
    T xi, tau, beta;
    reflector_scalars(nrm2, A[i + i * lda], xi, tau, beta);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        scal[B_LTAU] = tau;
        scal[B_LXI] = xi;
        scal[B_LBETA] = beta;
        taul[i] = tau;
    }
    const int64_t C = n - i - 1;
    if (C <= 0) return;
    const int64_t rb = blockIdx.x / ncb, cb = blockIdx.x % ncb;
    const int t = threadIdx.x, a = t & 15, b = t >> 4, lane = t & 63, wv = t >> 6;
    // rows RB + 16u (whole cache lines per load instruction), columns
    // C0 + cc; unconditional loads from clamped indices
    const int64_t RB = i + rb * kTB + a, C0 = i + 1 + cb * kTB + 4 * b;
    T vr[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int64_t r = RB + 16 * u;
        vr[u] = r < m ? (r == i ? T(1) : A[r + i * lda] / xi) : T(0);
    }
    T x[4][4];
#pragma unroll
    for (int cc = 0; cc < 4; ++cc)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
            const int64_t gr = RB + 16 * rr, gc = C0 + cc;
            const int64_t grc = gr < m ? gr : m - 1, gcc = gc < n ? gc : n - 1;
            const T v = A[grc + gcc * lda];
            x[cc][rr] = (gr < m && gc < n) ? v : T(0);
        }
    T qc[4];
#pragma unroll
    for (int cc = 0; cc < 4; ++cc) {
        T acc = T(0);
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) acc += x[cc][rr] * vr[rr];
        qc[cc] = acc;
    }
#pragma unroll
    for (int cc = 0; cc < 4; ++cc) qc[cc] = row_sum16(qc[cc]);
    if (a == 0)
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {
            const int64_t c = cb * kTB + 4 * b + cc;
            if (c < C) P[rb * C + c] = qc[cc];
        }
    if (cb == 0) {
        const int64_t gr = i + rb * kTB + lane;
        const int64_t grc = gr < m ? gr : m - 1;
        const T vg = gr < m ? (gr == i ? T(1) : A[gr + i * lda] / xi) : T(0);
        T a1[kPanel / 4], a2[kPanel / 4];
#pragma unroll
        for (int u = 0; u < kPanel / 4; ++u) {
            const int l = wv + 4 * u, lc = l < j ? l : 0;
            a1[u] = V[grc + (int64_t)lc * ldm];
            a2[u] = X[grc + (int64_t)lc * ldm];
        }
#pragma unroll
        for (int u = 0; u < kPanel / 4; ++u) {
            const int l = wv + 4 * u;
            if (l < j) {
                const T c1 = wave_sum(a1[u] * vg);
                const T c2 = wave_sum(a2[u] * vg);
                if (lane == 0) {
                    Cv1[rb * kPanel + l] = c1;
                    Cv2[rb * kPanel + l] = c2;
                }
            }
        }
    }
}

// Sum of the per-block partials part[b·kPanel + l] over b < nb for l < lmax,
// by the whole workgroup in a fixed order (eight interleaved parts, then
// the parts in order); the result in out[l] (zero for l ≥ lmax).
template <typename T>
__device__ __forceinline__ void panel_partials(const T *part, int64_t nb, int lmax, T *out,
                                               T (*cs)[kPanel])
{
    const int t = threadIdx.x, l = t & (kPanel - 1), pp = t / kPanel;
    T s = T(0);
    if (l < lmax)
        for (int64_t b = pp; b < nb; b += 8) s += part[b * kPanel + l];
    cs[pp][l] = s;
    __syncthreads();
    if (t < kPanel) {
        T r = T(0);
#pragma unroll
        for (int q = 0; q < 8; ++q) r += cs[q][t];
        out[t] = r;
    }
}

// Item it of the workgroup (64 items, four lanes each) covers column
// c = i+1+it (y_c = τ (Ãᵀv − Y c1 − U c2)_c, row i brought up to date,
// partial ‖row‖²; lane k takes the row-block partials rb ≡ k and the
// reflectors l ≡ k (mod 4), summed over the quad) and row r = i+it (v into
// A and V).
template <typename T>
__global__ __launch_bounds__(256) void bd_y_kernel(int64_t m, int64_t n, int64_t i, int j, T *A,
                                                   int64_t lda, T *V, const T *X, int64_t ldm,
                                                   T *Y, const T *U, int64_t ldn, const T *P,
                                                   int64_t nrb, const T *Cv1, const T *Cv2,
                                                   const T *scal, T *npart2)
{
    __shared__ T sh[8];
    __shared__ T c1[kPanel], c2[kPanel], vi[kPanel], xi_[kPanel];
    __shared__ T cs[8][kPanel];
    const int t = threadIdx.x, k = t & 3;
    const T tau = scal[B_LTAU], xi = scal[B_LXI], beta = scal[B_LBETA];
    if (t < kPanel) {
        vi[t] = t < j ? V[i + (int64_t)t * ldm] : T(0);
        xi_[t] = t < j ? X[i + (int64_t)t * ldm] : T(0);
    }
    panel_partials(Cv1, nrb, j, c1, cs);
    __syncthreads();
    panel_partials(Cv2, nrb, j, c2, cs);
    __syncthreads();
    const int64_t it = (int64_t)blockIdx.x * kRPB + (t >> 2);
    const int64_t C = n - i - 1;
    T sq = T(0);
    if (C > 0) {
        const bool in = it < C;
        const int64_t tc = in ? it : C - 1, c = i + 1 + tc;
        T p0 = T(0), p1 = T(0);
        int64_t rb = k;
        for (; rb + 4 < nrb; rb += 8) {
            p0 += P[rb * C + tc];
            p1 += P[(rb + 4) * C + tc];
        }
        if (rb < nrb) p0 += P[rb * C + tc];
        T p = p0 + p1, rp = T(0);
        if (j > 0) {
            T yv[kPanel / 4], uv[kPanel / 4];
#pragma unroll
            for (int u = 0; u < kPanel / 4; ++u) {
                const int l = k + 4 * u, lc = l < j ? l : 0;
                yv[u] = Y[c + (int64_t)lc * ldn];
                uv[u] = U[c + (int64_t)lc * ldn];
            }
#pragma unroll
            for (int u = 0; u < kPanel / 4; ++u) {
                const int l = k + 4 * u;
                if (l < j) {
                    p -= yv[u] * c1[l] + uv[u] * c2[l];
                    rp += vi[l] * yv[u] + xi_[l] * uv[u];
                }
            }
        }
        p = quad_sum(p);
        rp = quad_sum(rp);
        if (in && k == 0) {
            const T y = tau * p;
            Y[c + (int64_t)j * ldn] = y;
            const T r = A[i + c * lda] - y - rp;
            A[i + c * lda] = r;
            sq = r * r;
        }
    }
    const int64_t r = i + it;
    if (k == 0 && r < m) {
        const T v = r == i ? T(1) : A[r + i * lda] / xi;
        V[r + (int64_t)j * ldm] = v;
        A[r + i * lda] = r == i ? beta : v;
    }
    sq = wave_sum(sq);
    if ((t & 63) == 0) sh[t >> 6] = sq;
    __syncthreads();
    if (t == 0) npart2[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// Right reflector scalars of row i, then P[cb·R + r'] = Σ over the 64-column
// block cb of Ã[i+1+r', c] u_c (Ã u), and on rb = 0 blocks
// Cu1[cb·kPanel + l] = Σ Y[c,l] u_c (l ≤ j), Cu2 = Σ U[c,l] u_c (l < j).
template <typename T>
__global__ __launch_bounds__(256) void bd_gemvn_kernel(int64_t m, int64_t n, int64_t i, int j,
                                                       const T *A, int64_t lda, const T *Y,
                                                       const T *U, int64_t ldn,
                                                       const T *npart2, int ncnt, int64_t ncb,
                                                       T *P, T *Cu1, T *Cu2, T *scal, T *taur)
{
    __shared__ T sh[8];
    __shared__ T srow[4][kTB];
    const T nrm2 = block_sum_fixed(npart2, ncnt, sh);
    T xi, tau, beta;
    reflector_scalars(nrm2, A[i + (i + 1) * lda], xi, tau, beta);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        scal[B_RTAU] = tau;
        scal[B_RXI] = xi;
        scal[B_RBETA] = beta;
        taur[i] = tau;
    }
    const int64_t R = m - i - 1;
    const int64_t rb = blockIdx.x / ncb, cb = blockIdx.x % ncb;
    const int t = threadIdx.x, a = t & 15, b = t >> 4, lane = t & 63, wv = t >> 6;
    // rows RB + 16u (whole cache lines per load instruction), columns
    // C0 + cc; unconditional loads from clamped indices
    const int64_t RB = i + 1 + rb * kTB + a, C0 = i + 1 + cb * kTB + 4 * b;
    T uc[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int64_t c = C0 + u;
        uc[u] = c < n ? (c == i + 1 ? T(1) : A[i + c * lda] / xi) : T(0);
    }
    T x[4][4];
#pragma unroll
    for (int cc = 0; cc < 4; ++cc)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
            const int64_t gr = RB + 16 * rr, gc = C0 + cc;
            const int64_t grc = gr < m ? gr : m - 1, gcc = gc < n ? gc : n - 1;
            const T v = A[grc + gcc * lda];
            x[cc][rr] = (gr < m && gc < n) ? v : T(0);
        }
    T s[4];
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
        T acc = T(0);
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) acc += x[cc][rr] * uc[cc];
        s[rr] = acc;
    }
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
        s[rr] += __shfl_xor(s[rr], 16);
        s[rr] += __shfl_xor(s[rr], 32);
    }
    if (lane < 16)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) srow[wv][a + 16 * rr] = s[rr];
    __syncthreads();
    if (t < kTB) {
        const int64_t r = rb * kTB + t;
        if (r < R) P[cb * R + r] = srow[0][t] + srow[1][t] + srow[2][t] + srow[3][t];
    }
    if (rb == 0) {
        const int64_t gc = i + 1 + cb * kTB + lane;
        const int64_t gcc = gc < n ? gc : n - 1;
        const T ug = gc < n ? (gc == i + 1 ? T(1) : A[i + gc * lda] / xi) : T(0);
        T a1[kPanel / 4], a2[kPanel / 4];
#pragma unroll
        for (int u = 0; u < kPanel / 4; ++u) {
            const int l = wv + 4 * u, l1 = l <= j ? l : 0, l2 = l < j ? l : 0;
            a1[u] = Y[gcc + (int64_t)l1 * ldn];
            a2[u] = U[gcc + (int64_t)l2 * ldn];
        }
#pragma unroll
        for (int u = 0; u < kPanel / 4; ++u) {
            const int l = wv + 4 * u;
            if (l <= j) {
                const T c1 = wave_sum(a1[u] * ug);
                const T c2 = wave_sum(l < j ? a2[u] * ug : T(0));
                if (lane == 0) {
                    Cu1[cb * kPanel + l] = c1;
                    Cu2[cb * kPanel + l] = c2;
                }
            }
        }
    }
}

// Item it (64 per workgroup, four lanes each) covers row r = i+1+it
// (x_r = τ (Ã u − V c3 − X c4)_r; then, unless `last`, column i+1 brought
// up to date with reflectors 0..j and its partial ‖·‖²; lane k takes the
// column-block partials cb ≡ k and the reflectors l ≡ k (mod 4), summed over
// the quad) and column c = i+1+it (u into A and U).
template <typename T>
__global__ __launch_bounds__(256) void bd_x_kernel(int64_t m, int64_t n, int64_t i, int j,
                                                   int last, T *A, int64_t lda, const T *V, T *X,
                                                   int64_t ldm, const T *Y, T *U, int64_t ldn,
                                                   const T *P, int64_t ncb, const T *Cu1,
                                                   const T *Cu2, const T *scal, T *npart)
{
    __shared__ T sh[8];
    __shared__ T c3[kPanel], c4[kPanel], yn[kPanel], un[kPanel];
    __shared__ T cs[8][kPanel];
    const int t = threadIdx.x, k = t & 3;
    const T tau = scal[B_RTAU], xi = scal[B_RXI], beta = scal[B_RBETA];
    const int64_t i1 = i + 1;
    if (t < kPanel) {
        yn[t] = t <= j ? Y[i1 + (int64_t)t * ldn] : T(0);
        un[t] = t <= j ? (t == j ? T(1) : U[i1 + (int64_t)t * ldn]) : T(0);
    }
    panel_partials(Cu1, ncb, j + 1, c3, cs);
    __syncthreads();
    panel_partials(Cu2, ncb, j, c4, cs);
    __syncthreads();
    const int64_t it = (int64_t)blockIdx.x * kRPB + (t >> 2);
    const int64_t R = m - i - 1;
    T sq = T(0);
    if (R > 0) {
        const bool in = it < R;
        const int64_t tr = in ? it : R - 1, r = i1 + tr;
        T q0 = T(0), q1 = T(0);
        int64_t cb = k;
        for (; cb + 4 < ncb; cb += 8) {
            q0 += P[cb * R + tr];
            q1 += P[(cb + 4) * R + tr];
        }
        if (cb < ncb) q0 += P[cb * R + tr];
        T q = q0 + q1, ap = T(0);
        T vv[kPanel / 4], xv[kPanel / 4];
#pragma unroll
        for (int u = 0; u < kPanel / 4; ++u) {
            const int l = k + 4 * u, lv = l <= j ? l : 0, lx = l < j ? l : 0;
            vv[u] = V[r + (int64_t)lv * ldm];
            xv[u] = X[r + (int64_t)lx * ldm];
        }
#pragma unroll
        for (int u = 0; u < kPanel / 4; ++u) {
            const int l = k + 4 * u;
            if (l <= j) q -= vv[u] * c3[l];
            if (l < j) {
                q -= xv[u] * c4[l];
                ap += vv[u] * yn[l] + xv[u] * un[l];
            }
        }
        q = quad_sum(q);
        ap = quad_sum(ap);
        if (in && k == 0) {
            const T x = tau * q;
            X[r + (int64_t)j * ldm] = x;
            if (!last && i1 < n) {
                // the l = j term: V[r][j] y_n[j] + x u_n[j]
                const T a = A[r + i1 * lda] - ap - (V[r + (int64_t)j * ldm] * yn[j] + x * un[j]);
                A[r + i1 * lda] = a;
                sq = a * a;
            }
        }
    }
    const int64_t c = i1 + it;
    if (k == 0 && c < n) {
        const T u = c == i1 ? T(1) : A[i + c * lda] / xi;
        U[c + (int64_t)j * ldn] = u;
        A[i + c * lda] = c == i1 ? beta : u;
    }
    sq = wave_sum(sq);
    if ((t & 63) == 0) sh[t >> 6] = sq;
    __syncthreads();
    if (t == 0) npart[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// ---- bidiagonalize! with the matrix in registers ----
// One launch for a tall matrix that fits 128×128 elements per workgroup on
// ⌈m/128⌉ × ⌈n/128⌉ ≤ 256 of them.  Workgroup (gr, gc) of the PR × PC grid
// holds rows ≡ gr (mod PR) and columns ≡ gc (mod PC): thread (row group rg,
// column group cg) rows 4 rg + k, columns 8 cg + q of the block.  It also
// keeps, for its own rows or columns, the column x to be reflected and the
// vectors v, w and y, z, u.  Column i (src/svd.jl:333-345), A as it stands:
//   L  publish d = Σ_{r>i} x_r A[r, ·] over the own rows, Σ x_r², row i and
//      x_i;  gather over the grid column;  ‖x‖, ξ, τ;  y = A[i, ·] + d/ξ
//      (= Aᵀv), z = A[i, ·] − τ y;  A −= τ v yᵀ;
//   R  publish e = Σ_{c>i+1} z_c A[·, c] over the own columns, Σ z_c², column
//      i + 1 and z_{i+1};  gather over the grid row;  w = A[·, i+1] + e/ξ
//      (= A u);  the next column x = A[·, i+1] − τ w;  A −= τ w uᵀ.
// Two exchanges per column; the sums travel before the norm is known, since
// they are formed with the unscaled vector.  Arrival marks as in the
// tridiagonal kernel; the partial sums go through a ring of three slots,
// marked again by their owner one step after they were gathered: a
// workgroup that gathers step i + 1 knows that its peers are done with step
// i, and its publication of step i + 2, after which the slot's next use can
// begin, follows the new mark.  All workgroups must be resident, as there.
// The grid is two-dimensional since a workgroup then exchanges with a row or
// a column of it (20 of 240 for 2500×1501) and not with all.
// Bound: latency, two exchanges and six barriers a column.  2500×1501 FP64
// 10.2 ms, 6.8 µs a column; the four launches per column of the deferred form
// took 50.0 ms.  The same kernel with some of the block spilled to memory
// took 24.4 ms: no wide stores of the block, no exit inside the loop, places
// worked out anew per column.
// Line: wherever the block fits.  Deferred form -> this, FP64 ms: 2×2
// 0.072 -> 0.063, 64×64 1.28 -> 0.36, 8192×20 0.67 -> 0.18, 8192×512
// 22.2 -> 4.3, 2048² 65.9 -> 14.9, 3000×2000 (panels first) 72.7 -> 32.3;
// FP32 64×64 1.15 -> 0.28, 2048² 57.0 -> 14.7.
// Accuracy: over 84 matrices of 17×17…140×64 the error against a __float128
// evaluation is 0.69 of the FP64 oracle's (1.03 the deferred form), in FP32
// 0.70 of the FP32 oracle's (0.84).
constexpr int kBRLoc = 128;                 // rows and columns per workgroup
constexpr int kBRBlk = 136;                 // an exchanged vector with its scalar
constexpr int kBRMaxPR = 64;

template <typename T>
struct BdResP {
    T *A;
    int64_t lda;
    int m, n, PR, PC;
    T *taul, *taur;
    T *e1, *e2;          // [3][P][kBRBlk], grid column and grid row major; e1 starts the
                         // workspace, which ends below 4 GiB
    T *rowb, *colb;      // [n][PC][kBRBlk], [n][PR][kBRBlk]
    unsigned spin_limit;
};

template <typename T>
__global__ __launch_bounds__(512, 4) void bd_resident_kernel(BdResP<T> q)
{
    typedef typename NaNMark<T>::bits B;
    __shared__ T red[8][kBRLoc], gsum[4][kBRLoc];
    __shared__ T X[kBRLoc], V[kBRLoc], Wv[kBRLoc], Y[kBRLoc], Z[kBRLoc], Uv[kBRLoc];
    __shared__ T sp[2], ss[2], xpiv, piv;
    const int PR = q.PR, PC = q.PC, m = q.m, n = q.n;
    const int gr = blockIdx.x % PR, gc = blockIdx.x / PR;
    const int64_t lda = q.lda, slot = (int64_t)PR * PC * kBRBlk;

    auto mark = [](T *p) {
        store_coherent(reinterpret_cast<B *>(p), NaNMark<T>::value);
    };
    auto publish = [](T *p, T v) {
        store_coherent(reinterpret_cast<B *>(p), __builtin_bit_cast(B, v));
    };

    T a[4][8];
    {
        const int t = threadIdx.x, lane = t & 63, cg = lane & 15, rg = 4 * (t >> 6) + (lane >> 4);
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const int r = gr + PR * (4 * rg + k), cc = gc + PC * (8 * cg + c);
                const bool in = r < m && cc < n;
                const T v = q.A[in ? r + (int64_t)cc * lda : 0];
                a[k][c] = in ? quiet(v) : T(0);
            }
        if (t < kBRLoc) {
            const int r = gr + PR * t;
            const T v = quiet(q.A[r < m ? r : 0]);      // x_0 is published as it is
            const T x = r < m && r > 0 ? v : T(0);
            X[t] = x;
            if (r == 0) xpiv = v;
            const T sq = wave_sum(x * x);
            if (lane == 0) ss[t >> 6] = sq;
        }
    }
    bool lost = false;

    // Sum over the cnt partial vectors at base + e·kBRBlk (element tl, those
    // ≡ h mod 4) into gsum, and with them the scalar parts: quarter 0 returns
    // `line`'s element, quarter 1 sums the partials' scalars into sp, one
    // thread of quarter 2 takes line's scalar into piv.
    auto gather = [&](const T *base, int cnt, const T *line, int t) -> T {
        const int tl = t & (kBRLoc - 1), h = t >> 7, lane = t & 63, wv = t >> 6;
        T s = T(0), extra = T(0);
        // places in the workspace, in elements
        const unsigned b0 = (unsigned)(base - q.e1), l0 = (unsigned)(line - q.e1);
        unsigned xo = b0;
        if (h == 0) xo = l0 + tl;
        else if (h == 1 && tl < cnt) xo = b0 + tl * kBRBlk + kBRLoc;
        else if (h == 2) xo = l0 + kBRLoc;
        for (int e0 = h; e0 == h || e0 < cnt; e0 += 28) {
            unsigned off[8];
            T v[8];
#pragma unroll
            for (int u = 0; u < 7; ++u) {
                const int e = e0 + 4 * u;
                off[u] = (b0 + (e < cnt ? e : 0) * kBRBlk + tl) * (unsigned)sizeof(T);
            }
            off[7] = xo * (unsigned)sizeof(T);
            for (unsigned spins = 0;; ++spins) {
                load8_coherent(q.e1, off, v);
                bool ok = true;
#pragma unroll
                for (int u = 0; u < 8; ++u) ok = ok && !is_mark(v[u]);
                if (__all(ok) || lost) break;
                if (spins >= q.spin_limit) lost = true;
            }
#pragma unroll
            for (int u = 0; u < 7; ++u)
                if (e0 + 4 * u < cnt) s += v[u];
            extra = v[7];
        }
        gsum[h][tl] = s;
        if (h == 1) {
            const T sc = wave_sum(tl < cnt ? extra : T(0));
            if (lane == 0) sp[wv - 2] = sc;
        }
        if (t == 2 * kBRLoc) piv = extra;
        return extra;
    };

    lds_barrier();
    for (int i = 0; i < n; ++i) {
        // the thread's places are worked out anew for every column: kept over
        // the loop, they and what follows from them push the block out of the
        // registers
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));
        const int lane = t & 63, wv = t >> 6, cg = lane & 15, rg = 4 * wv + (lane >> 4);
        const int tl = t & (kBRLoc - 1);                  // element of an exchanged vector
        T *e1 = q.e1 + (i % 3) * slot + ((int64_t)gc * PR) * kBRBlk;   // this grid column
        T *e2 = q.e2 + (i % 3) * slot + ((int64_t)gr * PC) * kBRBlk;   // this grid row
        T *rowi = q.rowb + ((int64_t)i * PC + gc) * kBRBlk;
        T *coli = q.colb + ((int64_t)i * PR + gr) * kBRBlk;
        const int li = i / PR, lc1 = (i + 1) / PC;
        const bool has_row = i % PR == gr, has_col = i + 1 < n && (i + 1) % PC == gc;
        // ---- L: row i, d
        if (has_row) {
            if (rg == li >> 2) {
                // (one value per store: wider ones would tie the block's
                // registers together)
                auto put = [&](const T (&r)[8]) {
#pragma unroll
                    for (int c = 0; c < 8; ++c) publish(rowi + 8 * cg + c, r[c]);
                };
                switch (li & 3) {
                case 0: put(a[0]); break;
                case 1: put(a[1]); break;
                case 2: put(a[2]); break;
                default: put(a[3]); break;
                }
            }
            if (t == 0) publish(rowi + kBRLoc, xpiv);
        }
        {
            T d[8];
            const T x0 = X[4 * rg], x1 = X[4 * rg + 1], x2 = X[4 * rg + 2], x3 = X[4 * rg + 3];
#pragma unroll
            for (int c = 0; c < 8; ++c)
                d[c] = fma_t(x3, a[3][c], fma_t(x2, a[2][c], fma_t(x1, a[1][c], x0 * a[0][c])));
            // over the wave's four row groups: lanes keep columns
            // 4·bit5 + 2·bit4 and the next of their eight
            T u[4], w[2];
#pragma unroll
            for (int k = 0; k < 4; ++k) u[k] = pair_sum32<T>(d[k], d[k + 4]);
#pragma unroll
            for (int k = 0; k < 2; ++k) w[k] = pair_sum16<T>(u[k], u[k + 2]);
            const int c = 8 * cg + 4 * (lane >> 5) + 2 * ((lane >> 4) & 1);
            red[wv][c] = w[0];
            red[wv][c + 1] = w[1];
        }
        lds_barrier();
        if (t < kBRLoc) {
            T s = T(0);
#pragma unroll
            for (int w = 0; w < 8; ++w) s += red[w][t];
            publish(e1 + gr * kBRBlk + t, s);
            if (t == 0) publish(e1 + gr * kBRBlk + kBRLoc, ss[0] + ss[1]);
        }
        T line = gather(e1, PR, rowi, t);
        lds_barrier();
        // the left reflector
        const T xi_ = piv;
        const T nrm = sqrt(fma_t(xi_, xi_, sp[0] + sp[1]));
        const bool live = nrm != T(0);
        const T nu = copysign(nrm, xi_), xi = xi_ + nu;
        const T tau = live ? xi / nu : T(0), rxi = live ? T(1) / xi : T(1);
        if (t < kBRLoc) {
            const int c = gc + PC * t;
            const T d = (gsum[0][t] + gsum[1][t]) + (gsum[2][t] + gsum[3][t]);
            const bool in = c > i && c < n;
            const T y = in ? fma_t(d, rxi, line) : T(0);
            const T z = in ? fma_t(-tau, y, line) : T(0);
            Y[t] = y;
            Z[t] = c > i + 1 ? z : T(0);
            if (c == i + 1) xpiv = z;                     // z's first element
            const T sq = wave_sum(c > i + 1 ? z * z : T(0));
            if (lane == 0) ss[wv] = sq;
        } else if (t < 2 * kBRLoc) {
            const int r = gr + PR * tl;
            V[tl] = r > i ? X[tl] * rxi : (r == i ? T(1) : T(0));
        }
        // the grid column's peers are done with the previous step's sums (by
        // waves with nothing else to do here)
        if (i > 0 && t >= 2 * kBRLoc && t < 3 * kBRLoc) {
            T *old = q.e1 + ((i + 2) % 3) * slot + ((int64_t)gc * PR + gr) * kBRBlk;
            mark(old + tl);
            if (tl == 0) mark(old + kBRLoc);
        }
        if (blockIdx.x == 0 && t == 0) q.taul[i] = tau;
        const T beta_l = live ? -nu : xi_;
        lds_barrier();
        if (i + 1 < n) {     // the last column has no right reflector (src/svd.jl:339)
            // A −= τ v yᵀ, then e
            {
                T tv[4], e[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    tv[k] = -tau * V[4 * rg + k];
                    e[k] = T(0);
                }
                // two columns at a time: the block leaves no more registers
#pragma unroll
                for (int c = 0; c < 8; c += 2) {
                    const T y0 = Y[8 * cg + c], y1 = Y[8 * cg + c + 1];
                    const T z0 = Z[8 * cg + c], z1 = Z[8 * cg + c + 1];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        a[k][c] = fma_t(tv[k], y0, a[k][c]);
                        a[k][c + 1] = fma_t(tv[k], y1, a[k][c + 1]);
                        e[k] = fma_t(z1, a[k][c + 1], fma_t(z0, a[k][c], e[k]));
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                // over the row's 16 lanes: lane keeps row 2·bit3 + bit2 of its four
                const bool b3 = lane & 8, b2 = lane & 4;
                T w0 = (b3 ? e[2] : e[0]) + dppmov<0x128>(b3 ? e[0] : e[2]);   // row_ror:8
                T w1 = (b3 ? e[3] : e[1]) + dppmov<0x128>(b3 ? e[1] : e[3]);
                T s = (b2 ? w1 : w0) + dppmov<0x141>(b2 ? w0 : w1);            // half mirror
                s += dppmov<0xB1>(s);
                s += dppmov<0x4E>(s);
                if ((lane & 3) == 0)
                    publish(e2 + gc * kBRBlk + 4 * rg + 2 * ((lane >> 3) & 1) + ((lane >> 2) & 1), s);
            }
            if (has_col && cg == lc1 >> 3) {
                auto put = [&](T r0, T r1, T r2, T r3) {
                    publish(coli + 4 * rg, r0);
                    publish(coli + 4 * rg + 1, r1);
                    publish(coli + 4 * rg + 2, r2);
                    publish(coli + 4 * rg + 3, r3);
                };
                switch (lc1 & 7) {
                case 0: put(a[0][0], a[1][0], a[2][0], a[3][0]); break;
                case 1: put(a[0][1], a[1][1], a[2][1], a[3][1]); break;
                case 2: put(a[0][2], a[1][2], a[2][2], a[3][2]); break;
                case 3: put(a[0][3], a[1][3], a[2][3], a[3][3]); break;
                case 4: put(a[0][4], a[1][4], a[2][4], a[3][4]); break;
                case 5: put(a[0][5], a[1][5], a[2][5], a[3][5]); break;
                case 6: put(a[0][6], a[1][6], a[2][6], a[3][6]); break;
                default: put(a[0][7], a[1][7], a[2][7], a[3][7]); break;
                }
            }
            if (t == 0) {
                publish(e2 + gc * kBRBlk + kBRLoc, ss[0] + ss[1]);
                if (has_col) publish(coli + kBRLoc, xpiv);
            }
            // ---- R
            line = gather(e2, PC, coli, t);
            lds_barrier();
            const T zi = piv;
            const T nrmr = sqrt(fma_t(zi, zi, sp[0] + sp[1]));
            const bool liver = nrmr != T(0);
            const T nur = copysign(nrmr, zi), xir = zi + nur;
            const T taur = liver ? xir / nur : T(0), rxir = liver ? T(1) / xir : T(1);
            if (t < kBRLoc) {
                const int r = gr + PR * t;
                const T e = (gsum[0][t] + gsum[1][t]) + (gsum[2][t] + gsum[3][t]);
                const bool in = r > i && r < m;
                const T w = in ? fma_t(e, rxir, line) : T(0);
                const T x = in ? fma_t(-taur, w, line) : T(0);
                Wv[t] = w;
                X[t] = r > i + 1 ? x : T(0);
                if (r == i + 1) xpiv = x;
                const T sq = wave_sum(r > i + 1 ? x * x : T(0));
                if (lane == 0) ss[wv] = sq;
            } else if (t < 2 * kBRLoc) {
                const int c = gc + PC * tl;
                Uv[tl] = c > i + 1 ? Z[tl] * rxir : (c == i + 1 ? T(1) : T(0));
            }
            if (i > 0 && t >= 2 * kBRLoc && t < 3 * kBRLoc) {
                T *old = q.e2 + ((i + 2) % 3) * slot + ((int64_t)gr * PC + gc) * kBRBlk;
                mark(old + tl);
                if (tl == 0) mark(old + kBRLoc);
            }
            if (blockIdx.x == 0 && t == 0) q.taur[i] = taur;
            lds_barrier();
            {
                T tw[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) tw[k] = -taur * Wv[4 * rg + k];
#pragma unroll
                for (int c = 0; c < 8; c += 2) {
                    const T u0 = Uv[8 * cg + c], u1 = Uv[8 * cg + c + 1];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        a[k][c] = fma_t(tw[k], u0, a[k][c]);
                        a[k][c + 1] = fma_t(tw[k], u1, a[k][c + 1]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            // row i of the result, by its holders
            if (has_row && t >= kBRLoc && t < 2 * kBRLoc) {
                const int c = gc + PC * tl;
                if (c > i && c < n)
                    q.A[i + (int64_t)c * lda] = c == i + 1 ? (liver ? -nur : zi) : Uv[tl];
            }
        }
        // column i of the result, by its holders.  Only now: the grid row's
        // peers have published e, so they have read x
        if (i % PC == gc && t < kBRLoc) {
            const int r = gr + PR * t;
            if (r >= i && r < m) q.A[r + (int64_t)i * lda] = r == i ? beta_l : V[t];
        }
    }
}

// Shapes the resident kernel takes (m ≥ n), and its workspace in elements.
inline bool bd_resident_fits(int64_t m, int64_t n, int num_cus)
{
    const int64_t PR = cdiv(m, kBRLoc), PC = cdiv(n, kBRLoc);
    return n >= 2 && m >= n && PR <= kBRMaxPR && PR * PC <= std::min(256, num_cus);
}
inline size_t bd_resident_elems(int64_t m, int64_t n)
{
    const int64_t PR = cdiv(m, kBRLoc), PC = cdiv(n, kBRLoc);
    return (size_t)(6 * PR * PC + n * (PR + PC)) * kBRBlk;
}

template <typename T>
int bd_resident(Handle *h, hipStream_t s, int64_t m, int64_t n, T *A, int64_t lda, T *taul, T *taur,
                T *ws, bool *done)
{
    *done = resident_begin(h, s, cdiv(m, kBRLoc) * cdiv(n, kBRLoc));
    if (!*done) return GLA_OK;
    BdResP<T> q;
    q.A = A;
    q.lda = lda;
    q.m = (int)m;
    q.n = (int)n;
    q.PR = (int)cdiv(m, kBRLoc);
    q.PC = (int)cdiv(n, kBRLoc);
    q.taul = taul;
    q.taur = taur;
    const size_t ring = 3 * (size_t)q.PR * q.PC * kBRBlk;
    q.e1 = ws;
    q.e2 = q.e1 + ring;
    q.rowb = q.e2 + ring;
    q.colb = q.rowb + (size_t)n * q.PC * kBRBlk;
    q.spin_limit = h->spin_limit;
    const int64_t cnt = (int64_t)bd_resident_elems(m, n);
    hipLaunchKernelGGL((mark_kernel<T>), dim3((unsigned)cdiv(cnt, 256)), dim3(256), 0, s, cnt, ws);
    hipLaunchKernelGGL((bd_resident_kernel<T>), dim3((unsigned)(q.PR * q.PC)), dim3(512), 0, s, q);
    const int rc = resident_end(h, s);
    GLA_LAUNCH_CHECK();
    return rc;
}

// B (n×m, ld ldb) = Aᵀ for A m×n.
template <typename T>
__global__ void transpose_kernel(int64_t m, int64_t n, const T *A, int64_t lda, T *B, int64_t ldb)
{
    __shared__ T tile[16][17];
    const int64_t r0 = (int64_t)blockIdx.x * 16, c0 = (int64_t)blockIdx.y * 16;
    const int tx = threadIdx.x, ty = threadIdx.y;
    if (r0 + tx < m && c0 + ty < n) tile[ty][tx] = A[(r0 + tx) + (c0 + ty) * lda];
    __syncthreads();
    if (c0 + tx < n && r0 + ty < m) B[(c0 + tx) + (r0 + ty) * ldb] = tile[tx][ty];
}

}  // namespace

// Workspace elements of symtri for order n.
// (resident: with the resident kernel's exchange, which a captured call never uses)
size_t symtri_scratch(int64_t n, bool resident)
{
    const int64_t ldv = (n + 3) / 4 * 4;
    const int64_t nbk = cdiv(n, kTB);
    const int64_t g = cdiv(n, kRPB);
    const int64_t nr = resident ? std::min<int64_t>(n, kTRMax) : 0;
    return 2 * (size_t)ldv * kPanel +
           std::max((size_t)nbk * n + 2 * (size_t)nbk * kPanel + 2 * g, 2 * (size_t)nr * (nr + 8)) + 64;
}

// symtriLower! on the lower triangle of A (n×n); τ (n − 1 entries, device):
// panels of deferred updates until the trailing block fits the resident
// kernel, which takes the rest.
template <typename T>
int symtri_lower_dev(Handle *h, hipStream_t s, int64_t n, T *A, int64_t lda, T *tau, T *ws)
{
    if (n < 1) return GLA_OK;
    if (n > 1) {
        hipLaunchKernelGGL((zero_kernel<T>), dim3((unsigned)cdiv(n - 1, 256)), dim3(256), 0, s,
                           n - 1, tau);
        GLA_LAUNCH_CHECK();
    }
    if (n <= 2) return GLA_OK;
    const int64_t ldv = (n + 3) / 4 * 4;
    const int64_t nbk_max = cdiv(n, kTB);
    const int64_t gmax = cdiv(n, kRPB);
    // (P starts on 16 bytes: ldv is a multiple of 4)
    T *V = ws, *W = V + ldv * kPanel, *P = W + ldv * kPanel, *Y1 = P + nbk_max * n,
      *Y2 = Y1 + nbk_max * kPanel, *npart = Y2 + nbk_max * kPanel, *qpart = npart + gmax,
      *scal = qpart + gmax;
    const int64_t ncols = n - 2;   // columns with a reflector (:462)
    for (int64_t k = 0; k < ncols; k += kPanel) {
        if (tri_resident_fits(n - k, h->num_cus)) {
            bool done = false;
            GLA_TRY(tri_resident<T>(h, s, n - k, A + k * (lda + 1), lda, tau + k, P, &done));
            if (done) break;
        }
        const int w = (int)std::min<int64_t>(kPanel, ncols - k);
        for (int j = 0; j < w; ++j) {
            const int64_t c = k + j;
            const int64_t m = n - c - 1;
            const unsigned g1 = (unsigned)cdiv(n - c, kRPB);
            const int qcnt = (int)cdiv(n - c, kRPB);   // the previous column's tri_w grid
            hipLaunchKernelGGL((tri_col_kernel<T>), dim3(g1), dim3(256), 0, s, n, c, j, A, lda, V,
                               W, ldv, qpart, qcnt, scal, npart);
            GLA_LAUNCH_CHECK();
            const int64_t nbk = cdiv(m, kTB);
            hipLaunchKernelGGL((tri_symv_kernel<T>), dim3((unsigned)(nbk * (nbk + 1) / 2)),
                               dim3(256), 0, s, n, c, j, (const T *)A, lda, (const T *)V,
                               (const T *)W, ldv, (const T *)npart, (int)g1, P, Y1, Y2, scal, tau);
            GLA_LAUNCH_CHECK();
            const unsigned g4 = (unsigned)cdiv(m, kRPB);
            hipLaunchKernelGGL((tri_w_kernel<T>), dim3(g4), dim3(256), 0, s, n, c, j, A, lda, V, W,
                               ldv, (const T *)P, (int)nbk, (const T *)Y1, (const T *)Y2, scal,
                               qpart);
            GLA_LAUNCH_CHECK();
        }
        // W's last column: u -> w over rows ≥ k + w
        const int64_t c1 = k + w;
        hipLaunchKernelGGL((tri_wfin_kernel<T>), dim3((unsigned)cdiv(n - c1, 256)), dim3(256), 0,
                           s, n, c1, w - 1, V, W, ldv, (const T *)qpart, (int)cdiv(n - c1, kRPB),
                           (const T *)scal);
        GLA_LAUNCH_CHECK();
        // Ã[c1:, c1:] −= V Wᵀ + W Vᵀ (lower triangle)
        const int64_t mt = n - c1;
        if (mt > 0) {
            GLA_TRY(gemm<T>(s, 'N', 'T', 1, mt, mt, w, T(-1), V + c1, ldv, W + c1, ldv, T(1),
                            A + c1 + c1 * lda, lda, 0));
            GLA_TRY(gemm<T>(s, 'N', 'T', 1, mt, mt, w, T(-1), W + c1, ldv, V + c1, ldv, T(1),
                            A + c1 + c1 * lda, lda, 0));
        }
    }
    return GLA_OK;
}

template <typename T>
int symtri_dev(Handle *h, hipStream_t s, char uplo, int64_t n, T *A, int64_t lda, T *tau, T *ws)
{
    const dim3 rg((unsigned)cdiv(n, 16), (unsigned)cdiv(n, 16));
    if (uplo == 'U') {
        hipLaunchKernelGGL((reverse_kernel<T>), rg, dim3(16, 16), 0, s, n, A, lda);
        GLA_LAUNCH_CHECK();
    }
    GLA_TRY(symtri_lower_dev<T>(h, s, n, A, lda, tau, ws));
    if (uplo == 'U') {
        hipLaunchKernelGGL((reverse_kernel<T>), rg, dim3(16, 16), 0, s, n, A, lda);
        GLA_LAUNCH_CHECK();
    }
    return GLA_OK;
}

template int symtri_dev<double>(Handle *, hipStream_t, char, int64_t, double *, int64_t, double *, double *);
template int symtri_dev<float>(Handle *, hipStream_t, char, int64_t, float *, int64_t, float *, float *);

// Workspace elements of bidiagonalize! for m×n.
size_t bidiag_scratch(int64_t m, int64_t n, bool resident)
{
    const int64_t M = std::max(m, n), N = std::min(m, n);   // the tall problem
    const int64_t ldm = (M + 3) / 4 * 4, ldn = (N + 3) / 4 * 4;
    const int64_t nrb = cdiv(M, kTB), ncb = cdiv(N, kTB), g = cdiv(M, kRPB) + 1;
    // the GEMVs' partials, or the resident kernel's exchange for the largest
    // trailing block that fits it
    size_t pe = std::max((size_t)nrb * N, (size_t)ncb * M), re = 0;
    for (int64_t k = 0; resident && k < N; k += kPanel)
        if (bd_resident_fits(M - k, N - k, 256)) {
            re = bd_resident_elems(M - k, N - k);
            break;
        }
    pe = std::max(pe, re);
    const size_t tr = m < n ? (size_t)ldm * N : 0;   // Aᵀ for the wide case
    return 2 * (size_t)ldm * kPanel + 2 * (size_t)ldn * kPanel + pe +
           2 * (size_t)nrb * kPanel + 2 * (size_t)ncb * kPanel + 2 * (size_t)g + 16 + tr;
}

// bidiagonalize! of a tall A (m ≥ n): panels of deferred updates until the
// trailing block fits the resident kernel, which takes the rest.
template <typename T>
int bidiag_tall_dev(Handle *h, hipStream_t s, int64_t m, int64_t n, T *A, int64_t lda, T *taul, T *taur,
                    T *ws)
{
    const int64_t ldm = (m + 3) / 4 * 4, ldn = (n + 3) / 4 * 4;
    const int64_t nrb_max = cdiv(m, kTB), ncb_max = cdiv(n, kTB), gmax = cdiv(m, kRPB) + 1;
    T *V = ws, *X = V + ldm * kPanel, *Y = X + ldm * kPanel, *U = Y + ldn * kPanel;
    T *P = U + ldn * kPanel;
    T *Cv1 = P + std::max(nrb_max * n, ncb_max * m), *Cv2 = Cv1 + nrb_max * kPanel;
    T *Cu1 = Cv2 + nrb_max * kPanel, *Cu2 = Cu1 + ncb_max * kPanel;
    T *npart = Cu2 + ncb_max * kPanel, *npart2 = npart + gmax, *scal = npart2 + gmax;
    for (int64_t k = 0; k < n; k += kPanel) {
        if (bd_resident_fits(m - k, n - k, h->num_cus)) {
            bool done = false;
            GLA_TRY(bd_resident<T>(h, s, m - k, n - k, A + k * (lda + 1), lda, taul + k, taur + k, P,
                                   &done));
            if (done) break;
        }
        const int w = (int)std::min<int64_t>(kPanel, n - k);
        int ncnt = (int)cdiv(m - k, 256);
        hipLaunchKernelGGL((bd_col0_kernel<T>), dim3((unsigned)ncnt), dim3(256), 0, s, m, k,
                           (const T *)A, lda, npart);
        GLA_LAUNCH_CHECK();
        for (int j = 0; j < w; ++j) {
            const int64_t i = k + j;
            const int64_t C = n - i - 1, R = m - i;
            const int64_t nrb = cdiv(R, kTB), ncb = std::max<int64_t>(1, cdiv(C, kTB));
            const unsigned g2 = (unsigned)(C > 0 ? nrb * ncb : 1);
            hipLaunchKernelGGL((bd_gemvt_kernel<T>), dim3(g2), dim3(256), 0, s, m, n, i, j,
                               (const T *)A, lda, (const T *)V, (const T *)X, ldm,
                               (const T *)npart, ncnt, ncb, P, Cv1, Cv2, scal, taul);
            GLA_LAUNCH_CHECK();
            const unsigned g3 = (unsigned)cdiv(std::max(R, C), kRPB);
            hipLaunchKernelGGL((bd_y_kernel<T>), dim3(g3), dim3(256), 0, s, m, n, i, j, A, lda, V,
                               (const T *)X, ldm, Y, (const T *)U, ldn, (const T *)P,
                               C > 0 ? nrb : 0, (const T *)Cv1, (const T *)Cv2, (const T *)scal,
                               npart2);
            GLA_LAUNCH_CHECK();
            if (C == 0) break;   // the last column: no right reflector (src/svd.jl:339)
            const int64_t R1 = m - i - 1;
            const int64_t nrb1 = cdiv(R1, kTB), ncb1 = cdiv(C, kTB);
            hipLaunchKernelGGL((bd_gemvn_kernel<T>), dim3((unsigned)(nrb1 * ncb1)), dim3(256), 0,
                               s, m, n, i, j, (const T *)A, lda, (const T *)Y, (const T *)U, ldn,
                               (const T *)npart2, (int)g3, ncb1, P, Cu1, Cu2, scal, taur);
            GLA_LAUNCH_CHECK();
            const int last = j == w - 1;
            const unsigned g5 = (unsigned)cdiv(std::max(R1, C), kRPB);
            hipLaunchKernelGGL((bd_x_kernel<T>), dim3(g5), dim3(256), 0, s, m, n, i, j, last, A,
                               lda, (const T *)V, X, ldm, (const T *)Y, U, ldn, (const T *)P,
                               ncb1, (const T *)Cu1, (const T *)Cu2, (const T *)scal, npart);
            GLA_LAUNCH_CHECK();
            ncnt = (int)g5;
        }
        const int64_t c1 = k + w;
        if (c1 < n) {   // Ã[c1:, c1:] −= V Yᵀ + X Uᵀ
            GLA_TRY(gemm<T>(s, 'N', 'T', 0, m - c1, n - c1, w, T(-1), V + c1, ldm, Y + c1, ldn,
                            T(1), A + c1 + c1 * lda, lda, 0));
            GLA_TRY(gemm<T>(s, 'N', 'T', 0, m - c1, n - c1, w, T(-1), X + c1, ldm, U + c1, ldn,
                            T(1), A + c1 + c1 * lda, lda, 0));
        }
    }
    return GLA_OK;
}

// bidiagonalize!: tall directly, wide (m < n) as the tall problem of Aᵀ
// (its left reflectors are A's right ones, src/svd.jl:356-375 mirrors
// :332-349), transposed back.
template <typename T>
int bidiag_dev(Handle *h, hipStream_t s, int64_t m, int64_t n, T *A, int64_t lda, T *taul, T *taur,
               T *ws)
{
    if (m == 0 || n == 0) return GLA_OK;
    if (m >= n) return bidiag_tall_dev<T>(h, s, m, n, A, lda, taul, taur, ws);
    const int64_t ldt = (n + 3) / 4 * 4;
    T *At = ws;
    T *rest = ws + (size_t)ldt * m;
    hipLaunchKernelGGL((transpose_kernel<T>), dim3((unsigned)cdiv(m, 16), (unsigned)cdiv(n, 16)),
                       dim3(16, 16), 0, s, m, n, (const T *)A, lda, At, ldt);
    GLA_LAUNCH_CHECK();
    GLA_TRY(bidiag_tall_dev<T>(h, s, n, m, At, ldt, taur, taul, rest));
    hipLaunchKernelGGL((transpose_kernel<T>), dim3((unsigned)cdiv(n, 16), (unsigned)cdiv(m, 16)),
                       dim3(16, 16), 0, s, n, m, (const T *)At, ldt, A, lda);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}

template int bidiag_dev<double>(Handle *, hipStream_t, int64_t, int64_t, double *, int64_t, double *,
                                double *, double *);
template int bidiag_dev<float>(Handle *, hipStream_t, int64_t, int64_t, float *, int64_t, float *, float *,
                               float *);

}  // namespace gla

// ------------------------------------------------------------------ C ABI --
namespace {

template <typename T>
int symtri_entry(gla_handle_t hh, char uplo, int64_t n, T *A, int64_t lda, T *tau, void *stream)
{
    gla::Handle *h = reinterpret_cast<gla::Handle *>(hh);
    if (!h) { gla::set_error("null handle"); return -1; }
    if (uplo != 'L' && uplo != 'U') { gla::set_error("uplo must be 'L' or 'U'"); return -2; }
    if (n < 0) { gla::set_error("n < 0"); return -3; }
    if (!A && n > 0) { gla::set_error("A is null"); return -4; }
    if (lda < std::max<int64_t>(1, n)) { gla::set_error("lda < max(1,n)"); return -5; }
    if (!tau && n > 1) { gla::set_error("tau is null"); return -6; }
    if (n == 0) return GLA_OK;
    GLA_HIP_TRY(hipSetDevice(h->device));
    const hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    GLA_TRY(gla::ensure_workspace(h, gla::symtri_scratch(n, !gla::capturing(s)) * sizeof(T)));
    return gla::symtri_dev<T>(h, s, uplo, n, A, lda, tau,
                              reinterpret_cast<T *>(h->ws));
}


template <typename T>
int bidiag_entry(gla_handle_t hh, int64_t m, int64_t n, T *A, int64_t lda, T *taul, T *taur,
                 void *stream)
{
    gla::Handle *h = reinterpret_cast<gla::Handle *>(hh);
    if (!h) { gla::set_error("null handle"); return -1; }
    if (m < 0) { gla::set_error("m < 0"); return -2; }
    if (n < 0) { gla::set_error("n < 0"); return -3; }
    if (!A && m > 0 && n > 0) { gla::set_error("A is null"); return -4; }
    if (lda < std::max<int64_t>(1, m)) { gla::set_error("lda < max(1,m)"); return -5; }
    const int64_t k = std::min(m, n);
    const int64_t nl = m >= n ? k : k - 1, nr = m >= n ? k - 1 : k;
    if (!taul && nl > 0) { gla::set_error("taul is null"); return -6; }
    if (!taur && nr > 0) { gla::set_error("taur is null"); return -7; }
    if (k == 0) return GLA_OK;
    GLA_HIP_TRY(hipSetDevice(h->device));
    const hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    GLA_TRY(gla::ensure_workspace(h, gla::bidiag_scratch(m, n, !gla::capturing(s)) * sizeof(T)));
    return gla::bidiag_dev<T>(h, s, m, n, A, lda, taul, taur,
                              reinterpret_cast<T *>(h->ws));
}

}  // namespace

extern "C" {

int gla_symtri_d(gla_handle_t h, char uplo, int64_t n, double *A, int64_t lda, double *tau,
                 void *stream)
{
    return symtri_entry<double>(h, uplo, n, A, lda, tau, stream);
}
int gla_symtri_s(gla_handle_t h, char uplo, int64_t n, float *A, int64_t lda, float *tau,
                 void *stream)
{
    return symtri_entry<float>(h, uplo, n, A, lda, tau, stream);
}

int gla_bidiag_d(gla_handle_t h, int64_t m, int64_t n, double *A, int64_t lda, double *taul,
                 double *taur, void *stream)
{
    return bidiag_entry<double>(h, m, n, A, lda, taul, taur, stream);
}
int gla_bidiag_s(gla_handle_t h, int64_t m, int64_t n, float *A, int64_t lda, float *taul,
                 float *taur, void *stream)
{
    return bidiag_entry<float>(h, m, n, A, lda, taul, taur, stream);
}

}  // extern "C"
