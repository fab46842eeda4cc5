// Reverse-mode derivatives (adjoints) of the Cholesky and QR factorisations.
// No counterpart in the reference (src/cholesky.jl and src/qr.jl define the
// forward factorisations only).  Formulas:
//
// Cholesky, A = L Lᵀ (Murray 2016, arXiv:1602.07527, eq. 10):
//   P  = Φ(Lᵀ L̄)            Φ: lower triangle with the diagonal halved
//   Ā  = ½ L⁻ᵀ (P + Pᵀ) L⁻¹  (symmetric convention)
//   or tril(2Ā) − diag(Ā)    (lower-only convention: the derivative with
//                             respect to the lower triangle the
//                             factorisation reads)
//   Note ½(P + Pᵀ) = ½ copyltu(Lᵀ L̄), copyltu(M) = tril(M) + tril(M,−1)ᵀ.
// QR, A = Q R, m ≥ n, Q̄ = 0 (Walter & Lehmann 2018; Liao et al. 2019):
//   M = R R̄ᵀ,  Ā = Q [copyltu(M) R⁻ᵀ ; 0]
//
// Device plan.  A batch: one launch for the factors and one for all the rest,
// with the matrix in one workgroup (chol_adjoint_kernel).  Single matrices: the
// triangle–triangle products run on the MFMA GEMM with
// the K range of each tile starting at its first row (kfrom_row), so the
// work is that of the triangular product.  Both right-side solves
// X ← X L⁻¹ use the Cholesky driver's solve B ← B L⁻ᵀ with the reversed
// matrix Lr = J Lᵀ J (J the reversal): X L⁻¹ = ((X J) Lr⁻ᵀ) J.  For QR,
// R⁻ᵀ = (Rᵀ)⁻¹ with Rᵀ lower, reversed as Kr = J R J.  The final Q product
// is the compact-WY apply of the factorisation's own reflectors.
#include <algorithm>

#include "gla_internal.hpp"

namespace gla {

namespace {

#define GLA_TRY(expr)                  \
    do {                               \
        int _rc = (expr);              \
        if (_rc != GLA_OK) return _rc; \
    } while (0)

#define GLA_COLS(j, ncols) for (int64_t j = blockIdx.y; j < (ncols); j += gridDim.y)
#define GLA_ROW(i) const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x

inline dim3 g2(int64_t rows, int64_t cols)
{
    return dim3((unsigned)cdiv(rows, 256), (unsigned)std::min<int64_t>(cols, 65535));
}

// D (n×n) <- op(tri(S)), zeros elsewhere.  src_lower: the lower triangle of
// S is taken (else the upper); trans: D = tri(S)ᵀ.
template <typename T>
__global__ void tri_copy(int64_t n, const T *S, int64_t lds, T *D, int64_t ldd, int src_lower,
                         int trans)
{
    GLA_ROW(i);
    GLA_COLS(j, n)
    if (i < n) {
        const int64_t si = trans ? j : i, sj = trans ? i : j;
        const bool keep = src_lower ? si >= sj : si <= sj;
        D[i + j * ldd] = keep ? S[si + sj * lds] : T(0);
    }
}

// D[i][n-1-j] = scale · M[max(i,j)][min(i,j)]: scale·copyltu(M), columns
// reversed (reads the lower triangle of M only).
template <typename T>
__global__ void sym_lower_rev(int64_t n, const T *M, int64_t ldm, T scale, T *D, int64_t ldd)
{
    GLA_ROW(i);
    GLA_COLS(j, n)
    if (i < n) {
        const int64_t a = i > j ? i : j, b = i > j ? j : i;
        D[i + (n - 1 - j) * ldd] = scale * M[a + b * ldm];
    }
}

// D = J Sᵀ J: D[i][j] = S[n-1-j][n-1-i], n×n.
template <typename T>
__global__ void rev_transpose(int64_t n, const T *S, int64_t lds, T *D, int64_t ldd)
{
    GLA_ROW(i);
    GLA_COLS(j, n) if (i < n) D[i + j * ldd] = S[(n - 1 - j) + (n - 1 - i) * lds];
}

// Lower-triangular reversals (the strict upper part is not written):
// transpose = 1: Lr = J Lᵀ J of a lower L, Lr[i][j] = L[n-1-j][n-1-i];
// transpose = 0: Kr = J R J of an upper R,  Kr[i][j] = R[n-1-i][n-1-j].
template <typename T>
__global__ void rev_lower(int64_t n, const T *S, int64_t lds, T *D, int64_t ldd, int transpose)
{
    GLA_ROW(i);
    GLA_COLS(j, n)
    if (i < n && i >= j)
        D[i + j * ldd] = transpose ? S[(n - 1 - j) + (n - 1 - i) * lds]
                                   : S[(n - 1 - i) + (n - 1 - j) * lds];
}

// Cholesky output from Res2 (Z = J Res2ᵀ = Res2 J in exact arithmetic):
// Z[i][j] = ½(Res2[i][n-1-j] + Res2[j][n-1-i]), exactly symmetric.
// lower_only: 2Z below the diagonal, Z on it, 0 above.
template <typename T>
__global__ void chol_adj_out(int64_t n, const T *R, int64_t ldr, T *Ab, int64_t ldab,
                             int lower_only)
{
    GLA_ROW(i);
    GLA_COLS(j, n)
    if (i < n) {
        const T z = T(0.5) * (R[i + (n - 1 - j) * ldr] + R[j + (n - 1 - i) * ldr]);
        T v = z;
        if (lower_only) v = i > j ? T(2) * z : (i == j ? z : T(0));
        Ab[i + j * ldab] = v;
    }
}

// QR: Ab[i][j] = Res[i][n-1-j] for i < n, 0 for n ≤ i < m.
template <typename T>
__global__ void qr_adj_top(int64_t m, int64_t n, const T *R, int64_t ldr, T *Ab, int64_t ldab)
{
    GLA_ROW(i);
    GLA_COLS(j, n) if (i < m) Ab[i + j * ldab] = i < n ? R[i + (n - 1 - j) * ldr] : T(0);
}

#undef GLA_COLS
#undef GLA_ROW

template <typename T>
int launch_tri_copy(hipStream_t s, int64_t n, const T *S, int64_t lds, T *D, int src_lower,
                    int trans)
{
    hipLaunchKernelGGL((tri_copy<T>), g2(n, n), dim3(256), 0, s, n, S, lds, D, n,
                       src_lower, trans);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}

// ---- the batched Cholesky adjoint, orders up to 16·NT ----
// One workgroup per matrix, one wave per column of 16×16 tiles, L's strictly
// lower tiles and the inverses of the diagonal ones in LDS, everything else
// in registers:
//   1  the wave's column of W = Lᵀ L̄ (tiles on and below the diagonal), and
//      S = ½ copyltu(W) by one exchange of tiles through LDS;
//   2  Y = L⁻ᵀ S, substitution from the last row on, each wave by itself;
//   3  Yᵀ's column by another exchange, Zᵀ = L⁻ᵀ Yᵀ the same way;
//   4  ½ (Z + Zᵀ) by a third.
// A tile in the accumulator's layout is the B operand of a product over its
// rows, and kept that way in LDS ("register order") the A operand of its
// transpose, so no product moves data: only the exchanges transpose.
// Accuracy: sums with a triangular tile run from its far end to the diagonal,
// which holds the largest term.  Error against a wider evaluation, in eps, from
// the diagonal on and to it (the twelve launches' in brackets): FP64 n = 16 1.03
// and 0.77 (0.85), 128 2.22 and 2.10 (2.16); FP32 n = 16 0.93 and 0.87 (0.92).
// Bound: memory and the matrix cores in turn (one workgroup per CU at NT = 8):
// per matrix of order 128 696 tile products, FP64 19 µs, and L, L̄ and Ā, 12 µs
// at a CU's share of the bandwidth.  512 matrices of order 128, FP64: 100 µs, two
// per CU, after 31 µs for the factors; the whole call 667 -> 181 µs against
// twelve launches that carried every step through memory.
// NT of 2, 4 and 8, so that small matrices share a CU: 1000 of order 16
// 208 -> 69 µs, of 64 512 -> 123, 65535 of order 5 5.8 -> 0.65 ms.
template <typename T, int NT>
struct AdjLds {
    T L[NT * (NT - 1) / 2][256];   // tile (k, j), k > j, at k (k − 1)/2 + j, register order
    T inv[NT][256];                // L_jj⁻¹, register order
    T E[NT * NT / 2][256];         // exchange
};

template <typename T, int NT>
__global__ __launch_bounds__(64 * NT, NT == 8 ? 2 : 1) void chol_adjoint_kernel(
    int n, const T *Lw, const T *Lb, int64_t ldlb, int64_t sLb,
    T *Ab, int64_t ldab, int64_t sAb, int lower_only)
{
    typedef PanelMfma<T> M;
    typedef typename M::acc_t acc_t;
    constexpr int H = NT / 2;
    __shared__ AdjLds<T, NT> sh;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int lc = lane & 15;
    // the wave's tile column: waves that share a SIMD take c and NT − 1 − c
    // (product 1 is a triangle)
    const int c = w < H ? w : NT - 1 - (w - H);
    const int nt = (n + 15) / 16;
    Lw += (int64_t)blockIdx.x * n * n;
    Lb += blockIdx.x * sLb;
    Ab += blockIdx.x * sAb;

    // a tile to LDS and its transpose back; rows rotated against columns, so
    // that both ways are free of bank conflicts
    auto put = [&](int slot, const acc_t &v) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = M::row(lane, r);
            sh.E[slot][row * 16 + (lc ^ row)] = v[r];
        }
    };
    auto take = [&](int slot) {
        acc_t v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = sh.E[slot][lc * 16 + (M::row(lane, r) ^ lc)];
        return v;
    };
    const acc_t zero = {T(0), T(0), T(0), T(0)};

    // L̄'s column c, rows from the diagonal; L to LDS (its diagonal tiles are
    // needed here only, and come last, from memory)
    acc_t g[NT], s[NT];
#pragma unroll
    for (int k = 0; k < NT; ++k) {
        g[k] = zero;
        if (k >= c && k < nt) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * k + M::row(lane, r), col = 16 * c + lc;
                const bool in = row < n && col <= row;
                const T v = Lb[in ? row + (int64_t)col * ldlb : 0];
                g[k][r] = in ? v : T(0);
            }
        }
    }
    for (int e = w; e < nt * (nt - 1) / 2; e += NT) {
        int k = 1;
        while (k * (k + 1) / 2 <= e) ++k;
        const int j = e - k * (k - 1) / 2;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * k + M::row(lane, r), col = 16 * j + lc;
            const T v = Lw[row < n ? row + (int64_t)col * n : 0];
            sh.L[e][r * 64 + lane] = row < n ? v : T(0);
        }
    }
    // the inverse X of diagonal tile w, a row per lane from X L = I (not L X:
    // what is applied below is Xᵀ, and Lᵀ Xᵀ is to be I)
    if (w < nt) {
        T *D = sh.E[w];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = lc, j = M::row(lane, r), row = 16 * w + i, col = 16 * w + j;
            const bool in = row < n && j <= i;
            const T v = Lw[in ? row + (int64_t)col * n : 0];
            D[i * 16 + j] = in ? v : (i == j ? T(1) : T(0));
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        T x[16];
#pragma unroll
        for (int i = 15; i >= 0; --i) {
            T t = i == lc ? T(1) : T(0);
#pragma unroll
            for (int j = i + 1; j < 16; ++j) t = fma_t(-D[j * 16 + i], x[j], t);
            x[i] = t / D[i * 17];
        }
        // register order
        const int at = sizeof(T) == 8 ? (lc >> 2) * 64 + (lc & 3) * 16 : (lc & 3) * 64 + (lc >> 2) * 16;
#pragma unroll
        for (int i = 0; i < 16; ++i) sh.inv[w][at + i] = x[i];
    }
    __syncthreads();

    // 1: W's column c, tiles i ≥ c
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        s[i] = zero;
        if (i < c || i >= nt) continue;
        // L_iiᵀ
        T d[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int row = 16 * i + M::row(lane, q), col = 16 * i + lc;
            const bool in = row < n && col <= row;
            const T v = Lw[in ? row + (int64_t)col * n : 0];
            d[q] = in ? v : T(0);
        }
#pragma unroll
        for (int k = i + 1; k < NT; ++k) {
            if (k >= nt) continue;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                s[i] = M::mma(sh.L[k * (k - 1) / 2 + i][q * 64 + lane], g[k][q], s[i]);
        }
        // the diagonal tile last and its rows from the last: the sums then
        // end with L_ii, their largest term
#pragma unroll
        for (int q = 3; q >= 0; --q) s[i] = M::mma(d[q], g[i][q], s[i]);
    }
    // S: the diagonal tile mirrored by itself, tiles above from their owners
#pragma unroll
    for (int i = 0; i < NT; ++i)
        if (i == c) put(c, s[i]);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    {
        const acc_t t = take(c);
#pragma unroll
        for (int i = 0; i < NT; ++i)
            if (i == c) {
#pragma unroll
                for (int r = 0; r < 4; ++r) s[i][r] = M::row(lane, r) < lc ? t[r] : s[i][r];
            }
    }
    lds_barrier();
#pragma unroll
    for (int i = 1; i < NT; ++i)
        if (i > c && i < nt) put(i * (i - 1) / 2 + c, s[i]);
    lds_barrier();
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        if (i < c && c < nt) s[i] = take(c * (c - 1) / 2 + i);
#pragma unroll
        for (int r = 0; r < 4; ++r) s[i][r] *= T(0.5);
    }
    lds_barrier();

    // s <- L⁻ᵀ s
    auto sweep = [&](acc_t (&x)[NT]) {
        if (c >= nt) return;
#pragma unroll
        for (int j = NT - 1; j >= 0; --j) {
            if (j >= nt) continue;
            acc_t y = zero;
#pragma unroll
            for (int q = 3; q >= 0; --q) y = M::mma(sh.inv[j][q * 64 + lane], x[j][q], y);
            x[j] = y;
#pragma unroll
            for (int i = 0; i < j; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    x[i] = M::mma(sh.L[j * (j - 1) / 2 + i][q * 64 + lane], -y[q], x[i]);
        }
    };
    // x (column c of X) <- column c of Xᵀ, half of the rows at a time
    auto transpose = [&](const acc_t (&x)[NT], acc_t (&o)[NT]) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int i = 0; i < H; ++i) put(i * NT + c, x[h * H + i]);
            lds_barrier();
            if (c / H == h) {
#pragma unroll
                for (int i = 0; i < NT; ++i) o[i] = take((c - h * H) * NT + i);
            }
            lds_barrier();
        }
    };
    sweep(s);
    transpose(s, g);
    sweep(g);
    transpose(g, s);
    // Ā is symmetric: its tile (i, c) is written as tile (c, i), whose columns
    // are the lanes' rows
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        if (i >= nt || c >= nt) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * c + lc, col = 16 * i + M::row(lane, r);
            const T z = T(0.5) * (g[i][r] + s[i][r]);
            T v = z;
            if (lower_only) v = row > col ? T(2) * z : (row == col ? z : T(0));
            if (row < n && col < n) Ab[row + (int64_t)col * ldab] = v;
        }
    }
}

template <typename T, int NT>
int launch_chol_adjoint(hipStream_t s, int64_t n, int64_t batch, const T *Lw, const T *Lb, int64_t ldlb, int64_t sLb, T *Ab, int64_t ldab,
                        int64_t sAb, int lower_only)
{
    hipLaunchKernelGGL((chol_adjoint_kernel<T, NT>), dim3((unsigned)batch), dim3(64 * NT),
                       0, s, (int)n, Lw, Lb, ldlb, sLb, Ab, ldab,
                       sAb, lower_only);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}

}  // namespace

size_t chol_adjoint_scratch(int64_t n) { return 4 * (size_t)n * n + tile_inverse_elems(n) + 64; }

// Ā for one matrix; L, L̄ lower (their strict upper parts are not read).
template <typename T>
int chol_adjoint_dev(hipStream_t s, int64_t n, const T *L, int64_t ldl, const T *Lb,
                     int64_t ldlb, T *Ab, int64_t ldab, int lower_only, T *scratch)
{
    if (n <= 0) return GLA_OK;
    const size_t nn = (size_t)n * n;
    T *Lt = scratch, *Gt = Lt + nn, *W = Gt + nn, *Lr = W + nn, *Linv = Lr + nn;
    GLA_TRY(launch_tri_copy<T>(s, n, L, ldl, Lt, 1, 1));     // Lt = tril(L)ᵀ
    GLA_TRY(launch_tri_copy<T>(s, n, Lb, ldlb, Gt, 1, 1));   // Gt = tril(L̄)ᵀ
    // W (lower) = Lt · Gtᵀ = Lᵀ L̄, k from each tile's first row
    GLA_TRY(gemm<T>(s, 'N', 'T', 1, n, n, n, T(1), Lt, n, Gt, n, T(0), W, n, 0, nullptr, 0, 1));
    // Lt <- ½ copyltu(W) J
    hipLaunchKernelGGL((sym_lower_rev<T>), g2(n, n), dim3(256), 0, s, n, W, n, T(0.5), Lt, n);
    GLA_LAUNCH_CHECK();
    hipLaunchKernelGGL((rev_lower<T>), g2(n, n), dim3(256), 0, s, n, L, ldl, Lr, n, 1);
    GLA_LAUNCH_CHECK();
    GLA_TRY(tile_inverses<T>(s, n, Lr, n, Linv));
    GLA_TRY(trsm_rlt<T>(s, n, n, Lr, n, Linv, Lt, n));        // Res1 = Psym J Lr⁻ᵀ
    hipLaunchKernelGGL((rev_transpose<T>), g2(n, n), dim3(256), 0, s, n, Lt, n, W, n);
    GLA_LAUNCH_CHECK();
    GLA_TRY(trsm_rlt<T>(s, n, n, Lr, n, Linv, W, n));         // Res2 = J Res1ᵀ J Lr⁻ᵀ
    hipLaunchKernelGGL((chol_adj_out<T>), g2(n, n), dim3(256), 0, s, n, W, n, Ab, ldab,
                       lower_only);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}

// Per-matrix scratch of the batched form (n ≤ 128): L.
size_t chol_adjoint_batched_scratch(int64_t n) { return (size_t)n * n; }

// Ā for a strided batch of SPD matrices of order n ≤ 128, recomputing each
// factor L from A.  info[b] = first failing pivot of matrix b.
template <typename T>
int chol_adjoint_batched_dev(hipStream_t s, int64_t n, int64_t batch, const T *A, int64_t lda,
                             int64_t sA, const T *Lb, int64_t ldlb, int64_t sLb, T *Ab,
                             int64_t ldab, int64_t sAb, int lower_only, int *info, T *scratch)
{
    if (n <= 0 || batch <= 0) return GLA_OK;
    const int64_t nn = n * n;
    T *Lw = scratch;
    GLA_TRY(chol_factor_batched<T>(s, (int)n, A, lda, sA, Lw, n, nn, info, batch));
    if (n <= 32)
        return launch_chol_adjoint<T, 2>(s, n, batch, Lw, Lb, ldlb, sLb, Ab, ldab, sAb,
                                         lower_only);
    if (n <= 64)
        return launch_chol_adjoint<T, 4>(s, n, batch, Lw, Lb, ldlb, sLb, Ab, ldab, sAb,
                                         lower_only);
    return launch_chol_adjoint<T, 8>(s, n, batch, Lw, Lb, ldlb, sLb, Ab, ldab, sAb,
                                     lower_only);
}

size_t qr_adjoint_scratch(int64_t m, int64_t n)
{
    return 5 * (size_t)n * n + tile_inverse_elems(n) +
           std::max(qr_tblock_scratch(m, n), qr_apply_scratch(m, n, n)) + 64;
}

// Ā (m×n) for A = QR as stored by qrBlocked!/qrUnblocked! (F, τ), R̄ upper.
template <typename T>
int qr_adjoint_dev(hipStream_t s, int64_t m, int64_t n, const T *F, int64_t ldf, const T *tau,
                   const T *Rb, int64_t ldrb, T *Ab, int64_t ldab, T *scratch)
{
    if (n <= 0 || m <= 0) return GLA_OK;
    const size_t nn = (size_t)n * n;
    T *Rz = scratch, *Gz = Rz + nn, *W = Gz + nn, *Kr = W + nn, *Tm = Kr + nn, *Linv = Tm + nn;
    T *rest = Linv + tile_inverse_elems(n);
    GLA_TRY(launch_tri_copy<T>(s, n, F, ldf, Rz, 0, 0));     // R
    GLA_TRY(launch_tri_copy<T>(s, n, Rb, ldrb, Gz, 0, 0));   // triu(R̄)
    // W (lower) = R R̄ᵀ
    GLA_TRY(gemm<T>(s, 'N', 'T', 1, n, n, n, T(1), Rz, n, Gz, n, T(0), W, n, 0, nullptr, 0, 1));
    hipLaunchKernelGGL((sym_lower_rev<T>), g2(n, n), dim3(256), 0, s, n, W, n, T(1), Gz, n);
    GLA_LAUNCH_CHECK();
    hipLaunchKernelGGL((rev_lower<T>), g2(n, n), dim3(256), 0, s, n, Rz, n, Kr, n, 0);
    GLA_LAUNCH_CHECK();
    GLA_TRY(tile_inverses<T>(s, n, Kr, n, Linv));
    GLA_TRY(trsm_rlt<T>(s, n, n, Kr, n, Linv, Gz, n));        // copyltu(M) J Kr⁻ᵀ
    hipLaunchKernelGGL((qr_adj_top<T>), g2(m, n), dim3(256), 0, s, m, n, Gz, n, Ab, ldab);
    GLA_LAUNCH_CHECK();
    GLA_TRY(qr_tblock_dev<T>(s, m, n, F, ldf, tau, Tm, n, rest));
    return qr_apply_dev<T>(s, 'N', m, n, n, F, ldf, Tm, n, Ab, ldab, rest);
}

}  // namespace gla

// ------------------------------------------------------------------ C ABI --
namespace {

using gla::Handle;

// (a kernel rather than a memset, so the call can be captured in a graph)
__global__ void zero_ints(int64_t n, int *p)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

template <typename T>
int chol_adjoint_entry(gla_handle_t hh, char conv, int64_t n, const T *L, int64_t ldl,
                       const T *Lb, int64_t ldlb, T *Ab, int64_t ldab, void *stream)
{
    Handle *h = reinterpret_cast<Handle *>(hh);
    if (!h) { gla::set_error("null handle"); return -1; }
    if (conv != 'S' && conv != 'L') { gla::set_error("convention must be 'S' or 'L'"); return -2; }
    if (n < 0) return -3;
    if (ldl < std::max<int64_t>(1, n)) return -5;
    if (ldlb < std::max<int64_t>(1, n)) return -7;
    if (ldab < std::max<int64_t>(1, n)) return -9;
    if (n == 0) return GLA_OK;
    GLA_HIP_TRY(hipSetDevice(h->device));
    GLA_TRY(gla::ensure_workspace(h, gla::chol_adjoint_scratch(n) * sizeof(T)));
    return gla::chol_adjoint_dev<T>(reinterpret_cast<hipStream_t>(stream), n, L, ldl, Lb, ldlb,
                                    Ab, ldab, conv == 'L', reinterpret_cast<T *>(h->ws));
}

template <typename T>
int chol_adjoint_batched_entry(gla_handle_t hh, char conv, int64_t n, int64_t batch, const T *A,
                               int64_t lda, int64_t sA, const T *Lb, int64_t ldlb, int64_t sLb,
                               T *Ab, int64_t ldab, int64_t sAb, int32_t *info, void *stream)
{
    Handle *h = reinterpret_cast<Handle *>(hh);
    if (!h) { gla::set_error("null handle"); return -1; }
    if (conv != 'S' && conv != 'L') { gla::set_error("convention must be 'S' or 'L'"); return -2; }
    if (n < 0) return -3;
    if (n > 128) {
        gla::set_error("batched Cholesky adjoint: order %lld exceeds 128", (long long)n);
        return GLA_ERR_UNSUPPORTED;
    }
    if (batch < 0) return -4;
    if (lda < std::max<int64_t>(1, n)) return -6;
    if (ldlb < std::max<int64_t>(1, n)) return -9;
    if (ldab < std::max<int64_t>(1, n)) return -12;
    if (n == 0 || batch == 0) return GLA_OK;
    GLA_HIP_TRY(hipSetDevice(h->device));
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    // chunks of at most 65535 matrices (one grid dimension each)
    const int64_t chunk = std::min<int64_t>(batch, 65535);
    const size_t per = gla::chol_adjoint_batched_scratch(n) * sizeof(T);
    const size_t data = ((size_t)chunk * per + 255) / 256 * 256;
    GLA_TRY(gla::ensure_workspace(h, data + 4 * (size_t)batch + 256));
    int *dinfo = info ? reinterpret_cast<int *>(info)
                      : reinterpret_cast<int *>(reinterpret_cast<char *>(h->ws) + data);
    hipLaunchKernelGGL(zero_ints, dim3((unsigned)gla::cdiv(batch, 256)), dim3(256), 0, s, batch,
                       dinfo);
    GLA_LAUNCH_CHECK();
    for (int64_t b0 = 0; b0 < batch; b0 += chunk) {
        const int64_t nb = std::min<int64_t>(chunk, batch - b0);
        GLA_TRY(gla::chol_adjoint_batched_dev<T>(s, n, nb, A + b0 * sA, lda, sA, Lb + b0 * sLb,
                                                 ldlb, sLb, Ab + b0 * sAb, ldab, sAb, conv == 'L',
                                                 dinfo + b0, reinterpret_cast<T *>(h->ws)));
    }
    return GLA_OK;
}

template <typename T>
int qr_adjoint_entry(gla_handle_t hh, int64_t m, int64_t n, const T *F, int64_t ldf,
                     const T *tau, const T *Rb, int64_t ldrb, T *Ab, int64_t ldab, void *stream)
{
    Handle *h = reinterpret_cast<Handle *>(hh);
    if (!h) { gla::set_error("null handle"); return -1; }
    if (m < 0) return -2;
    if (n < 0 || n > m) { gla::set_error("the QR adjoint needs 0 <= n <= m"); return -3; }
    if (ldf < std::max<int64_t>(1, m)) return -5;
    if (ldrb < std::max<int64_t>(1, n)) return -8;
    if (ldab < std::max<int64_t>(1, m)) return -10;
    if (n == 0) return GLA_OK;
    GLA_HIP_TRY(hipSetDevice(h->device));
    GLA_TRY(gla::ensure_workspace(h, gla::qr_adjoint_scratch(m, n) * sizeof(T)));
    return gla::qr_adjoint_dev<T>(reinterpret_cast<hipStream_t>(stream), m, n, F, ldf, tau, Rb,
                                  ldrb, Ab, ldab, reinterpret_cast<T *>(h->ws));
}

}  // namespace

extern "C" {

int gla_chol_adjoint_d(gla_handle_t h, char conv, int64_t n, const double *L, int64_t ldl,
                       const double *Lbar, int64_t ldlbar, double *Abar, int64_t ldabar,
                       void *stream)
{
    return chol_adjoint_entry<double>(h, conv, n, L, ldl, Lbar, ldlbar, Abar, ldabar, stream);
}
int gla_chol_adjoint_s(gla_handle_t h, char conv, int64_t n, const float *L, int64_t ldl,
                       const float *Lbar, int64_t ldlbar, float *Abar, int64_t ldabar,
                       void *stream)
{
    return chol_adjoint_entry<float>(h, conv, n, L, ldl, Lbar, ldlbar, Abar, ldabar, stream);
}
int gla_chol_adjoint_batched_d(gla_handle_t h, char conv, int64_t n, int64_t batch,
                               const double *A, int64_t lda, int64_t strideA, const double *Lbar,
                               int64_t ldlbar, int64_t strideLbar, double *Abar, int64_t ldabar,
                               int64_t strideAbar, int32_t *info, void *stream)
{
    return chol_adjoint_batched_entry<double>(h, conv, n, batch, A, lda, strideA, Lbar, ldlbar,
                                              strideLbar, Abar, ldabar, strideAbar, info, stream);
}
int gla_chol_adjoint_batched_s(gla_handle_t h, char conv, int64_t n, int64_t batch,
                               const float *A, int64_t lda, int64_t strideA, const float *Lbar,
                               int64_t ldlbar, int64_t strideLbar, float *Abar, int64_t ldabar,
                               int64_t strideAbar, int32_t *info, void *stream)
{
    return chol_adjoint_batched_entry<float>(h, conv, n, batch, A, lda, strideA, Lbar, ldlbar,
                                             strideLbar, Abar, ldabar, strideAbar, info, stream);
}
int gla_qr_adjoint_d(gla_handle_t h, int64_t m, int64_t n, const double *F, int64_t ldf,
                     const double *tau, const double *Rbar, int64_t ldrbar, double *Abar,
                     int64_t ldabar, void *stream)
{
    return qr_adjoint_entry<double>(h, m, n, F, ldf, tau, Rbar, ldrbar, Abar, ldabar, stream);
}
int gla_qr_adjoint_s(gla_handle_t h, int64_t m, int64_t n, const float *F, int64_t ldf,
                     const float *tau, const float *Rbar, int64_t ldrbar, float *Abar,
                     int64_t ldabar, void *stream)
{
    return qr_adjoint_entry<float>(h, m, n, F, ldf, tau, Rbar, ldrbar, Abar, ldabar, stream);
}

}  // extern "C"
