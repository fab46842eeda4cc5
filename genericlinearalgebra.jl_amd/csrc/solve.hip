// Solves with the factors: A X = B from a Cholesky factor (LAPACK potrs,
// Julia's ldiv! with a Cholesky) and the least-squares solution of A X ≈ B
// from a Householder QR (Julia's ldiv! with a QR: lmul!(Hᴴ, B) of
// src/householder.jl:119-157, then back-substitution with R).  The
// reference defines the factorisations only (src/cholesky.jl:3-55,
// src/qr.jl:86-146); these are the solves a caller applies to their
// results.
//
// Device plan.  Up to kFewRhs right-hand sides: one launch per triangle
// (tri_solve), which reads the factor where it lies.  More: right-side solves
// on the transposed right-hand sides (rows of length n, one per right-hand
// side) with the Cholesky driver's B <- B L⁻ᵀ (16×16 tile inverses, MFMA
// GEMMs between 128-wide leaves):
//   L y = b           ⇔  yᵀ = bᵀ L⁻ᵀ;
//   Lᵀ x = y          ⇔  xᵀ = yᵀ L⁻¹ = ((yᵀ J) Lr⁻ᵀ) J,  Lr = J Lᵀ J lower;
//   R x = y (R upper) ⇔  xᵀ = yᵀ R⁻ᵀ = ((yᵀ J) Kr⁻ᵀ) J,  Kr = J R J lower,
// J the reversal (Lr⁻ᵀ = J L⁻¹ J).  Qᵀ B is the compact-WY apply of the
// factorisation's own reflectors.
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

// Y (nrhs×n, row k = right-hand side k) from B (n×nrhs):
// Y[k][i] = B[rev ? n−1−i : i][k].
template <typename T>
__global__ void to_rows_k(int64_t n, int64_t nrhs, const T *B, int64_t ldb, T *Y, int rev)
{
    GLA_ROW(i);
    GLA_COLS(k, nrhs)
    if (i < n) Y[k + i * nrhs] = B[(rev ? n - 1 - i : i) + k * ldb];
}

// Z = Y J for Y nrhs×n: Z[k][j] = Y[k][n−1−j].
template <typename T>
__global__ void colrev_k(int64_t n, int64_t nrhs, const T *Y, T *Z)
{
    GLA_ROW(k);
    GLA_COLS(j, n)
    if (k < nrhs) Z[k + j * nrhs] = Y[k + (n - 1 - j) * nrhs];
}

// B (n×nrhs) = (Z J)ᵀ: B[i][k] = Z[k][n−1−i].
template <typename T>
__global__ void from_rows_rev_k(int64_t n, int64_t nrhs, const T *Z, T *B, int64_t ldb)
{
    GLA_ROW(i);
    GLA_COLS(k, nrhs)
    if (i < n) B[i + k * ldb] = Z[k + (n - 1 - i) * nrhs];
}

// Lower-triangular reversals (strict upper part not written):
// transpose = 1: D = J Sᵀ J of a lower S;  transpose = 0: D = J S J of an upper S.
template <typename T>
__global__ void rev_lower_k(int64_t n, const T *S, int64_t lds, T *D, int64_t ldd, int transpose)
{
    GLA_ROW(i);
    GLA_COLS(j, n)
    if (i < n && i >= j)
        D[i + j * ldd] = transpose ? S[(n - 1 - j) + (n - 1 - i) * lds]
                                   : S[(n - 1 - i) + (n - 1 - j) * lds];
}

// D (lower) = Sᵀ of an upper S.
template <typename T>
__global__ void upper_to_lower_k(int64_t n, const T *S, int64_t lds, T *D, int64_t ldd)
{
    GLA_ROW(i);
    GLA_COLS(j, n)
    if (i < n && i >= j) D[i + j * ldd] = S[j + i * lds];
}

// *info = 1 + the first index with a zero diagonal entry of R (unchanged if
// none; the caller sets it to n + 1 first).
template <typename T>
__global__ void first_zero_diag_k(int64_t n, const T *R, int64_t ldr, int *info)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && R[i + i * ldr] == T(0)) atomicMin(info, (int)(i + 1));
}

// info: the first zero of the diagonal, and whether a wait has given up
__global__ void set_info_k(int *p, int v)
{
    p[0] = v;
    p[1] = 0;
}

// S (rows×cols, ld lds) = 0.
template <typename T>
__global__ void set_zero_k(int64_t rows, int64_t cols, T *S, int64_t lds)
{
    GLA_ROW(i);
    GLA_COLS(j, cols)
    if (i < rows) S[i + j * lds] = T(0);
}

// Y (n×nrhs, column-major) <- D Y, D the diagonal of F.
template <typename T>
__global__ void scale_rows_k(int64_t n, int64_t nrhs, const T *F, int64_t ldf, T *Y, int64_t ldy)
{
    GLA_ROW(i);
    GLA_COLS(k, nrhs)
    if (i < n) Y[i + k * ldy] *= F[i + i * ldf];
}

// Lx (n×n, lower, explicit unit diagonal) = the unit lower factor of LDLᵀ
// data F: L = F's strict lower triangle (upper = 0), or Uᵀ (upper = 1).
template <typename T>
__global__ void unit_lower_k(int64_t n, const T *F, int64_t ldf, T *Lx, int upper)
{
    GLA_ROW(i);
    GLA_COLS(j, n)
    if (i < n && i >= j)
        Lx[i + j * n] = i == j ? T(1) : (upper ? F[j + i * ldf] : F[i + j * ldf]);
}

// Y (nrhs×n, row k = right-hand side k): Y[k][i] /= d_i, d the diagonal of F.
template <typename T>
__global__ void div_rows_k(int64_t n, int64_t nrhs, const T *F, int64_t ldf, T *Y)
{
    GLA_ROW(k);
    GLA_COLS(i, n)
    if (k < nrhs) Y[k + i * nrhs] = Y[k + i * nrhs] / F[i + i * ldf];
}

// G <- I + stril(G) D, D = diag(d); the upper triangle is left alone.
template <typename T>
__global__ void unit_scale_k(int64_t n, T *G, const T *d)
{
    GLA_ROW(i);
    GLA_COLS(j, n)
    if (i < n && i >= j) G[i + j * n] = i == j ? T(1) : G[i + j * n] * d[j];
}

// W (n×nrhs) = D Zᵀ for Z nrhs×n.
template <typename T>
__global__ void scaled_cols_k(int64_t n, int64_t nrhs, const T *Z, const T *d, T *W)
{
    GLA_ROW(i);
    GLA_COLS(k, nrhs)
    if (i < n) W[i + k * n] = d[i] * Z[k + i * nrhs];
}

#undef GLA_COLS
#undef GLA_ROW

// With Z = yᵀ J (nrhs×n): Z <- Z M⁻ᵀ for the lower M, then B[0:n] = (Z J)ᵀ.
template <typename T>
int reversed_tail(hipStream_t s, int64_t n, int64_t nrhs, const T *M, int64_t ldm, T *Minv,
                  T *Z, T *B, int64_t ldb)
{
    GLA_TRY(tile_inverses<T>(s, n, M, ldm, Minv));
    GLA_TRY(trsm_rlt<T>(s, nrhs, n, M, ldm, Minv, Z, nrhs));
    hipLaunchKernelGGL((from_rows_rev_k<T>), g2(n, nrhs), dim3(256), 0, s, n, nrhs, Z, B, ldb);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}

}  // namespace

// Up to here one tri_solve launch per triangle, which reads the factor where
// it lies; beyond, the GEMM form, whose tiles of L serve more columns at a
// time.  Two solves with a Cholesky factor, GEMM form -> tri_solve, µs: FP64
// n = 5001 3507 -> 473 (16 right-hand sides) and 4243 -> 1088 (512), 4096
// 3621 -> 2736 (2000) but 7359 -> 10435 (8192), 1000 541 -> 106 (16),
// 646 -> 153 (1000) and 1745 -> 1930 (20000); FP32 5001 2768 -> 312 (16),
// 4096 4645 -> 3945 (8192).
constexpr int64_t kFewRhs = 2048;

// L Lᵀ X = B or L D Lᵀ X = B, L the lower triangle of F or the transposed
// upper one (unit: its diagonal is taken as 1 and F's is D).
template <typename T>
int few_rhs_solve(const Handle *h, hipStream_t s, char uplo, int unit, int64_t n, int64_t nrhs,
                  const T *F, int64_t ldf, T *B, int64_t ldb, T *scratch)
{
    const size_t ye = tri_solve_elems(n, nrhs);
    int *ticket = reinterpret_cast<int *>(scratch + 2 * ye);
    GLA_TRY(tri_solve_prepare<T>(s, (int64_t)(2 * ye), scratch, ticket, 2));
    TriSolve<T> p{};
    p.n = n;
    p.unit = unit;
    p.nrhs = (int)nrhs;
    p.spin_limit = h->spin_limit;
    // L y = b
    p.M = F;
    p.si = uplo == 'U' ? ldf : 1;
    p.sj = uplo == 'U' ? 1 : ldf;
    p.R = B;
    p.ri = 1;
    p.rk = ldb;
    p.rp = 16 * ldb;
    p.Y = scratch;
    p.ticket = ticket;
    GLA_TRY(tri_solve<T>(s, p));
    // Lᵀ x = y (D⁻¹ y), rows and columns from the last
    const int64_t l = n - 1;
    p.M = F + l * (ldf + 1);
    const int64_t t = p.si;
    p.si = -p.sj;
    p.sj = -t;
    p.R = scratch + l * 16;
    p.ri = -16;
    p.rk = 1;
    p.rp = (int64_t)(ye / cdiv(nrhs, 16));
    if (unit) {
        p.div = F + l * (ldf + 1);
        p.ds = -(ldf + 1);
    }
    p.Y = scratch + ye;
    p.out = B + l;
    p.oi = -1;
    p.ok = ldb;
    p.ticket = ticket + 1;
    return tri_solve<T>(s, p);
}

// Scratch elements of the Cholesky solve: two exchanges and their tickets, or
// Uᵀ (uplo 'U'), Lr, two tile-inverse sets, two nrhs×n row blocks.
size_t chol_solve_scratch(int64_t n, int64_t nrhs)
{
    if (nrhs <= kFewRhs) return 2 * tri_solve_elems(n, nrhs) + 64;
    return 2 * (size_t)n * n + 2 * tile_inverse_elems(n) + 2 * (size_t)nrhs * n + 256;
}

// B (n×nrhs) <- A⁻¹ B with A = L Lᵀ (uplo 'L', L lower) or A = Uᵀ U
// (uplo 'U', U upper); the other triangle of F is not read.
template <typename T>
int chol_solve_dev(const Handle *h, hipStream_t s, char uplo, int64_t n, int64_t nrhs, const T *F, int64_t ldf,
                   T *B, int64_t ldb, T *scratch)
{
    if (n <= 0 || nrhs <= 0) return GLA_OK;
    if (nrhs <= kFewRhs)
        return few_rhs_solve<T>(h, s, uplo, 0, n, nrhs, F, ldf, B, ldb, scratch);
    const size_t nn = (size_t)n * n, ti = tile_inverse_elems(n);
    T *Lx = scratch, *Lr = Lx + nn, *Li = Lr + nn, *Lri = Li + ti, *Y = Lri + ti,
      *Z = Y + (size_t)nrhs * n;
    const T *L = F;
    int64_t ldl = ldf;
    if (uplo == 'U') {   // L = Uᵀ
        hipLaunchKernelGGL((upper_to_lower_k<T>), g2(n, n), dim3(256), 0, s, n, F, ldf, Lx, n);
        GLA_LAUNCH_CHECK();
        L = Lx;
        ldl = n;
    }
    // yᵀ = bᵀ L⁻ᵀ
    hipLaunchKernelGGL((to_rows_k<T>), g2(n, nrhs), dim3(256), 0, s, n, nrhs, B, ldb, Y, 0);
    GLA_LAUNCH_CHECK();
    GLA_TRY(tile_inverses<T>(s, n, L, ldl, Li));
    GLA_TRY(trsm_rlt<T>(s, nrhs, n, L, ldl, Li, Y, nrhs));
    // xᵀ = ((yᵀ J) Lr⁻ᵀ) J
    hipLaunchKernelGGL((colrev_k<T>), g2(nrhs, n), dim3(256), 0, s, n, nrhs, Y, Z);
    GLA_LAUNCH_CHECK();
    hipLaunchKernelGGL((rev_lower_k<T>), g2(n, n), dim3(256), 0, s, n, L, ldl, Lr, n, 1);
    GLA_LAUNCH_CHECK();
    return reversed_tail<T>(s, n, nrhs, Lr, n, Lri, Z, B, ldb);
}

// B (n×nrhs) <- L⁻ᵀ D⁻¹ L⁻¹ B for LDLᵀ factor data F (uplo 'L': L in the
// strict lower triangle, D on the diagonal; 'U': L = Uᵀ) — ldiv!(F::LDLt, X),
// src/ldlt.jl:225-228.  Same scratch as the Cholesky solve.
template <typename T>
int ldlt_solve_dev(const Handle *h, hipStream_t s, char uplo, int64_t n, int64_t nrhs, const T *F, int64_t ldf,
                   T *B, int64_t ldb, T *scratch)
{
    if (n <= 0 || nrhs <= 0) return GLA_OK;
    if (nrhs <= kFewRhs)
        return few_rhs_solve<T>(h, s, uplo, 1, n, nrhs, F, ldf, B, ldb, scratch);
    const size_t nn = (size_t)n * n, ti = tile_inverse_elems(n);
    T *Lx = scratch, *Lr = Lx + nn, *Li = Lr + nn, *Lri = Li + ti, *Y = Lri + ti,
      *Z = Y + (size_t)nrhs * n;
    hipLaunchKernelGGL((unit_lower_k<T>), g2(n, n), dim3(256), 0, s, n, F, ldf, Lx,
                       uplo == 'U' ? 1 : 0);
    GLA_LAUNCH_CHECK();
    // yᵀ = bᵀ L⁻ᵀ (ldiv!(L, X)), then ldiv!(D, X)
    hipLaunchKernelGGL((to_rows_k<T>), g2(n, nrhs), dim3(256), 0, s, n, nrhs, B, ldb, Y, 0);
    GLA_LAUNCH_CHECK();
    GLA_TRY(tile_inverses<T>(s, n, Lx, n, Li));
    GLA_TRY(trsm_rlt<T>(s, nrhs, n, Lx, n, Li, Y, nrhs));
    hipLaunchKernelGGL((div_rows_k<T>), g2(nrhs, n), dim3(256), 0, s, n, nrhs, F, ldf, Y);
    GLA_LAUNCH_CHECK();
    // ldiv!(L', X): xᵀ = ((yᵀ J) Lr⁻ᵀ) J
    hipLaunchKernelGGL((colrev_k<T>), g2(nrhs, n), dim3(256), 0, s, n, nrhs, Y, Z);
    GLA_LAUNCH_CHECK();
    hipLaunchKernelGGL((rev_lower_k<T>), g2(n, n), dim3(256), 0, s, n, Lx, n, Lr, n, 1);
    GLA_LAUNCH_CHECK();
    return reversed_tail<T>(s, n, nrhs, Lr, n, Lri, Z, B, ldb);
}

// B (n×nrhs) <- L D Lᵀ B — lmul!(F::LDLt, X), src/ldlt.jl:229-232 (and
// F * X, :234): two MFMA products with the explicit unit factor.
// Scratch: n² + n·nrhs elements.
template <typename T>
int ldlt_lmul_dev(hipStream_t s, char uplo, int64_t n, int64_t nrhs, const T *F, int64_t ldf,
                  T *B, int64_t ldb, T *scratch)
{
    if (n <= 0 || nrhs <= 0) return GLA_OK;
    T *Lx = scratch, *Y = Lx + (size_t)n * n;
    hipLaunchKernelGGL((set_zero_k<T>), g2(n, n), dim3(256), 0, s, n, n, Lx, n);
    GLA_LAUNCH_CHECK();
    hipLaunchKernelGGL((unit_lower_k<T>), g2(n, n), dim3(256), 0, s, n, F, ldf, Lx,
                       uplo == 'U' ? 1 : 0);
    GLA_LAUNCH_CHECK();
    // Y = Lᵀ B (lmul!(L', X)), then D Y (lmul!(D, X)), then B = L Y (lmul!(L, X))
    GLA_TRY(gemm<T>(s, 'T', 'N', 0, n, nrhs, n, T(1), Lx, n, B, ldb, T(0), Y, n, 0));
    hipLaunchKernelGGL((scale_rows_k<T>), g2(n, nrhs), dim3(256), 0, s, n, nrhs, F, ldf, Y, n);
    GLA_LAUNCH_CHECK();
    return gemm<T>(s, 'N', 'N', 0, n, nrhs, n, T(1), Lx, n, Y, n, T(0), B, ldb, 0);
}

// Scratch elements of the QR solve: explicit V, G = VᵀV (then J Rᵀ J), tile
// inverses, three nrhs×n blocks, split-K partials.
size_t qr_solve_scratch(int64_t m, int64_t n, int64_t nrhs)
{
    return (size_t)m * n + (size_t)n * n + tile_inverse_elems(n) + 3 * (size_t)nrhs * n +
           8 * (size_t)nrhs * n + (nrhs <= kFewRhs ? 32 + 2 * tri_solve_elems(n, nrhs) : 0) + 256;
}

// Least squares for m ≥ n: B (m×nrhs) <- Qᵀ B, then B[0:n] <- R⁻¹ B[0:n],
// with (F, τ) as stored by qrBlocked!/qrUnblocked!.  info (device, two ints):
// 1 + the first zero diagonal entry of R, n + 1 when R is nonsingular; and 1
// when a wait gave up.
// Qᵀ B = B − V Tᵀ Vᵀ B with T = (I + D striu(VᵀV))⁻¹ D, D = diag(τ)
// (src/qr.jl:64-83, src/householder.jl:119-157), so TᵀW = D L⁻¹ W for the
// unit lower L = I + stril(VᵀV) D: a solve with nrhs rows instead of T's
// explicit inverse (1501×700: 1.0 ms of 128-wide inverses).
template <typename T>
int qr_solve_dev(const Handle *h, hipStream_t s, int64_t m, int64_t n, int64_t nrhs, const T *F, int64_t ldf,
                 const T *tau, T *B, int64_t ldb, int *info, T *scratch)
{
    if (n <= 0 || nrhs <= 0) return GLA_OK;
    const size_t nr = (size_t)nrhs * n;
    T *Vw = scratch, *G = Vw + (size_t)m * n, *Gi = G + (size_t)n * n,
      *W = Gi + tile_inverse_elems(n), *Z = W + nr, *W2 = Z + nr, *split = W2 + nr;
    hipLaunchKernelGGL(set_info_k, dim3(1), dim3(1), 0, s, info, (int)(n + 1));
    GLA_LAUNCH_CHECK();
    hipLaunchKernelGGL((first_zero_diag_k<T>), dim3((unsigned)cdiv(n, 256)), dim3(256), 0, s, n, F,
                       ldf, info);
    GLA_LAUNCH_CHECK();
    GLA_TRY(unit_lower_explicit<T>(s, m, n, F, ldf, Vw, m));
    GLA_TRY(gemm<T>(s, 'T', 'N', 0, n, n, m, T(1), Vw, m, Vw, m, T(0), G, n));
    hipLaunchKernelGGL((unit_scale_k<T>), g2(n, n), dim3(256), 0, s, n, G, tau);
    GLA_LAUNCH_CHECK();
    // W = VᵀB, Z = (L⁻¹ W)ᵀ, W2 = D Zᵀ, B -= V W2
    GLA_TRY(gemm<T>(s, 'T', 'N', 0, n, nrhs, m, T(1), Vw, m, B, ldb, T(0), W, n, 0, split, 8 * nr));
    if (nrhs <= kFewRhs) {
        const size_t ye = tri_solve_elems(n, nrhs);
        T *Y = scratch + (split + 8 * nr - scratch + 31) / 32 * 32;   // on 16 bytes (scratch is)
        int *ticket = reinterpret_cast<int *>(Y + 2 * ye);
        GLA_TRY(tri_solve_prepare<T>(s, (int64_t)(2 * ye), Y, ticket, 2));
        TriSolve<T> p{};
        p.n = n;
        p.nrhs = (int)nrhs;
        p.spin_limit = h->spin_limit;
        p.err = info + 1;
        p.unit = 1;                       // W2 = D L⁻¹ W
        p.M = G;
        p.si = 1;
        p.sj = n;
        p.R = W;
        p.ri = 1;
        p.rk = n;
        p.rp = 16 * n;
        p.Y = Y;
        p.out = W2;
        p.oi = 1;
        p.ok = n;
        p.mul = tau;
        p.ms = 1;
        p.ticket = ticket;
        GLA_TRY(tri_solve<T>(s, p));
        GLA_TRY(gemm<T>(s, 'N', 'N', 0, m, nrhs, n, T(-1), Vw, m, W2, n, T(1), B, ldb));
        const int64_t l = n - 1;          // R x = y, rows and columns from the last
        p.unit = 0;
        p.M = F + l * (ldf + 1);
        p.si = -1;
        p.sj = -ldf;
        p.R = B + l;
        p.ri = -1;
        p.rk = ldb;
        p.rp = 16 * ldb;
        p.Y = Y + ye;
        p.out = B + l;
        p.oi = -1;
        p.ok = ldb;
        p.mul = nullptr;
        p.ticket = ticket + 1;
        return tri_solve<T>(s, p);
    }
    hipLaunchKernelGGL((to_rows_k<T>), g2(n, nrhs), dim3(256), 0, s, n, nrhs, W, n, Z, 0);
    GLA_LAUNCH_CHECK();
    GLA_TRY(tile_inverses<T>(s, n, G, n, Gi));
    GLA_TRY(trsm_rlt<T>(s, nrhs, n, G, n, Gi, Z, nrhs));
    hipLaunchKernelGGL((scaled_cols_k<T>), g2(n, nrhs), dim3(256), 0, s, n, nrhs, Z, tau, W2);
    GLA_LAUNCH_CHECK();
    GLA_TRY(gemm<T>(s, 'N', 'N', 0, m, nrhs, n, T(-1), Vw, m, W2, n, T(1), B, ldb));
    // R x = y: Z = yᵀ J, Z <- Z Kr⁻ᵀ, x = (Z J)ᵀ
    T *Kr = G, *Kri = Gi;
    hipLaunchKernelGGL((to_rows_k<T>), g2(n, nrhs), dim3(256), 0, s, n, nrhs, B, ldb, Z, 1);
    GLA_LAUNCH_CHECK();
    hipLaunchKernelGGL((rev_lower_k<T>), g2(n, n), dim3(256), 0, s, n, F, ldf, Kr, n, 0);
    GLA_LAUNCH_CHECK();
    return reversed_tail<T>(s, n, nrhs, Kr, n, Kri, Z, B, ldb);
}

}  // namespace gla

// ------------------------------------------------------------------ C ABI --
namespace {

using gla::Handle;

template <typename T>
int chol_solve_entry(gla_handle_t hh, char uplo, int64_t n, int64_t nrhs, const T *F, int64_t ldf,
                     T *B, int64_t ldb, void *stream)
{
    Handle *h = reinterpret_cast<Handle *>(hh);
    if (!h) { gla::set_error("null handle"); return -1; }
    if (uplo != 'L' && uplo != 'U') { gla::set_error("uplo must be 'L' or 'U'"); return -2; }
    if (n < 0) return -3;
    if (nrhs < 0) return -4;
    if (ldf < std::max<int64_t>(1, n)) return -6;
    if (ldb < std::max<int64_t>(1, n)) return -8;
    if (n == 0 || nrhs == 0) return GLA_OK;
    GLA_HIP_TRY(hipSetDevice(h->device));
    GLA_TRY(gla::ensure_workspace(h, gla::chol_solve_scratch(n, nrhs) * sizeof(T)));
    return gla::chol_solve_dev<T>(h, reinterpret_cast<hipStream_t>(stream), uplo, n, nrhs, F, ldf, B,
                                  ldb, reinterpret_cast<T *>(h->ws));
}

// mode 0: ldiv!(F::LDLt, B); 1: lmul!(F::LDLt, B).
template <typename T>
int ldlt_apply_entry(gla_handle_t hh, int mode, char uplo, int64_t n, int64_t nrhs, const T *F,
                     int64_t ldf, T *B, int64_t ldb, void *stream)
{
    Handle *h = reinterpret_cast<Handle *>(hh);
    if (!h) { gla::set_error("null handle"); return -1; }
    if (uplo != 'L' && uplo != 'U') { gla::set_error("uplo must be 'L' or 'U'"); return -2; }
    if (n < 0) return -3;
    if (nrhs < 0) return -4;
    if (ldf < std::max<int64_t>(1, n)) { gla::set_error("ldf < max(1,n)"); return -6; }
    if (ldb < std::max<int64_t>(1, n)) { gla::set_error("ldb < max(1,n)"); return -8; }
    if (n == 0 || nrhs == 0) return GLA_OK;
    GLA_HIP_TRY(hipSetDevice(h->device));
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const size_t need = mode == 0 ? gla::chol_solve_scratch(n, nrhs)
                                  : (size_t)n * n + (size_t)n * nrhs + 64;
    GLA_TRY(gla::ensure_workspace(h, need * sizeof(T)));
    T *ws = reinterpret_cast<T *>(h->ws);
    if (mode == 0) return gla::ldlt_solve_dev<T>(h, s, uplo, n, nrhs, F, ldf, B, ldb, ws);
    return gla::ldlt_lmul_dev<T>(s, uplo, n, nrhs, F, ldf, B, ldb, ws);
}

template <typename T>
int qr_solve_entry(gla_handle_t hh, int64_t m, int64_t n, int64_t nrhs, const T *F, int64_t ldf,
                   const T *tau, T *B, int64_t ldb, int64_t *info, void *stream)
{
    Handle *h = reinterpret_cast<Handle *>(hh);
    if (!h) { gla::set_error("null handle"); return -1; }
    if (m < 0) return -2;
    if (n < 0 || n > m) { gla::set_error("the QR solve needs 0 <= n <= m"); return -3; }
    if (nrhs < 0) return -4;
    if (ldf < std::max<int64_t>(1, m)) return -6;
    if (!tau && n > 0) return -7;
    if (ldb < std::max<int64_t>(1, m)) return -9;
    if (info) *info = 0;
    if (n == 0 || nrhs == 0) return GLA_OK;
    GLA_HIP_TRY(hipSetDevice(h->device));
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    GLA_TRY(gla::ensure_workspace(h, gla::qr_solve_scratch(m, n, nrhs) * sizeof(T)));
    GLA_TRY(gla::qr_solve_dev<T>(h, s, m, n, nrhs, F, ldf, tau, B, ldb, h->dinfo + 8,
                                 reinterpret_cast<T *>(h->ws)));
    if (info) {
        int hv[2] = {0, 0};
        GLA_HIP_TRY(hipMemcpyAsync(hv, h->dinfo + 8, sizeof(hv), hipMemcpyDeviceToHost, s));
        GLA_HIP_TRY(hipStreamSynchronize(s));
        if (hv[1]) {
            gla::set_error("least squares: a device-side wait gave up after %u polls", h->spin_limit);
            return GLA_ERR_TIMEOUT;
        }
        *info = hv[0] > n ? 0 : hv[0];
    }
    return GLA_OK;
}

}  // namespace

extern "C" {

int gla_chol_solve_d(gla_handle_t h, char uplo, int64_t n, int64_t nrhs, const double *F,
                     int64_t ldf, double *B, int64_t ldb, void *stream)
{
    return chol_solve_entry<double>(h, uplo, n, nrhs, F, ldf, B, ldb, stream);
}
int gla_chol_solve_s(gla_handle_t h, char uplo, int64_t n, int64_t nrhs, const float *F,
                     int64_t ldf, float *B, int64_t ldb, void *stream)
{
    return chol_solve_entry<float>(h, uplo, n, nrhs, F, ldf, B, ldb, stream);
}
int gla_ldlt_solve_d(gla_handle_t h, char uplo, int64_t n, int64_t nrhs, const double *F,
                     int64_t ldf, double *B, int64_t ldb, void *stream)
{
    return ldlt_apply_entry<double>(h, 0, uplo, n, nrhs, F, ldf, B, ldb, stream);
}
int gla_ldlt_solve_s(gla_handle_t h, char uplo, int64_t n, int64_t nrhs, const float *F,
                     int64_t ldf, float *B, int64_t ldb, void *stream)
{
    return ldlt_apply_entry<float>(h, 0, uplo, n, nrhs, F, ldf, B, ldb, stream);
}
int gla_ldlt_lmul_d(gla_handle_t h, char uplo, int64_t n, int64_t nrhs, const double *F,
                    int64_t ldf, double *B, int64_t ldb, void *stream)
{
    return ldlt_apply_entry<double>(h, 1, uplo, n, nrhs, F, ldf, B, ldb, stream);
}
int gla_ldlt_lmul_s(gla_handle_t h, char uplo, int64_t n, int64_t nrhs, const float *F,
                    int64_t ldf, float *B, int64_t ldb, void *stream)
{
    return ldlt_apply_entry<float>(h, 1, uplo, n, nrhs, F, ldf, B, ldb, stream);
}
int gla_qr_solve_d(gla_handle_t h, int64_t m, int64_t n, int64_t nrhs, const double *F,
                   int64_t ldf, const double *tau, double *B, int64_t ldb, int64_t *info,
                   void *stream)
{
    return qr_solve_entry<double>(h, m, n, nrhs, F, ldf, tau, B, ldb, info, stream);
}
int gla_qr_solve_s(gla_handle_t h, int64_t m, int64_t n, int64_t nrhs, const float *F,
                   int64_t ldf, const float *tau, float *B, int64_t ldb, int64_t *info,
                   void *stream)
{
    return qr_solve_entry<float>(h, m, n, nrhs, F, ldf, tau, B, ldb, info, stream);
}

}  // extern "C"
