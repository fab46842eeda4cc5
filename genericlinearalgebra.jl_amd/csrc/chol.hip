// Cholesky on gfx950: cholUnblocked!, cholBlocked!, cholRecursive!
// (src/cholesky.jl:3-55) and the rdiv!/rankUpdate! steps they call.
//
// Kernels
//   chol_factor_kernel  One workgroup factors a diagonal block (≤128×128) in
//                       place.  The block is held as 16×16 MFMA accumulator
//                       tiles; waves 1–3 hold them, wave 0 factors and
//                       inverts one diagonal tile after another
//                       (tile_factor) while waves 1–3 apply the rank-16
//                       update C -= X_i X_jᵀ on MFMA.  The tile inverses are
//                       kept for the panel solve.
//   chol_solve_kernel   rdiv!(A21, LowerTriangular(A11)') (src/cholesky.jl:28,
//                       48) for a ≤128-wide L11: each workgroup takes 64 rows
//                       of A21, L11's tiles and tile inverses sit in LDS, and
//                       every 16-column step is X = B_kb·L_kk⁻ᵀ then
//                       B_j -= X·L_(j,kb)ᵀ on MFMA.  A batched form (grid y)
//                       inverts many diagonal blocks at once.
//   gemm (gemm.hip)     The trailing rankUpdate!(Hermitian(A22,:L), A21, -1)
//                       as an MFMA SYRK over lower tiles.
//
// Drivers
//   blocked    right-looking, block nb ≤ 128, depth-1 look-ahead: the update
//              of the next block column runs on the caller's stream right
//              after the panel, the rest of the trailing update runs on the
//              handle's side stream and overlaps the next panel.
//   look-ahead the same loop with wide blocks: the block column by one
//              dataflow launch (chol_df.hip), or the diagonal block by the
//              blocked driver and the panel by one launch or the recursive
//              rdiv!; the trailing SYRK with K = NB.
//   dataflow   cholRecursive! up to h->chol_df: the whole matrix in one
//              dataflow launch.
//   recursive  halves n as cholRecursive! does; below a threshold the blocked
//              driver factors the leaf.  rdiv! with a large L11 is itself
//              recursive (two half solves and a GEMM); its leaves are
//              chol_solve_kernel launches.
#include <algorithm>
#include <mutex>

#include "gla_internal.hpp"

namespace gla {

__global__ void k_set_int(int *p, int v) { *p = v; }

namespace {

constexpr int kPanelNB = 128;   // max diagonal block
constexpr int kPanelRB = 64;    // rows of A21 per solve workgroup
constexpr int kPanelThreads = 256;
constexpr int kXLD = 17;        // padded row length of the LDS column blocks

#define GLA_TRY(expr)                  \
    do {                               \
        int _rc = (expr);              \
        if (_rc != GLA_OK) return _rc; \
    } while (0)



// One wave holds a 16×16 tile with lane (i = l % 16, g = l / 16) owning row
// i, columns g, g+4, g+8, g+12 (v[t] = tile[i][g + 4t]).  Row i of column c
// therefore sits in lane i + 16*(c % 4), slot c / 4.

// v from lane `src` (a wave-uniform constant) to every lane, through SGPRs.
template <typename T>
__device__ __forceinline__ T lane_bcast(T v, int src)
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



// w <- L⁻¹ for a lower 16×16 tile L (rd = reciprocals of its diagonal), in
// the four-column layout (w[t] = W[i][g + 4t]).  Forward elimination of
// [L | I] with unscaled rows: V[i] = e_i − Σ_{k<i} m_ik V[k] with the
// multipliers m_ik = L[i][k]·rd[k] formed once (zero for i ≤ k, so every
// step is one broadcast and one unconditional FMA per column), then
// W[i] = rd[i]·V[i] (the steps are TileInvSteps).  L comes in row layout
// (li[k] = L[i][k]).
template <typename T>
__device__ __forceinline__ void tile_inverse_rows(const T li[16], const T rd[16], T w[4])
{
    const int lane = threadIdx.x & 63;
    const int i = lane & 15, g = lane >> 4;
    T m[16], ri = rd[0];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        m[k] = i > k ? li[k] * rd[k] : T(0);
        ri = i == k ? rd[k] : ri;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) w[t] = (i == g + 4 * t) ? T(1) : T(0);
    TileInvSteps<0, T>::run(m, w);
#pragma unroll
    for (int t = 0; t < 4; ++t) w[t] *= ri;
}

// The same from L in the four-column layout (v[t] = L[i][g + 4t]).
template <typename T>
__device__ __forceinline__ void tile_inverse(const T v[4], const T rd[16], T w[4])
{
    const int i = threadIdx.x & 15;
    T li[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) li[k] = __shfl(v[k >> 2], i + 16 * (k & 3));
    tile_inverse_rows<T>(li, rd, w);
}

// Orders one wave's LDS accesses, for data exchanged between its lanes.
__device__ __forceinline__ void wave_order() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront"); }

// Strictly-lower tile rows of waves 1..3: {7, 2}, {6, 3}, {5, 4, 1} (nine,
// nine and ten tiles), so that each 16-wide step spreads its panel tiles
// and its trailing updates evenly.  Slot q -> tile (bi, bj); bi = -1 past
// the wave's last tile.
__host__ __device__ constexpr int oslot_bi(int w, int q)
{
    return w == 1 ? (q < 7 ? 7 : (q < 9 ? 2 : -1))
         : w == 2 ? (q < 6 ? 6 : (q < 9 ? 3 : -1))
                  : (q < 5 ? 5 : (q < 9 ? 4 : (q < 10 ? 1 : -1)));
}
__host__ __device__ constexpr int oslot_bj(int w, int q)
{
    return w == 1 ? (q < 7 ? q : q - 7) : w == 2 ? (q < 6 ? q : q - 6) : (q < 5 ? q : (q < 9 ? q - 5 : q - 9));
}
// Every strictly-lower tile of the 8×8-tile block belongs to exactly one
// slot of waves 1–3, and every slot past a wave's last is marked unused.
constexpr bool oslots_cover()
{
    int seen[8][8] = {};
    for (int w = 1; w <= 3; ++w)
        for (int q = 0; q < 10; ++q) {
            const int bi = oslot_bi(w, q), bj = oslot_bj(w, q);
            if (bi < 0) continue;
            if (bi > 7 || bj < 0 || bj >= bi) return false;
            ++seen[bi][bj];
        }
    for (int i = 0; i < 8; ++i)
        for (int j = 0; j < i; ++j)
            if (seen[i][j] != 1) return false;
    return true;
}
static_assert(oslots_cover(), "the tile slots of waves 1-3 must cover the strictly-lower tiles once");

// LDLᴴ and Cholesky tiles: slot q of wave W (LDLᴴ's wave 0: diagonal tile q).
template <int W>
__host__ __device__ constexpr int dslot_bi(int q) { return W == 0 ? q : oslot_bi(W, q); }
template <int W>
__host__ __device__ constexpr int dslot_bj(int q) { return W == 0 ? q : oslot_bj(W, q); }

// Tile rows of waves 1–3, whose diagonal tiles they keep up to date until
// wave 0 factors them: row number d of wave W (0: none).
template <int W>
__host__ __device__ constexpr int row_of(int d)
{
    return W == 1 ? (d == 0 ? 7 : d == 1 ? 2 : 0)
         : W == 2 ? (d == 0 ? 6 : d == 1 ? 3 : 0)
                  : (d == 0 ? 5 : d == 1 ? 4 : 1);
}

// Tile (bi, bj) of A transposed (lane: row bi·16 + l % 16 at columns bj·16 +
// row(l, r)); a diagonal tile symmetric, from its lower triangle.  Rows and
// columns past nb continue as the identity.  fetch_tile loads from addresses
// kept inside the block (nb ≥ 1), take_tile puts the identity in: a wave has
// all its tiles' loads in flight before the first is looked at (as loads under
// a branch each, 55 of the 144 FP32 ones and all of FP64-from-FP32 were waited
// for one by one; n = 100 FP64, whole call: 46.0 -> 45.4 µs).
// TS: storage type of A.
template <typename T, typename TS>
__device__ __forceinline__ void fetch_tile(int nb, const TS *__restrict__ A, int64_t lda, int bi,
                                           int bj, TS (&raw)[4])
{
    const int lane = threadIdx.x & 63, lc = lane & 15;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int a = bi * 16 + lc, b = bj * 16 + PanelMfma<T>::row(lane, r);
        const int gi = min(a > b ? a : b, nb - 1), gj = min(a > b ? b : a, nb - 1);
        raw[r] = A[gi + (int64_t)gj * lda];
    }
}

template <typename T, typename TS>
__device__ __forceinline__ typename PanelMfma<T>::acc_t take_tile(int nb, int bi, int bj,
                                                                 TS (&raw)[4])
{
    const int lane = threadIdx.x & 63, lc = lane & 15;
    typename PanelMfma<T>::acc_t v;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int a = bi * 16 + lc, b = bj * 16 + PanelMfma<T>::row(lane, r);
        hold(raw[r]);
        v[r] = max(a, b) < nb ? T(raw[r]) : (a == b ? T(1) : T(0));
    }
    return v;
}

// Stores tile (bi, bj) held transposed, its lower triangle only.
template <typename T, typename TS>
__device__ __forceinline__ void store_tile(int nb, TS *__restrict__ A, int64_t lda, int bi, int bj,
                                           const typename PanelMfma<T>::acc_t &v)
{
    typedef PanelMfma<T> M;
    const int lane = threadIdx.x & 63, lc = lane & 15;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int gi = bi * 16 + lc, gj = bj * 16 + M::row(lane, r);
        if (gi < nb && gj <= gi) A[gi + (int64_t)gj * lda] = TS(v[r]);
    }
}

// One workgroup factors the nb×nb (nb ≤ 128) diagonal block as 16×16 MFMA
// tiles.  Waves 1–3 own the tile rows below the first (row_of), diagonal
// tiles included, held transposed; wave 0 factors and inverts the diagonal
// tiles one after the other (tile_factor).  Step kb:
//   (A) waves 1–3: the panel tiles X = A_(i,kb) L_kk⁻ᵀ (rdiv!), as
//       Xᵀ = L_kk⁻¹ A_(i,kb)ᵀ with the B operand from registers; the owner of
//       row kb + 1 first, which at once takes X Xᵀ off its diagonal tile
//       (both operands in registers) and hands that tile to wave 0.  Wave 0
//       stores the tile it has factored.
//   (B) wave 0 factors diagonal tile kb + 1; waves 1–3 apply the rank-16
//       update (rankUpdate!), C_ijᵀ -= X_j X_iᵀ, to their tiles, their later
//       diagonal tiles among them, and store column block kb.
// LDS tiles are kept as the lanes hold them (element r·64 + lane: the
// accumulator layout of a tile is an MFMA operand of it with K permuted
// alike on both sides), so every access is free of bank conflicts, and the
// barriers leave global stores in flight.
// Bound by the serial chain: 2,900 cycles of tile_factor and 1,500 of hand
// over per step.  128×128 FP64: 17.5 µs; 31 µs when wave 0 also kept the
// diagonal tiles up to date, moved each through a row layout (6,300 cycles
// per tile) and every barrier waited for the stores of the tile inverse.
// TS: storage type of A (T, or FP32 for the mixed-precision driver, which
// factors its FP32 diagonal tiles in FP64); Linv32: optional FP32 copy of
// the tile inverses.  L is stored in D, which may be A.
constexpr int kFactorX = 2 * (kPanelNB / 16) * 256;   // LDS elements: Xb,
constexpr int kFactorLi = 2 * 16 * kXLD;              // Lib (Db: one tile, 256)
template <typename T, int W, typename TS = T>
__device__ __forceinline__ void factor_body(int nb, const TS *A, int64_t lda, TS *D, int64_t ldd,
                                             int *info, int64_t info_base, T *__restrict__ LinvG, T *Xb,
                                             T *Db, T *Lib, float *__restrict__ Linv32 = nullptr)
{
    typedef PanelMfma<T> M;
    typedef typename M::acc_t acc_t;
    constexpr int NBLK = kPanelNB / 16;
    constexpr int XS = NBLK * 256, LS = 16 * kXLD;
    const int lane = threadIdx.x & 63;
    const int lc = lane & 15, lg = lane >> 4;
    const int nkb = (nb + 15) / 16;
    if (nb <= 0) return;

    if constexpr (W == 0) {
        TS raw[4];
        fetch_tile<T, TS>(nb, A, lda, 0, 0, raw);
        acc_t d = take_tile<T, TS>(nb, 0, 0, raw);
#pragma unroll 1
        for (int kb = 0; kb < nkb; ++kb) {
            if (kb > 0) {
#pragma unroll
                for (int r = 0; r < 4; ++r) d[r] = Db[r * 64 + lane];
            }
            T w[4];
            tile_factor<T>(d, w, nb - kb * 16, info, info_base + kb * 16);
            T *Li = Lib + (kb & 1) * LS;
#pragma unroll
            for (int t = 0; t < 4; ++t) Li[lc * kXLD + lg + 4 * t] = w[t];
            lds_barrier();                                            // end of (B)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if (LinvG) LinvG[kb * 256 + lc * 16 + lg + 4 * t] = w[t];
                if (Linv32) Linv32[kb * 256 + lc * 16 + lg + 4 * t] = float(w[t]);
            }
            store_tile<T, TS>(nb, D, ldd, kb, kb, d);
            lds_barrier();                                            // end of (A)
        }
    } else {
        constexpr int NQ = W == 3 ? 10 : 9, ND = W == 3 ? 3 : 2;
        acc_t acc[NQ], dg[ND];
        TS raw[NQ + ND][4];
#pragma unroll
        for (int q = 0; q < NQ; ++q)
            fetch_tile<T, TS>(nb, A, lda, oslot_bi(W, q), oslot_bj(W, q), raw[q]);
#pragma unroll
        for (int d = 0; d < ND; ++d)
            fetch_tile<T, TS>(nb, A, lda, row_of<W>(d), row_of<W>(d), raw[NQ + d]);
        lds_barrier();
#pragma unroll
        for (int q = 0; q < NQ; ++q)
            acc[q] = take_tile<T, TS>(nb, oslot_bi(W, q), oslot_bj(W, q), raw[q]);
#pragma unroll
        for (int d = 0; d < ND; ++d)
            dg[d] = take_tile<T, TS>(nb, row_of<W>(d), row_of<W>(d), raw[NQ + d]);
#pragma unroll
        for (int kb = 0; kb < NBLK; ++kb) {
            if (kb >= nkb) break;
            T *X = Xb + (kb & 1) * XS;
            const T *Lik = Lib + (kb & 1) * LS;
            // (A), ascending tile rows: row kb + 1 is the first of its owner
#pragma unroll
            for (int bi = kb + 1; bi < NBLK; ++bi) {
#pragma unroll
                for (int q = 0; q < NQ; ++q) {
                    if (oslot_bi(W, q) != bi || oslot_bj(W, q) != kb) continue;
                    if (bi >= nkb) continue;
                    acc_t x = {T(0), T(0), T(0), T(0)};
#pragma unroll
                    for (int kq = 0; kq < 4; ++kq)
                        x = M::mma(Lik[lc * kXLD + M::row(lane, kq)], acc[q][kq], x);
                    acc[q] = x;
                    if (bi == kb + 1) {
#pragma unroll
                        for (int d = 0; d < ND; ++d) {
                            if (row_of<W>(d) != bi) continue;
#pragma unroll
                            for (int kq = 0; kq < 4; ++kq) dg[d] = M::mma(-x[kq], x[kq], dg[d]);
#pragma unroll
                            for (int r = 0; r < 4; ++r) Db[r * 64 + lane] = dg[d][r];
                        }
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r) X[bi * 256 + r * 64 + lane] = x[r];
                }
            }
            lds_barrier();                                            // end of (A)
            if (kb + 1 >= nkb) break;
            // (B)
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const int bi = oslot_bi(W, q), bj = oslot_bj(W, q);
                if (bj <= kb || bi >= nkb) continue;
#pragma unroll
                for (int kq = 0; kq < 4; ++kq)
                    acc[q] = M::mma(-X[bj * 256 + kq * 64 + lane], X[bi * 256 + kq * 64 + lane],
                                    acc[q]);
            }
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const int bi = oslot_bi(W, q);
                if (oslot_bj(W, q) != kb || bi >= nkb) continue;
#pragma unroll
                for (int d = 0; d < ND; ++d) {
                    if (row_of<W>(d) != bi || bi == kb + 1) continue;
#pragma unroll
                    for (int kq = 0; kq < 4; ++kq) dg[d] = M::mma(-acc[q][kq], acc[q][kq], dg[d]);
                }
                store_tile<T, TS>(nb, D, ldd, bi, kb, acc[q]);
            }
            lds_barrier();                                            // end of (B)
        }
    }
}

// The kernels below ask for two workgroups per CU: without that the compiler
// takes 288 registers, 80 of them in the accumulator file, and a batch runs one
// workgroup per CU (512 matrices of 128, factor and adjoint, whole call: 188 ->
// 176.5 µs); with it 182.
// Factors the nb×nb (nb ≤ 128) diagonal block at A in place (lower
// triangle; the strict upper triangle is not touched) and stores the
// inverses of its 16×16 diagonal tiles (row-major, 256 elements each) in
// LinvG for the solve that follows.  One workgroup.
template <typename T>
__global__ __launch_bounds__(kPanelThreads, 2) void chol_factor_kernel(int nb, T *__restrict__ A,
                                                                    int64_t lda, int *info,
                                                                    int64_t info_base,
                                                                    T *__restrict__ LinvG, int fresh)
{
    __builtin_amdgcn_s_setprio(3);
    __shared__ T Xb[kFactorX];
    __shared__ T Db[256];
    __shared__ T Lib[kFactorLi];
    if (fresh && threadIdx.x == 0) *info = 0;   // (by the lane that records a pivot)
    switch (threadIdx.x >> 6) {
    case 0: factor_body<T, 0>(nb, A, lda, A, lda, info, info_base, LinvG, Xb, Db, Lib); break;
    case 1: factor_body<T, 1>(nb, A, lda, A, lda, info, info_base, LinvG, Xb, Db, Lib); break;
    case 2: factor_body<T, 2>(nb, A, lda, A, lda, info, info_base, LinvG, Xb, Db, Lib); break;
    default: factor_body<T, 3>(nb, A, lda, A, lda, info, info_base, LinvG, Xb, Db, Lib); break;
    }
}

// ---------------------------------------------------------------- LDLᴴ --
// _ldlt_lower! (src/ldlt.jl:16-33) of a 16×16 tile in row layout, column C:
// δ = a_CC (broadcast from lane C), l_i = a_iC / δ (:21), then
// a_ij −= l_i (l_j δ) for C < j ≤ i (:24-26).  Lane C keeps δ on the
// diagonal, rows below take l; entries right of the diagonal are left
// meaningless (cleared by the caller).  dv[C] receives δ.  A zero pivot
// divides by zero and the Inf/NaN propagate, as in the reference.
template <int C, int J, typename T>
struct LdltColUpdate {
    static __device__ __forceinline__ void run(T a[16], T l, T ld)
    {
        a[J] = fma_t(-l, row_bcast<J>(ld), a[J]);
        LdltColUpdate<C, J + 1, T>::run(a, l, ld);
    }
};
template <int C, typename T>
struct LdltColUpdate<C, 16, T> {
    static __device__ __forceinline__ void run(T *, T, T) {}
};
template <int C, typename T>
struct LdltTileCols {
    static __device__ __forceinline__ void run(T a[16], T dv[16], int i)
    {
        const T d = row_bcast<C>(a[C]);
        dv[C] = d;
        const T l = a[C] / d;
        const T ld = l * d;
        LdltColUpdate<C, C + 1, T>::run(a, l, ld);
        a[C] = i == C ? d : l;
        LdltTileCols<C + 1, T>::run(a, dv, i);
    }
};
template <typename T>
struct LdltTileCols<16, T> {
    static __device__ __forceinline__ void run(T *, T *, int) {}
};

// w <- L⁻¹ (four-column layout) for the unit lower tile L in row layout
// (li[k] = L[i][k] for k < i): forward elimination with unit pivots.
template <typename T>
__device__ __forceinline__ void tile_inverse_unit_rows(const T li[16], T w[4])
{
    const int lane = threadIdx.x & 63;
    const int i = lane & 15, g = lane >> 4;
    T m[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) m[k] = i > k ? li[k] : T(0);
#pragma unroll
    for (int t = 0; t < 4; ++t) w[t] = (i == g + 4 * t) ? T(1) : T(0);
    TileInvSteps<0, T>::run(m, w);
}

// Wave 0: LDLᴴ of diagonal tile j (d, transposed) in row layout through
// the wave's LDS tile D (LdltTileCols), the inverse of its unit factor to
// Li (row-major) and LinvG, the pivots to dv; d keeps δ on the diagonal and
// L below it (transposed).
template <typename T>
__device__ __forceinline__ void ldlt_diag_factor(typename PanelMfma<T>::acc_t &d, int j, T *D,
                                                 T *Li, T *dv, T *__restrict__ LinvG)
{
    typedef PanelMfma<T> M;
    const int lane = threadIdx.x & 63;
    const int lc = lane & 15;
    const int i = lane & 15, g = lane >> 4;
#pragma unroll
    for (int r = 0; r < 4; ++r) D[lc * kXLD + M::row(lane, r)] = d[r];
    wave_order();
    T a[16], w[4], dd[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) a[c] = c <= i ? D[i * kXLD + c] : T(0);
    LdltTileCols<0, T>::run(a, dd, i);
#pragma unroll
    for (int c = 0; c < 16; ++c) a[c] = c <= i ? a[c] : T(0);
    tile_inverse_unit_rows<T>(a, w);
    wave_order();
    if (g == 0)
#pragma unroll
        for (int c = 0; c < 16; ++c) D[i * kXLD + c] = a[c];
    if (lane < 16) {
        T dl = dd[0];   // the pivots are the same in every lane: lane c stores δ_c
#pragma unroll
        for (int c = 1; c < 16; ++c) dl = lane == c ? dd[c] : dl;
        dv[lane] = dl;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        Li[i * kXLD + g + 4 * t] = w[t];
        if (LinvG) LinvG[j * 256 + i * 16 + g + 4 * t] = w[t];
    }
    wave_order();
#pragma unroll
    for (int r = 0; r < 4; ++r) d[r] = D[lc * kXLD + M::row(lane, r)];
}

// d (a diagonal tile, transposed) −= W_j L_jᵀ for tile row j of W (X) and
// of L (Y) in LDS
template <typename T>
__device__ __forceinline__ void ldlt_diag_update(typename PanelMfma<T>::acc_t &d, const T *X,
                                                 const T *Y, int j)
{
    typedef PanelMfma<T> M;
    const int lane = threadIdx.x & 63;
    const int lc = lane & 15;
#pragma unroll
    for (int kq = 0; kq < 4; ++kq) {
        const int kk = (lane >> 4) + 4 * kq;
        d = M::mma(-Y[(j * 16 + lc) * kXLD + kk], X[(j * 16 + lc) * kXLD + kk], d);
    }
}

// The LDLᴴ of the nb×nb (nb ≤ 128) diagonal block at A, with the tiles held
// as in factor_body (transposed; wave 0 the diagonal tiles, waves 1–3 the
// rest) and the same two-barrier step: (A) waves 1–3 form W = A L_kk⁻ᵀ
// (rdiv! by UnitLowerTriangular, src/ldlt.jl:86) and L = W D_kk⁻¹ (rdiv! by
// Diagonal, :87, a division) for their panel tiles while wave 0 applies the
// previous step's update to the diagonal tiles beyond kb + 1; (B) wave 0
// updates diagonal tile kb + 1, factors it (LdltTileCols) and inverts its
// unit factor while waves 1–3 apply C −= W Lᵀ (:88-95) on MFMA.  Writes D
// on the diagonal and L below it, and the inverses of the unit 16×16
// diagonal tiles (row-major, 256 elements each) to LinvG.
template <typename T, int W>
__device__ __forceinline__ void ldlt_body(int nb, T *__restrict__ A, int64_t lda,
                                          T *__restrict__ LinvG, T *Xb, T *Yb, T *Db, T *Lib,
                                          T *dvs)
{
    typedef PanelMfma<T> M;
    typedef typename M::acc_t acc_t;
    constexpr int NQ = W == 0 ? 8 : 10;
    constexpr int NBLK = kPanelNB / 16;
    constexpr int XS = kPanelNB * kXLD, LS = 16 * kXLD;
    const int lane = threadIdx.x & 63;
    const int lc = lane & 15;
    const int nkb = (nb + 15) / 16;

    acc_t acc[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int bi = dslot_bi<W>(q), bj = dslot_bj<W>(q);
        if (bi < 0) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int gi = bi * 16 + lc, gj = bj * 16 + M::row(lane, r);
            T v = T(0);
            if (gj <= gi) v = gi < nb ? A[gi + (int64_t)gj * lda] : (gi == gj ? T(1) : T(0));
            acc[q][r] = v;
        }
    }
    if constexpr (W == 0) ldlt_diag_factor<T>(acc[0], 0, Db, Lib, dvs, LinvG);
    __syncthreads();
#pragma unroll
    for (int kb = 0; kb < NBLK; ++kb) {
        if (kb >= nkb) break;
        T *X = Xb + (kb & 1) * XS;   // W of column block kb
        T *Y = Yb + (kb & 1) * XS;   // L of column block kb
        // (A)
        if constexpr (W == 0) {
            if (kb > 0) {
                const T *Xp = Xb + ((kb - 1) & 1) * XS, *Yp = Yb + ((kb - 1) & 1) * XS;
#pragma unroll
                for (int j = kb + 1; j < NBLK; ++j) {
                    if (j >= nkb) break;
                    ldlt_diag_update<T>(acc[j], Xp, Yp, j);
                }
            }
        } else {
            const T *Lik = Lib + (kb & 1) * LS;
            const T *dv = dvs + (kb & 1) * 16;
            T dcol[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) dcol[r] = dv[M::row(lane, r)];
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const int bi = dslot_bi<W>(q), bj = dslot_bj<W>(q);
                if (bi < 0 || bj != kb) continue;
                if (bi >= nkb) continue;
                acc_t x = {T(0), T(0), T(0), T(0)};
#pragma unroll
                for (int kq = 0; kq < 4; ++kq)
                    x = M::mma(Lik[lc * kXLD + M::row(lane, kq)], acc[q][kq], x);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    acc[q][r] = x[r] / dcol[r];
                    X[(bi * 16 + lc) * kXLD + M::row(lane, r)] = x[r];
                    Y[(bi * 16 + lc) * kXLD + M::row(lane, r)] = acc[q][r];
                }
            }
        }
        __syncthreads();
        // (B)
        if constexpr (W == 0) {
            if (kb + 1 < nkb) {
                ldlt_diag_update<T>(acc[kb + 1], X, Y, kb + 1);
                ldlt_diag_factor<T>(acc[kb + 1], kb + 1, Db, Lib + ((kb + 1) & 1) * LS,
                                    dvs + ((kb + 1) & 1) * 16, LinvG);
            }
        } else {
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const int bi = dslot_bi<W>(q), bj = dslot_bj<W>(q);
                if (bi < 0 || bj <= kb) continue;
                if (bi >= nkb) continue;
#pragma unroll
                for (int kq = 0; kq < 4; ++kq) {
                    const int kk = (lane >> 4) + 4 * kq;
                    const T a = -Y[(bj * 16 + lc) * kXLD + kk];
                    const T b = X[(bi * 16 + lc) * kXLD + kk];
                    acc[q] = M::mma(a, b, acc[q]);
                }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int bi = dslot_bi<W>(q), bj = dslot_bj<W>(q);
        if (bi < 0) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int gi = bi * 16 + lc, gj = bj * 16 + M::row(lane, r);
            if (gi < nb && gj <= gi) A[gi + (int64_t)gj * lda] = acc[q][r];
        }
    }
}

template <typename T>
__global__ __launch_bounds__(kPanelThreads) void ldlt_tile_factor_kernel(int nb, T *__restrict__ A,
                                                                         int64_t lda,
                                                                         T *__restrict__ LinvG)
{
    __shared__ T Xb[2 * kPanelNB * kXLD];
    __shared__ T Yb[2 * kPanelNB * kXLD];
    __shared__ T Db[2 * 16 * kXLD];
    __shared__ T Lib[2 * 16 * kXLD];
    __shared__ T dvs[2 * 16];
    switch (threadIdx.x >> 6) {
    case 0: ldlt_body<T, 0>(nb, A, lda, LinvG, Xb, Yb, Db, Lib, dvs); break;
    case 1: ldlt_body<T, 1>(nb, A, lda, LinvG, Xb, Yb, Db, Lib, dvs); break;
    case 2: ldlt_body<T, 2>(nb, A, lda, LinvG, Xb, Yb, Db, Lib, dvs); break;
    default: ldlt_body<T, 3>(nb, A, lda, LinvG, Xb, Yb, Db, Lib, dvs); break;
    }
}

// The same for a block that an earlier kernel has classified through
// flags: flags[0] != 0 — nothing to do (the caller's path failed);
// flags[1] == 0 — A = I + E with ‖E‖_F ≤ 0.1·√eps, whose factor is
// L = I + Φ(E), Φ(E) = the strictly lower part of E plus half its diagonal,
// since (I + F)(I + F)ᵀ = I + E gives F = Φ(E − F Fᵀ) and ‖F Fᵀ‖ ≤ ‖E‖² ≤
// 0.01·eps, below the rounding of any entry; likewise the 16×16 tile
// inverses (I + F_tt)⁻¹ = I − F_tt; otherwise the full factorisation.
template <typename T>
__global__ __launch_bounds__(kPanelThreads, 2) void chol_factor_near_identity_kernel(
    int nb, T *__restrict__ A, int64_t lda, int *info, int64_t info_base, T *__restrict__ LinvG,
    const int *flags)
{
    __builtin_amdgcn_s_setprio(3);
    __shared__ T Xb[kFactorX];
    __shared__ T Db[256];
    __shared__ T Lib[kFactorLi];
    if (flags[0] != 0) return;
    if (flags[1] == 0) {
        const int nt = (nb + 15) / 16;
        for (int e = threadIdx.x; e < nt * 256; e += kPanelThreads) {
            const int t = e >> 8, i = (e >> 4) & 15, j = e & 15;
            const int gi = 16 * t + i, gj = 16 * t + j;
            T v;
            if (gi >= nb || gj >= nb) v = gi == gj ? T(1) : T(0);
            else if (gi == gj) v = T(1) - (A[gi + (int64_t)gi * lda] - T(1)) * T(0.5);
            else v = gi > gj ? -A[gi + (int64_t)gj * lda] : T(0);
            LinvG[e] = v;
        }
        __syncthreads();
        for (int e = threadIdx.x; e < nb; e += kPanelThreads)
            A[e + (int64_t)e * lda] = T(1) + (A[e + (int64_t)e * lda] - T(1)) * T(0.5);
        return;
    }
    switch (threadIdx.x >> 6) {
    case 0: factor_body<T, 0>(nb, A, lda, A, lda, info, info_base, LinvG, Xb, Db, Lib); break;
    case 1: factor_body<T, 1>(nb, A, lda, A, lda, info, info_base, LinvG, Xb, Db, Lib); break;
    case 2: factor_body<T, 2>(nb, A, lda, A, lda, info, info_base, LinvG, Xb, Db, Lib); break;
    default: factor_body<T, 3>(nb, A, lda, A, lda, info, info_base, LinvG, Xb, Db, Lib); break;
    }
}

// The same factorisation of an FP32 diagonal block computed in FP64: the
// block is read and written back in FP32, the tile inverses are stored in
// FP32 (Linv32).
__global__ __launch_bounds__(kPanelThreads, 2) void chol_factor_f32io_kernel(int nb,
                                                                          float *__restrict__ A,
                                                                          int64_t lda, int *info,
                                                                          int64_t info_base,
                                                                          float *__restrict__ Linv32)
{
    __shared__ double Xb[kFactorX];
    __shared__ double Db[256];
    __shared__ double Lib[kFactorLi];
    switch (threadIdx.x >> 6) {
    case 0: factor_body<double, 0, float>(nb, A, lda, A, lda, info, info_base, nullptr, Xb, Db, Lib, Linv32); break;
    case 1: factor_body<double, 1, float>(nb, A, lda, A, lda, info, info_base, nullptr, Xb, Db, Lib, Linv32); break;
    case 2: factor_body<double, 2, float>(nb, A, lda, A, lda, info, info_base, nullptr, Xb, Db, Lib, Linv32); break;
    default: factor_body<double, 3, float>(nb, A, lda, A, lda, info, info_base, nullptr, Xb, Db, Lib, Linv32); break;
    }
}

// A strided batch of diagonal-block factorisations (nb ≤ 128 each), one
// workgroup per matrix: matrix b at A + b·sA, its factor at D + b·sD,
// its first failing pivot in info[b] (info zeroed by the caller).
template <typename T>
__global__ __launch_bounds__(kPanelThreads, 2) void chol_factor_batched_kernel(
    int nb, const T *A, int64_t lda, int64_t sA, T *D, int64_t ldd, int64_t sD, int *info)
{
    __shared__ T Xb[kFactorX];
    __shared__ T Db[256];
    __shared__ T Lib[kFactorLi];
    const int64_t b = blockIdx.x;
    const T *Ab = A + b * sA;
    T *Lb = D + b * sD;
    int *ib = info + b;
    switch (threadIdx.x >> 6) {
    case 0: factor_body<T, 0>(nb, Ab, lda, Lb, ldd, ib, 0, nullptr, Xb, Db, Lib); break;
    case 1: factor_body<T, 1>(nb, Ab, lda, Lb, ldd, ib, 0, nullptr, Xb, Db, Lib); break;
    case 2: factor_body<T, 2>(nb, Ab, lda, Lb, ldd, ib, 0, nullptr, Xb, Db, Lib); break;
    default: factor_body<T, 3>(nb, Ab, lda, Lb, ldd, ib, 0, nullptr, Xb, Db, Lib); break;
    }
}

// Inverses of the 16×16 diagonal tiles of a lower n×n L (tiles past n are
// padded with the identity); one wave per tile.
template <typename T>
__global__ __launch_bounds__(256) void tile_inverse_kernel(int64_t n, const T *__restrict__ L,
                                                           int64_t ldl, T *__restrict__ LinvG)
{
    const int64_t tile = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (tile * 16 >= n) return;
    const int lane = threadIdx.x & 63;
    const int i = lane & 15, g = lane >> 4;
    T v[4], w[4], rd[16];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int j = g + 4 * t;
        const int64_t gi = tile * 16 + i, gj = tile * 16 + j;
        v[t] = (j <= i) ? (gi < n ? L[gi + gj * ldl] : (i == j ? T(1) : T(0))) : T(0);
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) rd[k] = T(1) / __shfl(v[k >> 2], k + 16 * (k & 3));
    tile_inverse<T>(v, rd, w);
#pragma unroll
    for (int t = 0; t < 4; ++t) LinvG[tile * 256 + i * 16 + g + 4 * t] = w[t];
}

// Tile q of the strictly-lower tiles (bj, kb), bj > kb, of an 8×8-tile
// block, stored column block after column block: its kb and bj.
__host__ __device__ constexpr int lt_kb(int q)
{
    int kb = 0, base = 0;
    while (base + (7 - kb) <= q) {
        base += 7 - kb;
        ++kb;
    }
    return kb;
}
__host__ __device__ constexpr int lt_bj(int q)
{
    int kb = 0, base = 0;
    while (base + (7 - kb) <= q) {
        base += 7 - kb;
        ++kb;
    }
    return kb + 1 + (q - base);
}

// Index of tile (bj, kb), bj > kb, in Lt: column blocks stored one after
// another.
__device__ __forceinline__ int lt_index(int bj, int kb) { return 7 * kb - kb * (kb - 1) / 2 + (bj - kb - 1); }

// Stages the strictly-lower 16×16 tiles of the nb×nb (nb ≤ 128) lower L and
// the inverses of its diagonal tiles into LDS (row-major tiles, padded rows),
// all loads issued before the first store.  L is read with 16 consecutive
// rows of one column per 16 lanes (thread t: row t % 16, column t / 16 % 16
// of every tile), the inverses as stored (row-major, 256 per tile).
template <typename T>
__device__ __forceinline__ void stage_l_tiles(int nb, const T *__restrict__ L, int64_t ldl,
                                              const T *__restrict__ LinvG, T *Lt, T *Li)
{
    constexpr int NBLK = kPanelNB / 16;
    constexpr int NLT = NBLK * (NBLK - 1) / 2;
    constexpr int TS = 16 * kXLD;
    static_assert(kPanelThreads == 256, "one tile element per thread");
    const int nkb = (nb + 15) / 16;
    const int ri = threadIdx.x & 15, rj = (threadIdx.x >> 4) & 15;
    const int i = (threadIdx.x >> 4) & 15, j = threadIdx.x & 15;
    // unconditional loads from clamped indices, so that all of them stay in
    // flight; out-of-range values replaced afterwards
    T lv[NLT], iv[NBLK];
#pragma unroll
    for (int q = 0; q < NLT; ++q) {
        const int kb = lt_kb(q), bj = lt_bj(q);
        const int gi = bj * 16 + ri, gj = kb * 16 + rj;
        const int gic = gi < nb ? gi : nb - 1, gjc = gj < nb ? gj : nb - 1;
        lv[q] = L[gic + (int64_t)gjc * ldl];
    }
#pragma unroll
    for (int q = 0; q < NBLK; ++q) iv[q] = LinvG[(q < nkb ? q : nkb - 1) * 256 + threadIdx.x];
#pragma unroll
    for (int q = 0; q < NLT; ++q) hold(lv[q]);
#pragma unroll
    for (int q = 0; q < NBLK; ++q) hold(iv[q]);
#pragma unroll
    for (int q = 0; q < NLT; ++q) {
        const bool in = lt_bj(q) * 16 + ri < nb && lt_kb(q) * 16 + rj < nb;
        Lt[q * TS + ri * kXLD + rj] = in ? lv[q] : T(0);
    }
#pragma unroll
    for (int q = 0; q < NBLK; ++q) Li[q * TS + i * kXLD + j] = q < nkb ? iv[q] : T(0);
}

// acc (this wave's 16 rows × 128 columns as eight 16×16 tiles, each held
// TRANSPOSED: acc[bj] = B_bjᵀ in accumulator layout) <- acc L⁻ᵀ with L's
// tiles and tile inverses staged in LDS.  The accumulator layout of Bᵀ is
// the MFMA's B-operand layout with K index row(lane, kq) in step kq, so for
// each column block kb the wave forms X_kbᵀ = L_kk⁻¹ B_kbᵀ and updates
// B_jᵀ -= L_(j,kb) X_kbᵀ (j > kb) with the B operands straight from
// registers and only L read from LDS: no LDS round trip and no barrier
// (every wave touches only its own rows).  The column-block loop is
// unrolled, so every tile index is static.
template <typename T, bool FULL>
__device__ __forceinline__ void solve_tiles_of(int nkb, typename PanelMfma<T>::acc_t acc[8],
                                               const T *Lt, const T *Li)
{
    typedef PanelMfma<T> M;
    typedef typename M::acc_t acc_t;
    constexpr int NBLK = kPanelNB / 16;
    constexpr int TS = 16 * kXLD;
    const int lane = threadIdx.x & 63;
    const int lc = lane & 15;
#pragma unroll
    for (int kb = 0; kb < NBLK; ++kb) {
        if (!FULL && kb >= nkb) break;
        const T *Lik = Li + kb * TS;
        acc_t x = {T(0), T(0), T(0), T(0)};
#pragma unroll
        for (int kq = 0; kq < 4; ++kq)
            x = M::mma(Lik[lc * kXLD + M::row(lane, kq)], acc[kb][kq], x);
        acc[kb] = x;
        T nx[4];
#pragma unroll
        for (int kq = 0; kq < 4; ++kq) nx[kq] = -x[kq];
#pragma unroll
        for (int bj = kb + 1; bj < NBLK; ++bj) {
            if (!FULL && bj >= nkb) break;
            const T *Lt_jk = Lt + lt_index(bj, kb) * TS;
#pragma unroll
            for (int kq = 0; kq < 4; ++kq)
                acc[bj] = M::mma(Lt_jk[lc * kXLD + M::row(lane, kq)], nx[kq], acc[bj]);
        }
    }
}
// (a full block without branches, so that L's reads run ahead of their use)
template <typename T>
__device__ __forceinline__ void solve_tiles(int nkb, typename PanelMfma<T>::acc_t acc[8],
                                            const T *Lt, const T *Li)
{
    if (nkb == kPanelNB / 16)
        solve_tiles_of<T, true>(nkb, acc, Lt, Li);
    else
        solve_tiles_of<T, false>(nkb, acc, Lt, Li);
}

// B (nrows×nb) <- B L⁻ᵀ for the lower nb×nb L (nb ≤ 128) whose 16×16
// diagonal-tile inverses are in LinvG — rdiv!(A21, LowerTriangular(A11)'),
// src/cholesky.jl:28,48.  Each workgroup takes 64 rows; wave w holds tile
// row w of them (8 tiles).  L's 28 strictly-lower tiles and the 8 inverses
// are read into LDS once, then solve_tiles runs the column sweep.  Bound by
// the sweep, 36 tile products a wave (FP64 4 µs), between two memory round
// trips: 1501×128 FP64 12 µs (22 with the loads under branches, one round trip
// after another, and a branch per tile in the sweep).
template <typename T>
__global__ __launch_bounds__(kPanelThreads) void chol_solve_kernel(int nb, const T *__restrict__ L,
                                                                   int64_t ldl,
                                                                   const T *__restrict__ LinvG,
                                                                   T *__restrict__ B, int64_t ldb,
                                                                   int64_t nrows)
{
    __builtin_amdgcn_s_setprio(3);
    typedef PanelMfma<T> M;
    typedef typename M::acc_t acc_t;
    constexpr int NBLK = kPanelNB / 16;             // 8
    constexpr int NLT = NBLK * (NBLK - 1) / 2;       // 28 strictly-lower tiles
    constexpr int TS = 16 * kXLD;                    // one padded tile
    __shared__ T Lt[NLT * TS];                       // tile (bj, kb), bj > kb
    __shared__ T Li[NBLK * TS];                      // inverses of the diagonal tiles
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    const int lc = lane & 15;
    const int64_t row0 = (int64_t)blockIdx.x * kPanelRB;
    const int nkb = (nb + 15) / 16;

    // the wave's rows, tiles transposed (lane: row lc, columns row(lane, r)),
    // loaded first so that their latency overlaps L's
    acc_t acc[NBLK];
    const int64_t gr = row0 + w * 16 + lc;
    const int64_t grc = gr < nrows ? gr : nrows - 1;
#pragma unroll
    for (int bj = 0; bj < NBLK; ++bj)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int gj = bj * 16 + M::row(lane, r);
            const int gjc = gj < nb ? gj : nb - 1;
            acc[bj][r] = B[grc + (int64_t)gjc * ldb];
        }
    stage_l_tiles<T>(nb, L, ldl, LinvG, Lt, Li);
#pragma unroll
    for (int bj = 0; bj < NBLK; ++bj)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            T v = acc[bj][r];
            hold(v);
            acc[bj][r] = (gr < nrows && bj * 16 + M::row(lane, r) < nb) ? v : T(0);
        }
    __syncthreads();
    solve_tiles<T>(nkb, acc, Lt, Li);
#pragma unroll
    for (int bj = 0; bj < NBLK; ++bj)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int gj = bj * 16 + M::row(lane, r);
            if (gr < nrows && gj < nb) B[gr + (int64_t)gj * ldb] = acc[bj][r];
        }
}

// B (nrows×nb) <- B L⁻ᵀ for a wide lower L (nb a multiple of 128, up to
// kPsolveMaxNB), already factored, with its 16×16 diagonal-tile inverses in
// LinvG: rdiv!(A21, LowerTriangular(A11)') (src/cholesky.jl:28) of a whole
// look-ahead panel in one launch.  Each workgroup takes 64 rows and sweeps
// the 128-wide column blocks left to right: block c first takes the
// products of the blocks already solved, B_c -= Σ_{c'<c} X_c' L(c,c')ᵀ, as
// one MFMA product over K = 128c with operands staged through LDS in
// 32-wide slabs, then X_c = B_c L_cc⁻ᵀ by solve_tiles.  A workgroup reads
// only L and its own rows, so no workgroup waits for another.
constexpr int kPsolveMaxNB = 768;   // wider panels: the recursive solve is faster
constexpr int kPsolveKC = 32;                 // K slab of the product
constexpr int kPsolveGLD = kPsolveKC + 1;     // padded LDS row
template <typename T>
__global__ __launch_bounds__(kPanelThreads) void chol_psolve_kernel(int nb, const T *__restrict__ L,
                                                                    int64_t ldl,
                                                                    const T *__restrict__ LinvG,
                                                                    T *__restrict__ B, int64_t ldb,
                                                                    int64_t nrows)
{
    typedef PanelMfma<T> M;
    typedef typename M::acc_t acc_t;
    constexpr int NBLK = kPanelNB / 16;
    constexpr int NLT = NBLK * (NBLK - 1) / 2;
    constexpr int TS = 16 * kXLD;
    __shared__ T Lt[NLT * TS];
    __shared__ T Li[NBLK * TS];
    __shared__ T Gx[kPanelRB * kPsolveGLD];   // this workgroup's solved rows, one K slab
    __shared__ T Gl[kPanelNB * kPsolveGLD];   // rows of block c of L, the same K slab
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    const int lc = lane & 15;
    const int64_t row0 = (int64_t)blockIdx.x * kPanelRB;
    const int64_t gr = row0 + w * 16 + lc;   // this lane's row in every tile
    const int nc = nb / kPanelNB;
    for (int c = 0; c < nc; ++c) {
        // block c of the wave's rows, tiles transposed as solve_tiles takes them
        acc_t acc[NBLK];
#pragma unroll
        for (int bj = 0; bj < NBLK; ++bj)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t gj = (int64_t)c * kPanelNB + bj * 16 + M::row(lane, r);
                acc[bj][r] = gr < nrows ? B[gr + gj * ldb] : T(0);
            }
        // B_cᵀ -= L[128c : 128c+128, 0:128c] X[:, 0:128c]ᵀ, the global loads
        // of slab s + 1 in flight while slab s is multiplied
        const T *Lc = L + (int64_t)c * kPanelNB;
        constexpr int XE = kPanelRB * kPsolveKC / kPanelThreads;   // 8 per thread
        constexpr int LE = kPanelNB * kPsolveKC / kPanelThreads;   // 16 per thread
        const int kend = c * kPanelNB;
        T xv[XE], lv[LE];
        auto fetch = [&](int k0) {
#pragma unroll
            for (int e = 0; e < XE; ++e) {
                const int idx = threadIdx.x + e * kPanelThreads;
                const int i = idx % kPanelRB, kk = idx / kPanelRB;
                xv[e] = row0 + i < nrows ? B[row0 + i + (int64_t)(k0 + kk) * ldb] : T(0);
            }
#pragma unroll
            for (int e = 0; e < LE; ++e) {
                const int idx = threadIdx.x + e * kPanelThreads;
                const int i = idx % kPanelNB, kk = idx / kPanelNB;
                lv[e] = Lc[i + (int64_t)(k0 + kk) * ldl];
            }
        };
        // block c − 1 was stored by other waves at the end of the last sweep
        __syncthreads();
        if (kend > 0) fetch(0);
        for (int k0 = 0; k0 < kend; k0 += kPsolveKC) {
            __syncthreads();   // the previous slab has been read
#pragma unroll
            for (int e = 0; e < XE; ++e) {
                const int idx = threadIdx.x + e * kPanelThreads;
                Gx[(idx % kPanelRB) * kPsolveGLD + idx / kPanelRB] = xv[e];
            }
#pragma unroll
            for (int e = 0; e < LE; ++e) {
                const int idx = threadIdx.x + e * kPanelThreads;
                Gl[(idx % kPanelNB) * kPsolveGLD + idx / kPanelNB] = lv[e];
            }
            __syncthreads();
            if (k0 + kPsolveKC < kend) fetch(k0 + kPsolveKC);
#pragma unroll
            for (int kq = 0; kq < kPsolveKC / 4; ++kq) {
                const int kk = 4 * kq + (lane >> 4);
                const T xb = -Gx[(w * 16 + lc) * kPsolveGLD + kk];
#pragma unroll
                for (int bj = 0; bj < NBLK; ++bj)
                    acc[bj] = M::mma(Gl[(bj * 16 + lc) * kPsolveGLD + kk], xb, acc[bj]);
            }
        }
        // X_c = B_c L_cc⁻ᵀ
        __syncthreads();   // Lt/Li of the previous block have been read
        stage_l_tiles<T>(kPanelNB, L + (int64_t)c * kPanelNB * (1 + ldl), ldl,
                         LinvG + (int64_t)c * NBLK * 256, Lt, Li);
        __syncthreads();
        solve_tiles<T>(NBLK, acc, Lt, Li);
#pragma unroll
        for (int bj = 0; bj < NBLK; ++bj)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t gj = (int64_t)c * kPanelNB + bj * 16 + M::row(lane, r);
                if (gr < nrows) B[gr + gj * ldb] = acc[bj][r];
            }
        // the stores of block c are read back by this workgroup's later
        // slabs (workgroup-scope visibility at the barrier that opens them)
    }
}

// Swaps the strict upper and strict lower triangles of an n×n matrix, in
// place (A <- Aᵀ off the diagonal).  Used for the Val{:U} convention.  One
// workgroup per pair of mirrored 64×64 tiles, both transposed through LDS, so
// that memory is read and written down its columns.  Bound: memory.  n = 5001
// FP32: 47 µs; 95 with the mirrored element read and written across the rows.
constexpr int kSwT = 64;
template <typename T>
__global__ __launch_bounds__(256) void swap_triangles_kernel(int64_t n, T *A, int64_t lda)
{
    __shared__ T lo[kSwT][kSwT + 1], up[kSwT][kSwT + 1];   // [column][row]
    const int64_t i0 = (int64_t)blockIdx.x * kSwT, j0 = (int64_t)blockIdx.y * kSwT;
    if (i0 < j0) return;
    const int r = threadIdx.x & 63, w = threadIdx.x >> 6;
    T a[16], b[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int c = w + 4 * u;
        const int64_t li = i0 + r < n ? i0 + r : n - 1, lj = j0 + c < n ? j0 + c : n - 1;
        const int64_t ui = j0 + r < n ? j0 + r : n - 1, uj = i0 + c < n ? i0 + c : n - 1;
        a[u] = A[li + lj * lda];
        b[u] = A[ui + uj * lda];
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        lo[w + 4 * u][r] = a[u];
        up[w + 4 * u][r] = b[u];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int c = w + 4 * u;
        // strictly lower (i0 + r, j0 + c), and strictly upper (j0 + r, i0 + c)
        if (i0 + r < n && i0 + r > j0 + c) A[i0 + r + (j0 + c) * lda] = up[r][c];
        if (i0 + c < n && j0 + r < i0 + c) A[j0 + r + (i0 + c) * lda] = lo[r][c];
    }
}

template <typename T>
int launch_factor(hipStream_t s, int nb, T *A, int64_t lda, int *info, int64_t info_base,
                  T *LinvG, int fresh = 0)
{
    hipLaunchKernelGGL((chol_factor_kernel<T>), dim3(1), dim3(kPanelThreads), 0, s, nb, A, lda,
                       info, info_base, LinvG, fresh);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}

template <typename T>
int launch_solve(hipStream_t s, int nb, const T *L, int64_t ldl, const T *LinvG, T *B,
                 int64_t ldb, int64_t nrows)
{
    if (nrows <= 0 || nb <= 0) return GLA_OK;
    hipLaunchKernelGGL((chol_solve_kernel<T>), dim3((unsigned)cdiv(nrows, kPanelRB)),
                       dim3(kPanelThreads), 0, s, nb, L, ldl, LinvG, B, ldb, nrows);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}

template <typename T>
int launch_psolve(hipStream_t s, int nb, const T *L, int64_t ldl, const T *LinvG, T *B,
                  int64_t ldb, int64_t nrows)
{
    if (nrows <= 0) return GLA_OK;
    hipLaunchKernelGGL((chol_psolve_kernel<T>), dim3((unsigned)cdiv(nrows, kPanelRB)),
                       dim3(kPanelThreads), 0, s, nb, L, ldl, LinvG, B, ldb, nrows);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}

template <typename T>
int launch_tile_inverse(hipStream_t s, int64_t n, const T *L, int64_t ldl, T *LinvG)
{
    if (n <= 0) return GLA_OK;
    hipLaunchKernelGGL((tile_inverse_kernel<T>), dim3((unsigned)cdiv(cdiv(n, 16), 4)), dim3(256),
                       0, s, n, L, ldl, LinvG);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}

// Elements of the per-call workspace: the 16×16 diagonal-tile inverses of
// one 128-wide panel (blocked driver) or of L11 (recursive rdiv!).
inline size_t linv_elems(int64_t n) { return (size_t)(cdiv(n, 16) + 8) * 256; }

// Right-looking blocked Cholesky of the lower triangle with look-ahead.
// keep_linv: every block's 16×16 tile inverses stay in Linv at the block's
// own offset (tile q of the whole matrix at q·256), for a solve that
// follows; otherwise each block reuses the start of Linv.
template <typename T>
int chol_blocked_dev(Handle *h, hipStream_t s, int64_t n, T *A, int64_t lda, int nb,
                     int64_t info_base, T *Linv, bool use_side = true, bool keep_linv = false)
{
    if (n <= 0) return GLA_OK;
    const int64_t nsteps = cdiv(n, nb);
    const bool overlap = use_side && nsteps > 2;
    if (overlap) {
        GLA_HIP_TRY(hipEventRecord(h->ev_fork, s));
        GLA_HIP_TRY(hipStreamWaitEvent(h->side, h->ev_fork, 0));
    }
    int64_t k = 0;
    for (int64_t step = 0; step < nsteps; ++step, k += nb) {
        const int kb = (int)std::min<int64_t>(nb, n - k);
        const int64_t below = n - k - kb;
        T *Akk = A + k + k * lda;
        T *A21 = Akk + kb;
        T *Lv = keep_linv ? Linv + (k / 16) * 256 : Linv;
        GLA_TRY(launch_factor<T>(s, kb, Akk, lda, h->dinfo, info_base + k, Lv));    // :25
        GLA_TRY(launch_solve<T>(s, kb, Akk, lda, Lv, A21, lda, below));             // :27-28
        if (below == 0) break;
        if (!overlap) {
            // :30-31 rankUpdate! of all of A22 in one launch: with nothing
            // beside it, splitting off the next block column only adds a
            // launch (same products, same order)
            GLA_TRY(gemm<T>(s, 'N', 'T', 1, below, below, kb, T(-1), A21, lda, A21, lda, T(1),
                            A21 + kb * lda, lda, 0));
            continue;
        }
        const int kb2 = (int)std::min<int64_t>(nb, below);
        const int64_t rest = below - kb2;
        if (overlap && rest > 0) GLA_HIP_TRY(hipEventRecord(h->ev_step[0], s));
        if (overlap && step > 0) GLA_HIP_TRY(hipStreamWaitEvent(s, h->ev_step[1], 0));
        // :30-31 rankUpdate! on the next block column first (look-ahead) ...
        GLA_TRY(gemm<T>(s, 'N', 'T', 1, below, kb2, kb, T(-1), A21, lda, A21, lda, T(1),
                        A21 + kb * lda, lda, 0));
        // ... and on the rest of A22 beside the next panels
        if (rest > 0) {
            hipStream_t us = overlap ? h->side : s;
            if (overlap) GLA_HIP_TRY(hipStreamWaitEvent(h->side, h->ev_step[0], 0));
            T *X2 = A21 + kb2;
            GLA_TRY(gemm<T>(us, 'N', 'T', 1, rest, rest, kb, T(-1), X2, lda, X2, lda, T(1),
                            X2 + (kb + kb2) * lda, lda, 0));
            if (overlap) GLA_HIP_TRY(hipEventRecord(h->ev_step[1], h->side));
        }
    }
    if (overlap) {
        GLA_HIP_TRY(hipEventRecord(h->ev_join, h->side));
        GLA_HIP_TRY(hipStreamWaitEvent(s, h->ev_join, 0));
    }
    return GLA_OK;
}

// B (m×n) <- B L⁻ᵀ, L n×n lower, already factored, with the inverses of its
// 16×16 diagonal tiles in Linv.  Recursive on L: two half solves and a GEMM.
template <typename T>
int trsm_rlt_dev(hipStream_t s, int64_t m, int64_t n, const T *L, int64_t ldl, const T *Linv,
                 T *B, int64_t ldb)
{
    if (m <= 0 || n <= 0) return GLA_OK;
    if (n <= kPanelNB) return launch_solve<T>(s, (int)n, L, ldl, Linv, B, ldb, m);
    // split at a multiple of the panel width
    int64_t n1 = ((n / 2) + kPanelNB - 1) / kPanelNB * kPanelNB;
    if (n1 >= n) n1 = n - kPanelNB;
    GLA_TRY(trsm_rlt_dev<T>(s, m, n1, L, ldl, Linv, B, ldb));
    // B2 -= X1 * L21ᵀ, L21 = L[n1:n, 0:n1]
    GLA_TRY(gemm<T>(s, 'N', 'T', 0, m, n - n1, n1, T(-1), B, ldb, L + n1, ldl, T(1),
                    B + n1 * ldb, ldb, 0));
    return trsm_rlt_dev<T>(s, m, n - n1, L + n1 + n1 * ldl, ldl, Linv + (n1 / 16) * 256,
                           B + n1 * ldb, ldb);
}

// Blocked right-looking Cholesky with wide blocks (NB > 128) and depth-1
// look-ahead — cholBlocked!'s loop (src/cholesky.jl:17-35) with the
// diagonal block factored by the 128-wide driver on the caller's stream,
// the panel solved in one chol_psolve_kernel launch (or the recursive
// rdiv!), the next block column updated on
// the caller's stream and the rest of the trailing rankUpdate! (K = NB, an
// efficient MFMA SYRK) on the side stream, where it overlaps the next
// diagonal factor and panel solve.
template <typename T>
int chol_la_dev(Handle *h, hipStream_t s0, int64_t n, T *A, int64_t lda, int NB,
                int64_t info_base, T *Linv, bool df = false)
{
    if (n <= 0) return GLA_OK;
    if (NB <= kPanelNB || n <= NB) return chol_blocked_dev<T>(h, s0, n, A, lda, kPanelNB, info_base, Linv);
    const int64_t nsteps = cdiv(n, NB);
    const bool overlap = nsteps > 2;
    // df: each block column in one dataflow launch, which fills the chip, so
    // the SYRK beside it runs on every CU (n = 16384 FP64, 2048-wide: 28.3
    // ms; with 32 CUs kept from the SYRK 29.3 ms).
    // Else, with CUs reserved from the SYRK, the chain runs on an internal stream
    // with every CU and the SYRK on the masked one, both forked from (and
    // joined back to) the caller's stream.
    const bool masked = overlap && !df && h->masked != nullptr;
    hipStream_t s = masked ? h->chain : s0;
    hipStream_t side = masked ? h->masked : h->side;
    if (overlap) {
        GLA_HIP_TRY(hipEventRecord(h->ev_fork, s0));
        GLA_HIP_TRY(hipStreamWaitEvent(side, h->ev_fork, 0));
        if (masked) GLA_HIP_TRY(hipStreamWaitEvent(s, h->ev_fork, 0));
    }
    int64_t k = 0;
    for (int64_t step = 0; step < nsteps; ++step, k += NB) {
        const int64_t kb = std::min<int64_t>(NB, n - k);
        const int64_t below = n - k - kb;
        T *Akk = A + k + k * lda;
        T *A21 = Akk + kb;
        // :27-28 the diagonal block and rdiv! of the panel: one dataflow launch,
        // or the 128-wide driver and one launch over the panel when the block
        // is a whole number of 128-wide tiles, else the recursive solve
        const bool fused = h->chol_psolve != 0 && kb % kPanelNB == 0 && kb <= kPsolveMaxNB;
        if (df)
            GLA_TRY(chol_df<T>(h, s, n - k, kb, Akk, lda, info_base + k, nullptr));
        else
            GLA_TRY(chol_blocked_dev<T>(h, s, kb, Akk, lda, kPanelNB, info_base + k, Linv, false,
                                        fused));
        if (below == 0) break;
        if (!df && fused) {
            GLA_TRY(launch_psolve<T>(s, (int)kb, Akk, lda, Linv, A21, lda, below));
        } else if (!df) {
            GLA_TRY(launch_tile_inverse<T>(s, kb, Akk, lda, Linv));
            GLA_TRY(trsm_rlt_dev<T>(s, below, kb, Akk, lda, Linv, A21, lda));
        }
        const int64_t kb2 = std::min<int64_t>(NB, below);
        const int64_t rest = below - kb2;
        // the side stream's SYRK is released after the next-block-column
        // update (chol_syrk_late, default), which then runs without the
        // SYRK's workgroups crowding it, or right after the panel solve
        const bool late = h->chol_syrk_late != 0;
        if (overlap && rest > 0 && !late) GLA_HIP_TRY(hipEventRecord(h->ev_step[0], s));
        if (overlap && step > 0) GLA_HIP_TRY(hipStreamWaitEvent(s, h->ev_step[1], 0));
        GLA_TRY(gemm<T>(s, 'N', 'T', 1, below, kb2, kb, T(-1), A21, lda, A21, lda, T(1),
                        A21 + kb * lda, lda, 0));
        if (overlap && rest > 0 && late) GLA_HIP_TRY(hipEventRecord(h->ev_step[0], s));
        if (rest > 0) {
            hipStream_t us = overlap ? side : s;
            if (overlap) GLA_HIP_TRY(hipStreamWaitEvent(side, h->ev_step[0], 0));
            T *X2 = A21 + kb2;
            GLA_TRY(gemm<T>(us, 'N', 'T', 1, rest, rest, kb, T(-1), X2, lda, X2, lda, T(1),
                            X2 + (kb + kb2) * lda, lda, 0));
            if (overlap) GLA_HIP_TRY(hipEventRecord(h->ev_step[1], side));
        }
    }
    if (overlap) {
        GLA_HIP_TRY(hipEventRecord(h->ev_join, side));
        GLA_HIP_TRY(hipStreamWaitEvent(s0, h->ev_join, 0));
        if (masked) {
            GLA_HIP_TRY(hipEventRecord(h->ev_fork, s));
            GLA_HIP_TRY(hipStreamWaitEvent(s0, h->ev_fork, 0));
        }
    }
    return GLA_OK;
}

// cholRecursive! (src/cholesky.jl:37-55): halve until n <= leaf, then the
// blocked driver.
// use_side = false keeps every launch on the caller's stream (the leaves'
// look-ahead then runs in order: the same arithmetic, no side stream).
template <typename T>
int chol_recursive_dev(Handle *h, hipStream_t s, int64_t n, T *A, int64_t lda, int64_t leaf,
                       int64_t info_base, T *Linv, bool use_side = true)
{
    if (n <= leaf)
        return chol_blocked_dev<T>(h, s, n, A, lda, kPanelNB, info_base, Linv, use_side);
    int64_t n2 = n / 2;                                              // :44
    if (n2 > kPanelNB) n2 = n2 / kPanelNB * kPanelNB;                // keep blocks aligned
    GLA_TRY(chol_recursive_dev<T>(h, s, n2, A, lda, leaf, info_base, Linv, use_side));   // :46
    GLA_TRY(launch_tile_inverse<T>(s, n2, A, lda, Linv));            // :48 rdiv!
    GLA_TRY(trsm_rlt_dev<T>(s, n - n2, n2, A, lda, Linv, A + n2, lda));
    GLA_TRY(gemm<T>(s, 'N', 'T', 1, n - n2, n - n2, n2, T(-1), A + n2, lda, A + n2, lda, T(1),
                    A + n2 + n2 * lda, lda, 0));                     // :51 rankUpdate!
    return chol_recursive_dev<T>(h, s, n - n2, A + n2 + n2 * lda, lda, leaf,
                                 info_base + n2, Linv, use_side);    // :52
}

template <typename T>
int swap_triangles(hipStream_t s, int64_t n, T *A, int64_t lda)
{
    dim3 grid((unsigned)cdiv(n, kSwT), (unsigned)cdiv(n, kSwT));
    hipLaunchKernelGGL((swap_triangles_kernel<T>), grid, dim3(256), 0, s, n, A, lda);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}

}  // namespace

// Building blocks shared with the mixed-precision driver.
template <typename T>
int chol_factor_block(hipStream_t s, int nb, T *A, int64_t lda, int *info, int64_t info_base,
                      T *LinvG)
{
    return launch_factor<T>(s, nb, A, lda, info, info_base, LinvG);
}
template <typename T>
int ldlt_factor_block(hipStream_t s, int nb, T *A, int64_t lda, T *LinvG)
{
    hipLaunchKernelGGL((ldlt_tile_factor_kernel<T>), dim3(1), dim3(kPanelThreads), 0, s, nb, A,
                       lda, LinvG);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}
template <typename T>
int chol_factor_block_near_identity(hipStream_t s, int nb, T *A, int64_t lda, int *info,
                                    int64_t info_base, T *LinvG, const int *flags)
{
    hipLaunchKernelGGL((chol_factor_near_identity_kernel<T>), dim3(1), dim3(kPanelThreads), 0, s,
                       nb, A, lda, info, info_base, LinvG, flags);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}
int chol_factor_block_f32io(hipStream_t s, int nb, float *A, int64_t lda, int *info,
                            int64_t info_base, float *Linv32)
{
    hipLaunchKernelGGL(chol_factor_f32io_kernel, dim3(1), dim3(kPanelThreads), 0, s, nb, A, lda,
                       info, info_base, Linv32);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}
template <typename T>
int chol_solve_block(hipStream_t s, int nb, const T *L, int64_t ldl, const T *LinvG, T *B,
                     int64_t ldb, int64_t nrows)
{
    return launch_solve<T>(s, nb, L, ldl, LinvG, B, ldb, nrows);
}
template <typename T>
int tile_inverses(hipStream_t s, int64_t n, const T *L, int64_t ldl, T *LinvG)
{
    return launch_tile_inverse<T>(s, n, L, ldl, LinvG);
}
template <typename T>
int trsm_rlt(hipStream_t s, int64_t m, int64_t n, const T *L, int64_t ldl, const T *Linv, T *B,
             int64_t ldb)
{
    return trsm_rlt_dev<T>(s, m, n, L, ldl, Linv, B, ldb);
}
template <typename T>
int chol_factor_batched(hipStream_t s, int nb, const T *A, int64_t lda, int64_t sA, T *L,
                        int64_t ldl, int64_t sL, int *info, int64_t batch)
{
    if (batch <= 0 || nb <= 0) return GLA_OK;
    hipLaunchKernelGGL((chol_factor_batched_kernel<T>), dim3((unsigned)batch), dim3(kPanelThreads),
                       0, s, nb, A, lda, sA, L, ldl, sL, info);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}
size_t tile_inverse_elems(int64_t n) { return linv_elems(n); }

#define GLA_INST_BLOCKS(T)                                                                    \
    template int chol_factor_block<T>(hipStream_t, int, T *, int64_t, int *, int64_t, T *);  \
    template int ldlt_factor_block<T>(hipStream_t, int, T *, int64_t, T *);                  \
    template int chol_factor_block_near_identity<T>(hipStream_t, int, T *, int64_t, int *,   \
                                                    int64_t, T *, const int *);              \
    template int chol_solve_block<T>(hipStream_t, int, const T *, int64_t, const T *, T *,   \
                                     int64_t, int64_t);                                      \
    template int tile_inverses<T>(hipStream_t, int64_t, const T *, int64_t, T *);            \
    template int trsm_rlt<T>(hipStream_t, int64_t, int64_t, const T *, int64_t, const T *,   \
                             T *, int64_t); \
    template int chol_factor_batched<T>(hipStream_t, int, const T *, int64_t, int64_t, T *,   \
                                        int64_t, int64_t, int *, int64_t);

GLA_INST_BLOCKS(double)
GLA_INST_BLOCKS(float)
#undef GLA_INST_BLOCKS

// Driver of cholRecursive! for chol_block −1 (the default), from sweeps on
// MI355X (ms, copy of A included; FP64 | FP32):
//                                       n = 1000   5001       8192       12288      16384
//   whole matrix in one dataflow launch  0.21|0.18  1.52|0.99  4.72|2.48
//   look-ahead, 3072-wide dataflow                             4.81|2.87  12.9|7.33  28.4|15.9
//   look-ahead, 2048-wide dataflow                             4.89|2.99  13.3|7.55  27.6|15.5
//   a launch per 128-wide step           0.53|0.49  3.37|3.05  7.38|5.65  16.9|11.7  33.2|21.9
// so: one launch up to h->chol_df (8192: its packed tiles take 266 MB in
// FP64), then 3072-wide steps, then 2048.  Without the dataflow buffer
// (chol_df 0, or no memory for it) the step width is 0 (recursive halving)
// below 3072, then 256, 512 and 1024.
inline int64_t auto_chol_block(int64_t n, bool df)
{
    if (df) return n < 14336 ? 3072 : 2048;
    if (n < 3072) return 0;
    if (n < 10240) return 256;
    if (n < 14336) return 512;
    return 1024;
}

// algo: 0 unblocked, 1 blocked (param = blocksize), 2 recursive (param = cutoff)
template <typename T>
int chol_device(Handle *h, hipStream_t s, int64_t n, T *A, int64_t lda, int algo, int64_t param,
                T *Linv)
{
    if (n == 0) return GLA_OK;
    if (!Linv) {
        GLA_TRY(ensure_workspace(h, sizeof(T) * linv_elems(n)));
        Linv = reinterpret_cast<T *>(h->ws);
    }
    if (algo == 0) {
        // cholUnblocked!: one factor launch when the matrix fits the 128×128
        // block, otherwise the same column sweep blocked by 128.
        return chol_blocked_dev<T>(h, s, n, A, lda, kPanelNB, 0, Linv);
    }
    if (algo == 1) {
        int nb = (int)std::min<int64_t>(std::max<int64_t>(param, 1), kPanelNB);
        return chol_blocked_dev<T>(h, s, n, A, lda, nb, 0, Linv);
    }
    if (algo == 3) return chol_la_dev<T>(h, s, n, A, lda, (int)param, 0, Linv);
    // cholRecursive!: the reference recurses to 1×1 (cutoff does not reach
    // the A11 branch, :46); on the device the recursion stops at a leaf of
    // at least 2048 (or `cutoff` if larger) that the blocked driver factors.
    // (an order above a lowered chol_df that one block column would hold takes
    // the drivers without the buffer)
    bool df = false;
    if (h->chol_block < 0 && h->chol_df > 0 && n > kPanelNB) {
        const bool whole = n <= h->chol_df;
        const int64_t w = whole ? n : auto_chol_block(n, true);
        df = (whole || w < n) && ensure_df(h, s, chol_df_bytes(n, w, sizeof(T)));
        if (df && whole) return chol_df<T>(h, s, n, n, A, lda, 0, nullptr);
    }
    const int64_t NB = h->chol_block < 0 ? auto_chol_block(n, df) : h->chol_block;
    if (NB > kPanelNB) return chol_la_dev<T>(h, s, n, A, lda, (int)NB, 0, Linv, df);
    int64_t leaf = std::max<int64_t>(param, 2048);
    return chol_recursive_dev<T>(h, s, n, A, lda, leaf, 0, Linv);
}

template int chol_device<double>(Handle *, hipStream_t, int64_t, double *, int64_t, int, int64_t,
                                 double *);
template int chol_device<float>(Handle *, hipStream_t, int64_t, float *, int64_t, int, int64_t,
                                float *);

// ------------------------------------------------------------------ C ABI --
namespace {

template <typename T>
int chol_entry(gla_handle_t hh, char uplo, int64_t n, T *A, int64_t lda, int algo, int64_t param,
               int64_t *info, void *stream)
{
    Handle *h = reinterpret_cast<Handle *>(hh);
    if (!h) { set_error("null handle"); return -1; }
    if (uplo != 'L' && uplo != 'U' && uplo != 'l' && uplo != 'u') {
        set_error("uplo must be 'L' or 'U'");
        return -2;
    }
    if (n < 0) { set_error("n < 0"); return -3; }
    if (!A && n > 0) { set_error("A is null"); return -4; }
    if (lda < std::max<int64_t>(1, n)) { set_error("lda < max(1,n)"); return -5; }
    if (algo == 1 && param < 1) { set_error("blocksize < 1"); return -6; }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    GLA_HIP_TRY(hipSetDevice(h->device));
    // A matrix of one diagonal block is one launch, which also clears info
    // (n = 100 FP64, with the copy before and the read of info after it: 48.0 -> 46.0 µs).
    const bool one = n > 0 && n <= kPanelNB && (algo == 0 || algo == 2 || (algo == 1 && param >= n));
    if (!one) {
        hipLaunchKernelGGL(k_set_int, dim3(1), dim3(1), 0, s, h->dinfo, 0);
        GLA_LAUNCH_CHECK();
    }
    const bool upper = (uplo == 'U' || uplo == 'u');
    if (upper) GLA_TRY(swap_triangles<T>(s, n, A, lda));
    if (one)
        GLA_TRY(launch_factor<T>(s, (int)n, A, lda, h->dinfo, 0, nullptr, 1));
    else
        GLA_TRY(chol_device<T>(h, s, n, A, lda, algo, param));
    if (upper) GLA_TRY(swap_triangles<T>(s, n, A, lda));
    if (info) {
        int hv = 0;
        GLA_HIP_TRY(hipMemcpyAsync(&hv, h->dinfo, sizeof(int), hipMemcpyDeviceToHost, s));
        GLA_HIP_TRY(hipStreamSynchronize(s));
        if (hv < 0) {
            set_error("Cholesky: a device-side wait gave up after %u polls", h->spin_limit);
            return GLA_ERR_TIMEOUT;
        }
        *info = hv;
    }
    return GLA_OK;
}

template <typename T>
int rank_update_entry(gla_handle_t hh, char uplo, int64_t n, int64_t k, T alpha, const T *A,
                      int64_t lda, T *C, int64_t ldc, void *stream)
{
    Handle *h = reinterpret_cast<Handle *>(hh);
    if (!h) { set_error("null handle"); return -1; }
    if (uplo != 'L' && uplo != 'U') { set_error("uplo must be 'L' or 'U'"); return -2; }
    if (n < 0) return -3;
    if (k < 0) return -4;
    if (lda < std::max<int64_t>(1, n)) { set_error("lda < max(1,n)"); return -7; }
    if (ldc < std::max<int64_t>(1, n)) { set_error("ldc < max(1,n)"); return -9; }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    GLA_HIP_TRY(hipSetDevice(h->device));
    if (uplo == 'L') return gemm<T>(s, 'N', 'T', 1, n, n, k, alpha, A, lda, A, lda, T(1), C, ldc, 0);
    return gemm<T>(s, 'N', 'T', 2, n, n, k, alpha, A, lda, A, lda, T(1), C, ldc, 0);
}

template <typename T>
int trsm_entry(gla_handle_t hh, int64_t m, int64_t n, const T *L, int64_t ldl, T *B, int64_t ldb,
               void *stream)
{
    Handle *h = reinterpret_cast<Handle *>(hh);
    if (!h) { set_error("null handle"); return -1; }
    if (m < 0) return -2;
    if (n < 0) return -3;
    if (ldl < std::max<int64_t>(1, n)) { set_error("ldl < max(1,n)"); return -5; }
    if (ldb < std::max<int64_t>(1, m)) { set_error("ldb < max(1,m)"); return -7; }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    GLA_HIP_TRY(hipSetDevice(h->device));
    if (m == 0 || n == 0) return GLA_OK;
    GLA_TRY(ensure_workspace(h, sizeof(T) * linv_elems(n)));
    T *Linv = reinterpret_cast<T *>(h->ws);
    GLA_TRY(launch_tile_inverse<T>(s, n, L, ldl, Linv));
    return trsm_rlt_dev<T>(s, m, n, L, ldl, Linv, B, ldb);
}

}  // namespace

// ------------------------------------------------ no-allocation entry point --
// cholRecursive! for callers that cannot allocate device memory (code under
// HIP graph capture, serving loops): no handle, no hipMalloc.  Its scratch —
// the 16×16 diagonal-tile inverses of the panel solves and the info word —
// is this file-scope array, one copy per GPU, held until the process ends.
// Host code never passes `scratch` itself: its device address on the
// current GPU comes from hipGetSymbolAddress, taken once per device.
constexpr int64_t kNoAllocMaxN = 32768;
constexpr size_t kNoAllocLinvBytes = (size_t)(kNoAllocMaxN / 16 + 8) * 256 * sizeof(double);
constexpr size_t kNoAllocBytes = kNoAllocLinvBytes + 256;   // + the info word
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current GPU.
int scratch_address(void **out)
{
    int dev = 0;
    GLA_HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) {
        set_error("device ordinal %d beyond the %d this library tracks", dev, kMaxDevices);
        return GLA_ERR_UNSUPPORTED;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        GLA_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return GLA_OK;
}

int chol_recursive_noalloc(char uplo, int64_t n, double *A, int64_t lda, int64_t cutoff,
                           int64_t *info, void *stream)
{
    if (uplo != 'L' && uplo != 'U' && uplo != 'l' && uplo != 'u') {
        set_error("uplo must be 'L' or 'U'");
        return -1;
    }
    if (n < 0) { set_error("n < 0"); return -2; }
    if (n > kNoAllocMaxN) {
        set_error("n = %lld exceeds the no-allocation entry point's maximum %lld (its fixed "
                  "scratch holds the tile inverses of n <= %lld); use gla_chol_recursive_d",
                  (long long)n, (long long)kNoAllocMaxN, (long long)kNoAllocMaxN);
        return GLA_ERR_UNSUPPORTED;
    }
    if (!A && n > 0) { set_error("A is null"); return -3; }
    if (lda < std::max<int64_t>(1, n)) { set_error("lda < max(1,n)"); return -4; }
    void *base = nullptr;
    GLA_TRY(scratch_address(&base));
    double *Linv = reinterpret_cast<double *>(base);
    int *dinfo = reinterpret_cast<int *>(static_cast<unsigned char *>(base) + kNoAllocLinvBytes);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(k_set_int, dim3(1), dim3(1), 0, s, dinfo, 0);   // a kernel, not a memset
    GLA_LAUNCH_CHECK();
    // A handle-shaped view of the scratch: the drivers read only its info
    // word when use_side is false.
    Handle view;
    view.dinfo = dinfo;
    const bool upper = (uplo == 'U' || uplo == 'u');
    if (upper) GLA_TRY(swap_triangles<double>(s, n, A, lda));
    if (n > 0)
        GLA_TRY(chol_recursive_dev<double>(&view, s, n, A, lda, std::max<int64_t>(cutoff, 2048), 0,
                                           Linv, false));
    if (upper) GLA_TRY(swap_triangles<double>(s, n, A, lda));
    if (info) {
        int hv = 0;
        GLA_HIP_TRY(hipMemcpyAsync(&hv, dinfo, sizeof(int), hipMemcpyDeviceToHost, s));
        GLA_HIP_TRY(hipStreamSynchronize(s));
        *info = hv;
    }
    return GLA_OK;
}
}  // namespace
}  // namespace gla

using gla::chol_entry;

extern "C" {

int gla_chol_unblocked_d(gla_handle_t h, char uplo, int64_t n, double *A, int64_t lda,
                         int64_t *info, void *stream)
{
    return chol_entry<double>(h, uplo, n, A, lda, 0, 0, info, stream);
}
int gla_chol_unblocked_s(gla_handle_t h, char uplo, int64_t n, float *A, int64_t lda,
                         int64_t *info, void *stream)
{
    return chol_entry<float>(h, uplo, n, A, lda, 0, 0, info, stream);
}
int gla_chol_blocked_d(gla_handle_t h, char uplo, int64_t n, double *A, int64_t lda,
                       int64_t blocksize, int64_t *info, void *stream)
{
    return chol_entry<double>(h, uplo, n, A, lda, 1, blocksize, info, stream);
}
int gla_chol_blocked_s(gla_handle_t h, char uplo, int64_t n, float *A, int64_t lda,
                       int64_t blocksize, int64_t *info, void *stream)
{
    return chol_entry<float>(h, uplo, n, A, lda, 1, blocksize, info, stream);
}
int gla_chol_recursive_d(gla_handle_t h, char uplo, int64_t n, double *A, int64_t lda,
                         int64_t cutoff, int64_t *info, void *stream)
{
    return chol_entry<double>(h, uplo, n, A, lda, 2, cutoff, info, stream);
}
int gla_chol_recursive_s(gla_handle_t h, char uplo, int64_t n, float *A, int64_t lda,
                         int64_t cutoff, int64_t *info, void *stream)
{
    return chol_entry<float>(h, uplo, n, A, lda, 2, cutoff, info, stream);
}
int gla_chol_recursive_noalloc_d(char uplo, int64_t n, double *A, int64_t lda, int64_t cutoff,
                                 int64_t *info, void *stream)
{
    return gla::chol_recursive_noalloc(uplo, n, A, lda, cutoff, info, stream);
}
int gla_rank_update_d(gla_handle_t h, char uplo, int64_t n, int64_t k, double alpha,
                      const double *A, int64_t lda, double *C, int64_t ldc, void *stream)
{
    return gla::rank_update_entry<double>(h, uplo, n, k, alpha, A, lda, C, ldc, stream);
}
int gla_rank_update_s(gla_handle_t h, char uplo, int64_t n, int64_t k, float alpha,
                      const float *A, int64_t lda, float *C, int64_t ldc, void *stream)
{
    return gla::rank_update_entry<float>(h, uplo, n, k, alpha, A, lda, C, ldc, stream);
}
int gla_trsm_rlt_d(gla_handle_t h, int64_t m, int64_t n, const double *L, int64_t ldl,
                   double *B, int64_t ldb, void *stream)
{
    return gla::trsm_entry<double>(h, m, n, L, ldl, B, ldb, stream);
}
int gla_trsm_rlt_s(gla_handle_t h, int64_t m, int64_t n, const float *L, int64_t ldl, float *B,
                   int64_t ldb, void *stream)
{
    return gla::trsm_entry<float>(h, m, n, L, ldl, B, ldb, stream);
}

}  // extern "C"
