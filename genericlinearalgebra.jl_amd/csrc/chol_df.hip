// Dataflow Cholesky: the factor of an m×n block column (m ≥ n, the first n
// rows its symmetric diagonal block) in one launch, cholBlocked!'s products
// (src/cholesky.jl:17-35) tile by tile.
//
// The matrix is cut into 64×64 tiles and every workgroup owns one tile
// (i, j) below the diagonal, or the diagonal tile (j, j) together with its
// left neighbour (j, j − 1).  It keeps the tile in accumulators, subtracts
// X(i, k) X(j, k)ᵀ for k = 0, 1, … as the factored tiles X arrive, then
// solves with L(j, j) or factors.  A finished tile goes to the matrix, and to
// a packed copy in the layout the MFMA operands have (16-byte pieces,
// consecutive over the lanes), written with device-coherent stores and read
// straight into LDS by coherent 16-byte loads.  Row i's tiles finish in
// column order, so one counter per row announces them, and one flag per
// diagonal tile its L.
//
// Order and progress: tiles are numbered by columns, diagonal tile first, and
// a tile reads tiles of smaller numbers only.  A workgroup takes its number by
// a ticket when it starts, so whatever else runs on the device the unfinished
// tile with the smallest number is always one that is running, and has
// everything it waits for; the launch needs no more workgroups resident than
// fit.  (Numbers by blockIdx, which would hold for a launch that has the device
// to itself, spread the tiles better: FP64 n = 5001 1.45 ms, 8192 4.56.  By
// ticket 1.57 and 4.84, and with the diagonal tiles' waves, which the chain
// goes through, at a higher priority 1.52 and 4.72.)
// Every wait is bounded by spin_limit polls; one that gives up puts −1 in *info
// before its workgroup publishes anything.  A workgroup looks there after its
// own waits, and when it finds −1 leaves NaN for its tile: whatever was formed
// from data that had not come, at any remove, is NaN in the matrix.
//
// Bound: for small n the chain along the diagonal, per 64 columns the tile
// factor of four 16×16 tiles (≈7 µs), one flag and tile exchange between
// workgroups (≈2 µs) and the 64-wide solve and update (≈2 µs): FP64 n = 1000
// takes 0.21 ms (0.53 ms with a launch per factor, solve and update of 128
// columns).  For large n the products, at about half the MFMA rate (n = 8192
// FP64: 4.72 ms, 39 TFLOP/s): three workgroups per CU cover each other's
// waits, which is why a slab is 16 columns (53 KB of LDS); with 32-column
// slabs and two workgroups per CU n = 8192 took 5.07 ms.  Coherent or plain
// operand loads took the same time, so the coherent ones stay.
// Accuracy: sums are formed from zero over 256 columns at a time, as the
// launch-per-step driver's; FP64 n = 1000 is 1.5e-16 from an 80-bit
// evaluation (2.1e-16 that driver).
#include <algorithm>

#include "gla_coherent.hpp"
#include "gla_internal.hpp"

namespace gla {

namespace {

constexpr int kDT = 64;               // tile
constexpr int kTE = kDT * kDT;        // elements of a tile
constexpr int kLE = 10 * 256;         // elements of a packed L: 4 inverses, 6 tiles
constexpr int kDThreads = 256;
constexpr int kXLD = 17;              // padded row of the inverse's row-major copy

template <typename T>
struct DfP {
    T *A;
    int64_t lda;
    int64_t m, n;
    int mt, nt;           // tile rows, tile columns
    T *X;                 // packed tiles below the diagonal
    T *L;                 // packed diagonal tiles
    int *prog;            // per tile row: finished tiles left of the diagonal
    int *ldone;           // per tile column: 1 when L(j, j) is published
    int *ticket;          // workgroups started
    int *info;
    int64_t info_base;
    T *LinvG;             // 16×16 tile inverses, row-major (optional)
    unsigned spin_limit;
};

// 16×16 piece in operand order: value r of `lane` (accumulator element r, or
// K step r of an operand); 16-byte vectors of one lane, lanes consecutive.
__device__ __forceinline__ void put16(double *p, const d4 &v)
{
    const int lane = threadIdx.x & 63;
    typedef double d2 __attribute__((ext_vector_type(2)));
    *reinterpret_cast<d2 *>(p + 2 * lane) = d2{v[0], v[1]};
    *reinterpret_cast<d2 *>(p + 128 + 2 * lane) = d2{v[2], v[3]};
}
__device__ __forceinline__ void put16(float *p, const f4 &v)
{
    *reinterpret_cast<f4 *>(p + 4 * (threadIdx.x & 63)) = v;
}
__device__ __forceinline__ d4 get16(const double *p)
{
    const int lane = threadIdx.x & 63;
    typedef double d2 __attribute__((ext_vector_type(2)));
    const d2 a = *reinterpret_cast<const d2 *>(p + 2 * lane);
    const d2 b = *reinterpret_cast<const d2 *>(p + 128 + 2 * lane);
    return d4{a[0], a[1], b[0], b[1]};
}
__device__ __forceinline__ f4 get16(const float *p)
{
    return *reinterpret_cast<const f4 *>(p + 4 * (threadIdx.x & 63));
}
// The same to global memory, device-coherent (sc1).  The s_nop keeps the data
// registers unwritten for the cycle a store of over 8 bytes needs them.
__device__ __forceinline__ void publish16(double *p, const d4 &v)
{
    const int lane = threadIdx.x & 63;
    typedef double d2 __attribute__((ext_vector_type(2)));
    const d2 a{v[0], v[1]}, b{v[2], v[3]};
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p + 2 * lane), "v"(a) : "memory");
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p + 128 + 2 * lane), "v"(b) : "memory");
}
__device__ __forceinline__ void publish16(float *p, const f4 &v)
{
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p + 4 * (threadIdx.x & 63)), "v"(v)
                 : "memory");
}

// This wave's share of copying `elems` packed elements (16-byte pieces, 1 KB
// per wave instruction) to LDS, coherent and asynchronous: complete after
// this wave's vmcnt(0) and a barrier.
template <typename T>
__device__ __forceinline__ void stage(const T *g, T *l, int elems)
{
    constexpr int E = 1024 / sizeof(T);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int e = w * E; e < elems; e += 4 * E)
        __builtin_amdgcn_global_load_lds((const void *)(g + e + lane * (16 / sizeof(T))),
                                         (__attribute__((address_space(3))) void *)(l + e), 16, 0,
                                         16);
}

// Waits until *f ≥ need; returns the value seen (need after a time-out).
__device__ __forceinline__ int wait_ge(const int *f, int need, unsigned limit, int *info)
{
    int v = __builtin_amdgcn_readfirstlane(load_coherent(f));
    for (unsigned spins = 0; v < need; v = __builtin_amdgcn_readfirstlane(load_coherent(f))) {
        __builtin_amdgcn_s_sleep(1);
        if (++spins > limit || ((spins & 255) == 0 && load_coherent(info) < 0)) {
            if ((threadIdx.x & 63) == 0) store_coherent(info, -1);
            return need;
        }
    }
    return v;
}

template <typename T>
__device__ __forceinline__ T *x_tile(const DfP<T> &p, int i, int k)
{
    const int64_t q = i < p.nt ? (int64_t)i * (i - 1) / 2 + k
                               : (int64_t)p.nt * (p.nt - 1) / 2 + (int64_t)(i - p.nt) * p.nt + k;
    return p.X + q * kTE;
}

// Strip of tile (i, j) this wave owns (tile row w), transposed: acc[b] holds
// rows 64 i + 16 w + l % 16 at columns 64 j + 16 b + row(l, r); zero past m.
template <typename T>
__device__ __forceinline__ void load_strip(const DfP<T> &p, int i, int j, int w,
                                           typename PanelMfma<T>::acc_t acc[4])
{
    const int lane = threadIdx.x & 63;
    const int64_t gr = (int64_t)i * kDT + 16 * w + (lane & 15);
    const int64_t grc = gr < p.m ? gr : p.m - 1;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const T v = p.A[grc + ((int64_t)j * kDT + 16 * b + PanelMfma<T>::row(lane, r)) * p.lda];
            acc[b][r] = gr < p.m ? v : T(0);
        }
}
template <typename T>
__device__ __forceinline__ void store_strip(const DfP<T> &p, int i, int j, int w,
                                            const typename PanelMfma<T>::acc_t acc[4])
{
    const int lane = threadIdx.x & 63;
    const int64_t gr = (int64_t)i * kDT + 16 * w + (lane & 15);
    if (gr >= p.m) return;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            p.A[gr + ((int64_t)j * kDT + 16 * b + PanelMfma<T>::row(lane, r)) * p.lda] = acc[b][r];
}

// acc <- acc L⁻ᵀ for the packed L in LDS: the strip's column blocks left to
// right, operands in registers and LDS alone.
template <typename T>
__device__ __forceinline__ void solve_strip(const T *Ls, typename PanelMfma<T>::acc_t acc[4])
{
    typedef PanelMfma<T> M;
    typedef typename M::acc_t acc_t;
    int q = 4;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
        const acc_t li = get16(Ls + kb * 256);
        acc_t x = {T(0), T(0), T(0), T(0)};
#pragma unroll
        for (int kq = 0; kq < 4; ++kq) x = M::mma(li[kq], acc[kb][kq], x);
        acc[kb] = x;
#pragma unroll
        for (int b = kb + 1; b < 4; ++b, ++q) {
            const acc_t l = get16(Ls + q * 256);
#pragma unroll
            for (int kq = 0; kq < 4; ++kq) acc[b] = M::mma(l[kq], -x[kq], acc[b]);
        }
    }
}

// The diagonal tile: strips of its lower tiles in c (b < w), its diagonal
// 16×16 tile in dg (symmetric).  Wave r owns tile row r; wave 0 factors and
// inverts the diagonal tiles in turn (tile_factor), as chol_factor_kernel.
// The other waves' barriers match wave 0's: two per 16 columns.
template <typename T>
__device__ __forceinline__ void factor_diag(const DfP<T> &p, int j, int w,
                                            typename PanelMfma<T>::acc_t c[3],
                                            typename PanelMfma<T>::acc_t &dg, T *Db, T *Lib, T *Xs)
{
    typedef PanelMfma<T> M;
    typedef typename M::acc_t acc_t;
    constexpr int LS = 16 * kXLD;
    const int lane = threadIdx.x & 63, lc = lane & 15, lg = lane >> 4;
    const int64_t r0 = (int64_t)j * kDT;
    const int nv = (int)(p.n - r0 < kDT ? p.n - r0 : kDT);   // valid rows and columns
    const int nkb = (nv + 15) / 16;
    T *Lp = p.L + (int64_t)j * kLE;
    T *D0 = p.A + r0 * (1 + p.lda);

    auto store_lower = [&](int bi, int bj, const acc_t &v) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int gi = bi * 16 + lc, gj = bj * 16 + M::row(lane, r);
            if (gi < nv && gj <= gi) D0[gi + (int64_t)gj * p.lda] = v[r];
        }
    };
    if (w == 0) {
#pragma unroll 1
        for (int kb = 0; kb < nkb; ++kb) {
            if (kb > 0) dg = get16(Db);
            T iv[4];
            tile_factor<T>(dg, iv, nv - kb * 16, p.info, p.info_base + r0 + kb * 16);
            T *Li = Lib + (kb & 1) * LS;
#pragma unroll
            for (int t = 0; t < 4; ++t) Li[lc * kXLD + lg + 4 * t] = iv[t];
            if (kb == 0) stores_done();            // the solved strip's publication
            lds_barrier();                                            // end of (B)
            if (kb == 0 && lane == 0 && j > 0) store_coherent(p.prog + j, j);
            acc_t op;
#pragma unroll
            for (int r = 0; r < 4; ++r) op[r] = Li[lc * kXLD + M::row(lane, r)];
            publish16(Lp + kb * 256, op);
            if (p.LinvG)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    p.LinvG[((int64_t)4 * j + kb) * 256 + lc * 16 + lg + 4 * t] = iv[t];
            store_lower(kb, kb, dg);
            lds_barrier();                                            // end of (A)
        }
    } else {
        stores_done();
        lds_barrier();
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
            if (kb >= nkb) break;
            T *X = Xs + (kb & 1) * 768;           // tile rows 1–3
            acc_t x = {T(0), T(0), T(0), T(0)};
            if (w > kb && w < nkb) {
                const T *Li = Lib + (kb & 1) * LS;
                const acc_t a = c[kb < 3 ? kb : 2];
#pragma unroll
                for (int kq = 0; kq < 4; ++kq) x = M::mma(Li[lc * kXLD + M::row(lane, kq)], a[kq], x);
                if (w == kb + 1) {
#pragma unroll
                    for (int kq = 0; kq < 4; ++kq) dg = M::mma(-x[kq], x[kq], dg);
                    put16(Db, dg);
                }
                put16(X + (w - 1) * 256, x);
            }
            lds_barrier();                                            // end of (A)
            if (kb + 1 >= nkb) break;
            if (w > kb && w < nkb) {
                if (w > kb + 1) {
#pragma unroll
                    for (int b = kb + 1; b < 3; ++b)
                        if (b < w) {
                            const acc_t xb = get16(X + (b - 1) * 256);
#pragma unroll
                            for (int kq = 0; kq < 4; ++kq) c[b] = M::mma(-xb[kq], x[kq], c[b]);
                        }
#pragma unroll
                    for (int kq = 0; kq < 4; ++kq) dg = M::mma(-x[kq], x[kq], dg);
                }
                // packed tile (w, kb) after the four inverses, by columns
                publish16(Lp + (4 + (kb == 0 ? w - 1 : kb == 1 ? 1 + w : 5)) * 256, x);
                store_lower(w, kb, x);
            }
            lds_barrier();                                            // end of (B)
        }
    }
    stores_done();
    lds_barrier();
    if (threadIdx.x == 0) store_coherent(p.ldone + j, 1);
}

template <typename T>
__global__ __launch_bounds__(kDThreads, sizeof(T) == 8 ? 3 : 4) void chol_df_kernel(DfP<T> p)
{
    typedef PanelMfma<T> M;
    typedef typename M::acc_t acc_t;
    constexpr int H = kTE / 4;                        // a quarter tile: 16 columns
    // a ring of three slabs of two operands; then the packed L and the solved
    // tile.  53 KB in FP64: three workgroups per CU
    __shared__ __align__(16) T buf[kLE + kTE];
    static_assert(3 * 2 * H <= kLE + kTE, "slab ring");
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;

    // this workgroup's tile: column j, then the diagonal tile or row i
    __shared__ int place;
    if (threadIdx.x == 0) place = atomicAdd(p.ticket, 1);
    lds_barrier();
    int j = 0, id = __builtin_amdgcn_readfirstlane(place);
    for (; j < p.nt; ++j) {
        const int c = 1 + p.mt - (j + 1 < p.nt ? j + 2 : j + 1);
        if (id < c) break;
        id -= c;
    }
    const bool diag = id == 0;
    const int i = diag ? j : id + (j + 1 < p.nt ? j + 1 : j);
    const int jo = diag ? j - 1 : j;                  // the column of acc and of operand X(jo, k)
    const int nk = diag ? (j > 0 ? j - 1 : 0) : j;    // products of 64 columns
    if (diag) __builtin_amdgcn_s_setprio(3);          // the chain goes through it

    acc_t acc[4], c[3], dg;
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[b] = acc_t{T(0), T(0), T(0), T(0)};
    if (jo >= 0) load_strip<T>(p, i, jo, w, acc);
    if (diag) {
        // tile row w of the diagonal tile, the identity past n
        const int lc = lane & 15;
        auto elem = [&](int a, int b) {
            const int gi = a > b ? a : b, gj = a > b ? b : a;
            const int64_t r = (int64_t)j * kDT + gi, cc = (int64_t)j * kDT + gj;
            const T v = p.A[(r < p.n ? r : p.n - 1) + (cc < p.n ? cc : p.n - 1) * p.lda];
            return r < p.n ? v : (gi == gj ? T(1) : T(0));
        };
#pragma unroll
        for (int b = 0; b < 3; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                c[b][r] = b < w ? elem(16 * w + lc, 16 * b + M::row(lane, r)) : T(0);
#pragma unroll
        for (int r = 0; r < 4; ++r) dg[r] = elem(16 * w + lc, 16 * w + M::row(lane, r));
    }

    // the products, in slabs of 16 columns: slab s of X(i, ·) and X(jo, ·) in
    // place s % 3 of a ring, two slabs in flight while one is multiplied
    const int ns = 4 * nk;
    // products are summed from zero and taken off the tile every kFold slabs:
    // a sum that runs through the tile rounds every product at the tile's own
    // magnitude (FP32 n = 5001: 4x the error)
    constexpr int kFold = 16;
    const acc_t zero = {T(0), T(0), T(0), T(0)};
    acc_t sa[4], sc[3], sd = zero;
#pragma unroll
    for (int b = 0; b < 4; ++b) sa[b] = zero;
#pragma unroll
    for (int b = 0; b < 3; ++b) sc[b] = zero;
    int av = 0, next = 0;                             // products available, next slab to load
    auto issue = [&]() {
        T *d = buf + (next % 3) * 2 * H;
        stage<T>(x_tile<T>(p, i, next >> 2) + (next & 3) * H, d, H);
        stage<T>(x_tile<T>(p, jo, next >> 2) + (next & 3) * H, d + H, H);
        ++next;
    };
    for (int s = 0; s < ns; ++s) {
        if (next <= s) {
            const int a = wait_ge(p.prog + i, (s >> 2) + 1, p.spin_limit, p.info);
            const int b = wait_ge(p.prog + jo, (s >> 2) + 1, p.spin_limit, p.info);
            av = a < b ? a : b;
            issue();
        }
        // this wave's loads of slab s have landed, those of later ones may not
        constexpr int PER = 2 * H * sizeof(T) / 4096;
        const int later = next - s - 1;
        if (later == 0) __builtin_amdgcn_s_waitcnt(0x0F70);
        else if (later == 1) __builtin_amdgcn_s_waitcnt(0x0F70 | PER);
        else __builtin_amdgcn_s_waitcnt(0x0F70 | (2 * PER));
        lds_barrier();      // everyone's have, and slab s − 1 has been read
        while (next < ns && next <= s + 2) {
            if (av < (next >> 2) + 1) {
                const int a = load_coherent(p.prog + i), b = load_coherent(p.prog + jo);
                av = __builtin_amdgcn_readfirstlane(a < b ? a : b);
                if (av < (next >> 2) + 1) break;
            }
            issue();
        }
        const T *bi = buf + (s % 3) * 2 * H, *bj = bi + H;
        const acc_t xi = get16(bi + w * 256);
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const acc_t xj = get16(bj + b * 256);
#pragma unroll
            for (int kq = 0; kq < 4; ++kq) sa[b] = M::mma(xj[kq], xi[kq], sa[b]);
        }
        if (diag) {
#pragma unroll
            for (int b = 0; b < 3; ++b)
                if (b < w) {
                    const acc_t xb = get16(bi + b * 256);
#pragma unroll
                    for (int kq = 0; kq < 4; ++kq) sc[b] = M::mma(xb[kq], xi[kq], sc[b]);
                }
#pragma unroll
            for (int kq = 0; kq < 4; ++kq) sd = M::mma(xi[kq], xi[kq], sd);
        }
        if ((s & (kFold - 1)) == kFold - 1 || s + 1 == ns) {
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                acc[b] -= sa[b];
                sa[b] = zero;
            }
            if (diag) {
#pragma unroll
                for (int b = 0; b < 3; ++b) {
                    c[b] -= sc[b];
                    sc[b] = zero;
                }
                dg -= sd;
                sd = zero;
            }
        }
    }

    int state = 0;
    // X = acc L(jo, jo)⁻ᵀ
    T *Ls = buf;                                      // 2560 elements
    T *Xr = buf + kLE;                                // 4096: the solved tile
    if (jo >= 0) {
        wait_ge(p.ldone + jo, 1, p.spin_limit, p.info);
        lds_barrier();                                // the last slab has been read
        stage<T>(p.L + (int64_t)jo * kLE, Ls, kLE);
        stores_done();
        lds_barrier();
        state = load_coherent(p.info);                // (looked at in the end)
        solve_strip<T>(Ls, acc);
        if (i < p.nt || jo + 1 < p.nt) {              // someone reads it
            T *xp = x_tile<T>(p, i, jo);
#pragma unroll
            for (int b = 0; b < 4; ++b) publish16(xp + (b * 4 + w) * 256, acc[b]);
        }
        if (!diag) {
            stores_done();
            lds_barrier();
            if (threadIdx.x == 0) store_coherent(p.prog + i, jo + 1);
        }
    }
    if (diag) {
        if (j > 0) {
            // the diagonal tile's own last product, operands from registers
            // and the other waves' strips from LDS
#pragma unroll
            for (int b = 0; b < 4; ++b) put16(Xr + (b * 4 + w) * 256, acc[b]);
            lds_barrier();
#pragma unroll
            for (int bk = 0; bk < 4; ++bk)
#pragma unroll
                for (int kq = 0; kq < 4; ++kq) sd = M::mma(acc[bk][kq], acc[bk][kq], sd);
            dg -= sd;
#pragma unroll
            for (int b = 0; b < 3; ++b)
                if (b < w) {
#pragma unroll
                    for (int bk = 0; bk < 4; ++bk) {
                        const acc_t xb = get16(Xr + (bk * 4 + b) * 256);
#pragma unroll
                        for (int kq = 0; kq < 4; ++kq) sc[b] = M::mma(xb[kq], acc[bk][kq], sc[b]);
                    }
                    c[b] -= sc[b];
                }
        }
        // Ls is free: every wave is past its solve (the barrier above; j = 0 has none)
        static_assert(256 + 2 * 16 * kXLD + 2 * 768 <= kLE, "LDS regions");
        factor_diag<T>(p, j, w, c, dg, buf, buf + 256, buf + 256 + 2 * 16 * kXLD);
    }
    if (__builtin_amdgcn_readfirstlane(state) < 0) {
        const T nan = T(__builtin_nan(""));
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[b] = acc_t{nan, nan, nan, nan};
        // (the diagonal tile is in the matrix: factor_diag ended with its stores)
        if (diag)
            for (int e = threadIdx.x; e < kTE; e += kDThreads) {
                const int64_t r = (int64_t)j * kDT + e % kDT, cc = (int64_t)j * kDT + e / kDT;
                if (r < p.n && cc <= r) p.A[r + cc * p.lda] = nan;
            }
    }
    if (jo >= 0) store_strip<T>(p, i, jo, w, acc);
}

// Clears the counters, flags and ticket of one launch.
__global__ void df_clear_kernel(int *f, int n)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e < n) f[e] = 0;
}

}  // namespace

size_t chol_df_bytes(int64_t m, int64_t n, size_t esz)
{
    const int64_t mt = cdiv(m, kDT), nt = cdiv(n, kDT);
    return (size_t)(nt * (nt - 1) / 2 + (mt - nt) * nt) * kTE * esz + (size_t)nt * kLE * esz +
           (size_t)(mt + nt + 1) * sizeof(int) + 256;
}

// The factor of the m×n block column at A.  h->df holds the packed copies;
// the caller has made it large enough (ensure_df).
template <typename T>
int chol_df(Handle *h, hipStream_t s, int64_t m, int64_t n, T *A, int64_t lda, int64_t info_base,
            T *LinvG)
{
    if (n <= 0) return GLA_OK;
    DfP<T> p;
    p.A = A;
    p.lda = lda;
    p.m = m;
    p.n = n;
    p.mt = (int)cdiv(m, kDT);
    p.nt = (int)cdiv(n, kDT);
    // rows below a partial last diagonal tile would share its tile row
    if (m < n || (m > n && n % kDT != 0) || h->df_bytes < chol_df_bytes(m, n, sizeof(T))) {
        set_error("chol_df: %lld x %lld does not fit", (long long)m, (long long)n);
        return GLA_ERR_UNSUPPORTED;
    }
    const int64_t tiles = (int64_t)p.nt * (p.nt - 1) / 2 + (int64_t)(p.mt - p.nt) * p.nt;
    p.X = reinterpret_cast<T *>(h->df);
    p.L = p.X + tiles * kTE;
    p.prog = reinterpret_cast<int *>(p.L + (int64_t)p.nt * kLE);
    p.ldone = p.prog + p.mt;
    p.ticket = p.ldone + p.nt;
    p.info = h->dinfo;
    p.info_base = info_base;
    p.LinvG = LinvG;
    p.spin_limit = h->spin_limit;
    const int nf = p.mt + p.nt + 1;
    hipLaunchKernelGGL(df_clear_kernel, dim3((unsigned)cdiv(nf, 256)), dim3(256), 0, s, p.prog, nf);
    GLA_LAUNCH_CHECK();
    // one workgroup per tile, the left neighbour of each diagonal tile but
    // the first going with it
    const int64_t grid = tiles + p.nt - (p.nt - 1);
    hipLaunchKernelGGL((chol_df_kernel<T>), dim3((unsigned)grid), dim3(kDThreads), 0, s, p);
    GLA_LAUNCH_CHECK();
    return GLA_OK;
}

template int chol_df<double>(Handle *, hipStream_t, int64_t, int64_t, double *, int64_t, int64_t,
                             double *);
template int chol_df<float>(Handle *, hipStream_t, int64_t, int64_t, float *, int64_t, int64_t,
                            float *);

}  // namespace gla
