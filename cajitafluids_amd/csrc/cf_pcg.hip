// cf_pcg.hip -- matrix-free Jacobi-PCG (FP64, and FP32 inside an FP64
// defect-correction loop) for the pressure solve of
// src/VelocityCorrector.hpp:266-282.
//
// Control flow (this library's statement of Cajita's ReferenceConjugateGradient,
// called at src/VelocityCorrector.hpp:276), from x = 0:
//   r = b; rho = r.(D^-1 r); bnorm = ||b||            (bnorm = 0: done)
//   iteration k:
//     p = D^-1 r                      (k = 1)
//     p = fma(beta, p, D^-1 r)        (k > 1)
//     q = A p; alpha = rho / p.q
//     x = fma(alpha, p, x); r = fma(-alpha, q, r)
//     stop if ||r|| / bnorm < tol, or k = maxit
//     beta = r.(D^-1 r) / rho; rho = r.(D^-1 r)
//
// One iteration is two streaming kernels:
//   dir_spmv: p_new = fma(beta, p_old, D^-1 r) at the cell, and at each
//             stencil neighbour recomputed from r and p_old there; q = A p_new;
//             p_new.q -> alpha.                reads r, p_old; writes p_new
//   update:   q = A p_new again (same expression, same bits); x += alpha p_new;
//             r -= alpha q; r.r, r.(D^-1 r) -> convergence test, beta, rho.
//                                              reads x, p_new, r; writes x, r
// 8 vector words per cell per iteration instead of the 11 of the
// SpMV / update / direction split.  p is double-buffered because dir_spmv
// reads the old direction around each cell while writing the new one.  The
// 3-D FP64 update takes x every second iteration (XUpdate: the skipped step
// and the current one are applied together, in order, from the two
// direction buffers), 7.5 words per iteration.  The
// last block of each kernel to finish computes the scalars on the device;
// every kernel returns at once when the device-side `done` flag is set, so
// the host queues iterations in batches and polls once per batch.
#include <hip/hip_runtime.h>

#include "cf_pcg_state.hpp"
#include "cf_solver.hpp"
#include "cf_stream.hpp"
#include "cf_tile3.hpp"


namespace cfmi
{

// ---- PCG initialisation ------------------------------------------------------
__global__ __launch_bounds__(256) void k_pcg_init64(
    Geo g, const double* __restrict__ b, double* __restrict__ x,
    double* __restrict__ r, PcgState* st, double tol, int maxit, RedBuf rb)
{
    double hi[2] = {0.0, 0.0}, lo[2] = {0.0, 0.0};
    for_owned_rows(g, [&](int64_t base, int j, int k) {
        const int ryz = wall_count(g, 1, j) + wall_count(g, 2, k);
        for (int i = threadIdx.x; i < g.n[0]; i += kBlock) {
            const int64_t c = base + i;
            const double bc = b[c];
            const double z = dinv_pick<double>(g, ryz, wall_count(g, 0, i)) * bc;
            r[c] = bc; // r = b - A 0 = b
            x[c] = 0.0;
            dd_add_prod(hi[0], lo[0], bc, z);
            dd_add_prod(hi[1], lo[1], bc, bc);
        }
    });
    grid_reduce<2>(hi, lo, rb,
                   [&](double* s) { init_state(st, s[0], s[1], tol, maxit); });
}

// Relative FP32 reduction that ends a defect-correction pass started from a
// residual of norm rref: inner_tol, or less when half the final target
// (0.5 tol ||b||) is closer, so the last pass stops near the target instead
// of a full inner_tol past it.
__device__ __forceinline__ double pass_tol(double itol, double gtol,
                                           double bnorm, double rref)
{
    return fmax(itol, (0.5 * gtol * bnorm) / rref);
}

__global__ __launch_bounds__(256) void k_pcg_init32(
    Geo g, const float* __restrict__ r, float* __restrict__ d, PcgState* st,
    const RefineState* rs, double itol, double gtol, int maxit, RedBuf rb)
{
    double hi[2] = {0.0, 0.0}, lo[2] = {0.0, 0.0};
    for_owned_rows(g, [&](int64_t base, int j, int k) {
        const int ryz = wall_count(g, 1, j) + wall_count(g, 2, k);
        for (int i = threadIdx.x; i < g.n[0]; i += kBlock) {
            const int64_t c = base + i;
            const float rc = r[c];
            const float z = dinv_pick<float>(g, ryz, wall_count(g, 0, i)) * rc;
            d[c] = 0.0f;
            dd_add_prod(hi[0], lo[0], (double)rc, (double)z);
            dd_add_prod(hi[1], lo[1], (double)rc, (double)rc);
        }
    });
    grid_reduce<2>(hi, lo, rb, [&](double* s) {
        const double r0 = sqrt(s[1]);
        init_state(st, s[0], s[1], pass_tol(itol, gtol, rs->bnorm, r0), maxit);
    });
}

// ---- one PCG iteration --------------------------------------------------------
// The two halves of an iteration over this block's owned rows (the row
// partition of for_owned_rows), accumulating the block's double-double
// partials.
template <int DIM, class T>
__device__ __forceinline__ void dir_spmv_rows(const Geo& g, const T* __restrict__ r,
                                              const T* __restrict__ p_old,
                                              T* __restrict__ p_new, bool first, T beta,
                                              double (&hi)[1], double (&lo)[1])
{
    const T s = offdiag<T>(g);
    for_owned_rows(g, [&](int64_t base, int j, int k) {
        const RowStencil rs = row_stencil(g, j, k);
        for (int i = threadIdx.x; i < g.n[0]; i += kBlock) {
            const int64_t c = base + i;
            const LaneX lx = lane_x(g, i);
            // new direction at cell `at` whose wall count is ubase + wx
            auto pdir = [&](int64_t at, int ubase, int wx) -> T {
                const T z = dinv_pick<T>(g, ubase, wx) * r[at];
                return first ? z : fma_t<T>(beta, p_old[at], z);
            };
            const T pc = pdir(c, rs.cnt, lx.cnt);
            T y = diag_pick<T>(g, rs.cnt, lx.cnt) * pc;
#pragma unroll
            for (int side = 0; side < 2; ++side) {
                const T pn = pdir(c + lx.off[side], rs.cnt, lx.ncnt[side]);
                y = fma_t<T>(lx.wall[side] ? (T)0 : s, lx.wall[side] ? (T)0 : pn, y);
            }
#pragma unroll
            for (int d = 1; d < DIM; ++d) {
#pragma unroll
                for (int side = 0; side < 2; ++side) {
                    const T pn = pdir(c + rs.off[d][side], rs.ncnt[d][side], lx.cnt);
                    y = fma_t<T>(rs.wall[d][side] ? (T)0 : s,
                                 rs.wall[d][side] ? (T)0 : pn, y);
                }
            }
            p_new[c] = pc;
            dd_add_prod(hi[0], lo[0], (double)pc, (double)y);
        }
    });
}

template <int DIM, class T>
__device__ __forceinline__ void update_rows(const Geo& g, T* __restrict__ x, T* __restrict__ r,
                                            const T* __restrict__ p, T alpha, double (&hi)[2],
                                            double (&lo)[2])
{
    for_owned_rows(g, [&](int64_t base, int j, int k) {
        const RowStencil rs = row_stencil(g, j, k);
        for (int i = threadIdx.x; i < g.n[0]; i += kBlock) {
            const int64_t c = base + i;
            const LaneX lx = lane_x(g, i);
            const T q = apply_A<DIM, T>(g, rs, lx, p, c);
            x[c] = fma_t<T>(alpha, p[c], x[c]);
            const T rn = fma_t<T>(-alpha, q, r[c]);
            r[c] = rn;
            const T z = dinv_pick<T>(g, rs.cnt, lx.cnt) * rn;
            dd_add_prod(hi[0], lo[0], (double)rn, (double)rn);
            dd_add_prod(hi[1], lo[1], (double)rn, (double)z);
        }
    });
}

template <int DIM, class T>
__global__ __launch_bounds__(256) void k_pcg_dir_spmv(
    Geo g, const T* __restrict__ r, const T* __restrict__ p_old,
    T* __restrict__ p_new, PcgState* st, RedBuf rb)
{
    if (st->done)
        return;
    double hi[1] = {0.0}, lo[1] = {0.0};
    dir_spmv_rows<DIM, T>(g, r, p_old, p_new, st->iter == 0, (T)st->beta, hi, lo);
    grid_reduce<1>(hi, lo, rb, [&](double* sm) { st->alpha = st->rho / sm[0]; });
}

template <int DIM, class T>
__global__ __launch_bounds__(256) void k_pcg_update(
    Geo g, T* __restrict__ x, T* __restrict__ r, const T* __restrict__ p,
    PcgState* st, RedBuf rb)
{
    if (st->done)
        return;
    double hi[2] = {0.0, 0.0}, lo[2] = {0.0, 0.0};
    update_rows<DIM, T>(g, x, r, p, (T)st->alpha, hi, lo);
    grid_reduce<2>(hi, lo, rb, [&](double* sm) { finish_update(st, sm[0], sm[1]); });
}

// ---- 3-D kernels (cf_tile3.hpp) ------------------------------------------------
// Products of two floats are exact in double, so the FP32 kernels skip the
// TwoProd error term.
template <class T>
constexpr bool exact_products()
{
    return std::is_same<T, float>::value;
}

// Cells per lane along x of the 3-D kernels: 2 for FP32 (8-byte accesses);
// CF_CPL64 for FP64.
#ifndef CF_CPL64
#define CF_CPL64 1
#endif
template <class T>
constexpr int cpl_of()
{
    return std::is_same<T, float>::value ? 2 : CF_CPL64;
}

template <class T, int CPL>
struct DirEpiT
{
    const Geo& g;
    T* __restrict__ p_new;
    double hi[1] = {0.0}, lo[1] = {0.0};
    template <int B>
    __device__ void prefetch(const Tile3Ctx<CPL>&, const Plane3Meta&, int)
    {
    }
    __device__ void shift() {}
    __device__ void rotate() {}
    template <int B>
    __device__ void cells(const Tile3Ctx<CPL>& c, const Plane3Meta& m, int q,
                          const T (&pc)[CPL], const T (&y)[CPL])
    {
        vstore_valid<T, CPL>(p_new + c.colb[q] + m.off, pc, c.valid[q]);
#pragma unroll
        for (int j = 0; j < CPL; ++j)
            if (c.valid[q][j])
                dd_acc_prod<exact_products<T>()>(hi[0], lo[0], (double)pc[j], (double)y[j]);
    }
};

// The update's epilogue; XM is its x mode (XUpdate).
//
// X_EACH and X_SKIP: x and r of the next plane load into the second of two
// buffers (prefetch) while the march works on the current one.  X_PAIR
// reads one more vector; it loads x, r and the previous direction of the
// next plane after each step's barrier instead (kLate), into one buffer,
// which keeps it at 4 waves per SIMD in FP32 (double-buffered it would take
// 143 VGPRs, 3 waves).
//
// R32: the update also writes (float) r, the FP32 right-hand side of a
// multigrid V-cycle whose finest level runs in FP32 (the V-cycle then needs
// no cast of its own).
template <class T, int CPL, int XM, bool R32 = false>
struct UpdEpiT
{
    const Geo& g;
    T* __restrict__ x;
    T* __restrict__ r;
    T alpha;
    const T* __restrict__ p_lag; // X_PAIR: the previous direction
    T alpha_lag;
    float* __restrict__ r32;     // R32: (float) r
    double hi[2] = {0.0, 0.0}, lo[2] = {0.0, 0.0};
    static constexpr bool kReadX = XM != X_SKIP;
    static constexpr bool kLate = XM == X_PAIR;
    // x and r of a plane, in two buffers that alternate with the march's
    // steps (X_EACH, X_SKIP)
    T xb[2][tile3::RY][CPL], rb[2][tile3::RY][CPL];
    // kLate: x, r and p_lag of the current plane, and where the next one is
    T xs[tile3::RY][CPL], rs[tile3::RY][CPL], ls[tile3::RY][CPL];
    int next_k = 0;
    int64_t next_off = 0;

    __device__ void late(const Tile3Ctx<CPL>& c)
    {
#pragma unroll
        for (int q = 0; q < tile3::RY; ++q) {
            // a group with a valid first cell lies inside its padded row
            const bool ok = next_k >= c.k0 && next_k < c.k1 && c.valid[q][0];
            const int64_t at = c.colb[q] + next_off;
            if constexpr (CPL == 1) {
                xs[q][0] = load_any<T>(x, ok, at, c.safe);
                ls[q][0] = load_any<T>(p_lag, ok, at, c.safe);
                rs[q][0] = load_any<T>(r, ok, at, c.safe);
                continue;
            }
            const int64_t ap = ok ? at : c.safe;
            vload<T, CPL>(x + ap, xs[q]);
            vload<T, CPL>(p_lag + ap, ls[q]);
            vload<T, CPL>(r + ap, rs[q]);
        }
    }
    template <int B>
    __device__ void prefetch(const Tile3Ctx<CPL>& c, const Plane3Meta& m, int k)
    {
        if constexpr (kLate) { // late() loads it
            next_k = k;
            next_off = m.off;
            return;
        }
#pragma unroll
        for (int q = 0; q < tile3::RY; ++q) {
            // a group with a valid first cell lies inside its padded row
            const bool ok = k >= c.k0 && k < c.k1 && c.valid[q][0];
            const int64_t at = c.colb[q] + m.off;
            if constexpr (CPL == 1) {
                // raw: cells() reads only valid rows of planes below k1
                if constexpr (kReadX)
                    xb[B][q][0] = load_any<T>(x, ok, at, c.safe);
                rb[B][q][0] = load_any<T>(r, ok, at, c.safe);
                continue;
            }
            // an aligned pair on every path (raw, as above)
            const int64_t ap = ok ? at : c.safe;
            if constexpr (kReadX)
                vload<T, CPL>(x + ap, xb[B][q]);
            vload<T, CPL>(r + ap, rb[B][q]);
        }
    }
    __device__ void shift()
    {
        if constexpr (!kLate) {
#pragma unroll
            for (int q = 0; q < tile3::RY; ++q)
#pragma unroll
                for (int j = 0; j < CPL; ++j) {
                    if constexpr (kReadX)
                        xb[0][q][j] = xb[1][q][j];
                    rb[0][q][j] = rb[1][q][j];
                }
        }
    }
    __device__ void rotate() {}
    template <int B>
    __device__ void cells(const Tile3Ctx<CPL>& c, const Plane3Meta& m, int q,
                          const T (&pc)[CPL], const T (&qv)[CPL])
    {
        const int64_t at = c.colb[q] + m.off;
        T ro[CPL];
#pragma unroll
        for (int j = 0; j < CPL; ++j)
            ro[j] = fma_t<T>(-alpha, qv[j], kLate ? rs[q][j] : rb[B][q][j]);
        if constexpr (kReadX) {
            T xo[CPL];
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                // X_PAIR: the skipped step first, then this one
                const T xl = kLate ? fma_t<T>(alpha_lag, ls[q][j], xs[q][j]) : xb[B][q][j];
                xo[j] = fma_t<T>(alpha, pc[j], xl);
            }
            vstore_valid<T, CPL>(x + at, xo, c.valid[q]);
        }
        vstore_valid<T, CPL>(r + at, ro, c.valid[q]);
        if constexpr (R32) {
            float rf[CPL];
#pragma unroll
            for (int j = 0; j < CPL; ++j)
                rf[j] = (float)ro[j];
            vstore_valid<float, CPL>(r32 + at, rf, c.valid[q]);
        }
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
            if (!c.valid[q][j])
                continue;
            const T z = ctx_dinv<T, 0>(g, c, c.wy[q] + m.wz, c.wx[j]) * ro[j];
            dd_acc_prod<exact_products<T>()>(hi[0], lo[0], (double)ro[j], (double)ro[j]);
            dd_acc_prod<exact_products<T>()>(hi[1], lo[1], (double)ro[j], (double)z);
        }
    }
};

// TR: the element type of r (float: an FP32 multigrid V-cycle's z, widened
// on load; its values are the FP64 z's exactly).
template <class T, int CPL, bool PX, class TR = T>
__global__ __launch_bounds__(kTileBlock) void k_pcg_dir_spmv3(
    Geo g, Tile3Grid tg, const TR* __restrict__ r, const T* __restrict__ p_old,
    T* __restrict__ p_new, PcgState* st, RedBuf rb)
{
    using namespace tile3;
    if (st->done)
        return;
    __shared__ __align__(16) T pl[2][TY + 2][prow<CPL>()];
    const bool first = st->iter == 0;
    const T beta = (T)st->beta;
    DirEpiT<T, CPL> epi{g, p_new};
    tile3_march<T, true, CPL, PX, false, TR>(g, tg, r, p_old, first, beta, pl, epi);
    dd_norm(epi.hi[0], epi.lo[0]);
    grid_reduce<1, kTileBlock>(epi.hi, epi.lo, rb,
                   [&](double* sm) { st->alpha = st->rho / sm[0]; });
}

template <class T, int CPL, bool PX, int XM, bool R32>
__global__ __launch_bounds__(kTileBlock) void k_pcg_update3(
    Geo g, Tile3Grid tg, T* __restrict__ x, T* __restrict__ r,
    const T* __restrict__ p, const T* __restrict__ p_lag, float* __restrict__ r32,
    PcgState* st, RedBuf rb)
{
    using namespace tile3;
    if (st->done)
        return;
    __shared__ __align__(16) T pl[2][TY + 2][prow<CPL>()];
    UpdEpiT<T, CPL, XM, R32> epi{g, x, r, (T)st->alpha, p_lag, (T)st->alpha_lag, r32};
    // downwards: the direction kernel marches up, so each kernel starts on
    // the planes the other touched last (Infinity Cache hits; FP64 256^3:
    // update 127 -> 121 us, direction 101 -> 95 us)
    tile3_march<T, false, CPL, PX, true>(g, tg, p, nullptr, false, (T)0, pl, epi);
    dd_norm(epi.hi[0], epi.lo[0]);
    dd_norm(epi.hi[1], epi.lo[1]);
    grid_reduce<2, kTileBlock>(epi.hi, epi.lo, rb, [&](double* sm) {
        if (XM == X_SKIP) // every block has read the state by now
            st->alpha_lag = st->alpha;
        finish_update(st, sm[0], sm[1]);
    });
}

// x = fma(alpha, p, x): the x step an X_SKIP update left out, when it was
// the last of a run (alpha is still that iteration's).
template <class T>
__global__ __launch_bounds__(256) void k_pcg_xfix(Geo g, T* __restrict__ x,
                                                  const T* __restrict__ p,
                                                  const PcgState* st)
{
    const T a = (T)st->alpha;
    for_owned_cells(g, [&](int64_t c, int, int, int) { x[c] = fma_t<T>(a, p[c], x[c]); });
}

// ---- defect correction ---------------------------------------------------------
//   x = 0; r64 = b; bnorm = ||b||; res = ||r64|| / bnorm
//   pass: r32 = (float) r64; inner FP32 PCG d ~ A^-1 r32;
//         x = x + (double) d; r64 = b - A x; res = ||r64|| / bnorm
__global__ __launch_bounds__(256) void k_refine_init(
    Geo g, const double* __restrict__ b, double* __restrict__ x64,
    float* __restrict__ r32, RefineState* rst, RedBuf rb)
{
    double hi[1] = {0.0}, lo[1] = {0.0};
    for_owned_cells(g, [&](int64_t c, int, int, int) {
        const double bc = b[c];
        x64[c] = 0.0;
        r32[c] = (float)bc;
        dd_add_prod(hi[0], lo[0], bc, bc);
    });
    grid_reduce<1>(hi, lo, rb, [&](double* s) {
        const double bnorm = sqrt(s[0]);
        rst->bnorm = bnorm;
        rst->res = bnorm == 0.0 ? 0.0 : sqrt(s[0]) / bnorm;
    });
}

__global__ __launch_bounds__(256) void k_refine_add(Geo g,
                                                     double* __restrict__ x64,
                                                     float* __restrict__ d)
{
    for_owned_cells(g, [&](int64_t c, int, int, int) {
        x64[c] = x64[c] + (double)d[c];
        d[c] = 0.0f;
    });
}

template <int DIM>
__global__ __launch_bounds__(256) void k_refine_residual(
    Geo g, const double* __restrict__ b, const double* __restrict__ x64,
    float* __restrict__ r32, RefineState* rst, RedBuf rb)
{
    double hi[1] = {0.0}, lo[1] = {0.0};
    for_owned_rows(g, [&](int64_t base, int j, int k) {
        const RowStencil rs = row_stencil(g, j, k);
        for (int i = threadIdx.x; i < g.n[0]; i += kBlock) {
            const int64_t c = base + i;
            const LaneX lx = lane_x(g, i);
            const double y = apply_A<DIM, double>(g, rs, lx, x64, c);
            const double r = b[c] - y;
            r32[c] = (float)r;
            dd_add_prod(hi[0], lo[0], r, r);
        }
    });
    grid_reduce<1>(hi, lo, rb,
                   [&](double* s) { rst->res = sqrt(s[0]) / rst->bnorm; });
}

// ---- defect correction with the search direction carried across passes -----
//   x = 0; bnorm = ||b||; r32 = (float) b; d = 0; rref = ||r32||;
//   rho = r32.(D32^-1 r32); then one FP32 PCG run (the iteration kernels
//   above, which stop when ||r|| / rref < pass_tol).  At each pass boundary:
//   x = x + (double) d; d = 0; r64 = b - A x; res = ||r64|| / bnorm;
//   r32 = (float) r64; rref = ||r32||; beta = r32.(D32^-1 r32) / rho;
//   rho = r32.(D32^-1 r32); the PCG resumes with the same direction.
__global__ __launch_bounds__(256) void k_refine_init_carry(
    Geo g, const double* __restrict__ b, double* __restrict__ x64,
    float* __restrict__ r32, float* __restrict__ d32, RefineState* rst,
    PcgState* st, double itol, double gtol, int maxit, RedBuf rb)
{
    double hi[3] = {0.0, 0.0, 0.0}, lo[3] = {0.0, 0.0, 0.0};
    for_owned_rows(g, [&](int64_t base, int j, int k) {
        const int ryz = wall_count(g, 1, j) + wall_count(g, 2, k);
        for (int i = threadIdx.x; i < g.n[0]; i += kBlock) {
            const int64_t c = base + i;
            const double bc = b[c];
            const float rc = (float)bc;
            const float z = dinv_pick<float>(g, ryz, wall_count(g, 0, i)) * rc;
            x64[c] = 0.0;
            r32[c] = rc;
            d32[c] = 0.0f;
            dd_add_prod(hi[0], lo[0], bc, bc);
            dd_add_prod(hi[1], lo[1], (double)rc, (double)rc);
            dd_add_prod(hi[2], lo[2], (double)rc, (double)z);
        }
    });
    grid_reduce<3>(hi, lo, rb, [&](double* s) {
        const double bnorm = sqrt(s[0]);
        const double rref = sqrt(s[1]);
        rst->bnorm = bnorm;
        rst->res = 1.0;
        st->bnorm = rref;
        st->tol = pass_tol(itol, gtol, bnorm, rref);
        st->maxit = maxit;
        st->iter = 0;
        st->rho = s[2];
        st->alpha = 0.0;
        st->beta = 0.0;
        st->alpha_lag = 0.0;
        st->mg = 0;
        // a non-finite ||b|| is reported by the host from rst->bnorm
        st->nonfinite = isfinite(bnorm) ? 0 : 1;
        st->done = bnorm == 0.0 || st->nonfinite ? 1 : (maxit <= 0 ? 1 : 0);
        st->converged = bnorm == 0.0 ? 1 : 0;
        if (bnorm == 0.0)
            rst->res = 0.0;
    });
}

template <int DIM>
__global__ __launch_bounds__(256) void k_refine_residual_carry(
    Geo g, const double* __restrict__ b, const double* __restrict__ x64,
    float* __restrict__ r32, RefineState* rst, PcgState* st, double itol,
    double gtol, RedBuf rb)
{
    double hi[3] = {0.0, 0.0, 0.0}, lo[3] = {0.0, 0.0, 0.0};
    for_owned_rows(g, [&](int64_t base, int j, int k) {
        const RowStencil rs = row_stencil(g, j, k);
        for (int i = threadIdx.x; i < g.n[0]; i += kBlock) {
            const int64_t c = base + i;
            const LaneX lx = lane_x(g, i);
            const double y = apply_A<DIM, double>(g, rs, lx, x64, c);
            const double r = b[c] - y;
            const float rc = (float)r;
            const float z = dinv_pick<float>(g, rs.cnt, lx.cnt) * rc;
            r32[c] = rc;
            dd_add_prod(hi[0], lo[0], r, r);
            dd_add_prod(hi[1], lo[1], (double)rc, (double)rc);
            dd_add_prod(hi[2], lo[2], (double)rc, (double)z);
        }
    });
    grid_reduce<3>(hi, lo, rb, [&](double* s) {
        rst->res = sqrt(s[0]) / rst->bnorm;
        const double rref = sqrt(s[1]);
        st->bnorm = rref;
        st->tol = pass_tol(itol, gtol, rst->bnorm, rref);
        st->beta = s[2] / st->rho;
        st->rho = s[2];
        st->done = 0;
        st->converged = 0;
    });
}

// ---- RHS mean removal --------------------------------------------------------
__global__ __launch_bounds__(256) void k_rhs_sum(Geo g, const double* rhs,
                                                  double* out, RedBuf rb)
{
    double hi[1] = {0.0}, lo[1] = {0.0};
    for_owned_cells(g, [&](int64_t c, int, int, int) {
        dd_add(hi[0], lo[0], rhs[c], 0.0);
    });
    grid_reduce<1>(hi, lo, rb, [&](double* s) { out[0] = s[0]; });
}

__global__ __launch_bounds__(256) void k_rhs_shift(Geo g, double* rhs,
                                                    const double* sum)
{
    const double cnt = (double)g.n[0] * (double)g.n[1] * (double)g.n[2];
    const double mean = sum[0] / cnt;
    for_owned_cells(g, [&](int64_t c, int, int, int) { rhs[c] = rhs[c] - mean; });
}

// ---- launchers -------------------------------------------------------------------
#define CF_STREAM_LAUNCH(kernel, ...)                                         \
    hipLaunchKernelGGL(kernel, dim3(stream_blocks(g)), dim3(kBlock), 0, s,    \
                       __VA_ARGS__)

void launch_rhs_sum(const Geo& g, const double* rhs, double* out_sum,
                    RedBuf rb, hipStream_t s)
{
    CF_STREAM_LAUNCH(k_rhs_sum, g, rhs, out_sum, rb);
}

void launch_rhs_shift(const Geo& g, double* rhs, const double* sum,
                      hipStream_t s)
{
    CF_STREAM_LAUNCH(k_rhs_shift, g, rhs, sum);
}

void launch_pcg_init64(const Geo& g, const double* b, double* x, double* r,
                       PcgState* st, double tol, int maxit, RedBuf rb,
                       hipStream_t s)
{
    CF_STREAM_LAUNCH(k_pcg_init64, g, b, x, r, st, tol, maxit, rb);
}

void launch_pcg_init32(const Geo& g, const float* r, float* d, PcgState* st,
                       const RefineState* rs, double itol, double gtol,
                       int maxit, RedBuf rb, hipStream_t s)
{
    CF_STREAM_LAUNCH(k_pcg_init32, g, r, d, st, rs, itol, gtol, maxit, rb);
}

void launch_refine_init_carry(const Geo& g, const double* b, double* x64,
                              float* r32, float* d32, RefineState* rs,
                              PcgState* st, double itol, double gtol, int maxit,
                              RedBuf rb, hipStream_t s)
{
    CF_STREAM_LAUNCH(k_refine_init_carry, g, b, x64, r32, d32, rs, st, itol,
                     gtol, maxit, rb);
}

void launch_refine_residual_carry(const Geo& g, const double* b,
                                  const double* x64, float* r32,
                                  RefineState* rs, PcgState* st, double itol,
                                  double gtol, RedBuf rb, hipStream_t s)
{
    if (g.dim == 2)
        CF_STREAM_LAUNCH(k_refine_residual_carry<2>, g, b, x64, r32, rs, st,
                         itol, gtol, rb);
    else
        CF_STREAM_LAUNCH(k_refine_residual_carry<3>, g, b, x64, r32, rs, st,
                         itol, gtol, rb);
}

// The two-cell (FP32) tile kernels come in a periodic-x instantiation,
// which also reads the wrapped first cell of an odd row, and a plain one.
template <class T, bool PX>
static void dir_spmv3_t(const Geo& g, const T* r, const T* p_old, T* p_new, PcgState* st,
                        RedBuf rb, hipStream_t s)
{
    hipLaunchKernelGGL((k_pcg_dir_spmv3<T, cpl_of<T>(), PX>),
                       dim3(tile3_blocks<cpl_of<T>()>(g)), dim3(kTileBlock), 0, s, g,
                       tile3_grid<cpl_of<T>()>(g), r, p_old, p_new, st, rb);
}

template <class T, bool PX, int XM, bool R32>
static void update3_t(const Geo& g, T* x, T* r, const T* p, const T* p_lag, float* r32,
                      PcgState* st, RedBuf rb, hipStream_t s)
{
    hipLaunchKernelGGL((k_pcg_update3<T, cpl_of<T>(), PX, XM, R32>),
                       dim3(tile3_blocks<cpl_of<T>()>(g)), dim3(kTileBlock), 0, s, g,
                       tile3_grid<cpl_of<T>()>(g), x, r, p, p_lag, r32, st, rb);
}

template <class T, bool PX, bool R32>
static void update3_x(const Geo& g, T* x, T* r, const T* p, const T* p_lag, float* r32,
                      PcgState* st, RedBuf rb, hipStream_t s, int xmode)
{
    if (xmode == X_EACH) {
        update3_t<T, PX, X_EACH, R32>(g, x, r, p, p_lag, r32, st, rb, s);
        return;
    }
    if (xmode == X_SKIP) {
        update3_t<T, PX, X_SKIP, R32>(g, x, r, p, p_lag, r32, st, rb, s);
        return;
    }
    if (xmode == X_PAIR) {
        if (!p_lag || p_lag == p)
            throw CfError(CF_EINVAL, "X_PAIR update needs the previous direction buffer");
        update3_t<T, PX, X_PAIR, R32>(g, x, r, p, p_lag, r32, st, rb, s);
        return;
    }
    throw CfError(CF_EINVAL, "x mode not available for this PCG update");
}

void launch_pcg_dir_spmv_z32(const Geo& g, const float* z, const double* p_old, double* p_new,
                             PcgState* st, RedBuf rb, hipStream_t s)
{
    if (g.dim != 3)
        throw CfError(CF_EINVAL, "an FP32 z is a 3-D multigrid V-cycle's");
    hipLaunchKernelGGL((k_pcg_dir_spmv3<double, 1, false, float>), dim3(tile3_blocks<1>(g)),
                       dim3(kTileBlock), 0, s, g, tile3_grid<1>(g), z, p_old, p_new, st, rb);
}

template <class T>
void launch_pcg_dir_spmv(const Geo& g, const T* r, const T* p_old, T* p_new,
                         PcgState* st, RedBuf rb, hipStream_t s)
{
    if (g.dim == 2) {
        CF_STREAM_LAUNCH((k_pcg_dir_spmv<2, T>), g, r, p_old, p_new, st, rb);
        return;
    }
    if constexpr (cpl_of<T>() > 1)
        if (g.periodic[0]) {
            dir_spmv3_t<T, true>(g, r, p_old, p_new, st, rb, s);
            return;
        }
    dir_spmv3_t<T, false>(g, r, p_old, p_new, st, rb, s);
}

template <class T>
void launch_pcg_update(const Geo& g, T* x, T* r, const T* p, PcgState* st,
                       RedBuf rb, hipStream_t s, int xmode, const T* p_lag, float* r32)
{
    if (g.dim == 2) {
        if (xmode != X_EACH || r32)
            throw CfError(CF_EINVAL, "the 2-D PCG update takes x every iteration and "
                                     "writes no FP32 copy of r");
        CF_STREAM_LAUNCH((k_pcg_update<2, T>), g, x, r, p, st, rb);
        return;
    }
    if constexpr (cpl_of<T>() > 1) {
        if (r32)
            throw CfError(CF_EINVAL, "the FP32 PCG update writes no FP32 copy of r");
        if (g.periodic[0]) {
            update3_x<T, true, false>(g, x, r, p, p_lag, nullptr, st, rb, s, xmode);
            return;
        }
        update3_x<T, false, false>(g, x, r, p, p_lag, nullptr, st, rb, s, xmode);
    } else {
        if (r32)
            update3_x<T, false, true>(g, x, r, p, p_lag, r32, st, rb, s, xmode);
        else
            update3_x<T, false, false>(g, x, r, p, p_lag, nullptr, st, rb, s, xmode);
    }
}

template <class T>
void launch_pcg_xfix(const Geo& g, T* x, const T* p, const PcgState* st, hipStream_t s)
{
    CF_STREAM_LAUNCH(k_pcg_xfix<T>, g, x, p, st);
}

int reduction_blocks_max(const Geo& g)
{
    // the largest tile grid (up to 64 cells along x, FP32 pairs have as many
    // tiles and chunks half as deep)
    const int t1 = g.dim == 3 ? tile3_blocks<1>(g) : 0;
    const int t2 = g.dim == 3 ? tile3_blocks<2>(g) : 0;
    const int t = t1 > t2 ? t1 : t2;
    return t > kRedBlocks ? t : kRedBlocks;
}

template void launch_pcg_dir_spmv<double>(const Geo&, const double*,
                                          const double*, double*, PcgState*,
                                          RedBuf, hipStream_t);
template void launch_pcg_dir_spmv<float>(const Geo&, const float*, const float*,
                                         float*, PcgState*, RedBuf, hipStream_t);
template void launch_pcg_update<double>(const Geo&, double*, double*,
                                        const double*, PcgState*, RedBuf,
                                        hipStream_t, int, const double*, float*);
template void launch_pcg_update<float>(const Geo&, float*, float*, const float*,
                                       PcgState*, RedBuf, hipStream_t, int, const float*,
                                       float*);
template void launch_pcg_xfix<double>(const Geo&, double*, const double*, const PcgState*,
                                      hipStream_t);
template void launch_pcg_xfix<float>(const Geo&, float*, const float*, const PcgState*,
                                     hipStream_t);

void launch_refine_init(const Geo& g, const double* b, double* x64,
                        float* r32, RefineState* rs, RedBuf rb, hipStream_t s)
{
    CF_STREAM_LAUNCH(k_refine_init, g, b, x64, r32, rs, rb);
}

void launch_refine_add(const Geo& g, double* x64, float* d32, hipStream_t s)
{
    CF_STREAM_LAUNCH(k_refine_add, g, x64, d32);
}

void launch_refine_residual(const Geo& g, const double* b, const double* x64,
                            float* r32, RefineState* rs, RedBuf rb,
                            hipStream_t s)
{
    if (g.dim == 2)
        CF_STREAM_LAUNCH(k_refine_residual<2>, g, b, x64, r32, rs, rb);
    else
        CF_STREAM_LAUNCH(k_refine_residual<3>, g, b, x64, r32, rs, rb);
}

} // namespace cfmi
