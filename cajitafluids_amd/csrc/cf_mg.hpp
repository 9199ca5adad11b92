// cf_mg.hpp -- geometric multigrid preconditioner for the FP64 pressure
// solve: level descriptions and kernel launchers (cf_mg.hip), and the host
// hierarchy (cf_mg_host.cpp).
//
// Level 0 is the pressure grid in the handle's padded layout with the
// matrix-free operator.  Coarser levels are compact arrays (x fastest, no
// ghosts).  Their Galerkin operators P^T A P (P piecewise constant over the
// aggregation) are matrix-free too: a coarse cell is a box of level-0 cells,
// every level-0 coupling is s = dt / (rho dx^2), so
//   coupling to the -/+ e_d neighbour = -(area_d s)   (0 without neighbour)
//   diagonal                         = K s,
// where area_d is the number of level-0 faces between two neighbouring boxes
// along d (the product of the box's extents along the other axes) and K
// counts the box's boundary faces that are not SOLID domain walls.  These
// are the integer face counts the aggregation produces level by level,
// rounded once; the Jacobi weight is omega / (K s).
#pragma once

#include <hip/hip_runtime.h>

#include <memory>
#include <vector>

#include "cf_kernels.hpp"

namespace cfmi
{

constexpr int kMgMaxLevels = 24;
// The coarsest levels whose vectors (3 per level), tables and infos fit this
// much LDS, and whose largest leaves a thread at most kMgTailCells cells, run
// inside one workgroup (k_mg_tail).  Against 64 KB, where 16^3 cells ran as
// legs of their own: 256^3 V-cycle 15 us shorter.
constexpr int kMgTailLdsBytes = 150 * 1024;
constexpr int kMgTailThreads = 1024;
constexpr int kMgTailCells = 4;

// omega * (1 / diag) on level 0, by the cell's SOLID wall count.
struct MgTab
{
    double v[7];
};

// One compact level as the kernels see it.
struct MgLev
{
    int n[3];
    int coarsen[3];   // axis coarsened from this level to the next
    int periodic[3];
    int shift[3];     // a cell spans 2^shift[d] level-0 cells along d (fewer at the end)
    int n0[3];        // level-0 cells per axis
    int solid[3][2];  // SOLID domain ends of non-periodic axes
    int dim;
    int ncell;
    double s;         // dt / (rho dx^2)
    double omega;
    double alpha;     // coarse-correction scale: x = fma(alpha, x_parent, x)
};

// Linear index of the parent of cell (i, j, k) in the next level's array:
// base + i/2 + sy j/2 + sz k/2 (compact or padded layout).
struct MgParentMap
{
    int64_t base, sy, sz;
};

// A level's operator by the place of a cell along each axis (class 0 in
// between, 1 first, 2 last, 3 both): diagonal and Jacobi weight at
// cx + 4 cy + 16 cz, couplings along x at cy + 4 cz, along y at cx + 4 cz,
// along z at cx + 4 cy.  A row outside the domain has class kMgOutside in place
// of cx + 4 cy, a plane outside it class 4: entries of 0.
constexpr int kMgOutside = 64;
template <class T>
struct MgOpTab
{
    T diag[2 * kMgOutside + 1], w[2 * kMgOutside + 1], cx[16], cy[16], cz[16];
};
struct MgOp
{
    MgOpTab<double> d;
    MgOpTab<float> f; // the FP64 entries rounded
};

// A cell of those levels: x, y, z hold the elements of its -/+ neighbours
// along each axis in bits 0-12 and 13-25, counted from 1 (0: none, across a
// wall); x its class (MgOpTab) in bits 26-31; y in bits 26-28 whether its box
// has a second child along each axis; w its parent's element, and in bits
// 16-31 its first child's.
using MgTailInfo = int4;

// The levels that k_mg_tail runs (l0 .. last): their LDS offsets (level l's
// vectors from element off[l], the operator tables from off[last + 1], the
// cells' infos after them), and the global arrays it reads (B[l0]) and writes
// (res[l0]).
struct MgTail
{
    int l0, last, nu, coarse;
    MgLev lev[kMgMaxLevels];
    int off[kMgMaxLevels + 1];
    double* B[kMgMaxLevels];
    double* res[kMgMaxLevels];
    int info_at[kMgMaxLevels + 1]; // level l's cells in MgTailTop::info
};

// What k_mg_tail starts with, by value: the top level's right-hand side and
// cells, and what it copies to LDS.
struct MgTailTop
{
    int l0, last, n_top, n_all; // cells of level l0, MgTailInfo in all
    const double* b;
    const MgTailInfo* info; // of the levels from l0 on
    const MgOp* op;         // of every level
};

// Which of a level's two vectors k_mg_tail's downward leg leaves the residual
// in: x = w b in X, then nu - 1 sweeps and the residual, alternating.  The
// upward leg's nu sweeps from there end in X.
template <class P>
__host__ __device__ inline P mg_tail_residual(P X, P T, int nu)
{
    return nu & 1 ? T : X;
}

// One level's legs in a launch each (cf_mg_fused.hip): its cells and its
// parents' storage, and the tiling.
struct MgFused
{
    int dim, n[3], periodic[3];
    int tiles_x, core_x, tiles_y, core_y, nchunk, kz, work;
    int waves; // of a block
    double alpha;
    double coupling; // of every pair of neighbours, or 0 if they differ
    MgParentMap lv, pm;
    // elements from a plane's first owned cell to its last, and plane strides
    unsigned len, plen, lsz, psz;
};

// Source of the values a smoothing sweep reads:
//   first:   x = w b (the sweep from zero, computed on the fly)
//   plain:   x = xi
//   prolong: x = fma(alpha, xc[parent], xi)
enum MgSrc
{
    MG_FIRST = 0,
    MG_PLAIN = 1,
    MG_PROLONG = 2
};

// Padded levels by row kernels (level 0 of 2-D or thin grids, and small
// tiled levels): xo = fma(w, b - A x, x) with x from `src` (the parent's
// value read at pm, scaled by alpha); with rz, also r.z = b.xo reduced into
// st (beta = r.z / rho after the first iteration, rho = r.z).
// launch_mg0_first: x = w b alone (a single sweep from zero).
void launch_mg0_smooth(const Geo& g, const MgTab& wd0, int src, bool rz, const double* xi,
                       const double* b, MgParentMap pm, double alpha, const double* xc,
                       double* xo, PcgState* st, RedBuf rb, hipStream_t s);
void launch_mg0_first(const Geo& g, const MgTab& wd0, const double* b, double* x,
                      const PcgState* st, hipStream_t s);
// Next level's b1 = sum over children (z, y, x order) of (b - A x); c1: the
// next level's dims, pm: where its cells are stored.
void launch_mg0_resrestrict(const Geo& g, const MgLev& c1, MgParentMap pm, const double* x,
                            const double* b, double* b1, const PcgState* st, hipStream_t s);

// Tiled levels (3-D, every axis coarsened further): level 0 and the coarse
// levels of full 2^l boxes in a padded layout with their own Geo.  The same
// sweeps (the parent read through pm, scaled by alpha) and
// residual-restriction as z-marching tiles; gw is the level's geometry with
// the Jacobi table omega / diag.
bool mg_tiled3(const Geo& g);
void launch_mg_smooth3(const Geo& g, const Geo& gw, int src, bool rz, const double* xi,
                       const double* b, const double* xc, MgParentMap pm, double alpha,
                       double* xo, PcgState* st, RedBuf rb, hipStream_t s);
void launch_mg_resrestrict3(const Geo& g, const double* x, const double* b, double* bc,
                            MgParentMap pm, const PcgState* st, hipStream_t s);

// FP32 level 0 (3-D, marched), and level 1 when it is a marched tiled level:
// the same sweeps and restriction on FP32 vectors.  b32 = (float) r (launch_mg_cast32, or the PCG update); a sweep
// with rz reads r64 instead of b32 (its sweep uses (float) r64) and reduces
// r.z with the FP64 r; the restriction sums the FP32 residuals as doubles
// into the FP64 level 1; the prolongation rounds the FP64 parent to FP32.
void launch_mg_cast32(const Geo& g, const double* r, float* b32, const PcgState* st,
                      hipStream_t s);
void launch_mg0_first_f32(const Geo& g, const MgTab& wd0, const float* b, float* x,
                          const PcgState* st, hipStream_t s);
// xc32 (non-null): an FP32 parent level instead of xc; cpl: cells per lane
// (2 on level 0, 1 on an FP32 level 1).
void launch_mg_smooth3_f32(const Geo& g, const Geo& gw, int src, bool rz, const float* xi,
                           const float* b32, const double* r64, const double* xc,
                           const float* xc32, MgParentMap pm, double alpha, float* xo,
                           PcgState* st, RedBuf rb, hipStream_t s, int cpl);
// bc32 (non-null): the sums rounded into an FP32 level 1 instead of bc.
void launch_mg_resrestrict3_f32(const Geo& g, const float* x, const float* b, double* bc,
                                float* bc32, MgParentMap pm, const PcgState* st, hipStream_t s,
                                int cpl);

// Whole legs of a level whose axes are all coarsened, with nu = 2 or 3 sweeps
// (false otherwise); fills f but for the storage maps.  f32: the level runs in
// FP32; coupling: a padded level's, 0 on a compact one.  Down: x = nu sweeps
// from zero on b, bc the parents' right-hand side.  Up: xo = nu sweeps from
// x + alpha xc; with rz also r.z = b . xo as above.  FP32 levels: as the FP32
// sweeps below (r64: the rz leg's right-hand side).
bool mg_fused_level(const MgLev& L, int nu, bool f32, double coupling, MgFused& f);
void launch_mg_down(const MgFused& f, const MgOp* op, int nu, const double* b, double* x,
                    double* bc, PcgState* st, RedBuf rb, hipStream_t s);
void launch_mg_up(const MgFused& f, const MgOp* op, int nu, bool rz, const double* b,
                  const double* x, const double* xc, double* xo, PcgState* st, RedBuf rb,
                  hipStream_t s);
void launch_mg_down_f32(const MgFused& f, const MgOp* op, int nu, const float* b, float* x,
                        double* bc, float* bc32, PcgState* st, RedBuf rb, hipStream_t s);
void launch_mg_up_f32(const MgFused& f, const MgOp* op, int nu, const float* b,
                      const double* r64, const float* x, const double* xc, const float* xc32,
                      float* xo, PcgState* st, RedBuf rb, hipStream_t s);

// Compact levels.
void launch_mg_first(const MgLev& L, const double* b, double* x, const PcgState* st,
                     hipStream_t s);
void launch_mg_smooth(const MgLev& L, int src, const double* xi, const double* b,
                      const MgLev& C, const double* xc, double* xo, const PcgState* st,
                      hipStream_t s);
void launch_mg_resrestrict(const MgLev& F, const MgLev& C, const double* x, const double* b,
                           double* bc, const PcgState* st, hipStream_t s);
// One workgroup runs the V-cycle of levels t->l0 .. t->last in lds_bytes of LDS.
void launch_mg_tail(const MgTailTop& top, const MgTail* t_dev, size_t lds_bytes,
                    const PcgState* st, hipStream_t s);

// MG-PCG: r = b, x = 0, ||b|| (sets st->mg); and rho / beta from r.z.
void launch_mgpcg_init(const Geo& g, const double* b, double* x, double* r,
                       PcgState* st, double tol, int maxit, RedBuf rb, hipStream_t s);
void launch_mgpcg_rz(const Geo& g, const double* r, const double* z, PcgState* st,
                     RedBuf rb, hipStream_t s);

// The device hierarchy of one handle.
class Multigrid
{
  public:
    Multigrid(const Geo& g, const cf_config& cfg, hipStream_t s);
    ~Multigrid();
    // z = B r (one V-cycle), then rho / beta from r.z; returns the level-0
    // buffer that holds z (one of the two the hierarchy owns).  Kernels
    // return at once when st->done.
    const double* vcycle(const double* r, PcgState* st, RedBuf rb);
    // The same with level 0 on FP32 vectors (3-D grids with more than 2
    // cells per axis, f32_supported()), the coarser levels in FP64; z comes
    // back in FP32.  b32_ready: the caller has written (float) r into b32()
    // (the PCG update does), so the V-cycle skips its own cast.
    const float* vcycle32(const double* r, PcgState* st, RedBuf rb, bool b32_ready);
    bool f32_supported() const { return _nt >= 1 && _lev.size() >= 2; }
    // the FP32 level 0's right-hand side (null before the first FP32 V-cycle)
    float* b32() const;
    int levels() const { return (int)_lev.size(); }
    const MgLev& level(int l) const { return _lev[l]; }

  private:
    struct Buffers;
    const void* cycle(const double* r, PcgState* st, RedBuf rb, bool f32, bool b32_ready);
    void first(int l, const double* b, double* x, PcgState* st);
    void smooth(int l, int src, bool rz, const double* xi, const double* b, double* xo,
                PcgState* st, RedBuf rb);
    void resrestrict(int l, const double* x, const double* b, PcgState* st);
    // one FP32 sweep on level l (launch_mg_smooth3_f32)
    void smooth32(int l, int src, bool rz, const float* xi, const float* b32, const double* r,
                  float* xo, const float* xc32, PcgState* st, RedBuf rb);
    // level 1 runs in FP32 too (with level 0): it is a marched tile level
    bool f32_level1() const;
    bool marched(int l) const;
    const Geo& _g;
    hipStream_t _s;
    int _nu, _coarse;
    int _tail0;              // first level run by k_mg_tail
    size_t _tail_lds;        // its LDS bytes
    int _nt;                 // levels 0 .. _nt-1 run the z-marching tile kernels
    std::vector<Geo> _lg;    // Geo of each tiled level (padded layout)
    std::vector<Geo> _lgw;   // ... with the Jacobi table omega / diag
    std::vector<MgTab> _wt;  // level 0 and tiled levels: omega / diag by wall count
    std::vector<MgParentMap> _pm; // parent index of level l's cells in level l + 1
    std::vector<MgLev> _lev; // _lev[0]: level-0 dims and coarsening only
    // levels whose legs run as one launch each (tiling; work 0: the others)
    // [0]: in FP64, [1]: in FP32 (levels 0 and 1)
    std::vector<MgFused> _fz[2];
    bool fused(int l) const { return _fz[0][l].work > 0; }
    MgOp op_table(int l) const;
    void tail_infos(int l, std::vector<MgTailInfo>& out) const;
    size_t tail_lds(int l0) const;
    std::unique_ptr<Buffers> _buf;
};

// Sweep-count parity of one cycle on a level: the cycle starts in X and
// ends in T when odd.
__host__ __device__ inline int mg_level_swaps(bool last, int nu, int coarse)
{
    if (last)
        return coarse >= 2 ? coarse - 2 : 0;
    return (nu >= 2 ? nu - 2 : 0) + nu;
}

} // namespace cfmi
