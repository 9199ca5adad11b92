// cf_mg_fused.hip -- one multigrid level's pre-smoothing and restriction in
// one launch, and its prolongation and post-smoothing in another.
//
// A level's downward leg (x from zero by nu Jacobi sweeps, then the summed
// residual of each parent) was nu launches, its upward leg nu more, and each
// read and wrote the level's vectors: 16.25 words per cell of a large level
// (nu = 3), and five to eight microseconds a launch on a small one.  Here a
// leg reads its inputs once and writes its outputs once (2.125 and 3.125
// words): a block takes a column of cells wider than the ones it owns by
// one cell a side for every sweep, and carries the sweeps one plane behind
// each other as it marches along z.  The cells of the overlap are computed
// by each block that needs them, with the same operations, so every value
// has the bits of the sweep-by-sweep kernels (cf_mg.hip).
//
// Split: a wave spans the 64 columns of the block's x extent, a lane one
// column and RY rows of it; a block is NW such waves.  The x neighbours are
// the neighbour lanes (wave shifts), the z neighbours the lane's own last
// planes, the y neighbours the lane's own rows, and only a wave's first and
// last rows pass through LDS.  A sweep's plane is exchanged in the step
// after the one that made it, so a step needs one barrier.
//
// Couplings and diagonals depend on a cell's place along each axis only as
// first, last or in between (the extent of its box and the walls), so each
// level has tables of 4 classes per axis; a lane keeps its rows' entries for
// inner planes in registers.
//
// What bounds it: vector issue.  A block computes its overlap too (at 256^3
// 1.8 cells per owned cell) and all its waves wait for each other at every
// plane.  Measured, six launches before and two now: 256^3 level 0 in FP64
// 400 -> 202 us (0.7 GB, 3.5 TB/s), 190 x 182 x 149 level 0 in FP32 130 -> 66
// us, a 2-D level of 391 x 263 31 -> 13 us.  The first forms were slower than
// the six launches: rows at a wall on a path of their own (every wave of the
// block waits for them at each plane: 175 us a leg), and loads in flight
// copied at the loop's end (settle()).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "cf_mg.hpp"
#include "cf_solver.hpp"
#include "cf_stream.hpp"

namespace cfmi
{

namespace
{

// Rows per lane.  Two: the two rows of a parent.  With four a lane's sweeps
// no longer fit the registers of three waves a SIMD (256^3, level 0, down and
// up in FP64: 121 and 313 us against 113 and 121).
constexpr int RY = 2;

// Waves per block of the large levels, all resident at once: as many as the registers of a leg
// allow (FP32 16 against 12: 29 and 39 against 34 and 43 us, 190 x 182 x 149).
template <class T, bool UNI>
constexpr int waves_of()
{
    return std::is_same<T, float>::value || UNI ? 16 : 12;
}
// Waves per block of the 3-D levels that fill the GPU no other way (tile_level).
constexpr int kSmallLeg = 8;
// Steps from a plane's loads to their use.
template <class T, bool UNI>
constexpr int ahead_of()
{
    return std::is_same<T, float>::value || !UNI ? 2 : 1;
}

// A lane's value from the lane below / above it (0 at the wave's ends).
__device__ __forceinline__ int lane_below(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, 0x138, 0xf, 0xf, true); // wave_shr:1
}
__device__ __forceinline__ int lane_above(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, 0x130, 0xf, 0xf, true); // wave_shl:1
}
__device__ __forceinline__ float shift_below(float v)
{
    return __int_as_float(lane_below(__float_as_int(v)));
}
__device__ __forceinline__ float shift_above(float v)
{
    return __int_as_float(lane_above(__float_as_int(v)));
}
__device__ __forceinline__ double shift_below(double v)
{
    return __hiloint2double(lane_below(__double2hiint(v)), lane_below(__double2loint(v)));
}
__device__ __forceinline__ double shift_above(double v)
{
    return __hiloint2double(lane_above(__double2hiint(v)), lane_above(__double2loint(v)));
}

// m in [0, n): the cell that index i of a periodic axis stands for
__device__ __forceinline__ int wrap_index(int i, int n)
{
    const int m = i % n;
    return m < 0 ? m + n : m;
}

// place of cell m of an axis of n cells: 1 first, 2 last, 3 both, 0 neither
__device__ __forceinline__ int axis_class(int m, int n)
{
    return (m == 0 ? 1 : 0) + (m == n - 1 ? 2 : 0);
}

// Element index of a lane with nothing to load or store: past the end of any
// plane, so the buffer access that uses it reads 0 or is dropped.
constexpr unsigned kNoCell = 0x1fffffffu;

// The block's place and a lane's constants.
template <class T>
struct Place
{
    int i0, j0, k0, k1, i1, j1; // owned cells: [i0, i1) x [j0, j1) x [k0, k1)
    int gi;                     // the lane's column
    int lane, w;
    int clx;                    // its class
    bool own_x, xm_cut, xp_cut;
    int gj0;                    // the wave's first row
    unsigned own_rows;          // bit q: row q is owned (wave-uniform)
    int rinfo[RY];              // class, and kCutLo / kCutHi (wave-uniform)
    int id[RY];                 // the cell's table entry on an inner plane
    unsigned at[RY], to[RY];    // elements in a plane: read, written
    unsigned par[RY];           // the parents' elements in their plane
    // operator entries on inner planes (one coupling: cx as row 0's, cy per
    // row and cz uniform)
    T diag[RY], wt[RY], cxm[RY], cxp[RY], cym[RY], cyp[RY], cz[RY];
    T s; // the level's one coupling (UNI)
};
constexpr int kCutLo = 4, kCutHi = 8;

// Stored plane of index k in [-n, 2 n) (-1 outside the domain).
__device__ __forceinline__ int plane_of(const MgFused& f, int k)
{
    const int n = f.n[2];
    if (f.periodic[2])
        return k < 0 ? k + n : (k >= n ? k - n : k);
    return k >= 0 && k < n ? k : -1;
}

// UNI: every coupling of the level is the same (padded levels).
template <class T, int H, int NW, bool UNI>
__device__ __forceinline__ bool place_block(const MgFused& f, const MgOpTab<T>* op,
                                            Place<T>& c)
{
    const int L = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (L >= f.work)
        return false;
    const int tx = L % f.tiles_x, rest = L / f.tiles_x;
    const int ty = rest % f.tiles_y, ch = rest / f.tiles_y;
    const int n0 = f.n[0], n1 = f.n[1];
    c.i0 = tx * f.core_x;
    c.i1 = tx == f.tiles_x - 1 ? n0 : c.i0 + f.core_x;
    c.j0 = ty * f.core_y;
    c.j1 = ty == f.tiles_y - 1 ? n1 : c.j0 + f.core_y;
    c.k0 = ch * f.kz;
    c.k1 = min(c.k0 + f.kz, f.n[2]);
    c.lane = threadIdx.x & (kWave - 1);
    c.w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    // no overlap on a wall's side; an even one below along y, so that a
    // parent's two rows are one lane's
    const int lox = c.i0 == 0 && !f.periodic[0] ? 0 : H;
    const int loy = c.j0 == 0 && !f.periodic[1] ? 0 : (H + 1) / 2 * 2;
    c.gi = c.i0 - lox + c.lane;
    const bool inx = f.periodic[0] || (c.gi >= 0 && c.gi < n0);
    const int mx = f.periodic[0] ? wrap_index(c.gi, n0) : (inx ? c.gi : 0);
    c.clx = inx ? axis_class(mx, n0) : 0;
    c.own_x = c.gi >= c.i0 && c.gi < c.i1;
    c.xm_cut = !f.periodic[0] && c.gi <= 0;
    c.xp_cut = !f.periodic[0] && c.gi >= n0 - 1;
    c.gj0 = c.j0 - loy + c.w * RY;
    c.own_rows = 0;
#pragma unroll
    for (int q = 0; q < RY; ++q) {
        const int gj = c.gj0 + q;
        const int my = f.periodic[1] ? wrap_index(gj, n1) : (gj >= 0 && gj < n1 ? gj : -1);
        const int cly = my < 0 ? 0 : axis_class(my, n1);
        const bool lo = !f.periodic[1] && gj <= 0, hi = !f.periodic[1] && gj >= n1 - 1;
        const bool in = inx && my >= 0;
        c.rinfo[q] = cly | (lo ? kCutLo : 0) | (hi ? kCutHi : 0);
        c.id[q] = in ? c.clx + 4 * cly : kMgOutside;
        const bool own = gj >= c.j0 && gj < c.j1;
        c.own_rows |= own ? 1u << q : 0u;
        c.at[q] = in ? (unsigned)(mx + (int)f.lv.sy * my) : kNoCell;
        c.par[q] = in ? (unsigned)((mx >> 1) + (int)f.pm.sy * (my >> 1)) : kNoCell;
        c.to[q] = own && c.own_x ? c.at[q] : kNoCell;
        c.diag[q] = op->diag[c.id[q]];
        c.wt[q] = op->w[c.id[q]];
        c.s = (T)f.coupling;
        c.cxm[q] = c.xm_cut ? (T)0 : (UNI ? c.s : op->cx[cly]);
        c.cxp[q] = c.xp_cut ? (T)0 : (UNI ? c.s : op->cx[cly]);
        c.cym[q] = lo ? (T)0 : (UNI ? c.s : op->cy[c.clx]);
        c.cyp[q] = hi ? (T)0 : (UNI ? c.s : op->cy[c.clx]);
        c.cz[q] = UNI ? c.s : op->cz[c.clx + 4 * cly];
    }
    return true;
}

// A plane of a vector as a buffer: stored plane m of `sz` elements' stride
// holding `len` elements, or one of none (m < 0): reads give 0, writes are
// dropped.  So are those of kNoCell.
using Buffer = __amdgpu_buffer_rsrc_t;
template <class TV>
__device__ __forceinline__ Buffer plane_buffer(const TV* v, int m, unsigned stride, unsigned len)
{
    const uint64_t off = (uint64_t)(unsigned)(m < 0 ? 0 : m) * (stride * (unsigned)sizeof(TV));
    const char* base = reinterpret_cast<const char*>(v) + off;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0,
                                             m < 0 ? 0 : (int)(len * (unsigned)sizeof(TV)),
                                             0x00020000);
}
typedef unsigned U32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void buffer_get(Buffer r, unsigned e, double& v)
{
    v = __builtin_bit_cast(double, (U32x2)__builtin_amdgcn_raw_buffer_load_b64(r, e * 8u, 0, 0));
}
__device__ __forceinline__ void buffer_get(Buffer r, unsigned e, float& v)
{
    v = __builtin_bit_cast(float, (unsigned)__builtin_amdgcn_raw_buffer_load_b32(r, e * 4u, 0, 0));
}
__device__ __forceinline__ void buffer_put(Buffer r, unsigned e, double v)
{
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U32x2, v), r, e * 8u, 0, 0);
}
__device__ __forceinline__ void buffer_put(Buffer r, unsigned e, float v)
{
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, e * 4u, 0, 0);
}
// A loaded value in a register of its own.  The copy is opaque, so that a
// prefetch buffer's register is free when its next load is issued and the
// loop needs no copy of a value still in flight (which would wait for it).
__device__ __forceinline__ double settle(double v)
{
    double r;
    asm("v_mov_b64 %0, %1" : "=v"(r) : "v"(v));
    return r;
}
__device__ __forceinline__ float settle(float v)
{
    float r;
    asm("v_mov_b32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}
template <class TV>
__device__ __forceinline__ void get_rows(Buffer r, const unsigned (&e)[RY], TV (&v)[RY])
{
#pragma unroll
    for (int q = 0; q < RY; ++q)
        buffer_get(r, e[q], v[q]);
}

// Class of plane k along z: as axis_class, 4 outside the domain.
__device__ __forceinline__ int plane_class(const MgFused& f, int k)
{
    const int m = plane_of(f, k);
    return m < 0 ? 4 : axis_class(m, f.n[2]);
}

// y = A v on one plane of the lane's rows: v the plane, vm and vp the planes
// below and above, up and dn the rows beside the wave's.  The stencil order
// and the zero couplings are those of the sweep kernels; a cell outside the
// domain has zero entries, so a sweep leaves its 0.
template <class T, int DIM>
__device__ __forceinline__ void apply_inner(const Place<T>& c, const T (&vm)[RY],
                                            const T (&v)[RY], const T (&vp)[RY], T up, T dn,
                                            T (&y)[RY])
{
#pragma unroll
    for (int q = 0; q < RY; ++q) {
        T a = c.diag[q] * v[q];
        a = fma_t<T>(c.cxm[q], shift_below(v[q]), a);
        a = fma_t<T>(c.cxp[q], shift_above(v[q]), a);
        a = fma_t<T>(c.cym[q], q == 0 ? up : v[q - 1], a);
        a = fma_t<T>(c.cyp[q], q == RY - 1 ? dn : v[q + 1], a);
        if constexpr (DIM == 3) {
            a = fma_t<T>(c.cz[q], vm[q], a);
            a = fma_t<T>(c.cz[q], vp[q], a);
        }
        y[q] = a;
    }
}

// The same on a plane that may be first, last or outside, with the entries
// from the tables; and the cells' Jacobi weights.
template <class T, bool UNI>
__device__ __forceinline__ void apply_outer(const MgFused& f, const MgOpTab<T>* op,
                                            const Place<T>& c, int k, const T (&vm)[RY],
                                            const T (&v)[RY], const T (&vp)[RY], T up, T dn,
                                            T (&y)[RY], T (&wt)[RY])
{
    const int clz = plane_class(f, k);
    const bool zm_cut = !f.periodic[2] && k <= 0, zp_cut = !f.periodic[2] && k >= f.n[2] - 1;
    const T cy = UNI ? c.s : op->cy[c.clx + 4 * (clz & 3)];
#pragma unroll
    for (int q = 0; q < RY; ++q) {
        const T cx = UNI ? c.s : op->cx[(c.rinfo[q] & 3) + 4 * (clz & 3)];
        wt[q] = op->w[c.id[q] + 16 * clz];
        T a = op->diag[c.id[q] + 16 * clz] * v[q];
        a = fma_t<T>(c.xm_cut ? (T)0 : cx, shift_below(v[q]), a);
        a = fma_t<T>(c.xp_cut ? (T)0 : cx, shift_above(v[q]), a);
        a = fma_t<T>(c.rinfo[q] & kCutLo ? (T)0 : cy, q == 0 ? up : v[q - 1], a);
        a = fma_t<T>(c.rinfo[q] & kCutHi ? (T)0 : cy, q == RY - 1 ? dn : v[q + 1], a);
        a = fma_t<T>(zm_cut ? (T)0 : c.cz[q], vm[q], a);
        a = fma_t<T>(zp_cut ? (T)0 : c.cz[q], vp[q], a);
        y[q] = a;
    }
}

// One sweep of a plane: out = fma(w, b - A v, v).  INNER: plane k is neither
// first, last nor outside.
template <bool INNER, class T, class TB, int DIM, bool UNI>
__device__ __forceinline__ void sweep_plane(const MgFused& f, const MgOpTab<T>* op,
                                            const Place<T>& c, int k, const T (&vm)[RY],
                                            const T (&v)[RY], const T (&vp)[RY],
                                            const TB (&b)[RY], T up, T dn, T (&out)[RY])
{
    T y[RY];
    if constexpr (INNER) {
        apply_inner<T, DIM>(c, vm, v, vp, up, dn, y);
#pragma unroll
        for (int q = 0; q < RY; ++q)
            out[q] = fma_t<T>(c.wt[q], (T)b[q] - y[q], v[q]);
    } else {
        T wt[RY];
        apply_outer<T, UNI>(f, op, c, k, vm, v, vp, up, dn, y, wt);
#pragma unroll
        for (int q = 0; q < RY; ++q)
            out[q] = fma_t<T>(wt[q], (T)b[q] - y[q], v[q]);
    }
}

// The residual of a plane, b - A v.
template <bool INNER, class T, class TB, int DIM, bool UNI>
__device__ __forceinline__ void residual_plane(const MgFused& f, const MgOpTab<T>* op,
                                               const Place<T>& c, int k, const T (&vm)[RY],
                                               const T (&v)[RY], const T (&vp)[RY],
                                               const TB (&b)[RY], T up, T dn, T (&out)[RY])
{
    T y[RY];
    if constexpr (INNER) {
        apply_inner<T, DIM>(c, vm, v, vp, up, dn, y);
    } else {
        T wt[RY];
        apply_outer<T, UNI>(f, op, c, k, vm, v, vp, up, dn, y, wt);
    }
#pragma unroll
    for (int q = 0; q < RY; ++q)
        out[q] = (T)b[q] - y[q];
}

// The lane's share of a parent's sum over its children, z, y, x order: the
// residuals of two rows of its column and of the column above (own_x lanes
// of even columns).
template <class T>
__device__ __forceinline__ void add_children(const MgFused& f, const Place<T>& c,
                                             const T (&res)[RY], double (&sum)[RY / 2])
{
    const bool x1 = c.gi + 1 < f.n[0];
#pragma unroll
    for (int p = 0; p < RY / 2; ++p) {
        const T a0 = res[2 * p], a1 = res[2 * p + 1];
        const T b0 = shift_above(a0), b1 = shift_above(a1);
        double s = sum[p] + (double)a0;
        s = x1 ? s + (double)b0 : s;
        if (c.gj0 + 2 * p + 1 < f.n[1]) {
            s = s + (double)a1;
            s = x1 ? s + (double)b1 : s;
        }
        sum[p] = s;
    }
}

template <class T, class TO>
__device__ __forceinline__ void store_parents(const MgFused& f, const Place<T>& c, int m,
                                              const double (&sum)[RY / 2], TO* __restrict__ bc)
{
    const Buffer r = plane_buffer(bc + f.pm.base, m, f.psz, f.plen);
#pragma unroll
    for (int p = 0; p < RY / 2; ++p) {
        // an owned row pair starts with an owned row
        const bool own = ((c.own_rows >> (2 * p)) & 1) && c.own_x && !(c.gi & 1);
        buffer_put(r, own ? c.par[2 * p] : kNoCell, (TO)sum[p]);
    }
}

// The first and last rows of every wave of one sweep's plane; wave w reads
// the last row of wave w - 1 and the first of w + 1 (0 beyond the block).
template <class T, int NW>
using EdgeRows = T[2][NW + 2][kWave];

template <class T, int NW>
__device__ __forceinline__ void put_edges(EdgeRows<T, NW>& e, const Place<T>& c, const T (&v)[RY])
{
    e[0][c.w + 1][c.lane] = v[0];
    e[1][c.w + 1][c.lane] = v[RY - 1];
}
template <class T, int NW>
__device__ __forceinline__ void get_edges(const EdgeRows<T, NW>& e, const Place<T>& c, T& up,
                                          T& dn)
{
    up = e[1][c.w][c.lane];
    dn = e[0][c.w + 2][c.lane];
}
// the rows beyond the block's first and last wave read as 0
template <class T, int NW>
__device__ __forceinline__ void clear_edges(EdgeRows<T, NW>& e)
{
    if (threadIdx.x < kWave) {
        e[1][0][threadIdx.x] = (T)0;
        e[0][NW + 1][threadIdx.x] = (T)0;
    }
}

__device__ __forceinline__ void finish_rz(PcgState* st, double rz)
{
    if (st->iter > 0)
        st->beta = rz / st->rho;
    st->rho = rz;
}

// Values a leg starts from on plane k: w b (down), or x plus alpha times the
// parent (up); 0 outside the domain, where all of these were read as 0.
template <bool INNER, class T, class TB, class TP, bool UP, int DIM>
__device__ __forceinline__ void start_plane(const MgFused& f, const MgOpTab<T>* op,
                                            const Place<T>& c, int k, const TB (&b)[RY],
                                            const T (&x)[RY], const TP (&xc)[RY], T alpha,
                                            T (&out)[RY])
{
    if constexpr (UP) {
#pragma unroll
        for (int q = 0; q < RY; ++q)
            out[q] = fma_t<T>(alpha, (T)xc[q], x[q]);
    } else if constexpr (INNER) {
#pragma unroll
        for (int q = 0; q < RY; ++q)
            out[q] = c.wt[q] * (T)b[q];
    } else {
        const int clz = plane_class(f, k);
#pragma unroll
        for (int q = 0; q < RY; ++q)
            out[q] = op->w[c.id[q] + 16 * clz] * (T)b[q];
    }
}

// The sweeps' planes a lane holds as the march stands at plane p.
template <class T, class TB, int NU>
struct Sweeps
{
    T V[NU][2][RY];      // sweep s: the plane before its last one, its last one
    TB B[NU + 1][RY];    // b of planes p, p - 1, ...
    T last[RY];          // the last sweep's plane (UP)
    double sum[RY / 2];  // the parents being summed, and finished (down)
    double sums[RY / 2];
    double hi[1], lo[1]; // r.z (RZ)
};

// One step: plane p enters; sweep s + 1 makes plane k = p - 1 - s from sweep
// s's planes k - 1, k, k + 1, for every s.
template <bool INNER, class T, class TB, class TP, int NU, bool UP, bool RZ, bool UNI, int NW>
__device__ __forceinline__ void leg_step(const MgFused& f, const MgOpTab<T>* op,
                                         const Place<T>& c, int p, T alpha,
                                         const T (&xn)[RY], const TP (&cn)[RY],
                                         const EdgeRows<T, NW> (&rd)[NU],
                                         EdgeRows<T, NW> (&wr)[NU], Sweeps<T, TB, NU>& S)
{
    T made[RY];
    start_plane<INNER, T, TB, TP, UP, 3>(f, op, c, p, S.B[0], xn, cn, alpha, made);
#pragma unroll
    for (int s = 0; s < NU; ++s) {
        const int k = p - 1 - s;
        T up, dn, out[RY];
        get_edges<T, NW>(rd[s], c, up, dn);
        put_edges<T, NW>(wr[s], c, made);
        if (UP || s < NU - 1) {
            sweep_plane<INNER, T, TB, 3, UNI>(f, op, c, k, S.V[s][0], S.V[s][1], made, S.B[s + 1],
                                             up, dn, out);
        } else {
            residual_plane<INNER, T, TB, 3, UNI>(f, op, c, k, S.V[s][0], S.V[s][1], made,
                                                S.B[s + 1], up, dn, out);
            // planes before the chunk are summed and dropped at the chunk's start
            add_children<T>(f, c, out, S.sum);
            if ((k & 1) || k == f.n[2] - 1) {
#pragma unroll
                for (int q = 0; q < RY / 2; ++q) {
                    S.sums[q] = S.sum[q];
                    S.sum[q] = 0.0;
                }
            }
        }
        if (UP && s == NU - 1) {
#pragma unroll
            for (int q = 0; q < RY; ++q)
                S.last[q] = out[q];
            if constexpr (RZ)
                if ((unsigned)(k - c.k0) < (unsigned)(c.k1 - c.k0)) {
#pragma unroll
                    for (int q = 0; q < RY; ++q) {
                        const bool own = c.to[q] != kNoCell;
                        dd_acc_prod<false>(S.hi[0], S.lo[0], own ? (double)S.B[s + 1][q] : 0.0,
                                           own ? (double)out[q] : 0.0);
                    }
                }
        }
#pragma unroll
        for (int q = 0; q < RY; ++q) {
            S.V[s][0][q] = S.V[s][1][q];
            S.V[s][1][q] = made[q];
            made[q] = out[q];
        }
    }
}

// A leg of a 3-D level.  UP = false: x = nu sweeps from zero on b, bc = the
// parents' summed residuals.  UP = true: xo = nu sweeps from x + alpha xc.
// RZ (level 0's upward leg): also r.z = b . xo, for beta and rho.  A plane's
// loads are issued one or two steps before the step that uses them, and a
// step's stores in the next step ahead of its loads, every one of them on
// every path, so that no step waits for younger memory traffic.
template <class T, class TB, class TP, int NU, bool UP, bool RZ, bool UNI, int NW>
__global__ __launch_bounds__(NW* kWave) void k_mg_leg3(
    MgFused f, const MgOpTab<T>* __restrict__ tab, const TB* __restrict__ b,
    const T* __restrict__ x, const TP* __restrict__ xc, T* __restrict__ xo, TP* __restrict__ bc,
    PcgState* st, RedBuf rb)
{
    constexpr int kThreads = NW * kWave;
    if (st->done)
        return;
    __shared__ MgOpTab<T> op;
    __shared__ EdgeRows<T, NW> edges[2][NU];
    for (int q = threadIdx.x; q < (int)(sizeof(MgOpTab<T>) / sizeof(T)); q += kThreads)
        reinterpret_cast<T*>(&op)[q] = reinterpret_cast<const T*>(tab)[q];
#pragma unroll
    for (int s = 0; s < NU; ++s) {
        clear_edges<T, NW>(edges[0][s]);
        clear_edges<T, NW>(edges[1][s]);
    }
    __syncthreads();
    Sweeps<T, TB, NU> S = {};
    Place<T> c;
    const bool active = place_block<T, NU, NW, UNI>(f, &op, c); // the same for the whole block
    if (active) {
        const T alpha = (T)f.alpha;
        constexpr int A = ahead_of<T, UNI>();
        T xn[A][RY] = {};
        TP cn[A][RY] = {};
        TB bn[A][RY] = {};
        const int p0 = c.k0 == 0 && !f.periodic[2] ? 0 : c.k0 - NU;
        const int p1 = c.k1 + NU; // steps of planes p0 .. p1 - 1
        const unsigned chunk = (unsigned)(c.k1 - c.k0);
        // steps with planes p - NU .. p all inner
        const unsigned inner = f.n[2] < NU + 3 ? 0u : (unsigned)(f.n[2] - 2 - NU);
        const TB* bl = b + f.lv.base;
        const T* xl = UP ? x + f.lv.base : nullptr;
        const TP* cl = UP ? xc + f.pm.base : nullptr;
        T* ol = xo + f.lv.base;
        auto load = [&](int p, int W) {
            const int m = p < p1 ? plane_of(f, p) : -1;
            get_rows<TB>(plane_buffer(bl, m, f.lsz, f.len), c.at, bn[W]);
            if constexpr (UP) {
                get_rows<T>(plane_buffer(xl, m, f.lsz, f.len), c.at, xn[W]);
                get_rows<TP>(plane_buffer(cl, m >> 1, f.psz, f.plen), c.par, cn[W]);
            }
        };
        auto store = [&](int p) { // what the step of plane p made
            const int k = p - (UP ? NU : NU - 1);
            const bool mine = (unsigned)(k - c.k0) < chunk;
            const Buffer o = plane_buffer(ol, mine ? k : -1, f.lsz, f.len);
#pragma unroll
            for (int q = 0; q < RY; ++q)
                buffer_put(o, c.to[q], UP ? S.last[q] : S.V[NU - 1][1][q]);
            if constexpr (!UP) {
                const int kp = p - NU;
                const bool done =
                    (unsigned)(kp - c.k0) < chunk && ((kp & 1) || kp == f.n[2] - 1);
                store_parents<T, TP>(f, c, done ? kp >> 1 : -1, S.sums, bc);
            }
        };
        auto step = [&](int p, auto parity) {
            constexpr int W = decltype(parity)::value; // edges written; W ^ 1 are read
            T xp[RY] = {};
            TP cp[RY] = {};
#pragma unroll
            for (int q = 0; q < RY; ++q) {
#pragma unroll
                for (int s = NU; s > 0; --s)
                    S.B[s][q] = S.B[s - 1][q];
                S.B[0][q] = settle(bn[W % A][q]);
                if constexpr (UP) {
                    xp[q] = settle(xn[W % A][q]);
                    cp[q] = settle(cn[W % A][q]);
                }
            }
            store(p - 1);
            load(p + A, W % A);
            if ((unsigned)(p - 1 - NU) < inner)
                leg_step<true, T, TB, TP, NU, UP, RZ, UNI, NW>(f, &op, c, p, alpha, xp, cp,
                                                              edges[W ^ 1], edges[W], S);
            else
                leg_step<false, T, TB, TP, NU, UP, RZ, UNI, NW>(f, &op, c, p, alpha, xp, cp,
                                                               edges[W ^ 1], edges[W], S);
            __syncthreads();
        };
        load(p0, 0);
        if constexpr (A > 1)
            load(p0 + 1, 1);
        // the first step reads the edge rows of planes of zeros
#pragma unroll
        for (int s = 0; s < NU; ++s)
            put_edges<T, NW>(edges[1][s], c, S.V[s][1]);
        __syncthreads();
        // two steps a turn, so that the planes rotate by renaming
#pragma unroll 1
        for (int p = p0; p < p1; p += 2) {
            step(p, std::integral_constant<int, 0>{});
            step(p + 1, std::integral_constant<int, 1>{});
        }
        // an odd number of steps ends with one past the chunk, whose planes
        // no store takes
        store(p0 + ((p1 - p0 + 1) / 2 * 2) - 1);
    }
    if constexpr (RZ) {
        dd_norm(S.hi[0], S.lo[0]);
        grid_reduce<1, kThreads>(S.hi, S.lo, rb, [&](double* sm) { finish_rz(st, sm[0]); });
    }
}

// A leg of a 2-D level: the same sweeps on the block's one plane.
template <class T, int NU, bool UP, bool RZ, bool UNI, int NW>
__global__ __launch_bounds__(NW* kWave) void k_mg_leg2(
    MgFused f, const MgOpTab<T>* __restrict__ tab, const T* __restrict__ b,
    const T* __restrict__ x, const T* __restrict__ xc, T* __restrict__ xo, T* __restrict__ bc,
    PcgState* st, RedBuf rb)
{
    constexpr int kThreads = NW * kWave;
    if (st->done)
        return;
    __shared__ MgOpTab<T> op;
    __shared__ EdgeRows<T, NW> edges[NU];
    for (int q = threadIdx.x; q < (int)(sizeof(MgOpTab<T>) / sizeof(T)); q += kThreads)
        reinterpret_cast<T*>(&op)[q] = reinterpret_cast<const T*>(tab)[q];
#pragma unroll
    for (int s = 0; s < NU; ++s)
        clear_edges<T, NW>(edges[s]);
    __syncthreads();
    double hi[1] = {0.0}, lo[1] = {0.0};
    Place<T> c;
    if (place_block<T, NU, NW, UNI>(f, &op, c)) {
        T v[RY], out[RY], x0[RY] = {}, c0[RY] = {}, none[RY] = {};
        T B[RY];
        get_rows<T>(plane_buffer(b + f.lv.base, 0, 0, f.len), c.at, B);
        if constexpr (UP) {
            get_rows<T>(plane_buffer(x + f.lv.base, 0, 0, f.len), c.at, x0);
            get_rows<T>(plane_buffer(xc + f.pm.base, 0, 0, f.plen), c.par, c0);
        }
        start_plane<true, T, T, T, UP, 2>(f, &op, c, 0, B, x0, c0, (T)f.alpha, v);
#pragma unroll
        for (int s = 0; s < NU; ++s) {
            put_edges<T, NW>(edges[s], c, v);
            __syncthreads();
            T up, dn;
            get_edges<T, NW>(edges[s], c, up, dn);
            if (UP || s < NU - 1) {
                sweep_plane<true, T, T, 2, UNI>(f, &op, c, 0, none, v, none, B, up, dn, out);
#pragma unroll
                for (int q = 0; q < RY; ++q)
                    v[q] = out[q];
                if (s == (UP ? NU - 1 : NU - 2)) {
                    const Buffer o = plane_buffer(xo + f.lv.base, 0, 0, f.len);
#pragma unroll
                    for (int q = 0; q < RY; ++q) {
                        buffer_put(o, c.to[q], v[q]);
                        if constexpr (RZ) {
                            const bool own = c.to[q] != kNoCell;
                            dd_acc_prod<false>(hi[0], lo[0], own ? (double)B[q] : 0.0,
                                               own ? (double)v[q] : 0.0);
                        }
                    }
                }
            } else {
                residual_plane<true, T, T, 2, UNI>(f, &op, c, 0, none, v, none, B, up, dn, out);
                double sum[RY / 2] = {};
                add_children<T>(f, c, out, sum);
                store_parents<T, T>(f, c, 0, sum, bc);
            }
        }
    }
    if constexpr (RZ) {
        dd_norm(hi[0], lo[0]);
        grid_reduce<1, kThreads>(hi, lo, rb, [&](double* sm) { finish_rz(st, sm[0]); });
    }
}

// Tiles of an axis: the cells a tile owns (even), and how many tiles.  A tile
// holds `ext` cells; a neighbour below costs `below` of them, one above
// `above`.  Walls cost none, so the last tile may be larger than a middle one.
void split_axis(int n, bool periodic, int ext, int below, int above, int& tiles, int& core)
{
    const int mid = (ext - below - above) / 2 * 2;
    if (!periodic && n <= ext) {
        tiles = 1;
        core = n;
        return;
    }
    tiles = periodic ? (n + mid - 1) / mid : (n - above + mid - 1) / mid;
    if (!periodic && tiles < 2)
        tiles = 2;
    core = ((n + tiles - 1) / tiles + 1) / 2 * 2;
    if (core > mid)
        core = mid;
}

// The tiling of a level: the waves of a block (`big`, or in 3-D kSmallLeg) and
// the planes of a chunk (even, so that a block has both children of a parent
// along z) that minimise the last CU's blocks times a block's steps times a
// step's time, which 8 waves take in 0.65 of 16's or 12's (1.2-1.35 us).  Half
// the rows a block cost a large level a third more overlap; a level that
// leaves CUs idle gets shorter steps.  us a leg, 16 or 12 waves and 8: 128^3
// 25.0, 29.1; 64^3 16.9, 12.2; 32^3 16.4, 11.6; 95 x 91 x 75 (boxes) 19.0,
// 16.8; 47 x 45 x 37 15.7, 13.0.
void tile_level(MgFused& f, int nu, int big)
{
    double best = 1e30;
    for (int waves : {big, kSmallLeg}) {
        if (waves != big && f.dim == 2)
            break;
        MgFused t = f;
        t.waves = waves;
        split_axis(t.n[0], t.periodic[0], kWave, nu, nu, t.tiles_x, t.core_x);
        split_axis(t.n[1], t.periodic[1], RY * waves, (nu + 1) / 2 * 2, nu, t.tiles_y, t.core_y);
        const int tiles = t.tiles_x * t.tiles_y;
        for (int kz = 2;; kz += 2) {
            t.kz = t.dim == 3 ? kz : 1;
            t.nchunk = (t.n[2] + t.kz - 1) / t.kz;
            t.work = tiles * t.nchunk;
            const double cost = (double)((t.work + 255) / 256) * (t.kz + 2 * nu) *
                                (waves == big ? 1.0 : 0.65);
            if (cost < best && t.work <= kRedBlocks) {
                best = cost;
                f = t;
            }
            if (t.dim == 2 || kz >= t.n[2])
                break;
        }
    }
}

} // namespace

bool mg_fused_level(const MgLev& L, int nu, bool f32, double coupling, MgFused& f)
{
    if (nu != 2 && nu != 3)
        return false;
    for (int d = 0; d < L.dim; ++d)
        if (!L.coarsen[d])
            return false;
    f.dim = L.dim;
    for (int d = 0; d < 3; ++d) {
        f.n[d] = L.n[d];
        f.periodic[d] = L.periodic[d];
    }
    f.alpha = L.alpha;
    f.coupling = coupling;
    f.work = 0;
    tile_level(f, nu,
               f32 ? waves_of<float, true>()
                   : (coupling != 0.0 ? waves_of<double, true>() : waves_of<double, false>()));
    return f.work > 0;
}

namespace
{

template <class T, class TB, class TP, int NU, bool UP, bool RZ, bool UNI>
void leg3(const MgFused& f, const MgOpTab<T>* tab, const TB* b, const T* x, const TP* xc, T* xo,
          TP* bc, PcgState* st, RedBuf rb, hipStream_t s)
{
    const dim3 grid((f.work + 7) / 8 * 8), block(f.waves * kWave);
    if (f.waves == kSmallLeg)
        hipLaunchKernelGGL((k_mg_leg3<T, TB, TP, NU, UP, RZ, UNI, kSmallLeg>), grid, block, 0, s,
                           f, tab, b, x, xc, xo, bc, st, rb);
    else
        hipLaunchKernelGGL((k_mg_leg3<T, TB, TP, NU, UP, RZ, UNI, waves_of<T, UNI>()>), grid,
                           block, 0, s, f, tab, b, x, xc, xo, bc, st, rb);
}

template <int NU, bool UP, bool RZ, bool UNI>
void leg2(const MgFused& f, const MgOpTab<double>* tab, const double* b, const double* x,
          const double* xc, double* xo, double* bc, PcgState* st, RedBuf rb, hipStream_t s)
{
    constexpr int NW = waves_of<double, UNI>();
    hipLaunchKernelGGL((k_mg_leg2<double, NU, UP, RZ, UNI, NW>), dim3((f.work + 7) / 8 * 8),
                       dim3(NW * kWave), 0, s, f, tab, b, x, xc, xo, bc, st, rb);
}

// An FP64 leg of any level; nu = NU.
template <int NU, bool UP>
void leg64(const MgFused& f, const MgOpTab<double>* tab, bool rz, const double* b,
           const double* x, const double* xc, double* xo, double* bc, PcgState* st, RedBuf rb,
           hipStream_t s)
{
    const bool uni = f.coupling != 0.0;
    using D = double;
    if (UP && rz) // level 0 has one coupling
        (f.dim == 2 ? leg2<NU, UP, UP, true> : leg3<D, D, D, NU, UP, UP, true>)(
            f, tab, b, x, xc, xo, bc, st, rb, s);
    else if (uni)
        (f.dim == 2 ? leg2<NU, UP, false, true> : leg3<D, D, D, NU, UP, false, true>)(
            f, tab, b, x, xc, xo, bc, st, rb, s);
    else
        (f.dim == 2 ? leg2<NU, UP, false, false> : leg3<D, D, D, NU, UP, false, false>)(
            f, tab, b, x, xc, xo, bc, st, rb, s);
}

} // namespace

void launch_mg_down(const MgFused& f, const MgOp* op, int nu, const double* b, double* x,
                    double* bc, PcgState* st, RedBuf rb, hipStream_t s)
{
    (nu == 2 ? leg64<2, false> : leg64<3, false>)(f, &op->d, false, b, nullptr, nullptr, x, bc,
                                                  st, rb, s);
}

void launch_mg_up(const MgFused& f, const MgOp* op, int nu, bool rz, const double* b,
                  const double* x, const double* xc, double* xo, PcgState* st, RedBuf rb,
                  hipStream_t s)
{
    if (rz && f.coupling == 0.0)
        throw CfError(CF_EINVAL, "the leg that reduces r.z is level 0's");
    (nu == 2 ? leg64<2, true> : leg64<3, true>)(f, &op->d, rz, b, x, xc, xo, nullptr, st, rb, s);
}

void launch_mg_down_f32(const MgFused& f, const MgOp* op, int nu, const float* b, float* x,
                        double* bc, float* bc32, PcgState* st, RedBuf rb, hipStream_t s)
{
    using F = float;
    if (bc32)
        (nu == 2 ? leg3<F, F, F, 2, false, false, true> : leg3<F, F, F, 3, false, false, true>)(
            f, &op->f, b, nullptr, nullptr, x, bc32, st, rb, s);
    else
        (nu == 2 ? leg3<F, F, double, 2, false, false, true>
                 : leg3<F, F, double, 3, false, false, true>)(f, &op->f, b, nullptr, nullptr, x,
                                                              bc, st, rb, s);
}

void launch_mg_up_f32(const MgFused& f, const MgOp* op, int nu, const float* b,
                      const double* r64, const float* x, const double* xc, const float* xc32,
                      float* xo, PcgState* st, RedBuf rb, hipStream_t s)
{
    using F = float;
    using D = double;
    if (!r64)
        (nu == 2 ? leg3<F, F, D, 2, true, false, true> : leg3<F, F, D, 3, true, false, true>)(
            f, &op->f, b, x, xc, xo, nullptr, st, rb, s);
    else if (xc32)
        (nu == 2 ? leg3<F, D, F, 2, true, true, true> : leg3<F, D, F, 3, true, true, true>)(
            f, &op->f, r64, x, xc32, xo, nullptr, st, rb, s);
    else
        (nu == 2 ? leg3<F, D, D, 2, true, true, true> : leg3<F, D, D, 3, true, true, true>)(
            f, &op->f, r64, x, xc, xo, nullptr, st, rb, s);
}

} // namespace cfmi
