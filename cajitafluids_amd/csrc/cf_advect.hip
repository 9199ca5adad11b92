// cf_advect.hip -- semi-Lagrangian advection for gfx950.
#include <hip/hip_runtime.h>

#include "cf_stream.hpp"

namespace cfmi
{

// ---- advection: TimeIntegrator::advect for every entity in one launch ------
// (src/TimeIntegrator.hpp:81-116): each lane owns one (i, j, k) of the union
// of the owned boxes and advects every entity owning that index.
//
// Occupancy: the 3-D kernels with linear velocity sampling keep the 64
// cubic taps of a field sample in flight and would take 146 VGPRs (3 waves
// per SIMD); capping them at 128 VGPRs (4 waves, a 36-byte spill) ran 256^3
// in 3.0 ms instead of 4.15 (64 x 4 x 1 blocks).  Higher caps spill more than
// they gain (5 waves: 4.2 ms, 6: 5.2 ms).
template <int DIM, int VORDER>
constexpr int advect_min_waves()
{
    return DIM == 3 && VORDER == 1 ? 4 : 1;
}

template <int DIM, int FORDER, int VORDER>
__global__ __launch_bounds__(256, (advect_min_waves<DIM, VORDER>())) void k_advect(Geo g,
                                                                                 Fields cur,
                                                                                 Fields next)
{
    const int i = g.h + blockIdx.x * blockDim.x + threadIdx.x;
    const int j = g.h + blockIdx.y * blockDim.y + threadIdx.y;
    const int k = g.own_lo(2) + blockIdx.z * blockDim.z + threadIdx.z;
    const int l[3] = {i, j, k};
    const double* u = cur.e[1];
    const double* v = cur.e[2];
    const double* w = cur.e[3];
#pragma unroll
    for (int e = 0; e <= DIM; ++e) {
        bool own = true;
#pragma unroll
        for (int d = 0; d < DIM; ++d)
            own = own && l[d] < g.own_hi[e][d];
        if (!own)
            continue;
        double x0[3] = {0, 0, 0}, tr[3];
#pragma unroll
        for (int d = 0; d < DIM; ++d)
            x0[d] = coord(g, e, d, l[d]);
        rk3<DIM, VORDER>(g, u, v, w, x0, tr);
        next.e[e][g.idx(i, j, k)] =
            interpolate<DIM, FORDER>(g, e, cur.e[e], tr);
    }
}

static dim3 union_grid(const Geo& g, dim3 blk)
{
    const int ex = g.uni_hi[0] - g.h, ey = g.uni_hi[1] - g.h;
    const int ez = g.dim == 3 ? g.uni_hi[2] - g.h : 1;
    return dim3((ex + blk.x - 1) / blk.x, (ey + blk.y - 1) / blk.y, (ez + blk.z - 1) / blk.z);
}

// 3-D blocks of 32 x 4 x 2 points: two z planes share the cubic stencils in
// the CU's caches (2.88 against 3.0 ms for 64 x 4 x 1 at 256^3).
template <int DIM, int FORDER, int VORDER>
static void advect_t(const Geo& g, Fields cur, Fields next, hipStream_t s)
{
    const dim3 blk = DIM == 3 ? dim3(32, 4, 2) : dim3(64, 4, 1);
    hipLaunchKernelGGL((k_advect<DIM, FORDER, VORDER>), union_grid(g, blk), blk,
                       0, s, g, cur, next);
}

// ---- the 3-D kernel with linear velocity sampling -----------------------------
// A point's trace takes 9 velocity samples of 8 taps for each of its 4
// entities, its field sample 64 (cubic) or 8 taps.  Gathered from memory, all
// of them are 272 16-byte loads a point in the CU's texture units, and
// forming their 64-bit addresses is a third of the vector instructions.  Here
// a block of 32 x 4 x 4 points keeps u, v and w with a reach of 2 cells below
// and 3 above in LDS (72 KB, two blocks a CU) and takes the velocity samples
// and its u, v and w from there; only q's taps are gathered, at one 32-bit
// offset a lane from a uniform row pointer.  The samples of a trace point
// share the 6 splines its face and centre coordinates have.  Inside the
// window the clamp of a coordinate is the identity and is left out; a wave
// with a lane outside (a step of more than about a cell, a NaN) clamps and
// gathers that sample from memory.  The arithmetic of every value is
// interpolate's and rk3's, in their order.
//
// Bound by vector issue (73% of the cycles at 256^3, 2240 of its ~2700
// instructions a wave FP64 arithmetic).  The cubic kernel fills the 128
// registers of four waves a SIMD and spills 25 (56 bytes a lane), the linear
// one takes 102.  Cubic field, against k_advect: 256^3
// 2.69 -> 1.87 ms, 190 x 182 x 149 817 -> 590 us, 128^3 338 -> 226, 64^3 64 ->
// 44; steps of six cells, whose waves mostly gather, 255^3 2.54 -> 2.13 ms.
// Linear field: 200^3 930 -> 634 us, 64^3 45 -> 33; thin and long grids: 4 x 512
// x 512 737 -> 608, 512 x 512 x 4 125 -> 103, 8 x 8 x 4096 105 -> 83.
// Blocks of 1024 with q in the window too: 2.06 ms (one block a CU: nothing
// runs while it loads).  256 points: one wave less per SIMD.
//
// Grids of fewer blocks than CUs take k_advect, whose 256-point blocks spread
// wider and wait for no window (24^3 18.7 against 21.8 us, 32^3 28.7 against
// 31.5; 48^3, 288 blocks, 37.0 against 31.1), and so do arrays of 4 GiB and
// more (about 800^3): their offsets do not fit 32 bits.
namespace advwin
{
constexpr int BX = 32, BY = 4, BZ = 4; // points of a block
constexpr int RL = 2, RH = 3;          // reach of the window below and above
constexpr int WX = BX + RL + RH, WY = BY + RL + RH, WZ = BZ + RL + RH;
constexpr int NT = BX * BY * BZ;
constexpr int NW = WX * WY * WZ;
__host__ __device__ constexpr int extent(int d)
{
    return d == 0 ? WX : d == 1 ? WY : WZ;
}
} // namespace advwin

// What the kernel needs of Geo, few enough scalars to stay in registers.  An
// axis has two kinds of coordinate: a face entity's (its normal axis) and a
// centre entity's; F selects.
struct AdvArgs
{
    Fields cur, next;
    double x0[2][3], rdx[2][3]; // [F][d]: Geo::x0, Geo::rdx
    double dx, dt;
    int n[3], h, faces[3];      // faces[d]: owned face layers along d beyond n
    int quirk;
    int nbx, nby, work;
    int extra[3];               // blocks of the layers past full blocks, summed over axes
    unsigned sx8, px8, pz8;     // byte offset of (0, 0, 0), byte strides
    int64_t px, pxy;
};

struct AdvWin
{
    const double* win; // u, v, w of the window in LDS
    unsigned base;     // byte offset of local index (0, 0, 0) in it (mod 2^32)
    // a sample whose face (linear) or own (cubic) coordinates xi have
    // |xi - mid| <= half on every axis is inside
    double mid[3], half[3];
};

// A block-uniform value, moved to scalar registers (the empty asm hides that
// it is uniform, or the move is dropped).  The lane reads are the compiler's,
// with the wait states they need after the write of what they read and before
// their result's use.
__device__ __forceinline__ double uniform(double v)
{
    int lo = __double2loint(v), hi = __double2hiint(v);
    asm("" : "+v"(lo), "+v"(hi));
    return __hiloint2double(__builtin_amdgcn_readfirstlane(hi),
                            __builtin_amdgcn_readfirstlane(lo));
}

// 8 bytes at a 32-bit byte offset from a uniform pointer.
__device__ __forceinline__ double at32(const double* __restrict__ p, unsigned off)
{
    return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(p) + off);
}

template <int F>
__device__ __forceinline__ double coord_of(const AdvArgs& g, int d, double p)
{
    return (p - g.x0[F][d]) * g.rdx[F][d];
}
template <int F, int ORDER>
__device__ __forceinline__ double clamp_of(const AdvArgs& g, int d, double xi)
{
    const int ext = g.n[d] + 2 * g.h + F;
    return fmin(fmax(xi, ORDER == 1 ? 0.0 : 1.0), (double)(ext - (ORDER == 1 ? 2 : 3)));
}
__device__ __forceinline__ unsigned win_at(const AdvWin& a, int sx, int sy, int sz)
{
    using namespace advwin;
    return a.base + (unsigned)(__mul24(sz, 8 * WX * WY) + __mul24(sy, 8 * WX) + 8 * sx);
}
// The window's element at byte offset `off` plus q elements.
__device__ __forceinline__ double win_get(const AdvWin& a, unsigned off, int q)
{
    return reinterpret_cast<const double*>(reinterpret_cast<const char*>(a.win) + off)[q];
}
// The offset of the next plane, kept from folding into the loads' own
// offsets, which reach 255 elements: the rows of a plane share one address.
__device__ __forceinline__ unsigned next_plane(unsigned off)
{
    off += 8u * advwin::WX * advwin::WY;
    asm("" : "+v"(off));
    return off;
}
__device__ __forceinline__ unsigned mem_at(const AdvArgs& g, int sx, int sy, int sz)
{
    return g.sx8 + 8u * sx + g.px8 * sy + g.pz8 * sz;
}

// velocity<3, 1> at x.
__device__ __forceinline__ void velocity_win(const AdvArgs& g, const AdvWin& a,
                                             const double (&x)[3], double (&vel)[3])
{
    using namespace advwin;
    double fx[3], cx[3];
    bool in = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        fx[d] = coord_of<1>(g, d, x[d]);
        cx[d] = coord_of<0>(g, d, x[d]);
        in &= fabs(fx[d] - a.mid[d]) <= a.half[d];
    }
    const bool lds = __ballot(!in) == 0;
    if (!lds) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            fx[d] = clamp_of<1, 1>(g, d, fx[d]);
            cx[d] = clamp_of<0, 1>(g, d, cx[d]);
        }
    }
    int fs[3], cs[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        fs[d] = (int)fx[d];
        cs[d] = (int)cx[d];
    }
    double t[3][2][2][2];
    if (lds) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            unsigned at = 8u * c * NW + win_at(a, c == 0 ? fs[0] : cs[0], c == 1 ? fs[1] : cs[1],
                                               c == 2 ? fs[2] : cs[2]);
            asm("" : "+v"(at));
#pragma unroll
            for (int k = 0; k < 2; ++k, at = next_plane(at))
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    t[c][0][j][k] = win_get(a, at, j * WX);
                    t[c][1][j][k] = win_get(a, at, j * WX + 1);
                }
        }
    } else {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const unsigned at = mem_at(g, c == 0 ? fs[0] : cs[0], c == 1 ? fs[1] : cs[1],
                                       c == 2 ? fs[2] : cs[2]);
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const double* row = g.cur.e[c + 1] + (j * g.px + k * g.pxy);
                    t[c][0][j][k] = at32(row, at);
                    t[c][1][j][k] = at32(row + 1, at);
                    // keeps the two branches' loads apart (merged, they
                    // would all be flat loads)
                    asm volatile("" : "+v"(t[c][0][j][k]), "+v"(t[c][1][j][k]));
                }
        }
    }
    double fw[3][2], cw[3][2];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        // xi >= 0: its fraction is xi - (double)(int)xi exactly
        spline_of<1>(__builtin_amdgcn_fract(fx[d]), fw[d]);
        spline_of<1>(__builtin_amdgcn_fract(cx[d]), cw[d]);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const double(&wx)[2] = c == 0 ? fw[0] : cw[0];
        const double(&wy)[2] = c == 1 ? fw[1] : cw[1];
        const double(&wz)[2] = c == 2 ? fw[2] : cw[2];
        double val = 0.0;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const double wab = wx[i] * wy[j];
#pragma unroll
                for (int k = 0; k < 2; ++k)
                    val = fma(wab * wz[k], t[c][i][j][k], val);
            }
        vel[c] = val;
    }
}

// interpolate<3, ORDER> of the array of entity E at the logical coordinates
// xi before their clamp.
template <int ORDER, int E>
__device__ __forceinline__ double field_mem(const AdvArgs& g, const double (&xi)[3])
{
    constexpr int N = ORDER + 1;
    int s0[3];
    double w[3][N];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const double c = E == d + 1 ? clamp_of<1, ORDER>(g, d, xi[d])
                                    : clamp_of<0, ORDER>(g, d, xi[d]);
        s0[d] = (int)c - (ORDER == 1 ? 0 : 1);
        spline_of<ORDER>(__builtin_amdgcn_fract(c), w[d]);
    }
    const unsigned at = mem_at(g, s0[0], s0[1], s0[2]);
    double val = 0.0;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const double wab = w[0][i] * w[1][j];
#pragma unroll
            for (int k = 0; k < N; ++k)
                val = fma(wab * w[2][k], at32(g.cur.e[E] + (i + j * g.px + k * g.pxy), at), val);
        }
    return val;
}

// interpolate<3, ORDER> of the array of entity E at p.
template <int ORDER, int E>
__device__ __forceinline__ double field_win(const AdvArgs& g, const AdvWin& a,
                                            const double (&p)[3])
{
    using namespace advwin;
    constexpr int N = ORDER + 1;
    double xi[3];
    bool in = E > 0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        xi[d] = E == d + 1 ? coord_of<1>(g, d, p[d]) : coord_of<0>(g, d, p[d]);
        in &= fabs(xi[d] - a.mid[d]) <= a.half[d];
    }
    if (E == 0 || __ballot(!in) != 0) {
        double v = field_mem<ORDER, E>(g, xi);
        if (E > 0)
            asm volatile("" : "+v"(v)); // keeps the branches apart, as above
        return v;
    }
    int s0[3];
    double w[3][N];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        s0[d] = (int)xi[d] - (ORDER == 1 ? 0 : 1);
        spline_of<ORDER>(__builtin_amdgcn_fract(xi[d]), w[d]);
    }
    unsigned at[N];
    at[0] = 8u * (E > 0 ? E - 1 : 0) * NW + win_at(a, s0[0], s0[1], s0[2]);
    asm("" : "+v"(at[0]));
#pragma unroll
    for (int k = 1; k < N; ++k)
        at[k] = next_plane(at[k - 1]);
    double val = 0.0;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const double wab = w[0][i] * w[1][j];
#pragma unroll
            for (int k = 0; k < N; ++k)
                val = fma(wab * w[2][k], win_get(a, at[k], j * WX + i), val);
        }
    return val;
}

// Entity E at the point p (counted from the first owned), where it owns it.
template <int FORDER, int E>
__device__ __forceinline__ void advect_entity(const AdvArgs& g, const AdvWin& a,
                                              const int (&p)[3])
{
    const int l[3] = {g.h + p[0], g.h + p[1], g.h + p[2]};
    bool own = true;
    double x0[3], x[3], v0[3], v1[3], v2[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        own &= p[d] < g.n[d] + (E == d + 1 ? g.faces[d] : 0);
        // coord(): the face coordinate of local index 0 is the low corner
        x0[d] = g.x0[1][d] + ((double)l[d] + (E == d + 1 ? 0.0 : 0.5)) * g.dx;
    }
    if (!own)
        return;
    const double dt = g.dt;
    velocity_win(g, a, x0, v0);
#pragma unroll
    for (int d = 0; d < 3; ++d)
        x[d] = x0[d] - 0.5 * dt * v0[d];
    velocity_win(g, a, x, v1);
#pragma unroll
    for (int d = 0; d < 3; ++d)
        x[d] = x0[d] - 0.75 * dt * (g.quirk ? v0[d] : v1[d]);
    velocity_win(g, a, x, v2);
#pragma unroll
    for (int d = 0; d < 3; ++d)
        x[d] = x0[d] -
               dt * ((2.0 / 9.0) * v0[d] + (3.0 / 9.0) * v1[d] + (4.0 / 9.0) * v2[d]);
    *reinterpret_cast<double*>(reinterpret_cast<char*>(g.next.e[E]) +
                               mem_at(g, l[0], l[1], l[2])) = field_win<FORDER, E>(g, a, x);
}

template <int FORDER>
__global__ __launch_bounds__(advwin::NT, 4) void k_advect_win(AdvArgs g)
{
    using namespace advwin;
    __shared__ double win[3 * NW];
    const int t = threadIdx.x;
    AdvWin a;
    a.win = win;
    int p[3]; // the lane's point, counted from the first owned
    const int ex8 = (g.extra[2] + 7) & ~7;
    if ((int)blockIdx.x >= ex8) {
        // an XCD takes consecutive blocks: their windows overlap in its L2
        const int bi = blockIdx.x - ex8;
        const int L = (bi & 7) * ((gridDim.x - ex8) >> 3) + (bi >> 3);
        if (L >= g.work)
            return;
        const int b[3] = {L % g.nbx, L / g.nbx % g.nby, L / g.nbx / g.nby};
        const int o[3] = {g.h + b[0] * BX - RL, g.h + b[1] * BY - RL, g.h + b[2] * BZ - RL};
        a.base = 0u - 8u * (unsigned)((o[2] * WY + o[1]) * WX + o[0]);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            // Every tap inside the window and the arrays, and the clamps the
            // identity: max(o, 0) + 1 <= xi <= min(o + W - 2, n + 2h - 3)
            // does for a linear sample of face and centre entities at face
            // coordinate xi, and for a cubic one at its own.  A 1/1024 cell
            // inside both ends.
            const double lo = (double)(max(o[d], 0) + 1);
            const double hi = (double)min(o[d] + extent(d) - 2, g.n[d] + 2 * g.h - 3);
            a.mid[d] = uniform(0.5 * (hi + lo));
            a.half[d] = uniform(0.5 * (hi - lo) - 0x1p-10);
        }
        // the window's elements; its lanes past the arrays' ends read the
        // last element, which no sample inside the window takes from there
        constexpr int NR = (NW + NT - 1) / NT;
        double v[NR][3];
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int q = min(t + r * NT, NW - 1);
            const int x = min(max(o[0] + q % WX, 0), g.n[0] + 2 * g.h);
            const int y = min(max(o[1] + q / WX % WY, 0), g.n[1] + 2 * g.h);
            const int z = min(max(o[2] + q / (WX * WY), 0), g.n[2] + 2 * g.h);
            const unsigned at = mem_at(g, x, y, z);
#pragma unroll
            for (int c = 0; c < 3; ++c)
                v[r][c] = at32(g.cur.e[c + 1], at);
        }
#pragma unroll
        for (int r = 0; r < NR; ++r)
            if (t + r * NT < NW) {
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    win[c * NW + t + r * NT] = v[r][c];
            }
        __syncthreads();
        p[0] = b[0] * BX + t % BX;
        p[1] = b[1] * BY + t / BX % BY;
        p[2] = b[2] * BZ + t / (BX * BY);
    } else {
        // A wall axis owns one more face layer than cells.  Where the cells
        // fill the blocks along it, extra blocks, the grid's first, take that
        // layer from memory (blocks with windows of their own cost 256^3 4%).
        const int q = blockIdx.x;
        if (q >= g.extra[2])
            return;
        const int d = q >= g.extra[1] ? 2 : q >= g.extra[0] ? 1 : 0;
        const int m = (q - (d == 0 ? 0 : d == 1 ? g.extra[0] : g.extra[1])) * NT + t;
        const int na = d == 0 ? g.n[1] : g.n[0];
        const int pa = m % na, pb = m / na;
        p[0] = d == 0 ? g.n[0] : pa;
        p[1] = d == 0 ? pa : d == 1 ? g.n[1] : pb;
        p[2] = d == 2 ? g.n[2] : pb;
        a.base = 0;
#pragma unroll
        for (int e = 0; e < 3; ++e) {
            a.mid[e] = 0.0;
            a.half[e] = -1.0; // no sample is inside
        }
    }
    advect_entity<FORDER, 0>(g, a, p);
    advect_entity<FORDER, 1>(g, a, p);
    advect_entity<FORDER, 2>(g, a, p);
    advect_entity<FORDER, 3>(g, a, p);
}

static int advect_win_blocks(const Geo& g)
{
    using namespace advwin;
    return ((g.n[0] + BX - 1) / BX) * ((g.n[1] + BY - 1) / BY) * ((g.n[2] + BZ - 1) / BZ);
}

template <int FORDER>
static void advect_win_t(const Geo& g, Fields cur, Fields next, hipStream_t s)
{
    using namespace advwin;
    AdvArgs a;
    a.cur = cur;
    a.next = next;
    for (int d = 0; d < 3; ++d) {
        for (int f = 0; f < 2; ++f) {
            a.x0[f][d] = g.x0[f ? d + 1 : 0][d];
            a.rdx[f][d] = g.rdx[f ? d + 1 : 0][d];
        }
        a.n[d] = g.n[d];
        a.faces[d] = g.periodic[d] ? 0 : 1;
    }
    a.dx = g.dx;
    a.dt = g.dt;
    a.h = g.h;
    a.quirk = (g.quirks & CF_QUIRK_RK3_V0) != 0;
    a.sx8 = (unsigned)g.sx * 8u;
    a.px8 = (unsigned)g.px * 8u;
    a.pz8 = (unsigned)(g.px * g.py) * 8u;
    a.px = g.px;
    a.pxy = g.px * g.py;
    // an axis' blocks also hold its extra face layer unless they are full
    a.nbx = (g.n[0] + BX - 1) / BX;
    a.nby = (g.n[1] + BY - 1) / BY;
    a.work = advect_win_blocks(g);
    int extra = 0;
    for (int d = 0; d < 3; ++d) {
        const int B = d == 0 ? BX : d == 1 ? BY : BZ;
        if (a.faces[d] && g.n[d] % B == 0)
            extra += (g.n[d == 0 ? 1 : 0] * g.n[d == 2 ? 1 : 2] + NT - 1) / NT;
        a.extra[d] = extra;
    }
    hipLaunchKernelGGL((k_advect_win<FORDER>), dim3((a.work + 7) / 8 * 8 + (extra + 7) / 8 * 8),
                       dim3(NT), 0, s, a);
}

void launch_advect(const Geo& g, Fields cur, Fields next, hipStream_t s)
{
    if (g.dim == 3 && g.vel_order == 1 && advect_win_blocks(g) >= 256 &&
        g.total * 8 < (int64_t)1 << 32) {
        if (g.field_order == 1)
            advect_win_t<1>(g, cur, next, s);
        else
            advect_win_t<3>(g, cur, next, s);
        return;
    }
    const int key = g.dim * 100 + g.field_order * 10 + g.vel_order;
    switch (key) {
    case 211: advect_t<2, 1, 1>(g, cur, next, s); break;
    case 231: advect_t<2, 3, 1>(g, cur, next, s); break;
    case 213: advect_t<2, 1, 3>(g, cur, next, s); break;
    case 233: advect_t<2, 3, 3>(g, cur, next, s); break;
    case 311: advect_t<3, 1, 1>(g, cur, next, s); break;
    case 331: advect_t<3, 3, 1>(g, cur, next, s); break;
    case 313: advect_t<3, 1, 3>(g, cur, next, s); break;
    case 333: advect_t<3, 3, 3>(g, cur, next, s); break;
    default: break;
    }
}

} // namespace cfmi
