// cf_pcg_coop.hip -- a whole FP64 PCG solve of a 2-D grid, or of a 3-D grid of
// up to about 100^3 cells, in one cooperative launch; on those 3-D grids also
// the FP32 iterations of a pass of a refined solve.
//
// A 2-D streaming iteration at 128^2-512^2 is two launches whose time goes
// to start-up, one sweep per lane group and the grid reduction's arrival
// chain (about 7.5 us each at 128^2), not to bandwidth.  Here one
// cooperative launch of G workgroups runs all iterations:
//   - workgroup g owns the rows [g R, g R + R) as a strip; lane t of it owns
//     strip cells t + NT m (m < CPT, x fastest); r, x and q = A p of those
//     cells stay in registers;
//   - the direction lives in the strip's LDS window: its rows, one halo row
//     above and below, and a one-cell ring in x.  Ring cells of periodic
//     axes are copies of the wrapped cells; the others hold a zero whose
//     sign is that of the coupling s, so that fma(s, ring, y) adds
//     s * ring = +0, the term fma(0, 0, y) the streaming kernels add across a
//     non-periodic boundary (the same bits for every y, -0 included);
//   - a halo row's direction is computed by the strip itself, by the same
//     expression, from its last one and the neighbour strip's boundary r,
//     which that strip publishes with the reduction below;
//   - each of an iteration's two reductions: a workgroup reduction, then the
//     workgroup's double-double partial published and every workgroup's
//     partials read and summed in one fixed order, so that every workgroup
//     holds the same alpha, beta and stop decision.  A wave of its own, with
//     no cells, does this part and the scalars (coop_scalars).
//
// What bounds it is the two exchanges' latency: a value travels as 64-bit
// words of 32 bits of it and the exchange's sequence number, stored and
// loaded at agent scope (past the L2s, which do not see each other's
// writes), and its readers poll the words themselves.  No store's completion
// is waited for, no separate flag is read, no fence is issued.  Measured per
// exchange (16 workgroups): 2.7 us with a flag per workgroup (store, its
// acknowledgement, flag, flag's poll, then the value's read), 2.1 us with the
// words, 1.9 us with the wave sums by lane moves instead of LDS permutes,
// 1.65 us with the workgroups on one XCD (every eighth block of the launch,
// while that many fit the GPU; the others return at once, and nothing but
// the latency depends on where the blocks really run).  Polling the XCD's own
// L2 (with an invalidate or an atomic a poll) was no faster than agent scope.
//
// Beside them, a strip's own chain, 2.9 -> 2.0 us of an iteration: sums whose
// steps wait for one addition (dd_merge), r.r and r.z summed in alternate
// lanes, the stop test's root and division beside the next direction, halo
// cells kept as D^-1 r, and no halo work where no strip is next.
//
// Every value is the streaming kernels' expression on the same operands, so
// x, r, the direction and the state come out with the same bits.  A poll
// that exceeds its bound sets PcgState::stalled and ends the launch (the
// host reports CF_EDEVICE).
#include <hip/hip_runtime.h>

#include <climits>
#include <cmath>

#include "cf_pcg_state.hpp"
#include "cf_solver.hpp"
#include "cf_stream.hpp"

namespace cfmi
{

namespace
{

constexpr int kCoopMaxGroups = 256;
constexpr int kCoopCells = 4096; // of a strip or pencil at most
constexpr unsigned kCoopSpin = 1u << 22; // polls (about 1 us each) before a wait counts as stalled

// The strips' shape: 4 cells a lane of 256 lanes while that makes at most 64
// strips, 4 of 512 up to 128 strips and where that makes one of two (45^2
// 3.9 -> 2.3 us an iteration; 3840 cells in one strip of 960 lanes gained 7%
// over two to four, 4096 in one of 448 nothing), else 10 of 448 (with the scalars' wave two
// waves a SIMD: 8 of 512 with it left 168 registers a lane, and spilled).
// Fewer, larger strips shorten the exchanges and lengthen the strip's own
// chain.  us per iteration at 4 of 256, 4 of 512 and 8 of 512 lanes, with the
// scalars in a wave of cells: 32^2 2.9 (one strip), 3.8, 5.0; 128^2 5.7, 5.8,
// 6.7; 256^2 6.8, 7.7, 8.4; 391 x 263 9.7, 7.7, 9.0; 512^2 13.4, 9.1, 9.4;
// 700 x 500 -, 14.9, 10.5; 1024^2 -, -, 16.9.  Now, at the shape chosen: 32^2
// 2.0, 128^2 4.3, 256^2 5.6, 391 x 263 6.2, 512^2 7.1, 700 x 500 9.0, 1024^2
// 14.7 (the streaming kernels 32.2).  1024 lanes, and 2 cells a lane, were
// slower or within 2% everywhere.  Rows of more than 1024 cells, whose halo is
// as large as the strip, gain too (300 iterations, over them, the kernels
// before and these): 1100 x 200 21.1, 9.8; 1700 x 250 29.1, 12.2; 2300 x 256
// 33.8, 21.2; 2300 x 30 32.5, 12.8.
CoopGrid coop_grid(const Geo& g)
{
    constexpr int shape[3][3] = {{256, 4, 64}, {512, 4, 128}, {448, 10, kCoopMaxGroups}};
    CoopGrid cg;
    for (const auto& sh : shape) {
        cg.nt = sh[0];
        cg.cpt = sh[1];
        cg.R = (cg.nt * cg.cpt < kCoopCells ? cg.nt * cg.cpt : kCoopCells) / g.n[0];
        if (cg.R > g.n[1])
            cg.R = g.n[1];
        cg.G = cg.R > 0 ? (g.n[1] + cg.R - 1) / cg.R : INT_MAX;
        if (cg.G > 1 && (int64_t)g.n[0] * g.n[1] <= 4 * 512 && cg.nt == 256)
            continue;
        if (cg.G <= sh[2])
            break;
    }
    cg.every = cg.G > 1 && cg.G <= 32 ? 8 : 1;
    cg.e0 = g.n[0] + 2;
    cg.nwin = cg.e0 * (cg.R + 2);
    cg.c00 = (int)g.idx(g.h, g.h, g.own_lo(2));
    cg.px = (int)g.px;
    return cg;
}

// Bytes of LDS: the window, the coefficient tables, the halo rows' r and D^-1.
size_t coop_lds(const Geo& g, const CoopGrid& cg)
{
    return ((size_t)cg.nwin + 14 + 4 * (size_t)g.n[0]) * sizeof(double);
}

using Word = unsigned long long;

// The exchange buffer: per strip 16 words of partials (p.q in words 0-3,
// r.r and r.z in 8-15), and per strip the two boundary rows' r, two words a
// cell (top row, then bottom row).
struct CoopXch
{
    Word* part; // [G][16]
    Word* halo; // [G][2][n0][2]
    unsigned seq0; // the launch's exchanges are numbered from seq0 + 1
};

__device__ __forceinline__ void put_word(Word* p, unsigned seq, unsigned v)
{
    __hip_atomic_store(p, (Word)seq << 32 | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ Word get_word(const Word* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double value_of(Word lo, Word hi)
{
    return __longlong_as_double((long long)(hi << 32 | (lo & 0xffffffffu)));
}

#define CF_STEP(MOVE)                                   \
    {                                                   \
        const double oh = MOVE(h), ol = MOVE(l);        \
        dd_merge(h, l, oh, ol);                         \
    }

// The sums over the even lanes and over the odd lanes, in each even and each
// odd lane, of values that repeat every `width` lanes or (width >= 16) are
// zero past them.  As in wave_sum, the two lanes of a step add the same two
// pairs, so every lane ends with the same (h, l) bits: the words of a
// published partial come from different lanes.
__device__ __forceinline__ void pair_sum(double& h, double& l, int width)
{
    CF_STEP(move_row<0x4E>)
    if (width > 8)
        CF_STEP(move_row<0x128>) // row_ror 8
    if (width > 4)
        CF_STEP(move_row<0x124>) // row_ror 4
    if (width > 16)
        CF_STEP(move_half<16>)
    if (width > 32)
        CF_STEP(move_half<32>)
}
#undef CF_STEP

// What the waves of a workgroup share.  A workgroup is NW waves of cells and
// one wave of scalars (coop_scalars): the cells' waves leave their wave sums
// in red, the scalars' wave forms the totals over all workgroups.
template <int NW>
struct CoopShared
{
    static constexpr int N = NW <= 4 ? 4 : 8; // NW rounded up, zeros past NW
    double pq[2][N];    // p.q of the waves, high and low parts
    double rr[2][2][N]; // r.r, r.z
    double alpha, beta;
    int stop, stall;

    // before the workgroup's first barrier
    __device__ __forceinline__ void clear(int t)
    {
        if (t < 2 * N)
            pq[t / N][t % N] = 0.0;
        if (t < 4 * N)
            rr[t / N / 2][t / N % 2][t % N] = 0.0;
        if (t == 0)
            stop = stall = 0;
    }
};

// A wave's sum of (h, l) for the scalars' wave; the sums of (h0, l0) and of
// (h1, l1), the first exchange handing each lane one of the two.
template <int NW>
__device__ __forceinline__ void leave_pq(CoopShared<NW>& sh, double h, double l)
{
    wave_sum(h, l, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0) {
        sh.pq[0][threadIdx.x / kWave] = h;
        sh.pq[1][threadIdx.x / kWave] = l;
    }
}
template <int NW>
__device__ __forceinline__ void leave_rr(CoopShared<NW>& sh, const double (&hi)[2],
                                         const double (&lo)[2])
{
    const int lane = threadIdx.x & (kWave - 1);
    const bool odd = lane & 1;
    double h = odd ? hi[1] : hi[0], l = odd ? lo[1] : lo[0];
    const double oh = move_row<0xB1>(odd ? hi[0] : hi[1]), ol = move_row<0xB1>(odd ? lo[0] : lo[1]);
    dd_merge(h, l, oh, ol);
    pair_sum(h, l, kWave);
    if (lane < 2) {
        sh.rr[lane][0][threadIdx.x / kWave] = h;
        sh.rr[lane][1][threadIdx.x / kWave] = l;
    }
}

// Polls the four words at each of `at` until all carry seq; false: stalled.
// With one place a lane, only the lanes that want theirs read (of up to 32
// workgroups most have none: 128^2 4.8 -> 4.4 us an iteration); with more, a
// branch for each costs more than the reads it saves (512^2 7.1 -> 8.3).
template <int N>
__device__ __forceinline__ bool poll_words(const Word* const (&at)[N], const bool (&want)[N],
                                           unsigned seq, Word (&w)[N][4])
{
    for (unsigned polls = 0; polls < kCoopSpin; ++polls) {
        bool all = true;
#pragma unroll
        for (int u = 0; u < N; ++u)
            if (N > 1 || want[u]) {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    w[u][k] = get_word(at[u] + k);
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    all = all && (unsigned)(w[u][k] >> 32) == seq;
            }
        if (__all(all))
            return true;
    }
    return false;
}

// The scalars' wave: per iteration p.q's total and alpha, then r.r's and
// r.z's and beta; it keeps the PCG state (the same in every workgroup) in its
// first lane.  The stop test's square root and division run beside the cells'
// next direction and stencil, so a stop is seen one direction later.  The
// barriers are the cells' waves' (A, after periodic x's copies again, B, C,
// D, E).  PQ: strips per lane of the gather of the two sums (32 lanes each).
template <int NW, int PQ>
__device__ __forceinline__ void coop_scalars(CoopShared<NW>& sh, PcgState& fs, int gid, int G,
                                             const CoopXch& xc, bool periodic_x, int max_its)
{
    constexpr int N = CoopShared<NW>::N;
    constexpr int P1 = PQ > 1 ? PQ / 2 : 1; // strips per lane of p.q's gather
    const int lane = threadIdx.x & (kWave - 1);
    unsigned seq = xc.seq0;
    double rr = 0.0, rz = 0.0;
    const int width = G <= 1 ? 1 : G < kWave ? 1 << (32 - __builtin_clz(G - 1)) : kWave;
    for (int its = 1;; ++its) {
        __syncthreads(); // A
        if (periodic_x)
            __syncthreads();
        if (its > 1 && lane == 0) {
            finish_update(&fs, rr, rz);
            sh.stop = fs.done;
        }
        __syncthreads(); // B
        if (sh.stop)
            break;
        double h = sh.pq[0][lane & (N - 1)], l = sh.pq[1][lane & (N - 1)];
        wave_sum(h, l, N);
        ++seq;
        if (G > 1) {
            if (lane < 4) {
                const double v = lane & 2 ? l : h;
                put_word(xc.part + (size_t)gid * 16 + lane, seq,
                         (unsigned)(lane & 1 ? __double2hiint(v) : __double2loint(v)));
            }
            const Word* at[P1];
            bool want[P1];
            Word w[P1][4];
#pragma unroll
            for (int u = 0; u < P1; ++u) {
                const int q = lane + kWave * u;
                want[u] = q < G;
                at[u] = xc.part + (size_t)(q < G ? q : 0) * 16;
            }
            if (!poll_words<P1>(at, want, seq, w) && lane == 0)
                sh.stall = 1;
            h = l = 0.0;
#pragma unroll
            for (int u = 0; u < P1; ++u)
                if (want[u])
                    dd_merge(h, l, value_of(w[u][0], w[u][1]), value_of(w[u][2], w[u][3]));
            wave_sum(h, l, width);
        }
        if (lane == 0) {
            fs.alpha = fs.rho / (h + l);
            sh.alpha = fs.alpha;
        }
        __syncthreads(); // C
        if (sh.stall)
            break;
        __syncthreads(); // D
        // r.r in the even lanes, r.z in the odd ones
        const int v = lane & 1, wv = lane >> 1 & (N - 1);
        h = sh.rr[v][0][wv];
        l = sh.rr[v][1][wv];
        pair_sum(h, l, 2 * N);
        ++seq;
        if (G > 1) {
            if (lane < 8) {
                const int k = lane >> 1;
                const double d = k & 2 ? l : h;
                put_word(xc.part + (size_t)gid * 16 + 8 + 4 * v + k, seq,
                         (unsigned)(k & 1 ? __double2hiint(d) : __double2loint(d)));
            }
            const Word* at[PQ];
            bool want[PQ];
            Word w[PQ][4];
#pragma unroll
            for (int u = 0; u < PQ; ++u) {
                const int q = (lane >> 1) + kWave / 2 * u;
                want[u] = q < G;
                at[u] = xc.part + (size_t)(q < G ? q : 0) * 16 + 8 + 4 * v;
            }
            if (!poll_words<PQ>(at, want, seq, w) && lane == 0)
                sh.stall = 1;
            h = l = 0.0;
#pragma unroll
            for (int u = 0; u < PQ; ++u)
                if (want[u])
                    dd_merge(h, l, value_of(w[u][0], w[u][1]), value_of(w[u][2], w[u][3]));
            pair_sum(h, l, width < 8 ? 16 : 2 * width);
        }
        rr = h + l;
        rz = move_row<0xB1>(rr);
        if (lane == 0)
            sh.beta = rz / fs.rho;
        __syncthreads(); // E
        if (sh.stall)
            break;
        if (its >= max_its) {
            if (lane == 0)
                finish_update(&fs, rr, rz);
            break;
        }
    }
}

template <int NT, int CPT, int PQ>
__global__ __launch_bounds__(NT + kWave) void k_pcg_solve_coop(Geo g, CoopGrid cg,
                                                               double* __restrict__ x,
                                                               double* __restrict__ r,
                                                               double* __restrict__ pg,
                                                               PcgState* st, CoopXch xc,
                                                               int max_its)
{
    if (blockIdx.x % cg.every)
        return;
    constexpr int NW = NT / kWave;
    extern __shared__ double lds[];
    double* pw = lds;             // the direction window
    double* tab = lds + cg.nwin;  // diag[0..6], then dinv[0..6]
    double* hz = tab + 14;        // halo rows' D^-1 r [2][n0]
    double* hd = hz + 2 * g.n[0]; // and their D^-1
    __shared__ CoopShared<NW> sh;
    // The state is read once, here; the scalars' wave of every workgroup keeps
    // the same copy in registers, and workgroup 0 stores it back at the end.
    // A read of *st after a write in this kernel could be served by the scalar
    // cache, which vector stores do not update.
    PcgState fs = *st;
    const int t = threadIdx.x;
    const int gid = blockIdx.x / cg.every, G = cg.G;
    const int n0 = g.n[0], n1 = g.n[1], e0 = cg.e0;
    const int j0 = gid * cg.R;
    const int nrows = (j0 + cg.R < n1 ? cg.R : n1 - j0);
    const int ncell = nrows * n0;
    const double s = offdiag<double>(g);
    const double ring0 = copysign(0.0, s);
    sh.clear(t);
    for (int e = t; e < cg.nwin; e += NT + kWave)
        pw[e] = ring0;
#pragma unroll
    for (int q = 0; q < 7; ++q)
        if (t == q) {
            tab[q] = g.diag[q];
            tab[7 + q] = g.dinv[q];
        }
    __syncthreads();
    if (fs.done)
        return;
    if (__builtin_amdgcn_readfirstlane(t / kWave) == NW) {
        __syncthreads(); // the cells are loaded
        coop_scalars<NW, PQ>(sh, fs, gid, G, xc, g.periodic[0], max_its);
        if (gid == 0 && t == NT) {
            if (sh.stall)
                fs.stalled = 1;
            *st = fs;
        }
        return;
    }
    bool first = fs.iter == 0;
    double beta = fs.beta;

    // halo rows: window rows 0 (global row j0 - 1) and nrows + 1 (row j0 +
    // nrows), when they exist; gtop / gbot the strips that own them
    const bool py = g.periodic[1];
    const bool has_top = j0 > 0 || py, has_bot = j0 + nrows < n1 || py;
    const int jtop = j0 > 0 ? j0 - 1 : n1 - 1, jbot = j0 + nrows < n1 ? j0 + nrows : 0;
    const int gtop = gid > 0 ? gid - 1 : G - 1, gbot = gid + 1 < G ? gid + 1 : 0;
    // SOLID wall count of a cell of global row j (in 2-D, z adds its own
    // count for k = 0 as the streaming kernels do)
    auto cell_cnt = [&](int i, int j) -> int { return row_stencil(g, j, 0).cnt + lane_x(g, i).cnt; };
    // window index of a halo cell
    auto halo_at = [&](int side, int i) -> int { return (i + 1) + (side == 0 ? 0 : e0 * (nrows + 1)); };
    // the two halo rows' r, and a resumed solve's direction, from the padded
    // arrays (start of a launch)
    for (int e = t; e < 2 * n0; e += NT) {
        const int side = e >= n0 ? 1 : 0, i = e - side * n0;
        if (side == 0 ? has_top : has_bot) {
            const int64_t c = cg.c00 + i + (int64_t)cg.px * (side == 0 ? jtop : jbot);
            hd[e] = tab[7 + cell_cnt(i, side == 0 ? jtop : jbot)];
            hz[e] = hd[e] * r[c];
            if (!first)
                pw[halo_at(side, i)] = pg[c];
        }
    }

    // Slots past the strip's last cell carry the first cell's window index;
    // their stores and sums are masked.
    int wi[CPT]; // window indices
    bool own[CPT];
    double rv[CPT], qv[CPT], xv[CPT], dg[CPT], dv[CPT], pn[CPT];
#pragma unroll
    for (int m = 0; m < CPT; ++m) {
        const int L = t + NT * m;
        const int i = L % n0, jj = L / n0;
        own[m] = L < ncell;
        wi[m] = 1 + e0; // strip cell (0, 0)
        rv[m] = qv[m] = xv[m] = pn[m] = 0.0;
        dg[m] = tab[0];
        dv[m] = tab[7];
        if (own[m]) {
            const int cnt = cell_cnt(i, j0 + jj);
            wi[m] = (i + 1) + e0 * (jj + 1);
            dg[m] = tab[cnt];
            dv[m] = tab[7 + cnt];
            const int64_t c = cg.c00 + i + (int64_t)cg.px * (j0 + jj);
            rv[m] = r[c];
            xv[m] = x[c];
            if (!first)
                pn[m] = pg[c];
        }
    }
    // padded index of a slot's cell
    auto padded = [&](int li) -> int64_t {
        const int jj = li / e0 - 1, i = li - e0 * (jj + 1) - 1;
        return cg.c00 + i + (int64_t)cg.px * (j0 + jj);
    };
    __syncthreads();
    unsigned seq = xc.seq0;
    for (int its = 1;; ++its) {
        // direction: p = D^-1 r, or fma(beta, p, D^-1 r), for the strip's
        // cells and its halo rows
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            const double z = dv[m] * rv[m];
            pn[m] = first ? z : fma(beta, pn[m], z);
        }
#pragma unroll
        for (int m = 0; m < CPT; ++m)
            if (own[m])
                pw[wi[m]] = pn[m];
        if (has_top || has_bot)
            for (int e = t; e < 2 * n0; e += NT) {
                const int side = e >= n0 ? 1 : 0, i = e - side * n0;
                if (side == 0 ? has_top : has_bot) {
                    double* pp = pw + halo_at(side, i);
                    *pp = first ? hz[e] : fma(beta, *pp, hz[e]);
                }
            }
        __syncthreads(); // A
        if (g.periodic[0]) {
            for (int jw = t; jw < nrows + 2; jw += NT) {
                double* row = pw + e0 * jw;
                row[0] = row[n0];
                row[n0 + 1] = row[1];
            }
            __syncthreads();
        }
        // q = A p in the stencil order {0}, -x, +x, -y, +y; p.q
        double h1 = 0.0, l1 = 0.0;
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            const double* pp = pw + wi[m];
            const double pc = own[m] ? pn[m] : 0.0;
            double y = dg[m] * pn[m];
            y = fma(s, pp[-1], y);
            y = fma(s, pp[1], y);
            y = fma(s, pp[-e0], y);
            y = fma(s, pp[e0], y);
            qv[m] = own[m] ? y : 0.0;
            dd_acc_prod(h1, l1, pc, qv[m]);
        }
        leave_pq(sh, h1, l1);
        __syncthreads(); // B
        if (sh.stop)
            break;
        ++seq;
        __syncthreads(); // C
        if (sh.stall)
            break;
        const double alpha = sh.alpha;
        // x = fma(alpha, p, x); r = fma(-alpha, q, r); r.r and r.(D^-1 r).
        // Past the strip's last cell q = r = 0, so rn = 0 and the sums are
        // unchanged.
        ++seq;
#pragma unroll
        for (int m = 0; m < CPT; ++m)
            rv[m] = fma(-alpha, qv[m], rv[m]);
        // boundary rows' new r for the neighbour strips (the one strip of a
        // periodic axis is its own), before the partials: sent with them (after
        // D) they held up each other, 128^2 4.9 -> 5.3 us, 64^3 8.2 -> 9.2
#pragma unroll
        for (int side = 0; side < 2; ++side) {
            if (!(side == 0 ? has_top : has_bot))
                continue;
            const int lo = side == 0 ? 0 : ncell - n0;
#pragma unroll
            for (int m = 0; m < CPT; ++m) {
                if (NT * m >= lo + n0 || NT * (m + 1) <= lo)
                    continue;
                const int i = t + NT * m - lo;
                if (i < 0 || i >= n0)
                    continue;
                if (G > 1) {
                    Word* hb = xc.halo + (((size_t)gid * 2 + side) * n0 + i) * 2;
                    put_word(hb, seq, (unsigned)__double2loint(rv[m]));
                    put_word(hb + 1, seq, (unsigned)__double2hiint(rv[m]));
                } else {
                    const int e = (side ^ 1) * n0 + i;
                    hz[e] = hd[e] * rv[m];
                }
            }
        }
        double hi[2] = {0.0, 0.0}, lo[2] = {0.0, 0.0};
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            const double z = dv[m] * rv[m];
            dd_acc_prod(hi[0], lo[0], rv[m], rv[m]);
            dd_acc_prod(hi[1], lo[1], rv[m], z);
        }
        leave_rr(sh, hi, lo);
        __syncthreads(); // D
#pragma unroll
        for (int m = 0; m < CPT; ++m)
            xv[m] = fma(alpha, pn[m], xv[m]);
        if (G > 1) {
            // the neighbours' boundary rows, a few cells a lane at a time so
            // that their words are in flight together
            constexpr int NB = 4;
            for (int e1 = t; e1 < 2 * n0; e1 += NB * NT) {
                Word w[NB][2];
                unsigned polls = 0;
                for (;;) {
                    bool all = true;
#pragma unroll
                    for (int b = 0; b < NB; ++b) {
                        const int e = e1 + b * NT;
                        const int side = e >= n0 ? 1 : 0, i = e - side * n0;
                        const bool want = e < 2 * n0 && (side == 0 ? has_top : has_bot);
                        // the top halo row is the bottom row of the strip above
                        const Word* hb =
                            xc.halo + (want ? (((size_t)(side == 0 ? gtop : gbot) * 2 +
                                                (side == 0 ? 1 : 0)) * n0 + i) * 2
                                            : 0);
                        w[b][0] = get_word(hb);
                        w[b][1] = get_word(hb + 1);
                        if (!want)
                            w[b][0] = w[b][1] = (Word)seq << 32;
                    }
#pragma unroll
                    for (int b = 0; b < NB; ++b)
                        all = all && (unsigned)(w[b][0] >> 32) == seq &&
                              (unsigned)(w[b][1] >> 32) == seq;
                    if (all)
                        break;
                    if (++polls >= kCoopSpin) {
                        sh.stall = 1;
                        break;
                    }
                }
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const int e = e1 + b * NT;
                    if (e < 2 * n0)
                        hz[e] = hd[e] * value_of(w[b][0], w[b][1]);
                }
            }
        }
        __syncthreads(); // E
        if (sh.stall || its >= max_its)
            break;
        beta = sh.beta;
        first = false;
    }
    // x, r and the direction back to memory (a later launch resumes from
    // them; after a stop the direction is one ahead and nobody's)
#pragma unroll
    for (int m = 0; m < CPT; ++m)
        if (own[m]) {
            const int64_t c = padded(wi[m]);
            x[c] = xv[m];
            r[c] = rv[m];
            pg[c] = pn[m];
        }
}

template <int NT, int CPT>
const void* coop_kernel(int G)
{
    static_assert(kCoopMaxGroups <= 8 * 32, "gather bucket");
    return G <= 32    ? (const void*)k_pcg_solve_coop<NT, CPT, 1>
           : G <= 64  ? (const void*)k_pcg_solve_coop<NT, CPT, 2>
           : G <= 128 ? (const void*)k_pcg_solve_coop<NT, CPT, 4>
                      : (const void*)k_pcg_solve_coop<NT, CPT, 8>;
}

// ---- 3-D grids ------------------------------------------------------------------------
// The same solve with a workgroup per pencil of by x bz whole x-rows.  The
// window holds the pencil's rows and one row around them; a boundary cell's
// new r goes out as two words at the cell's own place (a neighbour pencil
// polls that place), so no pencil needs to know which one owns its halo.  A
// halo cell's r stays in its lane's registers from the poll to the next
// direction.  The wave that gathers the partials has no halo cells.
constexpr int kCoopHalo = 8; // halo cells per lane at most

// A bit mask the compiler re-reads: its bits' tests are not all kept as lane
// masks across the loop (which spilled the scalar registers).
__device__ __forceinline__ unsigned fresh(unsigned v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// The words of a value at place `at`: two of a double, one of a float.
__device__ __forceinline__ void put_value(Word* base, int at, unsigned seq, double v)
{
    put_word(base + 2 * (size_t)at, seq, (unsigned)__double2loint(v));
    put_word(base + 2 * (size_t)at + 1, seq, (unsigned)__double2hiint(v));
}
__device__ __forceinline__ void put_value(Word* base, int at, unsigned seq, float v)
{
    put_word(base + at, seq, __float_as_uint(v));
}
template <class T>
struct ValueWords
{
    Word lo, hi;
    __device__ __forceinline__ void get(const Word* base, int at)
    {
        lo = get_word(base + 2 * (size_t)at);
        hi = get_word(base + 2 * (size_t)at + 1);
    }
    __device__ __forceinline__ bool is(unsigned seq) const
    {
        return (unsigned)(lo >> 32) == seq && (unsigned)(hi >> 32) == seq;
    }
    __device__ __forceinline__ T value() const { return value_of(lo, hi); }
};
template <>
struct ValueWords<float>
{
    Word w;
    __device__ __forceinline__ void get(const Word* base, int at) { w = get_word(base + at); }
    __device__ __forceinline__ bool is(unsigned seq) const { return (unsigned)(w >> 32) == seq; }
    __device__ __forceinline__ float value() const { return __uint_as_float((unsigned)w); }
};

template <class T, int NT, int CPT, int PQ>
__global__ __launch_bounds__(NT + kWave) void k_pcg_solve_coop3(Geo g, Coop3Grid cg,
                                                                T* __restrict__ x,
                                                                T* __restrict__ r,
                                                                T* __restrict__ pg,
                                                                PcgState* st, CoopXch xc,
                                                                int max_its)
{
    if (blockIdx.x % cg.every)
        return;
    constexpr int NW = NT / kWave;
    constexpr bool EXACT = std::is_same<T, float>::value; // products of two T in double
    extern __shared__ double lds[];
    T* pw = reinterpret_cast<T*>(lds); // the direction window
    T* tab = pw + cg.nwin;             // diag[0..6], then dinv[0..6]
    T* xl = tab + 14;                  // x of the lane's cells, CPT per lane
    __shared__ CoopShared<NW> sh;
    PcgState fs = *st; // read once, as in k_pcg_solve_coop
    const int t = threadIdx.x;
    const int gid = blockIdx.x / cg.every, G = cg.G;
    const int n0 = g.n[0], n1 = g.n[1], n2 = g.n[2], e0 = cg.e0, e1 = cg.e1;
    const int j0 = gid % cg.gy * cg.by, k0 = gid / cg.gy * cg.bz;
    const int nby = min(cg.by, n1 - j0), nbz = min(cg.bz, n2 - k0);
    const T s = offdiag<T>(g);
    const T ring0 = s < (T)0 ? -(T)0 : (T)0; // a zero of s's sign
    sh.clear(t);
    for (int e = t; e < cg.nwin; e += NT + kWave)
        pw[e] = ring0;
#pragma unroll
    for (int q = 0; q < 7; ++q)
        if (t == q) {
            tab[q] = diag_of<T>(g, q);
            tab[7 + q] = dinv_of<T>(g, q);
        }
    __syncthreads();
    if (fs.done)
        return;
    if (__builtin_amdgcn_readfirstlane(t / kWave) == NW) {
        __syncthreads(); // the cells are loaded
        coop_scalars<NW, PQ>(sh, fs, gid, G, xc, g.periodic[0], max_its);
        if (gid == 0 && t == NT) {
            if (sh.stall)
                fs.stalled = 1;
            *st = fs;
        }
        return;
    }
    bool first = fs.iter == 0;
    T beta = (T)fs.beta;
    auto cell_cnt = [&](int i, int j, int k) -> int {
        return wall_count(g, 0, i) + wall_count(g, 1, j) + wall_count(g, 2, k);
    };
    auto padded = [&](int i, int j, int k) -> int64_t {
        return cg.c00 + i + (int64_t)cg.px * j + cg.pxy * k;
    };

    // halo cells: the rows y-low, y-high (nbz each), z-low, z-high (nby each).
    // hw: window index (bits 0-15), SOLID wall count (bits 16-18), kept only
    // where the row exists; hs: the cell's number.
    const int nrow = 2 * (nby + nbz);
    int hw[kCoopHalo], hs[kCoopHalo];
    T hz[kCoopHalo]; // D^-1 r
    unsigned halo_bits = 0;
#pragma unroll
    for (int b = 0; b < kCoopHalo; ++b) {
        hw[b] = hs[b] = 0;
        hz[b] = (T)0;
        const int h = t + NT * b;
        const int row = h / n0, i = h - row * n0;
        if (row >= nrow)
            continue;
        int jj, kk; // pencil-relative
        if (row < 2 * nbz) {
            jj = row < nbz ? -1 : nby;
            kk = row < nbz ? row : row - nbz;
        } else {
            const int q = row - 2 * nbz;
            jj = q < nby ? q : q - nby;
            kk = q < nby ? -1 : nbz;
        }
        int j = j0 + jj, k = k0 + kk;
        if (j < 0 || j >= n1) {
            if (!g.periodic[1])
                continue;
            j = j < 0 ? n1 - 1 : 0;
        }
        if (k < 0 || k >= n2) {
            if (!g.periodic[2])
                continue;
            k = k < 0 ? n2 - 1 : 0;
        }
        halo_bits |= 1u << b;
        const int w = (i + 1) + e0 * (jj + 1) + e1 * (kk + 1);
        hw[b] = w | cell_cnt(i, j, k) << 16;
        hs[b] = i + n0 * (j + n1 * k);
        const int64_t c = padded(i, j, k);
        hz[b] = tab[7 + (hw[b] >> 16)] * r[c];
        if (!first)
            pw[w] = pg[c];
    }

    // own cells: window index, and SOLID wall count (bits 16-18)
    int wi[CPT], no[CPT]; // no: the cell's number
    T rv[CPT], qv[CPT], pn[CPT];
    T po[CPT]; // FP32: the direction before, which the next pass resumes from
    unsigned own_bits = 0, edge_bits = 0; // edge: some pencil's halo
    const int ncell = n0 * nby * nbz;
#pragma unroll
    for (int m = 0; m < CPT; ++m) {
        wi[m] = 1 + e0 + e1; // pencil cell (0, 0, 0)
        no[m] = 0;
        rv[m] = qv[m] = pn[m] = po[m] = (T)0;
        const int L = t + NT * m;
        if (L < ncell) {
            const int row = L / n0, i = L - row * n0;
            const int kk = row / nby, jj = row - kk * nby;
            no[m] = i + n0 * (j0 + jj + n1 * (k0 + kk));
            wi[m] = ((i + 1) + e0 * (jj + 1) + e1 * (kk + 1)) |
                    cell_cnt(i, j0 + jj, k0 + kk) << 16;
            own_bits |= 1u << m;
            edge_bits |= jj == 0 || jj == nby - 1 || kk == 0 || kk == nbz - 1 ? 1u << m : 0u;
            const int64_t c = padded(i, j0 + jj, k0 + kk);
            rv[m] = r[c];
            xl[L] = x[c];
            if (!first)
                pn[m] = pg[c];
        }
    }
    __syncthreads();
    unsigned seq = xc.seq0;
    for (int its = 1;; ++its) {
        const unsigned own = fresh(own_bits), edge = fresh(edge_bits), have = fresh(halo_bits);
        // direction: p = D^-1 r, or fma(beta, p, D^-1 r), own and halo cells
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            const T z = tab[7 + (wi[m] >> 16)] * rv[m];
            if constexpr (EXACT)
                po[m] = pn[m];
            pn[m] = first ? z : fma_t<T>(beta, pn[m], z);
        }
#pragma unroll
        for (int m = 0; m < CPT; ++m)
            if (own >> m & 1)
                pw[wi[m] & 0xffff] = pn[m];
#pragma unroll
        for (int b = 0; b < kCoopHalo; ++b)
            if (have >> b & 1) {
                T* pp = pw + (hw[b] & 0xffff);
                *pp = first ? hz[b] : fma_t<T>(beta, *pp, hz[b]);
            }
        __syncthreads(); // A
        if (g.periodic[0]) {
            for (int q = t; q < nby * nbz; q += NT) {
                T* row = pw + e0 * (q % nby + 1) + e1 * (q / nby + 1);
                row[0] = row[n0];
                row[n0 + 1] = row[1];
            }
            __syncthreads();
        }
        // q = A p in the stencil order {0}, -x, +x, -y, +y, -z, +z; p.q
        double h1 = 0.0, l1 = 0.0;
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            const T* pp = pw + (wi[m] & 0xffff);
            const bool mine = own >> m & 1;
            T y = tab[wi[m] >> 16] * pn[m];
            y = fma_t<T>(s, pp[-1], y);
            y = fma_t<T>(s, pp[1], y);
            y = fma_t<T>(s, pp[-e0], y);
            y = fma_t<T>(s, pp[e0], y);
            y = fma_t<T>(s, pp[-e1], y);
            y = fma_t<T>(s, pp[e1], y);
            qv[m] = mine ? y : (T)0;
            dd_acc_prod<EXACT>(h1, l1, mine ? (double)pn[m] : 0.0, (double)qv[m]);
        }
        leave_pq(sh, h1, l1);
        __syncthreads(); // B
        if (sh.stop) {
            if constexpr (EXACT) {
#pragma unroll
                for (int m = 0; m < CPT; ++m)
                    pn[m] = po[m];
            }
            break;
        }
        ++seq;
        __syncthreads(); // C
        if (sh.stall)
            break;
        const T alpha = (T)sh.alpha;
        // r = fma(-alpha, q, r), published where a neighbour needs it; r.r and
        // r.(D^-1 r); x = fma(alpha, p, x)
        double hi[2] = {0.0, 0.0}, lo[2] = {0.0, 0.0};
        ++seq;
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            rv[m] = fma_t<T>(-alpha, qv[m], rv[m]);
            if (edge >> m & 1) {
                put_value(xc.halo, no[m], seq, rv[m]);
            }
        }
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            const T z = tab[7 + (wi[m] >> 16)] * rv[m];
            dd_acc_prod<EXACT>(hi[0], lo[0], (double)rv[m], (double)rv[m]);
            dd_acc_prod<EXACT>(hi[1], lo[1], (double)rv[m], (double)z);
        }
        leave_rr(sh, hi, lo);
        __syncthreads(); // D
#pragma unroll
        for (int m = 0; m < CPT; ++m)
            xl[t + NT * m] = fma_t<T>(alpha, pn[m], xl[t + NT * m]);
        // the halo cells' new r, four a lane at a time
#pragma unroll
        for (int b0 = 0; b0 < kCoopHalo; b0 += 4) {
            if (!(have >> b0 & 15))
                continue;
            ValueWords<T> w[4];
            unsigned polls = 0;
            for (;;) {
                bool all = true;
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    w[b].get(xc.halo, hs[b0 + b]);
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    all = all && (!(have >> (b0 + b) & 1) || w[b].is(seq));
                if (all)
                    break;
                if (++polls >= kCoopSpin) {
                    sh.stall = 1;
                    break;
                }
            }
#pragma unroll
            for (int b = 0; b < 4; ++b)
                hz[b0 + b] = tab[7 + (hw[b0 + b] >> 16)] * w[b].value();
        }
        __syncthreads(); // E
        if (sh.stall || its >= max_its)
            break;
        beta = (T)sh.beta;
        first = false;
    }
#pragma unroll
    for (int m = 0; m < CPT; ++m)
        if (own_bits >> m & 1) {
            const int row = no[m] / n0, i = no[m] - row * n0;
            const int64_t c = padded(i, row % n1, row / n1);
            x[c] = xl[t + NT * m];
            r[c] = rv[m];
            pg[c] = pn[m];
        }
}

// Bytes of LDS: the window, the coefficient tables, x.
size_t coop3_lds(const Coop3Grid& c)
{
    return ((size_t)c.nwin + 14 + (size_t)c.nt * c.cpt) * sizeof(double);
}

// The pencils' shape: the one with the least estimate of an iteration's time
// in us, from measured parts: an exchange of G workgroups (twice), a cell of
// a lane per wave of a SIMD, the fixed chain, and the halo words' traffic.
// G = 0: none fits (more than 256 pencils of 4096 cells, about 100^3).  us per
// iteration, the streaming tiles and this: 45 x 52 x 61 22.6, 7.5; 64^3 22.9,
// 8.2; 96^3 30.6, 13.7; 100^3 32, 15.8.  FP32, a refined solve's time over its
// iterations: 32^3 22, 6.7; 64^3 25, 7.8; 96^3 30, 12.6.
Coop3Grid coop3_grid(const Geo& g)
{
    constexpr int shape[][2] = {{256, 2}, {256, 4}, {512, 4}, {448, 10}};
    Coop3Grid best{};
    double cost = 1e30;
    const int n0 = g.n[0], n1 = g.n[1], n2 = g.n[2];
    if (n0 > 1024)
        return best;
    for (int by = 1; by <= n1 && by <= 64; ++by)
        for (int bz = 1; bz <= n2 && bz <= 64; ++bz) {
            const int64_t cells = (int64_t)n0 * by * bz;
            const int64_t G64 = (int64_t)((n1 + by - 1) / by) * ((n2 + bz - 1) / bz);
            if (cells > kCoopCells || G64 > kCoopMaxGroups)
                continue;
            const int G = (int)G64;
            int q = 0;
            while (shape[q][0] * shape[q][1] < cells)
                ++q;
            const int nt = shape[q][0], cpt = shape[q][1];
            const int halo = 2 * (by + bz) * n0;
            Coop3Grid c{};
            c.G = G;
            c.by = by;
            c.bz = bz;
            c.gy = (n1 + by - 1) / by;
            c.e0 = n0 + 2;
            c.e1 = c.e0 * (by + 2);
            c.nwin = c.e1 * (bz + 2);
            c.nt = nt;
            c.cpt = cpt;
            if (halo > kCoopHalo * nt || c.nwin >= 1 << 16 ||
                coop3_lds(c) > 150 * 1024)
                continue;
            const double xch = G > 1 ? 1.3 + 0.1 * std::log2((double)G) + 0.006 * G : 0.15;
            const double us = 2.0 * xch + 1.5 +
                              0.25 * (nt * cpt) / 256.0 + 1e-3 * halo / nt * 200.0 +
                              3.2e-6 * halo * G;
            if (us < cost) {
                cost = us;
                best = c;
            }
        }
    best.every = best.G > 1 && best.G <= 32 ? 8 : 1;
    best.c00 = (int)g.idx(g.h, g.h, g.h);
    best.px = (int)g.px;
    best.pxy = g.px * g.py;
    return best;
}

template <class T, int NT, int CPT>
const void* coop3_kernel(int G)
{
    return G <= 32    ? (const void*)k_pcg_solve_coop3<T, NT, CPT, 1>
           : G <= 64  ? (const void*)k_pcg_solve_coop3<T, NT, CPT, 2>
           : G <= 128 ? (const void*)k_pcg_solve_coop3<T, NT, CPT, 4>
                      : (const void*)k_pcg_solve_coop3<T, NT, CPT, 8>;
}
template <class T>
const void* coop3_kernel(const Coop3Grid& c)
{
    return c.nt == 256 ? (c.cpt == 2 ? coop3_kernel<T, 256, 2>(c.G) : coop3_kernel<T, 256, 4>(c.G))
           : c.cpt == 4 ? coop3_kernel<T, 512, 4>(c.G)
                        : coop3_kernel<T, 448, 10>(c.G);
}

} // namespace

CoopPlan coop_plan(const Geo& g)
{
    CoopPlan c;
    if (g.dim == 3) {
        c.pencils = coop3_grid(g);
        c.groups = c.pencils.G;
        c.lds = coop3_lds(c.pencils);
        c.xch = ((size_t)c.groups * 16 + 2 * (size_t)g.n[0] * g.n[1] * g.n[2]) * sizeof(Word);
    } else {
        c.strips = coop_grid(g);
        if (c.strips.G > kCoopMaxGroups)
            return c;
        c.lds = coop_lds(g, c.strips);
        if (c.lds > 128 * 1024)
            return c;
        c.groups = c.strips.G;
        c.xch = (size_t)c.groups * (16 + 4 * (size_t)g.n[0]) * sizeof(Word);
    }
    return c;
}

template <class T>
bool launch_pcg_solve_coop(const Geo& g, CoopPlan& plan, T* x, T* r, T* p, PcgState* st,
                           void* xch, unsigned& seq, int max_its, hipStream_t s)
{
    if (std::is_same<T, float>::value && g.dim != 3)
        throw CfError(CF_EINVAL, "the cooperative FP32 PCG is 3-D");
    if (plan.groups < 1)
        throw CfError(CF_EINVAL, "grid does not fit the cooperative PCG");
    if (max_its < 1)
        throw CfError(CF_EINVAL, "the cooperative PCG runs at least one iteration per launch");
    // a word is new when it carries its exchange's number: the numbers go on
    // from launch to launch, and before they wrap the buffer is cleared
    if (seq > 0xffffffffu - 2u * (unsigned)max_its - 2u) {
        CF_HIP(hipMemsetAsync(xch, 0, plan.xch, s));
        seq = 0;
    }
    CoopXch xc;
    xc.part = (Word*)xch;
    xc.halo = xc.part + (size_t)plan.groups * 16;
    xc.seq0 = seq;
    Geo ga = g;
    CoopGrid cg = plan.strips;
    Coop3Grid c3 = plan.pencils;
    T *xa = x, *ra = r, *pa = p;
    PcgState* sta = st;
    int ma = max_its;
    void* args[] = {&ga, &cg, &xa, &ra, &pa, &sta, &xc, &ma};
    const void* fn;
    int* every;
    int lanes;
    if (g.dim == 3) {
        args[1] = &c3;
        fn = coop3_kernel<T>(c3);
        every = &plan.pencils.every;
        lanes = c3.nt;
    } else {
        fn = cg.nt == 256 ? coop_kernel<256, 4>(cg.G)
             : cg.cpt == 4 ? coop_kernel<512, 4>(cg.G)
                           : coop_kernel<448, 10>(cg.G);
        every = &plan.strips.every;
        lanes = cg.nt;
    }
    const bool ran = coop_spread(*every, [&](int spread) {
        cg.every = c3.every = spread;
        const dim3 grid(plan.groups * spread), block(lanes + kWave);
        // A lone workgroup waits for no other: an ordinary launch will do,
        // which costs 20 us less (a 32^2 step 232 -> 211 us).
        const hipError_t e =
            grid.x == 1 ? hipLaunchKernel(fn, grid, block, args, plan.lds, s)
                        : hipLaunchCooperativeKernel(fn, grid, block, args, (unsigned)plan.lds, s);
        if (e == hipErrorCooperativeLaunchTooLarge || e == hipErrorNotSupported) {
            (void)hipGetLastError(); // refused before anything ran
            return false;
        }
        CF_HIP(e);
        return true;
    });
    if (!ran)
        return false;
    seq += 2u * (unsigned)max_its;
    return true;
}
template bool launch_pcg_solve_coop<double>(const Geo&, CoopPlan&, double*, double*, double*,
                                            PcgState*, void*, unsigned&, int, hipStream_t);
template bool launch_pcg_solve_coop<float>(const Geo&, CoopPlan&, float*, float*, float*,
                                           PcgState*, void*, unsigned&, int, hipStream_t);

} // namespace cfmi
