// k_ppe.hip -- the pressure Poisson relaxations of pressure.f (Ppe 30-249).
//
//   SorRB / SorRBP (pressure.f:457-656), Cartesian grid without blockages:
//     k_sor_tiled runs several sweeps per launch on tiles held in registers
//     (temporal blocking, below), bit for bit the reference's iterates.
//   SorRB / SorRBP otherwise: two colour kernels per sweep.  Points of one
//     colour only read points of the other, so every point's arithmetic is
//     the reference's regardless of order; the unrelaxed |s| is max-reduced
//     through per-workgroup partials that the next sweep's kernel folds.
//   Sor (pressure.f:384-450): lexicographic Gauss-Seidel, on Cartesian grids
//     without blockages as a pipeline of sweeps on the same tiles (ST_LEX);
//     otherwise, and for short solves, a row a lane (k_sor_lex_rows) or, past
//     its rows, tile by tile (k_sor_lex).  There a point needs its
//     west and south neighbours of this sweep and its east and north neighbours
//     of the last one, so 64x64 tiles run in wavefront order (each workgroup
//     takes the next tile in row-major order from an atomic ticket and waits for
//     its west and south tiles), and inside a tile the points run along
//     anti-diagonals (a barrier between diagonals).
//   Slor / SlorRB / SlorRBP (pressure.f:673-1138): each j-line is an (nx-1)-row
//     AltTridLU; the lines of one colour are solved as one batch of chains.
//
// Sweep control stays on the device: the stopping test of a sweep (m > 1 and
// dif < sortol, pressure.f:443/534, or m = msorit) is evaluated on the device
// and raises sor_done; every later kernel of the solve returns at entry, so
// the host only looks at the flag every few dozen sweeps.
#include "wd2_dev.hpp"
#include "wd2_launch.hpp"
#include "wd2_sor.hpp"

namespace wd2 {

constexpr int RB_T = 256;

__device__ inline void sor_finish(Scalars *sc, double dif, double sortol, int msorit) {
    const int m = sc->sor_m + 1;
    sc->sor_m = m;
    sc->sor_dif = dif;
    if (m > 1 && dif < sortol) {
        sc->sor_done = 1;
        sc->sor_nconv = m;
    } else if (m >= msorit) {
        sc->sor_done = 1;
    }
}

__device__ inline bool last_arrival(unsigned int *counter, unsigned int nblocks, int tid) {
    __shared__ bool amlast;
    __threadfence();
    __syncthreads();
    if (tid == 0) {
        const unsigned int t = atomicAdd(counter, 1u);
        amlast = (t == nblocks - 1);
        if (amlast) *counter = 0;
    }
    __syncthreads();
    return amlast;
}

// One point update of Sor / SorRB / SorRBP (pressure.f:425-431); returns |s|.
template <bool COEF>
__device__ inline double sor_point(int ld, int i, int j, const double *__restrict__ rau,
                                   const double *__restrict__ rgv, const PpeCoef &cf, const double *__restrict__ b,
                                   double sorrel, double *p) {
    const size_t k = WD2_IX(i, j);
    double a1, a2, a3, a4, a5;
    if (COEF) {
        a1 = cf.a1[k]; a2 = cf.a2[k]; a3 = cf.a3[k]; a4 = cf.a4[k]; a5 = cf.a5[k];
    } else {
        a1 = rgv[WD2_IX(i, j - 1)];
        a2 = rau[WD2_IX(i - 1, j)];
        a4 = rau[k];
        a5 = rgv[k];
        a3 = -a4 - a2 - a5 - a1;
    }
    double sum = b[k] - a1 * p[WD2_IX(i, j - 1)] - a2 * p[WD2_IX(i - 1, j)] - a4 * p[WD2_IX(i + 1, j)] -
                 a5 * p[WD2_IX(i, j + 1)];
    const double pij = p[k];
    sum = sum / a3 - pij;
    p[k] = pij + sorrel * sum;
    return fabs(sum);
}

// Max of n published partial maxima (written by earlier kernels), folded by
// one workgroup; every thread gets the result.
__device__ inline double fold_partials(const double *__restrict__ part, int n, double *sh, int tid) {
    double r = 0.0;
    for (int k = tid; k < n; k += RB_T) r = dmaxf(r, part[k]);
    return block_max<RB_T>(r, sh, tid);
}

// Sweep m of SorRB/SorRBP, one colour.  Before doing any work every
// workgroup evaluates the stopping test of sweep m-1 from that sweep's
// published partial maxima (pressure.f:534: m-1 > 1 and dif < sortol); all
// workgroups of both colour kernels reach the same decision, so the solve
// stops after exactly the sweep the reference stops after.  No device-scope
// fence is needed: partials cross workgroups only through kernel boundaries.
template <int COLOR, bool COEF>
__global__ __launch_bounds__(RB_T) void k_sor_rb(int nx, int ny, int ld, const double *__restrict__ rau,
                                                 const double *__restrict__ rgv, PpeCoef cf,
                                                 const double *__restrict__ b, double sorrel, double sortol, int m,
                                                 double *p, const double *__restrict__ prev_part, int nprev,
                                                 double *__restrict__ cur_part, Scalars *sc) {
    if (sc->sor_done) return;
    __shared__ double sh[RB_T / 64];
    const int tid = threadIdx.x;
    if (m - 1 > 1) {
        const double d = fold_partials(prev_part, nprev, sh, tid);
        if (d < sortol) {
            if (COLOR == 0 && blockIdx.x == 0 && blockIdx.y == 0 && tid == 0) {
                sc->sor_done = 1;
                sc->sor_nconv = m - 1;
                sc->sor_dif = d;
            }
            return;
        }
    }
    double mx = 0.0;
    for (int j = 2 + blockIdx.y; j <= ny; j += gridDim.y) {
        const int i0 = COLOR == 0 ? 2 + (j % 2) : 2 + ((j + 1) % 2);
        const int i = i0 + 2 * (blockIdx.x * RB_T + tid);
        if (i <= nx) mx = dmaxf(mx, sor_point<COEF>(ld, i, j, rau, rgv, cf, b, sorrel, p));
    }
    mx = block_max<RB_T>(mx, sh, tid);
    const unsigned int nb = gridDim.x * gridDim.y, bid = blockIdx.x + gridDim.x * blockIdx.y;
    if (tid == 0) cur_part[COLOR * nb + bid] = mx;
}

// Stopping test of the last launched sweep m (one workgroup).
__global__ __launch_bounds__(RB_T) void k_sor_check(const double *__restrict__ part, int n, int m, double sortol,
                                                    int msorit, Scalars *sc) {
    if (sc->sor_done) return;
    __shared__ double sh[RB_T / 64];
    const double d = fold_partials(part, n, sh, threadIdx.x);
    if (threadIdx.x == 0) {
        sc->sor_dif = d;
        if (m > 1 && d < sortol) {
            sc->sor_done = 1;
            sc->sor_nconv = m;
        } else if (m >= msorit) {
            sc->sor_done = 1;
        }
    }
}

static dim3 rb_grid(int nx, int ny) {
    const int per_row = (nx / 2 + RB_T - 1) / RB_T;
    const int rows = min(ny - 1, max(1, 512 / per_row));
    return dim3(per_row, rows);
}

int sor_rb_partials(int nx, int ny) {
    const dim3 g = rb_grid(nx, ny);
    return 2 * g.x * g.y;
}

void launch_sor_rb_sweep(int nx, int ny, int ld, const Metrics &m, const PpeCoef *coef, const double *b,
                         double sorrel, double sortol, int sweep, double *p, double *partials, Scalars *sc,
                         hipStream_t s, hipEvent_t *ev) {
    const dim3 g = rb_grid(nx, ny);
    const int np = 2 * g.x * g.y;
    const double *prev = partials + (size_t)((sweep - 1) & 1) * np;
    double *cur = partials + (size_t)(sweep & 1) * np;
    PpeCoef cf = coef ? *coef : PpeCoef{nullptr, nullptr, nullptr, nullptr, nullptr};
    for (int color = 0; color < 2; color++) {
        if (ev) (void)hipEventRecord(ev[2 * color], s);
        if (coef) {
            if (color == 0)
                hipLaunchKernelGGL((k_sor_rb<0, true>), g, dim3(RB_T), 0, s, nx, ny, ld, m.rau, m.rgv, cf, b, sorrel,
                                   sortol, sweep, p, prev, np, cur, sc);
            else
                hipLaunchKernelGGL((k_sor_rb<1, true>), g, dim3(RB_T), 0, s, nx, ny, ld, m.rau, m.rgv, cf, b, sorrel,
                                   sortol, sweep, p, prev, np, cur, sc);
        } else {
            if (color == 0)
                hipLaunchKernelGGL((k_sor_rb<0, false>), g, dim3(RB_T), 0, s, nx, ny, ld, m.rau, m.rgv, cf, b,
                                   sorrel, sortol, sweep, p, prev, np, cur, sc);
            else
                hipLaunchKernelGGL((k_sor_rb<1, false>), g, dim3(RB_T), 0, s, nx, ny, ld, m.rau, m.rgv, cf, b,
                                   sorrel, sortol, sweep, p, prev, np, cur, sc);
        }
        if (ev) (void)hipEventRecord(ev[2 * color + 1], s);
    }
}

void launch_sor_rb_check(int nx, int ny, int sweep, double sortol, int msorit, const double *partials,
                         Scalars *sc, hipStream_t s) {
    const int np = sor_rb_partials(nx, ny);
    hipLaunchKernelGGL(k_sor_check, dim3(1), dim3(RB_T), 0, s, partials + (size_t)(sweep & 1) * np, np, sweep,
                       sortol, msorit, sc);
}

// --------------------------------------------- temporally blocked SorRB
// Cartesian grids without blockages: the right-hand side and the five
// coefficients do not change during the solve, so a workgroup can run many
// sweeps on a tile it holds.  A tile is ST_W x ST_W points with a halo of
// 2 * nsweep cells: a red-black sweep moves the dependence front by two cells
// (black points read red neighbours, red points read the new black ones), so
// after the sweeps every owned point has seen exactly the values it sees in
// the global sweep order, and its arithmetic is the reference's.  Points of
// the outermost ring are never updated.
//
// The tile lives in registers: a lane holds a strip of ST_R rows of a pair of
// columns (32 lanes a strip, 16 strips), with its right-hand side,
// coefficients and reciprocal diagonals.  A colour takes one point of each
// row's pair, the same one in every lane, so of its four neighbours one is the
// lane's own pair mate, two are its own rows above and below, and one comes by
// a lane shift; only the rows at a strip's ends cross through LDS.  A half
// sweep is bound by its instructions (about 22 double-precision ones a point,
// 2048 points over four SIMDs) and one LDS exchange; a launch by those and
// about 5 us of launch gap, stopping test, loads and stores.  With p in LDS,
// five LDS reads a point, a plain division and four sweeps a launch, a sweep
// took 3.1 us on 251 x 243 cells, 6.5 on 1000^2 and, with uniform coefficients,
// 2.8 on 64^2, 2.9 on 512^2 and 4.2 on 1024^2; here 1.5, 4.5, 0.9, 1.3 and 2.9.
//
// ST_WHOLE: a grid of at most ST_W x ST_W interior points is one tile without a
// halo: the ghost cells are constants, and one workgroup runs the sweeps of
// the whole solve with the stopping test after each (0.9 us a sweep where
// tiles of 14 sweeps a launch take 1.0).
//
// ST_LEX: Sor (pressure.f:384-450), the lexicographic sweeps.  A point needs
// its west and south neighbours of its own sweep and its east and north ones
// of the sweep before, so at half sweep T every point with i + j of T's parity
// can run its sweep m = (T - i - j) / 2: a lexicographic solve of M sweeps is
// a red-black one of (nx + ny) / 2 + M in which a point starts at its first
// sweep and stops after its last, value for value the reference's.  A sweep's
// stopping test is known when the last point has run it; the tiles gather it
// as bits of sweeps with a point not below sortol.  A row a lane, a sweep of
// 97 x 75 cells took 73 us; here 1.4.
//
// With ST_TILES and ST_LEX the kernel reads p_in and writes the owned points to p_out (tiles
// read their neighbours' points as halo, so it cannot work in place).  The
// stopping test of sweep m is max|s| < sortol over the whole grid
// (pressure.f:534), which holds exactly when it holds on every tile: each tile
// publishes a bit mask of its sweeps whose owned-point maximum is below
// sortol, and the test of a launch is the AND of the masks.  Before any work,
// every workgroup evaluates the previous launch's test; all reach the same
// decision, so a solve that stopped is never advanced further.
//
// Division by the fixed diagonal, MODE 0 and 1: with r = 1/d correctly rounded,
// two steps q += fma(-d, q, x) * r from q = x * r give the correctly rounded
// x / d (Markstein, IBM J. Res. Dev. 34, 1990: the first makes q faithful, the
// second rounds it correctly) as long as nothing under- or overflows; d is
// checked once, and a wavefront that meets a quotient that is tiny, zero or
// not a number divides instead.  MODE 2: every diagonal is a power of two, so
// x / d == x * (1 / d) bit for bit.
constexpr int ST_T = 512, ST_W = 64, ST_R = 4;
constexpr int ST_L = ST_W / 2;       // lanes of a strip
constexpr int ST_N = ST_W / ST_R;    // strips
constexpr double ST_TINY = 0x1p-400, ST_HUGE = 0x1p400;

enum { ST_TILES = 0, ST_WHOLE = 1, ST_LEX = 2 };

template <int CTRL>
__device__ inline double st_dpp(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

struct StArgs {
    int nx, ny, ld, nsweep, m0, msorit;
    int prev_nsweep, prev_m0, prev_launch;
    int ntx, ntiles, own, force;
    double sorrel, sortol, rau_c, rgv_c, d_c, rd_c;   // uniform: the diagonal and its reciprocal
    const double *rau, *rgv, *b, *p_in;
    double *p_out;
    unsigned *masks;
    const unsigned *prev_masks;
    Scalars *sc;
    int pair, cap;     // ST_LEX: first pair of half sweeps, last sweep
    unsigned *bits;    // ST_LEX: bit m - 1: some point's |s| in sweep m is not below sortol
};

// One lane's part of a tile.  [r][h]: row r of the strip, column h of the pair.
template <int MODE>
struct StTile {
    double p[ST_R][2], b[ST_R][2];
    double g[ST_R + 1][2], a[ST_R][2], aw[ST_R], d[ST_R][2], rd[ST_R][2];   // MODE 0
    bool up[ST_R][2];                  // the point is updated
    unsigned long long own[ST_R][2];   // lanes whose point is owned
    bool divide;
};

// The points of colour C ((i + j) & 1 == C) of one half sweep.  sS, sN: the
// rows below and above the strip; gw, ge: ST_WHOLE, the west ghosts of a
// strip's first lane and the east ones of its last.  act, ST_LEX: whether the
// points with (r + h) / 2 = 0, 1, 2 are within their sweeps.  big[] receives
// the lanes that own a point whose |s| is not below sortol (a NaN counts as
// not converged), by the same index with ST_LEX, else all in big[0].
template <int MODE, int KIND, int C>
__device__ __forceinline__ void st_half(StTile<MODE> &t, double sS, double sN, const double *gw, const double *ge,
                                        int l, const StArgs &A, const bool *act, unsigned long long *big) {
    constexpr bool WHOLE = KIND == ST_WHOLE, LEX = KIND == ST_LEX;
    double x[ST_R], q[ST_R];
    bool bad = MODE != 2 && t.divide;
    // the inner rows first, kept there by the empty asm: the end rows'
    // neighbours are on their way from LDS
#pragma unroll
    for (int k = 0; k < ST_R; k++) {
        const int r = (k + 1) % ST_R, h = (r ^ C) & 1;
        if (k == ST_R - 2) asm volatile("" : "+v"(sS), "+v"(sN) : "v"(q[1]), "v"(q[2]));
        double W, E;
        if (h) {
            W = t.p[r][0];
            E = st_dpp<0x130>(t.p[r][0]);   // wave_shl:1
            if (WHOLE) E = l == ST_L - 1 ? ge[r] : E;
        } else {
            W = st_dpp<0x138>(t.p[r][1]);   // wave_shr:1
            if (WHOLE) W = l == 0 ? gw[r] : W;
            E = t.p[r][1];
        }
        const double S = r > 0 ? t.p[r > 0 ? r - 1 : 0][h] : sS;
        const double N = r < ST_R - 1 ? t.p[r < ST_R - 1 ? r + 1 : 0][h] : sN;
        const double a1 = MODE ? A.rgv_c : t.g[r][h], a5 = MODE ? A.rgv_c : t.g[r + 1][h];
        const double a2 = MODE ? A.rau_c : (h ? t.a[r][0] : t.aw[r]), a4 = MODE ? A.rau_c : t.a[r][h];
        const double rd = MODE ? A.rd_c : t.rd[r][h], d = MODE ? A.d_c : t.d[r][h];
        // the reference's order: b - a1 pS - a2 pW - a4 pE - a5 pN
        x[r] = t.b[r][h] - a1 * S - a2 * W - a4 * E - a5 * N;
        q[r] = x[r] * rd;
        if (MODE != 2) {
            q[r] = __builtin_fma(__builtin_fma(-d, q[r], x[r]), rd, q[r]);
            q[r] = __builtin_fma(__builtin_fma(-d, q[r], x[r]), rd, q[r]);
            bad |= t.up[r][h] && (!LEX || act[(r + h) / 2]) && !(fabs(q[r]) > ST_TINY);
        }
    }
    if (MODE != 2 && __any(bad)) {
#pragma unroll
        for (int r = 0; r < ST_R; r++) q[r] = x[r] / (MODE ? A.d_c : t.d[r][(r ^ C) & 1]);
    }
#pragma unroll
    for (int r = 0; r < ST_R; r++) {
        const int h = (r ^ C) & 1, dl = (r + h) / 2;
        const bool up = t.up[r][h] && (!LEX || act[dl]);
        const double s = q[r] - t.p[r][h];
        const double pn = t.p[r][h] + A.sorrel * s;
        t.p[r][h] = up ? pn : t.p[r][h];
        const unsigned long long b = __ballot(!(fabs(s) < A.sortol)) & t.own[r][h];
        if (LEX) big[dl] |= b & __ballot(act[dl]);
        else big[0] |= b;
    }
}

template <int MODE, int KIND>
__global__ __launch_bounds__(ST_T, KIND == ST_WHOLE ? 2 : 4) void k_sor_tiled(StArgs A) {
    constexpr bool WHOLE = KIND == ST_WHOLE, LEX = KIND == ST_LEX;
    // the strips' first and last rows by colour; strips 0 and ST_N + 1 are the
    // rows below and above the tile (WHOLE: the ghost rows)
    __shared__ double EB[2][ST_N + 2][ST_L], ET[2][ST_N + 2][ST_L];
    __shared__ unsigned sh[ST_T / 64];
    __shared__ int more[2];
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & (ST_L - 1), st = tid / ST_L;
    const int nx = A.nx, ny = A.ny, ld = A.ld;
    // XCD-aware tile order: consecutive workgroups go to different XCDs, so
    // give each XCD a contiguous band of tiles (their halos then share an L2).
    const int per = (A.ntiles + 7) / 8;
    const int tile = WHOLE ? 0 : (blockIdx.x % 8) * per + blockIdx.x / 8;
    const int halo = WHOLE ? 0 : (ST_W - A.own) / 2;
    const int TI = tile % A.ntx, TJ = tile / A.ntx;
    const int i0 = 2 + TI * A.own - halo, j0 = 2 + TJ * A.own - halo;   // tile origin, both even
    const int x = 2 * l, y = ST_R * st, i = i0 + x, j = j0 + y;
    // the loads need no answer from the earlier launch: they are in flight
    // while its stopping test is evaluated
    StTile<MODE> t;
#pragma unroll
    for (int r = 0; r < ST_R; r++) {
        const double2 pv = load_pair_sel(A.p_in, ld, nx, ny, i, j + r);
        const double2 bv = load_pair_sel(A.b, ld, nx, ny, i, j + r);
        t.p[r][0] = pv.x; t.p[r][1] = pv.y;
        t.b[r][0] = bv.x; t.b[r][1] = bv.y;
    }
    if (MODE == 0) {
#pragma unroll
        for (int r = 0; r < ST_R; r++) {
            const double2 gv = load_pair_sel(A.rgv, ld, nx, ny, i, j + r - 1);
            const double2 av = load_pair_sel(A.rau, ld, nx, ny, i, j + r);
            t.g[r][0] = gv.x; t.g[r][1] = gv.y;
            t.a[r][0] = av.x; t.a[r][1] = av.y;
            t.aw[r] = A.rau[(size_t)min(max(i - 1, 0), ld - 1) + (size_t)ld * (size_t)min(max(j + r, 0), ny + 1)];
        }
        const double2 gv = load_pair_sel(A.rgv, ld, nx, ny, i, j + ST_R - 1);
        t.g[ST_R][0] = gv.x; t.g[ST_R][1] = gv.y;
    }
    double gw[ST_R] = {}, ge[ST_R] = {};
    if (WHOLE) {
#pragma unroll
        for (int r = 0; r < ST_R; r++) {
            gw[r] = load_pair_sel(A.p_in, ld, nx, ny, 0, j + r).y;
            ge[r] = load_pair_sel(A.p_in, ld, nx, ny, 2 + ST_W, j + r).x;
        }
    }
    if (!A.force && A.sc->sor_done) return;
    if (KIND == ST_TILES && !A.force && A.prev_nsweep > 0) {
        int conv = 0;
        const int k = tiled_stop(tiled_mask(A.prev_masks, A.ntiles, sh), A.prev_nsweep, A.prev_m0, A.msorit, &conv);
        if (k > 0) {
            if (blockIdx.x == 0 && tid == 0) {
                A.sc->sor_done = 1;
                A.sc->sor_nconv = conv ? A.prev_m0 + k : 0;
                A.sc->sor_m = A.prev_m0 + k;
                A.sc->redo_launch = A.prev_launch;
                A.sc->redo_sweeps = k;
            }
            return;
        }
    }
    if (tile >= A.ntiles) return;
    bool divide = false, any_up = false;
#pragma unroll
    for (int r = 0; r < ST_R; r++) {
        const int yy = y + r, jj = j + r;
        const bool row = jj >= 2 && jj <= ny && (WHOLE || (yy >= 1 && yy <= ST_W - 2));
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int xx = x + h, ii = i + h;
            const bool u = row && ii >= 2 && ii <= nx && (WHOLE || (xx >= 1 && xx <= ST_W - 2));
            t.up[r][h] = u;
            t.own[r][h] =
                __ballot(u && xx >= halo && xx < ST_W - halo && yy >= halo && yy < ST_W - halo);
            any_up = any_up || __any(u);
            if (MODE == 0) {
                // a3 = -a4 - a2 - a5 - a1, the reference's expression; a point
                // that is not updated keeps its value whatever it computes
                const double a2 = h ? t.a[r][0] : t.aw[r];
                const double d = -t.a[r][h] - a2 - t.g[r + 1][h] - t.g[r][h];
                t.d[r][h] = u ? d : -1.0;
                t.rd[r][h] = 1.0 / t.d[r][h];
                divide |= !(fabs(t.d[r][h]) > ST_TINY && fabs(t.d[r][h]) < ST_HUGE);
            }
        }
    }
    t.divide = divide;
    for (int k = tid; k < 4 * ST_L; k += ST_T) {
        // rows j0 - 1 (ET of strip 0) and j0 + ST_W (EB of strip ST_N + 1), by colour
        const int c = (k / ST_L) & 1, top = k / (2 * ST_L), kl = k % ST_L;
        double v = 0.0;
        if (WHOLE) {
            const int jj = top ? 2 + ST_W : 1, h = top ? c : 1 - c, ii = 2 + 2 * kl + h;
            if (jj <= ny + 1 && ii <= nx + 1) v = A.p_in[WD2_IX(ii, jj)];
        }
        if (top) EB[c][ST_N + 1][kl] = v;
        else ET[c][0][kl] = v;
    }
    EB[0][st + 1][l] = t.p[0][0];
    EB[1][st + 1][l] = t.p[0][1];
    ET[1][st + 1][l] = t.p[ST_R - 1][0];
    ET[0][st + 1][l] = t.p[ST_R - 1][1];
    if (tid < 2) more[tid] = 0;
    __syncthreads();
    const int lo_w = 8 * w, hi_w = 8 * w + 7;   // the wavefront's rows
    unsigned below = 0;   // bit s: the wavefront's owned max |s| of sweep s is < sortol
    // ST_LEX: the lane's sweep m - 1 at s = 0, (r + h) / 2 = 0, the
    // wavefront's first lane's, and the sweeps with a point not below sortol
    // (bit k: m - 1 = base_w - 35 + k)
    const int base_w = A.pair - (i0 + j0) / 2 - 1 - 4 * w, base = A.pair - (i0 + j0) / 2 - 1 - l - 2 * st;
    unsigned long long acc = 0;
    for (int s = 0; s < A.nsweep; s++) {
        // rows that the owned points still depend on: one less a side per half sweep
        const int rem = 2 * (A.nsweep - 1 - s);
        const bool act0 = WHOLE ? any_up : (hi_w >= halo - rem - 1 && lo_w <= ST_W - halo + rem);
        const bool act1 = WHOLE ? any_up : (hi_w >= halo - rem && lo_w <= ST_W - halo - 1 + rem);
        if (WHOLE && s > 0) {
            // the test of the sweep before
            const int m = A.m0 + s;
            if (m > 1 && !__builtin_amdgcn_readfirstlane(more[(s - 1) & 1])) {
                if (tid == 0) {
                    A.sc->sor_done = 1;
                    A.sc->sor_nconv = A.sc->sor_m = m;
                }
                below = 1;
                break;
            }
        }
        unsigned long long big[3] = {0, 0, 0};
        bool act[3] = {true, true, true};
        bool on = true;   // ST_LEX: some lane's points are within their sweeps
        if (LEX) {
#pragma unroll
            for (int d = 0; d < 3; d++) act[d] = (unsigned)(base + s - d) < (unsigned)A.cap;
            on = __any(act[0] || act[1] || act[2]);
        }
        if (act0 && on) {
            st_half<MODE, KIND, 0>(t, ET[1][st][l], EB[1][st + 2][l], gw, ge, l, A, act, big);
            EB[0][st + 1][l] = t.p[0][0];
            ET[0][st + 1][l] = t.p[ST_R - 1][1];
        }
        __syncthreads();
        if (WHOLE && tid == 0) more[(s + 1) & 1] = 0;
        if (act1 && on) {
            st_half<MODE, KIND, 1>(t, ET[0][st][l], EB[0][st + 2][l], gw, ge, l, A, act, big);
            EB[1][st + 1][l] = t.p[0][1];
            ET[1][st + 1][l] = t.p[ST_R - 1][0];
        }
        if (WHOLE) {
            if (big[0] != 0) more[s & 1] = 1;
        } else if (LEX) {
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const unsigned long long x = __brevll(big[d]);
                acc |= ((x & 0xffffffffull) | ((x >> 32) << 2)) << (s + 2 - d);
            }
        } else if (big[0] == 0) {
            below |= 1u << s;
        }
        __syncthreads();
    }
    if (WHOLE && !below && tid == 0) {   // ran all its sweeps: the last one's test
        const int m = A.m0 + A.nsweep;
        const bool ok = m > 1 && !more[(A.nsweep - 1) & 1];
        if (ok || m >= A.msorit) {
            A.sc->sor_done = 1;
            A.sc->sor_nconv = ok ? m : 0;
        }
        A.sc->sor_m = m;
    }
    const unsigned long long me = 1ull << (tid & 63);
#pragma unroll
    for (int r = 0; r < ST_R; r++) {
        double *q = A.p_out + WD2_IX(i, j + r);
        if ((t.own[r][0] & t.own[r][1]) & me) *reinterpret_cast<double2 *>(q) = make_double2(t.p[r][0], t.p[r][1]);
        else if (t.own[r][0] & me) q[0] = t.p[r][0];
        else if (t.own[r][1] & me) q[1] = t.p[r][1];
    }
    if (WHOLE) return;
    if (LEX) {
        const int lane = tid & 63, b0 = base_w - 35, off = b0 & 31;
        if (lane < 3) {
            const unsigned long long lo = acc << off;
            const unsigned v = lane == 0 ? (unsigned)lo : lane == 1 ? (unsigned)(lo >> 32)
                                                        : off ? (unsigned)(acc >> (64 - off)) : 0u;
            // most sweeps' bits are set by the first tile that gets there
            if (v) {
                unsigned *q = A.bits + (b0 >> 5) + lane;
                if ((__hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & v) != v) atomicOr(q, v);
            }
        }
        return;
    }
    // tile mask = AND over the wavefronts (below is the same in every lane of one)
    if ((tid & 63) == 0) sh[w] = below;
    __syncthreads();
    if (tid == 0) {
        unsigned r = ~0u;
        for (int k = 0; k < ST_T / 64; k++) r &= sh[k];
        A.masks[tile] = r;
    }
}

// Stopping test of the last launch of a batch (one workgroup).
__global__ __launch_bounds__(RB_T) void k_sor_tiled_check(const unsigned *__restrict__ masks, int ntiles,
                                                          int nsweep, int m0, int launch, int msorit, Scalars *sc) {
    if (sc->sor_done) return;
    __shared__ unsigned sh[RB_T / 64];
    int conv = 0;
    const int k = tiled_stop(tiled_mask(masks, ntiles, sh), nsweep, m0, msorit, &conv);
    if (threadIdx.x == 0 && k > 0) {
        sc->sor_done = 1;
        sc->sor_nconv = conv ? m0 + k : 0;
        sc->sor_m = m0 + k;
        sc->redo_launch = launch;
        sc->redo_sweeps = k;
    }
}

bool sor_whole(int nx, int ny) { return nx - 1 <= ST_W && ny - 1 <= ST_W; }

static int st_tiles(int nx, int ny, int k, int *ntx) {
    const int own = ST_W - 4 * k, tx = (nx - 1 + own - 1) / own, ty = (ny - 1 + own - 1) / own;
    if (ntx) *ntx = tx;
    return tx * ty;
}
// The sweeps of a launch, the fewest microseconds a sweep by a fit to measured
// launches (251 x 243 to 2048^2, array coefficients): with n tiles on the
// busiest of 256 CUs a launch of K sweeps takes 3 + 3.4 n + 0.5 (1 + n) K us.
// Few tiles make long launches pay (up to K = 14, when a tile owns 8 x 8 of
// its points); with every CU full the halo's work decides (K = 4 or 5).
int sor_tiled_sweeps(int nx, int ny) {
    int best = 4;
    double cost = 1e300;
    for (int k = 4; k <= 14; k++) {
        const int nt = st_tiles(nx, ny, k, nullptr);
        if (k > 8 && nt > 1024) break;   // (the mask buffers hold these)
        const int n = (nt + 255) / 256;
        const double c = (3.0 + 3.4 * n) / k + 0.5 * (1 + n);
        if (c < cost) {
            cost = c;
            best = k;
        }
    }
    return best;
}

int sor_tiled_tiles(int nx, int ny, int *ntx) { return st_tiles(nx, ny, sor_tiled_sweeps(nx, ny), ntx); }

// The uniform coefficients, their diagonal and its reciprocal, and the kernel's MODE.
static int st_uniform(const double *uni, StArgs &A) {
    if (!uni) return 0;
    A.rau_c = uni[0];
    A.rgv_c = uni[1];
    A.d_c = -uni[0] - uni[0] - uni[1] - uni[1];   // the kernel's order of operations
    A.rd_c = 1.0 / A.d_c;
    int e2 = 0;
    if (!(std::fabs(A.d_c) > ST_TINY && std::fabs(A.d_c) < ST_HUGE)) return 0;
    return std::frexp(A.d_c, &e2) == -0.5 ? 2 : 1;
}

void launch_sor_tiled(int nx, int ny, int ld, const Metrics &m, const double *b, double sorrel, int nsweep,
                      const double *p_in, double *p_out, unsigned *masks, const unsigned *prev_masks,
                      int prev_nsweep, int prev_m0, int prev_launch, double sortol, int msorit, Scalars *sc,
                      int force, const double *uni, hipStream_t s) {
    int ntx = 0;
    const int nt = sor_tiled_tiles(nx, ny, &ntx);
    StArgs A{nx, ny, ld, nsweep, 0, msorit, prev_nsweep, prev_m0, prev_launch, ntx, nt, ST_W - 4 * sor_tiled_sweeps(nx, ny), force,
                   sorrel, sortol, 0.0, 0.0, 0.0, 0.0, m.rau, m.rgv, b, p_in, p_out, masks,
             prev_masks, sc, 0, 0, nullptr};
    const dim3 g(8 * ((nt + 7) / 8));
    const int mode = st_uniform(uni, A);
    if (mode == 2) hipLaunchKernelGGL((k_sor_tiled<2, ST_TILES>), g, dim3(ST_T), 0, s, A);
    else if (mode == 1) hipLaunchKernelGGL((k_sor_tiled<1, ST_TILES>), g, dim3(ST_T), 0, s, A);
    else hipLaunchKernelGGL((k_sor_tiled<0, ST_TILES>), g, dim3(ST_T), 0, s, A);
}

void launch_sor_lex_tiled(int nx, int ny, int ld, const Metrics &m, const double *b, double sorrel, int npair,
                          int pair, int cap, const double *p_in, double *p_out, unsigned *bits, double sortol,
                          Scalars *sc, int force, const double *uni, hipStream_t s) {
    int ntx = 0;
    const int nt = sor_tiled_tiles(nx, ny, &ntx);
    StArgs A{nx, ny, ld, npair, 0, 0, 0, 0, 0, ntx, nt, ST_W - 4 * sor_tiled_sweeps(nx, ny), force,
             sorrel, sortol, 0.0, 0.0, 0.0, 0.0, m.rau, m.rgv, b, p_in, p_out, nullptr,
             nullptr, sc, pair, cap, bits};
    const dim3 g(8 * ((nt + 7) / 8));
    const int mode = st_uniform(uni, A);
    if (mode == 2) hipLaunchKernelGGL((k_sor_tiled<2, ST_LEX>), g, dim3(ST_T), 0, s, A);
    else if (mode == 1) hipLaunchKernelGGL((k_sor_tiled<1, ST_LEX>), g, dim3(ST_T), 0, s, A);
    else hipLaunchKernelGGL((k_sor_tiled<0, ST_LEX>), g, dim3(ST_T), 0, s, A);
}

// Start of a solve: the ghost frame of p (which no sweep writes) into the
// other buffers, and the sweeps' bits cleared.
__global__ __launch_bounds__(256) void k_lex_begin(int nx, int ny, int ld, const double *p, LexBufs o, unsigned *bits,
                                                   int nwords) {
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q < nwords) bits[q] = 0;
    const int nr = 3 * (nx + 2), n = nr + 3 * (ny + 2);
    if (q >= n) return;
    const int a = q < nr ? q % (nx + 2) : (q - nr) % (ny + 2), e = q < nr ? q / (nx + 2) : (q - nr) / (ny + 2);
    const size_t k = q < nr ? WD2_IX(a, e < 2 ? e : ny + 1) : WD2_IX(e < 2 ? e : nx + 1, a);
    const double v = p[k];
#pragma unroll
    for (int c = 0; c < LEX_BUFS; c++) o.b[c][k] = v;
}

void launch_lex_begin(int nx, int ny, int ld, const double *p, const LexBufs &o, unsigned *bits, int cap,
                      hipStream_t s) {
    const int nwords = (cap + 31) / 32, n = std::max(nwords, 3 * (nx + 2) + 3 * (ny + 2));
    hipLaunchKernelGGL(k_lex_begin, dim3((n + 255) / 256), dim3(256), 0, s, nx, ny, ld, p, o, bits, nwords);
}

// The stopping test of sweeps m_lo .. m_hi, all complete (one wavefront): the
// first of them, but not the solve's first sweep, without a point that is not
// below sortol; cap: the last sweep of the run (m0 sweeps came before it).
__global__ __launch_bounds__(64) void k_lex_check(const unsigned *bits, int m_lo, int m_hi, int m0, int cap,
                                                  Scalars *sc) {
    if (sc->sor_done) return;
    int best = 0x7fffffff;
    for (int w = (m_lo - 1) / 32 + threadIdx.x; w <= (m_hi - 1) / 32; w += 64) {
        unsigned ok = ~bits[w];
        if (32 * w + 1 < m_lo) ok &= ~0u << (m_lo - 1 - 32 * w);
        if (32 * w + 32 > m_hi) ok &= ~0u >> (32 * w + 32 - m_hi);
        if (m0 == 0 && w == 0) ok &= ~1u;
        if (ok) {
            best = 32 * w + __ffs(ok);
            break;
        }
    }
    for (int off = 32; off > 0; off >>= 1) best = min(best, __shfl_xor(best, off));
    if (threadIdx.x == 0 && (best <= m_hi || m_hi >= cap)) {
        sc->sor_done = 1;
        sc->sor_nconv = best <= m_hi ? m0 + best : 0;
        sc->sor_m = best <= m_hi ? best : cap;
    }
}

void launch_lex_check(const unsigned *bits, int m_lo, int m_hi, int m0, int cap, Scalars *sc, hipStream_t s) {
    hipLaunchKernelGGL(k_lex_check, dim3(1), dim3(64), 0, s, bits, m_lo, m_hi, m0, cap, sc);
}

void launch_sor_whole(int nx, int ny, int ld, const Metrics &m, const double *b, double sorrel, int nsweep, int m0,
                      double *p, double sortol, int msorit, Scalars *sc, const double *uni, hipStream_t s) {
    StArgs A{nx, ny, ld, nsweep, m0, msorit, 0, 0, 0, 1, 1, ST_W, 0,
                   sorrel, sortol, 0.0, 0.0, 0.0, 0.0, m.rau, m.rgv, b, p, p, nullptr,
             nullptr, sc, 0, 0, nullptr};
    const int mode = st_uniform(uni, A);
    if (mode == 2) hipLaunchKernelGGL((k_sor_tiled<2, ST_WHOLE>), dim3(1), dim3(ST_T), 0, s, A);
    else if (mode == 1) hipLaunchKernelGGL((k_sor_tiled<1, ST_WHOLE>), dim3(1), dim3(ST_T), 0, s, A);
    else hipLaunchKernelGGL((k_sor_tiled<0, ST_WHOLE>), dim3(1), dim3(ST_T), 0, s, A);
}

void launch_sor_tiled_check(int ntiles, int nsweep, int m0, int launch, int msorit, const unsigned *masks,
                            Scalars *sc, hipStream_t s) {
    hipLaunchKernelGGL(k_sor_tiled_check, dim3(1), dim3(RB_T), 0, s, masks, ntiles, nsweep, m0, launch, msorit, sc);
}

__global__ void k_sor_reset(Scalars *sc) {
    sc->sor_done = 0;
    sc->sor_nconv = 0;
    sc->sor_m = 0;
    sc->sor_dif = 0.0;
    sc->val[6] = 0.0;
    sc->redo_launch = 0;
    sc->redo_sweeps = 0;
}
void launch_sor_reset(Scalars *sc, hipStream_t s) { hipLaunchKernelGGL(k_sor_reset, dim3(1), dim3(1), 0, s, sc); }

// ------------------------------------------------------- lexicographic Sor
constexpr int LX_T = 64;          // one wavefront per tile
constexpr int LX_TI = 64, LX_TJ = 64;

template <bool COEF>
__global__ __launch_bounds__(LX_T) void k_sor_lex(int nx, int ny, int ld, const double *__restrict__ rau,
                                                  const double *__restrict__ rgv, PpeCoef cf,
                                                  const double *__restrict__ b, double sorrel, double sortol,
                                                  int msorit, double *p, int *tile_flags, int sweep,
                                                  double *__restrict__ partials, Scalars *sc) {
    if (sc->sor_done) return;
    __shared__ int ticket;
    __shared__ double sh[1];
    const int t = threadIdx.x;
    const int ntx = (nx - 1 + LX_TI - 1) / LX_TI, nty = (ny - 1 + LX_TJ - 1) / LX_TJ;
    const unsigned int ntiles = ntx * nty;
    if (t == 0) ticket = (int)atomicAdd(&sc->counter[5], 1u);
    __syncthreads();
    const int tile = ticket;
    const int TI = tile % ntx, TJ = tile / ntx;
    // wait for the west and south tiles of this sweep
    if (t == 0) {
        if (TI > 0)
            while (__hip_atomic_load(&tile_flags[tile - 1], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) < sweep)
                __builtin_amdgcn_s_sleep(1);
        if (TJ > 0)
            while (__hip_atomic_load(&tile_flags[tile - ntx], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) < sweep)
                __builtin_amdgcn_s_sleep(1);
    }
    __syncthreads();
    const int i0 = 2 + TI * LX_TI, j0 = 2 + TJ * LX_TJ;
    const int ni = min(LX_TI, nx - i0 + 1), nj = min(LX_TJ, ny - j0 + 1);
    // column i0 + t, rows j0 .. j0+nj-1, walked along anti-diagonals
    double mx = 0.0;
    for (int step = 0; step < nj + LX_T - 1; step++) {
        const int jj = step - t;
        if (t < ni && jj >= 0 && jj < nj) {
            const int i = i0 + t, j = j0 + jj;
            const size_t k = WD2_IX(i, j);
            double a1, a2, a3, a4, a5;
            if (COEF) {
                a1 = cf.a1[k]; a2 = cf.a2[k]; a3 = cf.a3[k]; a4 = cf.a4[k]; a5 = cf.a5[k];
            } else {
                a1 = rgv[WD2_IX(i, j - 1)]; a2 = rau[WD2_IX(i - 1, j)]; a4 = rau[k]; a5 = rgv[k];
                a3 = -a4 - a2 - a5 - a1;
            }
            // neighbours written during this sweep by other lanes or tiles are
            // read through the coherent path
            const double pS = ld_coherent(&p[WD2_IX(i, j - 1)]);
            const double pW = ld_coherent(&p[WD2_IX(i - 1, j)]);
            const double pE = p[WD2_IX(i + 1, j)], pN = p[WD2_IX(i, j + 1)];
            double sum = b[k] - a1 * pS - a2 * pW - a4 * pE - a5 * pN;
            const double pij = p[k];
            sum = sum / a3 - pij;
            const double pnew = pij + sorrel * sum;
            __hip_atomic_store((unsigned long long *)&p[k], dbits(pnew), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
            mx = dmaxf(mx, fabs(sum));
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __syncthreads();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }
    for (int off = 32; off > 0; off >>= 1) mx = dmaxf(mx, __shfl_xor(mx, off));
    if (t == 0) {
        partials[tile] = mx;
        __hip_atomic_store(&tile_flags[tile], sweep, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (last_arrival(&sc->counter[6], ntiles, t)) {
        double r = 0.0;
        for (unsigned int k = t; k < ntiles; k += LX_T) r = dmaxf(r, ld_coherent(&partials[k]));
        for (int off = 32; off > 0; off >>= 1) r = dmaxf(r, __shfl_xor(r, off));
        if (t == 0) {
            sc->counter[5] = 0;
            sor_finish(sc, r, sortol, msorit);
        }
    }
    (void)sh;
}

// Lexicographic Sor, whole solve in one workgroup (grids of up to LR_MAXROWS
// rows).  Each lane owns one grid row j = 2 + lane and walks it from i = 2 to
// nx; the lanes of a wavefront run skewed by one column per lane, so at every
// step lane L updates the point whose south neighbour lane L-1 updated in the
// previous step (passed by a lane shuffle) and whose west neighbour is the
// lane's own previous point: exactly the reference's i-then-j order.  East,
// north and the point's old value are read from the previous sweep's field.
// Wavefront w starts LR_LAG steps after wavefront w-1 and takes the south
// values of its first row from a ring that w-1's last lane fills; with a
// workgroup barrier every LR_K steps a ring value is always at least one
// barrier old when it is read.  The stopping test (pressure.f:443) is applied
// in the kernel after every sweep, so the whole solve is one launch.
// Non-Cartesian grids re-form the right-hand side before every sweep
// (pressure.f:RhsPpe, as in the reference).
constexpr int LR_K = 16;                // steps between two barriers
constexpr int LR_LAG = 64 + LR_K;       // step lag between consecutive wavefronts
constexpr int LR_RING = 64;             // ring slots (> LR_K + 1)
constexpr int LR_D = 4;                 // steps of operand prefetch (divides LR_K)
constexpr int LR_MAXW = 8;
constexpr int LR_MAXROWS = 64 * LR_MAXW;

template <bool COEF>
__global__ __launch_bounds__(64 * LR_MAXW) void k_sor_lex_rows(int nx, int ny, int ld, const double *__restrict__ rau,
                                                              const double *__restrict__ rgv, PpeCoef cf,
                                                              const double *__restrict__ rhs,
                                                              const double *__restrict__ rbu,
                                                              const double *__restrict__ rbv, double *beff, int cart,
                                                              double sorrel, double sortol, int msorit, double *p,
                                                              Scalars *sc) {
    __shared__ double ring[LR_MAXW][LR_RING];
    __shared__ double red[LR_MAXW];
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    const int nw = blockDim.x >> 6;
    const int j = 2 + t;
    const bool rowok = j <= ny;
    const int nc = nx - 1;                       // columns i = 2 .. nx
    // steps of a sweep, rounded up to whole blocks (the extra steps find no point)
    const int nsteps = (nc + LR_LAG * (nw - 1) + 63 + LR_K - 1) / LR_K * LR_K;
    const double *bb = cart ? rhs : beff;
    for (int m = 1;; m++) {
        if (!cart) {   // pressure.f:RhsPpe from the field at the start of the sweep
#define P(a, b) p[WD2_IX(a, b)]
            for (int q = t; q < (nx - 1) * (ny - 1); q += blockDim.x) {
                const int i = 2 + q % (nx - 1), jj = 2 + q / (nx - 1);
                beff[WD2_IX(i, jj)] =
                    rhs[WD2_IX(i, jj)] -
                    (rbu[WD2_IX(i, jj)] * (P(i + 1, jj + 1) + P(i, jj + 1) - P(i + 1, jj - 1) - P(i, jj - 1)) -
                     rbu[WD2_IX(i - 1, jj)] * (P(i, jj + 1) + P(i - 1, jj + 1) - P(i, jj - 1) - P(i - 1, jj - 1)) +
                     rbv[WD2_IX(i, jj)] * (P(i + 1, jj + 1) + P(i + 1, jj) - P(i - 1, jj + 1) - P(i - 1, jj)) -
                     rbv[WD2_IX(i, jj - 1)] * (P(i + 1, jj) + P(i + 1, jj - 1) - P(i - 1, jj) - P(i - 1, jj - 1)));
            }
#undef P
            __syncthreads();
        }
        // operands of the point LR_D steps ahead are loaded while the current
        // step runs (slot d holds column c + d of this lane's row)
        // (the point's old value is the previous column's east value, and on
        // the unit-coefficient path its a2 the previous column's a4)
        double oE[LR_D], oN[LR_D], oB[LR_D], o1[LR_D], o4[LR_D], o5[LR_D];
        double o2[COEF ? LR_D : 1], o3[COEF ? LR_D : 1];
        auto fetch = [&](int cc, int d) {
            if (rowok && cc >= 0 && cc < nc) {
                const int i = 2 + cc;
                const size_t k = WD2_IX(i, j);
                oE[d] = p[WD2_IX(i + 1, j)];
                oN[d] = p[WD2_IX(i, j + 1)];
                oB[d] = bb[k];
                if (COEF) {
                    o1[d] = cf.a1[k]; o2[d] = cf.a2[k]; o3[d] = cf.a3[k]; o4[d] = cf.a4[k]; o5[d] = cf.a5[k];
                } else {
                    o1[d] = rgv[WD2_IX(i, j - 1)];
                    o4[d] = rau[k];
                    o5[d] = rgv[k];
                }
            }
        };
        const int off = w * LR_LAG + lane;   // the lane's point at step st is column st - off
#pragma unroll
        for (int d = 0; d < LR_D; d++) fetch(d - off, d);
        double mx = 0.0, res = 0.0, prevE = 0.0, prevA4 = 0.0;
        for (int s0 = 0; s0 < nsteps; s0 += LR_K) {
#pragma unroll
            for (int q = 0; q < LR_K; q++) {
                const int st = s0 + q;
                const int d = q % LR_D;                   // slot of this step (LR_K is a multiple of LR_D)
                const int c = st - off;
                const double up = __shfl_up(res, 1);      // lane-1's point of the previous step
                if (rowok && c >= 0 && c < nc) {
                    const int i = 2 + c;
                    double pS;
                    if (lane > 0) pS = up;
                    else if (w > 0) pS = ring[w - 1][c % LR_RING];
                    else pS = p[WD2_IX(i, j - 1)];            // ghost row j = 1
                    const double pW = c > 0 ? res : p[WD2_IX(i - 1, j)];   // ghost column i = 1
                    const double pij = c > 0 ? prevE : p[WD2_IX(i, j)];
                    const double a1 = o1[d], a4 = o4[d], a5 = o5[d];
                    const double a2 = COEF ? o2[COEF ? d : 0] : (c > 0 ? prevA4 : rau[WD2_IX(i - 1, j)]);
                    const double a3 = COEF ? o3[COEF ? d : 0] : -a4 - a2 - a5 - a1;
                    double sum = oB[d] - a1 * pS - a2 * pW - a4 * oE[d] - a5 * oN[d];
                    sum = sum / a3 - pij;
                    res = pij + sorrel * sum;
                    p[WD2_IX(i, j)] = res;
                    mx = dmaxf(mx, fabs(sum));
                    if (lane == 63) ring[w][c % LR_RING] = res;
                }
                prevE = oE[d];        // the next column's old value and a2
                prevA4 = o4[d];
                fetch(c + LR_D, d);   // the slot is free again: column c + LR_D
            }
            __syncthreads();
        }
        // dif of the sweep and the stopping test (pressure.f:434-449)
        for (int off = 32; off > 0; off >>= 1) mx = dmaxf(mx, __shfl_xor(mx, off));
        if (lane == 0) red[w] = mx;
        __syncthreads();
        double dif = 0.0;
        for (int q = 0; q < nw; q++) dif = dmaxf(dif, red[q]);
        __syncthreads();
        const bool conv = m > 1 && dif < sortol;
        if (conv || m >= msorit) {
            if (t == 0) {
                sc->sor_m = m;
                sc->sor_dif = dif;
                sc->sor_nconv = conv ? m : 0;
                sc->sor_done = 1;
            }
            return;
        }
    }
}

int sor_lex_rows_max() { return LR_MAXROWS; }

void launch_sor_lex_rows(int nx, int ny, int ld, const Metrics &m, const PpeCoef *coef, const double *rhs,
                         double *beff, int cart, double sorrel, double sortol, int msorit, double *p, Scalars *sc,
                         hipStream_t s) {
    const int nw = (ny - 1 + 63) / 64;
    const PpeCoef cf = coef ? *coef : PpeCoef{nullptr, nullptr, nullptr, nullptr, nullptr};
    if (coef)
        hipLaunchKernelGGL(k_sor_lex_rows<true>, dim3(1), dim3(64 * nw), 0, s, nx, ny, ld, m.rau, m.rgv, cf, rhs,
                           m.rbu, m.rbv, beff, cart, sorrel, sortol, msorit, p, sc);
    else
        hipLaunchKernelGGL(k_sor_lex_rows<false>, dim3(1), dim3(64 * nw), 0, s, nx, ny, ld, m.rau, m.rgv, cf, rhs,
                           m.rbu, m.rbv, beff, cart, sorrel, sortol, msorit, p, sc);
}

void launch_sor_lex_sweep(int nx, int ny, int ld, const Metrics &m, const PpeCoef *coef, const double *b,
                          double sorrel, double sortol, int msorit, double *p, int *tile_flags, int sweep,
                          double *partials, Scalars *sc, hipStream_t s) {
    const int ntx = (nx - 1 + LX_TI - 1) / LX_TI, nty = (ny - 1 + LX_TJ - 1) / LX_TJ;
    PpeCoef cf = coef ? *coef : PpeCoef{nullptr, nullptr, nullptr, nullptr, nullptr};
    if (coef)
        hipLaunchKernelGGL(k_sor_lex<true>, dim3(ntx * nty), dim3(LX_T), 0, s, nx, ny, ld, m.rau, m.rgv, cf, b, sorrel,
                           sortol, msorit, p, tile_flags, sweep, partials, sc);
    else
        hipLaunchKernelGGL(k_sor_lex<false>, dim3(ntx * nty), dim3(LX_T), 0, s, nx, ny, ld, m.rau, m.rgv, cf, b,
                           sorrel, sortol, msorit, p, tile_flags, sweep, partials, sc);
}

// ------------------------------------------------------------- line SOR
// Chains of the lines j = first_line + line_step*q (q < nlines): row r of line q
// is i = 2 + r (r < nx-1), with (a, d, c) = (a2, a3, a4) and
// b = rhs - (a1*p(i,j-1) + a5*p(i,j+1))   (pressure.f:746-771)
template <bool COEF>
__global__ __launch_bounds__(256) void k_slor_assemble(int nx, int ny, int ld, const double *__restrict__ rau,
                                                       const double *__restrict__ rgv, PpeCoef cf,
                                                       const double *__restrict__ b, const double *__restrict__ p,
                                                       int first_line, int line_step, int nlines,
                                                       double *__restrict__ ca, double *__restrict__ cd,
                                                       double *__restrict__ cc, double *__restrict__ cb,
                                                       const Scalars *sc) {
    if (sc->sor_done) return;
    const int L = nx - 1;
    const long r = (long)blockIdx.x * 256 + threadIdx.x;
    if (r >= (long)L * nlines) return;
    const int q = (int)(r / L), i = 2 + (int)(r % L);
    const int j = first_line + line_step * q;
    const size_t k = WD2_IX(i, j);
    double a1, a2, a3, a4, a5;
    if (COEF) {
        a1 = cf.a1[k]; a2 = cf.a2[k]; a3 = cf.a3[k]; a4 = cf.a4[k]; a5 = cf.a5[k];
    } else {
        a1 = rgv[WD2_IX(i, j - 1)]; a2 = rau[WD2_IX(i - 1, j)]; a4 = rau[k]; a5 = rgv[k];
        a3 = -a4 - a2 - a5 - a1;
    }
    ca[r] = a2;
    cd[r] = a3;
    cc[r] = a4;
    cb[r] = b[k] - (a1 * p[WD2_IX(i, j - 1)] + a5 * p[WD2_IX(i, j + 1)]);
}

void launch_slor_assemble(int nx, int ny, int ld, const Metrics &m, const PpeCoef *coef, const double *b,
                          const double *p, int first_line, int line_step, int nlines, double *ca, double *cd,
                          double *cc, double *cb, const Scalars *sc, hipStream_t s) {
    const long n = (long)(nx - 1) * nlines;
    PpeCoef cf = coef ? *coef : PpeCoef{nullptr, nullptr, nullptr, nullptr, nullptr};
    if (coef)
        hipLaunchKernelGGL(k_slor_assemble<true>, dim3((n + 255) / 256), dim3(256), 0, s, nx, ny, ld, m.rau, m.rgv, cf,
                           b, p, first_line, line_step, nlines, ca, cd, cc, cb, sc);
    else
        hipLaunchKernelGGL(k_slor_assemble<false>, dim3((n + 255) / 256), dim3(256), 0, s, nx, ny, ld, m.rau, m.rgv,
                           cf, b, p, first_line, line_step, nlines, ca, cd, cc, cb, sc);
}

// Relaxation of the solved lines: p = plold + sorrel*(x - plold).  dif_mode 0:
// max |x - plold| (Slor, SlorRB); 1: max |plold - pnew| (SlorRBP, pressure.f:1122).
__global__ __launch_bounds__(256) void k_slor_relax(int nx, int ny, int ld, int first_line, int line_step,
                                                    int nlines, const double *__restrict__ x, double sorrel,
                                                    int dif_mode, double *__restrict__ p, Scalars *sc, int slot) {
    if (sc->sor_done) return;
    __shared__ double sh[4];
    const int L = nx - 1;
    const long r = (long)blockIdx.x * 256 + threadIdx.x;
    double mx = 0.0;
    if (r < (long)L * nlines) {
        const int q = (int)(r / L), i = 2 + (int)(r % L);
        const int j = first_line + line_step * q;
        const size_t k = WD2_IX(i, j);
        const double plold = p[k];
        const double sum = x[r] - plold;
        const double pnew = plold + sorrel * sum;
        p[k] = pnew;
        mx = dif_mode == 0 ? fabs(sum) : fabs(plold - pnew);
    }
    mx = block_max<256>(mx, sh, threadIdx.x);
    if (threadIdx.x == 0) atomicMax((unsigned long long *)&sc->val[slot], dbits(mx));
}

void launch_slor_relax(int nx, int ny, int ld, int first_line, int line_step, int nlines, const double *x,
                       double sorrel, int dif_mode, double *p, const double *pn, double *partials, Scalars *sc,
                       int slot, hipStream_t s) {
    const long n = (long)(nx - 1) * nlines;
    (void)pn;
    (void)partials;
    hipLaunchKernelGGL(k_slor_relax, dim3((n + 255) / 256), dim3(256), 0, s, nx, ny, ld, first_line, line_step,
                       nlines, x, sorrel, dif_mode, p, sc, slot);
}

__global__ void k_slor_finish(double sortol, int msorit, Scalars *sc) {
    if (sc->sor_done) return;
    const double dif = sc->val[6];
    sc->val[6] = 0.0;
    sor_finish(sc, dif, sortol, msorit);
}

void launch_slor_finish(int nparts, double sortol, int msorit, double *partials, Scalars *sc, hipStream_t s) {
    (void)nparts;
    (void)partials;
    hipLaunchKernelGGL(k_slor_finish, dim3(1), dim3(1), 0, s, sortol, msorit, sc);
}

void launch_slor_rbp_relax(int, int, int, int, double, const double *, double *, hipStream_t) {}

}  // namespace wd2
