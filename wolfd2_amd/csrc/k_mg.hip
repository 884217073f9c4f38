// k_mg.hip -- multigrid Poisson solver for the pressure equation, refined in
// FP64 (the tightly converged "tier B" solve; no counterpart in the reference,
// whose solvers are the six SOR / line-SOR variants of pressure.f).
//
// System: the 5-point operator of pressure.f:97-106 on the interior cells
// i = 2..nx, j = 2..ny, with the ghost pressures frozen at the values
// PresBoundCond set before the solve (main.f:797-803):
//     a1 p(i,j-1) + a2 p(i-1,j) + a3 p(i,j) + a4 p(i+1,j) + a5 p(i,j+1) = b(i,j)
//     a1 = rgv(i,j-1), a2 = rau(i-1,j), a4 = rau(i,j), a5 = rgv(i,j),
//     a3 = -a4 - a2 - a5 - a1.
// After Project, the divergence of an interior cell is dk (b - A p): the
// solve stops when max |dk (b - A p)| < sortol over the interior, the
// divergence the projection leaves (ghost-adjacent cells add the frozen-ghost
// lag of the reference's own algorithm).
//
// Defect correction: each cycle forms r = b - A p in FP64 on the fine grid,
// runs one V-cycle for A e = r in the arithmetic type T (float: the mixed
// path; double: the FP64 path), and adds e to p in FP64.
//
// V-cycle (cell-centred):
// * level 0 is the pressure grid, NX = nx-1 by NY = ny-1 cells; level l+1
//   has ceil(NX/2) x ceil(NY/2) cells, a coarse cell holding fine cells 2I,
//   2I+1 (and 2J, 2J+1) where they exist;
// * face coefficients: level 0 copies rau and rgv; a coarse face takes the
//   mean of the fine faces it covers; a boundary face (to the frozen ghost)
//   is scaled by s_l / s_(l-1) with s_l = 2^(l+1) / (2^l + 1), which keeps
//   the correction's zero at the fine ghost's centre on every level;
// * smoother: red-black Gauss-Seidel, NU sweeps before and after (colours
//   0, 1 down; 1, 0 up); restriction: the sum of a coarse cell's children;
//   prolongation: bilinear (9, 3, 3, 1) / 16 from the coarse cell and its
//   neighbours, zero outside the grid;
// * the wider levels run as 64 x 64 tiles, one launch per level down (smooth,
//   residual, restrict) and one up (prolong, smooth); the levels of at most
//   64 cells a side run in one workgroup (the bottom kernel), and
//   from the first level of at most 64 cells in all the rest of the V-cycle
//   is one product with its matrix, built with the coefficients.
//
// A level or tile is held in registers (SPt below): a lane keeps a strip of
// four rows of one column, so a colour's update reads three of its four
// neighbours by lane shifts and from its own registers, and only the two rows
// at a strip's ends cross through LDS.  The smoothing phases are latency (a
// barrier and a few dependent operations each): with the points in LDS and a
// point update of four loads and a division, a phase took 0.35 (a 44 x 44
// tile) to 0.9 us (a 64 x 64 bottom level); here about 0.15.  Launches on the
// 1024^2 cavity, points in LDS -> strips (FP32 | FP64): level 0 down 15.1 ->
// 12.0 | 17.1 -> 15.0 us, up 10.4 -> 9.1 | 11.6 -> 13.1 us, bottom 31.6 ->
// 17.1 | 31.0 -> 11.9 us, a whole V-cycle 101 -> 70 | 111 -> 93 us; on the
// 128^2 cavity (FP32) a V-cycle 54 -> 31 us.
//
// The down kernel of level 0 also reduces max |r| per tile; every workgroup
// of the next kernel evaluates the stopping test from those maxima (every
// later kernel returns at entry once it has stopped the solve).
#include <cmath>

#include "wd2_dev.hpp"
#include "wd2_launch.hpp"

namespace wd2 {

constexpr int MG_NU = 2;                       // smoothing sweeps before and after
constexpr int MG_TW = 64;                      // tile side, one column per lane
constexpr int MG_SR = 4;                       // rows per strip
constexpr int MG_NS = MG_TW / MG_SR;           // strips of a tile
constexpr int MG_NT = 64 * MG_NS;              // threads of a tile workgroup
constexpr int MG_HD = 2 * MG_NU + 2;           // down halo (2 NU + 1, even)
constexpr int MG_HU = 2 * MG_NU;               // up halo
constexpr int MG_OD = MG_TW - 2 * MG_HD;       // owned cells per tile side, down (52)
constexpr int MG_OU = MG_TW - 2 * MG_HU;       // up (56)
constexpr int MG_TAIL = 64;                    // cells of the widest level the tail matrix covers
constexpr int MG_NCOARSE = 6;                  // sweeps on the coarsest grid (at most 2 x 2 cells)
constexpr int MG_NREG = 3;                     // bottom levels wider than the tail, at most
static_assert(MG_HD % 2 == 0 && MG_HU % 4 == 0 && MG_OD % 2 == 0 && MG_OU % 4 == 0,
              "even tile origins keep the colours global; the up strips start on coarse row pairs");

// Level arrays (elements of T): cell (I, J), 0-based, at (I+1) + ld (J+1),
// with a zero ring (e, r, c); x-face west of cell I (I = 0..nx) at
// I + ld (J+1); y-face south of cell J (J = 0..ny) at (I+1) + ld J.
__device__ inline size_t mc(int ld, int I, int J) { return (size_t)(I + 1) + (size_t)ld * (J + 1); }
__device__ inline size_t mfx(int ld, int I, int J) { return (size_t)I + (size_t)ld * (J + 1); }
__device__ inline size_t mfy(int ld, int I, int J) { return (size_t)(I + 1) + (size_t)ld * J; }

// ------------------------------------------------------------ coefficients
// Level 0 faces from rau and rgv (field layout; uniform values when uni).
template <typename T>
__global__ void k_mg_coef0(int nx, int ny, int ld, const double *__restrict__ rau, const double *__restrict__ rgv,
                           int uni, double rau_c, double rgv_c, MgLevel L) {
    const int NX = nx - 1, NY = ny - 1;
    const int I = blockIdx.x * blockDim.x + threadIdx.x, J = blockIdx.y;
    T *ax = (T *)L.ax, *ay = (T *)L.ay;
    if (I <= NX && J < NY) ax[mfx(L.ld, I, J)] = (T)(uni ? rau_c : rau[WD2_IX(I + 1, J + 2)]);
    if (I < NX && J <= NY) ay[mfy(L.ld, I, J)] = (T)(uni ? rgv_c : rgv[WD2_IX(I + 2, J + 1)]);
}

// Coarse faces of level c from level f: the mean of the fine faces a coarse
// face covers, boundary faces scaled by sb.
template <typename T>
__global__ void k_mg_coarsen(MgLevel F, MgLevel C, T sb) {
    const int I = blockIdx.x * blockDim.x + threadIdx.x, J = blockIdx.y;
    const T *fx = (const T *)F.ax, *fy = (const T *)F.ay;
    T *cx = (T *)C.ax, *cy = (T *)C.ay;
    if (I <= C.nx && J < C.ny) {
        const int f = min(2 * I, F.nx);
        T v = fx[mfx(F.ld, f, 2 * J)];
        int n = 1;
        if (2 * J + 1 < F.ny) { v += fx[mfx(F.ld, f, 2 * J + 1)]; n = 2; }
        v = v / (T)n;
        if (I == 0 || I == C.nx) v *= sb;
        cx[mfx(C.ld, I, J)] = v;
    }
    if (I < C.nx && J <= C.ny) {
        const int f = min(2 * J, F.ny);
        T v = fy[mfy(F.ld, 2 * I, f)];
        int n = 1;
        if (2 * I + 1 < F.nx) { v += fy[mfy(F.ld, 2 * I + 1, f)]; n = 2; }
        v = v / (T)n;
        if (J == 0 || J == C.ny) v *= sb;
        cy[mfy(C.ld, I, J)] = v;
    }
}

// The stopping test before V-cycle `cycle` (1-based), evaluated by every
// workgroup of the first kernel after the level-0 down kernel from that
// kernel's per-tile maxima of |r|: stop when max |dk r| < tol and at least
// minc cycles are applied (mg_nconv = cycles applied), or when `maxcyc`
// cycles are applied (mg_nconv = -1, not converged; a NaN never passes).
// All workgroups reach the same answer; workgroup 0 records it (val[7] =
// max |dk r|).  sh: NT / 64 doubles of LDS.
template <int NT>
__device__ inline bool mg_decide(const double *__restrict__ part, int nt, double dk, double tol, int cycle,
                                 int maxcyc, int minc, Scalars *sc, double *sh) {
    double m = 0.0;
    for (int k = threadIdx.x; k < nt; k += NT)
        if (!(part[k] <= m)) m = part[k];
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(m, off);
        if (!(o <= m)) m = o;
    }
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
    __syncthreads();
    m = sh[0];
    for (int w = 1; w < NT / 64; w++)
        if (!(sh[w] <= m)) m = sh[w];
    __syncthreads();
    const double div = m * dk;
    const bool conv = div < tol && cycle - 1 >= minc, cap = !conv && cycle - 1 >= maxcyc;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc->val[7] = div;
        sc->mg_cycles = cycle - 1;
        if (conv || cap) {
            sc->mg_done = 1;
            sc->mg_nconv = conv ? cycle - 1 : -1;
        }
    }
    return conv || cap;
}

// Arguments of the stopping test for the kernel that evaluates it.
struct MgDecide {
    const double *part;
    int nt, cycle, maxcyc;   // nt = 0: this kernel does not decide
    double dk, tol;
    int minc;                // cycles to apply before the tolerance may stop the solve
};

// XCD-aware tile order: consecutive workgroups go to different XCDs; each XCD
// gets a contiguous band of tiles.
__device__ inline int mg_tile(int ntiles) {
    const int per = (ntiles + 7) / 8;
    return (blockIdx.x % 8) * per + blockIdx.x / 8;
}

// ------------------------------------------------------------ strips
// Lane shifts within a wavefront: the value of lane - 1 (sh_w) or lane + 1
// (sh_e), 0 past the ends, and of the lane whose number differs in the last
// bit (sh_x).
template <int CTRL>
__device__ inline float dpp_move(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ inline double dpp_move(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
template <typename T>
__device__ inline T sh_w(T v) { return dpp_move<0x138>(v); }   // wave_shr:1
template <typename T>
__device__ inline T sh_e(T v) { return dpp_move<0x130>(v); }   // wave_shl:1
template <typename T>
__device__ inline T sh_x(T v) { return dpp_move<0xB1>(v); }    // quad_perm [1,0,3,2]

// A lane's strip: four rows of column x, as two row pairs.  With q = x & 1
// (tile origins are even, so a point's colour is (x + row) & 1), pair k's
// point of colour 0 is row 2k + q (A[k]) and of colour 1 row 2k + 1 - q
// (B[k]).  The horizontal neighbours of A[k] are B[k] of lanes x - 1 and
// x + 1, its vertical ones are its mate B[k] and, on the other side, row
// 2k - 1 (q = 0) or 2k + 2 (q = 1): B[k - 1] or B[k + 1], past the strip's
// end a value of the next strip; and the same with the colours exchanged.
//
// A point's update is e = r' + w e_W + e e_E + m e_mate + o e_other with the
// face coefficients and the right-hand side divided by the diagonal once
// (and signs turned): the reference has no counterpart whose rounding it
// would have to keep.  Coefficients towards the ring, and all of a point
// outside the grid, are 0, so such a point stays 0.
template <typename T>
struct SPt {
    T w, e, m, o, r;
};
template <typename T>
struct Strip {
    T A[2], B[2];
    SPt<T> a[2], b[2];
    T d[2];   // diagonals of the A points (their residuals are restricted)
};

// The strip's coefficients from its rows' west and east faces, its five
// y-faces (fs[j] south of row j) and right-hand sides; in: the row's point
// is in the grid; I, NX: its column and the level's width.
template <typename T>
__device__ __forceinline__ void strip_build(Strip<T> &S, int q, const T (&fw)[4], const T (&fe)[4], const T (&fs)[5],
                                   const T (&r)[4], const bool (&in)[4], int I, int NX) {
    SPt<T> v[4];
    T d[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const T a3 = -(fw[j] + fe[j] + fs[j] + fs[j + 1]);
        const T i3 = in[j] ? T(1) / a3 : T(0);
        const T so = -fs[j] * i3, no = -fs[j + 1] * i3;
        // a row of even j has its mate north of it
        v[j] = SPt<T>{I > 0 ? -fw[j] * i3 : T(0), I < NX - 1 ? -fe[j] * i3 : T(0), (j & 1) ? so : no,
                      (j & 1) ? no : so, in[j] ? r[j] * i3 : T(0)};
        d[j] = in[j] ? a3 : T(0);
    }
#define SEL(c, x, y) SPt<T>{c ? x.w : y.w, c ? x.e : y.e, c ? x.m : y.m, c ? x.o : y.o, c ? x.r : y.r}
#pragma unroll
    for (int k = 0; k < 2; k++) {
        S.a[k] = SEL(q, v[2 * k + 1], v[2 * k]);
        S.b[k] = SEL(q, v[2 * k], v[2 * k + 1]);
        S.d[k] = q ? d[2 * k + 1] : d[2 * k];
    }
#undef SEL
}
// q ? x : y by value (a conditional of two members would keep the strip in
// memory).
template <typename T>
__device__ __forceinline__ T sel(bool q, T x, T y) {
    return q ? x : y;
}
template <typename T>
__device__ __forceinline__ T strip_eval(const SPt<T> &c, T row, T mate, T other) {
    // the value from the next strip, read from LDS, enters last
    return fma(c.o, other, fma(c.w, sh_w(row), fma(c.e, sh_e(row), fma(c.m, mate, c.r))));
}
// Row j's value.
template <typename T>
__device__ __forceinline__ T strip_row(const Strip<T> &S, int q, int j) {
    return sel((j & 1) == q, S.A[j >> 1], S.B[j >> 1]);
}

// The rows at the strips' ends in LDS: end (s, h) is strip s's row 0 (h = 0)
// or 3 (h = 1), for s = -1 .. NS (zero beyond the strips).  Of the two rows a
// colour's lanes need (below where q = 0, above where q = 1 for colour 0; the
// other way round for colour 1) all values are of the other colour, so no
// lane writes what another may still read in the same phase.
template <typename T>
struct Ends {
    T *p;   // this lane's column
    int lw; // column count
    __device__ T &at(int s, int h) const { return p[((s + 1) * 2 + h) * lw]; }
};

// Sweep phases; s: the lane's strip.
template <typename T>
__device__ __forceinline__ void phase_a(Strip<T> &S, int q, int s, const Ends<T> &E) {
    const T x = q ? E.at(s + 1, 0) : E.at(s - 1, 1);
    const T a0 = strip_eval(S.a[0], S.B[0], S.B[0], sel(q, S.B[1], x));
    const T a1 = strip_eval(S.a[1], S.B[1], S.B[1], sel(q, x, S.B[0]));
    S.A[0] = a0;
    S.A[1] = a1;
    E.at(s, q) = q ? a1 : a0;
}
template <typename T>
__device__ __forceinline__ void phase_b(Strip<T> &S, int q, int s, const Ends<T> &E) {
    const T x = q ? E.at(s - 1, 1) : E.at(s + 1, 0);
    const T b0 = strip_eval(S.b[0], S.A[0], S.A[0], sel(q, x, S.A[1]));
    const T b1 = strip_eval(S.b[1], S.A[1], S.A[1], sel(q, S.A[0], x));
    S.B[0] = b0;
    S.B[1] = b1;
    E.at(s, q ^ 1) = q ? b0 : b1;
}
// Both end rows (after a prolongation).
template <typename T>
__device__ __forceinline__ void ends_put(const Strip<T> &S, int q, int s, const Ends<T> &E) {
    E.at(s, 0) = sel(q, S.B[0], S.A[0]);
    E.at(s, 1) = sel(q, S.A[1], S.B[1]);
}
// NU sweeps from e = 0, colours 0 then 1 (the first phase's neighbours are 0).
// act: the lane holds a strip (others only take part in the syncs).
template <typename T, typename Sync>
__device__ __forceinline__ void sweep_down(Strip<T> &S, int q, int s, const Ends<T> &E, bool act, Sync sync) {
    S.A[0] = S.a[0].r;
    S.A[1] = S.a[1].r;
    if (act) E.at(s, q) = sel(q, S.A[1], S.A[0]);
    sync();
#pragma unroll
    for (int k = 0; k < MG_NU; k++) {
        if (k && act) phase_a(S, q, s, E);
        if (k) sync();
        if (act) phase_b(S, q, s, E);
        sync();
    }
}
template <typename T, typename Sync>
__device__ __forceinline__ void sweep_up(Strip<T> &S, int q, int s, const Ends<T> &E, bool act, Sync sync) {
    if (act) ends_put(S, q, s, E);
    sync();
#pragma unroll
    for (int k = 0; k < MG_NU; k++) {
        if (act) phase_b(S, q, s, E);
        sync();
        if (act) phase_a(S, q, s, E);
        if (k + 1 < MG_NU) sync();
    }
}
// Residuals of the strip's two row pairs summed over a coarse cell's
// children, for the lanes of even x.  Colour 1 was relaxed last, so its
// residuals are zero; colour 0's are the diagonal times what one more
// relaxation would add.
template <typename T>
__device__ __forceinline__ void strip_restrict(const Strip<T> &S, int q, int s, const Ends<T> &E, T (&rc)[2]) {
    const T x = q ? E.at(s + 1, 0) : E.at(s - 1, 1);
    const T g0 = strip_eval(S.a[0], S.B[0], S.B[0], sel(q, S.B[1], x));
    const T g1 = strip_eval(S.a[1], S.B[1], S.B[1], sel(q, x, S.B[0]));
    const T r0 = S.d[0] * (g0 - S.A[0]), r1 = S.d[1] * (g1 - S.A[1]);
    rc[0] = r0 + sh_x(r0);
    rc[1] = r1 + sh_x(r1);
}
// e += prolongation: h[k] = 3 c + c' of the coarse rows jc0 - 1 .. jc0 + 2 on
// the column's coarse cell (c) and its horizontal neighbour (c').
template <typename T>
__device__ __forceinline__ T prolong(const T (&h)[4], int j) {
    const int k = (j >> 1) + 1;
    return (T(3) * h[k] + h[(j & 1) ? k + 1 : k - 1]) * T(0.0625);
}

// ------------------------------------------------------------ down
// Level l: e = NU sweeps from 0 on A e = r, then r_(l+1) = restriction of
// r - A e.  L0: r = b - A p is formed here in FP64 from p and b (ghosts
// frozen), stored in T for the up pass, and max |r| of the owned points goes
// to part[tile].  D.nt > 0: this launch first evaluates the stopping test of
// the level-0 kernel before it.  A tile owns the MG_OD x MG_OD cells from
// (I0, J0); what its outermost lanes miss (the columns beyond the tile) moves
// inwards one column a phase and stays off the owned cells.  uni: rau and rgv
// are one value each (level 0 of a uniform Cartesian grid): no loads.
template <typename T, bool L0>
__global__ __launch_bounds__(MG_NT) void k_mg_down(MgLevel L, MgLevel C, int ntx, int ntiles, int nx, int ny, int ld,
                                                   const double *__restrict__ p, const double *__restrict__ b,
                                                   const double *__restrict__ rau, const double *__restrict__ rgv,
                                                   int uni, double rau_c, double rgv_c, double *__restrict__ part,
                                                   MgDecide D, Scalars *sc) {
    // below level 0 the tile's loads are in flight before the flag is looked
    // at (level 0's would cost a launch that returns here more than it saves
    // one that runs)
    const int stopped = sc->mg_done;
    if (L0 && stopped) return;
    __shared__ T ends[(MG_NS + 2) * 2 * MG_TW];
    __shared__ double red[MG_NT / 64];
    const int tile = mg_tile(ntiles);
    if (tile >= ntiles) return;
    const int I0 = (tile % ntx) * MG_OD, J0 = (tile / ntx) * MG_OD;
    const int NX = L.nx, NY = L.ny;
    const int x = threadIdx.x & 63, s = threadIdx.x >> 6, q = x & 1;
    const int I = I0 - MG_HD + x, Jb = J0 - MG_HD + MG_SR * s;
    const bool inx = I >= 0 && I < NX;
    const bool ownx = inx && x >= MG_HD && x < MG_HD + MG_OD;
    bool in[4];
    T fw[4], fe[4], fs[5], rv[4];
    double rmax = 0.0;
#pragma unroll
    for (int j = 0; j < 4; j++) in[j] = inx && Jb + j >= 0 && Jb + j < NY;
    if (L0) {
        // field (i, j) = (I + 2, J + 2); addresses are clamped to the field
        // (values outside serve only points outside the grid)
        const int i = min(max(I + 2, 0), nx + 1);
        auto row = [&](int J) { return min(max(J + 2, 0), ny + 1); };
        double pc[6], bb[4];
#pragma unroll
        for (int j = 0; j < 6; j++) pc[j] = p[WD2_IX(i, row(Jb + j - 1))];
#pragma unroll
        for (int j = 0; j < 4; j++) bb[j] = b[WD2_IX(i, row(Jb + j))];
        double a4[4], a5[5];
        if (uni) {
#pragma unroll
            for (int j = 0; j < 4; j++) a4[j] = rau_c;
#pragma unroll
            for (int j = 0; j < 5; j++) a5[j] = rgv_c;
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) a4[j] = rau[WD2_IX(i, row(Jb + j))];
#pragma unroll
            for (int j = 0; j < 5; j++) a5[j] = rgv[WD2_IX(i, row(Jb + j - 1))];
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const double a1 = a5[j], a2 = uni ? rau_c : sh_w(a4[j]);
            const double a3 = -a4[j] - a2 - a5[j + 1] - a1;
            const double res = bb[j] - (a1 * pc[j] + a2 * sh_w(pc[j + 1]) + a3 * pc[j + 1] + a4[j] * sh_e(pc[j + 1]) +
                                        a5[j + 1] * pc[j + 2]);
            rv[j] = in[j] ? (T)res : T(0);
            const int y = MG_SR * s + j;
            // a NaN residual wins the maximum (never converged)
            if (in[j] && ownx && y >= MG_HD && y < MG_HD + MG_OD && !(fabs(res) <= rmax)) rmax = fabs(res);
            fw[j] = (T)a2;
            fe[j] = (T)a4[j];
        }
#pragma unroll
        for (int j = 0; j < 5; j++) fs[j] = (T)a5[j];
    } else {
        const T *r = (const T *)L.r, *ax = (const T *)L.ax, *ay = (const T *)L.ay;
        // clamped addresses (values outside serve only points outside)
        const int Ic = min(max(I, 0), NX - 1), If = min(max(I, 0), NX);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int J = min(max(Jb + j, 0), NY - 1);
            rv[j] = r[mc(L.ld, Ic, J)];
            fw[j] = ax[mfx(L.ld, If, J)];
        }
#pragma unroll
        for (int j = 0; j < 5; j++) fs[j] = ay[mfy(L.ld, Ic, min(max(Jb + j, 0), NY))];
#pragma unroll
        for (int j = 0; j < 4; j++) fe[j] = sh_e(fw[j]);
    }
    if (stopped) return;
    if (D.nt > 0 && mg_decide<MG_NT>(D.part, D.nt, D.dk, D.tol, D.cycle, D.maxcyc, D.minc, sc, red)) return;
    if (s == 0 || s == MG_NS - 1) {   // the zero rows beyond the strips
        const int g = s == 0 ? -1 : MG_NS;
        ends[((g + 1) * 2) * MG_TW + x] = T(0);
        ends[((g + 1) * 2 + 1) * MG_TW + x] = T(0);
    }
    Strip<T> S;
    strip_build<T>(S, q, fw, fe, fs, rv, in, I, NX);
    const Ends<T> E{ends + x, MG_TW};
    if (L0) {
        for (int off = 32; off > 0; off >>= 1) {
            const double o = __shfl_xor(rmax, off);
            if (!(o <= rmax)) rmax = o;
        }
        if (x == 0) red[s] = rmax;
    }
    sweep_down<T>(S, q, s, E, true, [] { __syncthreads(); });
    if (L0 && threadIdx.x == 0) {
        double m = red[0];
        for (int w = 1; w < MG_NT / 64; w++)
            if (!(red[w] <= m)) m = red[w];
        part[tile] = m;
    }
    T rc[2];
    strip_restrict<T>(S, q, s, E, rc);
    T *e = (T *)L.e, *r = (T *)L.r, *cr = (T *)C.r;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int y = MG_SR * s + j;
        if (in[j] && ownx && y >= MG_HD && y < MG_HD + MG_OD) {
            e[mc(L.ld, I, Jb + j)] = strip_row(S, q, j);
            if (L0) r[mc(L.ld, I, Jb + j)] = rv[j];
        }
    }
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const int y = MG_SR * s + 2 * k, Ic = I >> 1, Jc = (Jb + 2 * k) >> 1;
        if (q == 0 && ownx && y >= MG_HD && y < MG_HD + MG_OD && Ic < C.nx && Jc < C.ny) cr[mc(C.ld, Ic, Jc)] = rc[k];
    }
}

// ------------------------------------------------------------ up
// Level l: c = e + prolongation of c_(l+1), then NU sweeps; c of the owned
// points is written (L0: p += c in FP64 instead).  The input e of the halos
// and the output c are separate arrays, so no tile reads what another writes.
template <typename T, bool L0>
__global__ __launch_bounds__(MG_NT) void k_mg_up(MgLevel L, MgLevel C, int ntx, int ntiles, int nx, int ny, int ld,
                                                 double *__restrict__ p, const double *__restrict__ rau,
                                                 const double *__restrict__ rgv, int uni, double rau_c, double rgv_c,
                                                 const Scalars *sc) {
    const int stopped = sc->mg_done;
    if (L0 && stopped) return;
    __shared__ T ends[(MG_NS + 2) * 2 * MG_TW];
    const int tile = mg_tile(ntiles);
    if (tile >= ntiles) return;
    const int I0 = (tile % ntx) * MG_OU, J0 = (tile / ntx) * MG_OU;
    const int NX = L.nx, NY = L.ny;
    const int x = threadIdx.x & 63, s = threadIdx.x >> 6, q = x & 1;
    const int I = I0 - MG_HU + x, Jb = J0 - MG_HU + MG_SR * s;
    const bool inx = I >= 0 && I < NX;
    const int Ic = min(max(I, 0), NX - 1);   // addresses are clamped to the grid
    const T *e = (const T *)L.e, *r = (const T *)L.r, *ec = (const T *)C.c;
    bool in[4];
    T fw[4], fe[4], fs[5], rv[4], ev[4], h[4];
#pragma unroll
    for (int j = 0; j < 4; j++) in[j] = inx && Jb + j >= 0 && Jb + j < NY;
    {
        const int ic = min(max(I >> 1, 0), C.nx - 1), in2 = ic + ((I & 1) ? 1 : -1), jc0 = Jb >> 1;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int jc = min(max(jc0 - 1 + k, -1), C.ny);
            h[k] = T(3) * ec[mc(C.ld, ic, jc)] + ec[mc(C.ld, in2, jc)];
        }
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int J = min(max(Jb + j, 0), NY - 1);
        ev[j] = e[mc(L.ld, Ic, J)];
        rv[j] = r[mc(L.ld, Ic, J)];
    }
    if (L0) {
        const int i = min(max(I + 2, 0), nx + 1);
        auto row = [&](int J) { return min(max(J + 2, 0), ny + 1); };
#pragma unroll
        for (int j = 0; j < 4; j++) fe[j] = (T)(uni ? rau_c : rau[WD2_IX(i, row(Jb + j))]);
#pragma unroll
        for (int j = 0; j < 5; j++) fs[j] = (T)(uni ? rgv_c : rgv[WD2_IX(i, row(Jb + j - 1))]);
#pragma unroll
        for (int j = 0; j < 4; j++) fw[j] = uni ? (T)rau_c : sh_w(fe[j]);
    } else {
        const T *ax = (const T *)L.ax, *ay = (const T *)L.ay;
        const int If = min(max(I, 0), NX);
#pragma unroll
        for (int j = 0; j < 4; j++) fw[j] = ax[mfx(L.ld, If, min(max(Jb + j, 0), NY - 1))];
#pragma unroll
        for (int j = 0; j < 5; j++) fs[j] = ay[mfy(L.ld, Ic, min(max(Jb + j, 0), NY))];
#pragma unroll
        for (int j = 0; j < 4; j++) fe[j] = sh_e(fw[j]);
    }
    if (stopped) return;
    if (s == 0 || s == MG_NS - 1) {
        const int g = s == 0 ? -1 : MG_NS;
        ends[((g + 1) * 2) * MG_TW + x] = T(0);
        ends[((g + 1) * 2 + 1) * MG_TW + x] = T(0);
    }
    Strip<T> S;
    strip_build<T>(S, q, fw, fe, fs, rv, in, I, NX);
    T v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = in[j] ? ev[j] + prolong<T>(h, j) : T(0);
#pragma unroll
    for (int k = 0; k < 2; k++) {
        S.A[k] = q ? v[2 * k + 1] : v[2 * k];
        S.B[k] = q ? v[2 * k] : v[2 * k + 1];
    }
    const Ends<T> E{ends + x, MG_TW};
    sweep_up<T>(S, q, s, E, true, [] { __syncthreads(); });
    if (!inx || x < MG_HU || x >= MG_HU + MG_OU) return;
    T *eo = (T *)L.c;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int y = MG_SR * s + j;
        if (!in[j] || y < MG_HU || y >= MG_HU + MG_OU) continue;
        if (L0)
            p[WD2_IX(I + 2, Jb + j + 2)] += (double)strip_row(S, q, j);
        else
            eo[mc(L.ld, I, Jb + j)] = strip_row(S, q, j);
    }
}

// ------------------------------------------------------------ bottom
// The bottom levels in one workgroup.  Levels of more than MG_TAIL cells are
// strips in registers (a level of NX cells a row takes lw = 2^k >= NX lanes a
// strip, so a narrow level packs several strips into a wavefront; a level
// that fits one wavefront is run by wavefront 0 alone, between wavefront
// syncs).  From the first level of at most MG_TAIL cells on, the rest of the
// V-cycle is linear in that level's right-hand side: c = M r, with M built by
// k_mg_tail when the coefficients are (about thirty dependent phases on a
// handful of points otherwise).  Level 0's r comes from the down kernel
// above; its correction goes to c for the up kernel above.  D.nt > 0: the
// stopping test is evaluated first.
//
// The kernel runs once through its code on one CU, whose instruction cache
// holds none of it at launch: unrolled over the levels it was 37 KB and took
// 20 us, most of it instruction fetches.  So the levels are a loop over one
// copy of each half, their strip coefficients come ready-made from memory
// (k_mg_pack), loaded one level ahead, and the strips wait in LDS while the
// coarser levels run.
struct MgBottom {
    MgLevel lev[MG_NREG + 1];
    const void *pack[MG_NREG];   // the register levels' strip coefficients
    int nreg;                    // register levels; lev[nreg] is the tail's level
    const void *tail;            // M, column j at [MG_TAIL j]
};
// (FP64 strips of a 64-wide level, with the next level's coefficients in
// flight, exceed the 128 registers 1024 lanes can have: 26 us a launch
// against 9 with the 64-wide level as a tile launch down and up of 5 us each)
template <typename T>
constexpr int mg_bottom_width() { return sizeof(T) == 4 ? 64 : 32; }

// Lanes of a level's strips.
struct BtGeo {
    int k, ns;   // 2^k lanes a strip, ns strips
    __device__ BtGeo(const MgLevel &L)
        : k(L.nx > 32 ? 6 : (L.nx > 16 ? 5 : (L.nx > 8 ? 4 : 3))), ns((L.ny + MG_SR - 1) / MG_SR) {}
    __device__ int lanes() const { return ns << k; }
    __device__ bool wave() const { return lanes() <= 64; }
};
// A lane's coefficients in a pack: value v of lane t at [v lanes + t], the
// points a[0], a[1], b[0], b[1] with r = 1, then the diagonals d.
constexpr int BT_PACK = 22;
template <typename T>
struct BtCoef {
    T v[BT_PACK];
    __device__ SPt<T> pt(int p, T r) const {
        return SPt<T>{v[5 * p], v[5 * p + 1], v[5 * p + 2], v[5 * p + 3], v[5 * p + 4] * r};
    }
};

template <typename T>
__global__ __launch_bounds__(1024) void k_mg_pack(MgLevel L, T *__restrict__ P) {
    const BtGeo g(L);
    const int t = threadIdx.x, x = t & ((1 << g.k) - 1), s = t >> g.k;
    if (s >= g.ns) return;
    const T *ax = (const T *)L.ax, *ay = (const T *)L.ay;
    T fw[4], fe[4], fs[5], one[4];
    bool in[4];
    for (int j = 0; j < 5; j++) {
        const int J = MG_SR * s + j;
        const bool c = x < L.nx && J < L.ny;
        fs[j] = (x < L.nx && J <= L.ny) ? ay[mfy(L.ld, x, J)] : T(0);
        if (j == 4) break;
        in[j] = c;
        one[j] = T(1);
        fw[j] = c ? ax[mfx(L.ld, x, J)] : T(0);
        fe[j] = c ? ax[mfx(L.ld, x + 1, J)] : T(0);
    }
    Strip<T> S;
    strip_build<T>(S, x & 1, fw, fe, fs, one, in, x, L.nx);
    for (int p = 0; p < 4; p++) {
        const SPt<T> &c = p < 2 ? S.a[p & 1] : S.b[p & 1];
        T *o = P + (size_t)5 * p * g.lanes() + t;
        o[0] = c.w;
        o[g.lanes()] = c.e;
        o[2 * g.lanes()] = c.m;
        o[3 * g.lanes()] = c.o;
        o[4 * g.lanes()] = c.r;
    }
    P[(size_t)20 * g.lanes() + t] = S.d[0];
    P[(size_t)21 * g.lanes() + t] = S.d[1];
}

// LDS of the bottom kernel.  Level l >= 1 has at most 32 x 32 (l = 1), 16 x 16
// (l = 2) cells and lanes 256, 64; the tail's level at most MG_TAIL cells, in
// at most (MG_TAIL + 2) x 3 places with its ring.
template <typename T, int NT>
struct BtShared {
    T ends[(MG_NS + 2) * 2 * 64];
    T r[32 * 32 + 16 * 16 + MG_TAIL];            // right-hand sides of the levels below the first
    T c[34 * 34 + 18 * 18 + (MG_TAIL + 2) * 3];  // their corrections, with a zero ring
    T sv[4 * (NT + 256 + 64)];                   // strips of the levels above the running one
    T m[MG_TAIL * MG_TAIL];
    double red[1024 / 64];
};
__device__ inline int bt_roff(int l) { return l == 1 ? 0 : (l == 2 ? 1024 : 1280); }
__device__ inline int bt_coff(int l) { return l == 1 ? 0 : (l == 2 ? 1156 : 1480); }
template <int NT>
__device__ inline int bt_soff(int l) { return l == 0 ? 0 : (l == 1 ? 4 * NT : 4 * (NT + 256)); }

__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename T, int NT>
__global__ __launch_bounds__(NT) void k_mg_bottom(MgBottom B, MgDecide D, Scalars *sc) {
    const int stopped = sc->mg_done;
    __shared__ BtShared<T, NT> H;
    const int t = threadIdx.x;
    auto load = [&](int l) {
        const int n = BtGeo(B.lev[l]).lanes();
        const T *P = (const T *)B.pack[l] + min(t, n - 1);
        BtCoef<T> K;
#pragma unroll
        for (int v = 0; v < BT_PACK; v++) K.v[v] = P[(size_t)v * n];
        return K;
    };
    // a lane's strip of level l from its coefficients and right-hand sides
    // (lanes past the level's points have clamped addresses)
    T r0[4] = {T(0), T(0), T(0), T(0)};   // the first level's right-hand sides
    auto strip = [&](int l, const MgLevel &L, int x, int s, int q, const BtCoef<T> &K, Strip<T> &S) {
        T rv[4];
#pragma unroll
        for (int j = 0; j < 4; j++)
            rv[j] = l == 0 ? r0[j] : H.r[bt_roff(l) + min(x, L.nx - 1) + L.nx * min(MG_SR * s + j, L.ny - 1)];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            S.a[k] = K.pt(k, sel(q, rv[2 * k + 1], rv[2 * k]));
            S.b[k] = K.pt(2 + k, sel(q, rv[2 * k], rv[2 * k + 1]));
            S.d[k] = K.v[20 + k];
        }
    };
    // the first level's right-hand side and coefficients, the tail matrix
    const MgLevel &L0 = B.lev[0];
    BtCoef<T> K{};
    if (B.nreg > 0) {
        const BtGeo g(L0);
        const int x = t & ((1 << g.k) - 1), s = t >> g.k;
#pragma unroll
        for (int j = 0; j < 4; j++)
            r0[j] = ((const T *)L0.r)[mc(L0.ld, min(x, L0.nx - 1), min(MG_SR * s + j, L0.ny - 1))];
        K = load(0);
    }
    constexpr int MV = MG_TAIL * MG_TAIL / NT;
    T mv[MV];
#pragma unroll
    for (int k = 0; k < MV; k++) mv[k] = ((const T *)B.tail)[t + NT * k];
    if (stopped) return;
    if (D.nt > 0 && mg_decide<NT>(D.part, D.nt, D.dk, D.tol, D.cycle, D.maxcyc, D.minc, sc, H.red)) return;
    if (B.nreg == 0 && t < L0.nx * L0.ny) H.r[bt_roff(0) + t] = ((const T *)L0.r)[mc(L0.ld, t % L0.nx, t / L0.nx)];
#pragma unroll
    for (int k = 0; k < MV; k++) H.m[t + NT * k] = mv[k];
    for (int k = t; k < (int)(sizeof(H.c) / sizeof(T)); k += NT) H.c[k] = T(0);
    __syncthreads();
#pragma unroll 1
    for (int l = 0; l < B.nreg; l++) {
        const MgLevel &L = B.lev[l], &C = B.lev[l + 1];
        const BtGeo g(L);
        const bool wave = g.wave();
        if (wave && t >= 64) break;
        const int x = t & ((1 << g.k) - 1), s = t >> g.k, q = x & 1, n = g.lanes();
        const bool act = s < g.ns;
        auto sync = [&] {
            if (wave)
                wave_sync();
            else
                __syncthreads();
        };
        BtCoef<T> N{};
        if (l + 1 < B.nreg) N = load(l + 1);
        Strip<T> S;
        strip(l, L, x, s, q, K, S);
        const Ends<T> E{H.ends + x, 1 << g.k};
        if (act && s == 0) E.at(-1, 0) = E.at(-1, 1) = T(0);
        if (act && s == g.ns - 1) E.at(g.ns, 0) = E.at(g.ns, 1) = T(0);
        sweep_down<T>(S, q, s, E, act, sync);
        if (act) {
            T rc[2];
            strip_restrict<T>(S, q, s, E, rc);
            T *sv = H.sv + bt_soff<NT>(l) + t;
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const int Ic = x >> 1, Jc = 2 * s + k;
                if (q == 0 && Ic < C.nx && Jc < C.ny) H.r[bt_roff(l + 1) + Ic + C.nx * Jc] = rc[k];
                sv[k * n] = S.A[k];
                sv[(2 + k) * n] = S.B[k];
            }
        }
        sync();
        if (l + 1 < B.nreg) K = N;
    }
    if (t < 64) {   // c = M r on the tail's level
        const MgLevel &L = B.lev[B.nreg];
        const int n = L.nx * L.ny;
        if (t < n) {
            const T *r = H.r + bt_roff(B.nreg);
            T acc[4] = {T(0), T(0), T(0), T(0)};
            constexpr int U = 16;   // LDS reads in flight
            for (int j = 0; j < n; j += U) {
                T mm[U], rr[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int c = min(j + u, n - 1);
                    mm[u] = H.m[MG_TAIL * c + t];
                    rr[u] = r[c];
                }
#pragma unroll
                for (int u = 0; u < U; u++) acc[u & 3] = fma(mm[u], j + u < n ? rr[u] : T(0), acc[u & 3]);
            }
            const T v = (acc[0] + acc[1]) + (acc[2] + acc[3]);
            const int I = t % L.nx, J = t / L.nx;
            if (B.nreg == 0)
                ((T *)L.c)[mc(L.ld, I, J)] = v;
            else
                H.c[bt_coff(B.nreg) + I + 1 + (L.nx + 2) * (J + 1)] = v;
        }
        wave_sync();
    }
#pragma unroll 1
    for (int l = B.nreg - 1; l >= 0; l--) {
        const MgLevel &L = B.lev[l], &C = B.lev[l + 1];
        const BtGeo g(L);
        const bool wave = g.wave();
        // the other wavefronts join where the levels outgrow one
        if (!wave && (l == B.nreg - 1 || BtGeo(C).wave())) __syncthreads();
        if (wave && t >= 64) {
            if (l > 0 && !BtGeo(B.lev[l - 1]).wave()) K = load(l - 1);
            continue;
        }
        const int x = t & ((1 << g.k) - 1), s = t >> g.k, q = x & 1, n = g.lanes();
        const bool act = s < g.ns;
        auto sync = [&] {
            if (wave)
                wave_sync();
            else
                __syncthreads();
        };
        BtCoef<T> N{};
        if (l > 0) N = load(l - 1);
        Strip<T> S;
        strip(l, L, x, s, q, K, S);
        const T *sv = H.sv + bt_soff<NT>(l) + min(t, n - 1);
        const int W = C.nx + 2;
        const T *c = H.c + bt_coff(l + 1);
        const int ic = min(x >> 1, C.nx - 1) + 1, i2 = ic + (q ? 1 : -1);
        T h[4], v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int jc = min(2 * s + k, C.ny + 1);   // padded row of 2 s - 1 + k
            h[k] = T(3) * c[ic + W * jc] + c[i2 + W * jc];
        }
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = (act && x < L.nx && MG_SR * s + j < L.ny) ? prolong<T>(h, j) : T(0);
#pragma unroll
        for (int k = 0; k < 2; k++) {
            S.A[k] = sv[k * n] + sel(q, v[2 * k + 1], v[2 * k]);
            S.B[k] = sv[(2 + k) * n] + sel(q, v[2 * k], v[2 * k + 1]);
        }
        const Ends<T> E{H.ends + x, 1 << g.k};
        if (act && s == 0) E.at(-1, 0) = E.at(-1, 1) = T(0);
        if (act && s == g.ns - 1) E.at(g.ns, 0) = E.at(g.ns, 1) = T(0);
        sweep_up<T>(S, q, s, E, act, sync);
        T e[4];
#pragma unroll
        for (int j = 0; j < 4; j++) e[j] = strip_row(S, q, j);
        if (l == 0) {
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (act && x < L.nx && MG_SR * s + j < L.ny) ((T *)L.c)[mc(L.ld, x, MG_SR * s + j)] = e[j];
        } else {
            T *o = H.c + bt_coff(l) + x + 1 + (L.nx + 2) * (MG_SR * s + 1);
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (act && x < L.nx && MG_SR * s + j < L.ny) o[j * (L.nx + 2)] = e[j];
        }
        sync();
        if (l > 0) K = N;
    }
}

// The tail matrix: workgroup j (one wavefront) runs the V-cycle of the levels
// t .. of the hierarchy on the j-th unit vector; its result is column j.
struct MgTailLevels {
    MgLevel lev[MG_MAXLEV];
    int nlev;
};
template <typename T>
__global__ __launch_bounds__(64) void k_mg_tail(MgTailLevels B, T *__restrict__ M) {
    constexpr int CAP = 512;   // all levels with their rings: 64 x 1 and its halvings take the most
    __shared__ T E[CAP], R[CAP];
    __shared__ int off[MG_MAXLEV + 1];
    const int t = threadIdx.x;
    if (t == 0) {
        off[0] = 0;
        for (int l = 0; l < B.nlev; l++) off[l + 1] = off[l] + (B.lev[l].nx + 2) * (B.lev[l].ny + 2);
    }
    for (int k = t; k < CAP; k += 64) E[k] = R[k] = T(0);
    __syncthreads();
    if (t == 0) {
        const int j = blockIdx.x, NX = B.lev[0].nx;
        R[(j % NX + 1) + (NX + 2) * (j / NX + 1)] = T(1);
    }
    __syncthreads();
    auto relax = [&](int l, int c, bool res) {   // a colour's relaxation, or (res) the point's residual into E's place
        const MgLevel &L = B.lev[l];
        const T *ax = (const T *)L.ax, *ay = (const T *)L.ay;
        T *El = E + off[l];
        const T *Rl = R + off[l];
        const int W = L.nx + 2, I = t % L.nx, J = t / L.nx, k = (I + 1) + W * (J + 1);
        T v = T(0);
        if (J < L.ny && (res || ((I + J) & 1) == c)) {
            const T aw = ax[mfx(L.ld, I, J)], ae = ax[mfx(L.ld, I + 1, J)];
            const T as = ay[mfy(L.ld, I, J)], an = ay[mfy(L.ld, I, J + 1)];
            const T a3 = -(aw + ae + as + an);
            const T sum = as * El[k - W] + aw * El[k - 1] + ae * El[k + 1] + an * El[k + W];
            if (res)
                v = Rl[k] - (sum + a3 * El[k]);
            else
                El[k] = (Rl[k] - sum) / a3;
        }
        __syncthreads();
        return v;
    };
    for (int l = 0; l + 1 < B.nlev; l++) {
        for (int k = 0; k < MG_NU; k++)
            for (int c = 0; c < 2; c++) relax(l, c, false);
        const T v = relax(l, 0, true);
        const MgLevel &L = B.lev[l], &C = B.lev[l + 1];
        T *Rc = R + off[l + 1];
        const int I = t % L.nx, J = t / L.nx;
        // children of a coarse cell added in turn
        for (int u = 0; u < 4; u++) {
            if (J < L.ny && (I & 1) == (u & 1) && (J & 1) == (u >> 1))
                Rc[(I / 2 + 1) + (C.nx + 2) * (J / 2 + 1)] += v;
            __syncthreads();
        }
    }
    for (int k = 0; k < MG_NCOARSE; k++)
        for (int c = 0; c < 2; c++) relax(B.nlev - 1, c, false);
    for (int l = B.nlev - 2; l >= 0; l--) {
        const MgLevel &L = B.lev[l], &C = B.lev[l + 1];
        const int I = t % L.nx, J = t / L.nx, Wc = C.nx + 2;
        if (J < L.ny) {
            const T *Ec = E + off[l + 1];
            const int ic = (I >> 1) + 1, jc = (J >> 1) + 1, dx = (I & 1) ? 1 : -1, dy = (J & 1) ? 1 : -1;
            E[off[l] + (I + 1) + (L.nx + 2) * (J + 1)] +=
                (T(9) * Ec[ic + Wc * jc] + T(3) * Ec[ic + dx + Wc * jc] + T(3) * Ec[ic + Wc * (jc + dy)] +
                 Ec[ic + dx + Wc * (jc + dy)]) * T(0.0625);
        }
        __syncthreads();
        for (int k = 0; k < MG_NU; k++)
            for (int c = 1; c >= 0; c--) relax(l, c, false);
    }
    const MgLevel &L = B.lev[0];
    T v = T(0);
    if (t < L.nx * L.ny) v = E[(t % L.nx + 1) + (L.nx + 2) * (t / L.nx + 1)];
    M[MG_TAIL * blockIdx.x + t] = v;
}

// ------------------------------------------------------------ control
__global__ void k_mg_reset(Scalars *sc) {
    sc->mg_done = 0;
    sc->mg_nconv = -1;
    sc->mg_cycles = 0;
    sc->val[7] = 0.0;
}

// ------------------------------------------------------------ host side
static int tiles_of(int NX, int NY, int own, int *ntx) {
    const int tx = (NX + own - 1) / own, ty = (NY + own - 1) / own;
    if (ntx) *ntx = tx;
    return tx * ty;
}
int mg_tiles(int NX, int NY, int *ntx) { return tiles_of(NX, NY, MG_OD, ntx); }
int mg_tail_cells() { return MG_TAIL; }
int mg_bottom_side(int fp32) { return fp32 ? mg_bottom_width<float>() : mg_bottom_width<double>(); }
size_t mg_tail_bytes() { return sizeof(double) * (MG_TAIL * MG_TAIL + MG_NREG * BT_PACK * 1024); }

// The tail's level, the first of at most MG_TAIL cells below level 0 (the
// tiled levels end there at the latest), and the first level the bottom
// kernel can take: the packs are those of the levels between.
static int tail_level(const MgHierarchy &H) {
    int l = 1;
    while (l + 1 < H.nlev && H.lev[l].nx * H.lev[l].ny > MG_TAIL) l++;
    return l;
}
static int pack_level(const MgHierarchy &H) {
    int l = 1;
    while (l < tail_level(H) && std::max(H.lev[l].nx, H.lev[l].ny) > mg_bottom_width<float>()) l++;
    return l;
}
template <typename T>
static T *pack_of(const MgHierarchy &H, int l) {
    return (T *)H.tail + MG_TAIL * MG_TAIL + (size_t)BT_PACK * 1024 * (l - pack_level(H));
}

template <typename T>
void launch_mg_coef(const MgHierarchy &H, int nx, int ny, int ld, const double *rau, const double *rgv,
                    const double *uni, hipStream_t s) {
    const MgLevel &L0 = H.lev[0];
    hipLaunchKernelGGL(k_mg_coef0<T>, dim3((L0.nx + 1 + 255) / 256, L0.ny + 1), dim3(256), 0, s, nx, ny, ld, rau,
                       rgv, uni ? 1 : 0, uni ? uni[0] : 0.0, uni ? uni[1] : 0.0, L0);
    for (int l = 1; l < H.nlev; l++) {
        const double sl = std::ldexp(1.0, l + 1) / (std::ldexp(1.0, l) + 1.0);
        const double sp = std::ldexp(1.0, l) / (std::ldexp(1.0, l - 1) + 1.0);
        const MgLevel &C = H.lev[l];
        hipLaunchKernelGGL(k_mg_coarsen<T>, dim3((C.nx + 1 + 255) / 256, C.ny + 1), dim3(256), 0, s, H.lev[l - 1], C,
                           (T)(sl / sp));
    }
    MgTailLevels B{};
    const int t = tail_level(H);
    B.nlev = H.nlev - t;
    for (int l = 0; l < B.nlev; l++) B.lev[l] = H.lev[t + l];
    for (int l = pack_level(H); l < t; l++)
        hipLaunchKernelGGL(k_mg_pack<T>, dim3(1), dim3(1024), 0, s, H.lev[l], pack_of<T>(H, l));
    hipLaunchKernelGGL(k_mg_tail<T>, dim3(B.lev[0].nx * B.lev[0].ny), dim3(64), 0, s, B, (T *)H.tail);
}

template <typename T>
static void down0(const MgHierarchy &H, int nx, int ny, int ld, const double *b, const double *p, const double *rau,
                  const double *rgv, const double *uni, double *part, Scalars *sc, hipStream_t s) {
    int ntx = 0;
    const int nt = mg_tiles(H.lev[0].nx, H.lev[0].ny, &ntx);
    const MgDecide none{nullptr, 0, 0, 0, 0.0, 0.0};
    hipLaunchKernelGGL((k_mg_down<T, true>), dim3(8 * ((nt + 7) / 8)), dim3(MG_NT), 0, s, H.lev[0], H.lev[1], ntx, nt,
                       nx, ny, ld, p, b, rau, rgv, uni ? 1 : 0, uni ? uni[0] : 0.0, uni ? uni[1] : 0.0, part, none, sc);
}

template <typename T>
static void up0(const MgHierarchy &H, int nx, int ny, int ld, double *p, const double *rau, const double *rgv,
                const double *uni, Scalars *sc, hipStream_t s) {
    int ntx = 0;
    const int nt = tiles_of(H.lev[0].nx, H.lev[0].ny, MG_OU, &ntx);
    hipLaunchKernelGGL((k_mg_up<T, true>), dim3(8 * ((nt + 7) / 8)), dim3(MG_NT), 0, s, H.lev[0], H.lev[1], ntx, nt, nx,
                       ny, ld, p, rau, rgv, uni ? 1 : 0, uni ? uni[0] : 0.0, uni ? uni[1] : 0.0, sc);
}

template <typename T>
static void launch_mg_bottom(const MgHierarchy &H, const MgDecide &D, Scalars *sc, hipStream_t s) {
    MgBottom B{};
    B.nreg = tail_level(H) - H.ntiled;
    for (int l = 0; l <= B.nreg; l++) B.lev[l] = H.lev[H.ntiled + l];
    for (int l = 0; l < B.nreg; l++) B.pack[l] = pack_of<T>(H, H.ntiled + l);
    B.tail = H.tail;
    // lanes of the first level: 256 serve up to 32 x 32 cells
    if constexpr (mg_bottom_width<T>() > 32)
        if (std::max(B.lev[0].nx, B.lev[0].ny) > 32) {
            hipLaunchKernelGGL((k_mg_bottom<T, 1024>), dim3(1), dim3(1024), 0, s, B, D, sc);
            return;
        }
    hipLaunchKernelGGL((k_mg_bottom<T, 256>), dim3(1), dim3(256), 0, s, B, D, sc);
}

// One V-cycle of defect correction (cycle is 1-based), every kernel
// returning at entry once the solve has stopped; the stopping test of the
// cycle's level-0 residual runs at the start of the next kernel.
template <typename T>
void launch_mg_cycle(const MgHierarchy &H, int nx, int ny, int ld, const double *b, double *p, const double *rau,
                     const double *rgv, const double *uni, double dk, double tol, int cycle, int maxcyc,
                     double *part, Scalars *sc, hipStream_t s, hipEvent_t *ev_down, hipEvent_t *ev_up, int minc) {
    int ntx = 0;
    const int nt0 = mg_tiles(H.lev[0].nx, H.lev[0].ny, &ntx);
    if (ev_down) (void)hipEventRecord(ev_down[0], s);
    down0<T>(H, nx, ny, ld, b, p, rau, rgv, uni, part, sc, s);
    if (ev_down) (void)hipEventRecord(ev_down[1], s);
    const MgDecide D{part, nt0, cycle, maxcyc, dk, tol, minc};
    const MgDecide none{nullptr, 0, 0, 0, 0.0, 0.0};
    for (int l = 1; l < H.ntiled; l++) {
        const int nt = mg_tiles(H.lev[l].nx, H.lev[l].ny, &ntx);
        hipLaunchKernelGGL((k_mg_down<T, false>), dim3(8 * ((nt + 7) / 8)), dim3(MG_NT), 0, s, H.lev[l], H.lev[l + 1],
                           ntx, nt, nx, ny, ld, p, b, rau, rgv, 0, 0.0, 0.0, part, l == 1 ? D : none, sc);
    }
    launch_mg_bottom<T>(H, H.ntiled == 1 ? D : none, sc, s);
    for (int l = H.ntiled - 1; l >= 1; l--) {
        const int nt = tiles_of(H.lev[l].nx, H.lev[l].ny, MG_OU, &ntx);
        hipLaunchKernelGGL((k_mg_up<T, false>), dim3(8 * ((nt + 7) / 8)), dim3(MG_NT), 0, s, H.lev[l], H.lev[l + 1],
                           ntx, nt, nx, ny, ld, p, rau, rgv, 0, 0.0, 0.0, sc);
    }
    if (ev_up) (void)hipEventRecord(ev_up[0], s);
    up0<T>(H, nx, ny, ld, p, rau, rgv, uni, sc, s);
    if (ev_up) (void)hipEventRecord(ev_up[1], s);
}

// `reps` back-to-back launches of the level-0 down (which = 2) or up
// (which = 3) kernel, or of the bottom kernel (4; it writes only the
// correction c of its first level), between one event pair, on the state of
// the last solve
// (the stop flag is cleared first and set again after; the up kernel adds
// the last correction to p each time, so the caller restores p).
template <typename T>
void launch_mg_kernel_bench(const MgHierarchy &H, int which, int reps, int nx, int ny, int ld, const double *b,
                            double *p, const double *rau, const double *rgv, const double *uni, double *part,
                            Scalars *sc, hipStream_t s, hipEvent_t e0, hipEvent_t e1) {
    launch_mg_reset(sc, s);
    const MgDecide none{nullptr, 0, 0, 0, 0.0, 0.0};
    (void)hipEventRecord(e0, s);
    for (int k = 0; k < reps; k++) {
        if (which == 2)
            down0<T>(H, nx, ny, ld, b, p, rau, rgv, uni, part, sc, s);
        else if (which == 3)
            up0<T>(H, nx, ny, ld, p, rau, rgv, uni, sc, s);
        else
            launch_mg_bottom<T>(H, none, sc, s);
    }
    (void)hipEventRecord(e1, s);
}

void launch_mg_reset(Scalars *sc, hipStream_t s) { hipLaunchKernelGGL(k_mg_reset, dim3(1), dim3(1), 0, s, sc); }

template void launch_mg_coef<float>(const MgHierarchy &, int, int, int, const double *, const double *,
                                    const double *, hipStream_t);
template void launch_mg_coef<double>(const MgHierarchy &, int, int, int, const double *, const double *,
                                     const double *, hipStream_t);
template void launch_mg_cycle<float>(const MgHierarchy &, int, int, int, const double *, double *, const double *,
                                     const double *, const double *, double, double, int, int, double *, Scalars *,
                                     hipStream_t, hipEvent_t *, hipEvent_t *, int);
template void launch_mg_cycle<double>(const MgHierarchy &, int, int, int, const double *, double *, const double *,
                                      const double *, const double *, double, double, int, int, double *, Scalars *,
                                      hipStream_t, hipEvent_t *, hipEvent_t *, int);
template void launch_mg_kernel_bench<float>(const MgHierarchy &, int, int, int, int, int, const double *, double *,
                                            const double *, const double *, const double *, double *, Scalars *,
                                            hipStream_t, hipEvent_t, hipEvent_t);
template void launch_mg_kernel_bench<double>(const MgHierarchy &, int, int, int, int, int, const double *, double *,
                                             const double *, const double *, const double *, double *, Scalars *,
                                             hipStream_t, hipEvent_t, hipEvent_t);

}  // namespace wd2
