// k_adjoint.hip -- adjoint (transposed) kernels of the time step, FP64.
//
// The forward map differentiated is the step of main.f:690-972 on the
// multigrid path with a fixed number of q-l iterations (no stopping test)
// and a converged Poisson solve, on a one-region domain with no-slip walls
// (boundary profiles allowed), Cartesian metrics.  Every map below is the
// transpose of one forward piece; products that are bilinear in the fields
// (the convective fluxes, the upwinded chain coefficients) are transposed at
// the forward state, which the caller recomputes from checkpoints.
//
// Scatter-form transposes accumulate with FP64 atomics, in LDS and between
// tiles (the adjoint of a gather is a scatter); the sums are therefore not
// bit-reproducible, which does not matter to a gradient.
//
// Pieces and the forward lines they transpose:
// * chain solves (AltTridLU, momentum.f:1307-1339, with the first-row pivot
//   quirk H1: row 1's super-diagonal is divided by row 2's diagonal, i.e. the
//   matrix solved has S(1,2) = c1 d1 / d2): the transposed system is built
//   here and solved by the same parallel solver, whose own first-row quirk is
//   compensated; the coefficient adjoints are -mu_k x_{k-1}, -mu_k x_k,
//   -mu_k x_{k+1}, with the quirk's chain rule on rows 1 and 2;
// * the upwinded assembly of XMomentum (momentum.f:350-384, 396-428) and
//   YMomentum (675-754), the ConvCoef cases 1, 2, 4, 5 (864-981), DConvU/V
//   and DDiffU/V (987-1109);
// * VelBoundCond and PresBoundCond for no-slip walls (bound_cond.f:561-840,
//   853-1024), replayed in reverse order of assignment;
// * Project (utility.f:314-321, 384-391) and Divergence case 1
//   (pressure.f:287-299); the Poisson solve is self-adjoint on Cartesian grids
//   (a1 = rgv(i,j-1) is row (i,j-1)'s a5, a2 = rau(i-1,j) row (i-1,j)'s a4),
//   so its transpose is a solve with the same operator, and the frozen ghosts
//   receive minus their coupling coefficient times the solution.
#include <algorithm>

#include "wd2_dev.hpp"
#include "wd2_launch.hpp"

namespace wd2 {

constexpr int AT = 256;

__device__ inline void aadd(double *p, double v) {
    if (v != 0.0) atomicAdd(p, v);
}

// ------------------------------------------------------------ chains
__device__ inline long apos(const Chains &cs, long k, long &L) {
    if (k < cs.n1) {
        L = cs.L1;
        return k % cs.L1;
    }
    L = cs.L2;
    return (k - cs.n1) % cs.L2;
}

// The transposed system of the one the chain solver solved for (A, D, C),
// in a form the same solver solves exactly: row k of S^T has sub-diagonal
// S(k-1,k) = C[k-1] (c1 d1 / d2 on a chain's first row), diagonal D[k] and
// super-diagonal S(k+1,k) = A[k+1]; on a chain's first row the super-diagonal
// is given as A[k+1] D[k+1] / D[k], which the solver's own first-row quirk
// turns back into A[k+1].  *dom (from +0) receives the largest (|sub| +
// |super|) / |diagonal| of the rows (a NaN wins).
__global__ __launch_bounds__(AT) void k_adj_tchain(long n, Chains cs, const double *__restrict__ A,
                                                   const double *__restrict__ D, const double *__restrict__ C,
                                                   double *__restrict__ At, double *__restrict__ Dt,
                                                   double *__restrict__ Ct, unsigned long long *dom) {
    double m = 0.0;
    for (long k = (long)blockIdx.x * AT + threadIdx.x; k < n; k += (long)gridDim.x * AT) {
        long L;
        const long r = apos(cs, k, L);
        Dt[k] = D[k];
        double sub = 0.0, sup = 0.0;
        if (r > 0) sub = (r - 1 == 0) ? C[k - 1] * D[k - 1] / D[k] : C[k - 1];
        if (r < L - 1) sup = (r == 0) ? A[k + 1] * D[k + 1] / D[k] : A[k + 1];
        At[k] = sub;
        Ct[k] = sup;
        const double q = (fabs(sub) + fabs(sup)) / fabs(D[k]);
        if (!(q <= m)) m = q;
    }
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(m, off);
        if (!(o <= m)) m = o;
    }
    if ((threadIdx.x & 63) == 0) atomicMax(dom, dbits(m));
}

// Coefficient adjoints -mu_k x_{k-1}, -mu_k x_k, -mu_k x_{k+1} of row k of the
// matrix S of a solve S x = b (S with the chain solver's first-row quirk
// S(1,2) = c1 d1 / d2).  x is taken as +0 on the rows not flagged in XK -- at
// a converged q-l fixed point the first split's x vanishes on every row but
// the second split's identity rows, and only those rows' columns of S carry a
// derivative.
struct AdjChain {
    const double *A, *D, *C, *mu, *x;
    const unsigned char *XK;
};
__device__ inline void adj_coef(const AdjChain &q, const Chains &cs, long k, double m, double &ab, double &db,
                                double &cb) {
    long L;
    const long r = apos(cs, k, L);
    auto xv = [&](long o) { return q.XK[o] ? q.x[o] : 0.0; };
    ab = cb = 0.0;
    db = -m * xv(k);
    if (r > 0) ab = -m * xv(k - 1);
    if (r < L - 1) {
        const double sb = -m * xv(k + 1);   // adjoint of the entry S(k, k+1)
        if (r == 0) {   // S(1,2) = c1 d1 / d2
            cb = sb * q.D[k] / q.D[k + 1];
            db += sb * q.C[k] / q.D[k + 1];
        } else {
            cb = sb;
        }
    }
    // row 2's diagonal also enters S(1,2): d(c1 d1 / d2)/d d2 = -c1 d1 / d2^2
    if (r == 1) db += q.mu[k - 1] * xv(k) * q.C[k - 1] * q.D[k - 1] / (q.D[k] * q.D[k]);
}

// lam in chain order from the adjoints of the increments (X rows i = 1..nx,
// j = 2..ny, then Y rows i = 2..nx, j = 1..ny).
// Rows flagged in Z (the second split's identity rows; null: none) get +0.
// Thread 0 also clears red[slot], red[slot + 1] (red null: none).
__global__ __launch_bounds__(AT) void k_adj_gather(int nx, int ny, int ld, const double *__restrict__ ub,
                                                   const double *__restrict__ vb, const unsigned char *__restrict__ Z,
                                                   double *__restrict__ lam, unsigned long long *red, int slot) {
    const long n1 = (long)nx * (ny - 1), n2 = (long)(nx - 1) * ny;
    const long k = (long)blockIdx.x * AT + threadIdx.x;
    if (red && k == 0) {
        red[slot] = 0ull;
        red[slot + 1] = 0ull;
    }
    if (Z && k < n1 + n2 && Z[k]) {
        lam[k] = 0.0;
        return;
    }
    if (k < n1) {
        const int i = 1 + (int)(k % nx), j = 2 + (int)(k / nx);
        lam[k] = ub[WD2_IX(i, j)];
    } else if (k < n1 + n2) {
        const long q = k - n1;
        const int i = 2 + (int)(q % (nx - 1)), j = 1 + (int)(q / (nx - 1));
        lam[k] = vb[WD2_IX(i, j)];
    }
}

__global__ __launch_bounds__(AT) void k_adj_zmask(long n, const unsigned char *__restrict__ Z,
                                                  const double *__restrict__ in, double *__restrict__ out) {
    const long k = (long)blockIdx.x * AT + threadIdx.x;
    if (k < n) out[k] = Z[k] ? 0.0 : in[k];
}

// ------------------------------------------------------------ assembly
// Forward values the transposes need, as the forward kernels form them.
#define F(a, b) f[WD2_IX(a, b)]
// ConvCoef case 4 (momentum.f:944-951), djac = 2: written for i = 0..nx, j = 1..ny
__device__ inline double cj1_x(const Metrics &m, int ld, const double *u, const double *v, int i, int j) {
    return 2.0 * m.yeu[WD2_IX(i, j)] * u[WD2_IX(i, j)] -
           m.xeu[WD2_IX(i, j)] * (v[WD2_IX(i + 1, j)] + v[WD2_IX(i, j)] + v[WD2_IX(i + 1, j - 1)] + v[WD2_IX(i, j - 1)]) /
               4.0;
}
// ConvCoef case 5 (momentum.f:953-961), djac = 2: written for i = 1..nx, j = 0..ny
__device__ inline double cj1_y(const Metrics &m, int ld, const double *u, const double *v, int i, int j) {
    return m.yev[WD2_IX(i, j)] * (u[WD2_IX(i, j + 1)] + u[WD2_IX(i - 1, j + 1)] + u[WD2_IX(i, j)] + u[WD2_IX(i - 1, j)]) /
               4.0 -
           2.0 * m.xev[WD2_IX(i, j)] * v[WD2_IX(i, j)];
}
// ConvCoef case 1 (X, metrics xzn, xec, yzn, yec), djac = 1:
// c1 written i = 1..nx+1, j = 1..ny+1; c2 written i = 1..nx, j = 1..ny
__device__ inline double c1_x(const Metrics &m, int ld, const double *u, const double *v, int i, int j) {
    return (m.yec[WD2_IX(i, j)] * (u[WD2_IX(i, j)] + u[WD2_IX(i - 1, j)]) -
            m.xec[WD2_IX(i, j)] * (v[WD2_IX(i, j)] + v[WD2_IX(i, j - 1)])) *
           0.5;
}
__device__ inline double c2_x(const Metrics &m, int ld, const double *u, const double *v, int i, int j) {
    return (m.xzn[WD2_IX(i, j)] * (v[WD2_IX(i + 1, j)] + v[WD2_IX(i, j)]) -
            m.yzn[WD2_IX(i, j)] * (u[WD2_IX(i, j + 1)] + u[WD2_IX(i, j)])) *
           0.5;
}
// ConvCoef case 2 (Y, metrics xzc, xen, yzc, yen), djac = 1:
// c1 written i = 1..nx, j = 1..ny; c2 written i = 1..nx+1, j = 1..ny+1
__device__ inline double c1_y(const Metrics &m, int ld, const double *u, const double *v, int i, int j) {
    return (m.yen[WD2_IX(i, j)] * (u[WD2_IX(i, j + 1)] + u[WD2_IX(i, j)]) -
            m.xen[WD2_IX(i, j)] * (v[WD2_IX(i + 1, j)] + v[WD2_IX(i, j)])) *
           0.5;
}
__device__ inline double c2_y(const Metrics &m, int ld, const double *u, const double *v, int i, int j) {
    return (m.xzc[WD2_IX(i, j)] * (v[WD2_IX(i, j)] + v[WD2_IX(i, j - 1)]) -
            m.yzc[WD2_IX(i, j)] * (u[WD2_IX(i, j)] + u[WD2_IX(i - 1, j)])) *
           0.5;
}

// The rows of one component transposed: the adjoints of the first split's
// chain coefficients and right-hand side (bb = nu) go through the assembly
// (momentum.f:350-384; 675-754), DConvU/V, DDiffU/V (1015-1045; 1079-1109) and
// the ConvCoef cases onto the fields us, vs and (with_n) un, vn.  The second
// split's coefficients need no adjoint: at a converged q-l fixed point they
// only precondition.  Without porous regions and buoyancy the porosity terms
// are +0.
//
// A workgroup takes GT_X x GT_Y rows and adds their contributions up in LDS: fb
// to the component's own field, cj, c1, c2 to the ConvCoef outputs.  All of it
// is linear in the rows, so the tile's ConvCoef adjoints are taken on to the
// fields at once, in gather form, whether or not a neighbouring tile adds to
// the same face, and only the fields' sums go to memory: about 3 FP64 atomics
// a row, where scattering each term took some 40 (five launches,
// 93 us an iteration on 512^2 cells, bound by the atomics; here 37; tiles of
// eight rows, 512 lanes at 128 registers, 40).
constexpr int GT_X = 64, GT_Y = 4, GT_T = GT_X * GT_Y;
constexpr int GT_W = GT_X + 6, GT_H = GT_Y + 6;   // the rows' reach is 2; a ring of zeros

struct GtArgs {
    int nx, ny, ld, with_n;
    double dk, re;
    Metrics m;
    const double *us, *vs, *un, *vn;
    AdjChain q;
    Chains cs;
    double *usb, *vsb, *unb, *vnb;
};

template <int COMP>
__device__ inline void gt_tile(const GtArgs &A, int tile, double *fb, double *cj, double *c1, double *c2) {
    const int nx = A.nx, ny = A.ny, ld = A.ld, tid = threadIdx.x;
    const Metrics &m = A.m;
    const int ib = COMP == 1 ? 1 : 2, jb = COMP == 1 ? 2 : 1, ni = nx - ib + 1, nj = ny - jb + 1;
    const int gx = (ni + GT_X - 1) / GT_X;
    const int I0 = ib + (tile % gx) * GT_X, J0 = jb + (tile / gx) * GT_Y;
    const int oi = I0 - 3, oj = J0 - 3;
    auto at = [&](int i, int j) { return (j - oj) * GT_W + (i - oi); };
    auto add = [&](double *f, int i, int j, double v) { atomicAdd(&f[at(i, j)], v); };
    const int i = I0 + (tid & (GT_X - 1)), j = J0 + tid / GT_X;
    const bool row = i <= nx && j <= ny;
    const size_t p = WD2_IX(i, j);
    double b = 0.0, rkj = 0.0, gc = 0.0, gd = 0.0;
    if (row) {
        const long k = (COMP == 1 ? 0 : A.cs.n1) + (long)(j - jb) * ni + (i - ib);
        b = A.q.mu[k];
        rkj = A.dk * 0.5 * (COMP == 1 ? m.dju : m.djv)[p];
        // right-hand side: b = un - us - rkj (cnvs + cnvn) + rkj re1 (difs + difn)
        gc = -rkj * b;
        gd = rkj * (1.0 / A.re) * b;
    }
    for (int lev = 0; lev < 1 + A.with_n; lev++) {
        const double *u = lev ? A.un : A.us, *v = lev ? A.vn : A.vs, *f = COMP == 1 ? u : v;
        for (int q = tid; q < GT_W * GT_H; q += GT_T) fb[q] = cj[q] = c1[q] = c2[q] = 0.0;
        __syncthreads();
        if (row && lev == 0) {
            // split 1: upwinding on cj1(i,j); cj1(nx+1, j) is never written (+0)
            const long k = (COMP == 1 ? 0 : A.cs.n1) + (long)(j - jb) * ni + (i - ib);
            double ab, db, cb;
            adj_coef(A.q, A.cs, k, b, ab, db, cb);
            if (ab != 0.0 || db != 0.0 || cb != 0.0) {
                const double c = COMP == 1 ? cj1_x(m, ld, u, v, i, j) : cj1_y(m, ld, u, v, i, j);
                if (c >= 0.0) {
                    add(cj, i - 1, j, -rkj * ab);
                    add(cj, i, j, rkj * db);
                } else {
                    add(cj, i, j, -rkj * db);
                    if (i + 1 <= nx) add(cj, i + 1, j, rkj * cb);
                }
            }
        }
        if (row && b != 0.0) {
            double c1w, c1e, c2s, c2n, aW, aE, bW, bE, bS, bN, gS, gN;
            if (COMP == 1) {
                c1w = c1_x(m, ld, u, v, i, j), c1e = c1_x(m, ld, u, v, i + 1, j);
                c2s = c2_x(m, ld, u, v, i, j - 1), c2n = c2_x(m, ld, u, v, i, j);
                aW = m.rac[p], aE = m.rac[WD2_IX(i + 1, j)];
                bW = m.rbc[p], bE = m.rbc[WD2_IX(i + 1, j)];
                bS = m.rbn[WD2_IX(i, j - 1)], bN = m.rbn[p];
                gS = m.rgn[WD2_IX(i, j - 1)], gN = m.rgn[p];
            } else {
                c1w = c1_y(m, ld, u, v, i - 1, j), c1e = c1_y(m, ld, u, v, i, j);
                c2s = c2_y(m, ld, u, v, i, j), c2n = c2_y(m, ld, u, v, i, j + 1);
                aW = m.ran[WD2_IX(i - 1, j)], aE = m.ran[p];
                bW = m.rbn[WD2_IX(i - 1, j)], bE = m.rbn[p];
                bS = m.rbc[p], bN = m.rbc[WD2_IX(i, j + 1)];
                gS = m.rgc[p], gN = m.rgc[WD2_IX(i, j + 1)];
            }
            add(fb, i, j - 1, (bW - bE + gS) * gd - c2s * gc);
            add(fb, i - 1, j, (aW - bN + bS) * gd - c1w * gc);
            add(fb, i, j, -(aE + aW + gN + gS) * gd + (c1e - c1w + c2n - c2s) * gc + (lev ? b : -b));
            add(fb, i + 1, j, (aE + bN - bS) * gd + c1e * gc);
            add(fb, i, j + 1, (bE - bW + gN) * gd + c2n * gc);
            if (bW != 0.0 || bE != 0.0 || bS != 0.0 || bN != 0.0) {   // none on a Cartesian grid
                add(fb, i - 1, j - 1, (bW + bS) * gd);
                add(fb, i + 1, j - 1, -(bE + bS) * gd);
                add(fb, i - 1, j + 1, -(bW + bN) * gd);
                add(fb, i + 1, j + 1, (bE + bN) * gd);
            }
            const double f0 = f[p];
            const int w1 = COMP == 1 ? 0 : 1;   // the west face is c1(i, j) / c1(i-1, j), the south one as well
            add(c1, i - w1, j, (-f[WD2_IX(i - 1, j)] - f0) * gc);
            add(c1, i + 1 - w1, j, (f0 + f[WD2_IX(i + 1, j)]) * gc);
            add(c2, i, j - 1 + w1, (-f[WD2_IX(i, j - 1)] - f0) * gc);
            add(c2, i, j + w1, (f0 + f[WD2_IX(i, j + 1)]) * gc);
        }
        __syncthreads();
        // a face's sum times a metric there (0 where no row of the tile added)
        auto mv = [&](const double *c, const double *mt, int a, int e) {
            const double x = c[at(a, e)];
            return x != 0.0 ? mt[WD2_IX(a, e)] * x : 0.0;
        };
        for (int q = tid; q < (GT_W - 2) * (GT_H - 2); q += GT_T) {
            const int a = oi + 1 + q % (GT_W - 2), e = oj + 1 + q / (GT_W - 2);
            if (a < 0 || a > nx + 1 || e < 0 || e > ny + 1) continue;
            double own = fb[at(a, e)], oth;
            if (COMP == 1) {
                // case 4: cj1 = 2 yeu u - xeu (4 v) / 4; case 1: c1, c2
                own += 2.0 * mv(cj, m.yeu, a, e) + 0.5 * (mv(c1, m.yec, a, e) + mv(c1, m.yec, a + 1, e)) -
                       0.5 * (mv(c2, m.yzn, a, e - 1) + mv(c2, m.yzn, a, e));
                oth = -0.25 * (mv(cj, m.xeu, a - 1, e) + mv(cj, m.xeu, a, e) + mv(cj, m.xeu, a - 1, e + 1) +
                               mv(cj, m.xeu, a, e + 1)) -
                      0.5 * (mv(c1, m.xec, a, e) + mv(c1, m.xec, a, e + 1)) +
                      0.5 * (mv(c2, m.xzn, a - 1, e) + mv(c2, m.xzn, a, e));
            } else {
                // case 5: cj1 = yev (4 u) / 4 - 2 xev v; case 2: c1, c2
                own += -2.0 * mv(cj, m.xev, a, e) - 0.5 * (mv(c1, m.xen, a - 1, e) + mv(c1, m.xen, a, e)) +
                       0.5 * (mv(c2, m.xzc, a, e) + mv(c2, m.xzc, a, e + 1));
                oth = 0.25 * (mv(cj, m.yev, a, e - 1) + mv(cj, m.yev, a + 1, e - 1) + mv(cj, m.yev, a, e) +
                              mv(cj, m.yev, a + 1, e)) +
                      0.5 * (mv(c1, m.yen, a, e - 1) + mv(c1, m.yen, a, e)) -
                      0.5 * (mv(c2, m.yzc, a, e) + mv(c2, m.yzc, a + 1, e));
            }
            double *ub = lev ? A.unb : A.usb, *vb = lev ? A.vnb : A.vsb;
            aadd(&(COMP == 1 ? ub : vb)[WD2_IX(a, e)], own);
            aadd(&(COMP == 1 ? vb : ub)[WD2_IX(a, e)], oth);
        }
        __syncthreads();
    }
}

// Workgroups [0, t1) take the x-momentum's tiles, the rest the y-momentum's.
__global__ __launch_bounds__(GT_T, 3) void k_adj_gtrans(GtArgs A, int t1) {
    __shared__ double fb[GT_W * GT_H], cj[GT_W * GT_H], c1[GT_W * GT_H], c2[GT_W * GT_H];
    if ((int)blockIdx.x < t1)
        gt_tile<1>(A, blockIdx.x, fb, cj, c1, c2);
    else
        gt_tile<2>(A, (int)blockIdx.x - t1, fb, cj, c1, c2);
}

// ------------------------------------------------------------ boundary fills
// VelBoundCond with no-slip walls on all four sides of one region covering
// the grid (iW = 1, iE = nx, jS = 1, jN = ny), replayed in reverse: sides N,
// S, E, W, and within a side the v assignments before the u ones.  The
// wall values (a profile value per line, else the constant) receive the
// adjoints of 2 U in bc_bar[side][var][line] (k = j on W/E, i on S/N).
__global__ __launch_bounds__(1024) void k_adj_vbc(Regions R, int ld, double *ub, double *vb, double *bcb) {
    const int nx = R.nx, ny = R.ny, t = threadIdx.x;
    const int W = (nx + 2 > ny + 2) ? nx + 2 : ny + 2;
    auto bc = [&](int side, int var, int k) -> double * { return bcb + ((side - 1) * 2 + (var - 1)) * (size_t)W + k; };
    // N: v(i, ny) = 0 (i = 1..nx); u(i, ny+1) = 2 U(i) - u(i, ny) (i = 2..nx)
    for (int i = 1 + t; i <= nx; i += 1024) vb[WD2_IX(i, ny)] = 0.0;
    __syncthreads();
    for (int i = 2 + t; i <= nx; i += 1024) {
        const double g = ub[WD2_IX(i, ny + 1)];
        ub[WD2_IX(i, ny)] -= g;
        *bc(NORTH, VU, i) += 2.0 * g;
        ub[WD2_IX(i, ny + 1)] = 0.0;
    }
    __syncthreads();
    // S: v(i, 1) = 0 (i = 1..nx); u(i, 1) = 2 U(i) - u(i, 2) (i = 2..nx)
    for (int i = 1 + t; i <= nx; i += 1024) vb[WD2_IX(i, 1)] = 0.0;
    __syncthreads();
    for (int i = 2 + t; i <= nx; i += 1024) {
        const double g = ub[WD2_IX(i, 1)];
        ub[WD2_IX(i, 2)] -= g;
        *bc(SOUTH, VU, i) += 2.0 * g;
        ub[WD2_IX(i, 1)] = 0.0;
    }
    __syncthreads();
    // E: v(nx+1, j) = 2 V(j) - v(nx, j) (j = 2..ny); u(nx, j) = 0 (j = 1..ny)
    for (int j = 2 + t; j <= ny; j += 1024) {
        const double g = vb[WD2_IX(nx + 1, j)];
        vb[WD2_IX(nx, j)] -= g;
        *bc(EAST, VV, j) += 2.0 * g;
        vb[WD2_IX(nx + 1, j)] = 0.0;
    }
    __syncthreads();
    for (int j = 1 + t; j <= ny; j += 1024) ub[WD2_IX(nx, j)] = 0.0;
    __syncthreads();
    // W: v(1, j) = 2 V(j) - v(2, j) (j = 2..ny); u(1, j) = 0 (j = 1..ny)
    for (int j = 2 + t; j <= ny; j += 1024) {
        const double g = vb[WD2_IX(1, j)];
        vb[WD2_IX(2, j)] -= g;
        *bc(WEST, VV, j) += 2.0 * g;
        vb[WD2_IX(1, j)] = 0.0;
    }
    __syncthreads();
    for (int j = 1 + t; j <= ny; j += 1024) ub[WD2_IX(1, j)] = 0.0;
}

// PresBoundCond with walls (p(ghost) = value + p(inner)) in reverse: N, S, E, W.
__global__ __launch_bounds__(1024) void k_adj_pbc(int nx, int ny, int ld, double *pb) {
    const int t = threadIdx.x;
    for (int i = 2 + t; i <= nx; i += 1024) {
        pb[WD2_IX(i, ny)] += pb[WD2_IX(i, ny + 1)];
        pb[WD2_IX(i, ny + 1)] = 0.0;
    }
    __syncthreads();
    for (int i = 2 + t; i <= nx; i += 1024) {
        pb[WD2_IX(i, 2)] += pb[WD2_IX(i, 1)];
        pb[WD2_IX(i, 1)] = 0.0;
    }
    __syncthreads();
    for (int j = 2 + t; j <= ny; j += 1024) {
        pb[WD2_IX(nx, j)] += pb[WD2_IX(nx + 1, j)];
        pb[WD2_IX(nx + 1, j)] = 0.0;
    }
    __syncthreads();
    for (int j = 2 + t; j <= ny; j += 1024) {
        pb[WD2_IX(2, j)] += pb[WD2_IX(1, j)];
        pb[WD2_IX(1, j)] = 0.0;
    }
}

// ------------------------------------------------------------ Project / Ppe
// Project transposed (utility.f:314-321, 384-391): u, v pass through; p
// receives minus the gradient operator's transpose of their adjoints.
__global__ __launch_bounds__(AT) void k_adj_project(int nx, int ny, int ld, double dk, Metrics m,
                                                    const double *__restrict__ ub, const double *__restrict__ vb,
                                                    double *pb) {
    const long q = (long)blockIdx.x * AT + threadIdx.x;
    if (q >= (long)(nx + 2) * (ny + 2)) return;
    const int i = (int)(q % (nx + 2)), j = (int)(q / (nx + 2));
    if (i >= 2 && i <= nx - 1 && j >= 2 && j <= ny) {
        const double g = ub[WD2_IX(i, j)], djk = m.dju[WD2_IX(i, j)] * dk;
        const double gx = djk * m.yeu[WD2_IX(i, j)] * g, gy = djk * m.yzu[WD2_IX(i, j)] * g / 4.0;
        aadd(&pb[WD2_IX(i + 1, j)], -gx);
        aadd(&pb[WD2_IX(i, j)], gx);
        aadd(&pb[WD2_IX(i + 1, j + 1)], gy);
        aadd(&pb[WD2_IX(i, j + 1)], gy);
        aadd(&pb[WD2_IX(i + 1, j - 1)], -gy);
        aadd(&pb[WD2_IX(i, j - 1)], -gy);
    }
    if (i >= 2 && i <= nx && j >= 2 && j <= ny - 1) {
        const double g = vb[WD2_IX(i, j)], djk = m.djv[WD2_IX(i, j)] * dk;
        const double gx = djk * m.xev[WD2_IX(i, j)] * g / 4.0, gy = djk * m.xzv[WD2_IX(i, j)] * g;
        aadd(&pb[WD2_IX(i + 1, j + 1)], gx);
        aadd(&pb[WD2_IX(i + 1, j)], gx);
        aadd(&pb[WD2_IX(i - 1, j + 1)], -gx);
        aadd(&pb[WD2_IX(i - 1, j)], -gx);
        aadd(&pb[WD2_IX(i, j + 1)], -gy);
        aadd(&pb[WD2_IX(i, j)], gy);
    }
}

// Divergence case 1 (pressure.f:287-299) transposed, for g = lam / dk on
// the pressure cells i = 2..nx, j = 2..ny; and the frozen ghosts' share of
// the Poisson solve: pb(ghost) -= coupling * lam.
__global__ __launch_bounds__(AT) void k_adj_div(int nx, int ny, int ld, double dk, Metrics m,
                                                const double *__restrict__ lam, double *ub, double *vb, double *pb) {
    const long q = (long)blockIdx.x * AT + threadIdx.x;
    if (q >= (long)(nx - 1) * (ny - 1)) return;
    const int i = 2 + (int)(q % (nx - 1)), j = 2 + (int)(q / (nx - 1));
    const double l = lam[WD2_IX(i, j)], g = l / dk;
    if (i == 2) aadd(&pb[WD2_IX(1, j)], -m.rau[WD2_IX(1, j)] * l);
    if (i == nx) aadd(&pb[WD2_IX(nx + 1, j)], -m.rau[WD2_IX(nx, j)] * l);
    if (j == 2) aadd(&pb[WD2_IX(i, 1)], -m.rgv[WD2_IX(i, 1)] * l);
    if (j == ny) aadd(&pb[WD2_IX(i, ny + 1)], -m.rgv[WD2_IX(i, ny)] * l);
    if (g == 0.0) return;
    // ucij = yeu(i,j) u(i,j) - xeu(i,j) (v(i+1,j) + v(i,j) + v(i+1,j-1) + v(i,j-1)) / 4
    aadd(&ub[WD2_IX(i, j)], m.yeu[WD2_IX(i, j)] * g);
    double gv = -m.xeu[WD2_IX(i, j)] * g / 4.0;
    aadd(&vb[WD2_IX(i + 1, j)], gv);
    aadd(&vb[WD2_IX(i, j)], gv);
    aadd(&vb[WD2_IX(i + 1, j - 1)], gv);
    aadd(&vb[WD2_IX(i, j - 1)], gv);
    // - uci1j
    aadd(&ub[WD2_IX(i - 1, j)], -m.yeu[WD2_IX(i - 1, j)] * g);
    gv = m.xeu[WD2_IX(i - 1, j)] * g / 4.0;
    aadd(&vb[WD2_IX(i, j)], gv);
    aadd(&vb[WD2_IX(i - 1, j)], gv);
    aadd(&vb[WD2_IX(i, j - 1)], gv);
    aadd(&vb[WD2_IX(i - 1, j - 1)], gv);
    // vcij = xzv(i,j) v(i,j) - yzv(i,j) (u(i,j+1) + u(i-1,j+1) + u(i,j) + u(i-1,j)) / 4
    aadd(&vb[WD2_IX(i, j)], m.xzv[WD2_IX(i, j)] * g);
    double gu = -m.yzv[WD2_IX(i, j)] * g / 4.0;
    aadd(&ub[WD2_IX(i, j + 1)], gu);
    aadd(&ub[WD2_IX(i - 1, j + 1)], gu);
    aadd(&ub[WD2_IX(i, j)], gu);
    aadd(&ub[WD2_IX(i - 1, j)], gu);
    // - vcij1
    aadd(&vb[WD2_IX(i, j - 1)], -m.xzv[WD2_IX(i, j - 1)] * g);
    gu = m.yzv[WD2_IX(i, j - 1)] * g / 4.0;
    aadd(&ub[WD2_IX(i, j)], gu);
    aadd(&ub[WD2_IX(i - 1, j)], gu);
    aadd(&ub[WD2_IX(i, j - 1)], gu);
    aadd(&ub[WD2_IX(i - 1, j - 1)], gu);
}

// nu += z over n elements with red[slot] = max |z| and red[slot + 1] =
// max |nu| (the slots start at +0; a NaN wins).
__global__ __launch_bounds__(AT) void k_adj_update(long n, const double *__restrict__ z, double *__restrict__ nu,
                                                   unsigned long long *red, int slot) {
    __shared__ double sh[2][AT / 64];
    double mz = 0.0, mn = 0.0;
    for (long k = (long)blockIdx.x * AT + threadIdx.x; k < n; k += (long)gridDim.x * AT) {
        const double zk = z[k], v = nu[k] + zk;
        nu[k] = v;
        if (!(fabs(zk) <= mz)) mz = fabs(zk);
        if (!(fabs(v) <= mn)) mn = fabs(v);
    }
    for (int off = 32; off > 0; off >>= 1) {
        const double a = __shfl_xor(mz, off), b = __shfl_xor(mn, off);
        if (!(a <= mz)) mz = a;
        if (!(b <= mn)) mn = b;
    }
    if ((threadIdx.x & 63) == 0) {
        sh[0][threadIdx.x >> 6] = mz;
        sh[1][threadIdx.x >> 6] = mn;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < AT / 64; w++) {
            if (!(sh[0][w] <= mz)) mz = sh[0][w];
            if (!(sh[1][w] <= mn)) mn = sh[1][w];
        }
        atomicMax(&red[slot], dbits(mz));
        atomicMax(&red[slot + 1], dbits(mn));
    }
}

// y += alpha x and y = 0 over n elements.
__global__ __launch_bounds__(AT) void k_adj_axpy(long n, double alpha, const double *__restrict__ x, double *y) {
    const long k = (long)blockIdx.x * AT + threadIdx.x;
    if (k < n) y[k] += alpha * x[k];
}
__global__ __launch_bounds__(AT) void k_adj_zero(long n, double *y) {
    const long k = (long)blockIdx.x * AT + threadIdx.x;
    if (k < n) y[k] = 0.0;
}

// The adjoint of a step's initial u (comp 1) or v (comp 2) from the
// converged q-l fixed point: out = fnb + fsb on the points the iterations
// leave at their initial value (us = un there), out = fnb on the points they
// update (u: i = 2..nx-1, j = 2..ny; v: i = 2..nx, j = 2..ny-1).
__global__ __launch_bounds__(AT) void k_adj_combine(int comp, int nx, int ny, int ld, const double *__restrict__ fsb,
                                                    const double *__restrict__ fnb, double *__restrict__ out) {
    const long q = (long)blockIdx.x * AT + threadIdx.x;
    if (q >= (long)(nx + 2) * (ny + 2)) return;
    const int i = (int)(q % (nx + 2)), j = (int)(q / (nx + 2));
    const bool act = comp == 1 ? (i >= 2 && i <= nx - 1 && j >= 2 && j <= ny)
                               : (i >= 2 && i <= nx && j >= 2 && j <= ny - 1);
    const size_t p = WD2_IX(i, j);
    out[p] = act ? fnb[p] : fnb[p] + fsb[p];
}

// red[slot] = max(red[slot], max |x|) over n elements (non-negative doubles
// order like their bit patterns; red must start at +0).  A NaN wins.
__global__ __launch_bounds__(AT) void k_adj_maxabs(long n, const double *__restrict__ x, unsigned long long *red,
                                                   int slot) {
    __shared__ double sh[AT / 64];
    double m = 0.0;
    for (long k = (long)blockIdx.x * AT + threadIdx.x; k < n; k += (long)gridDim.x * AT) {
        const double a = fabs(x[k]);
        if (!(a <= m)) m = a;
    }
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(m, off);
        if (!(o <= m)) m = o;
    }
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < AT / 64; w++)
            if (!(sh[w] <= m)) m = sh[w];
        atomicMax(&red[slot], dbits(m));
    }
}

// ------------------------------------------------------------ launchers
static inline dim3 ag(long n) { return dim3((unsigned)((n + AT - 1) / AT)); }

void launch_adj_tchain(long n, const Chains &cs, const double *A, const double *D, const double *C, double *At,
                       double *Dt, double *Ct, unsigned long long *dom, hipStream_t s) {
    const long nb = std::min<long>(512, (n + AT - 1) / AT);
    hipLaunchKernelGGL(k_adj_tchain, dim3((unsigned)std::max<long>(nb, 1)), dim3(AT), 0, s, n, cs, A, D, C, At, Dt, Ct,
                       dom);
}
void launch_adj_gather(int nx, int ny, int ld, const double *ub, const double *vb, const unsigned char *Z,
                       double *lam, unsigned long long *red, int slot, hipStream_t s) {
    const long n = (long)nx * (ny - 1) + (long)(nx - 1) * ny;
    hipLaunchKernelGGL(k_adj_gather, ag(n), dim3(AT), 0, s, nx, ny, ld, ub, vb, Z, lam, red, slot);
}
void launch_adj_update(long n, const double *z, double *nu, unsigned long long *red, int slot, hipStream_t s) {
    const long nb = std::min<long>(1024, (n + AT - 1) / AT);
    hipLaunchKernelGGL(k_adj_update, dim3((unsigned)std::max<long>(nb, 1)), dim3(AT), 0, s, n, z, nu, red, slot);
}
void launch_adj_zmask(long n, const unsigned char *Z, const double *in, double *out, hipStream_t s) {
    hipLaunchKernelGGL(k_adj_zmask, ag(n), dim3(AT), 0, s, n, Z, in, out);
}
void launch_adj_gtrans(int nx, int ny, int ld, double dk, double re, const Metrics &m, const double *us,
                       const double *vs, const double *un, const double *vn, const Chain &ch, const Chains &cs,
                       const double *nu, const unsigned char *XK, int with_n, double *usb, double *vsb, double *unb,
                       double *vnb, hipStream_t s) {
    const GtArgs A{nx, ny, ld, with_n, dk, re, m, us, vs, un, vn, AdjChain{ch.a, ch.d, ch.c, nu, ch.x, XK}, cs,
                   usb, vsb, unb, vnb};
    auto tiles = [](int ni, int nj) { return ((ni + GT_X - 1) / GT_X) * ((nj + GT_Y - 1) / GT_Y); };
    const int t1 = tiles(nx, ny - 1), t2 = tiles(nx - 1, ny);
    hipLaunchKernelGGL(k_adj_gtrans, dim3(t1 + t2), dim3(GT_T), 0, s, A, t1);
}
void launch_adj_vbc(const Regions &R, int ld, double *ub, double *vb, double *bcb, hipStream_t s) {
    hipLaunchKernelGGL(k_adj_vbc, dim3(1), dim3(1024), 0, s, R, ld, ub, vb, bcb);
}
void launch_adj_pbc(int nx, int ny, int ld, double *pb, hipStream_t s) {
    hipLaunchKernelGGL(k_adj_pbc, dim3(1), dim3(1024), 0, s, nx, ny, ld, pb);
}
void launch_adj_project(int nx, int ny, int ld, double dk, const Metrics &m, const double *ub, const double *vb,
                        double *pb, hipStream_t s) {
    hipLaunchKernelGGL(k_adj_project, ag((long)(nx + 2) * (ny + 2)), dim3(AT), 0, s, nx, ny, ld, dk, m, ub, vb, pb);
}
void launch_adj_div(int nx, int ny, int ld, double dk, const Metrics &m, const double *lam, double *ub, double *vb,
                    double *pb, hipStream_t s) {
    hipLaunchKernelGGL(k_adj_div, ag((long)(nx - 1) * (ny - 1)), dim3(AT), 0, s, nx, ny, ld, dk, m, lam, ub, vb, pb);
}
void launch_adj_axpy(long n, double alpha, const double *x, double *y, hipStream_t s) {
    hipLaunchKernelGGL(k_adj_axpy, ag(n), dim3(AT), 0, s, n, alpha, x, y);
}
void launch_adj_zero(long n, double *y, hipStream_t s) { hipLaunchKernelGGL(k_adj_zero, ag(n), dim3(AT), 0, s, n, y); }
void launch_adj_combine(int comp, int nx, int ny, int ld, const double *fsb, const double *fnb, double *out,
                        hipStream_t s) {
    hipLaunchKernelGGL(k_adj_combine, ag((long)(nx + 2) * (ny + 2)), dim3(AT), 0, s, comp, nx, ny, ld, fsb, fnb,
                       out);
}
void launch_adj_maxabs(long n, const double *x, unsigned long long *red, int slot, hipStream_t s) {
    const long nb = std::min<long>(1024, (n + AT - 1) / AT);
    hipLaunchKernelGGL(k_adj_maxabs, dim3((unsigned)std::max<long>(nb, 1)), dim3(AT), 0, s, n, x, red, slot);
}

}  // namespace wd2
