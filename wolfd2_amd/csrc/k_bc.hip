// k_bc.hip -- ghost-cell and wall fills (bound_cond.f:VelBoundCond 511-847,
// PresBoundCond 853-1024, VelOutflowBCs 1656-1874).
//
// These are O(nx+ny) line updates whose order matters: a later side reads
// values an earlier side wrote (corners), and the mass-conserving outlet
// formulas are first-order recurrences along the boundary.  One workgroup
// walks the regions and sides in the reference's order; each loop whose
// iterations are independent is spread over the workgroup, the recurrences
// run on one lane from LDS, and a barrier separates loops that depend on each
// other.  Launches and memory latency bound these kernels: one launch holds
// the velocity and the pressure fills (two workgroups), applied as often as a
// step applies them back to back.
//
// Boundary values: the reference's dBCVal holds one constant per region side
// and variable.  A side may instead carry a profile, one value per grid line
// (Regions::bcp); every formula is the reference's with the constant replaced
// by the line's value, so a profile of constant values gives the same bits.
#include "wd2_dev.hpp"
#include "wd2_launch.hpp"

namespace wd2 {

constexpr int BC_THREADS = 1024;
constexpr int BC_CH = 1024;   // outlet recurrence rows staged in LDS at a time

#define PAR(var, lo, hi) for (int var = (lo) + (int)threadIdx.x; var <= (hi); var += BC_THREADS)
#define SYNC() __syncthreads()

// A region's table entries, loaded by as many lanes at once into LDS: the
// fills then wait for one table load instead of a chain of them per side
// (profile offsets and constants of u, v, p on the four sides).
struct BcRegion {
    int brd[4], btp[4], rtype;
    int prof[4][3];
    double cst[4][3];
};
__device__ inline void bc_load(const Regions &R, int ir, int jr, BcRegion &g) {
    const int t = threadIdx.x;
    if (t < 4)
        g.brd[t] = R.border(ir, jr, t + 1);
    else if (t < 8)
        g.btp[t - 4] = R.btype(ir, jr, t - 3);
    else if (t == 8)
        g.rtype = R.type(ir, jr);
    else if (t >= 64 && t < 76)
        g.prof[(t - 64) / 3][(t - 64) % 3] = R.prof(ir, jr, (t - 64) / 3 + 1, (t - 64) % 3 + 1);
    else if (t >= 128 && t < 140)
        g.cst[(t - 128) / 3][(t - 128) % 3] = R.bc(ir, jr, (t - 128) / 3 + 1, (t - 128) % 3 + 1);
    SYNC();
}
// Regions::bcp from the loaded entries.
__device__ inline double bc_val(const Regions &R, const BcRegion &g, int side, int var, int k) {
    const int o = g.prof[side - 1][var - 1];
    return o >= 0 ? R.pval[o + k] : g.cst[side - 1][var - 1];
}

// The mass-conserving outlets' recurrence x_k = (neg ? -x_(k-1) : x_(k-1)) +
// t1_k + (sub ? -t2_k : t2_k) (left to right), k = lo..hi from x_(lo-1): the
// terms are formed by all lanes and staged in LDS, one lane runs the chain on
// them, all lanes store.  One lane reading each row's operands from memory
// took 140 ns a row (70 us for a 512-row outlet, now about 20); the chain
// itself is two dependent additions a row.
template <typename T, bool NEG, bool SUB, typename Term, typename Put>
__device__ inline void bc_chain(T prev, int lo, int hi, T (*st)[BC_CH], Term term, Put put) {
    for (int c0 = lo; c0 <= hi; c0 += BC_CH) {
        const int n = min(BC_CH, hi - c0 + 1);
        for (int q = threadIdx.x; q < n; q += BC_THREADS) term(c0 + q, st[0][q], st[1][q]);
        SYNC();
        if (threadIdx.x == 0) {
            constexpr int U = 8;
            T x = prev;
            for (int q0 = 0; q0 < n; q0 += U) {
                T a[U], b[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    a[u] = st[0][min(q0 + u, BC_CH - 1)];
                    b[u] = st[1][min(q0 + u, BC_CH - 1)];
                }
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const T s = (NEG ? -x : x) + a[u];
                    x = SUB ? s - b[u] : s + b[u];
                    if (q0 + u < n) st[0][q0 + u] = x;
                }
            }
        }
        SYNC();
        for (int q = threadIdx.x; q < n; q += BC_THREADS) put(c0 + q, st[0][q]);
        prev = st[0][n - 1];   // read by every lane before the next chunk's stores
        SYNC();
    }
}

// VelBoundCond (outflow_only = 0) and VelOutflowBCs (outflow_only = 1), by
// one workgroup.  A region's west and east fills touch disjoint columns when
// the region is at least two cells wide (west: columns iW-1..iW+1, east:
// iE-1..iE+1), and its south and north fills disjoint rows likewise, so each
// pair runs between the same two barriers; an outlet recurrence or a narrow
// region keeps the reference's side order with a barrier after each.
template <typename T>
__device__ inline void vel_fill(const Regions &R, int ld, T *__restrict__ u, T *__restrict__ v, int outflow_only,
                                int *__restrict__ err, BcRegion &g, T (*st)[BC_CH], bool loaded) {
    const T dTwo = 2, dThree = 3, dFour = 4, dFive = 5, dEight = 8;
    for (int jr = 1; jr <= R.nj; jr++)
        for (int ir = 1; ir <= R.ni; ir++) {
            if (!loaded) bc_load(R, ir, jr, g);
            const int iW = g.brd[WEST - 1], iE = g.brd[EAST - 1], jS = g.brd[SOUTH - 1], jN = g.brd[NORTH - 1];
#define U(i, j) u[WD2_IX(i, j)]
#define V(i, j) v[WD2_IX(i, j)]
#define BU(side, k) ((T)bc_val(R, g, side, VU, k))
#define BV(side, k) ((T)bc_val(R, g, side, VV, k))
            const int tw = g.btp[WEST - 1], te = g.btp[EAST - 1], ts = g.btp[SOUTH - 1], tn = g.btp[NORTH - 1];
            const bool we = tw != BM_OUTLT2 && te != BM_OUTLT2 && iE - iW >= 2;
            const bool sn = ts != BM_OUTLT2 && tn != BM_OUTLT2 && jN - jS >= 2;
            // ---- WEST
            {
                const int t = tw;
                if (!outflow_only && t == BM_WALL1) {
                    PAR(j, jS, jN) U(iW, j) = 0;
                    PAR(j, jS + 1, jN) V(iW, j) = dTwo * BV(WEST, j) - V(iW + 1, j);
                } else if (!outflow_only && t == BM_WALL2) {
                    PAR(j, jS, jN) U(iW, j) = 0;
                    PAR(j, jS + 1, jN) V(iW, j) = V(iW + 1, j);
                } else if (!outflow_only && t == BM_INLET) {
                    PAR(j, jS, jN) U(iW, j) = BU(WEST, j);
                    PAR(j, jS + 1, jN) V(iW, j) = dTwo * BV(WEST, j) - V(iW + 1, j);
                } else if (t == BM_OUTLT1) {
                    PAR(j, jS, jN) U(iW - 1, j) = BU(WEST, j) + U(iW, j);
                    PAR(j, jS + 1, jN) V(iW, j) = -V(iW + 1, j);
                } else if (t == BM_OUTLT2) {
                    if (!outflow_only) {
                        PAR(j, jS + 1, jN) U(iW, j) = U(iW + 1, j) + V(iW + 1, j) - V(iW + 1, j - 1);
                    } else {  // bound_cond.f:1727 has the opposite sign on the v terms
                        PAR(j, jS + 1, jN) U(iW, j) = U(iW + 1, j) - V(iW + 1, j) + V(iW + 1, j - 1);
                    }
                    SYNC();
                    bc_chain<T, true, false>(
                        V(iW, jS), jS + 1, jN, st,
                        [&](int j, T &a, T &b) {
                            a = dFive * (V(iW + 1, j) - V(iW + 1, j - 1));
                            b = dEight * (U(iW + 1, j) - U(iW, j));
                        },
                        [&](int j, T x) { V(iW, j) = x; });
                } else if (t < BM_INTERN || t > BM_OUTLT2) {
                    if (threadIdx.x == 0) *err = 1000 + WEST;
                }
                if (!we) SYNC();
            }
            // ---- EAST
            {
                const int t = te;
                if (!outflow_only && t == BM_WALL1) {
                    PAR(j, jS, jN) U(iE, j) = 0;
                    PAR(j, jS + 1, jN) V(iE + 1, j) = dTwo * BV(EAST, j) - V(iE, j);
                } else if (!outflow_only && t == BM_WALL2) {
                    PAR(j, jS, jN) U(iE, j) = 0;
                    PAR(j, jS + 1, jN) V(iE + 1, j) = V(iE, j);
                } else if (!outflow_only && t == BM_INLET) {
                    PAR(j, jS, jN) U(iE, j) = BU(EAST, j);
                    PAR(j, jS + 1, jN) V(iE + 1, j) = dTwo * BV(EAST, j) - V(iE, j);
                } else if (t == BM_OUTLT1) {
                    PAR(j, jS, jN) U(iE + 1, j) = BU(EAST, j) + U(iE, j);
                    PAR(j, jS + 1, jN) V(iE + 1, j) = -V(iE, j);
                } else if (t == BM_OUTLT2) {
                    PAR(j, jS + 1, jN) U(iE, j) = U(iE - 1, j) - (V(iE, j) - V(iE, j - 1));
                    SYNC();
                    bc_chain<T, false, true>(
                        V(iE + 1, jS), jS + 1, jN - 1, st,
                        [&](int j, T &a, T &b) {
                            a = dThree * (V(iE, j - 1) - V(iE, j));
                            b = dFour * (U(iE, j) - U(iE - 1, j));
                        },
                        [&](int j, T x) { V(iE + 1, j) = x; });
                } else if (t < BM_INTERN || t > BM_OUTLT2) {
                    if (threadIdx.x == 0) *err = 1000 + EAST;
                }
                SYNC();
            }
            // ---- SOUTH
            {
                const int t = ts;
                if (!outflow_only && t == BM_WALL1) {
                    PAR(i, iW + 1, iE) U(i, jS) = dTwo * BU(SOUTH, i) - U(i, jS + 1);
                    PAR(i, iW, iE) V(i, jS) = 0;
                } else if (!outflow_only && t == BM_WALL2) {
                    PAR(i, iW + 1, iE) U(i, jS) = U(i, jS + 1);
                    PAR(i, iW, iE) V(i, jS) = 0;
                } else if (!outflow_only && t == BM_INLET) {
                    PAR(i, iW + 1, iE) U(i, jS) = dTwo * BU(SOUTH, i) - U(i, jS + 1);
                    PAR(i, iW, iE) V(i, jS) = BV(SOUTH, i);
                } else if (t == BM_OUTLT1) {
                    PAR(i, iW + 1, iE) U(i, jS) = -U(i, jS + 1);
                    PAR(i, iW, iE) V(i, jS) = BV(SOUTH, i) + V(i, jS);
                } else if (t == BM_OUTLT2) {
                    PAR(i, iW + 1, iE) V(i, jS) = V(i, jS + 1) + (U(i, jS + 1) - U(i - 1, jS + 1));
                    SYNC();
                    bc_chain<T, false, true>(
                        U(iW, jS), iW + 1, iE - 1, st,
                        [&](int i, T &a, T &b) {
                            a = dThree * (U(i - 1, jS + 1) - U(i, jS + 1));
                            b = dFour * (V(i, jS + 1) - V(i, jS));
                        },
                        [&](int i, T x) { U(i, jS) = x; });
                } else if (t < BM_INTERN || t > BM_OUTLT2) {
                    if (threadIdx.x == 0) *err = 1000 + SOUTH;
                }
                if (!sn) SYNC();
            }
            // ---- NORTH
            {
                const int t = tn;
                if (!outflow_only && t == BM_WALL1) {
                    PAR(i, iW + 1, iE) U(i, jN + 1) = dTwo * BU(NORTH, i) - U(i, jN);
                    PAR(i, iW, iE) V(i, jN) = 0;
                } else if (!outflow_only && t == BM_WALL2) {
                    PAR(i, iW + 1, iE) U(i, jN + 1) = U(i, jN);
                    PAR(i, iW, iE) V(i, jN) = 0;
                } else if (!outflow_only && t == BM_INLET) {
                    PAR(i, iW + 1, iE) U(i, jN + 1) = dTwo * BU(NORTH, i) - U(i, jN);
                    PAR(i, iW, iE) V(i, jN) = BV(NORTH, i);
                } else if (t == BM_OUTLT1) {
                    PAR(i, iW + 1, iE) U(i, jN + 1) = -U(i, jN);
                    PAR(i, iW, iE) V(i, jN + 1) = BV(NORTH, i) + V(i, jN);
                } else if (t == BM_OUTLT2) {
                    PAR(i, iW, iE) V(i, jN) = V(i, jN - 1) - (U(i, jN) - U(i - 1, jN));
                    SYNC();
                    bc_chain<T, false, true>(
                        U(iW, jN + 1), iW + 1, iE - 1, st,
                        [&](int i, T &a, T &b) {
                            a = dThree * (U(i - 1, jN) - U(i, jN));
                            b = dFour * (V(i, jN) - V(i, jN - 1));
                        },
                        [&](int i, T x) { U(i, jN + 1) = x; });
                } else if (t < BM_INTERN || t > BM_OUTLT2) {
                    if (threadIdx.x == 0) *err = 1000 + NORTH;
                }
                SYNC();
            }
#undef U
#undef V
#undef BU
#undef BV
        }
}

// PresBoundCond, by one workgroup.  West and east (south and north) fills
// write columns (rows) outside those either reads, so each pair shares a
// barrier.
template <typename T>
__device__ inline void pres_fill(const Regions &R, int ld, T *__restrict__ p, int *__restrict__ err, BcRegion &g,
                                 bool loaded) {
    const T dTwo = 2;
#define P(i, j) p[WD2_IX(i, j)]
#define BP(side, k) ((T)bc_val(R, g, side, VP, k))
    for (int jr = 1; jr <= R.nj; jr++)
        for (int ir = 1; ir <= R.ni; ir++) {
            if (!loaded) bc_load(R, ir, jr, g);
            const int iW = g.brd[WEST - 1], iE = g.brd[EAST - 1], jS = g.brd[SOUTH - 1], jN = g.brd[NORTH - 1];
            if (g.rtype == RM_BLOCKG) {
                const int w = iE - iW, h = jN - jS;
                for (int k = threadIdx.x; k < w * h; k += BC_THREADS) P(iW + 1 + k % w, jS + 1 + k / w) = 0;
                SYNC();
                PAR(j, jS + 1, jN) P(iW + 1, j) = BP(WEST, j) + P(iW, j);
                SYNC();
                PAR(j, jS + 1, jN) P(iE, j) = BP(EAST, j) + P(iE + 1, j);
                SYNC();
                PAR(i, iW + 1, iE) P(i, jS + 1) = BP(SOUTH, i) + P(i, jS);
                SYNC();
                PAR(i, iW + 1, iE) P(i, jN) = BP(NORTH, i) + P(i, jN + 1);
                SYNC();
                continue;
            }
            int t = g.btp[WEST - 1];
            if (t == BM_WALL1 || t == BM_WALL2 || t == BM_INLET) {
                PAR(j, jS + 1, jN) P(iW, j) = BP(WEST, j) + P(iW + 1, j);
            } else if (t == BM_OUTLT1 || t == BM_OUTLT2) {
                PAR(j, jS + 1, jN) P(iW, j) = dTwo * BP(WEST, j) - P(iW + 1, j);
            } else if (t != BM_INTERN && threadIdx.x == 0) {
                *err = 1000 + WEST;
            }
            if (iE <= iW) SYNC();
            t = g.btp[EAST - 1];
            if (t == BM_WALL1 || t == BM_WALL2 || t == BM_INLET) {
                PAR(j, jS + 1, jN) P(iE + 1, j) = BP(EAST, j) + P(iE, j);
            } else if (t == BM_OUTLT1 || t == BM_OUTLT2) {
                PAR(j, jS + 1, jN) P(iE + 1, j) = dTwo * BP(EAST, j) - P(iE, j);
            } else if (t != BM_INTERN && threadIdx.x == 0) {
                *err = 1000 + EAST;
            }
            SYNC();
            t = g.btp[SOUTH - 1];
            if (t == BM_WALL1 || t == BM_WALL2 || t == BM_INLET) {
                PAR(i, iW + 1, iE) P(i, jS) = BP(SOUTH, i) + P(i, jS + 1);
            } else if (t == BM_OUTLT1 || t == BM_OUTLT2) {
                PAR(i, iW + 1, iE) P(i, jS) = dTwo * BP(SOUTH, i) - P(i, jS + 1);
            } else if (t != BM_INTERN && threadIdx.x == 0) {
                *err = 1000 + SOUTH;
            }
            if (jN <= jS) SYNC();
            t = g.btp[NORTH - 1];
            if (t == BM_WALL1 || t == BM_WALL2 || t == BM_INLET) {
                PAR(i, iW + 1, iE) P(i, jN + 1) = BP(NORTH, i) + P(i, jN);
            } else if (t == BM_OUTLT1 || t == BM_OUTLT2) {
                PAR(i, iW + 1, iE) P(i, jN + 1) = dTwo * BP(NORTH, i) - P(i, jN);
            } else if (t != BM_INTERN && threadIdx.x == 0) {
                *err = 1000 + NORTH;
            }
            SYNC();
        }
#undef P
#undef BP
}

// `reps` applications of VelBoundCond (workgroup 0) and of PresBoundCond
// (workgroup 1; none without p) in one launch: the two write separate fields.
// A one-region table is loaded once for all applications.
template <typename T>
__global__ __launch_bounds__(BC_THREADS) void k_fills(Regions R, int ld, T *__restrict__ u, T *__restrict__ v,
                                                      T *__restrict__ p, int outflow_only, int reps,
                                                      int *__restrict__ err, const int *stop) {
    if (stop && *stop) return;
    __shared__ BcRegion g;
    __shared__ T st[2][BC_CH];
    const bool one = R.ni == 1 && R.nj == 1;
    if (one) bc_load(R, 1, 1, g);
    for (int k = 0; k < reps; k++) {
        if (blockIdx.x == 0 && u)
            vel_fill<T>(R, ld, u, v, outflow_only, err, g, st, one);
        else
            pres_fill<T>(R, ld, p, err, g, one);
    }
}

template <typename T>
void launch_vel_bc(const Regions &R, int ld, T *u, T *v, bool outflow_only, int *err, hipStream_t s,
                   const int *stop) {
    hipLaunchKernelGGL(k_fills<T>, dim3(1), dim3(BC_THREADS), 0, s, R, ld, u, v, (T *)nullptr, outflow_only ? 1 : 0, 1,
                       err, stop);
}
template <typename T>
void launch_pres_bc(const Regions &R, int ld, T *p, int *err, hipStream_t s) {
    hipLaunchKernelGGL(k_fills<T>, dim3(1), dim3(BC_THREADS), 0, s, R, ld, (T *)nullptr, (T *)nullptr, p, 0, 1, err,
                       (const int *)nullptr);
}
void launch_fills(const Regions &R, int ld, double *u, double *v, double *p, int reps, int *err, hipStream_t s) {
    hipLaunchKernelGGL(k_fills<double>, dim3(2), dim3(BC_THREADS), 0, s, R, ld, u, v, p, 0, reps, err,
                       (const int *)nullptr);
}
template void launch_vel_bc<double>(const Regions &, int, double *, double *, bool, int *, hipStream_t,
                                    const int *);
template void launch_vel_bc<float>(const Regions &, int, float *, float *, bool, int *, hipStream_t, const int *);
template void launch_pres_bc<double>(const Regions &, int, double *, int *, hipStream_t);

}  // namespace wd2
