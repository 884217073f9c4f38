// wd2_trid.hpp -- row helpers shared by the tridiagonal chain kernels: the
// solvers of k_trid.hip (chains in memory) and the fused q-l iteration of
// k_ql.hip (both splits of a window of chain rows in one workgroup).
#pragma once

#include <type_traits>

#include "wd2_dev.hpp"
#include "wd2_launch.hpp"

namespace wd2 {

constexpr int TR_T = 256;   // threads per workgroup
constexpr int TR_S = 8;     // rows per thread
constexpr int TR_R = TR_T * TR_S;
constexpr int TR_P = TR_S + 1;   // padded LDS stride of a thread's rows

__device__ inline bool same(double x, double y) { return dbits(x) == dbits(y); }
__device__ inline bool same(float x, float y) { return __float_as_uint(x) == __float_as_uint(y); }

// One forward row.  kind: 0 interior, 1 chain start, 2 chain end.
template <typename T>
__device__ inline void fwd_row(int kind, T a, T d, T c, T b, T dnext, T cpv, T bpv, T &cpk, T &bpk) {
    if (kind == 1) {
        cpk = c / dnext;
        bpk = b / d;
    } else {
        const T dp = d - (a * cpv);
        cpk = (kind == 2) ? T(0) : c / dp;
        bpk = (b - a * bpv) / dp;
    }
}

// Position r of row k in its chain, and that chain's length Lk.
__device__ inline long chain_pos(const Chains &cs, long k, long &Lk) {
    if (k < cs.n1) {
        Lk = cs.L1;
        return k % cs.L1;
    }
    Lk = cs.L2;
    return (k - cs.n1) % cs.L2;
}
// (r, Lk) of row k + 1 from those of row k, and of row k - 1.
__device__ inline void chain_up(const Chains &cs, long k, long &r, long &Lk) {
    if (++r == Lk) {
        r = 0;
        if (k + 1 == cs.n1) Lk = cs.L2;
    }
}
__device__ inline void chain_down(const Chains &cs, long k, long &r, long &Lk) {
    if (r == 0) {
        if (k == cs.n1) Lk = cs.L1;
        r = Lk - 1;
    } else {
        r--;
    }
}
__device__ inline int kind_at(long r, long Lk) { return r == 0 ? 1 : (r == Lk - 1 ? 2 : 0); }
__device__ inline bool chain_end(long r, long Lk) { return r == Lk - 1 && r != 0; }
__device__ inline int row_kind(long k, const Chains &cs) {
    long Lk;
    const long r = chain_pos(cs, k, Lk);
    return kind_at(r, Lk);
}

// A thread's TR_S consecutive rows are read and written as 16-byte vectors
// (chain arrays start 128-byte aligned and a segment starts at a multiple of
// TR_S rows): a wavefront covers one contiguous span, every load in flight at
// once.  A partial last segment goes row by row.
template <typename T>
__device__ inline void seg_load(const T *__restrict__ G, long seg0, int len, T (&r)[TR_S]) {
    if (len == TR_S) {
        constexpr int V = 16 / sizeof(T);
        using V4 = typename std::conditional<sizeof(T) == 4, float4, double2>::type;
        const V4 *g = reinterpret_cast<const V4 *>(G + seg0);
#pragma unroll
        for (int q = 0; q < TR_S / V; q++) {
            const V4 v = g[q];
            const T *e = reinterpret_cast<const T *>(&v);
#pragma unroll
            for (int u = 0; u < V; u++) r[q * V + u] = e[u];
        }
    } else {
#pragma unroll
        for (int q = 0; q < TR_S; q++) r[q] = q < len ? G[seg0 + q] : T(0);
    }
}
template <typename T>
__device__ inline void seg_store(T *__restrict__ G, long seg0, int len, const T (&r)[TR_S]) {
    if (len == TR_S) {
        constexpr int V = 16 / sizeof(T);
        using V4 = typename std::conditional<sizeof(T) == 4, float4, double2>::type;
        V4 *g = reinterpret_cast<V4 *>(G + seg0);
#pragma unroll
        for (int q = 0; q < TR_S / V; q++) {
            V4 v;
            T *e = reinterpret_cast<T *>(&v);
#pragma unroll
            for (int u = 0; u < V; u++) e[u] = r[q * V + u];
            g[q] = v;
        }
    } else {
#pragma unroll
        for (int q = 0; q < TR_S; q++)
            if (q < len) G[seg0 + q] = r[q];
    }
}


// Kinds of the TR_S rows from seg0 on, two bits per row (one 64-bit modulo).
__device__ inline unsigned seg_kinds(long seg0, const Chains &cs) {
    long Lk;
    long r = chain_pos(cs, seg0, Lk);
    unsigned m = 0;
#pragma unroll
    for (int s = 0; s < TR_S; s++) {
        m |= (unsigned)kind_at(r, Lk) << (2 * s);
        chain_up(cs, seg0 + s, r, Lk);
    }
    return m;
}
#define SKIND(m, s) ((int)(((m) >> (2 * (s))) & 3u))

// Bit queries on a workgroup's per-lane flags (TR_T bits in 64-bit words).
__device__ inline int lowest_bit_in(const unsigned long long *m, int lo, int hi) {   // -1 if none
    for (int w = lo >> 6; lo <= hi && w <= (hi >> 6); w++) {
        unsigned long long x = m[w];
        if (w == (lo >> 6)) x &= ~0ull << (lo & 63);
        if (w == (hi >> 6) && (hi & 63) != 63) x &= (1ull << ((hi & 63) + 1)) - 1;
        if (x) return (w << 6) + __ffsll((long long)x) - 1;
    }
    return -1;
}
__device__ inline int highest_clear_at_or_below(const unsigned long long *m, int hi) {   // -1 if none
    for (int w = hi >> 6; w >= 0; w--) {
        unsigned long long x = ~m[w];
        if (w == (hi >> 6) && (hi & 63) != 63) x &= (1ull << ((hi & 63) + 1)) - 1;
        if (x) return (w << 6) + 63 - __clzll((long long)x);
    }
    return -1;
}
__device__ inline int highest_bit_in(const unsigned long long *m, int lo, int hi) {   // -1 if none
    for (int w = hi >> 6; lo <= hi && w >= (lo >> 6); w--) {
        unsigned long long x = m[w];
        if (w == (lo >> 6)) x &= ~0ull << (lo & 63);
        if (w == (hi >> 6) && (hi & 63) != 63) x &= (1ull << ((hi & 63) + 1)) - 1;
        if (x) return (w << 6) + 63 - __clzll((long long)x);
    }
    return -1;
}
__device__ inline int lowest_clear_at_or_above(const unsigned long long *m, int lo, int n) {   // n if none
    for (int w = lo >> 6; w < n / 64; w++) {
        unsigned long long x = ~m[w];
        if (w == (lo >> 6)) x &= ~0ull << (lo & 63);
        if (x) return (w << 6) + __ffsll((long long)x) - 1;
    }
    return n;
}
__device__ inline bool bit_at(const unsigned long long *m, int i) { return (m[i >> 6] >> (i & 63)) & 1ull; }

// Rounds after which a workgroup still changing looks for rounding cycles
// (the shortcut is described in k_trid.hip).
constexpr int TR_ACC = 3;

// Window shapes of the FP32 window solver (described in k_trid.hip).
constexpr int TW_S = 8, TW_H = 64;
template <int TW_T>
struct TwShape {
    static constexpr int N = TW_T * TW_S, O = N - 2 * TW_H, M = 2 * TW_T;
};
constexpr float TW_DOM = 0.9f;
constexpr float TW_EPS = 0x1p-48f;   // PCR stops once every coupling is below this share of its diagonal
// A window is usable if its rows couple to those TW_H rows away by at most
// this share of their diagonal, which PCR has at hand: its level h leaves the
// interface rows, two a segment of TW_S, coupled to those 2 h interface rows
// away.  A kept row's error is then at most 2^-24 of what was dropped, as one
// FP32 rounding.  The rows' ratio (|a| + |c|) / |d| alone does not tell: at
// 0.89 a value still weighs 0.61^64 = 2e-14 after 64 rows coupled evenly to
// both sides, but 0.89^64 = 6e-4 after 64 upwinded rows, coupled to one.
constexpr float TW_REACH = 0x1p-24f;
constexpr int TW_REACH_LEVEL = TW_H / TW_S;
static_assert((TW_REACH_LEVEL & (TW_REACH_LEVEL - 1)) == 0, "a PCR level spans the halo");

// Hardware reciprocal (1 ulp) for the window solver, which need not round
// like the reference.
__device__ inline float wrcp(float x) { return __builtin_amdgcn_rcpf(x); }

}  // namespace wd2
