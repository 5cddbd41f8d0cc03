// FP64 E-step of DA-GTM on gfx950: two streaming passes over the K x N
// distance matrix, which is never stored.
//
// Both passes take their cross term y.t from v_mfma_f64_16x16x4_f64: the FP64
// matrix and vector rates of this chip are the same (and the two share one
// pipe), but a matrix instruction needs one operand pair from LDS per 2048
// flops, where a 4 x 4 register tile of FMAs needs eight per 32.  An FP64 MFMA
// rounds like a chain of FMAs in the order of its inner index (measured: no
// bit differs), so every sum over d or n below is one FMA chain in ascending
// order, whatever the tiling; the results do not depend on it.
//
// Pass 1 (k_e1_f64): an online log-sum-exp per point, in sixteen
// slices: slice t holds the centres k = t (mod 16) in ascending order, its
// running maximum moving at most once per 64 centres.  The slices are merged
// in order at the end.  Output per point: x_max, log S2 (pass-2 normaliser),
// log g and log h, and their sums per workgroup.
//
// Pass 2 (k_e2_f64): one workgroup per (64-centre tile, N chunk) recomputes
// the same distances, forms R = exp((x - x_max)/temp - log S2) in registers
// and accumulates G = sum_n R and RT = sum_n R t_n, writing one partial per
// chunk; k_reduce_parts sums the chunks in a fixed order.
//
// The math restates mpicomm.c:316-414 (resp) and mpicomm.c:463-500 (qual):
// x = d * (-beta/2), E = exp(x), P = E^(1/temp), R = P / colsum(P), with
// exp underflow (x < -745.13) giving exactly 0 and an all-zero column
// falling back to R = 1/K (h = K; g = K in EM mode only).
#include <algorithm>
#include <cmath>
#include <limits>
#include <type_traits>

#include "dg_internal.h"

namespace {

typedef double d2 __attribute__((ext_vector_type(2)));
typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int NT = 256;   // threads per workgroup (4 waves of 64)
constexpr int TP = 64;    // points: a pass-2 chunk is a whole number of these
constexpr int DC = 16;    // d-chunk of the cross-term loop
constexpr int DCP = DC + 2;  // its row stride in LDS: 8 rows cover the banks once

// D[i][j] += sum_q A[i][q] B[q][j], 16 x 16 x 4: lane l holds A[l % 16][l / 16],
// B[l / 16][l % 16] and, in element r, D[4 r + l / 16][l % 16].
__device__ __forceinline__ d4 mfma64(double a, double b, d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Rows in LDS keep every eight d in the order 0 4 1 5 2 6 3 7, so that a lane
// finds its elements of two successive MFMAs (d and d + 4) in one 16-byte read.
__device__ __forceinline__ constexpr int dpos(int d) {
    return (d & ~7) + 2 * (d & 3) + ((d >> 2) & 1);
}
__device__ __forceinline__ void put_pair(double *row, int d, d2 v) {   // d even: d and d + 1
    row[dpos(d)] = v.x;
    row[dpos(d) + 2] = v.y;
}

// Exponent x = d * (-beta/2) with d = (-2 s + |y|^2) + |t|^2 in the
// reference's dgemm + dger order (comm.c:590-619); -inf when exp underflows
// (and for the +inf |y|^2 that stands for a centre past the end).
__device__ __forceinline__ double exponent(double s, double yk, double tn, double nbh) {
    const double d = fma(-2.0, s, yk) + tn;
    const double x = d * nbh;
    return (x > kExpUnderflowX) ? x : -INFINITY;
}

// ---------------------------------------------------------------- pass 1
// One slice's online sums: m its running maximum, s1 and s2 the sums of
// exp(x - m) and exp((x - m) / temp).
struct Slice {
    double m = -INFINITY, s1 = 0.0, s2 = 0.0;
    // a new running maximum rescales the sums
    __device__ __forceinline__ void raise(double top, double it, int two) {
        if (top > m) {
            const double r = m - top;
            s1 *= exp(r);
            if (two) s2 *= exp(r * it);
            m = top;
        }
    }
};

// Below this a term cannot change a sum: each slice's sums are at least 1 (its
// maximum's own term), and e^-37 is less than half a unit in their last place.
constexpr double kNoTerm = -37.0;

// log g and log h of a point from its merged sums (mpicomm.c:382-390 for a
// zero column), stored with the normalisers; returns its share of the sums
struct PointOut {
    double *pm, *pl, *logg, *logh;
    double it, logK;
    int two, isDA;
    __device__ __forceinline__ void put(long n, double M, double S1, double S2, double &lg,
                                        double &lh, double &zc) const {
        double l2 = 0.0;
        if (M == -INFINITY) {
            lg = isDA ? -INFINITY : logK;
            lh = logK;
            zc = 1.0;
        } else {
            const double l1 = log(S1);
            l2 = two ? log(S2) : l1;
            lg = M + l1;
            lh = M * it + l2;
        }
        pm[n] = M;
        pl[n] = l2;
        logg[n] = lg;
        logh[n] = lh;
    }
};

// the workgroup's sums of log g, log h and zero columns to partLog
__device__ __forceinline__ void put_logs(double lg, double lh, double zc,
                                         double (*sm)[NT / 64], double *__restrict__ partLog) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        lg += __shfl_xor(lg, o);
        lh += __shfl_xor(lh, o);
        zc += __shfl_xor(zc, o);
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { sm[0][w] = lg; sm[1][w] = lh; sm[2][w] = zc; }
    __syncthreads();
    if (threadIdx.x < 3) {
        const double *s = sm[threadIdx.x];
        partLog[3 * (long)blockIdx.x + threadIdx.x] = (s[0] + s[1]) + (s[2] + s[3]);
    }
}

// ---- the cross terms of 64 points with the centres
// 64 points (16 per wave) against the centres in tiles of 128: a wave holds
// eight 16 x 16 accumulators, whose lane (j, g) has point j and rows 4 r + g.
// Row i of accumulator a of tile t is centre 128 t + 16 a + i (S = 1), or one of
// the 64 centres from 64 (8 t + a) on, the (16 (i / 4) + 4 q + i % 4)-th (S = 4,
// q4 = 4 q).  The operands pass through LDS in 16-wide d chunks, double
// buffered, the next chunk's loads in registers while one is multiplied.
// close(t, yt, na, acc) gets each finished tile of [t0, t1): yt its |y|^2 in LDS
// (+inf past the last centre), na how many accumulators hold a centre.  With xs
// (S = 1), xs[t & 1][q] holds the centres' X[k][q], 0 for q >= L and past the end.
constexpr int P1 = 64, C1 = 128, RW = C1 / 16;

struct CrossSmem {
    double Ts[2][P1 * DCP];
    double Ys[2][C1 * DCP];
    double ys[2][C1];
};

// the centre in a row of a tile
template <int S>
__device__ __forceinline__ int centre_of(int t, int row, int q4) {
    const int i = row & 15;
    return t * C1 * S + (row >> 4) * 16 * S + (S == 1 ? i : 16 * (i >> 2) + q4 + (i & 3));
}

template <int S, typename Close>
__device__ __forceinline__ void cross_sweep(
    CrossSmem &sm, const double *__restrict__ T, long N, const double *__restrict__ Y,
    const double *__restrict__ yy, int K, int D, int ld, long n0, int t0, int t1, int q4,
    Close &&close, const double *__restrict__ X = nullptr, int L = 0,
    double (*xs)[3][C1] = nullptr) {
    constexpr int LT = P1 / 32, LY = C1 / 32;      // 16-byte loads per thread and chunk
    constexpr int CT = C1 * S;                     // centres from one tile to the next
    constexpr int CA = 16 * S;                     // from one accumulator to the next
    const int tid = threadIdx.x, l = tid & 63, w = tid >> 6, j = l & 15, g = l >> 4;
    const int nch = (D + DC - 1) / DC;                // d chunks per centre tile
    const int last8 = (D - (nch - 1) * DC + 7) / 8;   // 8-wide steps of the last one
    // staging: eight threads per row of a chunk, 16 bytes each; rows past the
    // end repeat the last one (|y|^2 = +inf there, and no point is stored).
    // Scalar bases and 32-bit lane offsets that change once per tile at most: a
    // vector instruction here holds up the FP64 matrix instructions of its SIMD.
    const int sr = tid >> 3, sp = tid & 7;
    const double *Tw = T + n0 * ld;
    unsigned ot[LT], oy[LY];
#pragma unroll
    for (int i = 0; i < LT; ++i) ot[i] = (unsigned)(min(n0 + sr + 32 * i, N - 1) - n0) * ld + 2 * sp;
    auto at = [](const double *base, unsigned o) { return *(const d2 *)(base + o); };
    d2 rt[LT], ry[LY];
    double ryy = INFINITY, rx[3] = {0.0, 0.0, 0.0};
    auto load = [&](int t, int q) {                    // tile t, d chunk q
        if (q == 0) {
#pragma unroll
            for (int i = 0; i < LY; ++i)
                oy[i] = (unsigned)min(centre_of<S>(t, sr + 32 * i, q4), K - 1) * ld + 2 * sp;
            if (tid < C1) {
                const int k = centre_of<S>(t, tid, q4);
                ryy = (k < K) ? yy[k] : INFINITY;
                if (xs)
#pragma unroll
                    for (int x = 0; x < 3; ++x) rx[x] = (k < K && x < L) ? X[(long)k * L + x] : 0.0;
            }
        }
#pragma unroll
        for (int i = 0; i < LT; ++i) rt[i] = at(Tw + q * DC, ot[i]);
#pragma unroll
        for (int i = 0; i < LY; ++i) ry[i] = at(Y + q * DC, oy[i]);
    };
    auto store = [&](int b, int t, int q) {
#pragma unroll
        for (int i = 0; i < LT; ++i) put_pair(&sm.Ts[b][(sr + 32 * i) * DCP], 2 * sp, rt[i]);
#pragma unroll
        for (int i = 0; i < LY; ++i) put_pair(&sm.Ys[b][(sr + 32 * i) * DCP], 2 * sp, ry[i]);
        if (q == 0 && tid < C1) {
            sm.ys[t & 1][tid] = ryy;
            if (xs)
#pragma unroll
                for (int x = 0; x < 3; ++x) xs[t & 1][x][tid] = rx[x];
        }
    };
    if (t0 >= t1) return;
    d4 acc[RW];
    load(t0, 0);
    store(0, t0, 0);
    __syncthreads();
    int b = 0;
    for (int t = t0; t < t1; ++t) {
        const int na = min(RW, (K - t * CT + CA - 1) / CA);
#pragma unroll
        for (int a = 0; a < RW; ++a) acc[a] = d4{0.0, 0.0, 0.0, 0.0};
        for (int q = 0; q < nch; ++q, b ^= 1) {
            const int tq = (q + 1 < nch) ? t : t + 1, qn = (q + 1 < nch) ? q + 1 : 0;
            const bool more = tq < t1;
            if (more) load(tq, qn);
            const int steps = (q + 1 < nch) ? DC / 8 : last8;
            for (int s = 0; s < steps; ++s) {
                const double *yr = &sm.Ys[b][j * DCP + 8 * s + 2 * g];
                const d2 bv = *(const d2 *)&sm.Ts[b][(16 * w + j) * DCP + 8 * s + 2 * g];
                if (na == RW) {
                    // the centre rows' operands are read one step ahead of
                    // their MFMAs (the sched_barrier keeps them there)
                    d2 av = *(const d2 *)yr;
#pragma unroll
                    for (int a = 0; a < RW; ++a) {
                        const d2 an = *(const d2 *)(yr + 16 * (a + 1 < RW ? a + 1 : a) * DCP);
                        __builtin_amdgcn_sched_barrier(0);
                        acc[a] = mfma64(av.x, bv.x, acc[a]);
                        acc[a] = mfma64(av.y, bv.y, acc[a]);
                        av = an;
                    }
                } else {
#pragma unroll
                    for (int a = 0; a < RW - 1; ++a)
                        if (a < na) {
                            const d2 av = *(const d2 *)(yr + 16 * a * DCP);
                            acc[a] = mfma64(av.x, bv.x, acc[a]);
                            acc[a] = mfma64(av.y, bv.y, acc[a]);
                        }
                }
            }
            if (more) store(b ^ 1, tq, qn);
            // (before the barrier: the next tile's |y|^2 goes to the other
            // half of ys, the one after it only past this barrier)
            if (q + 1 == nch) {
                // (opaque: else what close derives from t is computed, and kept
                // in registers, before the chunk loop)
                int tc = t;
                asm volatile("" : "+s"(tc));
                close(tc, sm.ys[tc & 1], na, acc);
            }
            __syncthreads();
        }
    }
}

// Pass 1.  S = 1: the workgroup takes every centre, its lanes keep slices
// 4 r + g, and it finishes its points.  S = 4: it takes the slices 4 q .. 4 q + 3,
// q = blockIdx.y, its lanes keep slice 4 q + g, and k_e1_merge finishes the points.
// Bound by the FP64 pipe, which the matrix instructions, the exponentials (two
// per element away from temperature 1, left out where no term of a wave can
// change its sum) and the exponents share: at N = 10^6, D = 166, K = 8000,
// temperature 2, 62 ms, of which the 2 K N D flops take 35 at the pipe's measured
// 77.7 TFLOP/s (4 x 4 register tiles of FMAs: 132 ms, their eight LDS reads per
// 16 FMAs cost twice the pipe's time).  N = 1640, K = 5832: 0.26 ms (3.27).
template <int S>
__global__ __launch_bounds__(NT, 2) void k_e1_f64(
    const double *__restrict__ T, const double *__restrict__ tt, long N,
    const double *__restrict__ Y, const double *__restrict__ yy, int K, int D, int ld, double nbh,
    PointOut po, double *__restrict__ partLog, double *__restrict__ part) {
    __shared__ __attribute__((aligned(16))) CrossSmem cs;
    __shared__ double sm[3][NT / 64];
    const int tid = threadIdx.x, l = tid & 63, w = tid >> 6, j = l & 15, g = l >> 4;
    const int q4 = 4 * blockIdx.y;
    const long n0 = (long)blockIdx.x * P1, n = n0 + 16 * w + j;
    const double it = po.it;
    const int two = po.two;
    const double tn = (n < N) ? tt[n] : 0.0;
    Slice sl[S == 1 ? 4 : 1];
    // slice s takes in the four centres it has of 64: exponents x of rows
    // row0 + step i
    auto take = [&](Slice &s, double (&x)[4], const double *yt, int row0, int step) {
        double top = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x[i] = exponent(x[i], yt[row0 + step * i + g], tn, nbh);
            top = fmax(top, x[i]);
        }
        s.raise(top, it, two);
        // (-inf: nothing in the slice yet; its x are all -inf too)
        const double m = (s.m == -INFINITY) ? 0.0 : s.m;
        const double near = top - m;
        if (__any(near > kNoTerm)) {
#pragma unroll
            for (int i = 0; i < 4; ++i) s.s1 += exp(x[i] - m);
        }
        if (two && __any(near * it > kNoTerm)) {
#pragma unroll
            for (int i = 0; i < 4; ++i) s.s2 += exp((x[i] - m) * it);
        }
    };
    cross_sweep<S>(cs, T, N, Y, yy, K, D, ld, n0, 0, (K + C1 * S - 1) / (C1 * S), q4,
                   [&](int, const double *yt, int na, d4 (&acc)[RW]) {
        if (S == 1) {
#pragma unroll
            for (int h = 0; h < RW; h += 4)
                if (h < na)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        double x[4] = {acc[h][r], acc[h + 1][r], acc[h + 2][r], acc[h + 3][r]};
                        take(sl[S == 1 ? r : 0], x, yt, 16 * h + 4 * r, 16);
                    }
        } else {
#pragma unroll
            for (int a = 0; a < RW; ++a)
                if (a < na) {
                    double x[4] = {acc[a][0], acc[a][1], acc[a][2], acc[a][3]};
                    take(sl[0], x, yt, 16 * a, 4);
                }
        }
    });
    if (S == 4) {
        if (n < N) {
            double *o = part + (long)(q4 + g) * 3 * N + n;
            o[0] = sl[0].m;
            o[N] = sl[0].s1;
            o[2 * N] = sl[0].s2;
        }
        return;
    }
    // merge the point's sixteen slices in order (slice 4 r + g is element r of
    // lane j + 16 g); every lane of the point gets the same sums
    double M = -INFINITY;
#pragma unroll
    for (int r = 0; r < (S == 1 ? 4 : 1); ++r) M = fmax(M, sl[r].m);
    M = fmax(M, __shfl_xor(M, 16));
    M = fmax(M, __shfl_xor(M, 32));
    double S1 = 0.0, S2 = 0.0;
#pragma unroll
    for (int r = 0; r < (S == 1 ? 4 : 1); ++r) {
        const double d = (M == -INFINITY) ? 0.0 : sl[r].m - M;
        const double f1 = exp(d), f2 = two ? exp(d * it) : 0.0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            S1 = fma(__shfl(sl[r].s1, j + 16 * q), __shfl(f1, j + 16 * q), S1);
            if (two) S2 = fma(__shfl(sl[r].s2, j + 16 * q), __shfl(f2, j + 16 * q), S2);
        }
    }
    double lg = 0.0, lh = 0.0, zc = 0.0;
    if (g == 0 && n < N) po.put(n, M, S1, S2, lg, lh, zc);
    put_logs(lg, lh, zc, sm, partLog);
}

// Finishes the points whose slices part holds: slice t's m, s1 and s2 of point
// n at part[(3 t + 0 .. 2) N + n].
__global__ __launch_bounds__(NT) void k_e1_merge(const double *__restrict__ part, long N,
                                                 PointOut po, double *__restrict__ partLog) {
    __shared__ double sm[3][NT / 64];
    const long n = (long)blockIdx.x * NT + threadIdx.x;
    double lg = 0.0, lh = 0.0, zc = 0.0;
    if (n < N) {
        double m[16], s1[16], s2[16], M = -INFINITY, S1 = 0.0, S2 = 0.0;
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            m[t] = part[3L * t * N + n];
            s1[t] = part[(3L * t + 1) * N + n];
            s2[t] = part[(3L * t + 2) * N + n];
        }
#pragma unroll
        for (int t = 0; t < 16; ++t) M = fmax(M, m[t]);
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            const double d = (M == -INFINITY) ? 0.0 : m[t] - M;
            S1 = fma(s1[t], exp(d), S1);
            if (po.two) S2 = fma(s2[t], exp(d * po.it), S2);
        }
        po.put(n, M, S1, S2, lg, lh, zc);
    }
    put_logs(lg, lh, zc, sm, partLog);
}

// ---------------------------------------------------------------- pass 2
// A workgroup owns 64 centres, 16 per wave with their rows in registers as
// the B operand, and one chunk of points, streamed in 16-point tiles through
// a double-buffered LDS copy (rows at ld + 4: both operand reads below touch
// every bank equally).  C[n][k] = T Y^T leaves R in the accumulator layout,
// which is the A operand layout of RT[k][d] += sum_n R[k][n] T[n][d] with the
// points of element r, 4 r .. 4 r + 3, as the inner index: R goes from the
// exponential straight into the second product.
// Bound by the FP64 pipe: at N = 10^6, D = 166, K = 8000, 105 ms, of which the
// 4 K N D flops (D padded to 168 and 176) take 71 at 77.7 TFLOP/s, the
// exponentials about 8 and the last, part-filled round of workgroups 12 (428 ms
// with FMAs from LDS; half as much again without the read-ahead and the split
// staging below).  Two workgroups share a CU: 256 registers hold the centre
// operand and the accumulators up to D = 192, with one half of the next tile's
// loads in flight.
template <int DB>
__global__ __launch_bounds__(NT, 2) void k_e2_f64(
    const double *__restrict__ T, const double *__restrict__ tt, long N,
    const double *__restrict__ Y, const double *__restrict__ yy, int K, int D,
    double nbh, double it, double invK,
    const double *__restrict__ pm, const double *__restrict__ pl, long chunk,
    double *__restrict__ partRT, double *__restrict__ partG) {
    constexpr int ld = 16 * DB, LD = ld + 4;
    constexpr int NL = (DB + 1) / 2;               // 16-byte loads per thread and tile
    __shared__ __attribute__((aligned(16))) double Tb[2][16 * LD];
    __shared__ double pt[2][3][16];                // |t|^2, x_max and log S2 of the tile

    const int tid = threadIdx.x, l = tid & 63, w = tid >> 6, j = l & 15, g = l >> 4;
    const int kw = blockIdx.x * 64 + 16 * w, k = kw + j;
    const long nb = (long)blockIdx.y * chunk;
    const long ne = (nb + chunk < N) ? nb + chunk : N;
    // (the last 8-wide step of d is all padding when D <= ld - 8)
    const bool full = D > ld - 8;

    d2 yb[2 * DB];
#pragma unroll
    for (int s = 0; s < 2 * DB; ++s)
        yb[s] = (k < K) ? d2{Y[(long)k * ld + 8 * s + g], Y[(long)k * ld + 8 * s + 4 + g]} : d2{0.0, 0.0};
    const double yk = (k < K) ? yy[k] : INFINITY;
    const double rz = (k < K) ? invK : 0.0;        // R of a zero column
    d4 acc[DB];
#pragma unroll
    for (int b = 0; b < DB; ++b) acc[b] = d4{0.0, 0.0, 0.0, 0.0};
    double gs[4] = {0.0, 0.0, 0.0, 0.0};           // points n = 4 r + g (mod 16)

    // staging: sixteen threads per row, 16 bytes each per load; rows past the
    // end are zero, and so is their R
    const int sr = tid >> 4, sp = tid & 15;
    const bool tail = DB % 2 == 0 || sp < 8;       // the last load of an odd row: half of them
    constexpr int H = (NL + 1) / 2;                // loads in flight: half a tile's
    d2 rt[H];
    double rp;
    const double *psrc = tt;                       // threads 0 .. 47: one of a point's three values
    if (sr == 1) psrc = pm;
    if (sr >= 2) psrc = pl;
    const double pend = (sr == 1) ? INFINITY : 0.0;   // past the end: x_max = +inf, so R = 0
    auto half_load = [&](int h, long n0) {
        // (a scalar base and a 32-bit lane offset, as in cross_sweep)
        const double *base = T + n0 * ld;
        const unsigned o = (unsigned)min(sr, (int)min(ne - 1 - n0, 15L)) * ld + 2 * sp;
#pragma unroll
        for (int i = 0; i < H; ++i) {
            const int f = h * H + i;
            if (f < NL && (f < NL - 1 || tail)) rt[i] = *(const d2 *)(base + 32 * f + o);
        }
        if (h == 0) {
            const double v = psrc[min(n0 + sp, ne - 1)];
            rp = (n0 + sp < ne) ? v : pend;
        }
    };
    auto half_store = [&](int h, int b, long n0) {
        if (n0 + sr >= ne) {
#pragma unroll
            for (int i = 0; i < H; ++i) rt[i] = d2{0.0, 0.0};
        }
#pragma unroll
        for (int i = 0; i < H; ++i) {
            const int f = h * H + i;
            if (f < NL && (f < NL - 1 || tail)) put_pair(&Tb[b][sr * LD + 32 * f], 2 * sp, rt[i]);
        }
        if (h == 0 && tid < 48) pt[b][sr][sp] = rp;
    };
    if (nb < ne) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            half_load(h, nb);
            half_store(h, 0, nb);
        }
    }
    __syncthreads();
    int b = 0;
    // (the sched_barriers keep each operand's LDS read one step ahead of the
    // MFMAs that use it; the compiler otherwise puts it right before them and
    // waits out its latency every two MFMAs)
    for (long n0 = nb; n0 < ne; n0 += 16, b ^= 1) {
        const bool more = n0 + 16 < ne;
        if (more) half_load(0, n0 + 16);
        d4 c = {0.0, 0.0, 0.0, 0.0};
        const double *ta = &Tb[b][j * LD + 2 * g];
        d2 a = *(const d2 *)ta;
#pragma unroll
        for (int s = 0; s < 2 * DB; ++s) {
            const d2 an = *(const d2 *)(ta + 8 * (s + 1 < 2 * DB ? s + 1 : s));
            __builtin_amdgcn_sched_barrier(0);
            if (s < 2 * DB - 1 || full) {
                c = mfma64(a.x, yb[s].x, c);
                c = mfma64(a.y, yb[s].y, c);
            }
            a = an;
        }
        if (more) {
            half_store(0, b ^ 1, n0 + 16);
            half_load(1, n0 + 16);
        }
        double R[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int n = 4 * r + g;
            const double x = exponent(c[r], yk, pt[b][0][n], nbh);
            R[r] = exp((x - pt[b][1][n]) * it - pt[b][2][n]);
            asm volatile("" : "+v"(R[r]));         // (no branch around the exponential)
        }
        const double *tb = &Tb[b][g * LD + dpos(j)];
        double t0 = tb[0], t1 = tb[DB > 1 ? 16 : 4 * LD];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            R[r] = (pt[b][1][4 * r + g] == -INFINITY) ? rz : R[r];
            gs[r] += R[r];
        }
#pragma unroll
        for (int i = 0; i < 4 * DB; ++i) {
            const int i2 = (i + 2 < 4 * DB) ? i + 2 : i;
            const double t2 = tb[(i2 / DB) * 4 * LD + 16 * (i2 % DB)];
            __builtin_amdgcn_sched_barrier(0);
            acc[i % DB] = mfma64(R[i / DB], t0, acc[i % DB]);
            t0 = t1;
            t1 = t2;
        }
        if (more) half_store(1, b ^ 1, n0 + 16);
        __syncthreads();
    }
    const long ch = blockIdx.y;
#pragma unroll
    for (int q = 0; q < DB; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int kk = kw + 4 * r + g, d = 16 * q + j;
            if (kk < K && d < D) partRT[(ch * K + kk) * D + d] = acc[q][r];
        }
    double G = 0.0;                                // the sixteen classes in order
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int q = 0; q < 4; ++q) G += __shfl(gs[r], j + 16 * q);
    if (g == 0 && k < K) partG[ch * K + k] = G;
}

// RT and G from the chunk partials, summed in chunk order with eight loads in
// flight; the last workgroup sums pass 1's partial log sums into scal and the host's
// copy of it (pinned: a copy of 64 bytes after the step took 5 us) instead.
__global__ __launch_bounds__(256) void k_reduce_parts(
    const double *__restrict__ partRT, const double *__restrict__ partG, int NC, int K, int D,
    double *__restrict__ RT, double *__restrict__ G, const double *__restrict__ partLog, long nlog,
    double *__restrict__ scal, double *__restrict__ hscal) {
    if (blockIdx.x == gridDim.x - 1) {
        __shared__ double s[3][256];
        double a[3] = {0.0, 0.0, 0.0};
        for (long i = threadIdx.x; i < nlog; i += 256)
            for (int x = 0; x < 3; ++x) a[x] += partLog[3 * i + x];
        for (int x = 0; x < 3; ++x) s[x][threadIdx.x] = a[x];
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            if ((int)threadIdx.x < o)
                for (int x = 0; x < 3; ++x) s[x][threadIdx.x] += s[x][threadIdx.x + o];
            __syncthreads();
        }
        if (threadIdx.x == 0) {
            scal[kScalSumLogG] = hscal[kScalSumLogG] = s[0][0];
            scal[kScalSumLogH] = hscal[kScalSumLogH] = s[1][0];
            scal[kScalNZero] = hscal[kScalNZero] = s[2][0];
        }
        return;
    }
    const long KD = (long)K * D;
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    auto sum = [&](const double *p, long stride) {
        double s = 0.0;
        int c = 0;
        for (; c + 8 <= NC; c += 8) {
            double v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = p[(c + u) * stride];
#pragma unroll
            for (int u = 0; u < 8; ++u) s += v[u];
        }
        for (; c < NC; ++c) s += p[c * stride];
        return s;
    };
    if (i < KD) RT[i] = sum(partRT + i, KD);
    else if (i < KD + K) G[i - KD] = sum(partG + (i - KD), K);
}

// ---------------------------------------------------------------- dense R, MAP
// R_kn of the centres from k0 = 0 .. K - 1 (K, Y and yy of a range of them) from
// the pass-1 normalisers, to R[k ldR + n].  Workgroup (point tile, range of
// tiles_per centre tiles).  Bound by the FP64 pipe for D beyond a few, else by
// the 8 K N bytes it writes: N = 6007, D = 12, K = 900 in 22 us (one thread per
// element over D, its row uncoalesced: 289).
__global__ __launch_bounds__(NT, 2) void k_resp_dense(
    const double *__restrict__ T, const double *__restrict__ tt, long N,
    const double *__restrict__ Y, const double *__restrict__ yy, int K, int D, int ld, double nbh,
    double it, double invK, const double *__restrict__ pm, const double *__restrict__ pl,
    int tiles_per, double *__restrict__ R, long ldR) {
    __shared__ __attribute__((aligned(16))) CrossSmem cs;
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6, j = l & 15, g = l >> 4;
    const long n0 = (long)blockIdx.x * P1, n = n0 + 16 * w + j, nn = min(n, N - 1);
    const int t0 = blockIdx.y * tiles_per, t1 = min((K + C1 - 1) / C1, t0 + tiles_per);
    const double tn = tt[nn], m = pm[nn], ls = pl[nn];
    const long off = g * ldR + 16 * w + j;
    cross_sweep<1>(cs, T, N, Y, yy, K, D, ld, n0, t0, t1, 0,
                   [&](int t, const double *yt, int na, d4 (&acc)[RW]) {
#pragma unroll
        for (int a = 0; a < RW; ++a)
            if (a < na) {
                double v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const double x = exponent(acc[a][r], yt[16 * a + 4 * r + g], tn, nbh);
                    v[r] = exp((x - m) * it - ls);
                    asm volatile("" : "+v"(v[r]));             // (no branch around it)
                }
                const int k = t * C1 + 16 * a;
                double *row = R + (long)k * ldR + n0;          // (wave-uniform)
#pragma unroll
                for (int r = 0; r < 4; ++r, row += 4 * ldR)
                    if (k + 4 * r + g < K && n < N) row[off] = (m == -INFINITY) ? invK : v[r];
            }
    });
}

// MAP in one pass: per point the online sums of p = exp((x - m) / temp) and of
// p X[k][l] (L <= 3) over a range of centres; k_map_merge makes M = sum p X /
// sum p of them.  No normaliser is needed beforehand, so a projection costs one
// pass over the K x N distances in either precision.  part[(5 range + f) N + n]:
// m, sum p, and the three sums.  FP64 pipe: 2 K N D flops, K N exponentials.
// N = 30011, D = 166, K = 8000: 1.95 ms (one thread per point over all centres,
// after two FP64 passes for its normaliser: 497).
__global__ __launch_bounds__(NT, 2) void k_map_f64(
    const double *__restrict__ T, const double *__restrict__ tt, long N,
    const double *__restrict__ Y, const double *__restrict__ yy, int K, int D, int ld, double nbh,
    double it, int tiles_per, const double *__restrict__ X, int L, double *__restrict__ part) {
    __shared__ __attribute__((aligned(16))) CrossSmem cs;
    __shared__ double xs[2][3][C1];
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6, j = l & 15, g = l >> 4;
    const long n0 = (long)blockIdx.x * P1, n = n0 + 16 * w + j;
    const int t0 = blockIdx.y * tiles_per, t1 = min((K + C1 - 1) / C1, t0 + tiles_per);
    const double tn = tt[min(n, N - 1)];
    double m = -INFINITY, s = 0.0, ax[3] = {0.0, 0.0, 0.0};
    auto take = [&](int t, int a, const double *yt, const d4 &c) {
        double x[4], top = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            x[r] = exponent(c[r], yt[16 * a + 4 * r + g], tn, nbh);
            top = fmax(top, x[r]);
        }
        if (top > m) {                             // new running max: rescale the sums
            const double f = exp((m - top) * it);
            s *= f;
#pragma unroll
            for (int q = 0; q < 3; ++q) ax[q] *= f;
            m = top;
        }
        const double ms = (m == -INFINITY) ? 0.0 : m;
        // (below this every p is exactly 0; a higher bound would drop a small p whose
        // coordinate is large)
        if (__any((top - ms) * it > kExpUnderflowX)) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const double v = exp((x[r] - ms) * it);
                s += v;
#pragma unroll
                for (int q = 0; q < 3; ++q) ax[q] = fma(v, xs[t & 1][q][16 * a + 4 * r + g], ax[q]);
            }
        }
    };
    cross_sweep<1>(cs, T, N, Y, yy, K, D, ld, n0, t0, t1, 0,
                   [&](int t, const double *yt, int na, d4 (&acc)[RW]) {
#pragma unroll
        for (int a = 0; a < RW; ++a)
            if (a < na) take(t, a, yt, acc[a]);
    }, X, L, xs);
    // the four lanes j, j + 16, j + 32, j + 48 hold the same point
    double M = fmax(m, __shfl_xor(m, 16));
    M = fmax(M, __shfl_xor(M, 32));
    const double f = exp((M == -INFINITY) ? 0.0 : (m - M) * it);
    double v[4] = {s * f, ax[0] * f, ax[1] * f, ax[2] * f};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        v[q] += __shfl_xor(v[q], 16);
        v[q] += __shfl_xor(v[q], 32);
    }
    if (g == 0 && n < N) {
        double *o = part + 5L * blockIdx.y * N + n;
        o[0] = M;
#pragma unroll
        for (int q = 0; q < 4; ++q) o[(q + 1) * N] = v[q];
    }
}

__global__ __launch_bounds__(NT) void k_map_merge(const double *__restrict__ part, int ranges,
                                                  long N, double it, int K, double invK,
                                                  const double *__restrict__ X, int L,
                                                  double *__restrict__ M) {
    const long n = (long)blockIdx.x * NT + threadIdx.x;
    if (n >= N) return;
    double top = -INFINITY, v[4] = {0.0, 0.0, 0.0, 0.0};
    for (int c = 0; c < ranges; ++c) top = fmax(top, part[5L * c * N + n]);
    if (top == -INFINITY) {                        // zero column: R = 1/K
        v[0] = 1.0;
        for (int k = 0; k < K; ++k)
            for (int q = 0; q < L; ++q) v[q + 1] = fma(invK, X[(long)k * L + q], v[q + 1]);
    } else {
        for (int c = 0; c < ranges; ++c) {
            const double *p = part + 5L * c * N + n;
            const double f = exp((p[0] - top) * it);
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = fma(p[(q + 1) * N], f, v[q]);
        }
    }
    for (int q = 0; q < L; ++q) M[n * L + q] = v[q + 1] / v[0];
}

// f(std::integral_constant<int, DB>) for DB = db in 1 .. 12, false otherwise
template <typename F>
bool with_db(int db, F &&f) {
    switch (db) {
#define DG_DB(V) case V: f(std::integral_constant<int, V>{}); return true;
        DG_DB(1) DG_DB(2) DG_DB(3) DG_DB(4) DG_DB(5) DG_DB(6)
        DG_DB(7) DG_DB(8) DG_DB(9) DG_DB(10) DG_DB(11) DG_DB(12)
#undef DG_DB
        default: return false;
    }
}

// ---------------------------------------------------------------- critical temperature
// Responsibility-weighted second moments of the data centred on one centre,
// S1 = sum_n r_kn x x^T and S2 = sum_n r_kn^2 x x^T with x = t_n - y_k (the
// 2 S1 and -S2 of mpicomm.c:580-597), r_kn = R[k N + n] of k_resp_dense.  One
// workgroup per (tile pair of the lower triangle, centre, N chunk); a tile is
// 16 RB wide and its waves take sixteen points in turn, straight from global
// memory: a lane's operands of four points are r x and r^2 x of its row and x of
// its column.  The waves' sums are added in order, and the chunk's partial goes
// to part[((chunk * KB + kb) * 2 + s) * D * D + a * D + b].
// Bound by the FP64 pipe: 4 flops for each entry, point and centre.  N = 5003,
// D = 32, K = 400: 143 us, and 14 for R (4 x 4 tiles of FMAs from LDS and one thread per
// point for its R: 1107 us).  D = 166: 69 % of the pipe's rate.
// diag: the pair's columns are its rows, and its upper tiles are not wanted.
template <int RB, bool diag>
__device__ __forceinline__ void moments_body(
    double (*red)[2 * RB * RB][256], const int ti, const int tj, const double *__restrict__ T, long N,
    const double *__restrict__ Y, int D, int ld, const double *__restrict__ R, long chunk,
    double *__restrict__ part) {
    const int tid = threadIdx.x, l = tid & 63, w = tid >> 6, j = l & 15, g = l >> 4;
    const long kb = blockIdx.y;
    const long n0 = (long)blockIdx.z * chunk, n1 = min(N, n0 + chunk);
    // (columns past the row's end repeat its last one; their results are not stored)
    int ca[RB], cb[RB];
    double ya[RB], yb[RB];
#pragma unroll
    for (int x = 0; x < RB; ++x) {
        ca[x] = min(16 * (RB * ti + x) + j, ld - 1);
        cb[x] = min(16 * (RB * tj + x) + j, ld - 1);
        ya[x] = Y[kb * ld + ca[x]];
        yb[x] = Y[kb * ld + cb[x]];
    }
    const double *r = R + kb * N;
    d4 s1[RB][RB], s2[RB][RB];
#pragma unroll
    for (int x = 0; x < RB; ++x)
#pragma unroll
        for (int y = 0; y < RB; ++y) s1[x][y] = s2[x][y] = d4{0.0, 0.0, 0.0, 0.0};
    double rv[4], ta[4][RB], tb[4][RB];    // the next sixteen points: four quads
    auto load = [&](long base) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const long n = base + 4 * u + g, nc = min(n, n1 - 1);
            const double v = r[nc];
            rv[u] = (n < n1) ? v : 0.0;
#pragma unroll
            for (int x = 0; x < RB; ++x) {
                ta[u][x] = T[nc * ld + ca[x]];
                if (!diag) tb[u][x] = T[nc * ld + cb[x]];
            }
        }
    };
    long base = n0 + 16 * w;
    if (base < n1) load(base);
    for (; base < n1; base += 64) {
        double a1[4][RB], a2[4][RB], bx[4][RB];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int x = 0; x < RB; ++x) {
                const double xa = ta[u][x] - ya[x];
                a1[u][x] = xa * rv[u];
                a2[u][x] = a1[u][x] * rv[u];
                bx[u][x] = diag ? xa : tb[u][x] - yb[x];
            }
        if (base + 64 < n1) load(base + 64);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int x = 0; x < RB; ++x)
#pragma unroll
                for (int y = 0; y < RB; ++y)
                    if (y <= x || !diag) {
                        s1[x][y] = mfma64(a1[u][x], bx[u][y], s1[x][y]);
                        s2[x][y] = mfma64(a2[u][x], bx[u][y], s2[x][y]);
                    }
    }
#pragma unroll
    for (int x = 0; x < RB; ++x)
#pragma unroll
        for (int y = 0; y < RB; ++y)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                red[w][2 * (RB * x + y)][64 * q + l] = s1[x][y][q];
                red[w][2 * (RB * x + y) + 1][64 * q + l] = s2[x][y][q];
            }
    __syncthreads();
    const long DD = (long)D * D;
    double *o = part + ((long)blockIdx.z * gridDim.y + kb) * 2 * DD;
#pragma unroll
    for (int x = 0; x < RB; ++x)
#pragma unroll
        for (int y = 0; y < RB; ++y) {
            // thread tid: element tid / 64 of lane tid % 64
            const int a = 16 * (RB * ti + x) + 4 * w + g, b = 16 * (RB * tj + y) + j;
            if (a < D && b < D && (y <= x || !diag))
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const int f = 2 * (RB * x + y) + s;
                    o[s * DD + (long)a * D + b] =
                        ((red[0][f][tid] + red[1][f][tid]) + red[2][f][tid]) + red[3][f][tid];
                }
        }
}

template <int RB>
__global__ __launch_bounds__(NT, 2) void k_ctemp_moments(
    const double *__restrict__ T, long N, const double *__restrict__ Y, int D, int ld,
    const double *__restrict__ R, long chunk, double *__restrict__ part) {
    __shared__ double red[4][2 * RB * RB][256];
    int p = blockIdx.x, ti = 0;            // lower-triangle pair p -> (ti >= tj)
    while (p > ti) { p -= ti + 1; ++ti; }
    if (p == ti) moments_body<RB, true>(red, ti, p, T, N, Y, D, ld, R, chunk, part);
    else moments_body<RB, false>(red, ti, p, T, N, Y, D, ld, R, chunk, part);
}

// out[i] = sum over the nc chunk partials of part[c * len + i], in chunk order.
__global__ void k_sum_chunks(const double *__restrict__ part, int nc, long len,
                             double *__restrict__ out) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= len) return;
    double s = 0.0;
    for (int c = 0; c < nc; ++c) s += part[(long)c * len + i];
    out[i] = s;
}

// x summed over the wave, the same bits in every lane: rotations within rows of
// sixteen, then the rows (row_ror and the row swaps cost a few cycles where a
// shuffle through LDS takes over a hundred).
template <int ROR>
__device__ __forceinline__ double add_rotated(double x) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
    const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)u, 0x120 + ROR, 0xf, 0xf, false);
    const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), 0x120 + ROR, 0xf, 0xf, false);
    return x + __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ double wave_sum(double x) {
    x = add_rotated<8>(x);
    x = add_rotated<4>(x);
    x = add_rotated<2>(x);
    x = add_rotated<1>(x);
    // (each half of a swapped pair is a row's sum: their sum is order-free)
    auto swapped = [](double y, bool rows32) {
        const unsigned long long u = __builtin_bit_cast(unsigned long long, y);
        unsigned a[2], b[2];
        for (int h = 0; h < 2; ++h) {
            const unsigned t = h ? (unsigned)(u >> 32) : (unsigned)u;
            const auto r = rows32 ? __builtin_amdgcn_permlane32_swap(t, t, false, false)
                                  : __builtin_amdgcn_permlane16_swap(t, t, false, false);
            a[h] = r[0];
            b[h] = r[1];
        }
        return __builtin_bit_cast(double, ((unsigned long long)a[1] << 32) | a[0]) +
               __builtin_bit_cast(double, ((unsigned long long)b[1] << 32) | b[0]);
    };
    x = swapped(x, false);
    return swapped(x, true);
}

// The eigenvalue of one centre's S that the critical temperature takes.  Workgroup
// (kb, part): of A = 2 S1 or 2 S1 - 2 S2, n x n, the largest eigenvalue below
// limit, and 0 in the place of those at or above it (comm.c:2149-2161):
// val[2 kb + part] = their maximum.  A's lower triangle is packed in LDS, scaled by
// a power of two to a largest entry in [1, 2) (a centre's weight, and so its S, may
// be any double down to the smallest, and the sums below square the entries), reduced to tridiagonal form by Householder reflections (Golub & Van Loan,
// Matrix Computations, 4th ed., 8.3.1), and the one eigenvalue wanted is found by
// Sturm counts (8.4.1) at 64 points of the interval at a time, one per lane.
// Bound by the chain of reflections (two reductions and a matrix-vector product
// each).  800 matrices of n = 32 in 125 us (178 with shuffled sums, rows loaded one
// at a time and updated one after the other), 1216 of n = 166 in 5.4 ms (6.1); on 16 host
// threads, with S to copy there first, the search took 2.7 ms longer at n = 32
// and 0.2 s at n = 166.
__global__ __launch_bounds__(256) void k_ctemp_eig(const double *__restrict__ S, int n,
                                                   const double *__restrict__ limit,
                                                   const double *__restrict__ asked,
                                                   double *__restrict__ val) {
    extern __shared__ double A[];                  // n (n + 1) / 2, then v, p, d, e of n each
    __shared__ double red[4];
    const int tid = threadIdx.x, nt = blockDim.x, l = tid & 63, w = tid >> 6;
    const long kb = blockIdx.x;
    const int sub = blockIdx.y;
    if (asked[kb] == 0.0) return;                  // a centre without weight
    double *v = A + n * (n + 1) / 2, *p = v + n, *d = p + n, *e = d + n;
    const double *S1 = S + kb * 2 * n * n, *S2 = S1 + (long)n * n;
    auto at = [&](int i, int j) -> double & { return A[i * (i + 1) / 2 + j]; };   // j <= i
    auto sum = [&](double x) {                     // over the workgroup, in every thread
        x = wave_sum(x);
        if (nt == 64) return x;
        __syncthreads();                           // the last sum's readers are done
        if (l == 0) red[w] = x;
        __syncthreads();
        return (red[0] + red[1]) + (red[2] + red[3]);
    };
    double top = 0.0;                              // the largest |entry| (NaN left out)
    for (int e0 = tid; e0 < n * n; e0 += 8 * nt) {  // (eight elements' loads in flight)
        double a[8], b[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int e = min(e0 + u * nt, n * n - 1);
            a[u] = S1[e];
            b[u] = sub ? S2[e] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int e = e0 + u * nt, i = e / n, j = e - i * n;
            const double x = sub ? 2.0 * a[u] - 2.0 * b[u] : 2.0 * a[u];
            if (i < n && j <= i) {
                at(i, j) = x;
                top = fmax(top, fabs(x));
            }
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) top = fmax(top, __shfl_xor(top, o));
    if (l == 0) red[w] = top;
    __syncthreads();
    for (int x = 0; x < nt / 64; ++x) top = fmax(top, red[x]);
    const int ex = (top > 0.0 && top < INFINITY) ? ilogb(top) : 0;   // 2^ex <= top < 2^(ex + 1)
    const double lim = ldexp(limit[kb], -ex);
    for (int x = tid; x < n * (n + 1) / 2; x += nt) A[x] = ldexp(A[x], -ex);
    __syncthreads();
    for (int k = 0; k + 2 < n; ++k) {
        // the reflection that annihilates A[k + 2 .., k]: v = x - alpha e1
        double s = 0.0;
        for (int i = k + 2 + tid; i < n; i += nt) s = fma(at(i, k), at(i, k), s);
        s = sum(s);
        const double x0 = at(k + 1, k), norm = sqrt(fma(x0, x0, s));
        const double alpha = (x0 > 0.0) ? -norm : norm, v0 = x0 - alpha, vv = fma(v0, v0, s);
        if (tid == 0) {
            d[k] = at(k, k);
            e[k] = alpha;
        }
        if (vv == 0.0 || s == 0.0) {               // (uniform) nothing to annihilate
            if (tid == 0) e[k] = x0;
            continue;
        }
        for (int i = k + 1 + tid; i < n; i += nt) v[i] = (i == k + 1) ? v0 : at(i, k);
        __syncthreads();
        // p = 2 A v / vv, then p -= (v.p / vv) v, and A -= v p^T + p v^T; a row of the
        // product to a thread (n <= nt): a column's elements, T(i) + j of row i, are
        // in different banks
        const int i = k + 1 + tid;
        double vi = 0.0, pi = 0.0;
        if (i < n) {
            double q[4] = {0.0, 0.0, 0.0, 0.0};    // (four chains, eight reads in flight)
            auto elem = [&](int j) { return A[j <= i ? i * (i + 1) / 2 + j : j * (j + 1) / 2 + i]; };
            int j = k + 1;
            for (; j + 8 <= n; j += 8) {
                double x[8], y[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) { x[u] = elem(j + u); y[u] = v[j + u]; }
#pragma unroll
                for (int u = 0; u < 8; ++u) q[u & 3] = fma(x[u], y[u], q[u & 3]);
            }
            for (; j < n; ++j) q[0] = fma(elem(j), v[j], q[0]);
            pi = 2.0 * ((q[0] + q[1]) + (q[2] + q[3])) / vv;
            vi = v[i];
        }
        const double c = sum(vi * pi) / vv;
        pi -= c * vi;
        if (i < n) p[i] = pi;
        __syncthreads();
        // the update: a row to a lane where one wave has them all (n = 32: 125 us, 154
        // with lanes along the rows, one row after the other; n = 64: 359 and 473),
        // else lanes along the rows (n = 166: 5.4 ms, and 6.4)
        if (nt == 64) {
            if (i < n) {
                double *row = A + i * (i + 1) / 2;
                int j = k + 1;
                for (; j + 8 <= n && __any(j <= i); j += 8) {
                    double x[8], y[8], z[8];
    #pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        x[u] = row[min(j + u, i)];
                        y[u] = p[j + u];
                        z[u] = v[j + u];
                    }
    #pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (j + u <= i) row[j + u] = x[u] - (vi * y[u] + pi * z[u]);
                }
                for (; j <= i; ++j) row[j] -= vi * p[j] + pi * v[j];
            }
        } else {
            for (int r = k + 1 + w; r < n; r += nt / 64) {
                const double vr = v[r], pr = p[r];
                for (int j = k + 1 + l; j <= r; j += 64) at(r, j) -= vr * p[j] + pr * v[j];
            }
        }
        __syncthreads();
    }
    if (tid == 0) {
        if (n > 1) {
            d[n - 2] = at(n - 2, n - 2);
            e[n - 2] = at(n - 1, n - 2);
        }
        d[n - 1] = at(n - 1, n - 1);
        e[n - 1] = 0.0;
    }
    __syncthreads();
    if (w > 0) return;
    // Gershgorin bounds, and the smallest pivot a count may divide by
    double lo = INFINITY, hi = -INFINITY;
    bool finite = true;
    for (int i = l; i < n; i += 64) {
        const double r = fabs(e[i]) + (i ? fabs(e[i - 1]) : 0.0);
        finite = finite && fabs(d[i]) + r < INFINITY;
        lo = fmin(lo, d[i] - r);
        hi = fmax(hi, d[i] + r);
    }
    if (!__all(finite)) {                          // NaN or infinite data: no eigenvalues
        if (l == 0) val[2 * kb + sub] = NAN;
        return;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        lo = fmin(lo, __shfl_xor(lo, o));
        hi = fmax(hi, __shfl_xor(hi, o));
    }
    const double tnorm = fmax(fabs(lo), fabs(hi));
    const double pivmin = fmax(2.3e-308, 2.3e-16 * 2.3e-16 * tnorm);
    auto below = [&](double x) {                   // eigenvalues below x
        int c = 0;
        double q = 1.0, e2 = 0.0;
        for (int i = 0; i < n; ++i) {
            q = d[i] - x - e2 / q;
            if (fabs(q) < pivmin) q = -pivmin;
            c += (q < 0.0) ? 1 : 0;
            e2 = e[i] * e[i];
        }
        return c;
    };
    const double pad = 4.0 * 2.3e-16 * n * tnorm + pivmin;
    const int idx = below(lim);                    // the idx-th smallest is the largest below
    double best = (idx < n) ? 0.0 : -INFINITY;
    double a = lo - pad, b = fmin(hi + pad, lim);
    if (idx > 0 && (idx == n || b > 0.0)) {
        if (idx < n && a < 0.0 && below(0.0) >= idx) {
            // none between 0 and the limit: 0 stands
        } else {
            for (int it = 0; it < 64; ++it) {
                const double h = (b - a) / 65.0, x = a + h * (l + 1);
                const unsigned long long up = __ballot(below(x) >= idx);
                const int f = up ? __builtin_ctzll(up) : 64;
                const double na = (f > 0) ? a + h * f : a, nb = (f < 64) ? a + h * (f + 1) : b;
                const bool done = !(nb - na < b - a) || nb - na <= 2.3e-16 * fmax(fabs(na), fabs(nb));
                a = na;
                b = nb;
                if (done) break;
            }
            best = fmax(best, 0.5 * (a + b));
        }
    }
    if (l == 0) val[2 * kb + sub] = ldexp(best, ex);
}

}  // namespace

// 1 / temp.  For an infinite temperature the smallest positive number: the same
// share for every centre whose exponent is finite, none for the others, where 0
// times their -inf would be NaN.
static double inv_temp(bool isDA, double temp) {
    return isDA ? std::max(1.0 / temp, std::numeric_limits<double>::denorm_min()) : 1.0;
}

// Pass 1 splits a point tile's slices over four workgroups up to 64 x 16 points
// per CU: below that, whole point tiles are too few to spread evenly (N = 10^5,
// D = 166, K = 8000: 6.4 ms split, 7.2 whole; N = 260000, K = 1000: 2.17 and
// 2.25).  Above it the slices' states (384 bytes a point) are not worth their
// way through memory.
constexpr long kSplitPoints = 64L * 16 * 256;
size_t dg_pass1_part(long N) { return N < kSplitPoints ? (size_t)48 * N : 0; }
long dg_pass1_wgs(long N) { return N < kSplitPoints ? (N + NT - 1) / NT : (N + P1 - 1) / P1; }

int dg_pass1_fp64(dg_ctx *c, int isDA, double temp) {
    const double nbh = -c->beta / 2.0;
    const double it = inv_temp(isDA, temp);
    const PointOut po{c->pm, c->pl, c->logg, c->logh, it, log((double)c->K),
                      (isDA && it != 1.0) ? 1 : 0, isDA};
    const unsigned tiles = (unsigned)((c->N + P1 - 1) / P1);
    auto go = [&](auto kernel, dim3 grid) {
        hipLaunchKernelGGL(kernel, grid, dim3(NT), 0, c->stream, c->T64, c->tt, c->N, c->Y64, c->yy,
                           c->K, c->D, c->ldt, nbh, po, c->partLog64, c->partRT);
    };
    if (c->N < kSplitPoints) {
        go(k_e1_f64<4>, dim3(tiles, 4));
        DG_HIP(c, hipGetLastError());
        hipLaunchKernelGGL(k_e1_merge, dim3((unsigned)dg_pass1_wgs(c->N)), dim3(NT), 0, c->stream,
                           c->partRT, c->N, po, c->partLog64);
    } else {
        go(k_e1_f64<1>, dim3(tiles));
    }
    DG_HIP(c, hipGetLastError());
    return DG_OK;
}

static int dg_pass2_fp64(dg_ctx *c, int isDA, double temp) {
    const double nbh = -c->beta / 2.0;
    const double it = inv_temp(isDA, temp);
    const long tiles = (c->N + TP - 1) / TP;
    const long chunk = ((tiles + c->NC - 1) / c->NC) * TP;
    const dim3 grid((unsigned)((c->K + 63) / 64), (unsigned)c->NC);
    auto go = [&](auto db) {
        hipLaunchKernelGGL(k_e2_f64<decltype(db)::value>, grid, dim3(NT), 0, c->stream, c->T64, c->tt,
                           c->N, c->Y64, c->yy, c->K, c->D, nbh, it, 1.0 / c->K, c->pm, c->pl,
                           chunk, c->partRT, c->partG);
    };
    if (!with_db(c->ldt / 16, go)) return dg_fail(c, DG_EINVAL, "FP64 path supports D <= 192");
    DG_HIP(c, hipGetLastError());
    return DG_OK;
}

int dg_stats_fp64(dg_ctx *c, int isDA, double temp) {
    int rc;
    if ((rc = dg_pass2_fp64(c, isDA, temp))) return rc;
    if (c->timing) DG_HIP(c, hipEventRecord(c->ev[2], c->stream));
    const long nred = (long)c->K * c->D + c->K;
    hipLaunchKernelGGL(k_reduce_parts, dim3((unsigned)((nred + 255) / 256 + 1)), dim3(256), 0,
                       c->stream, c->partRT, c->partG, c->NC, c->K, c->D, c->RT, c->G,
                       c->partLog64, dg_pass1_wgs(c->N), c->scal, c->m_scal);
    DG_HIP(c, hipGetLastError());
    return DG_OK;
}

int dg_estep_fp64(dg_ctx *c, int isDA, double temp) {
    int rc;
    if (c->timing) DG_HIP(c, hipEventRecord(c->ev[0], c->stream));
    if ((rc = dg_pass1_fp64(c, isDA, temp))) return rc;
    if (c->timing) DG_HIP(c, hipEventRecord(c->ev[1], c->stream));
    return dg_stats_fp64(c, isDA, temp);
}

// k_resp_dense and k_map_f64 split the centre tiles into ranges until there are
// about 2048 workgroups (two are resident on each of 256 CUs)
struct Ranges {
    int tiles_per, count;
};
static Ranges centre_ranges(long N, int K) {
    const long pt = (N + P1 - 1) / P1, ct = (K + C1 - 1) / C1;
    const long want = std::max(1L, std::min(ct, (2048 + pt - 1) / pt));
    const int per = (int)((ct + want - 1) / want);
    return {per, (int)((ct + per - 1) / per)};
}

size_t dg_map_part(long N, int K) { return (size_t)5 * N * centre_ranges(N, K).count; }

int dg_resp_dense_fp64(dg_ctx *c, double *dR, long ldR) {
    const double it = inv_temp(c->last_isDA, c->last_temp);
    const Ranges r = centre_ranges(c->N, c->K);
    hipLaunchKernelGGL(k_resp_dense, dim3((unsigned)((c->N + P1 - 1) / P1), (unsigned)r.count),
                       dim3(NT), 0, c->stream, c->T64, c->tt, c->N, c->Y64, c->yy, c->K, c->D,
                       c->ldt, -c->beta / 2.0, it, 1.0 / c->K, c->pm, c->pl, r.tiles_per, dR, ldR);
    DG_HIP(c, hipGetLastError());
    return DG_OK;
}

int dg_ctemp_fp64(dg_ctx *c, int k0, int KB, const DgCtempPlan &p, const double *dLimit,
                  double *buf, double *dVal) {
    const double it = inv_temp(c->last_isDA, c->last_temp);
    const int D = c->D;
    double *R = buf, *part = buf + p.r_len, *S = p.nc > 1 ? part + p.s_len * p.nc : part;
    // R of these centres, then their moments, then the eigenvalues
    const Ranges r = centre_ranges(c->N, KB);
    hipLaunchKernelGGL(k_resp_dense, dim3((unsigned)((c->N + P1 - 1) / P1), (unsigned)r.count),
                       dim3(NT), 0, c->stream, c->T64, c->tt, c->N, c->Y64 + (long)k0 * c->ldt,
                       c->yy + k0, KB, D, c->ldt, -c->beta / 2.0, it, 1.0 / c->K, c->pm, c->pl,
                       r.tiles_per, R, c->N);
    DG_HIP(c, hipGetLastError());
    const long chunk = ((c->N + (long)p.nc * 64 - 1) / ((long)p.nc * 64)) * 64;
    const dim3 grid((unsigned)p.pairs, (unsigned)KB, (unsigned)p.nc);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(NT), 0, c->stream, c->T64, c->N,
                           c->Y64 + (long)k0 * c->ldt, D, c->ldt, R, chunk, part);
    };
    if (D <= 16) go(k_ctemp_moments<1>);
    else go(k_ctemp_moments<2>);
    DG_HIP(c, hipGetLastError());
    if (p.nc > 1) {
        const long len = (long)KB * 2 * D * D;
        hipLaunchKernelGGL(k_sum_chunks, dim3((unsigned)((len + 255) / 256)), dim3(256), 0,
                           c->stream, part, p.nc, len, S);
        DG_HIP(c, hipGetLastError());
    }
    // (a wave is enough for 64 rows; 154368 bytes of LDS at D = 192)
    const size_t lds = ((size_t)D * (D + 1) / 2 + 4 * D) * sizeof(double);
    hipLaunchKernelGGL(k_ctemp_eig, dim3((unsigned)KB, 2), dim3(D <= 64 ? 64 : 256), lds, c->stream, S,
                       D, dLimit + 2 * (long)k0, dLimit + 2 * (long)k0 + KB, dVal + 2 * (long)k0);
    DG_HIP(c, hipGetLastError());
    return DG_OK;
}

// At most 256 MB of S1 and S2 and 1 GB of R to a batch of centres; about 2048
// workgroups of moments, with 256 points to each at least.
DgCtempPlan dg_ctemp_plan(const dg_ctx *c) {
    DgCtempPlan p;
    const long D = c->D, DD = D * D;
    p.KB = (int)std::max(1L, std::min({(long)c->K, (1L << 25) / (2 * DD), (1L << 27) / c->N}));
    const long nt = D <= 16 ? 1 : (D + 31) / 32;
    p.pairs = (int)(nt * (nt + 1) / 2);
    const long want = (2048 + (long)p.pairs * p.KB - 1) / ((long)p.pairs * p.KB);
    p.nc = (int)std::max(1L, std::min({want, 64L, (c->N + 255) / 256}));
    p.r_len = (size_t)p.KB * c->N;
    p.s_len = (size_t)p.KB * 2 * DD;
    return p;
}

int dg_map_fp64(dg_ctx *c, const double *dX, int L, double *dM) {
    const double it = inv_temp(c->last_isDA, c->last_temp);
    const Ranges r = centre_ranges(c->N, c->K);
    hipLaunchKernelGGL(k_map_f64, dim3((unsigned)((c->N + P1 - 1) / P1), (unsigned)r.count), dim3(NT),
                       0, c->stream, c->T64, c->tt, c->N, c->Y64, c->yy, c->K, c->D, c->ldt,
                       -c->beta / 2.0, it, r.tiles_per, dX, L, c->partRT);
    DG_HIP(c, hipGetLastError());
    hipLaunchKernelGGL(k_map_merge, dim3((unsigned)((c->N + NT - 1) / NT)), dim3(NT), 0, c->stream,
                       c->partRT, r.count, c->N, it, c->K, 1.0 / c->K, dX, L, dM);
    DG_HIP(c, hipGetLastError());
    return DG_OK;
}
