// FP64 M-step and the scalar reductions of DA-GTM on gfx950.
//
//   A  = FI^T diag(G) FI  (scale_by_row, then dgemm)  dagtm.cxx:1729-1738
//   B  = FI^T (R T) = FI^T RT                dagtm.cxx:1746-1761 (same product,
//                                            associated the other way)
//   W  = (A + lambda/beta I)^-1 B            Cholesky (dagtm_solve2 in the
//                                            reference, comm.c:1299-1348)
//   Y  = FI W                                dagtm.cxx:1769-1770
//   beta = N D / sum_kn R_kn |y_k - t_n|^2   mpicomm.c:276-302, evaluated as
//          sum_n |t_n|^2 - 2 sum_k y_k.RT_k + sum_k G_k |y_k|^2
//          (exact because every column of R sums to one, mpicomm.c:382-391)
#include <cmath>
#include <type_traits>
#include <utility>

#include "dg_internal.h"

namespace {

// out[r] = sum_d X[r][d]^2, sequential in d (the ddot loops of comm.c:604-618)
__global__ void k_rownorm(const double *__restrict__ X, long rows, int ld, int D,
                          double *__restrict__ out) {
    const long r = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    // eight loads in flight, then their FMAs in order
    double s = 0.0;
    int d = 0;
    for (; d + 8 <= D; d += 8) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = X[r * ld + d + u];
#pragma unroll
        for (int u = 0; u < 8; ++u) s = fma(v[u], v[u], s);
    }
    for (; d < D; ++d) {
        const double v = X[r * ld + d];
        s = fma(v, v, s);
    }
    out[r] = s;
}

// Deterministic block-tree sum of a vector into scal[slot].  Single workgroup, FP64.
__global__ __launch_bounds__(1024) void k_sum(const double *__restrict__ a, long n,
                                              double *__restrict__ scal, int slot) {
    __shared__ double sa[1024];
    double x = 0.0;
    for (long i = threadIdx.x; i < n; i += 1024) x += a[i];
    sa[threadIdx.x] = x;
    __syncthreads();
    for (int s = 512; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sa[threadIdx.x] += sa[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) scal[slot] = sa[0];
}

// tr(A0) into *out, summed by the first wave; every thread of the workgroup
// calls it (it ends with a barrier).  Only the jitter retries need it.
__device__ void block_trace(const double *__restrict__ A0, int n, double *out) {
    const int tid = threadIdx.x;
    if (tid < 64) {
        double s = 0.0;
        for (int i = tid; i < n; i += 64) s += A0[(long)i * n + i];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
        if (tid == 0) *out = s;
    }
    __syncthreads();
}

// Cholesky solve of (A0 + (ridge + jitter) I) W = B in one workgroup (the
// batched M-step's path for M + 1 > 126; a single instance uses the blocked
// kernels below), the factor built in place in A (right-looking; each entry
// receives its updates in the same column order as a left-looking loop).  On a
// non-positive pivot the factorisation restarts with jitter 1e-13 tr/n,
// growing x10 per retry, at most 8 retries.  scal[kScalSolveOK] = 1 on
// success, scal[kScalJitter] = the jitter used.
__device__ __forceinline__ void k_chol_solve_body(
    const double *__restrict__ A0, double *__restrict__ A, int n, double ridge,
    const double *__restrict__ B, int nrhs, double *__restrict__ Wout, double *__restrict__ scal) {
    __shared__ int fail;
    __shared__ double tr;
    const int tid = threadIdx.x, nt = blockDim.x;
    double jit = 0.0;
    int ok = 0;
    for (int attempt = 0; attempt < 9 && !ok; ++attempt) {
        if (attempt == 1) {
            block_trace(A0, n, &tr);
            jit = 1e-13 * tr / n;
        } else if (attempt > 1) {
            jit *= 10.0;
        }
        for (long e = tid; e < (long)n * n; e += nt) {
            const long i = e / n, j = e % n;
            A[e] = A0[e] + ((i == j) ? ridge + jit : 0.0);
        }
        if (tid == 0) fail = 0;
        __syncthreads();
        for (int j = 0; j < n; ++j) {
            if (tid == 0) {
                const double p = A[(long)j * n + j];
                if (!(p > 0.0)) fail = 1;
                else A[(long)j * n + j] = sqrt(p);
            }
            __syncthreads();
            if (fail) break;
            const double ljj = A[(long)j * n + j];
            for (int i = j + 1 + tid; i < n; i += nt) A[(long)i * n + j] /= ljj;
            __syncthreads();
            // trailing update of the lower triangle, columns j+1..n-1
            const int m = n - j - 1;
            const long pairs = (long)m * (m + 1) / 2;
            for (long e = tid; e < pairs; e += nt) {
                // e -> (r, c) with 0 <= c <= r < m
                long r = (long)((sqrt(8.0 * (double)e + 1.0) - 1.0) * 0.5);
                while ((r + 1) * (r + 2) / 2 <= e) ++r;
                while (r * (r + 1) / 2 > e) --r;
                const long cc = e - r * (r + 1) / 2;
                const long i = j + 1 + r, k = j + 1 + cc;
                A[i * n + k] = fma(-A[i * n + j], A[k * n + j], A[i * n + k]);
            }
            __syncthreads();
        }
        ok = !fail;
        __syncthreads();
    }
    if (tid == 0) {
        scal[kScalJitter] = jit;
        scal[kScalSolveOK] = ok ? 1.0 : 0.0;
    }
    if (!ok) return;
    // forward L y = b and backward L^T x = y, one right-hand side per thread
    for (int c = tid; c < nrhs; c += nt) {
        for (int i = 0; i < n; ++i) {
            double s = B[(long)i * nrhs + c];
            for (int p = 0; p < i; ++p) s = fma(-A[(long)i * n + p], Wout[(long)p * nrhs + c], s);
            Wout[(long)i * nrhs + c] = s / A[(long)i * n + i];
        }
        for (int i = n - 1; i >= 0; --i) {
            double s = Wout[(long)i * nrhs + c];
            for (int p = i + 1; p < n; ++p) s = fma(-A[(long)p * n + i], Wout[(long)p * nrhs + c], s);
            Wout[(long)i * nrhs + c] = s / A[(long)i * n + i];
        }
    }
}

// tr(A0) into scal[kScalJitter] (the retries' jitter scale)
__global__ __launch_bounds__(64) void k_bc_trace(const double *__restrict__ A0, int n,
                                                 double *__restrict__ scal) {
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 64) s += A0[(long)i * n + i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (threadIdx.x == 0) scal[kScalJitter] = s;
}

typedef double d4 __attribute__((ext_vector_type(4)));

// D[i][j] += sum_q A[i][q] B[q][j], 16 x 16 x 4: lane l holds A[l % 16][l / 16],
// B[l / 16][l % 16] and, in element r, D[4 r + l / 16][l % 16].  It rounds like a
// chain of FMAs in the order of q, so the products below have the bits of plain
// loops over their inner index.
__device__ __forceinline__ d4 mfma64(double a, double b, d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Split-K partials of [A | B] = FI^T [diag(G) FI | RT], an M1 x (M1 + D)
// product over the centres, part being nch x M1 x (M1 + D).  A wave computes one
// 16 RB x 16 RB block, number b of the dg_ab_blocks(M1, D) (A's lower triangle row by
// row: the factorisation takes no more; then B's), over centres [c kc, min(K,
// (c + 1) kc)), straight from global memory, where a row of FI or RT is a run of
// whole cache lines; 4 U centres are multiplied while the next ones are on their
// way.  dg_ab_edge chooses 32 x 32 blocks (RB = 2), which spread a small M1 over the
// chip, or for M1 > 256 64 x 64 (RB = 4), whose operands take half as much of L2's
// rate: at M1 = 1001 it bound the small ones.
// FP64 pipe.  K = 32768, M1 = 1001, D = 166: 3043 -> 1014 us (32 x 32 blocks: 2100;
// four blocks of a 128 x 128 tile to a workgroup, some of them above the diagonal or
// past the end, 1261: a wave runs for 150 us, and the last round left CUs idle for a
// fifth of the time); K = 8000, M1 = 126: 41 -> 27 us (4 x 4 register tiles of FMAs
// from LDS, and A's upper half computed too).
template <int RB>
__device__ __forceinline__ void k_partAB_body(
    const int b, const int c, const double *__restrict__ FI, const double *__restrict__ G,
    const double *__restrict__ RT, int K, int M1, int D, int kc, double *__restrict__ part) {
    const int NCOL = M1 + D, nA = bk_cdiv(M1, 16 * RB), tri = nA * (nA + 1) / 2;
    const bool isB = b >= tri;
    int bi = 0, bj = b;
    if (isB) {
        const int nB = bk_cdiv(D, 16 * RB);
        bi = (b - tri) / nB;
        bj = (b - tri) % nB;
    } else {
        while (bj > bi) bj -= ++bi;
    }
    if (bi >= nA) return;
    const int k0 = c * kc, k1 = (k0 + kc < K) ? k0 + kc : K;
    const int l = threadIdx.x & 63, j = l & 15, g = l >> 4;
    const int i0 = 16 * RB * bi, j0 = 16 * RB * bj, ncol = isB ? D : M1;
    const long E = (long)M1 * NCOL;
    // per lane: its columns of A's operand and of B's at centre k0 + g (past the
    // end: the last ones again, whose results are not stored), moved on by adds
    const double *pa[RB], *pb[RB], *pg = G + k0 + g, *R = isB ? RT : FI;
    const long sb = 4L * ncol;
#pragma unroll
    for (int x = 0; x < RB; ++x) {
        pa[x] = FI + (long)(k0 + g) * M1 + min(i0 + 16 * x + j, M1 - 1);
        pb[x] = R + (long)(k0 + g) * ncol + min(j0 + 16 * x + j, ncol - 1);
    }
    constexpr int U = RB == 2 ? 4 : 2;
    double ra[U][RB], rb[U][RB], rg[U];
    auto load = [&](int kb, bool whole) {          // centres kb .. kb + 4 U - 1
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool in = whole || kb + 4 * u + g < k1;
            rg[u] = in ? *pg : 0.0;
            pg += 4;
#pragma unroll
            for (int x = 0; x < RB; ++x) {
                ra[u][x] = in ? *pa[x] : 0.0;
                rb[u][x] = in ? *pb[x] : 0.0;
                pa[x] += 4L * M1;
                pb[x] += sb;
            }
        }
    };
    d4 acc[RB][RB];
#pragma unroll
    for (int x = 0; x < RB; ++x)
#pragma unroll
        for (int y = 0; y < RB; ++y) acc[x][y] = d4{0.0, 0.0, 0.0, 0.0};
    auto next = [&](int kb) {
        if (kb + 4 * U <= k1) load(kb, true);
        else if (kb < k1) load(kb, false);
    };
    next(k0);
    for (int kb = k0; kb < k1; kb += 4 * U) {
        double av[U][RB], bv[U][RB];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int x = 0; x < RB; ++x) {
                av[u][x] = ra[u][x];
                bv[u][x] = isB ? rb[u][x] : rg[u] * rb[u][x];
            }
        next(kb + 4 * U);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int x = 0; x < RB; ++x)
#pragma unroll
                for (int y = 0; y < RB; ++y) acc[x][y] = mfma64(av[u][x], bv[u][y], acc[x][y]);
    }
#pragma unroll
    for (int x = 0; x < RB; ++x)
#pragma unroll
        for (int y = 0; y < RB; ++y)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = i0 + 16 * x + 4 * r + g, jj = j0 + 16 * y + j;
                if (i < M1 && jj < ncol)
                    part[(long)c * E + (long)i * NCOL + (isB ? M1 : 0) + jj] = acc[x][y][r];
            }
}

// The hardware hands workgroup i to XCD i mod 8: all blocks of a chunk go to one
// XCD, whose L2 then holds the chunk's rows (4.7 MB at M1 = 1001, kc = 512).
// W waves to a workgroup: two where blocks are few (M1 = 65: 7.7 us, four 9.4), four
// of the large ones, which share lines in L1 (M1 = 1001: 1011 us; one 1021).
template <int RB, int W>
__global__ __launch_bounds__(64 * W, 2) void k_partAB(const double *__restrict__ FI,
                                                      const double *__restrict__ G,
                                                      const double *__restrict__ RT, int K, int M1,
                                                      int D, int kc, int nch,
                                                      double *__restrict__ part) {
    const int nw = bk_cdiv(dg_ab_blocks(M1, D), W), i = blockIdx.x >> 3;
    const int c = i / nw * 8 + (blockIdx.x & 7);
    const int b = i % nw * W + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (c < nch) k_partAB_body<RB>(b, c, FI, G, RT, K, M1, D, kc, part);
}

// A0 / B from the chunk partials, summed in chunk order (A0 without the blocks
// that k_partAB leaves out); the workgroups after those copy G to Gm, which the
// critical-temperature search reads (vggsub of dagtm.cxx:1715, still set when
// the next E-step converges).
__device__ __forceinline__ void k_sumAB_body(
    const int bx, const double *__restrict__ part,
    int nch, int M1, int D, double *__restrict__ A0, double *__restrict__ B, int K,
    const double *__restrict__ G, double *__restrict__ Gm) {
    const int NCOL = M1 + D;
    const long E = (long)M1 * NCOL;
    const long e = (long)bx * 256 + threadIdx.x;
    const int nE = bk_cdiv(E, 256);
    if (bx >= nE) {
        const int k = (bx - nE) * 256 + threadIdx.x;
        if (k < K) Gm[k] = G[k];
        return;
    }
    if (e >= E) return;
    const int i = (int)(e / NCOL), j = (int)(e % NCOL);
    const int edge = dg_ab_edge(M1);
    if (j < M1 && j / edge > i / edge) return;     // (above A's lower blocks)
    // eight loads in flight, then their sums in chunk order
    double s = 0.0;
    int c = 0;
    for (; c + 8 <= nch; c += 8) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = part[(long)(c + u) * E + e];
#pragma unroll
        for (int u = 0; u < 8; ++u) s += v[u];
    }
    for (; c < nch; ++c) s += part[(long)c * E + e];
    if (j < M1) A0[(long)i * M1 + j] = s;
    else B[(long)i * D + (j - M1)] = s;
}

__global__ __launch_bounds__(256) void k_sumAB(const double *__restrict__ part, int nch, int M1,
                                               int D, double *__restrict__ A0,
                                               double *__restrict__ B, int K,
                                               const double *__restrict__ G,
                                               double *__restrict__ Gm) {
    k_sumAB_body(blockIdx.x, part, nch, M1, D, A0, B, K, G, Gm);
}

constexpr int kLdsN = 126;   // largest M+1 whose factor fits in LDS
static_assert(kLdsN <= 128, "a wave holds two rows of a panel per lane, eight 16-row blocks");

// Broadcast lane l's value of x (l wave-uniform) to the whole wavefront.
__device__ __forceinline__ double lane_bcast(double x, int l) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)u, l);
    const unsigned hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), l);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

constexpr int kPB = 8;        // panel width of the blocked Cholesky

// put(i, k, A[i][k]) for the lower triangle of the n x n matrix A (n <= 128),
// rows spread over the workgroup's waves, eight rows' loads in flight
template <typename Put>
__device__ __forceinline__ void load_lower(const double *__restrict__ A, int n, Put &&put) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
    for (int i0 = wv; i0 < n; i0 += 8 * nw) {
        double v[8][2];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = i0 + u * nw;
#pragma unroll
            for (int h = 0; h < 2; ++h)
                v[u][h] = (i < n && lane + 64 * h <= i) ? A[(long)i * n + lane + 64 * h] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = i0 + u * nw;
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (i < n && lane + 64 * h <= i) put(i, lane + 64 * h, v[u][h]);
        }
    }
}

template <int... Is, typename F>
__device__ __forceinline__ void each_of(std::integer_sequence<int, Is...>, F &&f) {
    (f(std::integral_constant<int, Is>{}), ...);
}

// x of the four lanes j + 16 q, q = 0 .. 3, replaced by the one of q = G: the
// row swaps of v_permlane16_swap leave rows {0, 0, 2, 2} and {1, 1, 3, 3} of a
// value swapped with itself, v_permlane32_swap its halves.
template <int G>
__device__ __forceinline__ double row_bcast(double x) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
    unsigned h[2] = {(unsigned)u, (unsigned)(u >> 32)};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const auto a = __builtin_amdgcn_permlane16_swap(h[i], h[i], false, false);
        const unsigned t = (G & 1) ? (unsigned)a[1] : (unsigned)a[0];
        const auto b = __builtin_amdgcn_permlane32_swap(t, t, false, false);
        h[i] = (G & 2) ? (unsigned)b[1] : (unsigned)b[0];
    }
    return __builtin_bit_cast(double, ((unsigned long long)h[1] << 32) | h[0]);
}

// ---- blocked Cholesky and solves for M + 1 > 126 ---------------------------
// (A0 + (ridge + jitter) I) W = B by 64 x 64 blocks over many workgroups.  The
// right-hand sides, transposed, are further rows below A: their blocks of the
// factor are the forward substitution, with the same chain for every element.
// S is that (n + nrhs) x n matrix, row-major, factored in place; Ld takes the
// diagonal blocks' factors, transposed and filled up with the identity, 64 x 64
// each.  One launch per block column (k_bc_step), one for the whole backward
// substitution (k_bc_back).  failed[kc] is 1 where a pivot before block column kc was
// not positive: launch kc reads failed[kc] and writes failed[kc + 1], so that no
// workgroup reads what another one of its launch writes.  After a failure the
// kernels of the sequence return at once, and the host retries with a jitter.
constexpr int BC = 64;
constexpr int kBcLd = BC + 2;    // LDS row stride: 16 rows x 2 inner indexes hit 32 banks

__global__ __launch_bounds__(256) void k_bc_init(const double *__restrict__ A0,
                                                 double *__restrict__ S, int n, double ridge,
                                                 double jit, const double *__restrict__ B,
                                                 int nrhs, double *__restrict__ failed,
                                                 double *__restrict__ scal) {
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    const long nn = (long)n * n;
    if (e < nn) {
        S[e] = A0[e] + ((e / n == e % n) ? ridge + jit : 0.0);
    } else if (e < nn + (long)n * nrhs) {
        const long c = (e - nn) / n, p = (e - nn) % n;
        S[e] = B[p * nrhs + c];
    }
    if (e == 0) {
        failed[0] = 0.0;
        scal[kScalJitter] = jit;
    }
}

// Block column kc of the factorisation, with block column kc - 1's products:
// workgroup (x, 0) takes 64 rows below the diagonal block through all of it,
//   P = S[rows][kc] - L[rows][kc - 1] L[kc][kc - 1]^T,  P <- P L_kk^-T,
// and finds L_kk for itself, from the diagonal block less its own product
// (the same in every workgroup, none waits for another; workgroup 0 leaves it in
// Ld); workgroup (x, 1 + y) subtracts the product from one 64 x 64 tile of the
// columns after kc.  So a step is one launch, and the tiles run beside the panel.
//   Wave 0 factors 16 columns at a time in registers (a row to a lane, the pivot
// row broadcast with readlane), waves 1 .. 4 meanwhile solve their 16 rows of the
// panel against the 16 columns before, and all five apply the 16 columns to the
// rest of the diagonal block on matrix instructions.  The panel is held as
// [column][row], so that a solved 16 x 16 block in an accumulator is, as it lies,
// the operand of the products that follow.
// Bound by the chain of 64 square roots and divisions per step.  n = 1001, 166
// right-hand sides: 32 us a step; three launches for the factorisation and two
// for the forward substitution per block, each a third-full chain of its own,
// 86 + 46 + 20 and 32 + 20 us.
constexpr int kBcNT = 320;
__global__ __launch_bounds__(kBcNT) void k_bc_step(double *__restrict__ S, int n, int nrows, int kc,
                                                   double *__restrict__ Ld,
                                                   double *__restrict__ failed) {
    __shared__ double Pk[BC][kBcLd];               // L[kc][kc - 1], or a tile's columns
    __shared__ double Dg[BC][kBcLd];               // the diagonal block
    __shared__ int bad;
    const int tid = threadIdx.x, l = tid & 63, j = l & 15, g = l >> 4;
    if (failed[kc] != 0.0) {
        if (tid == 0 && blockIdx.x == 0 && blockIdx.y == 0) failed[kc + 1] = 1.0;
        return;
    }
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int k0 = kc * BC, kb = min(BC, n - k0), k1 = k0 + kb, kp = k0 - BC;
    const int i0 = k1 + blockIdx.x * BC;           // the first of this workgroup's rows
    const bool panel = blockIdx.y == 0;
    const int c0 = panel ? k0 : k1 + ((int)blockIdx.y - 1) * BC;
    if (!panel && c0 > i0 + BC - 1) return;        // above the diagonal
    const int cn = min(BC, n - c0);                // columns of this workgroup's tile
    if (kc > 0)
        for (int e = tid; e < BC * BC; e += kBcNT) {
            const int r = e >> 6, p = e & 63;
            Pk[r][p] = (r < cn) ? S[(long)(c0 + r) * n + kp + p] : 0.0;
        }
    const int wr = panel ? w - 1 : w;              // which 16 of the rows, if 0 .. 3
    const bool rows = wr >= 0 && wr < 4;
    const int ir = min(i0 + 16 * max(wr, 0) + j, nrows - 1);   // this lane's row (past the end: the last)
    double pa[16];                                 // L[ir][kp + 4 s + g]
#pragma unroll
    for (int s = 0; s < 16; ++s) pa[s] = (kc > 0 && rows) ? S[(long)ir * n + kp + 4 * s + g] : 0.0;
    if (!panel) {
        __syncthreads();
        if (!rows) return;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int s = 0; s < 16; ++s) acc = mfma64(pa[s], Pk[16 * t + j][4 * s + g], acc);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = i0 + 16 * wr + 4 * r + g, c = c0 + 16 * t + j;
                if (i < nrows && c < n && c <= i) S[(long)i * n + c] -= acc[r];
            }
        }
        return;
    }
    d4 x[4];                                       // P, [column 16 t + 4 r + g][row j]
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int p = 16 * t + 4 * r + g;
            x[t][r] = (rows && p < kb) ? S[(long)ir * n + k0 + p] : 0.0;
        }
    for (int e = tid; e < BC * BC; e += kBcNT) {
        const int r = e >> 6, c = e & 63;
        Dg[r][c] = (r < kb && c <= r) ? S[(long)(k0 + r) * n + k0 + c] : (r == c) ? 1.0 : 0.0;
    }
    if (tid == 0) bad = 0;
    __syncthreads();
    if (kc > 0) {
        for (int t = w; t < 10; t += 5) {          // the diagonal block's lower tiles
            const int ti = (t < 1) ? 0 : (t < 3) ? 1 : (t < 6) ? 2 : 3, tj = t - ti * (ti + 1) / 2;
            d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int s = 0; s < 16; ++s)
                acc = mfma64(Pk[16 * ti + j][4 * s + g], Pk[16 * tj + j][4 * s + g], acc);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = 16 * ti + 4 * r + g, c = 16 * tj + j;
                if (c <= i) Dg[i][c] -= acc[r];    // (0 past the end: Pk's rows are)
            }
        }
        if (rows)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int s = 0; s < 16; ++s) acc = mfma64(Pk[16 * t + j][4 * s + g], pa[s], acc);
#pragma unroll
                for (int r = 0; r < 4; ++r) x[t][r] -= acc[r];
            }
        __syncthreads();
    }
    // columns 16 t .. of the panel, once those of L_kk are there
    auto solve = [&](auto T) {
        constexpr int t = decltype(T)::value;
        each_of(std::make_integer_sequence<int, t>{}, [&](auto U) {
            constexpr int u = decltype(U)::value;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                x[t] = mfma64(-Dg[16 * t + j][16 * u + 4 * r + g], x[u][r], x[t]);
        });
        each_of(std::make_integer_sequence<int, 16>{}, [&](auto I) {
            constexpr int i = decltype(I)::value, R = i >> 2, Gi = i & 3;
            const double xi = row_bcast<Gi>(x[t][R]) / Dg[16 * t + i][16 * t + i];
#pragma unroll
            for (int r = R; r < 4; ++r) {
                const int p = 4 * r + g;
                const double v = fma(-xi, Dg[16 * t + max(p, i)][16 * t + i], x[t][r]);
                x[t][r] = (p == i) ? xi : (p > i) ? v : x[t][r];
            }
        });
    };
    each_of(std::make_integer_sequence<int, 4>{}, [&](auto T) {
        constexpr int t = decltype(T)::value;
        if (w == 0) {
            double a[16];
#pragma unroll
            for (int c = 0; c < 16; ++c) a[c] = Dg[l][16 * t + c];
            bool failed = false;
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const double piv = lane_bcast(a[q], 16 * t + q);
                failed = failed || !(piv > 0.0);
                const double sq = sqrt(piv);
                a[q] = (l == 16 * t + q) ? sq : a[q] / sq;
#pragma unroll
                for (int c = q + 1; c < 16; ++c)
                    a[c] = fma(-a[q], lane_bcast(a[q], 16 * t + c), a[c]);
            }
#pragma unroll
            for (int c = 0; c < 16; ++c)
                if (l >= 16 * t + c) Dg[l][16 * t + c] = a[c];
            if (failed && l == 0) bad = 1;
        } else if constexpr (t > 0) {
            solve(std::integral_constant<int, t - 1>{});
        }
        __syncthreads();
        if constexpr (t < 3) {
            constexpr int nt = 3 - t;              // 16 x 16 tiles a side after this column
            for (int q = w; q < nt * (nt + 1) / 2; q += 5) {
                const int a = (q < 1) ? 0 : (q < 3) ? 1 : 2;
                const int ti = t + 1 + a, tj = t + 1 + q - a * (a + 1) / 2;
                d4 c;
#pragma unroll
                for (int r = 0; r < 4; ++r) c[r] = Dg[16 * ti + 4 * r + g][16 * tj + j];
#pragma unroll
                for (int s = 0; s < 16; s += 4)
                    c = mfma64(-Dg[16 * ti + j][16 * t + s + g], Dg[16 * tj + j][16 * t + s + g], c);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (16 * tj + j <= 16 * ti + 4 * r + g) Dg[16 * ti + 4 * r + g][16 * tj + j] = c[r];
            }
            __syncthreads();
        }
    });
    if (tid == 0 && blockIdx.x == 0) failed[kc + 1] = bad ? 1.0 : 0.0;
    if (bad) return;                               // the same in every workgroup
    if (blockIdx.x == 0)
        for (int e = tid; e < BC * BC; e += kBcNT) {
            const int c = e >> 6, r = e & 63;
            Ld[(long)kc * BC * BC + e] = (c <= r) ? Dg[r][c] : 0.0;
        }
    if (w == 0) return;
    solve(std::integral_constant<int, 3>{});
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int p = 16 * t + 4 * r + g;
            if (p < kb && i0 + 16 * wr + j < nrows) S[(long)ir * n + k0 + p] = x[t][r];
        }
}

// L^T W = Y for sixteen right-hand sides, Y^T in the rows of S after the n-th:
// block by block from the last.  Wave 0 solves a block, a right-hand side to a
// lane, while waves 1 .. 4 subtract the products of the blocks solved before it
// from the next (16 of its rows each); the solved block's own product follows.
// Row i of a block takes x[i + 1], x[i + 2], .. in that order, so its chain can
// only begin when x[i + 1] is known: 2016 dependent FMAs and 64 divisions a block
// bound the kernel.  n = 1001, 166 right-hand sides: 289 us (two launches per
// block, 50 + 20 us each).
__global__ __launch_bounds__(kBcNT) void k_bc_back(const double *__restrict__ S, int n, int nrhs,
                                                   const double *__restrict__ Ld,
                                                   double *__restrict__ W,
                                                   const double *__restrict__ failed,
                                                   double *__restrict__ scal) {
    __shared__ __align__(16) double Lt[2][BC][kBcLd];   // L_kk transposed: Lt[i][p] = L[p][i]
    __shared__ double Ln[BC][kBcLd];                    // L[k][k - 1]
    __shared__ double Sx[BC][16], Xs[BC][16];           // the block's right side, its solution
    __shared__ double Sn[BC][16];                       // the next one's, but for the block's product
    const int tid = threadIdx.x, l = tid & 63, j = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = (n + BC - 1) / BC;
    const bool ok = failed[nb] == 0.0;
    if (tid == 0 && blockIdx.x == 0) scal[kScalSolveOK] = ok ? 1.0 : 0.0;
    if (!ok) return;
    const int col = min(16 * (int)blockIdx.x + j, nrhs - 1);   // past the end: the last again
    const bool live = 16 * (int)blockIdx.x + j < nrhs;
    const double *Yc = S + (long)(n + col) * n;
    const int ro = 16 * (w - 1);                   // waves 1 .. 4: their rows of a block
    auto stage = [&](int k) {                      // Ld of block k, by the threads of waves 1 .. 4
        for (int e = tid - 64; e < BC * BC; e += 256)
            Lt[k & 1][e >> 6][e & 63] = Ld[(long)k * BC * BC + e];
    };
    if (w > 0) {
        stage(nb - 1);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = ro + 4 * r + g, p = (nb - 1) * BC + i;
            Sx[i][j] = (p < n) ? Yc[p] : 0.0;
        }
    }
    __syncthreads();
    for (int k = nb - 1; k >= 0; --k) {
        const int k0 = k * BC, kb = min(BC, n - k0);
        if (w == 0) {
            // L's entries of a row are read sixteen at a time, one run ahead
            const double(*T)[kBcLd] = Lt[k & 1];
            double x[BC], cur[16], s = Sx[BC - 1][j], dg = T[BC - 1][BC - 1];
            each_of(std::make_integer_sequence<int, BC>{}, [&](auto I) {
                constexpr int i = BC - 1 - decltype(I)::value, m0 = (i + 1) / 16;
                double sn = 0.0, dn = 0.0;
                each_of(std::make_integer_sequence<int, 4 - m0>{}, [&](auto M) {
                    constexpr int m = m0 + decltype(M)::value;
                    constexpr int ni = (m < 3) ? i : i - 1;           // the run after this one
                    constexpr int nm = (m < 3) ? m + 1 : i / 16;
                    double nxt[16];
                    if constexpr (ni >= 0) {
#pragma unroll
                        for (int p = 0; p < 16; ++p) nxt[p] = (16 * nm + p > ni) ? T[ni][16 * nm + p] : 0.0;
                        if constexpr (m == 3) {
                            sn = Sx[ni][j];
                            dn = T[ni][ni];
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int p = 0; p < 16; ++p)
                        if (16 * m + p > i) s = fma(-cur[p], x[16 * m + p], s);
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (ni >= 0)
#pragma unroll
                        for (int p = 0; p < 16; ++p) cur[p] = nxt[p];
                });
                if constexpr (i == BC - 1) {
#pragma unroll
                    for (int p = 0; p < 16; ++p) cur[p] = T[BC - 2][BC - 16 + p];
                    sn = Sx[BC - 2][j];
                    dn = T[BC - 2][BC - 2];
                }
                x[i] = s / dg;
                s = sn;
                dg = dn;
                Xs[i][j] = x[i];                   // (the four lanes of a right-hand side alike)
            });
        } else if (k > 0) {
            stage(k - 1);
            // (opaque: the rows' offsets kept over the blocks would spill)
            int ld = n, ldw = nrhs;
            asm volatile("" : "+s"(ld), "+s"(ldw));
            const int r0 = k0 - BC + ro;           // this wave's first row in block k - 1
            d4 c;
#pragma unroll
            for (int r = 0; r < 4; ++r) c[r] = Yc[r0 + 4 * r + g];
            const double *Lr = S + r0 + j;
            for (int q = 0; q < 16; ++q)           // (wanted after the barrier)
                Ln[4 * q + g][ro + j] = Lr[(long)min(k0 + 4 * q + g, n - 1) * ld];
            // half a block's rows at a time, one half ahead (only the last block has
            // rows past the end: the last of L, zero of x)
            double lv[8], xv[8];
            auto load = [&](int b, int h) {
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const int p = b * BC + 32 * h + 4 * q + g, pc = min(p, n - 1);
                    lv[q] = Lr[(long)pc * ld];
                    xv[q] = W[(long)pc * ldw + col];
                    xv[q] = (p < n) ? xv[q] : 0.0;
                }
            };
            if (nb - 1 > k) load(nb - 1, 0);
            for (int b = nb - 1; b > k; --b) {
                d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    double lc[8], xc[8];
#pragma unroll
                    for (int q = 0; q < 8; ++q) { lc[q] = lv[q]; xc[q] = xv[q]; }
                    if (h == 0) load(b, 1);
                    else if (b - 1 > k) load(b - 1, 0);
#pragma unroll
                    for (int q = 0; q < 8; ++q) acc = mfma64(lc[q], xc[q], acc);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) c[r] -= acc[r];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) Sn[ro + 4 * r + g][j] = c[r];
        }
        __syncthreads();
        if (w > 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = ro + 4 * r + g;
                if (live && i < kb) W[(long)(k0 + i) * nrhs + col] = Xs[i][j];
            }
        }
        if (w > 0 && k > 0) {
            d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int p = 4 * q + g;
                acc = mfma64(Ln[p][ro + j], Xs[p][j], acc);   // (x is 0 past the end)
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
                Sx[ro + 4 * r + g][j] = Sn[ro + 4 * r + g][j] - acc[r];
        }
        __syncthreads();
    }
}

// W[:, c0 : c0 + 16] from (A0 + (ridge + jitter) I) W = B for n <= 126, the lower
// triangle resident in LDS; same pivots and retries as k_chol_solve_body.  Every
// workgroup factors the matrix for itself (they run side by side, and the factor
// need not go through memory to a second kernel).
//   Factor: blocked, right-looking.  Wave 0 takes each 8-column panel in registers
// (lane r holds rows p0 + r and p0 + r + 64; the pivot row and the L entries of
// later panel columns are broadcast with readlane, so the panel needs no barrier),
// then all waves apply the panel to the trailing lower triangle, a 16 x 16 tile
// at a time on matrix instructions (the chain over the panel's columns from 0,
// subtracted from the tile).  Two barriers per panel.
//   Solve: the right-hand sides in 16-row blocks, block t in the accumulator of
// wave t.  For each block in turn its wave solves the 16 x 16 triangle in the
// accumulator's layout, and the waves then apply the block's x to their blocks on
// matrix instructions.  Each row receives its updates in the order of the plain
// substitution: x_i = x_i (1 / L_ii), then one FMA per later row in ascending i
// (forward), or per earlier row in descending i (backward, the MFMA's inner index
// running down).
// Bound by the chains of square roots, reciprocals and blocks, one CU's latency.
// n = 126: 72 us, n = 65: 40, n = 26: 18.6; as two kernels, 55 + 35, 27 + 22
// and 13 + 9 and the gap between them, and 90 + 48, 45 + 27 and 17 + 15 with 4 x 4
// register tiles of FMAs and a wave per right-hand side.
constexpr int kCholNT = 1024;
__device__ __forceinline__ void k_solve_lds_body(
    const int bx, const double *__restrict__ A0, int n, double ridge, const double *__restrict__ B,
    int nrhs, double *__restrict__ W, double *__restrict__ scal) {
    __shared__ double As[128 * (kLdsN | 1) + 16];
    __shared__ double Pt[kPB][128 + 16];             // the factored panel, transposed
    __shared__ double tr;
    __shared__ int bad;
    __shared__ double rd[128];                       // 1 / L_pp
    __shared__ double xs[16][17];                    // the block just solved
    const int tid = threadIdx.x, nw = blockDim.x >> 6;
    const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15, g = lane >> 4;
    const int ld = n | 1;                            // odd: a column spreads over the banks
    const int nblk = (n + 15) / 16;
    const int col = 16 * bx + j;
    const bool live = col < nrhs;
    d4 x = {0.0, 0.0, 0.0, 0.0};                     // block wv
    if (wv < nblk)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int p = 16 * wv + 4 * r + g;
            x[r] = (live && p < n) ? B[(long)p * nrhs + col] : 0.0;
        }
    // rows past the end: zero entries of L, and zero right-hand sides
    for (int e = n * ld + tid; e < 16 * nblk * ld + 16; e += blockDim.x) As[e] = 0.0;
    double jit = 0.0;
    int ok = 0;
    for (int attempt = 0; attempt < 9 && !ok; ++attempt) {
        if (attempt == 1) {
            block_trace(A0, n, &tr);
            jit = 1e-13 * tr / n;
        } else if (attempt > 1) {
            jit *= 10.0;
        }
        load_lower(A0, n, [&](int i, int k, double v) {
            As[i * ld + k] = v + ((i == k) ? ridge + jit : 0.0);
        });
        if (tid == 0) bad = 0;
        __syncthreads();
        for (int p0 = 0; p0 < n; p0 += kPB) {
            const int pn = min(kPB, n - p0);
            if (wv == 0) {
                const int r0 = p0 + lane, r1 = r0 + 64;
                double a0[kPB], a1[kPB];
#pragma unroll
                for (int c = 0; c < kPB; ++c) {
                    a0[c] = (c < pn && r0 < n && c <= lane) ? As[r0 * ld + p0 + c] : 0.0;
                    a1[c] = (c < pn && r1 < n) ? As[r1 * ld + p0 + c] : 0.0;
                }
                bool failed = false;
#pragma unroll
                for (int q = 0; q < kPB; ++q) {
                    if (q < pn && !failed) {
                        const double piv = lane_bcast(a0[q], q);     // row p0 + q is lane q's
                        if (!(piv > 0.0)) {
                            failed = true;                           // the same in every lane
                        } else {
                            // (rows above the diagonal, lanes < c of column
                            // c, hold nothing that is read)
                            const double sq = sqrt(piv), inv = 1.0 / sq;
                            a0[q] = (lane == q) ? sq : a0[q] * inv;
                            a1[q] *= inv;
#pragma unroll
                            for (int c = q + 1; c < kPB; ++c) {
                                const double lcj = lane_bcast(a0[q], c);   // L[p0 + c][p0 + q]
                                a0[c] = fma(-a0[q], lcj, a0[c]);
                                a1[c] = fma(-a1[q], lcj, a1[c]);
                            }
                        }
                    }
                }
                // (rows past the end are zero: the tiles below need no bounds)
#pragma unroll
                for (int c = 0; c < kPB; ++c) {
                    if (c < pn && c <= lane && r0 < n) As[r0 * ld + p0 + c] = a0[c];
                    if (c < pn && r1 < n) As[r1 * ld + p0 + c] = a1[c];
                    Pt[c][lane] = (r0 < n) ? a0[c] : 0.0;
                    Pt[c][lane + 64] = (r1 < n) ? a1[c] : 0.0;
                    if (lane < 16) Pt[c][lane + 128] = 0.0;
                }
                if (failed && lane == 0) bad = 1;
            }
            __syncthreads();
            if (bad) break;                                  // read after the barrier: uniform
            // A[i][k] -= sum_q L[i][p0 + q] L[k][p0 + q] for q0 <= k <= i: tile
            // (ti, tj) of the triangle from q0 on, numbered row by row
            const int q0 = p0 + pn, nt = (n - q0 + 15) / 16;
            for (int t = wv; t < nt * (nt + 1) / 2; t += nw) {
                int ti = 0, tj = t;
                while (tj > ti) { tj -= ti + 1; ++ti; }
                const int oi = pn + 16 * ti + j, oj = pn + 16 * tj + j;   // panel-relative rows
                d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int s4 = 0; s4 < kPB; s4 += 4)
                    acc = mfma64(Pt[s4 + g][oi], Pt[s4 + g][oj], acc);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = q0 + 16 * ti + 4 * r + g, k = q0 + 16 * tj + j;
                    if (i < n && k <= i) As[i * ld + k] -= acc[r];
                }
            }
            __syncthreads();
        }
        ok = !bad;
        __syncthreads();                                     // before the next attempt resets bad
    }
    if (tid == 0 && bx == 0) {
        scal[kScalJitter] = jit;
        scal[kScalSolveOK] = ok ? 1.0 : 0.0;
    }
    if (!ok) return;
    if (tid < 128) rd[tid] = (tid < n) ? 1.0 / As[tid * ld + tid] : 0.0;
    __syncthreads();
    auto at = [&](int i, int k) { return As[i * ld + k]; };   // k <= i
    // block t's triangle, in the accumulator's layout: row i = 4 R + G goes from
    // its lanes to the others of its column, which update their later (earlier)
    // rows; xs gets the solved rows
    auto diag = [&](int t, d4 &c, auto fwd) {
        const int b0 = 16 * t;
        auto step = [&](auto I) {
            constexpr int i = decltype(fwd)::value ? decltype(I)::value : 15 - decltype(I)::value;
            constexpr int R = i >> 2, Gi = i & 3;
            const double xi = row_bcast<Gi>(c[R]) * rd[b0 + i];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (decltype(fwd)::value ? r < R : r > R) continue;
                const int p = 4 * r + g;
                const bool upd = decltype(fwd)::value ? p > i : p < i;
                const double lp = decltype(fwd)::value ? at(b0 + (upd ? p : i), b0 + i)
                                                       : at(b0 + i, b0 + (upd ? p : i));
                const double v = fma(-lp, xi, c[r]);
                c[r] = (p == i) ? xi : upd ? v : c[r];
            }
        };
        each_of(std::make_integer_sequence<int, 16>{}, step);
#pragma unroll
        for (int r = 0; r < 4; ++r) xs[4 * r + g][j] = c[r];
    };
    for (int t = 0; t < nblk; ++t) {                 // forward
        if (wv == t) diag(t, x, std::true_type{});
        __syncthreads();
        if (wv > t && wv < nblk)
#pragma unroll
            for (int s4 = 0; s4 < 16; s4 += 4)
                x = mfma64(-at(16 * wv + j, 16 * t + s4 + g), xs[s4 + g][j], x);
        __syncthreads();                             // xs is rewritten by the next block
    }
    for (int t = nblk - 1; t >= 0; --t) {            // backward with L^T, i descending
        if (wv == t) diag(t, x, std::false_type{});
        __syncthreads();
        if (wv < t)
#pragma unroll
            for (int s4 = 15; s4 > 0; s4 -= 4)
                x = mfma64(-at(16 * t + s4 - g, 16 * wv + j), xs[s4 - g][j], x);
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int p = 16 * wv + 4 * r + g;
        if (live && p < n) W[(long)p * nrhs + col] = x[r];
    }
}

__global__ __launch_bounds__(kCholNT) void k_solve_lds(const double *__restrict__ A0, int n,
                                                       double ridge, const double *__restrict__ B,
                                                       int nrhs, double *__restrict__ W,
                                                       double *__restrict__ scal) {
    k_solve_lds_body(blockIdx.x, A0, n, ridge, B, nrhs, W, scal);
}

// The new centres and what the M-step takes from them, sixteen centres to a
// workgroup:
//   Y = FI W into the padded layout (K x ld, columns >= D untouched),
//   yy_k = |y_k|^2, a chain in d,
//   part[bx] = sum over its centres of G_k |y_k|^2 - 2 y_k . RT_k, in order
//   (with part null, Y and yy only),
//   amax[bx] = max |Y| over them (with amax null: not wanted).
// FI's rows pass through LDS 64 functions at a time, the wave's share of W's
// columns (16 d-blocks w, w + 4, w + 8) straight from L2.  D <= 192.
// Bound by latency at M1 = 126 (32 steps of one load and one MFMA chain each) and
// by the FP64 pipe at M1 = 1001.  K = 8000, M1 = 126, D = 166: 23 us (Y, norms,
// sums and maximum as five kernels, the first with 4 x 4 tiles of FMAs: 71);
// K = 32768, M1 = 1001: 344 us (541); K = 400, M1 = 26, D = 12: 7 us (20, without
// a maximum).
constexpr int CW = 16;                             // centres per workgroup
__device__ __forceinline__ void k_centres_body(
    const int bx, const double *__restrict__ FI, const double *__restrict__ W, int K, int M1, int D,
    int ld, const double *__restrict__ G, const double *__restrict__ RT, double *__restrict__ Y,
    double *__restrict__ yy, double *__restrict__ part, double *__restrict__ amax) {
    constexpr int FC = 64, FP = FC + 4;            // functions per chunk, row stride in LDS
    constexpr int YP = 192 + 2;
    __shared__ double Fs[2][CW][FP];
    __shared__ double Yt[CW][YP];
    __shared__ double nrm[CW], dots[CW], mx[4];
    const int tid = threadIdx.x, l = tid & 63, w = tid >> 6, j = l & 15, g = l >> 4;
    const int k0 = bx * CW;
    const int nd = (D + 15) / 16;                  // d-blocks, w, w + 4, w + 8 this wave's
    const int sr = tid >> 4, sp = tid & 15;        // staging: 16 threads to a row of FI
    const double *frow = FI + (long)min(k0 + sr, K - 1) * M1;
    double rf[4];
    auto load = [&](int f0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int f = f0 + sp + 16 * i;
            rf[i] = (f < M1) ? frow[f] : 0.0;
        }
    };
    auto store = [&](int b) {
#pragma unroll
        for (int i = 0; i < 4; ++i) Fs[b][sr][sp + 16 * i] = rf[i];
    };
    int col[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) col[q] = min(16 * (w + 4 * q) + j, D - 1);
    d4 acc[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) acc[q] = d4{0.0, 0.0, 0.0, 0.0};
    load(0);
    store(0);
    __syncthreads();
    int b = 0;
    for (int f0 = 0; f0 < M1; f0 += FC, b ^= 1) {
        if (f0 + FC < M1) load(f0 + FC);
        const int steps = (min(FC, M1 - f0) + 3) / 4;
        if (w < nd) {
            // (functions past the end: FI's are 0 in LDS, W's row the last one)
            constexpr int U = 4;
            double wv[U][3];
            auto loadw = [&](int s0) {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const double *wr = W + (long)min(f0 + 4 * (s0 + u) + g, M1 - 1) * D;
#pragma unroll
                    for (int q = 0; q < 3; ++q)
                        if (q == 0 || w + 4 * q < nd) wv[u][q] = wr[col[q]];
                }
            };
            loadw(0);
            for (int s0 = 0; s0 < steps; s0 += U) {
                double av[U], bv[U][3];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int f = 4 * (s0 + u) + g;
                    av[u] = Fs[b][j][f < FC ? f : 0];
#pragma unroll
                    for (int q = 0; q < 3; ++q) bv[u][q] = wv[u][q];
                }
                if (s0 + U < steps) loadw(s0 + U);
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (s0 + u < steps)
#pragma unroll
                        for (int q = 0; q < 3; ++q)
                            if (q == 0 || w + 4 * q < nd) acc[q] = mfma64(av[u], bv[u][q], acc[q]);
            }
        }
        if (f0 + FC < M1) store(b ^ 1);
        __syncthreads();
    }
    double top = 0.0;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const int d = 16 * (w + 4 * q) + j;
        if (d < D)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int c = 4 * r + g, k = k0 + c;
                Yt[c][d] = acc[q][r];
                if (k < K) {
                    Y[(long)k * ld + d] = acc[q][r];
                    top = fmax(top, fabs(acc[q][r]));
                }
            }
    }
    if (amax) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) top = fmax(top, __shfl_xor(top, o));
        if (l == 0) mx[w] = top;
    }
    __syncthreads();
    // |y|^2: the last wave, one centre to a lane
    if (w == 3 && l < CW) {
        double s = 0.0;
        int d = 0;
        for (; d + 8 <= D; d += 8) {
            double v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = Yt[l][d + u];
#pragma unroll
            for (int u = 0; u < 8; ++u) s = fma(v[u], v[u], s);
        }
        for (; d < D; ++d) s = fma(Yt[l][d], Yt[l][d], s);
        nrm[l] = s;
        if (k0 + l < K) yy[k0 + l] = s;
    }
    if (!part) return;
    // y . RT: a wave to a centre, lanes along d, waves 0 .. 2 in turn (wave 3
    // once it has the norms)
    for (int c = w; c < CW; c += 4) {
        const int k = k0 + c;
        double dot = 0.0;
        if (k < K)
            for (int d = l; d < D; d += 64) dot = fma(Yt[c][d], RT[(long)k * D + d], dot);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) dot += __shfl_xor(dot, o);
        if (l == 0) dots[c] = dot;
    }
    __syncthreads();
    if (tid == 0) {
        double s = 0.0;
        for (int c = 0; c < CW; ++c) {
            if (k0 + c >= K) break;
            s += G[k0 + c] * nrm[c] - 2.0 * dots[c];
        }
        part[bx] = s;
        if (amax) amax[bx] = fmax(fmax(mx[0], mx[1]), fmax(mx[2], mx[3]));
    }
}

__global__ __launch_bounds__(256, 2) void k_centres(
    const double *__restrict__ FI, const double *__restrict__ W, int K, int M1, int D, int ld,
    const double *__restrict__ G, const double *__restrict__ RT, double *__restrict__ Y,
    double *__restrict__ yy, double *__restrict__ part, double *__restrict__ amax) {
    k_centres_body(blockIdx.x, FI, W, K, M1, D, ld, G, RT, Y, yy, part, amax);
}

// scal[kScalBetaSum] = the sum of the n sixteen-centre partials, four by four
// (64 centres) and then as a tree; with amax, scal[kScalYMax] = its largest.
__device__ __forceinline__ void k_beta_final_body(const double *__restrict__ part, int n,
                                                  const double *__restrict__ amax,
                                                  double *__restrict__ scal) {
    __shared__ double s[256], m[256];
    double a = 0.0, top = 0.0;
    for (int i = 4 * threadIdx.x; i < n; i += 4 * 256) {
        double v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = (i + u < n) ? part[i + u] : 0.0;
        a += (v[0] + v[1]) + (v[2] + v[3]);
        if (amax)
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (i + u < n) top = fmax(top, amax[i + u]);
    }
    s[threadIdx.x] = a;
    m[threadIdx.x] = top;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            s[threadIdx.x] += s[threadIdx.x + w];
            m[threadIdx.x] = fmax(m[threadIdx.x], m[threadIdx.x + w]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        scal[kScalBetaSum] = s[0];
        if (amax) scal[kScalYMax] = m[0];
    }
}

// (hscal: the host's copy of the M-step's scalars, in pinned memory)
__global__ __launch_bounds__(256) void k_beta_final(const double *__restrict__ part, int n,
                                                    const double *__restrict__ amax, double *scal,
                                                    double *__restrict__ hscal) {
    k_beta_final_body(part, n, amax, scal);
    __syncthreads();
    const int i = kScalBetaSum + (int)threadIdx.x;
    if (i <= kScalYMax) hscal[i] = scal[i];
}

// ---------------------------------------------------------------- batched
// The M-step of many instances per launch: tab holds one BInst per instance,
// list the table indices of the instances in this launch, and one grid
// dimension selects list[slot].  Each instance keeps its own grid extents;
// workgroups past them return before any barrier.  Every instance computes
// exactly what its own single-instance launch computes, but for kb_chol_solve
// (M + 1 > 126), whose chains differ from those of the blocked kernels.

static_assert(CW == kBCentres, "flat-grid tile sizes");

// Flat-grid kernels: workgroup blockIdx.x belongs to instance map[.].x and is
// its workgroup map[.].y (grids sized by bk_count for each instance).
__global__ __launch_bounds__(256, 2) void kb_partAB(const BInst *__restrict__ tab,
                                                 const int2 *__restrict__ map) {
    const int2 m = map[blockIdx.x];
    const BInst &I = tab[m.x];
    if (!I.do_m) return;
    const int kc = (I.K + I.nchAB - 1) / I.nchAB, nw = bk_cdiv(dg_ab_blocks(I.M1, I.D), 4);
    const int b = m.y % nw * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), c = m.y / nw;
    if (dg_ab_edge(I.M1) == 32) k_partAB_body<2>(b, c, I.FI, I.G, I.RT, I.K, I.M1, I.D, kc, I.partAB);
    else k_partAB_body<4>(b, c, I.FI, I.G, I.RT, I.K, I.M1, I.D, kc, I.partAB);
}

__global__ __launch_bounds__(256) void kb_sumAB(const BInst *__restrict__ tab, const int2 *__restrict__ map) {
    const int2 m = map[blockIdx.x];
    const BInst &I = tab[m.x];
    if (!I.do_m) return;
    k_sumAB_body(m.y, I.partAB, I.nchAB, I.M1, I.D, I.A0, I.Bm, I.K, I.G, I.Gm);
}

__global__ __launch_bounds__(kCholNT) void kb_solve_lds(const BInst *__restrict__ tab,
                                                        const int2 *__restrict__ map) {
    const int2 m = map[blockIdx.x];
    const BInst &I = tab[m.x];
    if (!I.do_m) return;
    k_solve_lds_body(m.y, I.A0, I.M1, I.ridge, I.Bm, I.D, I.W, I.scal);
}

__global__ __launch_bounds__(1024) void kb_chol_solve(const BInst *__restrict__ tab,
                                                      const int *__restrict__ list) {
    const BInst &I = tab[list[blockIdx.x]];
    if (!I.do_m) return;
    k_chol_solve_body(I.A0, I.A, I.M1, I.ridge, I.Bm, I.D, I.W, I.scal);
}

__global__ __launch_bounds__(256, 2) void kb_centres(const BInst *__restrict__ tab,
                                                     const int2 *__restrict__ map) {
    const int2 m = map[blockIdx.x];
    const BInst &I = tab[m.x];
    if (!I.do_m) return;
    k_centres_body(m.y, I.FI, I.W, I.K, I.M1, I.D, I.ldt, I.G, I.RT, I.Y64, I.yy, I.partAB,
                   I.partAB + bk_cdiv(I.K, CW));
}

__global__ __launch_bounds__(256) void kb_beta_final(const BInst *__restrict__ tab,
                                                     const int *__restrict__ list) {
    const BInst &I = tab[list[blockIdx.x]];
    if (!I.do_m) return;
    const int n = bk_cdiv(I.K, CW);
    k_beta_final_body(I.partAB, n, I.partAB + n, I.scal);
}

}  // namespace

// dst[r * ld + d] = src[r * lds + d] for d < D, 0 for D <= d < ld.
__global__ __launch_bounds__(256) void k_pad_rows(const double *__restrict__ src, long rows,
                                                  int D, long lds, int ld,
                                                  double *__restrict__ dst) {
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    if (e >= rows * ld) return;
    const long r = e / ld;
    const int d = (int)(e % ld);
    dst[e] = (d < D) ? src[r * lds + d] : 0.0;
}

int dg_pad_rows(dg_ctx *c, const double *src, long rows, int D, long lds, int ld, double *dst) {
    const long n = rows * ld;
    hipLaunchKernelGGL(k_pad_rows, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, src,
                       rows, D, lds, ld, dst);
    DG_HIP(c, hipGetLastError());
    return DG_OK;
}

int dg_rownorms(dg_ctx *c, const double *X, long rows, int ld, int D, double *out) {
    hipLaunchKernelGGL(k_rownorm, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, c->stream,
                       X, rows, ld, D, out);
    DG_HIP(c, hipGetLastError());
    return DG_OK;
}

int dg_sum_into(dg_ctx *c, const double *v, long n, int slot) {
    hipLaunchKernelGGL(k_sum, dim3(1), dim3(1024), 0, c->stream, v, n, c->scal, slot);
    DG_HIP(c, hipGetLastError());
    return DG_OK;
}

int dg_centres_from_w(dg_ctx *c) {
    hipLaunchKernelGGL(k_centres, dim3((unsigned)bk_cdiv(c->K, CW)), dim3(256), 0, c->stream, c->FI,
                       c->W, c->K, c->M1, c->D, c->ldt, nullptr, nullptr, c->Y64, c->yy, nullptr,
                       nullptr);
    DG_HIP(c, hipGetLastError());
    return DG_OK;
}

// (A0 + (ridge + jit) I) W = Bm for M + 1 > 126 by the blocked kernels, in the
// (consumed) partials of A and B; scal[kScalSolveOK] is 0 after a non-positive pivot
int blocked_chol_solve(dg_ctx *c, double ridge, double jit) {
    const int n = c->M1, D = c->D, nb = (n + BC - 1) / BC;
    // (n >= 127: n^2 > 64 (n + 63) + nb, the diagonal blocks and nb + 1 flags)
    double *S = c->partAB, *Ld = c->A, *failed = Ld + (size_t)nb * BC * BC;
    const long tot = (long)n * n + (long)n * D;
    hipLaunchKernelGGL(k_bc_init, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, c->stream,
                       c->A0, S, n, ridge, jit, c->Bm, D, failed, c->scal);
    for (int k = 0; k < nb; ++k) {
        const int k1 = std::min(n, (k + 1) * BC);
        const int rt = (n + D - k1 + BC - 1) / BC, ct = (k > 0) ? (n - k1 + BC - 1) / BC : 0;
        hipLaunchKernelGGL(k_bc_step, dim3((unsigned)rt, (unsigned)(1 + ct)), dim3(kBcNT), 0,
                           c->stream, S, n, n + D, k, Ld, failed);
    }
    hipLaunchKernelGGL(k_bc_back, dim3((unsigned)((D + 15) / 16)), dim3(kBcNT), 0, c->stream, S, n,
                       D, Ld, c->W, failed, c->scal);
    DG_HIP(c, hipGetLastError());
    return DG_OK;
}

int dg_mstep_trace(dg_ctx *c) {
    hipLaunchKernelGGL(k_bc_trace, dim3(1), dim3(64), 0, c->stream, c->A0, c->M1, c->scal);
    DG_HIP(c, hipGetLastError());
    return DG_OK;
}

int dg_mstep_run(dg_ctx *c, double jitter) {
    const int M1 = c->M1, D = c->D, K = c->K;
    const long E = (long)M1 * M1 + (long)M1 * D;
    const int nch = c->nchAB;
    const int kc = (K + nch - 1) / nch;
    const int nblk = dg_ab_blocks(M1, D);
    auto ab = [&](auto kernel, int w) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)(8 * bk_cdiv(nblk, w) * bk_cdiv(nch, 8))),
                           dim3(64 * w), 0, c->stream, c->FI, c->G, c->RT, K, M1, D, kc, nch,
                           c->partAB);
    };
    if (dg_ab_edge(M1) == 32) ab(k_partAB<2, 2>, 2);
    else ab(k_partAB<4, 4>, 4);
    DG_HIP(c, hipGetLastError());
    hipLaunchKernelGGL(k_sumAB, dim3((unsigned)(bk_cdiv(E, 256) + bk_cdiv(K, 256))), dim3(256), 0,
                       c->stream, c->partAB, nch, M1, D, c->A0, c->Bm, K, c->G, c->Gm);
    DG_HIP(c, hipGetLastError());
    const double ridge = (c->cfg.lambda > 0.0) ? c->cfg.lambda / c->beta : 0.0;
    if (M1 <= kLdsN) {
        hipLaunchKernelGGL(k_solve_lds, dim3((unsigned)bk_cdiv(D, 16)), dim3(kCholNT), 0, c->stream,
                           c->A0, M1, ridge, c->Bm, D, c->W, c->scal);
    } else {
        int rc = blocked_chol_solve(c, ridge, jitter);
        if (rc) return rc;
    }
    DG_HIP(c, hipGetLastError());
    // the centres' partials reuse the (now consumed) A/B partial buffer
    const int nb = bk_cdiv(K, CW);
    double *amax = c->mixed() ? c->partAB + nb : nullptr;
    hipLaunchKernelGGL(k_centres, dim3((unsigned)nb), dim3(256), 0, c->stream, c->FI, c->W, K, M1, D,
                       c->ldt, c->G, c->RT, c->Y64, c->yy, c->partAB, amax);
    DG_HIP(c, hipGetLastError());
    hipLaunchKernelGGL(k_beta_final, dim3(1), dim3(256), 0, c->stream, c->partAB, nb, amax, c->scal,
                       c->m_scal);
    DG_HIP(c, hipGetLastError());
    return DG_OK;
}

// M-step of the instances in list (n of them; nlds with M + 1 <= 126 first in
// list, the others after), on one stream; gr holds the flat grids over that
// list (the solves in LDS over its first nlds entries).  Each
// instance's steps are those of dg_mstep_run.
int dg_batch_mstep(hipStream_t st, const BInst *tab, const int *list, int n, int nlds,
                   const BGrids &gr) {
    if (n <= 0) return DG_OK;
    auto flat = [&](auto kernel, int kind, int threads) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)gr.wg[kind]), dim3(threads), 0, st, tab,
                           gr.map[kind]);
    };
    flat(kb_partAB, BK_PART_AB, 256);
    flat(kb_sumAB, BK_SUM_AB, 256);
    if (nlds > 0) flat(kb_solve_lds, BK_SOLVE_LDS, kCholNT);
    if (n > nlds)
        hipLaunchKernelGGL(kb_chol_solve, dim3((unsigned)(n - nlds)), dim3(1024), 0, st, tab,
                           list + nlds);
    flat(kb_centres, BK_CENTRES, 256);
    hipLaunchKernelGGL(kb_beta_final, dim3((unsigned)n), dim3(256), 0, st, tab, list);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? DG_OK : DG_EHIP;
}
