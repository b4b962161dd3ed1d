// mph_cr_body.h -- per-row / per-chunk bodies of the multigrid V-cycle and the
// conjugate-residual loop (source/main.cpp:4122-4421).
//
// The single-scene kernels (mph_solver.hip) and the scene-table kernels of the
// batched executor (mph_batch.hip) both call these functions, so a scene's
// arithmetic is the same instruction sequence whether it runs alone or in a batch.
// Every body keeps the reference's operand order (y = beta*y + sum, with the sum
// formed first, as myDcsrmv / myDdmv / myDcopy / myDscal of main.cpp:4015-4119).
#pragma once

#include "mph_kernels.h"

namespace mph {
namespace body {

__host__ __device__ inline int nblk(long long n, int bs) { return (int)((n + bs - 1) / bs); }

// launch(g0, n) for stretches of `cells` workgroups.  A launch of 2^32 threads or more runs
// only its remainder, without an error: 16.8 million workgroups of 256
template <class F>
inline void per_cell(int cells, F launch) {
    constexpr int kMost = 1 << 22;
    for (long long g0 = 0; g0 < cells; g0 += kMost)
        launch((int)g0, cells - g0 < kMost ? (int)(cells - g0) : kMost);
}

// CR scalars: rr0, rs0, rr, rho, rho_prev, tmp (= q.u), rs
enum { kRR0 = 0, kRS0 = 1, kRR = 2, kRHO = 3, kRHOP = 4, kTMP = 5, kRS = 6, kRSIter = 7, kNScal = 8,
       kRHON = 10 };

__device__ inline int cell_id(const DevParams& P, int cx, int cy, int cz) {
    const int* C = P.C;
    if (P.dim == 2) return ((cx) % C[0] + C[0]) % C[0] * C[1] + ((cy) % C[1] + C[1]) % C[1];
    return ((cx) % C[0] + C[0]) % C[0] * C[1] * C[2] + ((cy) % C[1] + C[1]) % C[1] * C[2] +
           ((cz) % C[2] + C[2]) % C[2];
}

// a level's S buffer by ping-pong parity, as a select: indexing the two-pointer array
// with a run-time value would keep a Level copied into a local in private memory
__device__ inline double* lv_s(const Level& L, unsigned parity) { return parity ? L.S[1] : L.S[0]; }

__device__ inline void grid_xyz(const Level& L, int g, int& gx, int& gy, int& gz) {
    gx = (g / (L.cnt[1] * L.cnt[2])) % L.cnt[0];
    gy = (g / L.cnt[2]) % L.cnt[1];
    gz = g % L.cnt[2];
}
__device__ inline int grid_id(const Level& L, int gx, int gy, int gz) {
    return (L.cnt[1] * L.cnt[2]) * gx + L.cnt[2] * gy + gz;
}

// pairwise tree over the 256 values of a workgroup (t[l] += t[l+h], h = 128..1);
// the result is valid in thread 0.  Every thread of the workgroup must call it.
__device__ inline double block_tree_sum(double t, double* sh) {
    sh[threadIdx.x] = t;
    __syncthreads();
    if (threadIdx.x < 128) sh[threadIdx.x] = sh[threadIdx.x] + sh[threadIdx.x + 128];
    __syncthreads();
    double v = 0.0;
    if (threadIdx.x < 64) {
        v = sh[threadIdx.x] + sh[threadIdx.x + 64];
        for (int h = 32; h >= 1; h >>= 1) v = v + __shfl_down(v, h, 64);
    }
    return v;
}

// which of the visited neighbour cells (ascending CellId, as the neighbour search)
// of cell g map to stencil cell c of level 0: bit q = run q of every particle's list
__device__ inline unsigned galerkin_mask(const DevParams& P, const Level& L, const int* __restrict__ cellStart,
                                         int g, int c) {
    int gx, gy, gz;
    grid_xyz(L, g, gx, gy, gz);
    const int cx = gx + L.mn[0], cy = gy + L.mn[1], cz = gz + L.mn[2];
    unsigned mask = 0;
    const int* C = P.C;
    const int rx = P.range[0], ry = P.range[1], rz = P.range[2];
    // cells lie in [0, C), so their neighbours wrap without a division; so does the offset
    // on the level grid, unless the domain's wrap takes it further than one cell
    auto wrap = [](int v, int n) { return v < 0 ? v + n : v >= n ? v - n : v; };
    auto slot = [](int d, int n) { return d >= -1 && d <= 1 && n >= 3 ? d + 1 : (d + 1 + n) % n; };
    const int bx = (2 * rx) - wrap(cx + rx, C[0]), by = (2 * ry) - wrap(cy + ry, C[1]), bz = (2 * rz) - wrap(cz + rz, C[2]);
    const int x0 = bx > 0 ? bx : 0, y0 = by > 0 ? by : 0, z0 = bz > 0 ? bz : 0;
    const int nx = 2 * rx + 1, ny = 2 * ry + 1, nz = 2 * rz + 1;
    int q = 0;
    for (int a = x0; a < x0 + nx; ++a) {
        const int ax = wrap(cx - rx + (a >= nx ? a - nx : a), C[0]);
        const int ix = slot((ax - L.mn[0]) - gx, L.cnt[0]);
        for (int b = y0; b < y0 + ny; ++b) {
            const int ay = wrap(cy - ry + (b >= ny ? b - ny : b), C[1]);
            const int iy = slot((ay - L.mn[1]) - gy, L.cnt[1]);
            for (int cc = z0; cc < z0 + nz; ++cc, ++q) {
                const int az = wrap(cz - rz + (cc >= nz ? cc - nz : cc), C[2]);
                const int iz = slot((az - L.mn[2]) - gz, L.cnt[2]);
                const int jc = (ax * C[1] + ay) * C[2] + az;
                if (cellStart[jc] == cellStart[jc + 1]) continue;  // no fluid there
                if (L.cs[2] * L.cs[1] * ix + L.cs[2] * iy + iz == c) mask |= 1u << q;
            }
        }
    }
    return mask;
}

// galerkin_mask's q of cell g's own cell: the run that holds each of its particles'
// self entry
__device__ inline int galerkin_self(const DevParams& P, const Level& L, int g) {
    int gx, gy, gz;
    grid_xyz(L, g, gx, gy, gz);
    const int cx = gx + L.mn[0], cy = gy + L.mn[1], cz = gz + L.mn[2];
    const int* C = P.C;
    const int rx = P.range[0], ry = P.range[1], rz = P.range[2];
    const int nx = 2 * rx + 1, ny = 2 * ry + 1, nz = 2 * rz + 1;
    const int bx = (2 * rx) - (cx + rx) % C[0], by = (2 * ry) - (cy + ry) % C[1], bz = (2 * rz) - (cz + rz) % C[2];
    const int x0 = bx > 0 ? bx : 0, y0 = by > 0 ? by : 0, z0 = bz > 0 ? bz : 0;
    // the own cell is the one visited with offset index r (jx[r] = cx): a % n == r
    auto at = [](int r, int o, int n) { return ((r - o) % n + n) % n; };
    return (at(rx, x0, nx) * ny + at(ry, y0, ny)) * nz + at(rz, z0, nz);
}

// ---------------------------------------------------------------------------
// multigrid rows (preconditionWithMultiGrid)

// myDscal(0.0, S), myDcopy(Q, R), then myDdmv(1.0, invD, R, 1.0, S) on the same row.  S*0.0
// is a zero and Q is never -0 (a sum from +0), so S = invD Q is formed without the old S.
__device__ inline void mg_begin_update_row(const Level& L, int row, double r) {
    L.R[row] = r;
    double y = 0.0;
    y += 1.0 * L.invD[row] * r;
    lv_s(L, L.cur)[row] = y;
}

// (v mod n) for 0 <= v < 3n without a division
__device__ inline int wrap3(int v, int n) {
    v -= v >= n ? n : 0;
    v -= v >= n ? n : 0;
    return v;
}

// The sum over the 27-point (9 in 2D) block stencil of -1.0*a*x.  Ordered: in shift
// order, one chain of up to 81 dependent adds (about 24 cycles each).  Otherwise (the
// factored form, which keeps no bits of the reference): four chains over the stencil
// cells [uQ, (u+1)Q), Q = cells/4 rounded up, with fused multiply-adds, combined as
// (c0 + c1) + (c2 + c3); the lane-split sweeps give each lane one chain, so every kernel
// that takes such a sum gets the same bits.  Per sweep of a level of 4k rows 4.3 us
// against 4.8 us ordered, of the one-workgroup cycle 12.0 against 13.4 us (64k drop).
template <bool kOrd>
struct RowSum {
    double c[kOrd ? 1 : 4];
    __device__ inline RowSum() {
        for (double& v : c) v = 0.0;
    }
    // the three entries of stencil cell q of N
    __device__ inline void add(int q, int Q, double a, double x) {
        if constexpr (kOrd) c[0] += -1.0 * a * x;
        else {
            const int u = q / Q;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (u == k) c[k] = __builtin_fma(-a, x, c[k]);
        }
    }
    __device__ inline double total() const {
        if constexpr (kOrd) return c[0];
        else return (c[0] + c[1]) + (c[2] + c[3]);
    }
};
__host__ __device__ constexpr int row_chain(int cells) { return (cells + 3) / 4; }

// The wrapped neighbour index (g + e - 1 + cnt) % cnt of the reference's periodic
// stencil (main.cpp:3323-3325) is formed by subtraction (its argument is < 3 cnt).
// Full stencils (3x3x3, 3x3x1) take an unrolled path that issues the loads of nine
// cells at a time before summing them; smaller levels take the loop.
template <class VT, int C0, int C1, int C2, bool kOrd>
__device__ inline double mg_row_sum_full(const Level& L, const VT* __restrict__ A, const double* __restrict__ x,
                                         int row, int gx, int gy, int gz) {
    constexpr int N = C0 * C1 * C2;
    const int c0 = L.cnt[0], c1 = L.cnt[1], c2 = L.cnt[2];
    const long long nrow = L.nrow;
    int jx[C0], jy[C1], jz[C2];
#pragma unroll
    for (int e = 0; e < C0; ++e) jx[e] = wrap3(gx + e - 1 + c0, c0);
#pragma unroll
    for (int e = 0; e < C1; ++e) jy[e] = wrap3(gy + e - 1 + c1, c1);
#pragma unroll
    for (int e = 0; e < C2; ++e) jz[e] = wrap3(gz + e - 1 + c2, c2);
    RowSum<kOrd> sum;
#pragma unroll
    for (int q0 = 0; q0 < N; q0 += 9) {
        VT av[27];
        double xv[27];
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            const int q = q0 + t;
            if (q < N) {
                const int ex = q / (C1 * C2), ey = (q / C2) % C1, ez = q % C2;
                const double* xc = x + 3 * ((c1 * c2) * jx[ex] + c2 * jy[ey] + jz[ez]);
#pragma unroll
                for (int sd = 0; sd < 3; ++sd) {
                    av[3 * t + sd] = A[(3 * q + sd) * nrow + row];
                    xv[3 * t + sd] = xc[sd];
                }
            }
        }
#pragma unroll
        for (int t = 0; t < 9; ++t)
            if (q0 + t < N)
#pragma unroll
                for (int sd = 0; sd < 3; ++sd) sum.add(q0 + t, row_chain(N), (double)av[3 * t + sd], xv[3 * t + sd]);
    }
    return sum.total();
}

template <class VT, bool kOrd>
__device__ inline double mg_row_sum(const Level& L, const VT* __restrict__ A, const double* __restrict__ x, int row) {
    const int g = row / 3;
    int gx, gy, gz;
    grid_xyz(L, g, gx, gy, gz);
    if (L.cs[0] == 3 && L.cs[1] == 3 && L.cs[2] == 3)
        return mg_row_sum_full<VT, 3, 3, 3, kOrd>(L, A, x, row, gx, gy, gz);
    if (L.cs[0] == 3 && L.cs[1] == 3 && L.cs[2] == 1)
        return mg_row_sum_full<VT, 3, 3, 1, kOrd>(L, A, x, row, gx, gy, gz);
    const int c0 = L.cnt[0], c1 = L.cnt[1], c2 = L.cnt[2];
    const int nrow = L.nrow, Q = row_chain(L.cs[0] * L.cs[1] * L.cs[2]);
    const VT* a = A + row;  // entry sh of the row at a[sh * nrow]
    RowSum<kOrd> sum;
    int q = 0;
    for (int ex = 0; ex < L.cs[0]; ++ex) {
        const int jx = wrap3(gx + ex - 1 + c0, c0);
        for (int ey = 0; ey < L.cs[1]; ++ey) {
            const int jy = wrap3(gy + ey - 1 + c1, c1);
            const int bxy = (c1 * c2) * jx + c2 * jy;
            for (int ez = 0; ez < L.cs[2]; ++ez, ++q) {
                const int jz = wrap3(gz + ez - 1 + c2, c2);
                const double* xc = x + 3 * (bxy + jz);
                for (int sd = 0; sd < 3; ++sd, a += nrow) sum.add(q, Q, (double)a[0], xc[sd]);
            }
        }
    }
    return sum.total();
}

// myDcopy(Q, R); myDcsrmv(-1.0, A, S, 1.0, R)
template <class VT, bool kOrd>
__device__ inline void mg_residual_row(const Level& L, int row) {
    const VT* A = sizeof(VT) == 8 ? (const VT*)L.A : (const VT*)L.A32;
    const double sum = mg_row_sum<VT, kOrd>(L, A, lv_s(L, L.cur), row);
    double y = L.Q[row];
    y *= 1.0;
    y += sum;
    L.R[row] = y;
}

// residual then smoother update of the same row; the new iterate goes to the other
// S buffer so every thread still reads the old one
template <class VT, bool kOrd>
__device__ inline void mg_residual_update_row(const Level& L, int row) {
    const double* So = lv_s(L, L.cur);
    const VT* A = sizeof(VT) == 8 ? (const VT*)L.A : (const VT*)L.A32;
    const double sum = mg_row_sum<VT, kOrd>(L, A, So, row);
    double y = L.Q[row];
    y *= 1.0;
    y += sum;
    L.R[row] = y;
    double s = So[row];
    s *= 1.0;
    s += 1.0 * L.invD[row] * y;
    lv_s(L, L.cur ^ 1)[row] = s;
}

// The same sweeps with kRowLanes lanes per row, for levels too small to fill the GPU
// with one thread per row (a row's 81 loads are then latency-bound).  Lane u loads the
// entries of stencil cells [uQ, (u+1)Q).  Ordered: it forms their terms -1.0 a x and the
// row's first lane adds all terms in stencil order (the order of mg_row_sum), read back
// through LDS.  Otherwise each lane sums its own, one of RowSum's four chains.  So the
// sums are those of mg_residual_row and mg_residual_update_row either way.  Measured on
// a level of 73k rows, one thread per row is faster (12.4 against 18.6 us per ordered
// sweep, 12.1 against 15.5 us unordered); on levels of 10k rows and fewer the lanes take
// 20-30% off.  C0 C1 C2 give the stencil at compile time (3x3x3, 3x3x1); 0 0 0 reads it
// from the level (other shapes), at the price of runtime index arithmetic.
// t: the thread's number over the level's lanes; tb: kRowTerms doubles per thread of the
// workgroup (ordered only)
constexpr int kRowLanes = 4, kRowQ = 7;  // kRowQ: stencil cells per lane (27 / 4, rounded up)
constexpr int kRowTerms = 3 * kRowQ;

// the prolongation's value of level U for row rd of cell (gx, gy, gz) of level L (mg_prolong_row)
__device__ inline double mg_parent_value(const Level& U, const Level& L, int gx, int gy, int gz, int rd) {
    const int g = grid_id(U, ((gx + L.mn[0]) / 2) - U.mn[0], ((gy + L.mn[1]) / 2) - U.mn[1],
                          ((gz + L.mn[2]) / 2) - U.mn[2]);
    double sum = 0.0;
    sum += 1.0 * 1.0 * lv_s(U, U.cur)[3 * g + rd];
    return sum;
}

// lane u's part of the sum of `row`, for the four lanes of the row (on: it has one); the
// whole sum in its first lane.  kUp: on the iterate after the prolongation from U, formed
// as it is read (the same add as mg_prolong_row's); own: that of the row itself.
template <class VT, bool kOrd, bool kUp, int C0, int C1, int C2>
__device__ inline double mg_lanes_sum(const Level& L, const Level& U, int row, bool on, double* tb, double* own) {
    constexpr int T = kRowTerms;
    const int u = threadIdx.x & (kRowLanes - 1);
    const int cs1 = C0 ? C1 : L.cs[1], cs2 = C0 ? C2 : L.cs[2];
    const int N = (C0 ? C0 : L.cs[0]) * cs1 * cs2, Q = row_chain(N);  // N <= 27
    const VT* __restrict__ A = sizeof(VT) == 8 ? (const VT*)L.A : (const VT*)L.A32;
    const double* __restrict__ x = lv_s(L, L.cur);
    const long long nrow = L.nrow;
    double a[T], xv[T];
    if (on) {
        int gx, gy, gz;
        grid_xyz(L, row / 3, gx, gy, gz);
        const int c0 = L.cnt[0], c1 = L.cnt[1], c2 = L.cnt[2];
        double up[kUp ? T : 1];
#pragma unroll
        for (int k = 0; k < kRowQ; ++k) {
            const int q = u * Q + k;
            if (k < Q && q < N) {
                const int ex = q / (cs1 * cs2), ey = (q / cs2) % cs1, ez = q % cs2;
                const int jx = wrap3(gx + ex - 1 + c0, c0), jy = wrap3(gy + ey - 1 + c1, c1);
                const int jz = wrap3(gz + ez - 1 + c2, c2);
                const double* xc = x + 3 * ((c1 * c2) * jx + c2 * jy + jz);
#pragma unroll
                for (int sd = 0; sd < 3; ++sd) {
                    a[3 * k + sd] = (double)A[(3 * q + sd) * nrow + row];
                    xv[3 * k + sd] = xc[sd];
                    if constexpr (kUp) up[3 * k + sd] = mg_parent_value(U, L, jx, jy, jz, sd);
                }
            } else {
#pragma unroll
                for (int sd = 0; sd < 3; ++sd) {
                    a[3 * k + sd] = xv[3 * k + sd] = 0.0;
                    if constexpr (kUp) up[3 * k + sd] = 0.0;
                }
            }
        }
        if constexpr (kUp) {
            *own = x[row] + mg_parent_value(U, L, gx, gy, gz, row % 3);
#pragma unroll
            for (int e = 0; e < T; ++e) xv[e] += up[e];
        }
    } else {
#pragma unroll
        for (int e = 0; e < T; ++e) a[e] = xv[e] = 0.0;
    }
    double sum = 0.0;
    if constexpr (kOrd) {
#pragma unroll
        for (int e = 0; e < T; ++e) tb[T * threadIdx.x + e] = -1.0 * a[e] * xv[e];
        wave_sync();
        if (u == 0 && on)
            for (int v = 0; v < kRowLanes; ++v)
                for (int k = 0; k < Q && v * Q + k < N; ++k)
#pragma unroll
                    for (int sd = 0; sd < 3; ++sd) sum += tb[T * (threadIdx.x + v) + 3 * k + sd];
    } else {
#pragma unroll
        for (int e = 0; e < T; ++e) sum = __builtin_fma(-a[e], xv[e], sum);
        sum += __shfl_xor(sum, 1, 64);
        sum += __shfl_xor(sum, 2, 64);
    }
    return sum;
}

// kUp: the first sweep after the prolongation from U, whose launch it takes the place of
template <class VT, bool kUpdate, bool kOrd, bool kUp, int C0, int C1, int C2>
__device__ inline void mg_sweep_lanes(const Level& L, const Level& U, long long t, double* tb) {
    const int row = (int)(t / kRowLanes);
    const bool on = row < L.nrow;
    double own = 0.0;
    const double sum = mg_lanes_sum<VT, kOrd, kUp, C0, C1, C2>(L, U, row, on, tb, &own);
    if ((threadIdx.x & (kRowLanes - 1)) != 0 || !on) return;
    double y = L.Q[row];
    y *= 1.0;
    y += sum;
    L.R[row] = y;
    if (kUpdate) {
        double sv = kUp ? own : lv_s(L, L.cur)[row];
        sv *= 1.0;
        sv += 1.0 * L.invD[row] * y;
        lv_s(L, L.cur ^ 1)[row] = sv;
    }
}

// The residual of S (mg_residual_row), its restriction into L (mg_restrict_row), then
// begin and update of L: a group of 4 lanes per child (8 children, 4 where S is one cell
// deep in z, as in 2D) forms a coarse row's fine residuals, which are added in child
// order; a clipped child adds a zero, which changes no bit.  S.R is read by nothing else
// then and is not written.  One launch in the place of two of 3.8 and 4.6 us on the 64k
// drop.
template <int C0, int C2>
__host__ __device__ constexpr int restrict_lanes() { return kRowLanes * (C0 && C2 == 1 ? 4 : 8); }
template <class VT, bool kOrd, int C0, int C1, int C2>
__device__ inline void mg_residual_restrict_lanes(const Level& S, const Level& L, long long t, double* tb) {
    constexpr int G = restrict_lanes<C0, C2>(), KC = G / kRowLanes, KZ = KC / 4;
    const int lrow = (int)(t / G), c = (int)(t / kRowLanes) % KC, rd = lrow % 3;
    const bool own = lrow < L.nrow;
    int lx = 0, ly = 0, lz = 0;
    if (own) grid_xyz(L, lrow / 3, lx, ly, lz);
    const int fx = 2 * (lx + L.mn[0]) + c / (2 * KZ) - S.mn[0], fy = 2 * (ly + L.mn[1]) + (c / KZ) % 2 - S.mn[1];
    // KZ = 1: S is one cell deep in z, and that cell may be the coarse cell's second
    const int fz = KZ == 1 ? 0 : 2 * (lz + L.mn[2]) + c % KZ - S.mn[2];
    const bool on = own && fx >= 0 && fx < S.cnt[0] && fy >= 0 && fy < S.cnt[1] && fz >= 0 && fz < S.cnt[2];
    const int row = on ? 3 * grid_id(S, fx, fy, fz) + rd : 0;
    const double q = on ? S.Q[row] : 0.0;
    double y = mg_lanes_sum<VT, kOrd, false, C0, C1, C2>(S, S, row, on, tb, nullptr);
    y = on ? q * 1.0 + y : 0.0;
    double sum = 0.0;
    const int l0 = (int)(threadIdx.x & 63) & ~(G - 1);
#pragma unroll
    for (int k = 0; k < KC; ++k) sum += 1.0 * 1.0 * __shfl(y, l0 + kRowLanes * k, 64);
    if ((int)(threadIdx.x & 63) != l0 || !own) return;
    L.Q[lrow] = sum;  // Q*0.0 is a zero, the sum never -0
    mg_begin_update_row(L, lrow, sum);
}

// restriction (R of 3115-3175): Q_L = 0*Q_L + sum of the clipped 2x2x2 children of R_S,
// returned
__device__ inline double mg_restrict_row(const Level& S, const Level& L, int row) {
    const int g = row / 3, rd = row % 3;
    int lx, ly, lz;
    grid_xyz(L, g, lx, ly, lz);
    const int lcx = lx + L.mn[0], lcy = ly + L.mn[1], lcz = lz + L.mn[2];
    const int fmx = S.mn[0] > 2 * lcx, fmy = S.mn[1] > 2 * lcy, fmz = S.mn[2] > 2 * lcz;
    const int fMx = S.mx[0] < 2 * (lcx + 1), fMy = S.mx[1] < 2 * (lcy + 1), fMz = S.mx[2] < 2 * (lcz + 1);
    double sum = 0.0;
    for (int ax = 0; ax < 2 - fmx - fMx; ++ax)
        for (int ay = 0; ay < 2 - fmy - fMy; ++ay)
            for (int az = 0; az < 2 - fmz - fMz; ++az) {
                const int sg = grid_id(S, (2 * lcx + ax + fmx) - S.mn[0], (2 * lcy + ay + fmy) - S.mn[1],
                                       (2 * lcz + az + fmz) - S.mn[2]);
                sum += 1.0 * 1.0 * S.R[3 * sg + rd];
            }
    L.Q[row] = sum;  // Q*0.0 is a zero, the sum never -0
    return sum;
}

// prolongation (P of 3216-3241): S_S += injection of the parent's S_L
__device__ inline void mg_prolong_row(const Level& L, const Level& S, int row) {
    const int g = row / 3, rd = row % 3;
    int sx, sy, sz;
    grid_xyz(S, g, sx, sy, sz);
    const int lg = grid_id(L, ((sx + S.mn[0]) / 2) - L.mn[0], ((sy + S.mn[1]) / 2) - L.mn[1],
                           ((sz + S.mn[2]) / 2) - L.mn[2]);
    double sum = 0.0;
    sum += 1.0 * 1.0 * lv_s(L, L.cur)[3 * lg + rd];
    double* Sv = lv_s(S, S.cur);
    double y = Sv[row];
    y *= 1.0;
    y += sum;
    Sv[row] = y;
}

// Levels lc..D-1 of the V-cycle inside ONE workgroup, in the order of
// preconditionWithMultiGrid (4160-4255) for those levels: restriction into lc, the
// down sweep (S = invD R, then residual-update sweeps and a residual per level), the
// coarsest level (S = invD R, then four residual-update sweeps), the up sweep and the
// prolongations back into lc-1.  With lc = 0 the whole hierarchy is here: Q0 comes
// from the P2G launch and S0 goes back for the G2P.
//
// Every row of every fused level is owned by one thread for the whole cycle, which
// keeps the row's stencil values, its smoother weight, Q and S in registers; S and R
// go through LDS, a workgroup barrier after every sweep.  The rows' values and places
// are laid out per thread once per multigrid build (coarse_pack), so the cycle starts
// with one round of coalesced loads, all in flight together (2.3-3.4 us), and a sweep
// is 27 LDS reads and a chain of 81 ordered adds per row (9 and 27 in 2D).  The chain
// bounds it: about 24 cycles per add, 0.9 us per 3D sweep.  Measured per cycle, ordered
// and in chains: 13.4 and 12.0 us on the 64k-particle drop (320 threads), 14.0 and 14.3 us
// on the 1M-particle scene (256), 13.3 and 12.4 us on a 2D pool of 4,100 (448).
// Re-reading the stencils through L2 in every sweep, three dependent rounds of loads
// each, took 47.7, 63.9 and 60.4 us ordered.
//
// Invalid cells of a stencil narrower than 3 along an axis are padded with a zero
// value and the row's own cell: they add a zero, which changes no bit of a sum that
// starts at +0.  S*0.0 and Q*0.0 of the reference are zeros and are not formed.

// The per-thread layout: value k of thread t at v[k*stride + t] (3N stencil values, then
// invD; NaN-free zeros for threads without a row), int m of thread t at i[m*stride + t]:
// (N+1)/2 pairs of 16-bit LDS places of the stencil cells, then the meta words below;
// up[r] = the LDS place of the parent of row r of level lc-1.
enum { kCmLevel = 0, kCmChild = 1, kCmSx = 2, kCmSy = 3, kCmParent = 4, kCmShape = 5, kCmWords = 6 };

__device__ inline void coarse_pack(const Level* __restrict__ lvs, int lc, int D, bool f32, const CoarsePack& K) {
    const int N = K.cells, NZ = N / 9, tid = threadIdx.x + blockIdx.x * blockDim.x;
    if (lc > 0) {
        const Level &L = lvs[lc], &F = lvs[lc - 1];
        for (int r = tid; r < F.nrow; r += gridDim.x * blockDim.x) {
            int fx, fy, fz;
            grid_xyz(F, r / 3, fx, fy, fz);
            K.up[r] = 3 * grid_id(L, ((fx + F.mn[0]) / 2) - L.mn[0], ((fy + F.mn[1]) / 2) - L.mn[1],
                                  ((fz + F.mn[2]) / 2) - L.mn[2]) + r % 3;
        }
    }
    if (tid >= K.stride) return;
    int myl = -1, row = 0, base = 0, down = 0, upb = 0;  // first LDS places: own, finer, coarser level
    for (int l = lc, b = 0, bp = 0; l < D; ++l) {
        const int n = lvs[l].nrow;
        if (tid >= b && tid < b + n) {
            myl = l;
            row = tid - b;
            base = b;
            down = l == lc ? 0 : bp;
            upb = b + n;
        }
        bp = b;
        b += n;
    }
    int* const im = K.i + (long long)((N + 1) / 2) * K.stride + tid;
    im[kCmLevel * K.stride] = myl;
    if (myl < 0) {
        for (int k = 0; k <= 3 * N; ++k) K.v[(long long)k * K.stride + tid] = 0.0;
        for (int m = 0; m < (N + 1) / 2; ++m) K.i[m * K.stride + tid] = 0;
        for (int m = 1; m < kCmWords; ++m) im[m * K.stride] = 0;
        return;
    }
    const Level& L = lvs[myl];
    const int g = row / 3, rd = row % 3;
    int gx, gy, gz;
    grid_xyz(L, g, gx, gy, gz);
    int lo = 0;
    const bool half = f32 && L.A32;
    for (int k0 = 0; k0 < N; k0 += 9) {  // nine cells' values in flight
        double v[27];
        long long at[27];
        bool in[9];
#pragma unroll
        for (int u = 0; u < 9; ++u) {
            const int k = k0 + u, ex = k / (3 * NZ), ey = (k / NZ) % 3, ez = k % NZ;
            in[u] = ex < L.cs[0] && ey < L.cs[1] && ez < L.cs[2];
            const long long sh = in[u] ? 3 * ((L.cs[1] * ex + ey) * L.cs[2] + ez) : 0;
            for (int sd = 0; sd < 3; ++sd) at[3 * u + sd] = (sh + sd) * L.nrow + row;
            const int jx = wrap3(gx + ex - 1 + L.cnt[0], L.cnt[0]), jy = wrap3(gy + ey - 1 + L.cnt[1], L.cnt[1]);
            const int jz = NZ == 1 ? 0 : wrap3(gz + ez - 1 + L.cnt[2], L.cnt[2]);
            const int pl = base + 3 * (in[u] ? grid_id(L, jx, jy, jz) : g);
            if (k & 1) K.i[(k / 2) * K.stride + tid] = lo | (pl << 16);
            else lo = pl;
        }
        if (half) {
#pragma unroll
            for (int e = 0; e < 27; ++e) v[e] = (double)L.A32[at[e]];
        } else {
#pragma unroll
            for (int e = 0; e < 27; ++e) v[e] = L.A[at[e]];
        }
#pragma unroll
        for (int e = 0; e < 27; ++e) K.v[(long long)(3 * k0 + e) * K.stride + tid] = in[e / 3] ? v[e] : 0.0;
    }
    if (N & 1) K.i[(N / 2) * K.stride + tid] = lo;
    K.v[(long long)(3 * N) * K.stride + tid] = L.invD[row];
    int child = 0, sx = 0, sy = 0, shape = 0, parent = 0;
    if (myl > 0) {  // the clipped 2x2x2 children (mg_restrict_row)
        const Level& F = lvs[myl - 1];
        const int x = gx + L.mn[0], y = gy + L.mn[1], z = gz + L.mn[2];
        const int fmx = F.mn[0] > 2 * x, fmy = F.mn[1] > 2 * y, fmz = F.mn[2] > 2 * z;
        const int nx = 2 - fmx - (F.mx[0] < 2 * (x + 1)), ny = 2 - fmy - (F.mx[1] < 2 * (y + 1));
        const int nz = 2 - fmz - (F.mx[2] < 2 * (z + 1));
        shape = nx | (ny << 2) | (nz << 4);
        child = down + 3 * grid_id(F, (2 * x + fmx) - F.mn[0], (2 * y + fmy) - F.mn[1], (2 * z + fmz) - F.mn[2]) + rd;
        sx = 3 * F.cnt[1] * F.cnt[2];
        sy = 3 * F.cnt[2];
    }
    if (myl + 1 < D) {  // the parent (mg_prolong_row)
        const Level& U = lvs[myl + 1];
        parent = upb + 3 * grid_id(U, ((gx + L.mn[0]) / 2) - U.mn[0], ((gy + L.mn[1]) / 2) - U.mn[1],
                                   ((gz + L.mn[2]) / 2) - U.mn[2]) + rd;
    }
    im[kCmChild * K.stride] = child;
    im[kCmSx * K.stride] = sx;
    im[kCmSy * K.stride] = sy;
    im[kCmParent * K.stride] = parent;
    im[kCmShape * K.stride] = shape;
}

template <int T>
struct CoarseShared {
    double S[2][T], R[T];
};

// K: the packed levels lc..D-1; in: R of level lc-1 (Q of level 0 when lc = 0); io: S of
// level lc-1, which the prolongation updates (of level 0 when lc = 0, written); nio: its
// rows; plain: io is S of level lc, written in the place of that prolongation.
// XB: stencil cells whose LDS reads are in flight together.  halt: the CR stop
// flag or null, tested once the loads are under way.
template <int N, int T, int XB, bool kOrd>
__device__ inline void mg_coarse_cycle(const CoarsePack& K, int lc, int D, const double* __restrict__ in, double* io,
                                       int nio, bool plain, const int* halt, CoarseShared<T>& sh) {
    const int tid = threadIdx.x, st = K.stride;
    double a[3 * N], w, q = 0.0, s = 0.0;
    int po[(N + 1) / 2];  // pairs of LDS places
    // uniform bases and one lane offset
    auto value = [&](int k) { return (K.v + (long long)k * st)[(unsigned)tid]; };
    auto word = [&](int m) { return (K.i + (long long)m * st)[(unsigned)tid]; };
    constexpr int M = (N + 1) / 2;
    const int myl = word(M + kCmLevel), child = word(M + kCmChild), sx = word(M + kCmSx), sy = word(M + kCmSy);
    const int parent = word(M + kCmParent), shape = word(M + kCmShape);
    w = value(3 * N);
#pragma unroll
    for (int k = 0; k < M; ++k) po[k] = word(k);
#pragma unroll
    for (int k = 0; k < 3 * N; ++k) a[k] = value(k);
    auto children = [&](const double* R) {  // mg_restrict_row
        double v[8], sum = 0.0;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const bool on = (k >> 2) < (shape & 3) && ((k >> 1) & 1) < ((shape >> 2) & 3) && (k & 1) < (shape >> 4);
            v[k] = on ? R[(k >> 2) * sx + ((k >> 1) & 1) * sy + (k & 1) * 3] : 0.0;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) sum += 1.0 * 1.0 * v[k];
        return sum;
    };
    if (myl == lc) q = lc == 0 ? in[tid] : children(in + child);
    if (cr_halted(halt)) return;
    auto row_sum = [&](const double* x) {  // mg_row_sum
        // XB cells' LDS reads are under way while the XB before them are added
        RowSum<kOrd> sum;
        double xv[2][3 * XB];
        auto read = [&](int k0, double* v) {
#pragma unroll
            for (int u = 0; u < XB; ++u)
                if (k0 + u < N) {
                    const int k = k0 + u;
                    unsigned pl = po[k / 2];
                    asm volatile("" : "+v"(pl));  // unpacked here, not kept in 27 registers over the sweeps
                    const double* xc = x + (k & 1 ? pl >> 16 : pl & 0xffff);
#pragma unroll
                    for (int sd = 0; sd < 3; ++sd) v[3 * u + sd] = xc[sd];
                }
        };
        read(0, xv[0]);
#pragma unroll
        for (int k0 = 0; k0 < N; k0 += XB) {
            const int h = (k0 / XB) & 1;
            if (k0 + XB < N) read(k0 + XB, xv[h ^ 1]);
            asm volatile("" : : : "memory");  // the reads stay above, the adds below
#pragma unroll
            for (int u = 0; u < XB; ++u)
                if (k0 + u < N)
#pragma unroll
                    for (int sd = 0; sd < 3; ++sd) sum.add(k0 + u, row_chain(N), a[3 * (k0 + u) + sd], xv[h][3 * u + sd]);
#pragma unroll
            for (double& c : sum.c) asm volatile("" : "+v"(c) : : "memory");
        }
        return sum.total();
    };
    unsigned pc = 0;  // the S buffer of the own level
    auto sweeps = [&](int l, int n) {  // n residual-update sweeps of level l
        for (int k = 0; k < n; ++k) {
            if (myl == l) {
                double y = q;
                y *= 1.0;
                y += row_sum(sh.S[pc]);
                s *= 1.0;
                s += 1.0 * w * y;
                pc ^= 1;
                sh.S[pc][tid] = s;
            }
            __syncthreads();
        }
    };
    for (int l = lc; l < D; ++l) {
        if (myl == l) {  // restriction, then begin and update
            if (l > lc) {
                int c = child;
                asm volatile("" : "+v"(c));  // the places are formed here, not kept over the sweeps
                q = children(sh.R + c);
            }
            s += 1.0 * w * q;
            sh.S[0][tid] = s;
        }
        __syncthreads();
        sweeps(l, l == D - 1 ? 4 : l == 0 ? 1 : 2);
        if (l < D - 1) {
            if (myl == l) {
                double y = q;
                y *= 1.0;
                y += row_sum(sh.S[pc]);
                sh.R[tid] = y;
            }
            __syncthreads();
        }
    }
    // a level's S ends in buffer 0 after four sweeps (the coarsest), in 1 after five (or
    // three, level 0)
    for (int l = D - 2; l >= lc; --l) {
        if (myl == l) {
            double sum = 0.0;
            sum += 1.0 * 1.0 * sh.S[l + 1 == D - 1 ? 0 : 1][parent];
            s *= 1.0;
            s += sum;
            sh.S[pc][tid] = s;
        }
        __syncthreads();
        sweeps(l, l == 0 ? 2 : 3);
    }
    if (lc == 0) {
        if (myl == 0) io[tid] = s;
    } else {
        const double* x = sh.S[lc == D - 1 ? 0 : 1];
        if (plain) {
            if (myl == lc) io[tid] = s;
            return;
        }
        for (int r = tid; r < nio; r += st) {
            double sum = 0.0;
            sum += 1.0 * 1.0 * x[K.up[r]];
            double y = io[r];
            y *= 1.0;
            y += sum;
            io[r] = y;
        }
    }
}

// u = D^-1 q (4144-4148) + G2P S0 (4260), and the chunk partial of q.u (when part)
__device__ inline void mg_g2p_chunk(const DevParams& P, const Level& L, const int* __restrict__ cellIndex,
                                    const double* __restrict__ invDiagA, const double* __restrict__ q,
                                    double* __restrict__ u, double* __restrict__ part, int chunk, double* sh) {
    const int i = chunk * 256 + threadIdx.x;
    double t = 0.0;
    if (i < P.nf) {
        const int key = cellIndex[i];
        const int cx = key / (P.C[1] * P.C[2]) % P.C[0], cy = key / (P.C[2]) % P.C[1], cz = key % P.C[2];
        const int g = grid_id(L, cx - L.mn[0], cy - L.mn[1], cz - L.mn[2]);
        const double* S0 = lv_s(L, L.cur);
        double uu[3], qq[3], z[3], c[3];
        for (int r = 0; r < 3; ++r) {
            qq[r] = q[3 * i + r];
            z[r] = 1.0 * invDiagA[3 * i + r] * qq[r];
            c[r] = S0[3 * g + r];
        }
        // y = u*0.0 + D^-1 q: the zero only matters for the sign of a zero product
        if (z[0] == 0.0 || z[1] == 0.0 || z[2] == 0.0)
            for (int r = 0; r < 3; ++r) z[r] += u[3 * i + r] * 0.0;
        for (int r = 0; r < 3; ++r) {
            double sum = 0.0;
            sum += 1.0 * 1.0 * c[r];
            double y = z[r];
            y *= 1.0;
            y += sum;
            uu[r] = y;
            u[3 * i + r] = y;
        }
        t = (qq[0] * uu[0] + qq[1] * uu[1]) + qq[2] * uu[2];
    }
    if (part) {
        const double v = block_tree_sum(t, sh);
        if (threadIdx.x == 0) part[chunk] = v;
    }
}

// ---------------------------------------------------------------------------
// conjugate residual (solveWithConjugatedGradient, 4270-4421)

// initial guess x = v - F/m dt (4299-4309)
__device__ inline void cr_init_particle(const DevParams& P, const double* __restrict__ vel,
                                        const double* __restrict__ force, const double* __restrict__ mass,
                                        double* __restrict__ x, int i) {
    for (int d = 0; d < 3; ++d) x[3 * i + d] = vel[3 * i + d] - force[3 * i + d] / mass[i] * P.dt;
}

// The tail of every particle-matrix product, given particle i's row sums (s0, s1,
// s2): y = beta*yin + sum (the sum formed first, as myDcsrmvForA), optional second
// output y2 = beta*y2 + sum, optional copy p = x, and the chunk partial of dotx.y.
// Every thread of the workgroup calls it (i >= nf: no row).
__device__ inline void spmv_store(int nf, int i, double s0, double s1, double s2, const double* __restrict__ x,
                                  double beta, const double* yin, double* y, double* y2, double* p_copy,
                                  const double* __restrict__ dotx, double* __restrict__ part, int chunk,
                                  double* sh) {
    double t = 0.0;
    if (i < nf) {
        const double sm[3] = {s0, s1, s2};
        double out[3];
        for (int r = 0; r < 3; ++r) {
            double yy = yin[3 * i + r];
            yy *= beta;
            yy += sm[r];
            out[r] = yy;
        }
        if (y2)
            for (int r = 0; r < 3; ++r) {
                double yy = y2[3 * i + r];
                yy *= beta;
                yy += sm[r];
                y2[3 * i + r] = yy;
            }
        for (int r = 0; r < 3; ++r) y[3 * i + r] = out[r];
        if (p_copy)
            for (int r = 0; r < 3; ++r) p_copy[3 * i + r] = x[3 * i + r];
        if (part) {
            const double d0 = dotx[3 * i], d1 = dotx[3 * i + 1], d2 = dotx[3 * i + 2];
            t = (d0 * out[0] + d1 * out[1]) + d2 * out[2];
        }
    }
    if (part) {
        const double v = block_tree_sum(t, sh);
        if (threadIdx.x == 0) part[chunk] = v;
    }
}

// element k of y (and y2) from the row's sum sm, as spmv_store: the separate
// roundings of y = beta*yin + sum (compiled without contraction); yv and y2v are yin[k]
// and y2[k], read before
__device__ inline void store1(int k, double sm, double yv, double y2v, double beta, double* y, double* y2) {
    double yy = yv;
    yy *= beta;
    yy += sm;
    if (y2) {
        double zz = y2v;
        zz *= beta;
        zz += sm;
        y2[k] = zz;
    }
    y[k] = yy;
}

// y = beta*yin + sum_k (alpha*a_k)*x_k over the sliced A (myDcsrmvForA, 4033-4050);
// alpha is +1 or -1, so alpha*a is exact and is applied as a sign.  Optional second
// output y2 = beta*y2 + sum (same sum), optional copy p = x, and the chunk partial
// of dotx.y.  One chunk = 4 slices = 256 particles.  The row sums run over the
// blocks in list order, entries s = 0,1,2 within a block, as the CSR.
template <bool kNeg, class VT, int kUn>
__device__ inline void spmv_chunk(int nf, const int* __restrict__ nFluid, const long long* __restrict__ start,
                                  const int* __restrict__ col, const VT* __restrict__ val,
                                  const double* __restrict__ x, double beta, const double* yin, double* y,
                                  double* y2, double* p_copy, const double* __restrict__ dotx,
                                  double* __restrict__ part, int chunk, double* sh) {
    typedef int it2 __attribute__((ext_vector_type(2)));
    const int i = chunk * 256 + threadIdx.x;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
    if (i < nf) {
        const int w = nFluid[i];
        const int lane = i % kSlice;
        const long long sb = start[i / kSlice];
        // the matrix is read once per launch: streaming (nontemporal) loads of whole
        // block pairs (FP64, a_val_index) or quads (FP32, a_val32_index), kUn of them
        // per group with all their loads issued before the first use; columns are
        // pairs (a_col_index)
        const it2* cp = (const it2*)col + (sb / 2) * kSlice + lane;
        auto block = [&](int j, const double* c9) {
            const double x0 = x[3 * j], x1 = x[3 * j + 1], x2 = x[3 * j + 2];
            double c[9];
#pragma unroll
            for (int e = 0; e < 9; ++e) c[e] = kNeg ? -c9[e] : c9[e];
            s0 += c[0] * x0; s0 += c[1] * x1; s0 += c[2] * x2;
            s1 += c[3] * x0; s1 += c[4] * x1; s1 += c[5] * x2;
            s2 += c[6] * x0; s2 += c[7] * x1; s2 += c[8] * x2;
        };
        if constexpr (sizeof(VT) == 8) {
            typedef VT vt2 __attribute__((ext_vector_type(2)));
            const vt2* vp = (const vt2*)val + (sb / 2) * 9 * kSlice + lane;
            auto pair = [&](const it2 j, const vt2* a, int h) {  // blocks 2m, 2m+1 (h of them)
                for (int u = 0; u < h; ++u) {
                    double c9[9];
#pragma unroll
                    for (int e = 0; e < 9; ++e) c9[e] = (double)a[e][u];
                    block(j[u], c9);
                }
            };
            const int wp = w / 2;
            int m = 0;
            for (; m + kUn <= wp; m += kUn) {
                it2 j[kUn];
                vt2 a[kUn][9];
#pragma unroll
                for (int u = 0; u < kUn; ++u) j[u] = __builtin_nontemporal_load(cp + (long long)(m + u) * kSlice);
#pragma unroll
                for (int u = 0; u < kUn; ++u)
#pragma unroll
                    for (int e = 0; e < 9; ++e)
                        a[u][e] = __builtin_nontemporal_load(vp + ((long long)(m + u) * 9 + e) * kSlice);
#pragma unroll
                for (int u = 0; u < kUn; ++u) pair(j[u], a[u], 2);
            }
            for (; m <= wp; ++m) {  // the last full pairs, then the odd last block
                const int h = (m < wp) ? 2 : (w & 1);
                if (h == 0) break;
                const it2 j = __builtin_nontemporal_load(cp + (long long)m * kSlice);
                vt2 a[9];
#pragma unroll
                for (int e = 0; e < 9; ++e) a[e] = __builtin_nontemporal_load(vp + ((long long)m * 9 + e) * kSlice);
                pair(j, a, h);
            }
        } else {
            typedef VT vt4 __attribute__((ext_vector_type(4)));
            const vt4* vp = (const vt4*)val + (sb / 4) * 9 * kSlice + lane;
            auto quad = [&](const it2 j0, const it2 j1, const vt4* a, int h) {  // blocks 4q..4q+h-1
                for (int u = 0; u < h; ++u) {
                    double c9[9];
#pragma unroll
                    for (int e = 0; e < 9; ++e) c9[e] = (double)a[e][u];
                    block(u < 2 ? j0[u] : j1[u - 2], c9);
                }
            };
            const int wq = w / 4;
            int q = 0;
            for (; q + kUn <= wq; q += kUn) {
                it2 j[kUn][2];
                vt4 a[kUn][9];
#pragma unroll
                for (int u = 0; u < kUn; ++u) {
                    j[u][0] = __builtin_nontemporal_load(cp + (long long)(2 * (q + u)) * kSlice);
                    j[u][1] = __builtin_nontemporal_load(cp + (long long)(2 * (q + u) + 1) * kSlice);
                }
#pragma unroll
                for (int u = 0; u < kUn; ++u)
#pragma unroll
                    for (int e = 0; e < 9; ++e)
                        a[u][e] = __builtin_nontemporal_load(vp + ((long long)(q + u) * 9 + e) * kSlice);
#pragma unroll
                for (int u = 0; u < kUn; ++u) quad(j[u][0], j[u][1], a[u], 4);
            }
            for (; q <= wq; ++q) {  // the last full quads, then the partial last one
                const int h = (q < wq) ? 4 : (w & 3);
                if (h == 0) break;
                const it2 j0 = __builtin_nontemporal_load(cp + (long long)(2 * q) * kSlice);
                const it2 j1 = __builtin_nontemporal_load(cp + (long long)(2 * q + 1) * kSlice);
                vt4 a[9];
#pragma unroll
                for (int e = 0; e < 9; ++e) a[e] = __builtin_nontemporal_load(vp + ((long long)q * 9 + e) * kSlice);
                quad(j0, j1, a, h);
            }
        }
    }
    spmv_store(nf, i, s0, s1, s2, x, beta, yin, y, y2, p_copy, dotx, part, chunk, sh);
}

// The same product for scenes of few slices, a wavefront per component of a slice's
// rows (workgroup `slice` of three wavefronts): a row's three sums are independent, so
// each keeps its order of summation.  One wavefront per slice had 18 KB in flight against
// about 2 us of latency, and a scene of 9k particles has 144 slices for 256 CUs.  Rounds
// of 8 blocks are pipelined: the values and x of the next round and the columns of the
// one after it load while a round is added.  The matrix of such a scene stays in the
// caches, so its loads are not marked nontemporal.
// 9k particles in 3D: 89 us per product with a wavefront per slice, 32 us now (116 MB,
// 3.6 TB/s); 4.1k in 2D: 19.1 and 8.8 us.
template <bool kNeg, class VT>
__device__ inline void spmv_split(int nf, const int* __restrict__ nFluid, const long long* __restrict__ start,
                                  const int* __restrict__ col, const VT* __restrict__ val,
                                  const double* __restrict__ x, double beta, const double* yin, double* y,
                                  double* y2, double* p_copy, int slice) {
    constexpr int V = 16 / sizeof(VT), B = 8, U = B / V;  // blocks per 16-byte load, per round; loads per entry
    typedef int it2 __attribute__((ext_vector_type(2)));
    typedef VT vt __attribute__((ext_vector_type(V)));
    const int lane = threadIdx.x & 63, r = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int i = slice * kSlice + lane;
    const long long sb = start[slice];
    const int slots = (int)(start[slice + 1] - sb), rounds = (slots + B - 1) / B;  // slots: a multiple of 4
    const int w = i < nf ? nFluid[i] : 0;
    const it2* cp = (const it2*)col + (sb / 2) * kSlice + lane;
    const vt* vp = (const vt*)val + (sb / V) * 9 * kSlice + 3 * r * kSlice + lane;
    struct Round {
        vt a[U][3];
        double xv[B][3];
    };
    // past the slice's slots the last ones load again; past the row, particle 0's x
    auto columns = [&](int k0, it2* j) {
#pragma unroll
        for (int q = 0; q < B / 2; ++q) {
            const int m = k0 / 2 + q < slots / 2 ? k0 / 2 + q : slots / 2 - 1;
            j[q] = cp[(long long)m * kSlice];
        }
    };
    auto operands = [&](int k0, const it2* j, Round& o) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int m = k0 / V + u < slots / V ? k0 / V + u : slots / V - 1;
#pragma unroll
            for (int e = 0; e < 3; ++e) o.a[u][e] = vp[((long long)m * 9 + e) * kSlice];
        }
#pragma unroll
        for (int q = 0; q < B; ++q) {
            const long long j3 = 3 * (long long)(k0 + q < w ? j[q / 2][q & 1] : 0);
#pragma unroll
            for (int e = 0; e < 3; ++e) o.xv[q][e] = x[j3 + e];
        }
    };
    double s = 0.0;
    if (rounds > 0) {
        it2 j[B / 2];
        Round cur;
        columns(0, j);
        operands(0, j, cur);
        columns(B, j);
        for (int n = 0; n < rounds; ++n) {
            const int k0 = B * n;
            Round next;
            operands(k0 + B, j, next);
            columns(k0 + 2 * B, j);
#pragma unroll
            for (int q = 0; q < B; ++q) {
                double t = s;
#pragma unroll
                for (int e = 0; e < 3; ++e) {
                    const double c = (double)cur.a[q / V][e][q % V];
                    t += (kNeg ? -c : c) * cur.xv[q][e];
                }
                s = k0 + q < w ? t : s;
            }
            cur = next;
        }
    }
    if (i < nf) {
        const int k = 3 * i + r;
        store1(k, s, yin[k], y2 ? y2[k] : 0.0, beta, y, y2);
        if (p_copy) p_copy[k] = x[k];
    }
}

// ---------------------------------------------------------------------------
// the particle matrix in factored form (FacOp; the derivation is at the top of
// mph_factored.hip).  Not bit-identical to the assembled product: the same sums,
// associated differently, with multiply-adds contracted.  Both passes give each particle a group of G lanes
// (kFacLanes) that walk its neighbour list together: the list is in
// cell order, so the group's column and scalar loads are coalesced and its
// gathers of neighbours' records mostly hit consecutive records; each lane keeps a
// batch of entries in flight.  The group's partial sums are combined by a
// butterfly, in the same order for every launch.

// minimum-image displacement pos_j - pos_i (the reference's Mod form, used where
// the scalars are built); j's coordinates are loaded before the first min_image,
// whose branch would otherwise hold each load back until the previous one is done
__device__ inline void fac_disp(const DevParams& P, const double* __restrict__ pos, int j, double pi0, double pi1,
                                double pi2, double& r0, double& r1, double& r2) {
    const double x = pos[3 * j], y = pos[3 * j + 1], z = pos[3 * j + 2];
    r0 = min_image(x, pi0, P.W[0], P.hW[0]);
    r1 = min_image(y, pi1, P.W[1], P.hW[1]);
    r2 = min_image(z, pi2, P.W[2], P.hW[2]);
}

// the same displacement for the products: positions lie inside the domain, so one
// wrap by the domain width gives the minimum image (equal to the Mod form up to
// rounding).  Only scenes with pairs across the periodic boundary (FacOp::wrap)
// take it; the others use the plain difference (kWrap false).
template <bool kWrap>
__device__ inline double fac_wrap(double r, double w, double hw) {
    if (!kWrap) return r;
    return r > hw ? r - w : (r < -hw ? r + w : r);
}

// sum over the G lanes of each aligned group (G a power of two, <= 64); every lane
// of the wavefront calls it
__device__ inline double group_sum(double v, int G) {
    for (int m = G >> 1; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    return v;
}

// a row's sum s plus component r of its diagonal term, D_r . x_i + C_ii,r t_i, with
// the fused multiply-adds written out: every kernel of the factored product that
// forms it (whichever lane does) gets the same bits
__device__ inline double fac_diag_add(double s, double dr0, double dr1, double dr2, double x0, double x1, double x2,
                                      double c, double t) {
    double d = __builtin_fma(dr0, x0, dr1 * x1);
    d = __builtin_fma(dr2, x2, d);
    d = __builtin_fma(c, t, d);
    return s + d;
}

// one entry of FacOp::u32 / v32: three floats and the column
struct FacEntry32 {
    float a0, a1, a2;
    int col;
};
__device__ inline FacEntry32 fac_entry32(const float* __restrict__ base, long long e) {
    typedef float fv4 __attribute__((ext_vector_type(4)));
    const fv4 v = ((const fv4*)base)[e];
    return {v[0], v[1], v[2], __float_as_int(v[3])};
}

// 1/sqrt(v), v >= 1e-200, by the hardware's estimate (about 2^-24) and one step of third
// order: within 2 ulp
__device__ inline double rsqrt_ref(double v) {
    const double y = __builtin_amdgcn_rsq(v);
    const double e = __builtin_fma(-(v * y), y, 1.0);
    return __builtin_fma(y * e, __builtin_fma(0.375, e, 0.5), y);
}

// one fluid-neighbour entry of the second pass: adds (beta t - alpha r.x) r for the
// displacement r.  The scalars come from the distance, alpha = facV (1/d - invV)+ / d^2
// and beta = facP (1/d - invP)+ (DevParams; (.)+ clamps at 0, so the radii need no
// test); their constants are in the operands: x is -facV x, t is facP t.  At r = 0 (the
// row's own entry, the padding of a list, a coincident particle) everything is 0.
// kVar: fluid pairs of several viscosities, alpha is the stored a and x is plain.
// Written in explicit fused operations: every kernel that forms it gets the same bits.
template <bool kVar>
__device__ inline void fac_pair(const DevParams& P, double r0, double r1, double r2, double x0, double x1, double x2,
                                double t, double a, double& s0, double& s1, double& s2) {
    const double d2 = __builtin_fmax(__builtin_fma(r2, r2, __builtin_fma(r1, r1, r0 * r0)), 1.0e-200);
    const double y = rsqrt_ref(d2);
    const double dot = __builtin_fma(r2, x2, __builtin_fma(r1, x1, r0 * x0));
    double f;
    if (kVar) f = -(a * dot);
    else f = (__builtin_fmax(y - P.invV, 0.0) * (y * y)) * dot;
    f = __builtin_fma(__builtin_fmax(y - P.invP, 0.0), t, f);
    s0 = __builtin_fma(f, r0, s0);
    s1 = __builtin_fma(f, r1, s1);
    s2 = __builtin_fma(f, r2, s2);
}

// list entries each lane of a second-pass row has in flight per batch; the FP32 form's
// lanes per particle in both passes and entries in flight (viscous and P entries)
constexpr int kFacBatch = 4, kFacLanes32 = 8, kFacBatch32 = 8, kFacBatchP = 4;
// the first pass (k's P list up to its last fluid entry, about 20 entries): lanes per
// particle and entries in flight per lane, at six waves per SIMD (126 us on the 1M
// scene; 160 us before beta was recomputed and, with rows in series, 132 us where 8 in
// flight at their three waves took 140 us)
constexpr int kFacLanesT = 4, kFacBatchT = 4;
static_assert(kFacRowsT == 256 / kFacLanesT && kFacRowsY == 256 / kFacLanes && kFacRowsY == 256 / kFacLanes32, "");

// the four planes of FacOp::rec
struct FacPlanes {
    double* a;  // [np][2] x0 x1
    double* b;  // [np][2] x2 p0
    double* c;  // [np][2] p1 p2
    double* t;  // [np]
};
__device__ inline FacPlanes fac_planes(const DevParams& P, double* rec) {
    const long long n = P.np;
    return {rec, rec + 2 * n, rec + 4 * n, rec + 6 * n};
}

// first pass over the 256 particles of `chunk` (fluid or wall):
//   t_k = lambda_k (C_kk . x_k [k fluid] - sum_{j fluid, j != k} beta_kj r_kj . x_j),
// written to k's record together with x_k (fluid k).  Every thread calls it.
// beta is recomputed from the distance, as in fac_pair.  (Streaming a stored v = beta r
// instead of gathering positions measured slower: as many load instructions, more bytes.)
template <bool kWrap>
__device__ inline void fac_t_chunk(const DevParams& P, const FacOp& F, const double* __restrict__ x, int chunk) {
#pragma clang fp contract(fast)
    constexpr int G = kFacLanesT, U = kFacBatchT;
    const int g = threadIdx.x & (G - 1);
    const double W0 = P.W[0], W1 = P.W[1], W2 = P.W[2], h0 = P.hW[0], h1 = P.hW[1], h2 = P.hW[2];
    const int k = chunk * kFacRowsT + threadIdx.x / G;
    double acc = 0.0;
    const int run = k < P.np ? F.runP[k] : 0;
    if (run > 0) {
        const double pk0 = F.pos[3 * k], pk1 = F.pos[3 * k + 1], pk2 = F.pos[3 * k + 2];
        const long long c0 = F.nPtrP[k];
        for (int jb = 0; jb < run; jb += G * U) {
            int jx[U];
            bool use[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                // entries past the end load the run's last entry (run >= 1), so the
                // list loads need no branches and issue together
                const int jn = jb + g + u * G;
                const int je = F.nIndP[c0 + (jn < run ? jn : run - 1)];
                use[u] = jn < run && je < P.nf && je != k;
                jx[u] = use[u] ? je : 0;  // unused entries read particle 0 with weight 0
            }
            double v[U][6];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const long long j3 = 3 * (long long)jx[u];
                v[u][0] = F.pos[j3];
                v[u][1] = F.pos[j3 + 1];
                v[u][2] = F.pos[j3 + 2];
                v[u][3] = x[j3];
                v[u][4] = x[j3 + 1];
                v[u][5] = x[j3 + 2];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const double r0 = fac_wrap<kWrap>(v[u][0] - pk0, W0, h0);
                const double r1 = fac_wrap<kWrap>(v[u][1] - pk1, W1, h1);
                const double r2 = fac_wrap<kWrap>(v[u][2] - pk2, W2, h2);
                const double d2 = __builtin_fmax((r0 * r0 + r1 * r1) + r2 * r2, 1.0e-200);
                const double b = use[u] ? __builtin_fmax(rsqrt_ref(d2) - P.invP, 0.0) : 0.0;
                acc -= b * ((r0 * v[u][3] + r1 * v[u][4]) + r2 * v[u][5]);
            }
        }
        acc *= P.facP;
    }
    acc = group_sum(acc, G);
    if (g == 0 && k < P.np) {
        const FacPlanes R = fac_planes(P, F.rec);
        if (k < P.nf) {
            const double x0 = x[3 * k], x1 = x[3 * k + 1], x2 = x[3 * k + 2];
            acc += (F.selfC[3 * k] * x0 + F.selfC[3 * k + 1] * x1) + F.selfC[3 * k + 2] * x2;
            R.a[2 * k] = x0;
            R.a[2 * k + 1] = x1;
            R.b[2 * k] = x2;
        }
        R.t[k] = run > 0 ? acc * F.lambda[k] : 0.0;
    }
}

// the C Lambda C^T terms of row i's wall neighbours (the P entries after the fluid
// ones), one entry per lane and round; adds to the lane's sums
template <bool kWrap>
__device__ inline void fac_walls(const DevParams& P, const FacOp& F, const double* __restrict__ rt, int i, int g,
                                 double pi0, double pi1, double pi2, double& s0, double& s1, double& s2) {
    const double W0 = P.W[0], W1 = P.W[1], W2 = P.W[2], h0 = P.hW[0], h1 = P.hW[1], h2 = P.hW[2];
    const long long c0 = F.nPtrP[i];
    const int n = F.nCountP[i];
    for (int jn = F.runP[i] + g; jn < n; jn += kFacLanes) {
        const int k = F.nIndP[c0 + jn];
        const double f = F.beta[c0 + jn] * rt[k];
        const double r0 = fac_wrap<kWrap>(F.pos[3 * (long long)k] - pi0, W0, h0);
        const double r1 = fac_wrap<kWrap>(F.pos[3 * (long long)k + 1] - pi1, W1, h1);
        const double r2 = fac_wrap<kWrap>(F.pos[3 * (long long)k + 2] - pi2, W2, h2);
        s0 = __builtin_fma(f, r0, s0);
        s1 = __builtin_fma(f, r1, s1);
        s2 = __builtin_fma(f, r2, s2);
    }
}

// row i's sum over its fluid neighbours with every record gathered through the caches
// (the chunk kernel, and cells with more records than the staging holds): lane g takes
// entries g, g + 8, ... in order, as the staged walk does
template <bool kWrap, bool kVar>
__device__ inline void fac_row_gather(const DevParams& P, const FacOp& F, int i, int g, double pi0, double pi1,
                                      double pi2, double& s0, double& s1, double& s2) {
    typedef double dv2 __attribute__((ext_vector_type(2)));
    constexpr int G = kFacLanes, U = kFacBatch;
    const FacPlanes R = fac_planes(P, F.rec);
    const dv2* __restrict__ ra = (const dv2*)R.a;
    const dv2* __restrict__ rb = (const dv2*)R.b;
    const dv2* __restrict__ rc = (const dv2*)R.c;
    const double* __restrict__ rt = R.t;
    const double* __restrict__ alpha = (const double*)F.alpha;
    const double W0 = P.W[0], W1 = P.W[1], W2 = P.W[2], h0 = P.hW[0], h1 = P.hW[1], h2 = P.hW[2];
    const double sx = kVar ? 1.0 : -P.facV;
    const long long b0 = F.nPtr[i];
    const int w = F.nFluid[i];
    for (int jb = 0; jb < w; jb += G * U) {
        int j[U];
        double a[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int jn = jb + g + u * G;
            const long long e = b0 + (jn < w ? jn : w - 1);
            j[u] = F.nInd[e];
            a[u] = kVar ? alpha[e] : 0.0;
            if (jn >= w) {  // past the list: the row's own record adds nothing
                j[u] = i;
                a[u] = 0.0;
            }
        }
        dv2 q0[U], q1[U], q2[U];
        double q3[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            q0[u] = ra[j[u]];
            q1[u] = rb[j[u]];
            q2[u] = rc[j[u]];
            q3[u] = rt[j[u]];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const double r0 = fac_wrap<kWrap>(q1[u][1] - pi0, W0, h0);
            const double r1 = fac_wrap<kWrap>(q2[u][0] - pi1, W1, h1);
            const double r2 = fac_wrap<kWrap>(q2[u][1] - pi2, W2, h2);
            fac_pair<kVar>(P, r0, r1, r2, sx * q0[u][0], sx * q0[u][1], sx * q1[u][0], P.facP * q3[u], a[u], s0, s1,
                           s2);
        }
    }
}

// second pass over the kFacRowsY fluid rows of `chunk`, eight lanes a row:
//   y_i = D_i x_i + C_ii t_i - sum_j alpha_ij r_ij (r_ij . x_j) + sum_{k != i} beta_ik r_ik t_k,
// a fluid neighbour's alpha and beta terms added together (fac_pair); then the tail of
// spmv_store, one component to each of three lanes.
template <bool kNeg, bool kWrap, bool kVar>
__device__ inline void fac_y_chunk(const DevParams& P, const FacOp& F, const double* __restrict__ x, double beta,
                                   const double* yin, double* y, double* y2, double* p_copy, int chunk) {
    constexpr int G = kFacLanes;
    const int g = threadIdx.x & (G - 1);
    const double* __restrict__ rt = fac_planes(P, F.rec).t;
    const int i = chunk * kFacRowsY + threadIdx.x / G;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
    if (i < P.nf) {
        const double pi0 = F.pos[3 * i], pi1 = F.pos[3 * i + 1], pi2 = F.pos[3 * i + 2];
        fac_row_gather<kWrap, kVar>(P, F, i, g, pi0, pi1, pi2, s0, s1, s2);
        fac_walls<kWrap>(P, F, rt, i, g, pi0, pi1, pi2, s0, s1, s2);
    }
    s0 = group_sum(s0, G);
    s1 = group_sum(s1, G);
    s2 = group_sum(s2, G);
    if (g < 3 && i < P.nf) {
        const int k = 3 * i + g;
        const double* D = F.diag + 9 * i + 3 * g;
        const double sg = fac_diag_add(g == 0 ? s0 : g == 1 ? s1 : s2, D[0], D[1], D[2], x[3 * i], x[3 * i + 1],
                                       x[3 * i + 2], F.selfC[k], rt[i]);
        store1(k, kNeg ? -sg : sg, yin[k], y2 ? y2[k] : 0.0, beta, y, y2);
        if (p_copy) p_copy[k] = x[k];
    }
}

// the variant of fac_y_chunk that the scene's flags ask for (uniform)
template <bool kNeg>
__device__ inline void fac_y_chunk_any(const DevParams& P, const FacOp& F, const double* __restrict__ x, double beta,
                                       const double* yin, double* y, double* y2, double* p_copy, int chunk) {
#define MPH_Y(WRAP, VAR) fac_y_chunk<kNeg, WRAP, VAR>(P, F, x, beta, yin, y, y2, p_copy, chunk)
    const int wrap = F.wrap[0], var = F.wrap[1];
    if (!wrap && !var) MPH_Y(false, false);
    else if (!var) MPH_Y(true, false);
    else MPH_Y(true, true);  // the wrapped displacement of a pair inside the domain is the plain one
#undef MPH_Y
}

// FP32 form of the two passes (mixed-precision inner solves): the displacements are
// folded into the stored vectors (v_kj = beta_kj r_kj, u_ij = sqrt(alpha_ij) r_ij),
// so a pass gathers only a neighbour's 16-byte record (x, t as floats).  Arithmetic
// is FP64 on the FP32-stored values.
__device__ inline void fac_t32_chunk(const DevParams& P, const FacOp& F, const double* __restrict__ x, int chunk) {
#pragma clang fp contract(fast)
    constexpr int G = kFacLanes32, U = kFacBatchP;
    typedef float fv4 __attribute__((ext_vector_type(4)));
    const int g = threadIdx.x & (G - 1);
    const int k = chunk * kFacRowsY + threadIdx.x / G;
    double acc = 0.0;
    const int run = k < P.np ? F.runP[k] : 0;
    if (run > 0) {
        const long long c0 = F.nPtrP[k];
        for (int jb = 0; jb < run; jb += G * U) {
            int jx[U];
            float v[U][3];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int jn = jb + g + u * G;
                const FacEntry32 en = fac_entry32(F.v32, c0 + (jn < run ? jn : 0));
                const int j = jn < run ? en.col : k;
                const bool use = jn < run && j < P.nf && j != k;
                jx[u] = use ? j : 0;  // unused entries read particle 0 with weight 0
                v[u][0] = use ? en.a0 : 0.0f;
                v[u][1] = use ? en.a1 : 0.0f;
                v[u][2] = use ? en.a2 : 0.0f;
            }
            double xv[U][3];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const long long j3 = 3 * (long long)jx[u];
                xv[u][0] = x[j3];
                xv[u][1] = x[j3 + 1];
                xv[u][2] = x[j3 + 2];
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                acc -= ((double)v[u][0] * xv[u][0] + (double)v[u][1] * xv[u][1]) + (double)v[u][2] * xv[u][2];
        }
    }
    acc = group_sum(acc, G);
    if (g == 0 && k < P.np) {
        fv4 rk = {0.0f, 0.0f, 0.0f, 0.0f};
        if (k < P.nf) {
            const double x0 = x[3 * k], x1 = x[3 * k + 1], x2 = x[3 * k + 2];
            acc += (F.selfC[3 * k] * x0 + F.selfC[3 * k + 1] * x1) + F.selfC[3 * k + 2] * x2;
            rk[0] = (float)x0;
            rk[1] = (float)x1;
            rk[2] = (float)x2;
        }
        rk[3] = run > 0 ? (float)(acc * F.lambda[k]) : 0.0f;
        ((fv4*)F.rec32)[k] = rk;
    }
}

template <bool kNeg>
__device__ inline void fac_y32_chunk(const DevParams& P, const FacOp& F, const double* __restrict__ x, double beta,
                                     const double* yin, double* y, double* y2, double* p_copy, int chunk) {
#pragma clang fp contract(fast)
    typedef float fv4 __attribute__((ext_vector_type(4)));
    constexpr int G = kFacLanes32, U = kFacBatch32;
    const int g = threadIdx.x & (G - 1);
    const fv4* __restrict__ rec = (const fv4*)F.rec32;
    const int i = chunk * kFacRowsY + threadIdx.x / G;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
    if (i < P.nf) {
        // viscous part: -u (u . x_j).  Software-pipelined: the columns and u of the next
        // batch load while the current batch's records are gathered
        struct Batch {
            int j[U];
            float a[U][3];
        };
        const long long b0 = F.nPtr[i];
        const int w = F.nFluid[i];
        auto vload = [&](int jb, Batch& b) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int jn = jb + g + u * G;
                const bool in = jn < w;
                const FacEntry32 en = fac_entry32(F.u32, b0 + (in ? jn : 0));
                b.j[u] = in ? en.col : i;  // unused entries: i's own record, u = 0
                b.a[u][0] = in ? en.a0 : 0.0f;
                b.a[u][1] = in ? en.a1 : 0.0f;
                b.a[u][2] = in ? en.a2 : 0.0f;
            }
        };
        Batch nb;
        vload(0, nb);
        for (int jb = 0; jb < w; jb += G * U) {
            const Batch cb = nb;
            fv4 q[U];
#pragma unroll
            for (int u = 0; u < U; ++u) q[u] = rec[cb.j[u]];
            if (jb + G * U < w) vload(jb + G * U, nb);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const double a0 = cb.a[u][0], a1 = cb.a[u][1], a2 = cb.a[u][2];
                const double f = (a0 * (double)q[u][0] + a1 * (double)q[u][1]) + a2 * (double)q[u][2];
                s0 -= f * a0;
                s1 -= f * a1;
                s2 -= f * a2;
            }
        }
        // C Lambda C^T part: v_ik t_k
        const long long c0 = F.nPtrP[i];
        const int n = F.nCountP[i];
        for (int jb = 0; jb < n; jb += G * kFacBatchP) {
            constexpr int U = kFacBatchP;
            int k[U];
            float vv[U][3];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int jn = jb + g + u * G;
                const bool in = jn < n;
                const FacEntry32 en = fac_entry32(F.v32, c0 + (in ? jn : 0));
                k[u] = in ? en.col : i;
                vv[u][0] = in ? en.a0 : 0.0f;
                vv[u][1] = in ? en.a1 : 0.0f;
                vv[u][2] = in ? en.a2 : 0.0f;
            }
            fv4 q[U];
#pragma unroll
            for (int u = 0; u < U; ++u) q[u] = rec[k[u]];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const double t = q[u][3];
                s0 += (double)vv[u][0] * t;
                s1 += (double)vv[u][1] * t;
                s2 += (double)vv[u][2] * t;
            }
        }
    }
    s0 = group_sum(s0, G);
    s1 = group_sum(s1, G);
    s2 = group_sum(s2, G);
    if (g < 3 && i < P.nf) {
        const int k = 3 * i + g;
        const double* D = F.diag + 9 * i + 3 * g;
        double d = (D[0] * x[3 * i] + D[1] * x[3 * i + 1]) + D[2] * x[3 * i + 2];
        d += F.selfC[k] * (double)rec[i][3];
        const double sg = (g == 0 ? s0 : g == 1 ? s1 : s2) + d;
        store1(k, kNeg ? -sg : sg, yin[k], y2 ? y2[k] : 0.0, beta, y, y2);
        if (p_copy) p_copy[k] = x[k];
    }
}

// chunk partial of x.y: per particle (x0 y0 + x1 y1) + x2 y2, then the chunk tree
__device__ inline void dot_partial_chunk(int nf, const double* __restrict__ x, const double* __restrict__ y,
                                         double* __restrict__ part, int chunk, double* sh) {
    const int i = chunk * 256 + threadIdx.x;
    double t = 0.0;
    if (i < nf) t = (x[3 * i] * y[3 * i] + x[3 * i + 1] * y[3 * i + 1]) + x[3 * i + 2] * y[3 * i + 2];
    const double v = block_tree_sum(t, sh);
    if (threadIdx.x == 0) part[chunk] = v;
}

// lane l's sum of the chunk partials l, l + 256, ... from 0.0 in that order; eight loads
// are issued before their adds so the lane does not wait on each in turn
__device__ inline double dot_lane_sum(const double* __restrict__ part, int nchunks) {
    double acc = 0.0;
    for (int c0 = threadIdx.x; c0 < nchunks; c0 += 256 * 8) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = c0 + 256 * u < nchunks ? part[c0 + 256 * u] : 0.0;
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (c0 + 256 * u < nchunks) acc = acc + v[u];
    }
    return acc;
}

// fold the chunk partials: the lanes' sums, then the tree.
// scal[shift_slot] receives the previous scal[slot] first (rho -> rho_prev).
__device__ inline void dot_final_body(const double* __restrict__ part, int nchunks, double* scal, int slot,
                                      int shift_slot, double* sh, double* host = nullptr) {
    const double v = block_tree_sum(dot_lane_sum(part, nchunks), sh);
    if (threadIdx.x == 0) {
        if (shift_slot >= 0) scal[shift_slot] = scal[slot];
        scal[slot] = v;
        if (host) *host = v;  // coherent pinned host memory: the CR stop test reads it
    }
}

// The same dot product in every thread of a workgroup that needs it (sh: 257 doubles), so
// that a later iteration of a scene of up to kFoldChunks chunks launches no reduction of
// rho and tmp: the P2G folds rho's partials and keeps it in scal[kRHON] beside the previous
// rho in scal[kRHO], the x update folds tmp's, and the reduction of rr, which comes after
// both, moves scal[kRHON] to scal[kRHO].
__device__ inline double dot_fold(const double* __restrict__ part, int nchunks, double* sh) {
    const double v = block_tree_sum(dot_lane_sum(part, nchunks), sh);
    if (threadIdx.x == 0) sh[256] = v;
    __syncthreads();
    return sh[256];
}
__device__ inline void dot_shift_rho(double* scal) {
    scal[kRHOP] = scal[kRHO];
    scal[kRHO] = scal[kRHON];
}

// p = beta*p + 1.0*s, q = beta*q + 1.0*y with beta = rho/rho_prev (4360-4364)
// one element of p = beta p + s or q = beta q + y (myDscal then myDaxpy, 4362-4366),
// with the same roundings in every kernel that forms it
__device__ inline double pq_elem(double beta, double v, double w) {
    v *= beta;
    v += 1.0 * w;
    return v;
}

// P2G (2964-2997), then begin + update of level 0 on the same row, with kP2gLanes lanes
// per row: level 0 has one row per cell and component, too few to fill the GPU with one
// thread each.  Lane u loads q of the cell's particles p0 + u, p0 + u + kP2gLanes, ...
// (kP2gK per pass).  Ordered: the row's first lane adds them in particle order from
// LDS.  Otherwise each lane adds its own and a butterfly the lanes' sums.  kPq: the CR
// loop's q = beta q + y (4364-4366) is formed here as q is loaded and written back
// (every fluid particle lies in exactly one level-0 cell, so each element is updated
// once); q is written only then.  tb: 256 * kP2gK doubles of LDS (ordered only).
// Unordered, with the update, 19.5 us on the 1M scene (72 MB, 3.7 TB/s) and 6.1 us on
// the 64k drop; ordered 21.5 and 9.4 us, bound by the first lane's chain of adds.
constexpr int kP2gLanes = 8, kP2gK = 8;
// coef(): beta, called by every thread of the workgroup (kPq only)
template <bool kPq, bool kOrd, class F>
__device__ inline void mg_p2g_lanes(const DevParams& P, const Level& L, const int* __restrict__ cellStart, double* q,
                                    const double* __restrict__ yv, F coef, int block, double* tb) {
    const int u = threadIdx.x & (kP2gLanes - 1);
    const int row = (int)(((long long)block * 256 + threadIdx.x) / kP2gLanes);
    const bool on = row < L.nrow;
    int p0 = 0, p1 = 0;
    const int rd = row % 3;
    if (on) {
        int gx, gy, gz;
        grid_xyz(L, row / 3, gx, gy, gz);
        const int ic = cell_id(P, gx + L.mn[0], gy + L.mn[1], gz + L.mn[2]);
        p0 = cellStart[ic];
        p1 = cellStart[ic + 1];
    }
    const double beta = kPq ? coef() : 0.0;
    double sum = 0.0;
    for (int base = p0; base < p1; base += kP2gLanes * kP2gK) {  // the same trips in every lane of the row
        double t[kP2gK], yt[kP2gK];
#pragma unroll
        for (int k = 0; k < kP2gK; ++k) {
            const int ip = base + u + kP2gLanes * k;
            t[k] = ip < p1 ? q[3 * ip + rd] : 0.0;
            yt[k] = kPq && ip < p1 ? yv[3 * ip + rd] : 0.0;
        }
#pragma unroll
        for (int k = 0; k < kP2gK; ++k) {
            const int ip = base + u + kP2gLanes * k;
            if (kPq && ip < p1) {
                t[k] = pq_elem(beta, t[k], yt[k]);
                q[3 * ip + rd] = t[k];
            }
        }
        if constexpr (kOrd) {
#pragma unroll
            for (int k = 0; k < kP2gK; ++k) tb[kP2gK * threadIdx.x + k] = t[k];
            wave_sync();
            if (u == 0)
                for (int k = 0; k < kP2gK; ++k)
                    for (int v = 0; v < kP2gLanes; ++v)
                        if (base + v + kP2gLanes * k < p1) sum += 1.0 * 1.0 * tb[kP2gK * (threadIdx.x + v) + k];
            wave_sync();
        } else {
#pragma unroll
            for (int k = 0; k < kP2gK; ++k) sum += t[k];
        }
    }
    if constexpr (!kOrd)
        for (int m = 1; m < kP2gLanes; m <<= 1) sum += __shfl_xor(sum, m, 64);
    if (u != 0 || !on) return;
    L.Q[row] = sum;  // Q*0.0 is a zero, the sum never -0
    mg_begin_update_row(L, row, sum);
}

__device__ inline void pq_update_elem(const double* __restrict__ scal, const double* __restrict__ s,
                                      const double* __restrict__ y, double* __restrict__ p, double* __restrict__ q,
                                      long long k) {
    const double beta = scal[kRHO] / scal[kRHOP];
    p[k] = pq_elem(beta, p[k], s[k]);
    q[k] = pq_elem(beta, q[k], y[k]);
}

// alpha = rho/tmp; x += alpha p; r -= alpha q; s -= alpha u (4372-4375) + r.r partial.
// kPq: p = beta p + s first (with s before its update), written back; the CR loop's
// p update is then this kernel's, not a launch of its own
// coef(alpha, beta): called by every thread of the workgroup, the vectors' loads under way
template <bool kPq, class F>
__device__ inline void xrs_update_chunk(int nf, F coef, double* __restrict__ p,
                                        const double* __restrict__ q, const double* __restrict__ u,
                                        double* __restrict__ x, double* __restrict__ r, double* __restrict__ s,
                                        double* __restrict__ part, int chunk, double* sh) {
    const int i = chunk * 256 + threadIdx.x;
    double t = 0.0;
    double pv[3], qv[3], uv[3], xv[3], rv[3], sv[3], alpha, beta;
    if (i < nf)
        for (int d = 0; d < 3; ++d) {
            const int k = 3 * i + d;
            pv[d] = p[k];
            sv[d] = s[k];
            xv[d] = x[k];
            rv[d] = r[k];
            qv[d] = q[k];
            uv[d] = u[k];
        }
    coef(alpha, beta);
    if (i < nf) {
        const double ma = -alpha;
        double rr[3];
        for (int d = 0; d < 3; ++d) {
            const int k = 3 * i + d;
            if (kPq) {
                pv[d] = pq_elem(beta, pv[d], sv[d]);
                p[k] = pv[d];
            }
            x[k] = xv[d] + alpha * pv[d];
            rr[d] = rv[d] + ma * qv[d];
            r[k] = rr[d];
            s[k] = sv[d] + ma * uv[d];
        }
        t = (rr[0] * rr[0] + rr[1] * rr[1]) + rr[2] * rr[2];
    }
    const double v = block_tree_sum(t, sh);
    if (threadIdx.x == 0) part[chunk] = v;
}

}  // namespace body
}  // namespace mph
