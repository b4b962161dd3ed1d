// mph_factored.hip -- the particle matrix of the implicit solve applied in factored
// form, reading one scalar per stored block instead of nine.
//
// calculateMatrixA and multiplyMatrixC (source/main.cpp:2137-2336, 2562-2644) build,
// for fluid particles i and fluid neighbours j != i,
//   A_ij = -alpha_ij r_ij r_ij^T + sum_k C_ik lambda_k C_jk^T
//   A_ii = D_i + sum_k C_ik lambda_k C_ik^T,  D_i = V_i + m_i/(V dt) I
// where r_ij is the minimum-image displacement pos_j - pos_i, and:
//   - alpha_ij = visc mu_ij (-w_v'(d))/d^3 for 0 < d < RadiusV, 0 otherwise. The
//     viscous coefficient visc mu_ij e_s e_r (-w_v'(d))/d of main.cpp:2279-2288,
//     with e = r/d.
//   - V_i = sum_j alpha_ij r_ij r_ij^T over every neighbour, walls included. This is
//     the viscous self block, main.cpp:2290.
//   - C_ik = beta_ik r_ik, with beta_ik = -w_p'(d)/d for 0 < d < RadiusP. This is
//     C's entry e (-w_p'(d)) of main.cpp:2479-2493.
//   - C_ii = sum_k C_ik (main.cpp:2497-2504).
//   - k runs over the RadiusP neighbours shared by i and j, fluid or wall.
// So A x needs only alpha per A slot, beta per P-list entry, D and C_ii:
//   t_k = lambda_k sum_{j fluid, k in P(j)} C_jk . x_j        (every particle k)
//   (A x)_i = D_i x_i - sum_j alpha_ij r_ij (r_ij . x_j) + C_ii t_i + sum_{k != i} C_ik t_k
// The first pass sums over k's own P list, using C_jk = -beta_kj r_kj.  That holds
// because the RadiusP relation is symmetric up to rounding in the distance.
//
// The product is the assembled one up to rounding: the same terms, associated
// differently.  alpha and beta are functions of the distance alone where one viscosity
// fills the scene (FacOp::wrap[1] = 0), so the FP64 passes recompute them from the
// positions with a few fused operations (body::fac_pair) and read 2 to 4 bytes per
// neighbour where the assembled product reads 76.  A neighbour's x, position and t come
// from planes of 16-byte pairs (FacOp::rec), staged per cell in LDS or gathered through
// the caches.  Each row is walked by a group of 8 lanes, so that the reads of one load
// instruction fall on consecutive particles of the cell-ordered list.
//
// Scenes whose multigrid levels allow it assemble no 3x3 blocks at all: level 0
// and InvDiagA come from the same scalars (k_fac_g, k_fac_gal0, k_fac_invdiag).
#include "mph_batch.h"
#include "mph_cr_body.h"

namespace mph {
namespace {

using body::nblk;

// beta beside the P lists (and v = beta r in FP32 for the FP32 form), the extent of
// their fluid entries, C_ii of fluid particles, and the records (positions; x and t
// zero until the first pass)
__global__ void __launch_bounds__(256) k_fac_p(DevParams P, const double* __restrict__ pos,
                                               const int* __restrict__ nCountP, const long long* __restrict__ nPtrP,
                                               const int* __restrict__ nIndP, double* __restrict__ beta,
                                               float* __restrict__ v32, int* __restrict__ runP,
                                               double* __restrict__ selfC, double* __restrict__ rec) {
    // entry-parallel: lane g handles entries g, g + 8, ... (beta, v); the group's
    // first lane adds the C_ii terms in list order and finds the fluid extent
    constexpr int G = 8, K = 3;
    __shared__ double tb[256 * K];
    __shared__ int tf[256];  // bit 0: inside RadiusP (a C_ii term), bit 1: fluid neighbour
    const int g = threadIdx.x & (G - 1);
    const int k = (int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) / G);
    const bool own = k < P.np;
    const long long b0 = own ? nPtrP[k] : 0;
    const int n = own ? nCountP[k] : 0;
    const double pk0 = own ? pos[3 * k] : 0.0, pk1 = own ? pos[3 * k + 1] : 0.0, pk2 = own ? pos[3 * k + 2] : 0.0;
    double c0 = 0.0, c1 = 0.0, c2 = 0.0;
    int run = 0;
    for (int base = 0; base < n; base += G) {
        const int jn = base + g;
        int f = 0;
        double t[K] = {0.0, 0.0, 0.0};
        if (jn < n) {
            const int j = nIndP[b0 + jn];
            double b = 0.0, r0 = 0.0, r1 = 0.0, r2 = 0.0;
            if (j != k) {
                body::fac_disp(P, pos, j, pk0, pk1, pk2, r0, r1, r2);
                const double r2s = (r0 * r0 + r1 * r1 + r2 * r2);
                if (r2s != 0.0 && P.radP2 - r2s > 0) {
                    const double d = sqrt(r2s);
                    b = -dwq_k(P.Kp, P.m2P, d, P.radP) / d;
                    t[0] = b * r0;
                    t[1] = b * r1;
                    t[2] = b * r2;
                    f = 1;
                }
            }
            if (j < P.nf) f |= 2;
            beta[b0 + jn] = b;
            if (v32) {
                typedef float fv4 __attribute__((ext_vector_type(4)));
                ((fv4*)v32)[b0 + jn] = fv4{(float)(b * r0), (float)(b * r1), (float)(b * r2), __int_as_float(j)};
            }
        }
        for (int e = 0; e < K; ++e) tb[K * threadIdx.x + e] = t[e];
        tf[threadIdx.x] = f;
        wave_sync();
        if (g == 0)
            for (int u = 0; u < G && base + u < n; ++u) {
                const int sl = threadIdx.x + u;
                const int fu = tf[sl];
                if (fu & 1) {
                    c0 += tb[K * sl];
                    c1 += tb[K * sl + 1];
                    c2 += tb[K * sl + 2];
                }
                if (fu & 2) run = base + u + 1;
            }
        wave_sync();
    }
    if (g != 0 || !own) return;
    runP[k] = run;
    const body::FacPlanes R = body::fac_planes(P, rec);
    R.a[2 * k] = 0.0;
    R.a[2 * k + 1] = 0.0;
    R.b[2 * k] = 0.0;
    R.b[2 * k + 1] = pk0;
    R.c[2 * k] = pk1;
    R.c[2 * k + 1] = pk2;
    R.t[k] = 0.0;
    if (k < P.nf) {
        selfC[3 * k] = c0;
        selfC[3 * k + 1] = c1;
        selfC[3 * k + 2] = c2;
    }
}

// u = sqrt(alpha) r per fluid-neighbour entry of fluid rows, eight lanes per row
// (coalesced writes beside the list)
__global__ void __launch_bounds__(256) k_fac_u(DevParams P, const int* __restrict__ nFluid,
                                               const long long* __restrict__ nPtr, const int* __restrict__ nInd,
                                               const double* __restrict__ alpha, const double* __restrict__ pos,
                                               float* __restrict__ u32) {
    constexpr int G = 8;
    const int g = threadIdx.x & (G - 1);
    const int i = (blockIdx.x * blockDim.x + threadIdx.x) / G;
    if (i >= P.nf) return;
    const double pi0 = pos[3 * i], pi1 = pos[3 * i + 1], pi2 = pos[3 * i + 2];
    const long long b0 = nPtr[i];
    const int w = nFluid[i];
    for (int jn = g; jn < w; jn += G) {
        const int j = nInd[b0 + jn];
        double r0, r1, r2;
        body::fac_disp(P, pos, j, pi0, pi1, pi2, r0, r1, r2);
        const double s = sqrt(alpha[b0 + jn]);  // alpha >= 0: visc, mu and -w' are not negative
        typedef float fv4 __attribute__((ext_vector_type(4)));
        ((fv4*)u32)[b0 + jn] = fv4{(float)(s * r0), (float)(s * r1), (float)(s * r2), __int_as_float(j)};
    }
}

// ---------------------------------------------------------------------------
// Multigrid level 0 and the particle-level inverse diagonal from the factored form,
// so a factored scene never assembles the 3x3 blocks.  Level 0 of
// calculateMultiGridCsrA (main.cpp:3336-3410) is, for row cell g and stencil cell h,
//   A0(g, h) = sum_{i in g} sum_{j in h} A_ij
//            = sum_{i in g} [D_i if h = g] - sum_{i in g, j in h, j != i} alpha_ij r r^T
//              + sum_k lambda_k G_gk G_hk^T,     G_gk = sum_{i in g, k in P(i)} C_ik,
// k over every particle with fluid P neighbours in both cells.  A particle's P
// neighbours lie in its own or the adjacent cells (cells are at least MaxRadius >=
// 2 RadiusP wide), so G_k is a 27-slot table around k's cell.

// slot of cell (tx, ty, tz) in the 3x3x3 block around (kx, ky, kz), -1 if outside
__device__ inline int fac_slot(const DevParams& P, int tx, int ty, int tz, int kx, int ky, int kz) {
    int d[3] = {tx - kx, ty - ky, tz - kz};
    for (int a = 0; a < 3; ++a) {
        if (d[a] > 1) d[a] -= P.C[a];
        if (d[a] < -1) d[a] += P.C[a];
        if (d[a] < -1 || d[a] > 1) return -1;
    }
    return 9 * (d[0] + 1) + 3 * (d[1] + 1) + (d[2] + 1);
}

__device__ inline void cell_xyz(const DevParams& P, int key, int& x, int& y, int& z) {
    const int c = key % P.T;  // wall keys carry +T
    x = c / (P.C[1] * P.C[2]);
    y = (c / P.C[2]) % P.C[1];
    z = c % P.C[2];
}

// G_k (27 slots x 3; only the slots in the mask, those where a fluid P neighbour
// lies, are written) and the mask, summed over k's P list in order; C_kk = C_ii of
// fluid k, C_jk = -beta r_kj
__global__ void k_fac_g(DevParams P, const int* __restrict__ cellIndex, const int* __restrict__ runP,
                        const long long* __restrict__ nPtrP, const int* __restrict__ nIndP,
                        const double* __restrict__ beta, const double* __restrict__ pos,
                        const double* __restrict__ selfC, double* __restrict__ gtab, int* __restrict__ gmask) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= P.np) return;
    double* G = gtab + 81 * (long long)k;
    int kx, ky, kz;
    cell_xyz(P, cellIndex[k], kx, ky, kz);
    const double pk0 = pos[3 * k], pk1 = pos[3 * k + 1], pk2 = pos[3 * k + 2];
    const long long c0 = nPtrP[k];
    const int run = runP[k];
    unsigned mask = 0;
    // the list visits each neighbour cell in one run, so a slot's sum is kept in
    // registers and stored when the run ends; slots outside the mask are never
    // read and stay unwritten (a slot met again would continue from its stored sum)
    int cur = -1;
    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
    // U entries at a time: their columns and beta, then their cell keys and positions,
    // load together (a wall or past-the-end entry loads k's own); the entries are
    // then added one by one in list order
    constexpr int U = 4;
    for (int jb = 0; jb < run; jb += U) {
        int jj[U], key[U];
        double bb[U], q[U][3];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const long long e = c0 + (jb + u < run ? jb + u : run - 1);
            jj[u] = nIndP[e];
            bb[u] = beta[e];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = jj[u] < P.nf ? jj[u] : k;
            key[u] = cellIndex[j];
            for (int d = 0; d < 3; ++d) q[u][d] = pos[3 * j + d];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = jj[u];
            if (jb + u >= run || j >= P.nf) continue;
            int jx, jy, jz;
            cell_xyz(P, key[u], jx, jy, jz);
            const int slot = fac_slot(P, jx, jy, jz, kx, ky, kz);
            if (slot < 0) continue;  // cannot happen: P neighbours are in adjacent cells
            if (slot != cur) {
                if (cur >= 0) {
                    G[3 * cur] = a0;
                    G[3 * cur + 1] = a1;
                    G[3 * cur + 2] = a2;
                }
                cur = slot;
                const bool seen = (mask >> slot) & 1u;
                a0 = seen ? G[3 * slot] : 0.0;
                a1 = seen ? G[3 * slot + 1] : 0.0;
                a2 = seen ? G[3 * slot + 2] : 0.0;
            }
            double c[3];
            if (j == k) {
                c[0] = selfC[3 * k];
                c[1] = selfC[3 * k + 1];
                c[2] = selfC[3 * k + 2];
            } else {  // body::fac_disp on the loaded position
                const double r0 = min_image(q[u][0], pk0, P.W[0], P.hW[0]);
                const double r1 = min_image(q[u][1], pk1, P.W[1], P.hW[1]);
                const double r2 = min_image(q[u][2], pk2, P.W[2], P.hW[2]);
                const double b = bb[u];
                c[0] = -(b * r0);
                c[1] = -(b * r1);
                c[2] = -(b * r2);
            }
            a0 += c[0];
            a1 += c[1];
            a2 += c[2];
            mask |= 1u << slot;
        }
    }
    if (cur >= 0) {
        G[3 * cur] = a0;
        G[3 * cur + 1] = a1;
        G[3 * cur + 2] = a2;
    }
    gmask[k] = (int)mask;
}

// level-0 row cell g (workgroup): the 3x3 blocks A0(g, c) of its ncs stencil cells.
// Thread t works on stencil cell c = t % ncs in partition t / ncs; the partitions split
// the row cell's particles (viscous part) and the candidate list (C Lambda C^T part)
// round robin, and their sums are added in partition order at the end.  The viscous part
// and the diagonal blocks come from the run sums of the matrix-A pass (blk): a particle's
// record of each visited cell that falls in stencil cell c.  (Walking the runs entry by
// entry here took 3.95 ms of 4.7 on the 1M scene.)  The candidates are the particles of
// the cells around g whose G table holds g, compacted in order into a list in LDS
// (flushed when full).  The list and the partition sums share one LDS buffer.  A walk is
// a chain of loads, so many short ones: 145 us at 4.9k particles, 168 at 64k and 799 at 1M
// (22k cells) with one wavefront and two partitions per cell, now 22, 62 and 636.
// T threads: 64 in 2D (12 rows a cell and few candidates; 160k particles 67 us, 85 with
// 128), 512 in 3D up to kGal0Cells cells, beyond it 256 (1M: 636 us, 831 with 512): enough
// workgroups are there to wait for one another.
constexpr int kGal0Cells = 4096;
template <int T>
__global__ void __launch_bounds__(T) k_fac_gal0(DevParams P, Level L, FacOp F, const int* __restrict__ cellStart,
                                                const double* __restrict__ blk, const double* __restrict__ gtab,
                                                const int* __restrict__ gmask, int g0) {
    typedef double dv2 __attribute__((ext_vector_type(2)));
    constexpr int kRanges = 54, kGal0List = 6 * T;  // ranges: fluid, then wall particles of 27 cells
    __shared__ double sbuf[T * 9];    // the list, then the partition sums
    static_assert(3 * kGal0List * sizeof(int) <= sizeof(sbuf), "list exceeds the shared buffer");
    int* const lk = (int*)sbuf;       // candidate particle
    int* const lc = lk + kGal0List;   // its cell's offset from g, (dx+1) + 3 (dy+1) + 9 (dz+1)
    int* const lm = lc + kGal0List;   // its G mask
    __shared__ signed char slots[27][27];  // [stencil cell][offset]: the G slot, -1 none
    __shared__ int rlo[64], roff[64], rsg[64], hits[T / 64];  // roff: candidates before the range
    __shared__ unsigned char rcell[64];
    const int ncs = L.cs[0] * L.cs[1] * L.cs[2];
    const int nparts = T / ncs;
    const int g = g0 + blockIdx.x, t = threadIdx.x, lane = t & 63, wave = t / 64;
    const int c = t % ncs, part = t / ncs;
    const bool active = part < nparts;
    int gx, gy, gz;
    body::grid_xyz(L, g, gx, gy, gz);
    const int ax = gx + L.mn[0], ay = gy + L.mn[1], az = gz + L.mn[2];
    const int ic = body::cell_id(P, ax, ay, az);
    const int p0 = cellStart[ic], p1 = cellStart[ic + 1];
    const int* C = P.C;
    const int wx = ((ax % C[0]) + C[0]) % C[0], wy = ((ay % C[1]) + C[1]) % C[1], wz = ((az % C[2]) + C[2]) % C[2];
    auto wrapc = [](int v, int cnt) { return v < 0 ? v + cnt : (v >= cnt ? v - cnt : v); };
    auto inside = [&](int o) {  // offset within the neighbour range (2D: no z offsets)
        const int dx = o % 3 - 1, dy = (o / 3) % 3 - 1, dz = o / 9 - 1;
        return abs(dx) <= P.range[0] && abs(dy) <= P.range[1] && abs(dz) <= P.range[2];
    };
    // slot, in the G table of a particle at offset o, of stencil cell h (level-0 counts of
    // at least 3 per axis: the caller checks)
    for (int e = t; e < 27 * ncs; e += T) {
        const int h = e / 27, o = e % 27;
        const int iX = h / (L.cs[1] * L.cs[2]), iY = (h / L.cs[2]) % L.cs[1], iZ = h % L.cs[2];
        const int hx = (((L.mn[0] + (gx + (L.cs[0] == 3 ? iX - 1 : 0) + L.cnt[0]) % L.cnt[0]) % C[0]) + C[0]) % C[0];
        const int hy = (((L.mn[1] + (gy + (L.cs[1] == 3 ? iY - 1 : 0) + L.cnt[1]) % L.cnt[1]) % C[1]) + C[1]) % C[1];
        const int hz = (((L.mn[2] + (gz + (L.cs[2] == 3 ? iZ - 1 : 0) + L.cnt[2]) % L.cnt[2]) % C[2]) + C[2]) % C[2];
        slots[h][o] = !inside(o) ? -1
                                 : (signed char)fac_slot(P, hx, hy, hz, wrapc(wx + o % 3 - 1, C[0]),
                                                         wrapc(wy + (o / 3) % 3 - 1, C[1]), wrapc(wz + o / 9 - 1, C[2]));
    }
    if (wave == 0) {  // the candidates' ranges, cells by x, y, z offset
        int cnt = 0, lo = 0, sg = -1, o = 0;
        if (lane < kRanges) {
            const int q = lane / 2, half = lane % 2;
            o = q / 9 + 3 * ((q / 3) % 3) + 9 * (q % 3);
            if (inside(o)) {
                const int kx = wrapc(wx + o % 3 - 1, C[0]), ky = wrapc(wy + (o / 3) % 3 - 1, C[1]);
                const int kz = wrapc(wz + o / 9 - 1, C[2]);
                sg = fac_slot(P, wx, wy, wz, kx, ky, kz);
                const int kc = half * P.T + body::cell_id(P, kx, ky, kz);
                if (sg >= 0) {
                    lo = cellStart[kc];
                    cnt = cellStart[kc + 1] - lo;
                }
            }
        }
        int incl = cnt;
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(incl, d, 64);
            if (lane >= d) incl += v;
        }
        rlo[lane] = lo;
        roff[lane] = incl - cnt;  // lanes past the ranges: the total
        rsg[lane] = sg;
        rcell[lane] = (unsigned char)o;
    }
    double acc[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    // viscous part and the diagonal blocks: the run sums of the row cell's particles
    // in the visited cells that fall in stencil cell c, then the particle's diagonal
    // block where c holds the row cell itself
    const unsigned vmask = active ? body::galerkin_mask(P, L, cellStart, g, c) : 0u;
    const bool dself = (vmask >> body::galerkin_self(P, L, g)) & 1u;
    if (vmask)
        for (int ip = p0 + part; ip < p1; ip += nparts) {
            const double* rb = blk + (long long)ip * kBlkRuns * kBlkStride;
            for (unsigned m = vmask; m; m &= m - 1) {  // symmetric: the upper triangle twice
                const dv2* o = (const dv2*)(rb + __builtin_ctz(m) * kBlkStride);
                const dv2 v0 = o[0], v1 = o[1], v2 = o[2];
                acc[0] += v0.x;
                acc[1] += v0.y;
                acc[2] += v1.x;
                acc[3] += v0.y;
                acc[4] += v1.y;
                acc[5] += v2.x;
                acc[6] += v1.x;
                acc[7] += v2.x;
                acc[8] += v2.y;
            }
            if (dself)
                for (int e = 0; e < 9; ++e) acc[e] += F.diag[9 * (long long)ip + e];
        }
    __syncthreads();
    // C Lambda C^T part: lambda_k G_gk G_hk^T for the listed k; h is stencil cell c
    int n = 0;  // entries in the list (uniform)
    auto consume = [&]() {
        if (active)
            for (int e0 = part; e0 < n; e0 += 2 * nparts) {  // two entries' loads under way
                bool ok[2];
                double lv[2], gg[2][3], gh[2][3];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int e = e0 + u * nparts < n ? e0 + u * nparts : e0;
                    const int o = lc[e], sh = slots[c][o], k = lk[e];
                    ok[u] = e0 + u * nparts < n && sh >= 0 && ((unsigned)lm[e] >> sh & 1u);
                    const int sg = rsg[2 * (9 * (o % 3) + 3 * ((o / 3) % 3) + o / 9)];
                    const double* G = gtab + 81 * (long long)k;
                    lv[u] = F.lambda[k];
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        gg[u][d] = G[3 * sg + d];
                        gh[u][d] = G[(ok[u] ? 3 * sh : 3 * sg) + d];
                    }
                }
#pragma unroll
                for (int u = 0; u < 2; ++u)
                    if (ok[u]) {
                        const double lg[3] = {lv[u] * gg[u][0], lv[u] * gg[u][1], lv[u] * gg[u][2]};
                        for (int rr = 0; rr < 3; ++rr) {
                            acc[3 * rr] += lg[rr] * gh[u][0];
                            acc[3 * rr + 1] += lg[rr] * gh[u][1];
                            acc[3 * rr + 2] += lg[rr] * gh[u][2];
                        }
                    }
            }
        __syncthreads();
        n = 0;
    };
    const int total = roff[63];
    for (int base = 0; base < total; base += T) {
        const int idx = base + t;
        int q = 0;  // the last range starting at or before the candidate
#pragma unroll
        for (int step = 32; step >= 1; step >>= 1)
            if (q + step < kRanges && roff[q + step] <= idx) q += step;
        const int k = rlo[q] + idx - roff[q];
        const unsigned km = idx < total ? (unsigned)gmask[k] : 0u;
        const bool hit = idx < total && (km >> rsg[q] & 1u);
        const unsigned long long bal = __ballot(hit);
        if (lane == 0) hits[wave] = __popcll(bal);
        __syncthreads();
        int before = __popcll(bal & ((1ull << lane) - 1ull)), cnt = 0;
        for (int w = 0; w < T / 64; ++w) {
            before += w < wave ? hits[w] : 0;
            cnt += hits[w];
        }
        if (n + cnt > kGal0List) consume();
        if (hit) {
            lk[n + before] = k;
            lc[n + before] = rcell[q];
            lm[n + before] = (int)km;
        }
        n += cnt;
        __syncthreads();
    }
    consume();  // ends with a barrier: the list is dead, sbuf takes the partition sums
    if (active)
        for (int e = 0; e < 9; ++e) sbuf[9 * t + e] = acc[e];
    __syncthreads();
    for (int h9 = t; h9 < 9 * ncs; h9 += T) {  // (stencil cell, entry)
        double v = sbuf[h9];
        for (int q = 1; q < nparts; ++q) v += sbuf[9 * ncs * q + h9];
        const int h = h9 / 9, e = h9 % 9;
        L.A[(long long)(3 * h + e % 3) * L.nrow + 3 * g + e / 3] = v;
    }
}

// InvDiagA (calculateInvDiagA, main.cpp:3045-3068): 1/A_ii[r][r] with
// A_ii[r][r] = D_i[r][r] + sum_{k in P(i)} lambda_k C_ik[r]^2
__global__ void __launch_bounds__(256) k_fac_invdiag(DevParams P, FacOp F, double* __restrict__ invDiagA) {
    // entry-parallel: lane g forms the terms of entries g, g + 8, ...; the group's
    // first lane adds them in list order
    constexpr int G = 8, K = 3;
    __shared__ double tb[256 * K];
    const int g = threadIdx.x & (G - 1);
    const int i = (int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) / G);
    const bool own = i < P.nf;
    const double pi0 = own ? F.pos[3 * i] : 0.0, pi1 = own ? F.pos[3 * i + 1] : 0.0, pi2 = own ? F.pos[3 * i + 2] : 0.0;
    double d[3] = {0.0, 0.0, 0.0};
    if (own) {
        d[0] = F.diag[9 * i];
        d[1] = F.diag[9 * i + 4];
        d[2] = F.diag[9 * i + 8];
    }
    const long long c0 = own ? F.nPtrP[i] : 0;
    const int n = own ? F.nCountP[i] : 0;
    for (int base = 0; base < n; base += G) {
        const int jn = base + g;
        double t[K] = {0.0, 0.0, 0.0};
        if (jn < n) {
            const int k = F.nIndP[c0 + jn];
            double cv[3];
            if (k == i) {
                cv[0] = F.selfC[3 * i];
                cv[1] = F.selfC[3 * i + 1];
                cv[2] = F.selfC[3 * i + 2];
            } else {
                double r0, r1, r2;
                body::fac_disp(P, F.pos, k, pi0, pi1, pi2, r0, r1, r2);
                const double b = F.beta[c0 + jn];
                cv[0] = b * r0;
                cv[1] = b * r1;
                cv[2] = b * r2;
            }
            const double lk = F.lambda[k];
            for (int a = 0; a < 3; ++a) t[a] = lk * cv[a] * cv[a];
        }
        for (int e = 0; e < K; ++e) tb[K * threadIdx.x + e] = t[e];
        wave_sync();
        if (g == 0)
            for (int u = 0; u < G && base + u < n; ++u)
                for (int a = 0; a < 3; ++a) d[a] += tb[K * (threadIdx.x + u) + a];
        wave_sync();
    }
    if (g == 0 && own)
        for (int a = 0; a < 3; ++a) invDiagA[3 * i + a] = d[a] != 0.0 ? 1.0 / d[a] : 0.0;
}

// the wrap flag is uniform, so the branch is taken by the whole launch; the FP32
// form has no displacements to wrap
template <class VT>
__global__ void __launch_bounds__(256, 6) k_fac_t(DevParams P, FacOp F, const double* __restrict__ x) {
    if (cr_halted(P.halt)) return;
    if constexpr (sizeof(VT) == 4) body::fac_t32_chunk(P, F, x, blockIdx.x);
    else if (*F.wrap) body::fac_t_chunk<true>(P, F, x, blockIdx.x);
    else body::fac_t_chunk<false>(P, F, x, blockIdx.x);
}

template <bool kNeg, class VT>
__global__ void __launch_bounds__(256, 4) k_fac_y(DevParams P, FacOp F, const double* __restrict__ x, double beta,
                                               const double* yin, double* y, double* y2, double* p_copy) {
    if (cr_halted(P.halt)) return;
    if constexpr (sizeof(VT) == 4) body::fac_y32_chunk<kNeg>(P, F, x, beta, yin, y, y2, p_copy, blockIdx.x);
    else body::fac_y_chunk_any<kNeg>(P, F, x, beta, yin, y, y2, p_copy, blockIdx.x);
}

// ---------------------------------------------------------------------------
// The FP64 second pass with its gathers from LDS.
//
// Every row of one cell visits the same 27 (9 in 2D) cells, so one workgroup per row
// cell stages the records (x, position, t) of the fluid particles of those cells in LDS
// once, and its rows read their fluid neighbours' records from there instead of
// gathering them through L1 and L2 per entry (each gather instruction of the chunk
// kernel touched about 21 cache lines).  An entry is a 2-byte place; alpha and beta are
// recomputed from the distance (body::fac_pair), and as the RadiusP neighbours are among
// the fluid neighbours, one walk forms both terms.  On the 1M-particle scene the pass
// takes 428 us; it took 726 us when it streamed alpha beside the places and walked the P
// lists on their own (10 bytes per entry at 4.3 TB/s, a dependent round of list loads
// per 32 entries, and the P part's gathers).  The VALU issues 52% of the time, the rest
// is LDS reads with their bank conflicts and a workgroup's waits for its loads at two
// workgroups per CU.
// A row's entries, lanes and order of summation are those of body::fac_row_gather, so
// the results are the chunk kernel's.  The rows go straight to y; the dot partials of
// the fused epilogue come from a dot-partial launch afterwards (the chunks of 256 rows
// do not follow cells).
//
// Everything a workgroup needs of its cell is in a descriptor built once per step
// (k_fac_slots), so it waits for two rounds of loads before it computes: the
// descriptor, then the staged records, the first places and the rows' diagonal terms
// together.
constexpr int kCellTable = 32;     // visited cells (27 in 3D) padded for the binary search

// words of FacOp::cellDesc, per cell of the fluid bounding box
enum {
    kFdRow = 0,     // first fluid row
    kFdRows = 1,    // rows (0: nothing to do)
    kFdTotal = 2,   // staged records; -1: more than the staging holds
    kFdBatches = 3, // batches of 4 entries per lane of the longest row
    kFdOwn = 4,     // place of the first row's own record
    kFdWalls = 5,   // some row has wall neighbours within RadiusP
    kFdPieces = 6,  // pieces of up to 64 consecutive particles; (first place | count << 16, first particle) of each
    kFdPiece0 = 8
};
static_assert(kFdPiece0 + 2 * (27 + kFacCellSlots[kFacCell3DWide] / 64) <= kFacDesc, "the pieces fit the descriptor");

typedef double dv2c __attribute__((ext_vector_type(2)));

// the cell of bounding-box index b (z fastest)
__device__ inline void fac_cell_xyz(const FacOp& F, int b, int& cx, int& cy, int& cz) {
    cz = F.cellLo[2] + b % F.cellCnt[2];
    cy = F.cellLo[1] + (b / F.cellCnt[2]) % F.cellCnt[1];
    cx = F.cellLo[0] + b / (F.cellCnt[2] * F.cellCnt[1]);
}

// FacOp::cellDesc and the places of every row of bounding-box cell blockIdx.x
__global__ void __launch_bounds__(256) k_fac_slots(DevParams P, FacOp F, int cap) {
    __shared__ int vlo[kCellTable], voff[kCellTable], vex[kCellTable], total, most, walls;
    const int t = threadIdx.x;
    int cx, cy, cz;
    fac_cell_xyz(F, blockIdx.x, cx, cy, cz);
    int* const D = F.cellDesc + (long long)kFacDesc * blockIdx.x;
    const int* C = P.C;
    const int c = (cx * C[1] + cy) * C[2] + cz;
    const int rs = F.cellStart[c], nrows = F.cellStart[c + 1] - rs;
    if (t == 0) D[kFdRows] = nrows;
    if (nrows <= 0) return;
    const int nx = 2 * P.range[0] + 1, ny = 2 * P.range[1] + 1, nz = 2 * P.range[2] + 1, nv = nx * ny * nz;
    if (t < 64) {  // the visited cells in the neighbour search's order (ascending CellId)
        int lo = 0x7fffffff, cnt = 0;
        if (t < nv) {
            const int bx = 2 * P.range[0] - (cx + P.range[0]) % C[0];
            const int by = 2 * P.range[1] - (cy + P.range[1]) % C[1];
            const int bz = 2 * P.range[2] - (cz + P.range[2]) % C[2];
            const int a = (bx > 0 ? bx : 0) + t / (ny * nz), bb = (by > 0 ? by : 0) + (t / nz) % ny;
            const int cc = (bz > 0 ? bz : 0) + t % nz;
            const int jx = ((cx - P.range[0] + a % nx) % C[0] + C[0]) % C[0];
            const int jy = ((cy - P.range[1] + bb % ny) % C[1] + C[1]) % C[1];
            const int jz = ((cz - P.range[2] + cc % nz) % C[2] + C[2]) % C[2];
            const int jc = (jx * C[1] + jy) * C[2] + jz;
            lo = F.cellStart[jc];
            cnt = F.cellStart[jc + 1] - lo;
        }
        int incl = cnt;  // inclusive scan of the counts over the wavefront
        for (int d = 1; d < 64; d <<= 1) {
            const int u = __shfl_up(incl, d, 64);
            if (t >= d) incl += u;
        }
        if (t < kCellTable) {
            vlo[t] = lo;
            voff[t] = (incl - cnt) - (t < nv ? lo : 0);
            vex[t] = t < nv ? incl - cnt : 0x7fffffff;
        }
        if (t == 63) {
            total = incl;
            most = 0;
            walls = 0;
        }
    }
    __syncthreads();
    // the place of fluid particle j: j + voff of the last visited range starting at or
    // before j
    auto place = [&](int j) {
        int v = 0;
#pragma unroll
        for (int step = kCellTable / 2; step >= 1; step >>= 1)
            if (vlo[v + step] <= j) v += step;
        return j + voff[v];
    };
    for (int r = t; r < nrows; r += 256) {
        atomicMax(&most, F.nFluid[rs + r]);
        if (F.nCountP[rs + r] > F.runP[rs + r]) atomicOr(&walls, 1);
    }
    __syncthreads();
    constexpr int G = kFacLanes;
    const int nb = (most + 4 * G - 1) / (4 * G);
    if (t == 0) {
        D[kFdRow] = rs;
        D[kFdTotal] = total <= cap ? total : -1;
        D[kFdBatches] = nb;
        D[kFdOwn] = place(rs);
        D[kFdWalls] = walls;
        int m = 0;
        for (int v = 0; v < nv && total <= cap;) {  // cells with consecutive particles share pieces
            const int p0 = vex[v], j0 = vlo[v];
            int p1 = p0;
            do {
                p1 = v + 1 < nv ? vex[v + 1] : total;
                ++v;
            } while (v < nv && vlo[v] == j0 + (p1 - p0));
            for (int p = p0; p < p1; p += 64, ++m) {
                D[kFdPiece0 + 2 * m] = p | (p1 - p < 64 ? p1 - p : 64) << 16;
                D[kFdPiece0 + 2 * m + 1] = j0 + (p - p0);
            }
        }
        D[kFdPieces] = m;
    }
    if (total > cap) return;  // that cell's rows gather from global memory
    // 32 lanes write a row's places, two each
    for (int r = t / 32; r < nrows; r += 8) {
        const int i = rs + r;
        const long long b0 = F.nPtr[i];
        const int w = F.nFluid[i];
        unsigned* const sl = (unsigned*)(F.slot + (long long)i * F.slotRow);
        const int own = place(i);
        for (int q = 2 * (t & 31); q < 8 * G * ((nb + 1) / 2); q += 64) {
            // places q and q + 1 of block q / 8G: lane (q / 8) mod G, entries q mod 8 and the next
            const int e = q / (8 * G) * (8 * G) + (q & 7) * G + (q >> 3) % G;
            const int a = e < w ? place(F.nInd[b0 + e]) : own, b = e + G < w ? place(F.nInd[b0 + e + G]) : own;
            sl[q / 2] = (unsigned)a | (unsigned)b << 16;
        }
    }
}

// the staged records in four planes: t (facP t), x0 x1, x2 p0, p1 p2 (x scaled as
// body::fac_pair takes it)
template <int kCap>
struct FacCellShared {
    double t[kCap];
    dv2c a[kCap], b[kCap], c[kCap];
};

// one batch of a row's walk: the four entries whose places are in w0, w1
template <bool kWrap, bool kVar, int kCap>
__device__ inline void fac_cell_batch(const DevParams& P, const FacCellShared<kCap>& L, unsigned w0, unsigned w1,
                                      const double* al, double pi0, double pi1, double pi2, double& s0, double& s1,
                                      double& s2) {
    const unsigned sl[4] = {w0 & 0xffffu, w0 >> 16, w1 & 0xffffu, w1 >> 16};
    dv2c q0[4], q1[4], q2[4];
    double q3[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        q0[u] = L.a[sl[u]];
        q1[u] = L.b[sl[u]];
        q2[u] = L.c[sl[u]];
        q3[u] = L.t[sl[u]];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const double r0 = body::fac_wrap<kWrap>(q1[u][1] - pi0, P.W[0], P.hW[0]);
        const double r1 = body::fac_wrap<kWrap>(q2[u][0] - pi1, P.W[1], P.hW[1]);
        const double r2 = body::fac_wrap<kWrap>(q2[u][1] - pi2, P.W[2], P.hW[2]);
        body::fac_pair<kVar>(P, r0, r1, r2, q0[u][0], q0[u][1], q1[u][0], q3[u], kVar ? al[u] : 0.0, s0, s1, s2);
    }
}

// workgroup b of the pass over scene (P, F); kThreads, kCap: kFacCell* of F.cellShape
template <bool kNeg, bool kWrap, bool kVar, int kThreads, int kCap>
__device__ inline void fac_y_cell_body(const DevParams& P, const FacOp& F, const double* __restrict__ x, double beta,
                                       const double* yin, double* y, double* y2, double* p_copy,
                                       FacCellShared<kCap>& L, int b) {
    constexpr int G = kFacLanes, kRows = kThreads / G;
    if (F.cellXcd) {
        // workgroups are dealt to the 8 XCDs in turn: XCD x = b mod 8 takes a contiguous
        // range of cells instead, so that the cells running on one XCD at a time are
        // neighbours and share their visited cells' records in that XCD's L2
        const int nb = F.cellCnt[0] * F.cellCnt[1] * F.cellCnt[2], per = nb / 8, rem = nb % 8, xc = b % 8;
        b = xc * per + (xc < rem ? xc : rem) + b / 8;
    }
    const int* __restrict__ D = F.cellDesc + (long long)kFacDesc * b;
    const int rs = D[kFdRow], nrows = D[kFdRows], total = D[kFdTotal], nb = D[kFdBatches], own = D[kFdOwn];
    const int walls = D[kFdWalls], m = D[kFdPieces];
    if (nrows <= 0) return;  // the whole workgroup
    const int t = threadIdx.x, g = t & (G - 1);
    const body::FacPlanes R = body::fac_planes(P, F.rec);
    const double* __restrict__ rt = R.t;
    const unsigned short* __restrict__ slot = F.slot;
    const long long srow = F.slotRow;
    auto places = [&](int i, int blk) {  // the lane's 8 entries of block blk of row i
        return *(const uint4*)(slot + (long long)i * srow + 8 * G * blk + 8 * g);
    };
    uint4 pl = {0, 0, 0, 0};
    const bool staged = total >= 0;
    if (staged) {
        if (t / G < nrows) pl = places(rs + t / G, 0);
        // wavefront w stages pieces w, w + kWaves, ...: uniform bases, the records of a
        // piece consecutive, and every load of a round of pieces issued before the first
        // store
        const dv2c* __restrict__ ra = (const dv2c*)R.a;
        const dv2c* __restrict__ rb = (const dv2c*)R.b;
        const dv2c* __restrict__ rc = (const dv2c*)R.c;
        constexpr int kWaves = kThreads / 64, K = 3;
        const int lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t / 64);
        const double sx = kVar ? 1.0 : -P.facV;
        for (int k0 = wv; k0 < m; k0 += kWaves * K) {
            dv2c qa[K], qb[K], qc[K];
            double qt[K];
            int p0[K], n[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const int pc = k0 + k * kWaves;
                const int h = pc < m ? D[kFdPiece0 + 2 * pc] : 0, j0 = pc < m ? D[kFdPiece0 + 2 * pc + 1] : 0;
                p0[k] = h & 0xffff;
                n[k] = h >> 16;
                if (lane < n[k]) {
                    qa[k] = (ra + j0)[(unsigned)lane];
                    qb[k] = (rb + j0)[(unsigned)lane];
                    qc[k] = (rc + j0)[(unsigned)lane];
                    qt[k] = (rt + j0)[(unsigned)lane];
                }
            }
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (lane < n[k]) {
                    const int r = p0[k] + lane;
                    L.a[r] = dv2c{sx * qa[k][0], sx * qa[k][1]};
                    L.b[r] = dv2c{sx * qb[k][0], qb[k][1]};
                    L.c[r] = qc[k];
                    L.t[r] = P.facP * qt[k];
                }
        }
        __syncthreads();
    }
    const int passes = (nrows + kRows - 1) / kRows;
    for (int ps = 0; ps < passes; ++ps) {  // uniform trip count: every lane reaches the group sums
        const int r = ps * kRows + t / G;
        const bool on = r < nrows;
        const int i = rs + (on ? r : 0);
        double s0 = 0.0, s1 = 0.0, s2 = 0.0;
        double dA = 0.0, dB = 0.0, dC = 0.0, xi0 = 0.0, xi1 = 0.0, xi2 = 0.0, ti = 0.0, sc = 0.0, yv = 0.0, y2v = 0.0;
        if (on) {
            // lanes 0..2 of the row: the loads of their component of the diagonal term
            // and of y, in flight during the walk
            if (g < 3) {
                const double* Dg = F.diag + 9 * i + 3 * g;
                dA = Dg[0];
                dB = Dg[1];
                dC = Dg[2];
                xi0 = x[3 * i];
                xi1 = x[3 * i + 1];
                xi2 = x[3 * i + 2];
                ti = rt[i];
                sc = F.selfC[3 * i + g];
                yv = yin[3 * i + g];
                if (y2) y2v = y2[3 * i + g];
            }
            double pi0, pi1, pi2;
            if (staged) {
                if (ps > 0) pl = places(i, 0);
                pi0 = L.b[own + r][1];
                pi1 = L.c[own + r][0];
                pi2 = L.c[own + r][1];
                // kVar: the row's stored alphas.  Past its end the last one again, which the
                // row's own record multiplies by r = 0.  (Loads guarded by the row's length
                // took 322 us per product at 294k particles of two viscosities, these 290;
                // loading a round ahead spills: 353)
                const double* al0 = nullptr;
                int last = 0;
                if (kVar) {
                    al0 = (const double*)F.alpha + F.nPtr[i];
                    last = F.nFluid[i] - 1;
                }
                auto alphas = [&](int jb, double* al) {
#pragma unroll
                    for (int u = 0; u < 4; ++u) al[u] = kVar ? al0[min(jb + g + u * G, last)] : 0.0;
                };
                for (int k = 0; k < nb; k += 2) {
                    const uint4 cur = pl;
                    if (k + 2 < nb) pl = places(i, k / 2 + 1);
                    double al[4];
                    alphas(4 * G * k, al);
                    fac_cell_batch<kWrap, kVar>(P, L, cur.x, cur.y, al, pi0, pi1, pi2, s0, s1, s2);
                    if (k + 1 < nb) {
                        alphas(4 * G * (k + 1), al);
                        fac_cell_batch<kWrap, kVar>(P, L, cur.z, cur.w, al, pi0, pi1, pi2, s0, s1, s2);
                    }
                }
            } else {
                pi0 = F.pos[3 * i];
                pi1 = F.pos[3 * i + 1];
                pi2 = F.pos[3 * i + 2];
                body::fac_row_gather<kWrap, kVar>(P, F, i, g, pi0, pi1, pi2, s0, s1, s2);
            }
            if (walls) body::fac_walls<kWrap>(P, F, rt, i, g, pi0, pi1, pi2, s0, s1, s2);
        }
        s0 = body::group_sum(s0, G);  // every lane of the group holds the sums
        s1 = body::group_sum(s1, G);
        s2 = body::group_sum(s2, G);
        if (g < 3 && on) {  // lane g: component g, as body::fac_y_chunk computes it
            const double sg = body::fac_diag_add(g == 0 ? s0 : g == 1 ? s1 : s2, dA, dB, dC, xi0, xi1, xi2, sc, ti);
            body::store1(3 * i + g, kNeg ? -sg : sg, yv, y2v, beta, y, y2);
            if (p_copy) p_copy[3 * i + g] = g == 0 ? xi0 : g == 1 ? xi1 : xi2;
        }
    }
}

template <bool kNeg, int kThreads, int kCap>
__device__ inline void fac_y_cell_any(const DevParams& P, const FacOp& F, const double* __restrict__ x, double beta,
                                      const double* yin, double* y, double* y2, double* p_copy,
                                      FacCellShared<kCap>& L, int b) {
#define MPH_Y(WRAP, VAR) \
    fac_y_cell_body<kNeg, WRAP, VAR, kThreads, kCap>(P, F, x, beta, yin, y, y2, p_copy, L, b)
    const int wrap = F.wrap[0], var = F.wrap[1];  // uniform: the whole launch takes one branch
    if (!wrap && !var) MPH_Y(false, false);
    else if (!var) MPH_Y(true, false);
    else MPH_Y(true, true);
#undef MPH_Y
}

// four waves per SIMD: two workgroups of 512 threads on a CU.  The three bodies share one
// kernel of 128 registers.  What spills (4 registers, 7 in the batch) does so in the body of
// several viscosities alone; the others have no scratch access
template <bool kNeg, int kShape>
__global__ void __launch_bounds__(kFacCellThreads[kShape], kShape == kFacCell3DWide ? 2 : 4)
    k_fac_y_cell(DevParams P, FacOp F, const double* __restrict__ x, double beta, const double* yin, double* y,
                 double* y2, double* p_copy) {
    if (cr_halted(P.halt)) return;
    __shared__ FacCellShared<kFacCellSlots[kShape]> L;
    fac_y_cell_any<kNeg, kFacCellThreads[kShape], kFacCellSlots[kShape]>(P, F, x, beta, yin, y, y2, p_copy, L,
                                                                         blockIdx.x);
}

// The same pass for the scenes of a batch (the scene-table launches of mph_batch.hip):
// workgroup b belongs to the scene s with R.pre[s] <= b < R.pre[s+1] and runs that
// scene's cell b - R.pre[s] with its FP64 factored operator.  The grid covers the
// scenes of the launch's set and shape only (the others have empty ranges).  The scenes
// of `first` also write y2 and p_copy.
template <bool kNeg, int kShape>
__global__ void __launch_bounds__(kFacCellThreads[kShape], kShape == kFacCell3DWide ? 2 : 4)
    kb_fac_y_cell(const batch::BScene* __restrict__ tab, batch::CellRanges R, int ns, batch::SceneSet first, int x,
                  double beta, int yin, int y, int y2, int p_copy) {
    int lo = 0, hi = ns;  // the last s with R.pre[s] <= b
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (R.pre[mid] <= (int)blockIdx.x) lo = mid;
        else hi = mid;
    }
    const int s = lo, lb = (int)blockIdx.x - R.pre[lo];
    const batch::BScene& B = tab[s];
    if (batch::halted(B)) return;
    __shared__ FacCellShared<kFacCellSlots[kShape]> L;
    // the scene's parameters as values: uniform loads into scalar registers (read
    // through the table, the compiler keeps them in vector registers and spills)
    const DevParams P = B.P;
    const FacOp F = B.fac[0];
    const bool f = batch::in_set(first, s);
    double* y2p = f && y2 >= 0 ? B.vec[y2] : nullptr;
    double* pc = f && p_copy >= 0 ? B.vec[p_copy] : nullptr;
    fac_y_cell_any<kNeg, kFacCellThreads[kShape], kFacCellSlots[kShape]>(P, F, B.vec[x], beta, B.vec[yin], B.vec[y],
                                                                         y2p, pc, L, lb);
}

template <bool kNeg, class VT>
void fac_launch(hipStream_t st, const DevParams& P, const FacOp& F, const double* x, double beta, const double* yin,
                double* y, double* y2, double* p_copy, const double* dotx, double* part, int passes) {
    constexpr bool f32 = sizeof(VT) == 4;
    if (passes & 1)
        hipLaunchKernelGGL(k_fac_t<VT>, dim3(nblk(P.np, f32 ? kFacRowsY : kFacRowsT)), dim3(256), 0, st,
                           P, F, x);
    if (!(passes & 2)) return;
    const long long cells = (long long)F.cellCnt[0] * F.cellCnt[1] * F.cellCnt[2];
    if (!f32 && F.slot && cells > 0) {
#define MPH_CELL(SHAPE)                                                                                           \
    hipLaunchKernelGGL((k_fac_y_cell<kNeg, SHAPE>), dim3((unsigned)cells), dim3(kFacCellThreads[SHAPE]), 0, st, P, F, \
                       x, beta, yin, y, y2, p_copy)
        if (F.cellShape == kFacCell2D) MPH_CELL(kFacCell2D);
        else if (F.cellShape == kFacCell3D) MPH_CELL(kFacCell3D);
        else MPH_CELL(kFacCell3DWide);
#undef MPH_CELL
    } else {
        hipLaunchKernelGGL((k_fac_y<kNeg, VT>), dim3(nblk(P.nf, kFacRowsY)), dim3(256), 0,
                           st, P, F, x, beta, yin, y, y2, p_copy);
    }
    if (part) launch_dot_partial(st, P, dotx, y, part);
}

}  // namespace

void launch_fac_p(hipStream_t st, const DevParams& P, const double* pos, const int* nCountP, const long long* nPtrP,
                  const int* nIndP, double* beta, float* v32, int* runP, double* selfC, double* rec) {
    if (P.np == 0) return;
    hipLaunchKernelGGL(k_fac_p, dim3(nblk(8LL * P.np, 256)), dim3(256), 0, st, P, pos, nCountP, nPtrP, nIndP, beta,
                       v32, runP, selfC, rec);
}

void launch_fac_level0(hipStream_t st, const DevParams& P, const Level& L0, const FacOp& F, const int* cellIndex,
                       const int* cellStart, const double* blk, double* gtab, int* gmask, double* invDiagA) {
    if (P.nf == 0) return;
    hipLaunchKernelGGL(k_fac_g, dim3(nblk(P.np, 128)), dim3(128), 0, st, P, cellIndex, F.runP, F.nPtrP, F.nIndP,
                       F.beta, F.pos, F.selfC, gtab, gmask);
    hipLaunchKernelGGL(k_fac_invdiag, dim3(nblk(8LL * P.nf, 256)), dim3(256), 0, st, P, F, invDiagA);
#define MPH_GAL0(T)                                                                                               \
    body::per_cell(L0.cells, [&](int g0, int n) {                                                                 \
        hipLaunchKernelGGL(k_fac_gal0<T>, dim3(n), dim3(T), 0, st, P, L0, F, cellStart, blk, gtab, gmask, g0);    \
    })
    if (P.dim == 2) MPH_GAL0(64);
    else if (L0.cells < kGal0Cells) MPH_GAL0(512);
    else MPH_GAL0(256);
#undef MPH_GAL0
}

void launch_fac_u(hipStream_t st, const DevParams& P, const int* nFluid, const long long* nPtr, const int* nInd,
                  const double* alpha, const double* pos, float* u32) {
    if (P.nf == 0) return;
    hipLaunchKernelGGL(k_fac_u, dim3(nblk(8LL * P.nf, 256)), dim3(256), 0, st, P, nFluid, nPtr, nInd, alpha, pos,
                       u32);
}

__global__ void __launch_bounds__(256) k_fac_rec_positions(DevParams P, const double* __restrict__ from,
                                                           double* __restrict__ to) {
    const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= P.np) return;
    const body::FacPlanes F = body::fac_planes(P, const_cast<double*>(from)), T = body::fac_planes(P, to);
    T.b[2 * k + 1] = F.b[2 * k + 1];  // p0
    T.c[2 * k] = F.c[2 * k];          // p1
    T.c[2 * k + 1] = F.c[2 * k + 1];  // p2
}

void launch_fac_rec_positions(hipStream_t st, const DevParams& P, const double* from, double* to) {
    if (P.np == 0) return;
    hipLaunchKernelGGL(k_fac_rec_positions, dim3(nblk(P.np, 256)), dim3(256), 0, st, P, from, to);
}

void launch_fac_slots(hipStream_t st, const DevParams& P, const FacOp& F) {
    const long long cells = (long long)F.cellCnt[0] * F.cellCnt[1] * F.cellCnt[2];
    if (P.nf == 0 || !F.slot || cells <= 0) return;
    hipLaunchKernelGGL(k_fac_slots, dim3((unsigned)cells), dim3(256), 0, st, P, F, kFacCellSlots[F.cellShape]);
}

namespace batch {
void spmv_fac_cells(const Tables& T, const SceneSet& on, const char* shapes, const SceneSet& first, double alpha,
                    int x, double beta, int yin, int y, int y2, int p_copy) {
    const int* o = T.hoff + (size_t)kOffCell * (T.ns + 1);
    for (int shape = 0; shape < kFacCellShapes; ++shape) {
        CellRanges R;
        int g = 0;
        for (int s = 0; s < T.ns; ++s) {
            R.pre[s] = g;
            if (((on.w[s >> 6] >> (s & 63)) & 1ull) && shapes[s] == shape) g += o[s + 1] - o[s];
        }
        R.pre[T.ns] = g;
        if (g <= 0) continue;
#define MPH_CELL(NEG, SHAPE)                                                                                        \
    hipLaunchKernelGGL((kb_fac_y_cell<NEG, SHAPE>), dim3(g), dim3(kFacCellThreads[SHAPE]), 0, T.st, T.tab, R, T.ns, \
                       first, x, beta, yin, y, y2, p_copy)
#define MPH_SIGN(SHAPE)                       \
    do {                                      \
        if (alpha < 0) MPH_CELL(true, SHAPE); \
        else MPH_CELL(false, SHAPE);          \
    } while (0)
        if (shape == kFacCell2D) MPH_SIGN(kFacCell2D);
        else if (shape == kFacCell3D) MPH_SIGN(kFacCell3D);
        else MPH_SIGN(kFacCell3DWide);
#undef MPH_SIGN
#undef MPH_CELL
    }
}
}  // namespace batch

void launch_fac_spmv(hipStream_t st, const DevParams& P, const FacOp& F, double alpha, const double* x, double beta,
                     const double* yin, double* y, double* y2, double* p_copy, const double* dotx, double* part,
                     bool f32, int passes) {
    // alpha is +1 or -1 at every call site (main.cpp:4337, 4353, 4357)
    if (P.nf == 0) return;
    if (f32) {
        if (alpha < 0) fac_launch<true, float>(st, P, F, x, beta, yin, y, y2, p_copy, dotx, part, passes);
        else fac_launch<false, float>(st, P, F, x, beta, yin, y, y2, p_copy, dotx, part, passes);
    } else {
        if (alpha < 0) fac_launch<true, double>(st, P, F, x, beta, yin, y, y2, p_copy, dotx, part, passes);
        else fac_launch<false, double>(st, P, F, x, beta, yin, y, y2, p_copy, dotx, part, passes);
    }
}

}  // namespace mph
