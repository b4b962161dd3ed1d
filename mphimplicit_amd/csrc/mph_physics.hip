// mph_physics.hip -- kinematics, explicit particle interactions and implicit assembly.
//
// Replaces calculateConvection/Wall/PeriodicBoundary/resetForce, the explicit force
// loops (source/main.cpp:1678-2128, 4741-4752), calculateMatrixA/C and
// multiplyMatrixC (2137-2643), and the output-step diagnostics (1932-2063,
// 4494-4738).  Each of a particle's sums runs over the neighbour list in list
// order, so every value is bit-identical to the reference.  The list walks of the
// densities, forces and matrix A are entry-parallel: a group of kLanes lanes owns
// the particle, lane g computes the terms of entries g, g + kLanes, ..., and a lane per
// component adds them, read back through LDS, in list order.
#include "mph_kernels.h"

namespace mph {

namespace {

inline int nblk(long long n, int bs) { return (int)((n + bs - 1) / bs); }

struct Rel {
    double x[3];
    double r2;
};

// both positions are loaded before the first min_image, whose branch would otherwise
// hold each coordinate's load back until the previous one is done
__device__ inline Rel rel(const DevParams& P, const double* __restrict__ pos, int i, int j) {
    Rel o;
    double pj[3], pi[3];
    for (int d = 0; d < 3; ++d) {
        pj[d] = pos[3 * j + d];
        pi[d] = pos[3 * i + d];
    }
    for (int d = 0; d < 3; ++d) o.x[d] = min_image(pj[d], pi[d], P.W[d], P.hW[d]);
    o.r2 = (o.x[0] * o.x[0] + o.x[1] * o.x[1] + o.x[2] * o.x[2]);
    return o;
}

// lanes per particle of the entry-parallel list walks (a workgroup is 256 lanes):
// kLanes for the MaxRadius lists (about 180 entries in 3D), kLanesP for the RadiusP
// lists (about 20).  32 lanes on the long lists: matrix A 48 against 58 us at 4.9k
// particles, but 4.26 against 3.76 ms at 1M (fewer particles to a wavefront share an
// addition)
constexpr int kLanes = 16, kLanesP = 8;

// The terms of a round of kLanes entries, a row per component: the lane that owns a
// component adds its row in list order, two terms to a read.  A term that the entry does
// not have is +0: a sum starts at +0 and so is never -0, and adding it changes nothing.
// One lane adding every component of its particle's entries, four lanes to a particle,
// spent most of the walk there, one dependent LDS read after the other, in 45 rounds of
// loads for a list of 180.  Densities, forces, matrix A at 4.9k particles: 71, 47, 160 us
// then, 26, 23, 58 now; at 64k 130, 115, 285 and 83, 77, 253; at 1M 1.57, 1.34, 3.97 ms
// and 1.18, 1.19, 3.76, of which matrix A's divisions and stores are most.
template <int K>
struct TermRows {
    double v[256 / kLanes][K][kLanes + 2];
    __device__ inline double add(int row, double s) const {  // s + the row's terms
        typedef double dv2 __attribute__((ext_vector_type(2)));
        const dv2* t = (const dv2*)v[threadIdx.x / kLanes][row];
#pragma unroll
        for (int o = 0; o < kLanes / 2; ++o) {
            const dv2 w = t[o];
            s += w[0];
            s += w[1];
        }
        return s;
    }
    __device__ inline double& at(int row) { return v[threadIdx.x / kLanes][row][threadIdx.x % kLanes]; }
};

// calculateConvection, calculateWall, calculatePeriodicBoundary, resetForce
__global__ void k_kinematics(DevParams P, WallKin wk, const int* __restrict__ type, double* __restrict__ pos,
                             double* __restrict__ vel, double* __restrict__ force) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P.np) return;
    double x[3] = {pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]};
    if (i < P.nf) {
        for (int d = 0; d < 3; ++d) x[d] += vel[3 * i + d] * P.dt;
    } else {
        const int t = type[i];
        const double(&R)[3][3] = wk.R[t];
        const double* w = wk.omega[t];
        const double* V = wk.vel[t];
        const double* c = wk.center[t];
        double r[3] = {x[0] - c[0], x[1] - c[1], x[2] - c[2]};
        r[0] = R[0][0] * r[0] + R[0][1] * r[1] + R[0][2] * r[2];  // in place, main.cpp:2108-2110
        r[1] = R[1][0] * r[0] + R[1][1] * r[1] + R[1][2] * r[2];
        r[2] = R[2][0] * r[0] + R[2][1] * r[1] + R[2][2] * r[2];
        vel[3 * i + 0] = w[1] * r[2] - w[2] * r[1] + V[0];
        vel[3 * i + 1] = w[2] * r[0] - w[0] * r[2] + V[1];
        vel[3 * i + 2] = w[0] * r[1] - w[1] * r[0] + V[2];
        x[0] = r[0] + c[0] + V[0] * P.dt;
        x[1] = r[1] + c[1] + V[1] * P.dt;
        x[2] = r[2] + c[2] + V[2] * P.dt;
    }
    for (int d = 0; d < 3; ++d) {
        const double t = x[d] - P.dmin[d];
        pos[3 * i + d] = (t - P.W[d] * floor(t / P.W[d])) + P.dmin[d];
        force[3 * i + d] = 0.0;
    }
}

// calculateDensityA, calculateGravityCenter, calculateDensityP (three sums, one list walk)
__global__ void __launch_bounds__(256) k_densities(DevParams P, const int* __restrict__ type,
                                                   const double* __restrict__ pos, const int* __restrict__ nCount,
                                                   const long long* __restrict__ nPtr, const int* __restrict__ nInd,
                                                   double* __restrict__ densA, double* __restrict__ gcen,
                                                   double* __restrict__ volStrainP) {
    // terms: DensityA, the three GravityCenter ones, DensityP
    constexpr int G = kLanes, K = 5;
    __shared__ TermRows<K> T;
    const int g = threadIdx.x & (G - 1);
    const int i = (int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) / G);
    if (i >= P.np) return;  // the whole group
    const int ti = type[i];
    double pi[3];
    for (int d = 0; d < 3; ++d) pi[d] = pos[3 * i + d];
    double s = 0.0;
    const long long b = nPtr[i];
    const int n = nCount[i];
    int jnext = g < n ? nInd[b + g] : 0;  // each lane's next entry loads one round ahead
    for (int base = 0; base < n; base += G) {
        const int jn = base + g, j = jnext;
        jnext = jn + G < n ? nInd[b + jn + G] : 0;
        double t[K] = {0.0, 0.0, 0.0, 0.0, 0.0};
        const int tj = type[j];  // before any branch (entries past the list read particle 0)
        double pj[3];
        for (int d = 0; d < 3; ++d) pj[d] = pos[3 * j + d];
        if (jn < n && i != j) {
            const double ratio = P.ratio[ti][tj];
            Rel q;  // rel() on the loaded positions
            for (int d = 0; d < 3; ++d) q.x[d] = min_image(pj[d], pi[d], P.W[d], P.hW[d]);
            q.r2 = (q.x[0] * q.x[0] + q.x[1] * q.x[1] + q.x[2] * q.x[2]);
            const double r = sqrt(q.r2);
            if (P.radA2 - q.r2 >= 0) t[0] = ratio * wa_k(P.Ka, r, P.radA);
            if (P.radG2 - q.r2 >= 0) {
                const double weight = ratio * wq_k(P.Kg, r, P.radG);
                t[1] = q.x[0] * weight / P.R2g * P.radG;
                t[2] = q.x[1] * weight / P.R2g * P.radG;
                t[3] = q.x[2] * weight / P.R2g * P.radG;
            }
            if (P.radP2 - q.r2 >= 0) t[4] = wq_k(P.Kp, r, P.radP);
        }
        for (int e = 0; e < K; ++e) T.at(e) = t[e];
        wave_sync();
        if (g < K) s = T.add(g, s);
        wave_sync();
    }
    if (g == 0) densA[i] = s;
    else if (g < 4) gcen[3 * i + g - 1] = s;
    else if (g == 4) volStrainP[i] = (s - P.N0p);
}

// calculatePhysicalCoefficients (1704-1735) and the PressureA values (1807-1812)
__global__ void k_coefficients(DevParams P, const int* __restrict__ type, const double* __restrict__ densA,
                               const double* __restrict__ volStrainP, double* __restrict__ mass,
                               double* __restrict__ kappa, double* __restrict__ lambda, double* __restrict__ mu,
                               double* __restrict__ pressA) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P.np) return;
    const int t = type[i];
    mass[i] = P.density[t] * P.V;
    kappa[i] = volStrainP[i] < 0.0 ? 0.0 : P.bulk[t];
    lambda[i] = P.bulkVisc[t];
    mu[i] = P.shear[t];
    double pa = P.cofA[t] * (densA[i] - P.N0a) / P.l;
    if (P.N0a <= densA[i]) pa = 0.0;
    pressA[i] = pa;
}

// calculatePressureA forces (1814-1848), calculateDiffuseInterface (1851-1901),
// calculateGravity (2065-2074), calculateAcceleration (2076-2086)
// kSurf false: every type's CofA is 0 (no surface tension).  The DiffuseInterface
// terms are then zeros of either sign, and fd, which starts at +0, stays +0 under
// fd -= (+-0); they are not formed, and the force keeps every bit.
template <bool kSurf>
__global__ void __launch_bounds__(256) k_forces(DevParams P, const int* __restrict__ type,
                                                const double* __restrict__ pos, const int* __restrict__ nCount,
                                                const long long* __restrict__ nPtr, const int* __restrict__ nInd,
                                                const double* __restrict__ pressA, const double* __restrict__ gcen,
                                                const double* __restrict__ mass, double* __restrict__ force,
                                                double* __restrict__ vel) {
    // terms: PressureA force, the two DiffuseInterface ones (3 each)
    constexpr int G = kLanes, K = kSurf ? 9 : 3;
    __shared__ TermRows<K> T;
    const int g = threadIdx.x & (G - 1);
    const int i = (int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) / G);
    if (i >= P.np) return;  // the whole group
    const int ti = type[i];
    const double ai = P.ai[ti];
    const double aj = P.ai[ti];  // the reference uses i's type for aj (main.cpp:1863)
    const double VoL = P.V / P.l;
    const double pai = pressA[i];
    const double gi[3] = {gcen[3 * i], gcen[3 * i + 1], gcen[3 * i + 2]};
    double s = 0.0;  // lanes 0-2: the PressureA force, lanes 3-5: the DiffuseInterface force
    const long long b = nPtr[i];
    const int n = nCount[i];
    double pi[3];
    for (int d = 0; d < 3; ++d) pi[d] = pos[3 * i + d];
    int jnext = g < n ? nInd[b + g] : 0;  // each lane's next entry loads one round ahead
    for (int base = 0; base < n; base += G) {
        const int jn = base + g, j = jnext;
        jnext = jn + G < n ? nInd[b + jn + G] : 0;
        const int tj = type[j];  // j's values load with its position (past the list: particle 0)
        const double paj = pressA[j];
        double pj[3], gj[3];
        for (int d = 0; d < 3; ++d) {
            pj[d] = pos[3 * j + d];
            gj[d] = kSurf ? gcen[3 * j + d] : 0.0;
        }
        double t[K];
        for (int e = 0; e < K; ++e) t[e] = 0.0;
        if (jn < n) {
            Rel q;  // rel() on the loaded positions
            for (int d = 0; d < 3; ++d) q.x[d] = min_image(pj[d], pi[d], P.W[d], P.hW[d]);
            q.r2 = (q.x[0] * q.x[0] + q.x[1] * q.x[1] + q.x[2] * q.x[2]);
            if (i != j && q.r2 != 0.0) {
                const double rij_ = P.ratio[ti][tj], rji_ = P.ratio[tj][ti];
                if (P.radA2 - q.r2 > 0) {
                    const double r = sqrt(q.r2);
                    const double dwij = rij_ * dwadr_k(P.Ka, P.invA, r, P.radA);
                    const double dwji = rji_ * dwadr_k(P.Ka, P.invA, r, P.radA);
                    for (int d = 0; d < 3; ++d) t[d] = (pai * dwij + paj * dwji) * (q.x[d] / r) * P.V;
                }
                if (kSurf && P.radG2 - q.r2 > 0) {
                    const double r = sqrt(q.r2);
                    const double wij = rij_ * wq_k(P.Kg, r, P.radG);
                    const double wji = rji_ * wq_k(P.Kg, r, P.radG);
                    for (int d = 0; d < 3; ++d)
                        t[3 + d] = (aj * gj[d] * wji - ai * gi[d] * wij) / P.R2g * P.radG * VoL;
                    const double dwij = rij_ * dwq_k(P.Kg, P.m2G, r, P.radG);
                    const double dwji = rji_ * dwq_k(P.Kg, P.m2G, r, P.radG);
                    double gr = 0.0;
                    for (int d = 0; d < 3; ++d) gr += (aj * gj[d] * dwji - ai * gi[d] * dwij) * q.x[d];
                    for (int d = 0; d < 3; ++d) t[6 + d] = (gr) * (q.x[d] / r) / P.R2g * P.radG * VoL;
                }
            }
        }
        for (int e = 0; e < K; ++e) T.at(e) = t[e];
        wave_sync();
        if (g < 3) s = T.add(g, s);
        if (kSurf && g >= 3 && g < 6) {  // both terms of an entry, then the next entry's
            const double* t1 = T.v[threadIdx.x / G][g];
            const double* t2 = T.v[threadIdx.x / G][g + 3];
#pragma unroll 8
            for (int o = 0; o < G; ++o) {
                s -= t1[o];
                s -= t2[o];
            }
        }
        wave_sync();
    }
    const double fd = __shfl_down(s, 3, G);
    if (g >= 3) return;
    double F = force[3 * i + g];
    F += s;
    F += kSurf ? fd : 0.0;
    if (i < P.nf) {
        const double m = mass[i];
        F += m * P.gravity[g];
        vel[3 * i + g] += F / m * P.dt;
    }
    force[3 * i + g] = F;
}

// calculateMatrixA values (2251-2335): viscous blocks, inertia, wall terms of b.
// kBlk: also the factored form's level-0 run sums (blk, from the run starts): lane q sums
// the -alpha r r^T (the negated blocks; 0 beyond RadiusV and for the self entry) of the
// fluid entries in visited cell q's run, all cells at a time.  There the blocks are not
// stored and the coefficients are alpha r r^T, six of them and three divisions an entry:
// the nine of the reference, ((((visc mu) e_s) e_r) w'/d), take fourteen, and FP64 divisions
// bound the kernel (3.7 ms on the 1M scene, of which 180M pairs' divisions about 2).
template <bool kBlk>
__global__ void __launch_bounds__(256, 4) k_matrix_a(DevParams P, const int* __restrict__ type,
                                                  const double* __restrict__ pos, const double* __restrict__ vel,
                                                  const double* __restrict__ mass, const double* __restrict__ mu,
                                                  const int* __restrict__ nCount, const int* __restrict__ nFluid,
                                                  const long long* __restrict__ nPtr, const int* __restrict__ nInd,
                                                  const long long* __restrict__ start, int* __restrict__ acol,
                                                  double* __restrict__ aval, int* __restrict__ selfIdx,
                                                  double* __restrict__ b, double* __restrict__ falpha,
                                                  double* __restrict__ fdiag, int* __restrict__ fwrap,
                                                  const unsigned short* __restrict__ runStart,
                                                  double* __restrict__ blk) {
    // terms: the 3x3 coefficients (kBlk: 00 01 02 11 12 22), then a wall neighbour's velocity
    constexpr int G = kLanes, C = kBlk ? 6 : 9, K = C + 3;
    __shared__ TermRows<K> T;
    __shared__ int wall[256];  // a wall neighbour inside RadiusV
    const int g = threadIdx.x & (G - 1), grp = threadIdx.x / G;
    const int i = (int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) / G);
    if (i >= P.nf) return;  // the whole group
    double s = 0.0, sv = 0.0;  // lanes 0..C-1: the diagonal block; lanes 0-2: the wall terms of b
    // lane g: the runs (upper triangles) of cells g, g + G
    constexpr int R = kBlk ? (kBlkRuns + G - 1) / G : 1;
    double run[R][6];
    for (int c = 0; c < R; ++c)
        for (int e = 0; e < 6; ++e) run[c][e] = 0.0;
    const double mui = mu[i];
    const long long b0 = nPtr[i];
    const int nfl = nFluid[i], nc = nCount[i];
    const long long sb = start[i / kSlice];
    const int lane = i % kSlice;
    // factored form: alpha_ij = visc mu_ij (-w_v'(d)) / d^3, the viscous block being
    // -alpha_ij r r^T (beside the neighbour list; 0 for self and beyond RadiusV)
    auto store_alpha = [&](int k, double a) {
        if (falpha) __builtin_nontemporal_store(a, falpha + b0 + k);
    };
    // the 3x3 blocks are stored unless aval is null (a factored scene that builds its
    // multigrid level 0 from the factored form needs none)
    const bool blocks = !kBlk && aval != nullptr;
    const int nv = (2 * P.range[0] + 1) * (2 * P.range[1] + 1) * (2 * P.range[2] + 1);
    int q0[R], q1[R];
    for (int c = 0; c < R; ++c) {
        const bool in = kBlk && g + c * G < nv;
        q0[c] = in ? runStart[(long long)i * kRuns + g + c * G] : 0;
        q1[c] = in ? runStart[(long long)i * kRuns + g + c * G + 1] : 0;
    }
    int iN = 0;
    bool flags[2] = {false, false};  // FacOp::wrap
    int jnext = g < nc ? nInd[b0 + g] : 0;  // each lane's next entry loads one round ahead
    for (int base = 0; base < nc; base += G) {
        const int jn = base + g;
        const int j = jnext;
        jnext = jn + G < nc ? nInd[b0 + jn + G] : 0;
        int f = 0;
        double t[K];
        for (int e = 0; e < K; ++e) t[e] = 0.0;
        if (jn < nc) {
            if (i == j) {
                iN = jn;
                if (blocks) acol[a_col_index(sb, jn, lane)] = j;
                if (jn < nfl) store_alpha(jn, 0.0);
            } else {
                double alpha = 0.0;
                // j's values load with its position, not after the distance test
                const double muj = mu[j];
                const int tj = type[j];
                const Rel q = rel(P, pos, i, j);
                // factored form: does any pair interact through the periodic boundary
                if (fwrap)
                    for (int d = 0; d < 3; ++d) flags[0] |= fabs(pos[3 * j + d] - pos[3 * i + d]) > P.hW[d];
                const bool inside = q.r2 != 0.0 && P.radV2 - q.r2 > 0;
                if (inside) {
                    const double dij = sqrt(q.r2);
                    const double wdrij = -dwq_k(P.Kv, P.m2V, dij, P.radV);
                    const double muij = 2.0 * (mui * muj) / (mui + muj);
                    if (kBlk || falpha) {
                        alpha = P.visc * muij * wdrij / (dij * dij * dij);
                        if (jn < nfl) flags[1] |= !(muij == P.mu0);
                    }
                    if constexpr (kBlk) {
                        const double ax = alpha * q.x[0], ay = alpha * q.x[1], az = alpha * q.x[2];
                        t[0] = ax * q.x[0];
                        t[1] = ax * q.x[1];
                        t[2] = ax * q.x[2];
                        t[3] = ay * q.x[1];
                        t[4] = ay * q.x[2];
                        t[5] = az * q.x[2];
                    } else {
                        const double e[3] = {q.x[0] / dij, q.x[1] / dij, q.x[2] / dij};
                        for (int r = 0; r < 3; ++r)
                            for (int sdim = 0; sdim < 3; ++sdim)
                                t[3 * r + sdim] = +P.visc * muij * e[sdim] * e[r] * wdrij / dij;
                    }
                    if (is_wall(tj)) {
                        t[C] = vel[3 * j];
                        t[C + 1] = vel[3 * j + 1];
                        t[C + 2] = vel[3 * j + 2];
                        f = 1;
                    }
                }
                if (jn < nfl) {
                    store_alpha(jn, alpha);
                    if (blocks) {
                        acol[a_col_index(sb, jn, lane)] = j;
                        for (int e9 = 0; e9 < 9; ++e9) aval[a_val_index(sb, jn, e9, lane)] = inside ? -t[e9] : 0.0;
                    }
                }
            }
        }
        const bool walls = __ballot(f) != 0;
        for (int e = 0; e < C; ++e) T.at(e) = t[e];
        if (walls) {
            for (int e = C; e < K; ++e) T.at(e) = t[e];
            wall[threadIdx.x] = f;
        }
        wave_sync();
        if (g < C) s = T.add(g, s);
        if (walls && g < 3) {
            const double(&c)[K][G + 2] = T.v[grp];
            const int c0 = kBlk ? g : 3 * g, c1 = kBlk ? (g == 0 ? 1 : g + 2) : 3 * g + 1;
            const int c2 = kBlk ? (g == 0 ? 2 : g + 3) : 3 * g + 2;
            for (int o = 0; o < G; ++o)
                if (wall[grp * G + o]) {
                    sv += c[c0][o] * c[C][o];
                    sv += c[c1][o] * c[C + 1][o];
                    sv += c[c2][o] * c[C + 2][o];
                }
        }
        if constexpr (kBlk) {
            const double(&c)[K][G + 2] = T.v[grp];
#pragma unroll
            for (int h = 0; h < R; ++h) {
                const int lo = q0[h] > base ? q0[h] - base : 0, hi = q1[h] < base + G ? q1[h] - base : G;
                for (int o = lo; o < hi; ++o) {
#pragma unroll
                    for (int e = 0; e < 6; ++e) run[h][e] += -c[e][o];
                }
            }
        }
        wave_sync();
    }
    // once per wavefront and behind a look: an atomic per entry took matrix A from 1.2 to
    // 5.5 ms in a scene of 294k fluid particles of two viscosities, now 0.96
    for (int k = 0; k < 2; ++k)
        if (flags[k] && __hip_atomic_load(fwrap + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
            atomicOr(fwrap + k, 1);
    for (int d = 1; d < G; d <<= 1) {  // the lane that met the self entry tells the others
        const int o = __shfl_xor(iN, d, G);
        iN = o > iN ? o : iN;
    }
    for (int h = 0; h < R; ++h)
        if (kBlk && g + h * G < nv) {
            typedef double dv2 __attribute__((ext_vector_type(2)));
            dv2* o = (dv2*)(blk + ((long long)i * kBlkRuns + g + h * G) * kBlkStride);
            o[0] = dv2{run[h][0], run[h][1]};
            o[1] = dv2{run[h][2], run[h][3]};
            o[2] = dv2{run[h][4], run[h][5]};
        }
    const double coef = mass[i] / P.V / P.dt;
    if (g < C) {
        const int r = kBlk ? (g < 3 ? 0 : g < 5 ? 1 : 2) : g / 3, c = kBlk ? (g < 3 ? g : g < 5 ? g - 2 : 2) : g % 3;
        if (r == c) s += coef;
        if (blocks) aval[a_val_index(sb, iN, g, lane)] = s;
        if (fdiag) {
            fdiag[9 * (long long)i + 3 * r + c] = s;
            if (kBlk) fdiag[9 * (long long)i + 3 * c + r] = s;
        }
    }
    if (g == 0) selfIdx[i] = iN;
    if (g < 3) {
        const double bv = 0.0 + sv;
        b[3 * i + g] = bv + coef * vel[3 * i + g];
    }
}

// calculateMatrixC values (2463-2507): C[3i+r][k] = e_r * (-w'_p).  Also
// D[3i+r][k] = C[3i+r][k] * Lambda[k], the left factor of every product of the
// C Lambda C^T sum (main.cpp:2614 evaluates (C_ik * Lambda_k) * C_jk).
__global__ void __launch_bounds__(256) k_matrix_c(DevParams P, const double* __restrict__ pos,
                                                  const int* __restrict__ nCountP, const long long* __restrict__ nPtrP,
                                                  const int* __restrict__ nIndP, const double* __restrict__ lambda,
                                                  double* __restrict__ cval, double* __restrict__ dval) {
    constexpr int G = kLanesP, K = 3;  // terms: the C block of an entry
    __shared__ double tb[256 * K];
    __shared__ int tf[256];  // bit 0: the self entry, bit 1: inside RadiusP
    const int g = threadIdx.x & (G - 1);
    const int i = (int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) / G);
    const bool own = i < P.nf;
    int iN = 0;
    double self[3] = {0.0, 0.0, 0.0};
    const long long b0 = own ? nPtrP[i] : 0;
    const int n = own ? nCountP[i] : 0;
    for (int base = 0; base < n; base += G) {
        const int jn = base + g;
        int f = 0;
        double c3[3] = {0.0, 0.0, 0.0};
        if (jn < n) {
            const int j = nIndP[b0 + jn];
            if (i == j) {
                f = 1;
            } else {
                const Rel q = rel(P, pos, i, j);
                if (q.r2 != 0.0 && P.radP2 - q.r2 > 0) {
                    const double dij = sqrt(q.r2);
                    const double e[3] = {q.x[0] / dij, q.x[1] / dij, q.x[2] / dij};
                    const double wpdrij = -dwq_k(P.Kp, P.m2P, dij, P.radP);
                    for (int r = 0; r < 3; ++r) c3[r] = e[r] * wpdrij;
                    f = 2;
                }
                // the self entry's block is written once its sum is complete
                for (int r = 0; r < 3; ++r) cval[3 * (b0 + jn) + r] = c3[r];
                if (dval) {  // D = C Lambda, read only by C Lambda C^T (assembled form)
                    const double lk = lambda[j];
                    for (int r = 0; r < 3; ++r) dval[3 * (b0 + jn) + r] = c3[r] * lk;
                }
            }
        }
        for (int e = 0; e < K; ++e) tb[K * threadIdx.x + e] = c3[e];
        tf[threadIdx.x] = f;
        wave_sync();
        if (g == 0)
            for (int u = 0; u < G && base + u < n; ++u) {
                const int sl = threadIdx.x + u;
                const int fu = tf[sl];
                if (fu & 1) iN = base + u;
                if (fu & 2)
                    for (int r = 0; r < 3; ++r) self[r] += tb[K * sl + r];
            }
        wave_sync();
    }
    if (g != 0 || !own) return;
    for (int r = 0; r < 3; ++r) cval[3 * (b0 + iN) + r] = self[r];
    if (dval) {
        const double li = lambda[i];
        for (int r = 0; r < 3; ++r) dval[3 * (b0 + iN) + r] = self[r] * li;
    }
}

// VectorP, main.cpp:2510-2549
__global__ void k_vector_p(DevParams P, const int* __restrict__ type, const double* __restrict__ pos,
                           const double* __restrict__ vel, const double* __restrict__ kappa,
                           const double* __restrict__ lambda, const double* __restrict__ volStrainP,
                           const int* __restrict__ nCountP, const long long* __restrict__ nPtrP,
                           const int* __restrict__ nIndP, double* __restrict__ vecP) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P.np) return;
    double pv = 0.0;
    if (volStrainP[i] > 0.0) pv = kappa[i] * volStrainP[i];
    const bool walli = is_wall(type[i]);
    const double li = lambda[i];
    const double pi[3] = {pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]};
    double sum = 0.0;
    const long long b0 = nPtrP[i];
    const int n = nCountP[i];
    // U entries at a time: columns, then types and positions, load together (past the
    // end: the last entry again, not visited); a pair adds terms only when i or j is a
    // wall, so fluid pairs stop after the distance test
    constexpr int U = 4;
    for (int jb = 0; jb < n; jb += U) {
        int jj[U], tj[U];
        double pj[U][3];
#pragma unroll
        for (int u = 0; u < U; ++u) jj[u] = nIndP[b0 + (jb + u < n ? jb + u : n - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            tj[u] = type[jj[u]];
            for (int d = 0; d < 3; ++d) pj[u][d] = pos[3 * jj[u] + d];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = jj[u];
            if (jb + u >= n || i == j) continue;
            Rel q;  // rel() on the loaded positions
            for (int d = 0; d < 3; ++d) q.x[d] = min_image(pj[u][d], pi[d], P.W[d], P.hW[d]);
            q.r2 = (q.x[0] * q.x[0] + q.x[1] * q.x[1] + q.x[2] * q.x[2]);
            if (q.r2 == 0.0) continue;
            const bool wallj = is_wall(tj[u]);
            if (P.radP2 - q.r2 > 0 && (walli || wallj)) {
                const double dij = sqrt(q.r2);
                const double e[3] = {q.x[0] / dij, q.x[1] / dij, q.x[2] / dij};
                const double wpdrij = -dwq_k(P.Kp, P.m2P, dij, P.radP);
                for (int s = 0; s < 3; ++s) {
                    if (walli) {
                        const double coef = +e[s] * wpdrij;
                        sum += li * coef * vel[3 * i + s];
                    }
                    if (wallj) {
                        const double coef = -e[s] * wpdrij;
                        sum += li * coef * vel[3 * j + s];
                    }
                }
            }
        }
    }
    vecP[i] = pv + sum;
}

// b -= C P (multiplyMatrixC, 2575-2584), accumulated directly into b
__global__ void __launch_bounds__(256) k_b_minus_cp(DevParams P, const int* __restrict__ nCountP,
                                                    const long long* __restrict__ nPtrP,
                                                    const int* __restrict__ nIndP, const double* __restrict__ cval,
                                                    const double* __restrict__ vecP, double* __restrict__ b) {
    constexpr int G = kLanesP, K = 3;  // terms: c_r * P_k
    __shared__ double tb[256 * K];
    const int g = threadIdx.x & (G - 1);
    const int i = (int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) / G);
    const bool own = i < P.nf;
    double b0 = own ? b[3 * i] : 0.0, b1 = own ? b[3 * i + 1] : 0.0, b2 = own ? b[3 * i + 2] : 0.0;
    const long long p0 = own ? nPtrP[i] : 0;
    const int n = own ? nCountP[i] : 0;
    for (int base = 0; base < n; base += G) {
        const int jn = base + g;
        double t[K] = {0.0, 0.0, 0.0};
        if (jn < n) {
            const double pk = vecP[nIndP[p0 + jn]];
            const double* c = &cval[3 * (p0 + jn)];
            for (int r = 0; r < 3; ++r) t[r] = c[r] * pk;
        }
        for (int e = 0; e < K; ++e) tb[K * threadIdx.x + e] = t[e];
        wave_sync();
        if (g == 0)
            for (int u = 0; u < G && base + u < n; ++u) {
                const double* tu = tb + K * (threadIdx.x + u);
                b0 -= tu[0];
                b1 -= tu[1];
                b2 -= tu[2];
            }
        wave_sync();
    }
    if (g != 0 || !own) return;
    b[3 * i] = b0;
    b[3 * i + 1] = b1;
    b[3 * i + 2] = b2;
}

// A += C Lambda C^T (multiplyMatrixC, 2586-2642): for each fluid i and each of its
// fluid neighbours j, the sum of D_ik (x) C_jk over the k in both P-neighbour lists
// (D = C*Lambda, left to right as the reference) in ascending order of k, added to the
// 3x3 block (i, j).  Workgroup = one slice of 64 particles, lane = particle; the
// wavefronts of gridDim.y workgroups share its block pairs.  The FP32 copy of the
// finished block is written when aval32 is non-null.
//
// i's list is a hash table in LDS, entry k << 6 | place, four to a bucket of one 16-byte
// read (a bucket is full before its successor takes entries).  A thread looks up the
// entries of j's list, four under way at a time; both lists ascend, so the t-th hit of
// one is the t-th of the other and the hits are two bit masks, from which the products
// are added without a search.  A lookup replaces two steps of a merge, and the lists
// need no copy in LDS: the merge kernel's copies (52 KB per workgroup of four
// wavefronts) left it waiting at three workgroups per CU.
// The values (0.8 GB read and written at 64k particles) go by pairs of blocks, whole lines:
// a block at a time moved 4.0 GB and took 1.22 ms.  0.90 ms at 64k particles (the merge
// kernel 1.67), 2.78 at 198k (3.84); with up to 16 workgroups to a slice 32 us at 216
// (367) and 100 us at 9k (516).  The gathers of the lists and of C and D, a cache line per
// lane, bound it next.
constexpr int kCacBuckets = 32;
__device__ inline unsigned cac_bucket(int k) { return ((unsigned)k * 0x9E3779B1u) >> 27; }

__global__ void __launch_bounds__(256) k_cac(DevParams P, const int* __restrict__ nFluid,
                                             const int* __restrict__ nCountP, const long long* __restrict__ nPtrP,
                                             const int* __restrict__ nIndP, const double* __restrict__ cval,
                                             const double* __restrict__ dval, const long long* __restrict__ start,
                                             const int* __restrict__ acol, double* __restrict__ aval,
                                             float* __restrict__ aval32) {
    typedef double dv2 __attribute__((ext_vector_type(2)));
    constexpr unsigned kEmpty = 0xffffffffu;
    __shared__ uint4 tab[kSlice][kCacBuckets];
    const int slice = blockIdx.x, base = slice * kSlice, t = threadIdx.x;
    for (int e = t; e < kSlice * kCacBuckets; e += 256) (&tab[0][0])[e] = uint4{kEmpty, kEmpty, kEmpty, kEmpty};
    __syncthreads();
    {  // four threads per list
        const int l = t / 4, i = base + l;
        if (i < P.nf) {
            const long long p = nPtrP[i];
            const int n = nCountP[i];
            for (int a = t & 3; a < n; a += 4) {
                const int k = nIndP[p + a];
                unsigned* const T = (unsigned*)tab[l];
                unsigned s = 4 * cac_bucket(k);  // at most 64 entries in 128 slots: ends
                while (atomicCAS(&T[s], kEmpty, (unsigned)k << 6 | a) != kEmpty) s = (s + 1) & (4 * kCacBuckets - 1);
            }
        }
    }
    __syncthreads();
    const int lane = t % kSlice, wave = t / kSlice;
    const int i = base + lane;
    if (i >= P.nf) return;
    const int nfl = nFluid[i];
    const double* di = dval + 3 * nPtrP[i];
    const long long sb = start[slice];
    const uint4* const ti = tab[lane];
    for (int k = 2 * (wave + 4 * blockIdx.y); k < nfl; k += 8 * gridDim.y) {
        int j[2], nj[2];
        long long pj[2];
        const int hn = k + 1 < nfl ? 2 : 1;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            j[h] = acol[a_col_index(sb, k + (h < hn ? h : 0), lane)];
            pj[h] = nPtrP[j[h]];
            nj[h] = h < hn ? nCountP[j[h]] : 0;
        }
        // both blocks of a pair of values are written together: 16 bytes a lane, whole lines
        dv2 v[9];
        double sum[2][9];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const long long p = pj[h];
            const int n = nj[h];
            unsigned long long mi = 0, mj = 0;  // hits: places in i's and in j's list
            for (int c0 = 0; c0 < n; c0 += 4) {
                unsigned q[4], b[4];
                uint4 w[4];
                __builtin_memcpy(q, nIndP + p + c0, 16);  // past the end: not taken (kListSpare)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    b[u] = cac_bucket((int)q[u]);
                    w[u] = ti[b[u]];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    auto hit = [&](const uint4& x) {  // the place, or 64 and more
                        const unsigned y = q[u] << 6;
                        const unsigned m0 = min(x.x ^ y, x.y ^ y), m1 = min(x.z ^ y, x.w ^ y);
                        return min(m0, m1);
                    };
                    unsigned a = hit(w[u]);
                    while (a >= 64 && w[u].w != kEmpty) {  // 64 entries leave a bucket that isn't full
                        b[u] = (b[u] + 1) & (kCacBuckets - 1);
                        w[u] = ti[b[u]];
                        a = hit(w[u]);
                    }
                    if (a < 64 && c0 + u < n) {
                        mi |= 1ull << a;
                        mj |= 1ull << (c0 + u);
                    }
                }
            }
            if (h == 1)
#pragma unroll
                for (int e = 0; e < 9; ++e) v[e] = *(const dv2*)(aval + a_val_index(sb, k, e, lane));
#pragma unroll
            for (int e = 0; e < 9; ++e) sum[h][e] = 0.0;
            double c[3], d[3];
            auto load = [&]() {
                const double* cj = cval + (mj ? 3 * (p + __builtin_ctzll(mj)) : 0);
                const double* da = mi ? di + 3 * __builtin_ctzll(mi) : dval;
#pragma unroll
                for (int e = 0; e < 3; ++e) {
                    c[e] = cj[e];
                    d[e] = da[e];
                }
            };
            load();
            while (mj) {
                const double c0 = c[0], c1 = c[1], c2 = c[2], d0 = d[0], d1 = d[1], d2 = d[2];
                mi &= mi - 1;
                mj &= mj - 1;
                load();  // the next hit's
                sum[h][0] += d0 * c0; sum[h][1] += d0 * c1; sum[h][2] += d0 * c2;
                sum[h][3] += d1 * c0; sum[h][4] += d1 * c1; sum[h][5] += d1 * c2;
                sum[h][6] += d2 * c0; sum[h][7] += d2 * c1; sum[h][8] += d2 * c2;
            }
        }
#pragma unroll
        for (int e = 0; e < 9; ++e) {
            v[e][0] += sum[0][e];
            v[e][1] += sum[1][e];  // past the row's last block: a value that is never read
            *(dv2*)(aval + a_val_index(sb, k, e, lane)) = v[e];
            if (aval32)
                for (int h = 0; h < hn; ++h) aval32[a_val32_index(sb, k + h, e, lane)] = (float)v[e][h];
        }
    }
}

// The same by merging the lists, for lists of more than 64 entries.  The products are a
// function of the two places: written out in the loop, they made the compiler copy the
// heads of the lists behind a wait for their loads (14.4 against 12.8 ms at 4.1k particles
// with lists of about 70 entries)
__global__ void __launch_bounds__(256) k_cac_merge(DevParams P, const int* __restrict__ nFluid,
                                                   const int* __restrict__ nCountP,
                                                   const long long* __restrict__ nPtrP,
                                                   const int* __restrict__ nIndP, const double* __restrict__ cval,
                                                   const double* __restrict__ dval,
                                                   const long long* __restrict__ start,
                                                   const int* __restrict__ acol, double* __restrict__ aval,
                                                   float* __restrict__ aval32) {
    const int slice = blockIdx.x;
    const int lane = threadIdx.x % kSlice, wave = threadIdx.x / kSlice;
    const int i = slice * kSlice + lane;
    if (i >= P.nf) return;
    const int nfl = nFluid[i];
    const long long pi = nPtrP[i];
    const int ni = nCountP[i];
    const int* ki = nIndP + pi;
    const double* di = dval + 3 * pi;
    const long long sb = start[slice];
    for (int k = wave; k < nfl; k += 4) {
        const int j = acol[a_col_index(sb, k, lane)];
        const long long pj = nPtrP[j];
        const int nj = nCountP[j];
        const int* kj = nIndP + pj;
        double sum[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        auto add = [&](int a, int c) {  // sum += D_i,k (x) C_j,k for the shared k
            const double* cj = &cval[3 * (pj + c)];
            const double c0 = cj[0], c1 = cj[1], c2 = cj[2];
            const double d0 = di[3 * a], d1 = di[3 * a + 1], d2 = di[3 * a + 2];
            sum[0] += d0 * c0; sum[1] += d0 * c1; sum[2] += d0 * c2;
            sum[3] += d1 * c0; sum[4] += d1 * c1; sum[5] += d1 * c2;
            sum[6] += d2 * c0; sum[7] += d2 * c1; sum[8] += d2 * c2;
        };
        int a = 0, c = 0;
        int ka = ni > 0 ? ki[0] : 0;
        int kc = nj > 0 ? kj[0] : 0;
        while (a < ni && c < nj) {
            if (ka == kc) {
                add(a, c);
                a++;
                c++;
                if (a < ni) ka = ki[a];
                if (c < nj) kc = kj[c];
            } else if (ka < kc) {
                a++;
                if (a < ni) ka = ki[a];
            } else {
                c++;
                if (c < nj) kc = kj[c];
            }
        }
        for (int e9 = 0; e9 < 9; ++e9) {
            const long long at = a_val_index(sb, k, e9, lane);
            const double v = aval[at] + sum[e9];
            aval[at] = v;
            if (aval32) aval32[a_val32_index(sb, k, e9, lane)] = (float)v;
        }
    }
}

}  // namespace

void launch_kinematics(hipStream_t st, const DevParams& P, const WallKin& wk, const int* type, double* pos,
                       double* vel, double* force) {
    hipLaunchKernelGGL(k_kinematics, dim3(nblk(P.np, 256)), dim3(256), 0, st, P, wk, type, pos, vel, force);
}

void launch_densities(hipStream_t st, const DevParams& P, const int* type, const double* pos, const int* nCount,
                      const long long* nPtr, const int* nInd, double* densA, double* gcen, double* volStrainP) {
    hipLaunchKernelGGL(k_densities, dim3(nblk((long long)kLanes * P.np, 256)), dim3(256), 0, st, P, type, pos, nCount,
                       nPtr, nInd, densA, gcen, volStrainP);
}

void launch_coefficients(hipStream_t st, const DevParams& P, const int* type, const double* densA,
                         const double* volStrainP, double* mass, double* kappa, double* lambda, double* mu,
                         double* pressA) {
    hipLaunchKernelGGL(k_coefficients, dim3(nblk(P.np, 256)), dim3(256), 0, st, P, type, densA, volStrainP, mass,
                       kappa, lambda, mu, pressA);
}

void launch_forces(hipStream_t st, const DevParams& P, const int* type, const double* pos, const int* nCount,
                   const long long* nPtr, const int* nInd, const double* pressA, const double* gcen,
                   const double* mass, double* force, double* vel) {
    const bool surf = !(P.ai[0] == 0.0 && P.ai[1] == 0.0 && P.ai[2] == 0.0 && P.ai[3] == 0.0);
    if (surf)
        hipLaunchKernelGGL(k_forces<true>, dim3(nblk((long long)kLanes * P.np, 256)), dim3(256), 0, st, P, type, pos,
                           nCount, nPtr, nInd, pressA, gcen, mass, force, vel);
    else
        hipLaunchKernelGGL(k_forces<false>, dim3(nblk((long long)kLanes * P.np, 256)), dim3(256), 0, st, P, type, pos,
                           nCount, nPtr, nInd, pressA, gcen, mass, force, vel);
}

void launch_matrix_a(hipStream_t st, const DevParams& P, const int* type, const double* pos, const double* vel,
                     const double* mass, const double* mu, const int* nCount, const int* nFluid,
                     const long long* nPtr, const int* nInd, ASlices A, int* selfIdx, double* b, double* alpha,
                     double* diag, int* wrap, const unsigned short* runStart, double* blk) {
    const dim3 grid(nblk((long long)kLanes * P.nf, 256));
    if (blk && runStart)
        hipLaunchKernelGGL(k_matrix_a<true>, grid, dim3(256), 0, st, P, type, pos, vel, mass, mu, nCount, nFluid, nPtr,
                           nInd, A.start, A.col, A.val, selfIdx, b, alpha, diag, wrap, runStart, blk);
    else
        hipLaunchKernelGGL(k_matrix_a<false>, grid, dim3(256), 0, st, P, type, pos, vel, mass, mu, nCount, nFluid,
                           nPtr, nInd, A.start, A.col, A.val, selfIdx, b, alpha, diag, wrap, nullptr, nullptr);
}

void launch_matrix_c(hipStream_t st, const DevParams& P, const double* pos, const int* nCountP,
                     const long long* nPtrP, const int* nIndP, const double* lambda, double* cval, double* dval) {
    hipLaunchKernelGGL(k_matrix_c, dim3(nblk((long long)kLanesP * P.nf, 256)), dim3(256), 0, st, P, pos, nCountP,
                       nPtrP, nIndP, lambda, cval, dval);
}

void launch_vector_p(hipStream_t st, const DevParams& P, const int* type, const double* pos, const double* vel,
                     const double* kappa, const double* lambda, const double* volStrainP, const int* nCountP,
                     const long long* nPtrP, const int* nIndP, double* vecP) {
    hipLaunchKernelGGL(k_vector_p, dim3(nblk(P.np, 128)), dim3(128), 0, st, P, type, pos, vel, kappa, lambda,
                       volStrainP, nCountP, nPtrP, nIndP, vecP);
}

void launch_b_minus_cp(hipStream_t st, const DevParams& P, const int* nCountP, const long long* nPtrP,
                       const int* nIndP, const double* cval, const double* vecP, double* b) {
    hipLaunchKernelGGL(k_b_minus_cp, dim3(nblk((long long)kLanesP * P.nf, 256)), dim3(256), 0, st, P, nCountP, nPtrP,
                       nIndP, cval, vecP, b);
}

void launch_cac(hipStream_t st, const DevParams& P, const int* nFluid, const int* nCountP, const long long* nPtrP,
                const int* nIndP, const double* cval, const double* dval, ASlices A, int maxP) {
    if (A.nslices == 0) return;
    // a hash entry has 6 bits for the place in the list and 26 for the particle (the last
    // number marks an empty one)
    if (maxP > 64 || P.np >= (1 << 26) - 1) {
        hipLaunchKernelGGL(k_cac_merge, dim3(A.nslices), dim3(256), 0, st, P, nFluid, nCountP, nPtrP, nIndP, cval, dval,
                           A.start, A.col, A.val, A.val32);
        return;
    }
    // few slices: up to 16 workgroups share one, towards 16 workgroups per CU
    const int want = (4096 + A.nslices - 1) / A.nslices, y = want > 16 ? 16 : want;
    hipLaunchKernelGGL(k_cac, dim3(A.nslices, y), dim3(256), 0, st, P, nFluid, nCountP, nPtrP, nIndP, cval, dval,
                       A.start, A.col, A.val, A.val32);
}

}  // namespace mph
