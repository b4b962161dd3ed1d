// mph_cells.hip -- cell list, bitonic particle order and neighbour search on gfx950.
//
// Replaces calculateCellParticle (source/main.cpp:1164-1379) and calculateNeighbor
// (1382-1667).  The particle order is the reference's bitonic network, emulated
// exactly (it is not stable, so a radix sort would order ties differently): the
// passes with distance < 8192 run inside a workgroup, the wider ones as global passes.
// Neighbour lists come out ascending (fluid block, then wall block) because the
// 27 (9 in 2D) cells are visited in ascending CellId, as in the reference.
#include "mph_kernels.h"

namespace mph {

namespace {

constexpr int kSortBlock = 8192;  // keys per workgroup (64 KB of LDS)
constexpr int kSortThreads = 1024;
constexpr int kScanShare = 32768;  // particles from which four share a wavefront of the neighbour search

__device__ inline int cell_id(const DevParams& P, int cx, int cy, int cz) {  // CellId, main.cpp:109-113
    const int* C = P.C;
    if (P.dim == 2) return ((cx) % C[0] + C[0]) % C[0] * C[1] + ((cy) % C[1] + C[1]) % C[1];
    return ((cx) % C[0] + C[0]) % C[0] * C[1] * C[2] + ((cy) % C[1] + C[1]) % C[1] * C[2] +
           ((cz) % C[2] + C[2]) % C[2];
}

// key of main.cpp:1168-1186, packed with the particle index for the sort
__global__ void k_hash(DevParams P, const double* __restrict__ pos, const int* __restrict__ type,
                       uint64_t* __restrict__ keys) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P.p2) return;
    if (i < P.np) {
        const int cx = ((int)floor((pos[3 * i + 0] - P.dmin[0]) / P.cw[0])) % P.C[0];
        const int cy = ((int)floor((pos[3 * i + 1] - P.dmin[1]) / P.cw[1])) % P.C[1];
        const int cz = ((int)floor((pos[3 * i + 2] - P.dmin[2]) / P.cw[2])) % P.C[2];
        int key = cell_id(P, cx, cy, cz);
        if (is_wall(type[i])) key += P.T;
        keys[i] = ((uint64_t)(uint32_t)key << 32) | (uint32_t)i;
    } else {
        keys[i] = ((uint64_t)(uint32_t)(2 * P.T) << 32) | (uint32_t)P.np;
    }
}

// one compare-exchange of the network of main.cpp:1190-1211 for global index i
__device__ inline void cmp_swap(uint64_t& a, uint64_t& b, bool up) {
    const uint32_t ka = (uint32_t)(a >> 32), kb = (uint32_t)(b >> 32);
    if ((ka > kb) == up) {
        const uint64_t t = a;
        a = b;
        b = t;
    }
}

__device__ inline int pair_lo(int t, int logd) {  // t-th pair (lo index) at distance 2^logd
    return ((t >> logd) << (logd + 1)) | (t & ((1 << logd) - 1));
}

// A block of n <= kSortBlock keys lives in registers, eight consecutive keys per thread: a
// pass at distance 1, 2 or 4 stays inside a thread, at 8 to 256 inside a wavefront (DPP and
// shuffles) and only from 512 on goes through LDS (10 of the 91 passes of 8192 keys).  The issue
// of one CU bounds it: 36 us for 4096 keys, 60 for 8192, 16 per merge.  With every pass in LDS,
// blocks of 2048 keys took 40 us and 10 per merge, and the passes from 2048 on a launch each: 36
// launches per sort of the 64k drop, now 21.  Blocks of 2048 keys in registers take 29 and 8 us,
// but their launches cost the smaller scenes more (batch of 12 scenes 20.3 against 19.6 ms).
constexpr int kSortKeys = kSortBlock / kSortThreads;
static_assert(kSortKeys == 8, "three distances inside a thread, six inside a wavefront");

// the compare-exchange of all keys of a thread at distance 2^L < kSortKeys; gi: its first index
template <int L>
__device__ inline void pass_thread(uint64_t (&v)[kSortKeys], int gi, int iMain) {
#pragma unroll
    for (int k = 0; k < kSortKeys; ++k)
        if (!(k & (1 << L))) cmp_swap(v[k], v[k | (1 << L)], (((gi + k) >> iMain) & 2) == 0);
}

// another lane's key without LDS: quad_perm [1,0,3,2] (0xB1, lane ^ 1) and [2,3,0,1] (0x4E,
// lane ^ 2), row_ror:8 (0x128, lane ^ 8 within a row of 16)
template <int kCtl>
__device__ inline uint64_t lane_dpp(uint64_t v) {
    const int lo = (int)(uint32_t)v, hi = (int)(uint32_t)(v >> 32);
    const uint32_t a = (uint32_t)__builtin_amdgcn_update_dpp(lo, lo, kCtl, 0xf, 0xf, false);
    const uint32_t b = (uint32_t)__builtin_amdgcn_update_dpp(hi, hi, kCtl, 0xf, 0xf, false);
    return ((uint64_t)b << 32) | a;
}

// the pass of stage iMain at distance 2^logd < n; every thread of the workgroup calls it
__device__ inline void block_pass(uint64_t (&v)[kSortKeys], int gi, int logd, int iMain, uint64_t* sh) {
    if (logd == 0) return pass_thread<0>(v, gi, iMain);
    if (logd == 1) return pass_thread<1>(v, gi, iMain);
    if (logd == 2) return pass_thread<2>(v, gi, iMain);
    const int t = threadIdx.x, td = 1 << (logd - 3);  // the partner is thread t ^ td
    uint64_t o[kSortKeys];
    if (td == 1) {
#pragma unroll
        for (int k = 0; k < kSortKeys; ++k) o[k] = lane_dpp<0xB1>(v[k]);
    } else if (td == 2) {
#pragma unroll
        for (int k = 0; k < kSortKeys; ++k) o[k] = lane_dpp<0x4E>(v[k]);
    } else if (td == 8) {
#pragma unroll
        for (int k = 0; k < kSortKeys; ++k) o[k] = lane_dpp<0x128>(v[k]);
    } else if (td < 64) {
#pragma unroll
        for (int k = 0; k < kSortKeys; ++k) o[k] = __shfl_xor((unsigned long long)v[k], td, 64);
    } else {
        __syncthreads();  // the previous pass through LDS has been read
#pragma unroll
        for (int k = 0; k < kSortKeys; ++k) sh[k * kSortThreads + t] = v[k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kSortKeys; ++k) o[k] = sh[k * kSortThreads + (t ^ td)];
    }
    const bool lo = !(t & td), up = ((gi >> iMain) & 2) == 0;
#pragma unroll
    for (int k = 0; k < kSortKeys; ++k) {
        const uint32_t a = (uint32_t)((lo ? v[k] : o[k]) >> 32), b = (uint32_t)((lo ? o[k] : v[k]) >> 32);
        if ((a > b) == up) v[k] = o[k];
    }
}

// kMerge: the passes of stage iMain0 with distance < n; else all stages below log2(n).  Keys
// past n (small sorts) take part in no exchange with the others: n is a power of two.
template <bool kMerge>
__global__ void __launch_bounds__(kSortThreads) k_bitonic_block(uint64_t* keys, int n, int logn, int iMain0) {
    __shared__ uint64_t sh[kSortBlock];
    const int base = blockIdx.x * n, at = kSortKeys * threadIdx.x, gi = base + at;
    uint64_t v[kSortKeys];
#pragma unroll
    for (int k = 0; k < kSortKeys; ++k) v[k] = at + k < n ? keys[gi + k] : 0;
    for (int iMain = kMerge ? iMain0 : 0; iMain < (kMerge ? iMain0 + 1 : logn); ++iMain)
        for (int logd = kMerge ? logn - 1 : iMain; logd >= 0; --logd) block_pass(v, gi, logd, iMain, sh);
#pragma unroll
    for (int k = 0; k < kSortKeys; ++k)
        if (at + k < n) keys[gi + k] = v[k];
}

// one pass at distance 2^logd >= block size
__global__ void k_bitonic_global(uint64_t* keys, int npairs, int logd, int iMain) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= npairs) return;
    const int lo = pair_lo(t, logd);
    const int hi = lo | (1 << logd);
    const bool up = ((lo >> iMain) & 2) == 0;
    uint64_t a = keys[lo], b = keys[hi];
    const uint32_t ka = (uint32_t)(a >> 32), kb = (uint32_t)(b >> 32);
    if ((ka > kb) == up) {
        keys[lo] = b;
        keys[hi] = a;
    }
}

// cellStart[c] = number of sorted keys < c, for c in [0, 2T]; this equals the
// cell Begin/End arrays built by boundary detection and scan at main.cpp:1213-1300
// (integer counts, so any evaluation order gives the same values).
__global__ void k_cell_start(DevParams P, const uint64_t* __restrict__ keys, int* __restrict__ cellStart) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c > 2 * P.T) return;
    int lo = 0, hi = P.np;  // first index in [0, np] whose key >= c (keys[np] = 2T)
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if ((int)(keys[mid] >> 32) < c) lo = mid + 1;
        else hi = mid;
    }
    cellStart[c] = lo;
}

// gather-reorder of ParticleIndex/Property/Position/Velocity, main.cpp:1315-1378
__global__ void k_reorder(DevParams P, const uint64_t* __restrict__ keys, const int* __restrict__ type,
                          const int* __restrict__ perm, const double* __restrict__ pos,
                          const double* __restrict__ vel, int* __restrict__ type2, int* __restrict__ perm2,
                          double* __restrict__ pos2, double* __restrict__ vel2, int* __restrict__ cellIndex) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P.np) return;
    const int src = (int)(uint32_t)keys[i];
    cellIndex[i] = (int)(keys[i] >> 32);
    type2[i] = type[src];
    perm2[i] = perm[src];
    for (int d = 0; d < 3; ++d) {
        pos2[3 * i + d] = pos[3 * src + d];
        vel2[3 * i + d] = vel[3 * src + d];
    }
}

// what the neighbour search writes (main.cpp:1406-1511, 1567-1666).  Count pass: the
// counts, `most` and, with lists, the lists themselves in
// per-particle scratch of capM / capP entries; a particle with more raises *overflow,
// which sends the search to the fill pass.  Fill pass: the lists at ptrM / ptrP.
// runStart: for fluid particles where the fluid neighbours of each visited cell start in
// the list (runStart[i][q], q in visiting order, runStart[i][ncells] = fluid count); the
// multigrid level-0 build reads these runs directly.
struct NeighborOut {
    int *nCount, *nFluid, *nCountP;
    int* most;  // [0], [1]: largest P and fluid count of a fluid particle (they size the LDS staging of
                // the C Lambda C^T kernel and the A rows); [2], [3]: largest count and P count of any
    int *listM, *listP;
    int capM, capP;
    const long long *ptrM, *ptrP;
    unsigned short* runStart;
    int* overflow;
};

// One wavefront scans the candidates of U consecutive particles, 64 at a time: the hits'
// ballot gives every lane its place in the list, so the lists come out in the visiting
// order (ascending CellId, main.cpp:1410-1445) with coalesced stores.  Visited cells that
// hold consecutive particles (the three along z) are scanned as one range of about 120
// candidates; U particles of one cell share its ranges and the candidates' coordinates.
// A particle per thread walked its 1100 candidates in series: 460 us for the smallest
// scene, 17 us now; at 1.3M particles its strided list stores also cost, 2.60 ms
// against 2.15 ms (U = 4).
template <int U, bool kFill>
__global__ void __launch_bounds__(256) k_neighbors(DevParams P, const double* __restrict__ pos,
                                                   const int* __restrict__ cellIndex,
                                                   const int* __restrict__ cellStart, NeighborOut O) {
    const int lane = threadIdx.x & 63;
    const int i0 = __builtin_amdgcn_readfirstlane((int)(((long long)blockIdx.x * 256 + threadIdx.x) >> 6) * U);
    if (i0 >= P.np) return;
    const int left = P.np - i0 < U ? P.np - i0 : U;
    double xi[U][3];
    int key[U], n[U], nfl[U], npp[U], rc[U];
    int *lm[U], *lp[U];
    const bool lists = O.listM != nullptr;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int i = i0 + (u < left ? u : 0);
        for (int d = 0; d < 3; ++d) xi[u][d] = pos[3 * (long long)i + d];
        key[u] = cellIndex[i];
        lm[u] = O.listM + (kFill ? O.ptrM[i] : (long long)i * O.capM);
        lp[u] = O.listP + (kFill ? O.ptrP[i] : (long long)i * O.capP);
        n[u] = nfl[u] = npp[u] = rc[u] = 0;
    }
    const int* C = P.C;
    const int nx = 2 * P.range[0] + 1, ny = 2 * P.range[1] + 1, nz = 2 * P.range[2] + 1, nv = nx * ny * nz;
    const double in0 = 0.4 * P.hW[0], in1 = 0.4 * P.hW[1], in2 = 0.4 * P.hW[2];
    unsigned todo = (1u << left) - 1;
    while (todo) {  // the particles of one cell at a time
        int k = key[0];
#pragma unroll
        for (int u = U - 1; u >= 0; --u)
            if (todo >> u & 1) k = key[u];
        unsigned set = 0;
#pragma unroll
        for (int u = 0; u < U; ++u)
            if ((todo >> u & 1) && key[u] == k) set |= 1u << u;
        todo &= ~set;
        // lane q < nv: the particle ranges of visited cell q, fluid and wall
        int lo[2] = {0, 0}, hi[2] = {0, 0};
        if (lane < nv) {
            const int cx = (k / (C[1] * C[2])) % P.T, cy = (k / C[2]) % C[1], cz = k % C[2];
            const int bx = 2 * P.range[0] - (cx + P.range[0]) % C[0], by = 2 * P.range[1] - (cy + P.range[1]) % C[1];
            const int bz = 2 * P.range[2] - (cz + P.range[2]) % C[2];
            const int a = ((bx > 0 ? bx : 0) + lane / (ny * nz)) % nx, b = ((by > 0 ? by : 0) + (lane / nz) % ny) % ny;
            const int c = ((bz > 0 ? bz : 0) + lane % nz) % nz;
            const int jc = cell_id(P, cx - P.range[0] + a, cy - P.range[1] + b, cz - P.range[2] + c);
            lo[0] = cellStart[jc];
            hi[0] = cellStart[jc + 1];
            lo[1] = cellStart[P.T + jc];
            hi[1] = cellStart[P.T + jc + 1];
        }
        int off = hi[0] - lo[0];  // fluid candidates before cell `lane`
        for (int d = 1; d < 32; d <<= 1) {
            const int v = __shfl_up(off, d, 64);
            if (lane >= d) off += v;
        }
        off = lane < nv ? off - (hi[0] - lo[0]) : 0x7fffffff;
#pragma unroll
        for (int wall = 0; wall < 2; ++wall) {
            if (wall) {
                // walls without fluid neighbours skip the wall scan (main.cpp:1474); walls
                // occupy [nf, np) after every sort
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (!(set >> u & 1)) continue;
                    nfl[u] = n[u];
                    if (i0 + u >= P.nf && n[u] == 0) set &= ~(1u << u);
                }
                if (!set) break;
            }
            const int before = __shfl_up(hi[wall], 1, 64);
            unsigned long long starts = __ballot(lane < nv && (lane == 0 || lo[wall] != before));
            int flat = 0;
            while (starts) {
                const int s = __builtin_ctzll(starts);
                starts &= starts - 1;
                const int e = starts ? __builtin_ctzll(starts) : nv;
                const int jlo = __builtin_amdgcn_readlane(lo[wall], s);
                const int jhi = __builtin_amdgcn_readlane(hi[wall], e - 1);
                for (int j0 = jlo; j0 < jhi; j0 += 128) {
                    double c[2][3];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {  // past the end: candidate jhi - 1, not taken
                        const int j = j0 + 64 * h + lane < jhi ? j0 + 64 * h + lane : jhi - 1;
                        for (int d = 0; d < 3; ++d) c[h][d] = pos[3 * (long long)j + d];
                    }
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int j = j0 + 64 * h + lane;
                        if (h && j0 + 64 >= jhi) break;
                        unsigned long long below = 0;  // the chunk's candidates before cell `lane`
                        if (!wall) {
                            const int b = off - flat;
                            below = b <= 0 ? 0 : b >= 64 ? ~0ull : (1ull << b) - 1;
                            flat += 64;  // only the last chunk of a range is shorter
                            if (j0 + 64 * (h + 1) > jhi) flat -= j0 + 64 * (h + 1) - jhi;
                        }
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                            if (!(set >> u & 1)) continue;
                            // min_image of a difference well inside the box is (e + hw) - hw; one
                            // branch for the wavefront instead of one per coordinate
                            double q0 = c[h][0] - xi[u][0], q1 = c[h][1] - xi[u][1], q2 = c[h][2] - xi[u][2];
                            const bool near = fabs(q0) <= in0 && fabs(q1) <= in1 && fabs(q2) <= in2;
                            if (__ballot(!near) == 0) {
                                q0 = q0 + P.hW[0] - P.hW[0];
                                q1 = q1 + P.hW[1] - P.hW[1];
                                q2 = q2 + P.hW[2] - P.hW[2];
                            } else {
                                q0 = min_image(c[h][0], xi[u][0], P.W[0], P.hW[0]);
                                q1 = min_image(c[h][1], xi[u][1], P.W[1], P.hW[1]);
                                q2 = min_image(c[h][2], xi[u][2], P.W[2], P.hW[2]);
                            }
                            const double r2 = q0 * q0 + q1 * q1 + q2 * q2;
                            const bool hit = j < jhi && r2 <= P.maxR2, hitP = hit && r2 <= P.radP2;
                            const unsigned long long M = __ballot(hit), MP = __ballot(hitP);
                            if (kFill || lists) {
                                const int at = n[u] + __builtin_amdgcn_mbcnt_hi((unsigned)(M >> 32),
                                                          __builtin_amdgcn_mbcnt_lo((unsigned)M, 0));
                                const int atP = npp[u] + __builtin_amdgcn_mbcnt_hi((unsigned)(MP >> 32),
                                                             __builtin_amdgcn_mbcnt_lo((unsigned)MP, 0));
                                if (hit && (kFill || at < O.capM)) lm[u][at] = j;
                                if (hitP && (kFill || atP < O.capP)) lp[u][atP] = j;
                                if (!wall) rc[u] += __popcll(M & below);
                            }
                            n[u] += __popcll(M);
                            npp[u] += __popcll(MP);
                        }
                    }
                }
            }
        }
    }
    if (kFill || lists)
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (u < left && i0 + u < P.nf && lane <= nv) O.runStart[(long long)(i0 + u) * kRuns + lane] = (unsigned short)rc[u];
    if (kFill) return;
    int m[4] = {0, 0, 0, 0}, vn = 0, vf = 0, vp = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (u >= left) continue;
        if (i0 + u < P.nf) {
            m[0] = npp[u] > m[0] ? npp[u] : m[0];
            m[1] = nfl[u] > m[1] ? nfl[u] : m[1];
        }
        m[2] = n[u] > m[2] ? n[u] : m[2];
        m[3] = npp[u] > m[3] ? npp[u] : m[3];
        if (lane == u) {
            vn = n[u];
            vf = nfl[u];
            vp = npp[u];
        }
    }
    if (lane < left) {
        O.nCount[i0 + lane] = vn;
        O.nFluid[i0 + lane] = vf;
        O.nCountP[i0 + lane] = vp;
    }
    if (lane < 4) {  // few wavefronts raise a maximum: look before the atomic
        const int v = lane == 0 ? m[0] : lane == 1 ? m[1] : lane == 2 ? m[2] : m[3];
        if (v > __hip_atomic_load(&O.most[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMax(&O.most[lane], v);
    }
    if (lists && lane == 0 && (m[2] > O.capM || m[3] > O.capP)) atomicOr(O.overflow, 1);
}

// the lists from the scratch of the count pass, 32 lanes per particle (coalesced)
__global__ void __launch_bounds__(256) k_neighbor_compact(DevParams P, const int* __restrict__ nCount,
                                                          const int* __restrict__ nCountP,
                                                          const long long* __restrict__ nPtr,
                                                          const long long* __restrict__ nPtrP,
                                                          const int* __restrict__ scrM, int capM,
                                                          const int* __restrict__ scrP, int capP,
                                                          int* __restrict__ nInd, int* __restrict__ nIndP) {
    constexpr int G = 32;
    const int g = threadIdx.x & (G - 1);
    const int i = (int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) / G);
    if (i >= P.np) return;
    const int n = nCount[i], npp = nCountP[i];
    const long long b = nPtr[i], bp = nPtrP[i];
    const int* sm = scrM + (long long)i * capM;
    const int* sp = scrP + (long long)i * capP;
    for (int k = g; k < n; k += G) nInd[b + k] = sm[k];
    for (int k = g; k < npp; k += G) nIndP[bp + k] = sp[k];
}

// ---- exclusive scan of int counts into int64 offsets (out[0]=0, out[n]=total) ----
constexpr int kScanThreads = 256, kScanItems = 8, kScanTile = kScanThreads * kScanItems;

__global__ void __launch_bounds__(kScanThreads) k_scan_tile_sums(const int* __restrict__ in, int n,
                                                                 long long* __restrict__ sums) {
    __shared__ long long red[kScanThreads];
    const int base = blockIdx.x * kScanTile;
    long long s = 0;
    for (int k = 0; k < kScanItems; ++k) {
        const int idx = base + threadIdx.x * kScanItems + k;
        if (idx < n) s += in[idx];
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int h = kScanThreads / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) sums[blockIdx.x] = red[0];
}

__device__ inline long long block_exclusive_scan(long long v, long long* sh, long long& total) {
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int off = 1; off < (int)blockDim.x; off <<= 1) {
        const long long t = (int)threadIdx.x >= off ? sh[threadIdx.x - off] : 0;
        __syncthreads();
        sh[threadIdx.x] += t;
        __syncthreads();
    }
    total = sh[blockDim.x - 1];
    const long long incl = sh[threadIdx.x];
    __syncthreads();
    return incl - v;
}

__global__ void __launch_bounds__(kScanThreads) k_scan_sums(long long* sums, int nt) {
    __shared__ long long sh[kScanThreads];
    long long carry = 0;
    for (int base = 0; base < nt; base += kScanThreads) {
        const int idx = base + threadIdx.x;
        const long long v = idx < nt ? sums[idx] : 0;
        long long total;
        const long long ex = block_exclusive_scan(v, sh, total);
        if (idx < nt) sums[idx] = carry + ex;
        carry += total;
    }
}

__global__ void __launch_bounds__(kScanThreads) k_scan_apply(const int* __restrict__ in, int n,
                                                             const long long* __restrict__ sums,
                                                             long long* __restrict__ out) {
    __shared__ long long sh[kScanThreads];
    const int base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    int v[kScanItems];
    long long s = 0;
    for (int k = 0; k < kScanItems; ++k) {
        v[k] = base + k < n ? in[base + k] : 0;
        s += v[k];
    }
    long long total;
    long long run = block_exclusive_scan(s, sh, total) + sums[blockIdx.x];
    for (int k = 0; k < kScanItems; ++k) {
        run += v[k];
        if (base + k < n) out[base + k + 1] = run;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) out[0] = 0;
}

__global__ void k_slice_width(int nf, int nslices, const int* __restrict__ nFluid, int* __restrict__ width) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nslices) return;
    int w = 0;
    for (int l = 0; l < kSlice; ++l) {
        const int i = s * kSlice + l;
        if (i < nf && nFluid[i] > w) w = nFluid[i];
    }
    width[s] = (w + 3) & ~3;  // block pairs / quads: every slice starts on a multiple of 4
}

inline int nblk(long long n, int bs) { return (int)((n + bs - 1) / bs); }

}  // namespace

void launch_hash(hipStream_t st, const DevParams& P, const double* pos, const int* type, uint64_t* keys) {
    hipLaunchKernelGGL(k_hash, dim3(nblk(P.p2, 256)), dim3(256), 0, st, P, pos, type, keys);
}

void launch_bitonic(hipStream_t st, const DevParams& P, uint64_t* keys) {
    const int n = P.p2 < kSortBlock ? P.p2 : kSortBlock;
    int logn = 0;
    while ((1 << logn) < n) ++logn;
    const int nb = P.p2 / n, nt = n / kSortKeys < 64 ? 64 : n / kSortKeys;
    hipLaunchKernelGGL(k_bitonic_block<false>, dim3(nb), dim3(nt), 0, st, keys, n, logn, 0);
    for (int iMain = logn; iMain < P.p2pow; ++iMain) {
        for (int logd = iMain; logd >= logn; --logd)
            hipLaunchKernelGGL(k_bitonic_global, dim3(nblk(P.p2 / 2, 256)), dim3(256), 0, st, keys, P.p2 / 2, logd,
                               iMain);
        hipLaunchKernelGGL(k_bitonic_block<true>, dim3(nb), dim3(nt), 0, st, keys, n, logn, iMain);
    }
}

void launch_cell_start(hipStream_t st, const DevParams& P, const uint64_t* keys, int* cellStart) {
    hipLaunchKernelGGL(k_cell_start, dim3(nblk(2 * (long long)P.T + 1, 256)), dim3(256), 0, st, P, keys, cellStart);
}

void launch_reorder(hipStream_t st, const DevParams& P, const uint64_t* keys, const int* type, const int* perm,
                    const double* pos, const double* vel, int* type2, int* perm2, double* pos2, double* vel2,
                    int* cellIndex) {
    hipLaunchKernelGGL(k_reorder, dim3(nblk(P.np, 256)), dim3(256), 0, st, P, keys, type, perm, pos, vel, type2,
                       perm2, pos2, vel2, cellIndex);
}

namespace {

// particles per wavefront: four share their cell's candidates where the scene fills the
// GPU's 8192 wavefronts several times over all the same, one otherwise
template <bool kFill>
void neighbors(hipStream_t st, const DevParams& P, const double* pos, const int* cellIndex, const int* cellStart,
               const NeighborOut& O) {
    if (P.np >= kScanShare)
        hipLaunchKernelGGL((k_neighbors<4, kFill>), dim3(nblk(64LL * ((P.np + 3) / 4), 256)), dim3(256), 0, st, P, pos,
                           cellIndex, cellStart, O);
    else
        hipLaunchKernelGGL((k_neighbors<1, kFill>), dim3(nblk(64LL * P.np, 256)), dim3(256), 0, st, P, pos, cellIndex,
                           cellStart, O);
}

}  // namespace

void launch_neighbor_count(hipStream_t st, const DevParams& P, const double* pos, const int* cellIndex,
                           const int* cellStart, int* nCount, int* nFluid, int* nCountP, int* maxFluidP, int* scrM,
                           int capM, int* scrP, int capP, unsigned short* runStart, int* overflow) {
    neighbors<false>(st, P, pos, cellIndex, cellStart,
                     {nCount, nFluid, nCountP, maxFluidP, scrM, scrP, capM, capP, nullptr, nullptr, runStart, overflow});
}

void launch_neighbor_compact(hipStream_t st, const DevParams& P, const int* nCount, const int* nCountP,
                             const long long* nPtr, const long long* nPtrP, const int* scrM, int capM,
                             const int* scrP, int capP, int* nInd, int* nIndP) {
    hipLaunchKernelGGL(k_neighbor_compact, dim3(nblk(32LL * P.np, 256)), dim3(256), 0, st, P, nCount, nCountP, nPtr,
                       nPtrP, scrM, capM, scrP, capP, nInd, nIndP);
}

void launch_neighbor_fill(hipStream_t st, const DevParams& P, const double* pos, const int* cellIndex,
                          const int* cellStart, const long long* nPtr, const long long* nPtrP, int* nInd, int* nIndP,
                          unsigned short* runStart) {
    neighbors<true>(st, P, pos, cellIndex, cellStart,
                    {nullptr, nullptr, nullptr, nullptr, nInd, nIndP, 0, 0, nPtr, nPtrP, runStart, nullptr});
}

int scan_scratch_len(int n) { return nblk(n > 0 ? n : 1, kScanTile); }

void launch_scan_i64(hipStream_t st, const int* in, long long* out, int n, long long* scratch, int scratch_len) {
    const int nt = nblk(n > 0 ? n : 1, kScanTile);
    (void)scratch_len;
    hipLaunchKernelGGL(k_scan_tile_sums, dim3(nt), dim3(kScanThreads), 0, st, in, n, scratch);
    hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(kScanThreads), 0, st, scratch, nt);
    hipLaunchKernelGGL(k_scan_apply, dim3(nt), dim3(kScanThreads), 0, st, in, n, scratch, out);
}

void launch_slice_width(hipStream_t st, int nf, int nslices, const int* nFluid, int* width) {
    hipLaunchKernelGGL(k_slice_width, dim3(nblk(nslices, 256)), dim3(256), 0, st, nf, nslices, nFluid, width);
}

}  // namespace mph
