// mph_kernels.h -- launchers of the HIP kernels (one scene, one stream).
//
// Layouts in HBM (all device pointers):
//   particles    AoS double[np][3] for Position/Velocity/Force (as the reference),
//                double[np] scalars, int Property[np], int perm[np]
//   cell keys    uint64 keys[p2] = (CellIndex << 32) | CellParticle while sorting;
//                int cellIndex[np] (sorted keys), int cellStart[2T+1]
//   neighbours   int64 ptr[np+1], int ind[E]; same for the RadiusP lists
//   A            sliced 3x3-block ELL: slice = 64 consecutive fluid particles,
//                width = max fluid-neighbour count in the slice rounded up to
//                a multiple of 4, sliceStart = prefix sum of widths.  Blocks
//                k = 2m, 2m+1 of a particle form a pair: its two columns are
//                adjacent ints and entry e = 3r+s of both blocks are adjacent
//                values (a_col_index / a_val_index), so a wavefront reads 512 B
//                of columns and 1 KiB (FP64) per entry of a block pair
//                with one 8/16-byte load per lane; the FP32 copy groups four
//                blocks per entry (a_val32_index)
//   C            cval[3*(ptrP[i] + jn) + r] for fluid i, P-neighbour jn
//   multigrid    per level: A stored [shift][row], vectors [row]
//   CR vectors   double[3*nf], row 3i+r as the reference
#pragma once

#include "mph_common.h"

namespace mph {

struct WallKin {  // per wall type: rotation, angular and linear velocity, centre
    double R[4][3][3];
    double omega[4][3];
    double vel[4][3];
    double center[4][3];
};

struct Level {  // geometry + storage of one multigrid level
    int mn[3], mx[3], cnt[3], cs[3];
    int cells, nrow, nshift;
    double* A;     // [nshift][nrow]
    double* invD;  // [nrow]
    double* S[2];  // ping-pong smoother iterate
    double* R;
    double* Q;
    int cur;       // which S buffer holds the current iterate
    float* A32;    // FP32 copy of A for the mixed-precision inner solve (or null)
    int f32;       // smoothers read A32 instead of A
    int lanes;     // sweeps split each row over lanes (small levels; set by the host)
    int ordered;   // sums run in the reference's order (the assembled form, bit for bit);
                   // 0: in fixed shorter chains (the factored form)
    const int* halt;  // the CR stop flag, as DevParams::halt
};

// The V-cycle's small levels, one thread per row, laid out for the one-workgroup cycle
// (body::mg_coarse_cycle) by launch_mg_coarse_pack: a longest run of levels up to the
// coarsest whose rows fit one workgroup.  A 3D row's stencil takes 162 registers of the
// 256 that 512 threads have, a 2D row's 54 of 128.  Depth bounds the coarsest level to
// three cells per axis, so it always fits.
constexpr int kCoarseRows3D = 512, kCoarseRows2D = 1024;
struct CoarsePack {
    double* v;   // [(3 cells + 1)][stride]: stencil values, then invD
    int* i;      // [(cells + 1) / 2 + 6][stride]: LDS places of the stencil cells, meta words
    int* up;     // [rows of level lc-1]: the LDS place of each row's parent
    int stride;  // threads (rows rounded up to whole wavefronts)
    int cells;   // 27, or 9 in 2D
    int ordered; // Level::ordered
};
inline size_t coarse_pack_values(int cells, int stride) { return (size_t)(3 * cells + 1) * stride; }
inline size_t coarse_pack_ints(int cells, int stride) { return (size_t)((cells + 1) / 2 + 6) * stride; }

// levels with fewer rows than this split their sweeps' rows over lanes by default
constexpr int kLaneRowsDefault = 32768;

struct ASlices {
    int nslices;
    const int* width;          // [nslices]
    const long long* start;    // [nslices+1]
    int* col;                  // [slots]
    double* val;               // [slots*9]
    float* val32;              // [slots*9] (mixed precision copy) or null
};

// The particle matrix in factored form (a scalar or a vector per neighbour-list
// entry instead of nine values per block; derivation in mph_factored.hip).  The
// values sit beside the neighbour lists, in their order: alpha[nPtr[i] + jn] for the
// fluid neighbours jn < nFluid[i] of fluid i, beta[nPtrP[k] + jn] for the P
// neighbours of every k.
struct FacOp {
    const int* nFluid;        // [np] fluid neighbours (they lead each list)
    const long long* nPtr;    // neighbour lists
    const int* nInd;
    const void* alpha;        // viscous scalar (double, or float in FP32 form)
    const double* diag;       // [nf][9] viscous self block + inertia
    const double* selfC;      // [nf][3] C_ii
    const int* nCountP;       // [np] P entries
    const int* runP;          // [np] P entries up to and including the last fluid one
    const long long* nPtrP;   // P lists
    const int* nIndP;
    const double* beta;       // -w_p'(d)/d per P entry
    const double* lambda;     // [np]
    const double* pos;        // [np][3]
    // [7 np] the operand x (fluid), the position and t = lambda_k C_k^T x of every
    // particle in four planes: [np] pairs x0 x1, [np] pairs x2 p0, [np] pairs p1 p2,
    // then [np] t (body::fac_planes).  The second pass gathers a neighbour's
    // operands with three 16-byte loads, and the eight lanes of a row, which walk
    // consecutive particles of the cell-ordered list, read consecutive 16-byte
    // pairs.  Positions are written with the P slices; x and t by every first pass.
    double* rec;
    // flags set by the matrix-A launch.  [0]: some neighbour pair interacts through the
    // periodic boundary (the displacements then take the minimum image).  [1]: some
    // fluid pair's viscosity is not DevParams::mu0 (the second pass then reads alpha
    // instead of recomputing it from the distance)
    const int* wrap;
    // FP32 form (the inner solves of mixed precision), which needs no positions:
    // u = sqrt(alpha) r per fluid-neighbour entry and v = beta r per P entry, each a
    // 16-byte entry beside the lists -- three floats and the column's bits in the
    // fourth (u32[4*(nPtr[i]+jn)+c], v32[4*(nPtrP[k]+jn)+c]; body::fac_entry32), so an
    // entry is one load -- and a 16-byte record x0 x1 x2 t per particle
    const float* u32;
    const float* v32;
    float* rec32;
    // cell-staged FP64 second pass (null slot: the chunk kernel): one workgroup per cell
    // of the fluid bounding box cellLo + [0, cellCnt), which stages the records of the
    // row cell's visited cells in LDS for the gathers
    const int* cellStart;
    int cellLo[3], cellCnt[3];
    int cellXcd;  // 1: each XCD takes a contiguous range of cells (else round robin)
    int cellShape;  // kFacCell*: the launch shape
    // built by launch_fac_slots.  cellDesc [cells][kFacDesc]: what a workgroup needs of
    // its cell.  slot [nf][slotRow]: per fluid row its fluid neighbours' places among
    // the staged records, in blocks of 8 G entries (G = kFacLanes lanes walk a row)
    // of which lane g reads the 8 consecutive places that stand for entries g, g + G,
    // ..., g + 7 G; padded with the row's own place
    int* cellDesc;
    unsigned short* slot;
    int slotRow;
};
constexpr int kFacDesc = 160;
// lanes per row of the FP64 second pass.  A 3D row has about 170 fluid neighbours, a 2D
// row about 37; a 3D cell about 41 rows, one pass of 512 threads.  (16 lanes in 3D, two
// passes: 444 against 428 us per second pass on the 1M scene.)
constexpr int kFacLanes = 8;
// rows of a 256-thread workgroup, one per group of lanes, of the FP64 first pass and of
// the second (FP32: both).  (Workgroups of 256 rows, each group of lanes walking four or
// eight in series, left most wavefront slots empty in scenes of less than about a million
// particles: first pass 9.6 us at 2.9k particles, 18.4 at 182k, 132 at 1.3M, now 4.7, 11.8
// and 126; FP32 second pass 62.9 us at 64k fluid particles, now 39 at 5 TB/s of entries.)
constexpr int kFacRowsT = 64, kFacRowsY = 32;
// launch shapes of the cell-staged pass: threads per workgroup and staged records (56
// bytes of LDS each).  The particles that a lattice has in the visited cells decide (fac_op).
// 3D: 1456 records (81,536 bytes) are the most that let two workgroups share a CU: 27 cells
// of 3.51 spacings hold at most 11^3 = 1331 lattice particles, with one axis of up to 4
// spacings 12 11 11 = 1452.  Domains of few cells have wider ones and take 2816, one
// workgroup per CU.  (With 1408 a film of 150 x 150 x 3, whose cells are 3.86 spacings deep,
// took the large shape: 78 us per product, now 63; a 34 x 38 x 42 pool 73, now 59.)  2D: a
// cell holds about 12 rows and its 9 visited cells 110-144 records,
// so 128 threads and 256 records keep many workgroups on a CU.  2D radii of more than 5
// spacings have larger cells and take the 3D shapes: with 256 records their rows would be
// gathered (us per product at radius 6, 8 and 12 spacings, 12k, 10k and 3.6k particles: 39,
// 57 and 146 gathered, 29, 31 and 52 staged; 75 and 59 at radius 6 and 90k).
enum { kFacCell3D = 0, kFacCell3DWide = 1, kFacCell2D = 2, kFacCellShapes = 3 };
constexpr int kFacCellThreads[kFacCellShapes] = {512, 512, 128};
// a launch of 2^32 threads or more runs only the remainder, without an error
constexpr long long kFacCellsMost = (1LL << 32) / 512 - 1;
constexpr int kFacCellSlots[kFacCellShapes] = {1456, 2816, 256};

constexpr int kSlice = 64;    // particles per A slice (one wavefront)

// block k of particle lane `lane` of the slice whose first slot is sb (even)
__host__ __device__ inline long long a_col_index(long long sb, int k, int lane) {
    return ((sb / 2 + k / 2) * 64 + lane) * 2 + (k & 1);
}
__host__ __device__ inline long long a_val_index(long long sb, int k, int e, int lane) {
    return (((sb / 2 + k / 2) * 9 + e) * 64 + lane) * 2 + (k & 1);
}
// the FP32 copy of A (mixed precision) groups blocks 4q..4q+3 per entry instead, so
// its loads are 16 bytes per lane as well
__host__ __device__ inline long long a_val32_index(long long sb, int k, int e, int lane) {
    return (((sb / 4 + k / 4) * 9 + e) * 64 + lane) * 4 + (k & 3);
}
// scenes of up to this many chunks fold rho and tmp where they are read (body::dot_fold)
constexpr int kFoldChunks = 1024;
constexpr int kChunk = 256;   // particles per dot-product chunk / CR workgroup
constexpr int kRuns = 28;     // run starts per fluid particle: 27 neighbour cells + end
// the factored form's level-0 run sums: per fluid particle and visited cell, the sums
// of -alpha r r^T over that cell's run of fluid entries, a symmetric block kept as its
// upper triangle (xx xy xz yy yz zz) in records of kBlkStride doubles
constexpr int kBlkRuns = kRuns - 1, kBlkStride = 6;
constexpr int kMaxLevels = 20;   // multigrid depth = floor(log2(cells per axis)) + 1

// ---- cells (calculateCellParticle) ----
void launch_hash(hipStream_t st, const DevParams& P, const double* pos, const int* type, uint64_t* keys);
void launch_bitonic(hipStream_t st, const DevParams& P, uint64_t* keys);
void launch_cell_start(hipStream_t st, const DevParams& P, const uint64_t* keys, int* cellStart);
void launch_reorder(hipStream_t st, const DevParams& P, const uint64_t* keys, const int* type, const int* perm,
                    const double* pos, const double* vel, int* type2, int* perm2, double* pos2, double* vel2,
                    int* cellIndex);
// ---- neighbours (calculateNeighbor) ----
// maxFluidP[4]: largest P count and fluid count of a fluid particle, largest count and
// P count of any particle.  With scrM set, the lists also go into per-particle
// scratch (capM / capP entries) and runStart is written; *overflow is raised if a
// list does not fit (then launch_neighbor_fill builds the lists instead).
void launch_neighbor_count(hipStream_t st, const DevParams& P, const double* pos, const int* cellIndex,
                           const int* cellStart, int* nCount, int* nFluid, int* nCountP, int* maxFluidP, int* scrM,
                           int capM, int* scrP, int capP, unsigned short* runStart, int* overflow);
// the lists from the count pass's scratch
void launch_neighbor_compact(hipStream_t st, const DevParams& P, const int* nCount, const int* nCountP,
                             const long long* nPtr, const long long* nPtrP, const int* scrM, int capM,
                             const int* scrP, int capP, int* nInd, int* nIndP);
void launch_scan_i64(hipStream_t st, const int* in, long long* out, int n, long long* scratch, int scratch_len);
int scan_scratch_len(int n);
void launch_neighbor_fill(hipStream_t st, const DevParams& P, const double* pos, const int* cellIndex,
                          const int* cellStart, const long long* nPtr, const long long* nPtrP, int* nInd, int* nIndP,
                          unsigned short* runStart);
void launch_slice_width(hipStream_t st, int nf, int nslices, const int* nFluid, int* width);
// ---- kinematics and explicit forces ----
void launch_kinematics(hipStream_t st, const DevParams& P, const WallKin& wk, const int* type, double* pos,
                       double* vel, double* force);
void launch_densities(hipStream_t st, const DevParams& P, const int* type, const double* pos, const int* nCount,
                      const long long* nPtr, const int* nInd, double* densA, double* gcen, double* volStrainP);
void launch_coefficients(hipStream_t st, const DevParams& P, const int* type, const double* densA,
                         const double* volStrainP, double* mass, double* kappa, double* lambda, double* mu,
                         double* pressA);
void launch_forces(hipStream_t st, const DevParams& P, const int* type, const double* pos, const int* nCount,
                   const long long* nPtr, const int* nInd, const double* pressA, const double* gcen,
                   const double* mass, double* force, double* vel);
// ---- implicit assembly ----
// alpha/diag/wrap (each may be null): the factored form's viscous scalar per
// fluid-neighbour entry (FacOp order), the diagonal block without C Lambda C^T, and
// the two flags of FacOp::wrap (0 before the launch).  blk (with runStart; may be null): the level-0 run sums
// [nf][kBlkRuns][kBlkStride] of the factored form, each in list order
void launch_matrix_a(hipStream_t st, const DevParams& P, const int* type, const double* pos, const double* vel,
                     const double* mass, const double* mu, const int* nCount, const int* nFluid,
                     const long long* nPtr, const int* nInd, ASlices A, int* selfIdx, double* b,
                     double* alpha = nullptr, double* diag = nullptr, int* wrap = nullptr,
                     const unsigned short* runStart = nullptr, double* blk = nullptr);
void launch_matrix_c(hipStream_t st, const DevParams& P, const double* pos, const int* nCountP,
                     const long long* nPtrP, const int* nIndP, const double* lambda, double* cval, double* dval);
void launch_vector_p(hipStream_t st, const DevParams& P, const int* type, const double* pos, const double* vel,
                     const double* kappa, const double* lambda, const double* volStrainP, const int* nCountP,
                     const long long* nPtrP, const int* nIndP, double* vecP);
void launch_b_minus_cp(hipStream_t st, const DevParams& P, const int* nCountP, const long long* nPtrP,
                       const int* nIndP, const double* cval, const double* vecP, double* b);
// maxP: the largest P-neighbour count of a fluid particle; above 64 the lists are merged
// instead of hashed (the same bits).  Also writes A.val32 when it is non-null
// (nIndP is read up to kListSpare entries past its lists)
constexpr int kListSpare = 3;
void launch_cac(hipStream_t st, const DevParams& P, const int* nFluid, const int* nCountP, const long long* nPtrP,
                const int* nIndP, const double* cval, const double* dval, ASlices A, int maxP);
// ---- multigrid ----
void launch_fluid_bbox(hipStream_t st, const DevParams& P, const int* cellStart, int* bbox);
void launch_inv_diag(hipStream_t st, const DevParams& P, const int* selfIdx, ASlices A, double* invDiagA);
// variant 0: per-thread sums straight from A; 1: the rows of four adjacent
// particles staged in LDS per round (rows of at most 216 blocks).  Same bits.
constexpr int kGalVariants = 2, kGalRowMax = 216;
void launch_mg_galerkin0(hipStream_t st, const DevParams& P, const Level& L, const int* cellStart,
                         const unsigned short* runStart, const int* nFluid, ASlices A, int variant);
void launch_mg_galerkinL(hipStream_t st, const Level& S, const Level& L);
void launch_mg_invd(hipStream_t st, const Level& L);
void launch_fill(hipStream_t st, double* x, long long n, double v);
void launch_fill_i32(hipStream_t st, int* x, long long n, int v);  // a kernel, not a memset node
void launch_mg_p2g_bu(hipStream_t st, const DevParams& P, Level& L, const int* cellStart, const double* q);
// the same after q = beta q + y (beta = rho / rho_prev from scal), written back to q
void launch_mg_p2g_bu_pq(hipStream_t st, const DevParams& P, Level& L, const int* cellStart, double* q,
                         const double* y, double* scal, const double* rho);  // rho: its partials, folded here, or null
void launch_mg_restrict_bu(hipStream_t st, const Level& S, Level& L);  // restriction, begin, update
void launch_mg_residual(hipStream_t st, Level& L);     // R = Q - A S
void launch_mg_residual_update(hipStream_t st, Level& L);  // R = Q - A S; S += invD R
void launch_mg_prolong(hipStream_t st, const Level& L, Level& S);
// levels lc..D-1 of the V-cycle in one workgroup, from their packed rows.  S is level
// lc-1 (its R is restricted, its current S takes the prolongation), or level 0 itself
// when lc = 0 (Q0 in, S0 out, three sweeps).  f32: pack the FP32 stencils where a level
// has one.  lvs: device copy of the levels.
void launch_mg_coarse_pack(hipStream_t st, const Level* lvs, int lc, int D, bool f32, const CoarsePack& K);
// S: level lc-1 (0 when lc = 0), F: level lc.  Where S takes the lane-split sweeps, S of F is
// written and the prolongation left to launch_mg_prolong_update
void launch_mg_coarse(hipStream_t st, const DevParams& P, const CoarsePack& K, int lc, int D, const Level& S,
                      const Level& F);
// residual of S, restriction into L, begin, update
void launch_mg_residual_restrict(hipStream_t st, Level& S, Level& L);
// prolongation U -> L (unless launch_mg_coarse has done it: prolonged), then a residual-update sweep of L
void launch_mg_prolong_update(hipStream_t st, const Level& U, Level& L, bool prolonged);
void launch_mg_g2p(hipStream_t st, const DevParams& P, const Level& L0, const int* cellIndex,
                   const double* invDiagA, const double* q, double* u, double* part);
// ---- conjugate residual ----
void launch_cr_init(hipStream_t st, const DevParams& P, const double* vel, const double* force,
                    const double* mass, double* x);
// SpMV variants differ only in how many block pairs are loaded per group (same
// bits): FP64 2, 3 or 4 block pairs; FP32 1 or 2 block quads
constexpr int kSpmvVariants64 = 3, kSpmvVariants32 = 2;
// up to this many slices of 64 rows a wavefront takes one component of a slice's rows
// (spmv_split in mph_cr_body.h), beyond it all three: the split reads x and the columns
// three times and reaches 4.2 TB/s, the other 6.3 TB/s once enough wavefronts are there.
// Split against whole, us per FP64 product with the 4.5 us of the dot partials that the
// split launches on their own: 2D 65 slices 13.3/19.1, 223: 15.7/20.3, 438: 21.9/22.3;
// 3D 144 slices 36.5/89.1, 216: 39.3/91.4, 436: 94.8/98.0, 631: 161/107, 1000: 196/129
constexpr int kSpmvSplit = 400;
void launch_spmv(hipStream_t st, const DevParams& P, ASlices A, const int* nFluid, double alpha, const double* x,
                 double beta, const double* yin, double* y, double* y2, double* p_copy, const double* dotx,
                 double* part, bool f32 = false, int variant = 0);
// factored form: beta, runP, C_ii and the records' positions (after matrix A has
// written alpha and the diagonal blocks), and y = beta*yin +- A x with the same
// outputs as launch_spmv (two launches: t over every particle, then the fluid rows)
void launch_fac_p(hipStream_t st, const DevParams& P, const double* pos, const int* nCountP, const long long* nPtrP,
                  const int* nIndP, double* beta, float* v32, int* runP, double* selfC, double* rec);
// multigrid level 0 (calculateMultiGridCsrA at level 0) and InvDiagA from the
// factored form, with per-particle scratch gtab [np][27][3] and gmask [np] (level-0
// counts of at least 3 per active axis: the caller checks)
// blk: the run sums launch_matrix_a wrote
void launch_fac_level0(hipStream_t st, const DevParams& P, const Level& L0, const FacOp& F, const int* cellIndex,
                       const int* cellStart, const double* blk, double* gtab, int* gmask, double* invDiagA);
// u32 of the FP32 form from alpha and the positions (after launch_fac_p)
void launch_fac_u(hipStream_t st, const DevParams& P, const int* nFluid, const long long* nPtr, const int* nInd,
                  const double* alpha, const double* pos, float* u32);
// passes: 1 the first pass (t from x) only, 2 the second only (t already in F.rec),
// 3 both
void launch_fac_spmv(hipStream_t st, const DevParams& P, const FacOp& F, double alpha, const double* x, double beta,
                     const double* yin, double* y, double* y2, double* p_copy, const double* dotx, double* part,
                     bool f32, int passes = 3);
// the positions of the FP64 records (planes b odd and c of FacOp::rec, 7*np doubles)
// copied from one record buffer into another; x and t are written by each product
void launch_fac_rec_positions(hipStream_t st, const DevParams& P, const double* from, double* to);
// FacOp::cellDesc and slot (after the lists and runP; the cell-staged pass)
void launch_fac_slots(hipStream_t st, const DevParams& P, const FacOp& F);

void launch_convert_f32(hipStream_t st, const double* in, float* out, long long n);
void launch_axpy(hipStream_t st, long long n, const double* x, double* y);  // y += 1.0*x
void launch_dot_partial(hipStream_t st, const DevParams& P, const double* x, const double* y, double* part);
// host: optional coherent pinned host memory that also receives the value
void launch_dot_final(hipStream_t st, const DevParams& P, const double* part, double* scal, int slot, int shift_slot,
                      double* host = nullptr, bool shiftRho = false);
// The CR loop's control block int[kNCtl] in device memory: the stop flag the
// iteration kernels test (DevParams::halt points at ctl[kCtlHalt]), the iterations
// done and a non-finite flag.
enum { kCtlHalt = 0, kCtlIter = 1, kCtlBad = 2, kNCtl = 4 };
// the r.r reduction of the CR loop (scal[2]) followed by the loop's stop test
// (main.cpp:4344-4346) on the device: ctl[kCtlIter] += step; then the loop stops
// (ctl[kCtlHalt] = 1) once ctl[kCtlIter] >= maxit, or on a residual that is not
// finite (also ctl[kCtlBad] = 1), or when rr/rr0 < tol, tested in that order.  A
// no-op once halted.  hctl and hrr: optional coherent pinned host memory that also
// receives ctl[0..2] and rr.
void launch_dot_final_stop(hipStream_t st, const DevParams& P, const double* part, double* scal, int* ctl, int step,
                           double tol, long long maxit, int* hctl, double* hrr, bool shiftRho);
// The convergence record of a CR iteration (main.cpp:4348-4351): the partials' sum
// r.s into scal[kRSIter], then rec[2 it] = rr (scal[kRR]) and rec[2 it + 1] = r.s
// for it = ctl[kCtlIter] (ctl null: the host's `it`), rows it >= cap skipped.  A
// no-op once halted.
void launch_dot_final_record(hipStream_t st, const DevParams& P, const double* part, double* scal, const int* ctl,
                             long long it, double* rec, long long cap);
void launch_pq_update(hipStream_t st, const DevParams& P, const double* scal, const double* s, const double* y,
                      double* p, double* q);
// pq: p = beta p + s first, written back
void launch_xrs_update(hipStream_t st, const DevParams& P, const double* scal, double* p, const double* q,
                       const double* u, double* x, double* r, double* s, double* part, bool pq = false,
                       const double* tmp = nullptr);  // tmp: its partials, folded here (pq only)
void launch_store_velocity(hipStream_t st, const DevParams& P, const double* x, double* vel);
// ---- output-step diagnostics ----
void launch_diagnostics(hipStream_t st, const DevParams& P, const int* type, const double* pos, const double* vel,
                        const double* mu, const double* lambda, const double* kappa, const double* volStrainP,
                        const double* pressA, const double* gcen, const int* nCount, const long long* nPtr,
                        const int* nInd, const int* nCountP, const long long* nPtrP, const int* nIndP, double* divP,
                        double* pressP, double* force, double* virialStress, double* virialP);

}  // namespace mph
