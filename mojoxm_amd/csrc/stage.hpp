// stage.hpp -- the fused DG stage kernel for gfx950 and its launcher.
//
// One launch computes, for every element, the weak-form right-hand side
//   rhs_i = sum_k sum_j D_k[i][j] (invJ F(q_j))_k
//           - inv_vol * sum_f sum_r Lift_f[i][r] s_f area_f F*_{f,r}
//           + S(q_i)
// and the Shu-Osher combine q_out = a q_a + b q_b + c dt rhs followed by the
// physics' positivity fix -- rk_stage_kernel, src/solver.mojo:161-337, and
// (for 2D) the face-flux + vol_lift_combine_rk kernel pair of
// src/local_mesh_2d_gpu_<phys>.mojo fused into one pass.
//
// One block (4 wave64, or 5 for the wide 2D P = 3 tile of the FP32-MFMA
// form, below) per tile of at most EPB elements, which are contiguous in
// device memory:
//   1. each thread starts the loads of its first face item (job record,
//      partner node, and the partner's trace when the partner lies outside
//      the tile); the block stages the q_in tile and the mesh's distinct
//      face and cell geometries in LDS;
//   2. per face item: the numerical flux (boundary faces: against the
//      physics' ghost state), signed and scaled by the face area, into LDS.
//      A face whose two elements are both in the tile is evaluated once by
//      its side-0 element, which also stores the negated value in the
//      partner's slot; faces to elements outside the tile are evaluated by
//      each side, as the reference evaluates every face from both sides;
//      side 0 is always the left state.  Per (element, node): the nodal
//      flux mapped to reference directions by invJ, into LDS;
//   3. the D and Lift contractions over LDS, the operator entries from the
//      scalar cache (FP64) or straight to the MFMA's lanes (FP32), then per
//      (element, node) the RK combine, limit_state and the store.
//
// Two arithmetic forms share the kernel:
//   R = double  plain FP64: the contractions run on the VALU in FP64;
//   R = float   FP32-MFMA: FP32 state, fluxes and traces; the volume and
//               LIFT contractions are one [D | Lift] x [F ; S] product per
//               tile on V_MFMA_F32_16X16X4F32 with FP32 accumulation, the
//               surface fluxes pre-scaled by -inv_vol s area; geometry is
//               formed in FP64 and rounded once to FP32, and the RK combine
//               and the positivity rescue are FP64; the stored state is
//               rounded stochastically.
// Blocks are mapped to tiles so that each of the 8 XCDs walks a contiguous
// range of tiles: face neighbours then mostly hit the XCD's own L2.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "bj.hpp"
#include "host.hpp"
#include "physics.hpp"

namespace mxm {

// Shu-Osher stage q_out = a q_a + b q_in + c dt L(q_in): in every SSPRK3
// stage of src/ssprk3.mojo:41-78 the b-term buffer is the stage input.
template <class R>
struct StageArgs {
  const R *q_in, *q_a;
  R *q_out;
  double a, b, c;         // stage coefficients; c dt multiplies the rhs
  // Instances: a tile belongs to one instance, whose physics parameters
  // (MXM_PRM_MAX doubles), time step and GLM decay the block reads.  One
  // solver is a single instance (tile_inst == nullptr: instance 0 with dt
  // and post_scale below); a batch sets the per-instance tables, and an
  // instance whose inst_active entry is 0 is skipped.
  const int *tile_inst;     // [ntiles] or nullptr
  const double *inst_prm;   // [n_inst][MXM_PRM_MAX]
  const double *inst_dt;    // [n_inst] or nullptr -> dt
  const double *inst_post;  // [n_inst] or nullptr -> post_scale
  const int *inst_active;   // [n_inst] or nullptr (all active)
  int *inst_fail;           // [n_inst] or nullptr: set to 1 when a stored value is not finite
  double *mean;             // [slots][NC] or nullptr: cell means sum_i w_i q_out_i of the stored state
  R *ext;                   // [slots][NCL][2] (with mean): smallest and largest stored node value of the
                            // limited components (all NC in 3D, component 0 in 2D)
  const double *w;          // [NP] node weights (with mean)
  // Limiter (mean != nullptr).  The factors pending on q_in are computed
  // from its means and node extrema as it is read (NaN extrema: nothing
  // pending); stage 1 stores those of its input, which is q_a of the others.  A value
  // read from q_in (tile and partner traces) or q_a is used as
  // mean + theta (q - mean) where its element's theta < 1, which is the state
  // the limiter would have stored.
  const double *lim_mn_in;               // q_in: means [slots][NC]
  const R *lim_ext_in;                   // q_in: extrema [slots][NCL][2]
  double *lim_th_in;                     // q_in: theta [slots], written for the tile's elements, or nullptr
  const double *lim_th_a, *lim_mn_a;     // q_a: theta, means
  const int *conn;                       // [slots][NF] partner slot of each face
  double lim_eps2;                       // Venkatakrishnan's eps^2
  double dt, post_scale;
  int post_comp;            // component scaled after the combine (GLM psi: Phys::kPost), -1 none
  const int *tile_count;  // [ntiles] elements in each tile (slots T*EPB ..)
  const R *geom;          // [n_inst][stage_geom_len]: the mesh's distinct face normals and areas
                          // ([max_face_geo][4]), then per element of a lattice cell invJ (ND*ND, rows =
                          // reference directions) and inv_vol (1/(6V) or 1/(2A)), in the FP32 form
                          // -inv_vol times each of those areas
  const int *tile_type;   // [ntiles] cell element of the tile's first slot
  const double *Dt;       // FP64 form: [ND*NP (k,j)][NPAD (i)] transposed D_ref, zero padded
  const double *Lt;       // FP64 form: [NF*NFP (f,r)][NPAD (i)] transposed Lift_ref, zero padded
  const float *Aop;       // FP32 form: [D_0 .. D_ND-1 | Lift], zero padded, in the order the MFMA operand reads it:
                          // [KPAD/4][MT][lane 16 g + r] = row 16 m + r, column 4 k + g
  const int *fmap;        // [NF][NFP] element node of each reference face slot
  const int2 *jobs;       // [ntiles*maxj] {el | lf<<7 | pin<<9 | plf<<16 | side<<18 | bc<<19 | geometry<<22
                          //  (-1: padding), partner slot}
  const unsigned short *ipr;  // [ntiles*maxj*NFP] partner node | partner slot << 8
  int maxj;               // job slots per tile
  int ntiles;
};

constexpr int kPrmMax = 32;  // MXM_PRM_MAX
// FP64 operators up to this size are read into the scalar cache (16 KB for
// two CUs) by the first blocks of a launch, one or so per CU
constexpr int kScalarWarmBytes = 4096, kScalarWarmBlocks = 256;
// read-only data in the constant address space: wave-uniform loads stay scalar
// whatever stands between them
typedef const double __attribute__((address_space(4))) *ScalarPtr;

// Launch configurations of the stage kernel: each is an occupancy target
// (waves per SIMD, e.g. 256-thread blocks per CU) that bounds the register
// allocation; all configurations compute the same bits.  The autotuner
// times them on the problem and keeps the fastest.  The FP64 kernels fit 5
// waves (<= 102 VGPRs; the 2D HLLEC Euler kernel's 80 let 6 run) or 4
// (<= 128: GLM-MHD); the FP32 kernels fit 5, 6 or 7 (<= 72 VGPRs), and the
// compiler's own choice (1: no bound) can be far off (e.g. 250 VGPRs, 1
// wave, for the 2D Euler kernels at P = 1).
template <class R>
struct StageCfg;
template <>
struct StageCfg<double> {
  static constexpr int count = 3, dflt = 0;
  static constexpr int waves[3] = {1, 5, 4};
};
template <>
struct StageCfg<float> {
  static constexpr int count = 4, dflt = 1;
  static constexpr int waves[4] = {1, 5, 6, 7};
};
constexpr int kStageCfgMax = 4;

// Elements per tile (one thread per element node): at most 256/NP for NP
// nodes per element, rounded down to whole lattice cells (2 triangles, 6
// tets) when a cell fits, then reduced -- by cells, then to runs of
// elements -- until the block's LDS at FP64 (the operand array -- the q_in
// tile and the face fluxes, later the ND*NP flux planes, rows of
// EPB*NC + 1 values -- and 8 bytes for each invJ entry and volume of the
// elements, an allowance for the geometry table and the limiter's arrays,
// which are of about that size; the kernel asserts its own sum) fits 64 KB,
// which only the two-fluid state (NC = 17) and, at P = 1, MHD (NC = 9) need.  Tiles are blocks of cells, so the LDS
// is sized for what a tile can hold; the host builds the tiles with the
// same value.
//
// The wide tile (wide = true; the FP32-MFMA form only, where the solver's
// autotuner times both tile sizes and keeps the faster): when 256 threads
// leave more than 5 % of the lanes without a node and whole cells fill a
// block of 5 to 8 waves exactly -- of the shapes built, 2D P = 3 (NP = 10:
// 24 triangles on 240 of 256 lanes, or 32 on all 320 lanes of 5 waves).
// It pays when all tiles are resident at once: a mesh of 128 x 128
// squares makes 1,024 wide tiles, 4 per CU and 5 waves per SIMD, against
// 1,370 narrow ones, 5 or 6 per CU and 6 waves on the busiest SIMDs.
// When tiles queue for the CUs the narrow tile is faster (an 8-wave tile
// of 50 triangles measured slower still): a CU then holds fewer, larger
// blocks, whose barriers idle more waves at once and whose phases overlap
// less.  The FP64 contraction layout (stage_groups) is sized for 4 waves
// and has no wide tile.
constexpr int stage_lds_bytes(int ND, int NP, int NFP, int NC, int epb) {
  return (epb * NP * NC + (ND + 1) * NFP * (epb * NC + 1) > ND * NP * (epb * NC + 1)
              ? epb * NP * NC + (ND + 1) * NFP * (epb * NC + 1)
              : ND * NP * (epb * NC + 1)) * 8 +
         epb * (ND * ND + 1) * 8 + (ND + 1) * NFP * 4;
}
constexpr int stage_epb(int ND, int NP, int NFP, int NC, bool wide = false) {
  const int cell = ND == 3 ? 6 : 2;
  int e = 256 / NP;
  if (e >= cell) e -= e % cell;
  if (wide && e >= cell && e * NP * 20 < 256 * 19)
    for (int w = 5; w <= 8; ++w) {
      const int t = 64 * w;
      if (t % NP == 0 && (t / NP) % cell == 0 && t / NP <= 126 &&
          stage_lds_bytes(ND, NP, NFP, NC, t / NP) <= 65536)
        return t / NP;
    }
  while (e > 1 && stage_lds_bytes(ND, NP, NFP, NC, e) > 65536) e = e > cell ? e - cell : e - 1;
  return e;
}
// Threads per block: 256, or the whole waves of a wide tile
constexpr int stage_block(int ND, int NP, int NFP, int NC, bool wide = false) {
  return stage_epb(ND, NP, NFP, NC, wide) * NP > 256 ? (stage_epb(ND, NP, NFP, NC, wide) * NP + 63) / 64 * 64 : 256;
}
// whether the shape has a wide tile distinct from the 256-thread one
constexpr bool stage_has_wide(int ND, int NP, int NFP, int NC) {
  return stage_epb(ND, NP, NFP, NC, true) != stage_epb(ND, NP, NFP, NC, false);
}

// FP64 contraction layout: the tile's (element, component) columns span
// ceil(EPB*NC/64) waves; the block's 4 waves form `groups` groups, each
// producing `IH` consecutive output nodes, so the operator entries a wave
// reads are wave-uniform.  The transposed operators are stored with
// groups*IH (>= NP) zero-padded node columns.
constexpr int stage_groups(int EPB, int NC) {
  return (EPB * NC + 63) / 64 >= 4 ? 1 : 4 / ((EPB * NC + 63) / 64);
}
constexpr int stage_node_pad(int EPB, int NP, int NC) {
  return stage_groups(EPB, NC) * ((NP + stage_groups(EPB, NC) - 1) / stage_groups(EPB, NC));
}

// FP32-MFMA operator shape: 16-row tiles of output nodes, K = ND*NP volume
// columns then NF*NFP lift columns, padded to the MFMA depth of 4.
constexpr int mfma_mtiles(int NP) { return (NP + 15) / 16; }
// FP32-MFMA operator columns: the ND*NP derivative columns padded to a
// multiple of 4, then the (ND+1)*NFP lift columns padded to a multiple of 4
constexpr int mfma_kvpad(int ND, int NP) { return (ND * NP + 3) / 4 * 4; }
constexpr int mfma_kpad(int ND, int NP, int NFP) { return mfma_kvpad(ND, NP) + ((ND + 1) * NFP + 3) / 4 * 4; }
constexpr int cmax(int a, int b) { return a > b ? a : b; }
// Length of the stage kernel's LDS operand array (in values): the q_in
// tile [0, TILE) with the face fluxes after it (NFF rows of NCOLS), and
// later the KV flux-plane rows from 0; the MFMA form also reads its
// padding rows and up to NTC columns of every row.
constexpr int stage_operand_len(bool mfma, int TILE, int NCOLS, int KV, int KVP, int NFF, int KPAD, int NTC) {
  return mfma ? cmax(cmax(TILE + NFF * NCOLS, KVP * NCOLS),
                     cmax(TILE + (KPAD - KVP - 1) * NCOLS + NTC, (KVP - 1) * NCOLS + NTC))
              : cmax(TILE + NFF * NCOLS, KV * NCOLS);
}

template <int ND, int P, int NC = 1, bool WIDE = false>
struct Shape {
  static constexpr int NP = ND == 3 ? (P + 1) * (P + 2) * (P + 3) / 6 : (P + 1) * (P + 2) / 2;
  static constexpr int NFP = ND == 3 ? (P + 1) * (P + 2) / 2 : P + 1;
  static constexpr int NF = ND + 1;
  static constexpr int BLOCK = stage_block(ND, NP, NFP, NC, WIDE);
  static constexpr int EPB = stage_epb(ND, NP, NFP, NC, WIDE);
  static constexpr bool kHasWide = stage_has_wide(ND, NP, NFP, NC);
};
// the stage kernel's shape for the state type R (the wide tile: FP32 only)
template <class Phys, int ND, int P, class R, bool WIDE>
using StageShape = Shape<ND, P, Phys::NC, WIDE && std::is_same<R, float>::value>;
template <class Phys, int ND, int P, class R, bool WIDE>
constexpr int kStageBlock = StageShape<Phys, ND, P, R, WIDE>::BLOCK;

// Bijective map from the hardware block index (dispatched round-robin over
// the 8 XCDs) to a tile index such that XCD x owns a contiguous tile range.
__device__ __forceinline__ int xcd_tile(int bid, int nb) {
  const int q = nb >> 3, r = nb & 7;
  const int x = bid & 7, loc = bid >> 3;
  return x < r ? x * (q + 1) + loc : r * (q + 1) + (x - r) * q + loc;
}

// One face item: slot r of a face job, with everything fetched from
// global memory before the flux is evaluated.  The records stay as they
// were loaded until the face phase: decoding or converting them where they
// are loaded would make the block wait for them before it issues the loads
// that follow.
template <class R, int NC>
struct FaceItem {
  int2 job;     // StageArgs::jobs
  unsigned pr;  // StageArgs::ipr
  R qp[NC];     // partner trace when the partner is outside the tile
};
// the partner's cell means (limited kernels)
template <int NC>
struct FaceMeans {
  double m[NC];
};

// A value of the state with its element's pending limiter factor applied:
// the expression of the limiter's own apply, so the bits are those the
// limiter would have stored.
template <class R>
__device__ __forceinline__ R lim_apply(R v, double th, double bm) {
  return th < 1.0 ? R(bm + th * (double(v) - bm)) : v;
}

// Quotient of x in [0, MAX) by a compile-time constant as a 24-bit multiply
// and a shift: the 32-bit multiplies of a general division run at a quarter
// of the rate.
constexpr bool small_div_exact(int d, int max) {
  for (int x = 0; x < max; ++x)
    if ((int)(((unsigned)x * ((65536u + d - 1) / d)) >> 16) != x / d) return false;
  return true;
}
template <int D, int MAX>
__device__ __forceinline__ int small_div(int x) {
  __builtin_assume(x >= 0 && x < MAX);
  if constexpr ((D & (D - 1)) == 0) {
    return (int)((unsigned)x / (unsigned)D);
  } else {
    static_assert(MAX <= 4096 && small_div_exact(D, MAX), "not exact over the range");
    return (int)(__umul24((unsigned)x, (65536u + D - 1) / D) >> 16);
  }
}

// Every record of face item t of a tile is addressed from the tile index,
// so all of them are in flight together (load_item_records); the partner
// trace of a face to another tile is the only load that waits for one of
// them (load_item_trace).
template <int NFP, int MAXT, class R, int NC>
__device__ __forceinline__ void load_item_records(const int2 *jobs, const unsigned short *ipr, int t,
                                                  FaceItem<R, NC> &it) {
  it.job = jobs[small_div<NFP, MAXT>(t)];
  it.pr = ipr[t];
}

// A partner slot in the tile's own range is in the tile: partners are real
// elements, which occupy the tile's first slots.  An item without a partner
// in another tile loads the tile's first node instead of branching around
// the loads: behind a branch, the waits for everything issued before would
// have to assume either path and wait for the traces too.
template <int NP, int EPB, bool LIM, class R, int NC>
__device__ __forceinline__ void load_item_trace(const StageArgs<R> &A, int e0, FaceItem<R, NC> &it,
                                                FaceMeans<LIM ? NC : 1> &fm) {
  const bool far = (unsigned)(it.job.y - e0) >= (unsigned)EPB;
  const size_t p = (size_t)(far ? it.job.y : e0);
  const R *g = A.q_in + (p * NP + (far ? it.pr & 255 : 0)) * NC;
#pragma unroll
  for (int c = 0; c < NC; ++c) it.qp[c] = g[c];
  if constexpr (LIM) {
#pragma unroll
    for (int c = 0; c < NC; ++c) fm.m[c] = A.lim_mn_in[p * NC + c];
  }
}

// Values per vector access of a tile: the widest of 16, 8 or 4 bytes that
// divides the tile, so that every tile starts aligned to it.
template <class R>
constexpr int tile_vec(int tile) {
  return sizeof(R) == 4 && tile % 4 == 0 ? 4 : tile % 2 == 0 ? 2 : 1;
}

typedef float mxm_float4 __attribute__((ext_vector_type(4)));

// FP64 -> FP32 with stochastic rounding, for the FP32-MFMA form's stored
// state.  Round-to-nearest storage loses every update smaller than half a
// float ulp and biases the rest, so over thousands of steps on a nearly
// steady background the state drifts from the FP64 solution; rounding up
// or down at random, with probabilities that make the expected stored
// value equal x, leaves only an unbiased random walk.  The 29 mantissa
// bits a float drops are cleared (the float of what is left is exact) and
// one float ulp is added away from zero when a 32-bit draw is below those
// bits scaled to 32 bits (lo << 3): probability (dropped bits) / 2^29.
// The draw is the bit reversal of x's low word xor `salt` (one value per
// node of an element), so its high bits are x's lowest, noisiest bits: a
// pure function of x and its node, so results do not depend on the launch
// configuration or on the other instances of a batch.  Infinities and the
// hardware's NaN have a zero low word and convert unchanged; any other NaN
// stays non-finite.
__device__ __forceinline__ float sr_f32(double x, unsigned salt) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(x);
  const unsigned lo = (unsigned)b;
  const float t = float(__longlong_as_double((long long)(b & ~0x1FFFFFFFull)));
  const unsigned up = __builtin_bitreverse32(lo ^ salt) < (lo << 3) ? 1u : 0u;
  return __uint_as_float(__float_as_uint(t) + up);
}

// W: occupancy target of the launch configuration, in waves per SIMD
// (amdgpu_waves_per_eu); 1 leaves the register budget to the compiler.
// WIDE: the wide tile (stage_epb).
template <class Phys, int ND, int P, class R, int W, bool LIM, bool WIDE>
__global__ __attribute__((amdgpu_flat_work_group_size(1, kStageBlock<Phys, ND, P, R, WIDE>),
                          amdgpu_waves_per_eu(W))) void
dg_stage_kernel(StageArgs<R> A) {
  using S = StageShape<Phys, ND, P, R, WIDE>;
  constexpr bool kMFMA = std::is_same<R, float>::value;
  static_assert(kMFMA || S::BLOCK == 256, "the FP64 contraction layout is sized for 4 waves");
  constexpr int NP = S::NP, NFP = S::NFP, NF = S::NF, EPB = S::EPB, NC = Phys::NC;
  constexpr int TILE = EPB * NP * NC;  // values of one element tile
  constexpr int NCOL = EPB * NC;       // (element, component) columns of a tile
  // Rows of (element, component) columns are NCOLS apart: one word of
  // padding, so that the node threads' row-strided writes of the flux
  // planes spread over the LDS banks.
  constexpr int NCOLS = NCOL + 1;
  // The contraction's right operands: NFF = NF*NFP face-flux rows, then
  // KV = ND*NP flux-plane rows in the same array (stage_operand_len).
  // FP32-MFMA: the products run over 4-deep steps of operator columns and
  // NT 16-column tiles; the array is long enough for every such read, and
  // the padding rows (face fluxes NFF..KPAD-KVP-1, planes KV..KVP-1) hold
  // zeros (their operator columns are zero; a column beyond NCOL only
  // feeds an output column that is never stored).
  constexpr int NFF = NF * NFP, KV = ND * NP;
  constexpr int KVP = kMFMA ? mfma_kvpad(ND, NP) : KV;
  constexpr int KPAD = kMFMA ? mfma_kpad(ND, NP, NFP) : KV + NFF;
  constexpr int MT = mfma_mtiles(NP);
  constexpr int NT = (NCOL + 15) / 16;
  // q_a is loaded by the node threads where they use it (2b), not with the
  // tile: held through the face phase, the register peak, it costs NC
  // registers (or as much LDS as the tile), and other blocks cover the wait.
  // The FP64 Euler kernel on triangles goes from 30.7 to 21 KB of LDS and
  // from 82 to 80 VGPRs, 5 to 6 waves per SIMD (us per stage: 128^2 vortex
  // 13.6 -> 13.1, 512^2 144 -> 138; 384^2 GLM-MHD FP64 110 -> 104, FP32 61.1
  // -> 59.6; limited 192^2 Sod FP64 32.5 -> 29.8).  The FP32 kernels of at
  // most 5 components fit 8 waves either way and keep the early load (512^2
  // vortex 81.5, late 83.3), and so do the FP64 ones of P = 5 tets, whose
  // blocks per CU the LDS bounds (small meshes, where nothing covers a wait:
  // 4 x 5 x 4 Euler 26.7, early 25.5).
  constexpr bool kQaLate = (kMFMA ? NC >= 6 : NP < 56) || LIM;
  constexpr int NB0 = stage_operand_len(kMFMA, TILE, NCOLS, KV, KVP, NFF, KPAD, NT * 16);
  // sW = sB: first the q_in tile as [el][j][c] (TILE contiguous values);
  // after the lift product the contravariant nodal fluxes as [k][j][el][c]
  // (row kj at kj*NCOLS); after the volume product the result as
  // [el][i][c].  sS = sB + TILE: face fluxes [f*NFP + r][el][c].
  __shared__ __align__(16) R sB[NB0];
  // the geometry (StageArgs::geom): face normals and areas, then invJ and
  // inv_vol of each element of a lattice cell.  A lattice has a handful of
  // each, so a tile reads 0.15 to 1.1 KB for them, the same for every tile,
  // where a record per face and per slot took 3 KB: 77 of the 251 MB that
  // the FP32 512^2 vortex stage fetched (90.6 -> 86.0 us; 32^3 Taylor-Green
  // FP64 186 -> 181, 16^3 P = 2 advection 7.9 -> 7.5).
  // The FP32 form's table is rounded to FP32 by the host, with the face scales
  // multiplied out, as it uses them: one read per face item where an FP64 product and
  // conversions stood (32^3 Taylor-Green 108.6 -> 107.0, 384^2 GLM-MHD 60.7
  // -> 59.8, 128^2 vortex 8.67 -> 8.57).
  constexpr int EPC = cell_elems(ND), GEL = stage_geom_elem(ND, kMFMA), GEOM = stage_geom_len(ND, kMFMA);
  static_assert(GEOM <= 256, "one geometry value per thread");
  __shared__ __align__(16) R sG[GEOM];
  const R *const sE = sG + 4 * max_face_geo(ND);
  __shared__ int sMap[NF * NFP];
  // limiter: the cell means of the tile's elements (q_in); the factors of
  // the tile's elements, then of the elements behind its face jobs
  constexpr int NL = EPB * NC;
  __shared__ double sLim[LIM ? NL : 1];
  __shared__ double sTh[LIM ? EPB * (1 + NF) : 1];
  // Where these slots alone do not fill the block and several components
  // are limited, a thread takes one component of a slot at a time and the
  // slot's factor is their minimum, formed in LDS (bit patterns of numbers
  // that are not negative compare as integers); until the face fluxes, their
  // rows hold each slot's element (-1: none) and neighbours.  A thread to a
  // slot leaves the block waiting for the components one after another: us
  // per limited stage, FP64, factors in a launch of their own / a thread to a
  // slot / to a component: two-fluid 22^3 P = 2 345 / 442 / 307, 18^3 P = 3
  // 432 / 501 / 319, 28^3 P = 1 391 / 495 / 331, MHD 18^3 P = 3 125 / 128 /
  // 109, Euler 18^3 P = 3 66 / 58.4 / 53.5.  P = 1 with up to 6 components
  // has more slots than threads (28^3 Euler 66 / 57.6 / 59.2).
  constexpr bool kThetaComp = LIM && ND == 3 && NC > 1 && EPB * (1 + NF) <= S::BLOCK;
  static_assert(!kThetaComp || EPB * (1 + NF) * (1 + NF) * sizeof(int) <= NFF * NCOLS * sizeof(R), "slots' neighbours");
  static_assert(sizeof(sB) + sizeof(sG) + sizeof(sMap) + sizeof(sLim) + sizeof(sTh) <= 65536, "LDS of a block");
  R *const sW = sB;
  R *const sS = sB + TILE;
  [[maybe_unused]] int *const sNb = reinterpret_cast<int *>(sS);  // [slot][1 + NF] (kThetaComp)

  const int tid = threadIdx.x;
  const int tile = xcd_tile(blockIdx.x, A.ntiles);
  const int e0 = tile * EPB;
  const int nitems = A.maxj * NFP;  // padding items have job.x < 0

  // ---- 1. loads --------------------------------------------------------
  // First everything addressed from the tile index: the first face item's
  // records (the partner trace waits for them, so they lead the queue), the
  // q_in tile, q_a, the geometry, the operator; then the partner trace, and
  // the scalars of the tile's instance.  Nothing between the issues waits:
  // values are used, converted or written to LDS only once all are in
  // flight.  Every tile owns EPB element slots in every per-slot array
  // (padding slots hold zeros), so the loads cover the whole tile and need
  // not wait for its element count, and the lanes past the end of a piece
  // load its last entry again instead of branching.  With the records
  // decoded where they were loaded, q_a and the trace left only after the
  // first round trip.  Together with the 16-byte tile accesses and the face
  // states read by LDS offset (2a), in us per stage: 2D P = 3 vortex 128^2
  // FP64 15.9 -> 14.4, FP32 9.95 -> 9.6; 512^2 FP64 163 -> 152, FP32 97.8 ->
  // 90.6; 384^2 GLM-MHD FP64 130 -> 114, FP32 71 -> 64.6; 16^2 5.4 -> 4.7.
  constexpr int VW = tile_vec<R>(TILE);                   // values per vector access
  typedef R TileVec __attribute__((ext_vector_type(VW)));
  constexpr int TV = TILE / VW;
  constexpr int QPT = (TV + S::BLOCK - 1) / S::BLOCK;     // tile vectors per thread
  constexpr int MAXT = EPB * NFF;                         // face items of a tile, at most
  const size_t tile0 = (size_t)tile * TILE;               // the tile's first value
  const size_t job0 = (size_t)tile * A.maxj;
  const int2 *const jobs = A.jobs + job0;
  const unsigned short *const ipr = A.ipr + NFP * job0;
  FaceItem<R, NC> it;
  [[maybe_unused]] FaceMeans<LIM ? NC : 1> itm;
  load_item_records<NFP, MAXT>(jobs, ipr, tid < nitems ? tid : nitems - 1, it);
  // Tets have more face items than threads.  With one component the second
  // item of a thread starts here too, and its trace waits in its face-flux
  // slot: two round trips less in a block's chain (16^3 P = 2 advection FP64
  // 6.68 -> 6.44 us, FP32 5.6 -> 5.45; 24^3 P = 3 FP64 42.5 -> 41.2).  With
  // more components it costs registers where the tile is loaded: Euler and
  // MHD gained up to 3 % on some meshes and lost as much on others.
  constexpr bool kTwo = ND == 3 && NC == 1 && !LIM && MAXT > S::BLOCK;
  const int t2 = tid + S::BLOCK;
  [[maybe_unused]] FaceItem<R, NC> it2;
  if constexpr (kTwo) load_item_records<NFP, MAXT>(jobs, ipr, t2 < nitems ? t2 : nitems - 1, it2);
  // limiter: slot i of the factors, and thread i's part of their loads, is
  // element i of the tile, then the partner of face job i - EPB if that lies
  // in another tile
  const int thj = tid - EPB;
  int2 thjob = int2{-1, 0};
  if constexpr (LIM) thjob = jobs[thj < 0 ? 0 : thj < A.maxj ? thj : A.maxj - 1];
  const TileVec *const src = reinterpret_cast<const TileVec *>(A.q_in + tile0);
  TileVec tq[QPT];
#pragma unroll
  for (int k = 0; k < QPT; ++k) {
    const int t = k * S::BLOCK + tid;
    tq[k] = src[(k + 1) * S::BLOCK <= TV || t < TV ? t : TV - 1];
  }
  // q_a of the own node, in the state precision until 2b; when q_a is the
  // stage input (SSPRK3 stage 1) it is read from the LDS copy of the tile
  const bool qa_is_in = A.q_a == A.q_in;
  R qa_in[NC];
  auto load_qa = [&] {
    const R *g = A.q_a + tile0 + (tid < EPB * NP ? tid : EPB * NP - 1) * NC;
#pragma unroll
    for (int c = 0; c < NC; ++c) qa_in[c] = g[c];
  };
  if constexpr (!kQaLate) {
    if (!qa_is_in) load_qa();
  }
  const int fm = A.fmap[tid < NFF ? tid : NFF - 1];
  constexpr int LPT = (NL + S::BLOCK - 1) / S::BLOCK;
  double tl[LIM ? LPT : 1];
  if constexpr (LIM) {
#pragma unroll
    for (int k = 0; k < LPT; ++k) {
      int t = k * S::BLOCK + tid;
      tl[k] = A.lim_mn_in[(size_t)e0 * NC + (t < NL ? t : NL - 1)];
    }
  }
  const int nE = A.tile_count[tile];
  const int type0 = EPB % EPC ? A.tile_type[tile] : 0;
  const int inst = A.tile_inst ? A.tile_inst[tile] : 0;
  const R tg = A.geom[(size_t)inst * GEOM + (tid < GEOM ? tid : GEOM - 1)];
  // the instance's switch, parameters and step
  const int on = A.inst_active ? A.inst_active[inst] : 1;
  const Phys phys = Phys::from(A.inst_prm + (size_t)inst * kPrmMax);
  const double cdt = A.c * (A.inst_dt ? A.inst_dt[inst] : A.dt);
  const double post = A.inst_post ? A.inst_post[inst] : A.post_scale;
  if (!on) return;
  load_item_trace<NP, EPB, LIM>(A, e0, it, itm);
  if constexpr (kTwo) load_item_trace<NP, EPB, LIM>(A, e0, it2, itm);
  int the = e0, thnb[NF] = {0};
  bool theta = false;
  if constexpr (LIM) {
    const bool far = thjob.x >= 0 && (unsigned)(thjob.y - e0) >= (unsigned)EPB && thj < A.maxj;
    theta = thj < 0 || far;
    the = thj < 0 ? e0 + tid : far ? thjob.y : e0;
    bj_neighbours<NF>(the, A.conn, thnb);
  }
  // FP64 form: the contraction streams the operator through the scalar
  // cache, which every launch starts with cold, a few rows at a time: a
  // chain of misses.  The launch's first blocks touch each line of a small
  // operator here, all at once and behind the tile's own loads (48^2 GLM-MHD
  // 7.5 -> 6.6 us, 33^2 P = 2 Euler 5.5 -> 5.1); done by every block, or for
  // operators beyond 4 KB, it cost more than it saved (16^3 P = 2 advection
  // 6.4 -> 7.7 us).
  if constexpr (!kMFMA) {
    constexpr int WAVES = S::BLOCK / 64, WORDS = stage_node_pad(EPB, NP, NC) * 2;
    constexpr int LD = (KV * WORDS + 15) / 16, LINES = LD + (NFF * WORDS + 15) / 16, LPW = (LINES + WAVES - 1) / WAVES;
    if (LINES * 64 <= kScalarWarmBytes && blockIdx.x < kScalarWarmBlocks) {
      typedef const unsigned __attribute__((address_space(4))) *Line;
      const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
      unsigned x[LPW], any = 0;
#pragma unroll
      for (int k = 0; k < LPW; ++k) {
        const int line = k * WAVES + w < LINES ? k * WAVES + w : LINES - 1;
        x[k] = line < LD ? ((Line)A.Dt)[line * 16] : ((Line)A.Lt)[(line - LD) * 16];
      }
#pragma unroll
      for (int k = 0; k < LPW; ++k) any |= x[k];
      asm volatile("" ::"s"(any));
    }
  }
  // thread tid owns output node (el, i) = (tid / NP, tid % NP): EPB*NP <= BLOCK
  const int nel = small_div<NP, S::BLOCK>(tid), nod = tid - nel * NP;
  const bool node = tid < nE * NP;
  auto limit_qa = [&] {
    if (LIM && !qa_is_in && tid < EPB * NP) {
      const size_t e = (size_t)e0 + nel;
      const double th = A.lim_th_a[e];
#pragma unroll
      for (int c = 0; c < NC; ++c) qa_in[c] = lim_apply(qa_in[c], th, A.lim_mn_a[e * NC + c]);
    }
  };
  if constexpr (!kQaLate) limit_qa();
#pragma unroll
  for (int k = 0; k < QPT; ++k) {
    const int t = k * S::BLOCK + tid;
    if ((k + 1) * S::BLOCK <= TV || t < TV) reinterpret_cast<TileVec *>(sW)[t] = tq[k];
  }
  if (tid < GEOM) sG[tid] = tg;
  if constexpr (kTwo) {
    if (t2 < nitems && it2.job.x >= 0 && (unsigned)(it2.job.y - e0) >= (unsigned)EPB) {
      R *const g = sS + (((it2.job.x >> 7) & 3) * NFP + t2 - small_div<NFP, MAXT>(t2) * NFP) * NCOLS + (it2.job.x & 127) * NC;
#pragma unroll
      for (int c = 0; c < NC; ++c) g[c] = it2.qp[c];
    }
  }
  if (tid < NFF) sMap[tid] = fm;
  if constexpr (kMFMA)
    for (int t = TILE + NFF * NCOLS + tid; t < NB0; t += S::BLOCK) sB[t] = R(0);
  if constexpr (LIM) {
#pragma unroll
    for (int k = 0; k < LPT; ++k)
      if (k * S::BLOCK + tid < NL) sLim[k * S::BLOCK + tid] = tl[k];
    if constexpr (kThetaComp) {
      if (tid < EPB * (1 + NF)) {
        sTh[tid] = 1.0;
        sNb[tid * (1 + NF)] = theta ? the : -1;
#pragma unroll
        for (int f = 0; f < NF; ++f) sNb[tid * (1 + NF) + 1 + f] = thnb[f];
      }
      __syncthreads();
      for (int t = tid; t < (EPB + A.maxj) * NC; t += S::BLOCK) {
        const int i = small_div<NC, EPB * (1 + NF) * NC>(t), e = sNb[i * (1 + NF)];
        if (e < 0) continue;
        int nb[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) nb[f] = sNb[i * (1 + NF) + 1 + f];
        const double th = bj_theta_comp<NC, true, NF>(e, t - i * NC, nb, A.lim_mn_in, A.lim_ext_in, A.lim_eps2, 1.0);
        if (th < 1.0)
          atomicMin(reinterpret_cast<unsigned long long *>(&sTh[i]), (unsigned long long)__double_as_longlong(th));
      }
    } else {
      if (theta) {
        const double th = bj_theta<NC, ND == 3, NF>(the, thnb, A.lim_mn_in, A.lim_ext_in, A.lim_eps2);
        sTh[tid] = th;
        if (thj < 0 && A.lim_th_in) A.lim_th_in[the] = th;
      }
      for (int i = tid + S::BLOCK; i < EPB + A.maxj; i += S::BLOCK) {  // more jobs than threads left
        const int2 job = jobs[i - EPB];
        if (job.x < 0 || (unsigned)(job.y - e0) < (unsigned)EPB) continue;
        bj_neighbours<NF>(job.y, A.conn, thnb);
        sTh[i] = bj_theta<NC, ND == 3, NF>(job.y, thnb, A.lim_mn_in, A.lim_ext_in, A.lim_eps2);
      }
    }
  }
  __syncthreads();
  // the q_in tile's pending limiter factors, applied in place to the
  // values this thread stored
  if constexpr (LIM) {
    if (kThetaComp && tid < EPB && A.lim_th_in) A.lim_th_in[e0 + tid] = sTh[tid];
#pragma unroll
    for (int k = 0; k < QPT; ++k) {
      const int t = k * S::BLOCK + tid;
      if (t < TV) {
#pragma unroll
        for (int v = 0; v < VW; ++v) {
          const int x = t * VW + v, el = x / (NP * NC), c = x % NC;
          sW[x] = lim_apply(tq[k][v], sTh[el], sLim[el * NC + c]);
        }
      }
    }
    __syncthreads();
  }
  const R *sQ = sW;  // the q_in tile, [el][j][c], until the flux planes are written
  // element el's place in its lattice cell
  auto cell_type = [&](int el) {
    if constexpr (EPB % EPC == 0)
      return el - small_div<EPC, 128>(el) * EPC;
    else
      return type0 + el - small_div<EPC, 128>(type0 + el) * EPC;
  };

  // ---- 2a. face fluxes ----------------------------------------------------
  // Both states of an item are read from LDS by offset: a trace that came
  // from another tile is first put into the item's own face-flux slot, which
  // only this thread touches until it writes the flux there.  Which state is
  // the left one is then a choice between two offsets.
  for (int t = tid; t < nitems; t += S::BLOCK) {
    const bool second = kTwo && t == t2;
    if (second) {
      it.job = it2.job, it.pr = it2.pr;
    } else if (t != tid) {
      load_item_records<NFP, MAXT>(jobs, ipr, t, it);
      load_item_trace<NP, EPB, LIM>(A, e0, it, itm);
    }
    if (it.job.x < 0) continue;
    const int el = it.job.x & 127, lf = (it.job.x >> 7) & 3, pin = (it.job.x >> 9) & 127;
    const int bc = (it.job.x >> 19) & 7;
    const int gi = it.job.x >> 22;
    const R *const geo = sG + 4 * gi;  // normal, area
    const int fr = lf * NFP + (t - small_div<NFP, MAXT>(t) * NFP);
    const int pl = it.job.y - e0, slot = TILE + fr * NCOLS + el * NC;
    const int mine = (el * NP + sMap[fr]) * NC;
    int other = __mul24(__mul24(pl, NP) + (int)(it.pr & 255), NC);
    if ((unsigned)pl >= (unsigned)EPB) {
      other = slot;
      if constexpr (LIM) {
        const double th = sTh[EPB + small_div<NFP, MAXT>(t)];
#pragma unroll
        for (int c = 0; c < NC; ++c) it.qp[c] = lim_apply(it.qp[c], th, itm.m[c]);
      }
      if (!second)
#pragma unroll
        for (int c = 0; c < NC; ++c) sB[slot + c] = it.qp[c];
    }
    // left = side-0 trace; right = side-1 trace or the ghost of the left
    const bool s0 = !(it.job.x & (1 << 18));
    const R *const pL = sB + (s0 ? mine : other), *const pR = sB + (s0 ? other : mine);
    const R n[3] = {geo[0], geo[1], ND == 3 ? geo[2] : R(0)};
    R ql[NC], qr[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) ql[c] = pL[c];
    if (bc)
      phys.ghost(ql, bc, n, qr);
    else
#pragma unroll
      for (int c = 0; c < NC; ++c) qr[c] = pR[c];
    R Fs[NC];
    phys.template numerical_flux<ND>(ql, qr, n, Fs);
    // FP64 form: s area F*, lifted and scaled by -inv_vol in the
    // contraction; FP32 form: -inv_vol s area F*, ready for the product
    const R w = kMFMA ? sE[cell_type(el) * GEL + ND * ND + gi] : geo[3], own = s0 ? w : -w;
#pragma unroll
    for (int c = 0; c < NC; ++c) sB[slot + c] = own * Fs[c];
    if (pin) {
      const int plf = (it.job.x >> 16) & 3, rs = it.pr >> 8;
      // (a paired job is its side-0 element's)
      const R oth = kMFMA ? -sE[cell_type(pin - 1) * GEL + ND * ND + gi] : -own;
#pragma unroll
      for (int c = 0; c < NC; ++c) sS[(plf * NFP + rs) * NCOLS + (pin - 1) * NC + c] = oth * Fs[c];
    }
  }

  // ---- 2b. nodal flux of the own node, and the RK terms of q_in ----------
  // qa becomes a q_a + b q_in + c dt S(q_in) (FP64); the flux, mapped to
  // reference directions by invJ in the form's own precision, waits in
  // registers until every read of the q_in tile is done.
  R Fk[ND * NC];
  double qa[NC];
  if constexpr (kQaLate) {
    if (!qa_is_in) {
      load_qa();
      limit_qa();
    }
  }
  if (node) {
    const R *q = &sQ[tid * NC];
    R F[ND * NC];
    phys.template flux<ND>(q, F);
    const R *iJ = sE + cell_type(nel) * GEL;
    if constexpr (kMFMA) {
      // FP32 form: the mapping in FP32 (invJ rounded to FP32), as
      // the volume product that takes its result is
#pragma unroll
      for (int k = 0; k < ND; ++k)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          float v = 0.f;
#pragma unroll
          for (int d = 0; d < ND; ++d) v += iJ[k * ND + d] * F[d * NC + c];
          Fk[k * NC + c] = v;
        }
    } else {
#pragma unroll
      for (int k = 0; k < ND; ++k)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          double v = 0.0;
#pragma unroll
          for (int d = 0; d < ND; ++d) v += iJ[k * ND + d] * double(F[d * NC + c]);
          Fk[k * NC + c] = R(v);
        }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) qa[c] = A.a * double(qa_is_in ? q[c] : qa_in[c]) + A.b * double(q[c]);
    if constexpr (Phys::kSource) {
      if (phys.source_active()) {
        R src[NC];
        phys.source(q, src);
#pragma unroll
        for (int c = 0; c < NC; ++c) qa[c] += cdt * double(src[c]);
      }
    }
  }
  // FP32-MFMA: the operator entries of a whole product go straight to the
  // registers of the lanes that feed them to the MFMA, one coalesced load
  // each, ahead of the barrier before the product.  Staged in LDS, the
  // operator took 12.8 of the 28.7 KB of a 3D P = 3 block and held it to 5
  // blocks per CU (us per stage: 32^3 Taylor-Green 115 -> 108, 19^3 30.7 ->
  // 29.3, 113^2 P = 4 Maxwell 11.3 -> 11.0, 128^2 vortex 8.8 -> 8.6).
  constexpr int KL = (KPAD - KVP) / 4, KD = KVP / 4;      // k-steps of the lift and volume products
  // Up to 30 entries a lane (3D P = 3); the 81 of P = 4 would take the registers
  // of other blocks (13^3 Euler 27.6 us loaded as it goes, 38.3 ahead, shallow
  // water 21.5 and 29.6).
  constexpr bool kAhead = kMFMA && MT * (KL > KD ? KL : KD) <= 32;
  constexpr int WAVES = S::BLOCK / 64, NTW = (NT + WAVES - 1) / WAVES;  // column tiles per wave
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // A wave without a column tile loads no operator and multiplies nothing.
  // One component (or three at P = 5) leaves one to three of the block's
  // waves without one; when they took part, the loads and MFMAs they
  // repeated held up the other blocks (us per stage, 18^3 P = 3 advection
  // 17.6 -> 10.8, 10^3 P = 5 36.4 -> 14.6, shallow water 37.4 -> 16.3).
  const bool cols = NT > (WAVES - 1) * NTW || wave * NTW < NT;
  const int l = tid & 63, lr = l & 15, lg = l >> 4;
  auto aop = [&](int k, int m) { return A.Aop[(k * MT + m) * 64 + l]; };
  [[maybe_unused]] float al[kAhead ? KL : 1][MT], ad[kAhead ? KD : 1][MT];
  if (kAhead && cols) {
#pragma unroll
    for (int k = 0; k < KL; ++k)
#pragma unroll
      for (int m = 0; m < MT; ++m) al[k][m] = aop(KD + k, m);
  }
  __syncthreads();

  // ---- 3. contractions ----------------------------------------------------
  // rhs_i = sum_k sum_j D_k[i][j] F_kj - inv_vol sum_fr Lift[fr][i] S_fr in
  // two products: first the lift over the face fluxes, then -- once the
  // face fluxes and the q_in tile are no longer read -- the flux planes are
  // written over them and the volume product accumulates onto the same
  // registers.  The result goes to [el][i][c] at the start of the array.
  //
  // FP32-MFMA: Out[i][col] = sum_k Aop[i][k] B[k][col] with the operator
  // columns [D (KVP) | Lift (KPAD - KVP)]; V_MFMA_F32_16X16X4F32 operands,
  // lane l = 16 g + r: A[r][k0 + g], B[k0 + g][col0 + r]; result rows
  // 4 g + v (v < 4), column col0 + r.
  mxm_float4 macc[kMFMA ? MT : 1][kMFMA ? NTW : 1];
  // FP64 on the VALU: the (element, component) columns are the lanes;
  // each wave group produces IH consecutive output nodes, so the operator
  // entries are wave-uniform (scalar loads)
  constexpr int GROUPS = stage_groups(EPB, NC);
  constexpr int GSIZE = S::BLOCK / GROUPS;
  constexpr int NPAD = stage_node_pad(EPB, NP, NC);
  constexpr int IH = NPAD / GROUPS;
  constexpr int ITER = (NCOL + GSIZE - 1) / GSIZE;  // columns per thread, at most
  const int grp = __builtin_amdgcn_readfirstlane(tid / GSIZE);
  const int i0 = grp * IH;
  const int lane = tid - grp * GSIZE;
  double dacc[kMFMA ? 1 : ITER][kMFMA ? 1 : IH];

  // acc[ii] += sum_r op[r][ii] col[r] over N rows: RB rows at a time, the next
  // rows' scalar and LDS loads in flight behind the FMAs of the present ones
  // (two sets of RB*IH operator entries in scalar registers).  Scalar
  // loads return out of order, so a wait for some is a wait for all: it
  // stands before the next rows are asked for.  Against one set, loaded and
  // waited for, us per stage: 512^2 vortex 149.7 -> 145.4, 128^2 14.1 -> 13.7,
  // 32^3 Taylor-Green 181 -> 176.5, 16^3 P = 2 advection 7.5 -> 6.7.
  // A set holds up to 16 entries; three rows of 3, since five (two sets of 30
  // scalar registers) gained nothing at best and made larger meshes slower (us
  // per stage, five rows / three: 320^2 P = 3 advection 22.1 / 19.0, limited
  // 36.9 / 31.2, 34^3 P = 2 34.0 / 31.6); and two rows of 9 or 10 where the product
  // is longer than a 2D P = 3 one (20 rows): with one row of 10 a wave had 10
  // FMAs to cover each wait (us per stage, one set / one row / two rows:
  // 18^3 P = 3 Maxwell 51.4 / 58.3 / 49.1, MHD 71.5 / 81.5 / 66.9, 13^3 P = 4
  // MHD 98 / 92 / 64; 100^2 P = 3 GLM-MHD 15.8 / 12.5 / 13.2).
  // P = 5 tets, 14 entries a row from 75 KB of operator, have no room for two
  // rows: with 3 to 9 components the plain loop, whose loads the compiler
  // batches, is faster (10^3 Euler 76.0 / 76.1 / plain loop 73.5, MHD 84.6 /
  // 97 / 79.3, Maxwell 72 / 72 / 65), with one or 17 this one (advection 124 /
  // 81, two-fluid 480 / 304).
  [[maybe_unused]] auto contract = [&](const R *col, ScalarPtr op, auto N, double (&acc)[kMFMA ? 1 : IH]) {
    if constexpr (NP == 56 && NC > 1 && NC < 17) {
#pragma unroll 4
      for (int r = 0; r < N; ++r) {
        const double v = col[r * NCOLS];
#pragma unroll
        for (int ii = 0; ii < IH; ++ii) acc[ii] += op[r * NPAD + ii] * v;
      }
      return;
    }
    constexpr int RB = IH == 3 ? 3 : IH <= 8 ? 16 / IH : IH <= 10 && N > 20 ? 2 : 1, SETS = (N + RB - 1) / RB;
    double o[2][RB][IH], v[2][RB];
    auto load = [&](int b, int s) {
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        const int row = b * RB + r < N ? b * RB + r : N - 1;  // past the end: loaded, not used
        v[s][r] = col[row * NCOLS];
#pragma unroll
        for (int ii = 0; ii < IH; ++ii) o[s][r][ii] = op[row * NPAD + ii];
      }
    };
    auto use = [&](int s, int n) {
#pragma unroll
      for (int r = 0; r < RB; ++r)
        if (r < n) {
#pragma unroll
          for (int ii = 0; ii < IH; ++ii) acc[ii] += o[s][r][ii] * v[s][r];
        }
    };
    auto arrived = [] {
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
      __builtin_amdgcn_sched_barrier(0);
    };
    // short products in full (16^3 P = 2 advection 8.0 -> 6.7 us); long ones
    // as a loop, which costs them nothing
    constexpr int pairs = N * IH <= 100 ? SETS : 1;
    load(0, 0);
#pragma unroll pairs
    for (int b = 0; b + 2 < SETS; b += 2) {
      arrived();
      load(b + 1, 1);
      __builtin_amdgcn_sched_barrier(0);
      use(0, RB);
      arrived();
      load(b + 2, 0);
      __builtin_amdgcn_sched_barrier(0);
      use(1, RB);
    }
    // the last set or two
    constexpr int left = SETS % 2 ? 1 : 2, last = N - (SETS - 1) * RB;
    arrived();
    if constexpr (left == 2) {
      load(SETS - 1, 1);
      __builtin_amdgcn_sched_barrier(0);
      use(0, RB);
      arrived();
      use(1, last);
    } else {
      use(0, last);
    }
  };
  // One 4-deep step of the MFMA product: operator entries a, operand rows
  // 4 kb .. of Bb.  Branch-free, so that the operand reads of many
  // steps are in flight together: a wave's column tile past the last one
  // repeats the last (its result is not stored).  With a branch around it
  // each step waited for its own LDS reads (us per stage: 128^2 vortex 9.4 ->
  // 8.8, 512^2 86 -> 82.3, 32^3 Taylor-Green 123.5 -> 115, 16^2 4.8 -> 4.3).
  int bcol[NTW];
#pragma unroll
  for (int w = 0; w < NTW; ++w) {
    const int nt = wave * NTW + w;
    bcol[w] = lg * NCOLS + (nt < NT ? nt : NT - 1) * 16 + lr;
  }
  auto kstep = [&](const R *Bb, const float (&a)[MT], int kb) {
#pragma unroll
    for (int w = 0; w < NTW; ++w) {
      const float bv = float(Bb[kb * 4 * NCOLS + bcol[w]]);
#pragma unroll
      for (int m = 0; m < MT; ++m) macc[m][w] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m], bv, macc[m][w], 0, 0, 0);
    }
  };
  // the product over the k-steps [k0, k1) of the operator, entries loaded as
  // it goes
  [[maybe_unused]] auto product = [&](const R *Bb, int k0, int k1) {
#pragma unroll 4
    for (int k = k0; k < k1; ++k) {
      float a[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) a[m] = aop(k, m);
      kstep(Bb, a, k - k0);
    }
  };

  // ---- 3a. lift product over the face fluxes -----------------------------
  if constexpr (kMFMA) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int w = 0; w < NTW; ++w) macc[m][w] = mxm_float4{0.f, 0.f, 0.f, 0.f};
    if (cols) {
      if constexpr (kAhead) {
#pragma unroll
        for (int k = 0; k < KL; ++k) kstep(sS, al[k], k);
      } else {
        product(sS, KD, KD + KL);
      }
    }
  } else {
#pragma unroll
    for (int m = 0; m < ITER; ++m) {
      const int p = lane + m * GSIZE;
#pragma unroll
      for (int ii = 0; ii < IH; ++ii) dacc[m][ii] = 0.0;
      if (p < nE * NC) {
        const int el = small_div<NC, ITER * GSIZE>(p);
        contract(sS + p, (ScalarPtr)A.Lt + i0, std::integral_constant<int, NFF>{}, dacc[m]);
        const double niv = -sE[cell_type(el) * GEL + ND * ND];
#pragma unroll
        for (int ii = 0; ii < IH; ++ii) dacc[m][ii] *= niv;
      }
    }
  }
  __syncthreads();

  // ---- 3b. flux planes over the face fluxes and the q_in tile -------------
  if (node) {
    R *const g = sW + nod * NCOLS + nel * NC;
#pragma unroll
    for (int k = 0; k < ND; ++k)
#pragma unroll
      for (int c = 0; c < NC; ++c) g[k * NP * NCOLS + c] = Fk[k * NC + c];
  }
  if constexpr (kMFMA && KVP > KV)
    for (int t = KV * NCOLS + tid; t < KVP * NCOLS; t += S::BLOCK) sB[t] = R(0);
  if (kAhead && cols) {
#pragma unroll
    for (int k = 0; k < KD; ++k)
#pragma unroll
      for (int m = 0; m < MT; ++m) ad[k][m] = aop(k, m);
  }
  __syncthreads();

  // ---- 3c. volume product, result as [el][i][c] ---------------------------
  if constexpr (kMFMA) {
    if (cols) {
      if constexpr (kAhead) {
#pragma unroll
        for (int k = 0; k < KD; ++k) kstep(sW, ad[k], k);
      } else {
        product(sW, 0, KD);
      }
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NTW; ++w) {
      const int col = (wave * NTW + w) * 16 + lr;
      if (wave * NTW + w < NT && col < nE * NC) {
        const int el = small_div<NC, NT * 16>(col);
        R *const g = sW + el * (NP * NC) + (col - el * NC);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int i = m * 16 + 4 * lg + v;
            if (i < NP) g[i * NC] = R(macc[m][w][v]);
          }
      }
    }
  } else {
#pragma unroll
    for (int m = 0; m < ITER; ++m) {
      const int p = lane + m * GSIZE;
      if (p < nE * NC) {
        contract(sW + p, (ScalarPtr)A.Dt + i0, std::integral_constant<int, KV>{}, dacc[m]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < ITER; ++m) {
      const int p = lane + m * GSIZE;
      if (p < nE * NC) {
        const int el = small_div<NC, ITER * GSIZE>(p);
        R *const g = sW + el * (NP * NC) + i0 * NC + (p - el * NC);
#pragma unroll
        for (int ii = 0; ii < IH; ++ii)
          if (i0 + ii < NP) g[ii * NC] = R(dacc[m][ii]);
      }
    }
  }
  __syncthreads();

  // ---- 4. RK combine (FP64), limit per (element, node), tile store -------
  // Each node thread writes its finished values over its own entries of the
  // [el][i][c] result (the tile's device order); after a barrier the block
  // stores the tile's real elements as one contiguous run, every lane
  // consecutive, so each cache line is written whole at once (per-node
  // stores at a stride of NC leave partly written lines in L2 that are
  // written back more than once when many blocks are resident).
  if (node) {
    double out[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) out[c] = qa[c] + cdt * double(sW[tid * NC + c]);
    if constexpr (Phys::kLimit) phys.limit(out);
    if constexpr (Phys::kPost >= 0)
      if (A.post_comp == Phys::kPost) out[Phys::kPost] *= post;
    const unsigned salt = unsigned(nod) * 0x85EBCA6Bu;  // node in its element
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if constexpr (kMFMA)
        sW[tid * NC + c] = sr_f32(out[c], salt);
      else
        sW[tid * NC + c] = R(out[c]);
    }
  }
  __syncthreads();
  {
    R *const g = A.q_out + tile0;
    const int nv = nE * NP * NC;
    bool bad = false;
    if (nE == EPB) {
      TileVec *const gv = reinterpret_cast<TileVec *>(g);
#pragma unroll
      for (int k = 0; k < QPT; ++k) {
        const int t = k * S::BLOCK + tid;
        if ((k + 1) * S::BLOCK <= TV || t < TV) {
          const TileVec v = reinterpret_cast<const TileVec *>(sW)[t];
          gv[t] = v;
          if (A.inst_fail) {
#pragma unroll
            for (int x = 0; x < VW; ++x) bad = bad || !__builtin_isfinite(v[x]);
          }
        }
      }
    } else {  // a tile with padding slots, which stay as they are
      for (int t = tid; t < nv; t += S::BLOCK) {
        const R v = sW[t];
        g[t] = v;
        bad = bad || !__builtin_isfinite(v);
      }
    }
    if (bad && A.inst_fail) atomicOr(&A.inst_fail[inst], 1);
  }
  // ---- 5. cell means of the stored state (limiter) -----------------------
  // sum_i w_i q_i per (element, component) in node order, FP64, from the
  // stored values: what a separate pass over q_out would compute
  if constexpr (LIM) {
    // FP64: 56 nodes are not read all at once.  Maxwell's kernel held 132 VGPRs
    // for that, 3 waves per SIMD where its LDS lets 4 run (15^3 limited, us per
    // stage: 242.7, in two halves 217.5); smaller elements and FP32 lose by it
    constexpr int kUnroll = !kMFMA && NP == 56 ? 28 : NP;
    for (int p = tid; p < nE * NC; p += S::BLOCK) {
      const int el = p / NC, c = p - el * NC;
      double sm = 0.0;
#pragma unroll kUnroll
      for (int n = 0; n < NP; ++n) sm += A.w[n] * double(sW[(el * NP + n) * NC + c]);
      A.mean[(size_t)(e0 + el) * NC + c] = sm;
      constexpr int NCL = ND == 3 ? NC : 1;  // the components the limiter bounds
      if (c < NCL) {
        double lo = double(sW[el * NP * NC + c]), hi = lo;
#pragma unroll kUnroll
        for (int n = 1; n < NP; ++n) {
          const double v = double(sW[(el * NP + n) * NC + c]);
          lo = v < lo ? v : lo;
          hi = v > hi ? v : hi;
        }
        A.ext[((size_t)(e0 + el) * NCL + c) * 2] = R(lo);
        A.ext[((size_t)(e0 + el) * NCL + c) * 2 + 1] = R(hi);
      }
    }
  }
}

// A shape without a distinct wide tile launches its one kernel for WIDE.
template <class Phys, int ND, int P, class R, int W, bool LIM, bool WIDE>
hipError_t launch_stage(const void *args, hipStream_t s) {
  constexpr bool kWide = WIDE && std::is_same<R, float>::value && Shape<ND, P, Phys::NC>::kHasWide;
  if constexpr (WIDE && !kWide) {
    return launch_stage<Phys, ND, P, R, W, LIM, false>(args, s);
  } else {
    using S = StageShape<Phys, ND, P, R, WIDE>;
    const StageArgs<R> &a = *static_cast<const StageArgs<R> *>(args);
    const int nb = a.ntiles;
    if (nb <= 0) return hipSuccess;
    // The 17 components of the two-fluid system spill 44 to 64 VGPRs of the
    // FP32 kernels at 5 waves, where the LDS lets 5 be asked for; their
    // 5-wave configuration is built for 4 (us per stage, 5 / 4 waves: 28^3
    // P = 1 86 / 58, 22^3 P = 2 87 / 64, 18^3 P = 3 98 / 81, 10^3 P = 5 111 / 85).
    constexpr int kWaves = std::is_same<R, float>::value && Phys::NC >= 17 && W == 5 ? 4 : W;
    hipLaunchKernelGGL((dg_stage_kernel<Phys, ND, P, R, kWaves, LIM, WIDE>), dim3(nb), dim3(S::BLOCK), 0, s, a);
    return hipGetLastError();
  }
}

// args points to StageArgs<double> (FP64 form) or StageArgs<float>
// (FP32-MFMA form); the tables are in stage_families.hpp.
using StageLaunch = hipError_t (*)(const void *args, hipStream_t);

}  // namespace mxm
