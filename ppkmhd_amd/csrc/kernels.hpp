// Interface between the host driver (capi.cpp) and the kernel translation units.  Each kernel
// file is compiled once per arithmetic variant into its own namespace (ppk::fast,
// ppk::strict); the driver picks one table of entry points per solver handle.
#pragma once

#include <hip/hip_runtime.h>

#include "mhd_device.hpp"

namespace ppk {

// slots of the device-resident time-loop control block (doubles)
enum {
  CTRL_T = 0,        // current time
  CTRL_DT = 1,       // dt of the step in flight
  CTRL_INVDT = 2,    // CFL maximum max_cells sum_d (c_f + |v_d|)/dx_d of the state (set_dt)
  CTRL_ITER = 3,     // iteration counter (exact in a double up to 2^53)
  CTRL_TEND = 4,
  CTRL_NSTEPMAX = 5,
  CTRL_ACTIVE = 6,   // 0 once SolverBase::finished() held before a checked step
  CTRL_SPARE = 7,
  CTRL_SLOTS = 8
};

// kernel stages bracketed by the optional per-stage GPU timers (ppk_mhd_timers_*)
enum Stage {
  ST_BOUNDARIES = 0,
  ST_PRIM_DT,
  ST_ELEC,
  ST_MAGSLOPES,
  ST_TRACE,
  ST_FLUXES,
  ST_EMF,
  ST_UPDATE,
  ST_CONTROL,
  ST_FUSED_HALF,     // fused: primitives + E + slopes + half step (compact records)
  ST_FUSED_RIEMANN,  // fused: Riemann problems at faces + EMFs at edges
  ST_FUSED_UPDATE,   // fused: update + CT + ghost copy (+ CFL of the new state)
  ST_FUSED_CFL,      // fused: standalone CFL reduction
  ST_FUSED_MARCH,    // single-pass step (half step, solves, update, CT, CFL in one kernel)
  ST_SUR_FACES,      // surrogate form: the network's face solves (inside ST_FUSED_RIEMANN)
  ST_SUR_FALLBACK,   // surrogate form: exact HLLD of the refused faces (same)
  ST_COUNT
};
// host-side hook the launchers call around each stage (implemented by the driver)
struct StageTimer {
  virtual void mark(int stage, bool start) = 0;
  virtual ~StageTimer() {}
};
#define PPK_TIMED(tm, stage, launch)   \
  do {                                 \
    if (tm) (tm)->mark((stage), true); \
    launch;                            \
    if (tm) (tm)->mark((stage), false); \
  } while (0)

// scratch of the stage-per-kernel form (all over the padded box, SoA)
struct StagedScratch {
  double *faces = nullptr;  // 2*dim face states x 8 vars
  double *edges = nullptr;  // 4*(3 in 3D, 1 in 2D) edge states x 8 vars
  double *flux = nullptr;   // dim fluxes x 8 vars
  double *emf = nullptr;    // 3 (3D) or 1 (2D) EMF components
  double *elec = nullptr;   // 3D: 3 E components
  double *dbf = nullptr;    // 3D: 6 transverse face-field slopes
};

// scratch of the fused form (padded-box indexing, SoA)
constexpr int kRec3 = 38;   // half-step record per cell, 3D
constexpr int kRec2 = 26;   // half-step record per cell, 2D
constexpr int kFluxComp3 = 5;  // ID IP IU IV IW per face direction, 3D
constexpr int kFluxComp2 = 6;  // ID IP IU IV IW IC per face direction, 2D
// the surrogate form of the face solves: network, gate, counters (device memory)
// blocks of a surrogate face launch (at most): three per CU of an MI355X, as many as its LDS
// holds (measured: 2D step 0.344 -> 0.324 ms, 3D 57.8 -> 56.6 ms against two per CU)
constexpr int kSurrogateBlocks = 768;
struct SurrogateCfg {
  const void *net = nullptr;            // packed network (MlpPacked, device)
  double gate_rho = 0.0, gate_p = 0.0;  // max relative jumps |a_R - a_L| / min(a_L, a_R)
  // per launch block b: [2b] faces by the network, [2b + 1] by HLLD (2 x kSurrogateBlocks
  // counters, accumulated over launches), or null
  unsigned long long *counters = nullptr;
  unsigned char *flags = nullptr;  // dim x cells: faces left to the HLLD pass (device scratch)
};
// element type of rec and flux: double, or float in the FP32-bulk form (DevParams::bulk32)
struct FusedScratch {
  void *rec = nullptr;   // kRec{2,3} x cells
  void *flux = nullptr;  // dim x kFluxComp{2,3} x cells
  void *emf = nullptr;   // 3 (3D) or 1 (2D) x cells, double in every form
  const SurrogateCfg *sur = nullptr;  // surrogate face solves when set
};

// dt modes of the set_dt kernel; SETDT_LATER: a prologue that leaves dt to a later set_dt
enum { SETDT_FIXED = 0, SETDT_CFL = 1, SETDT_REDUCE_ONLY = 2, SETDT_LATER = 3 };
// CFL partials that the prologue's one block of 256 threads reduces itself; more of them go to
// set_dt (1024 threads).  8192 take four rounds of eight loads per thread, about 3 us, which
// the ghost fill beside it covers.
constexpr int kPrologueParts = 8192;

// The CFL maximum is produced as per-block partial maxima (no same-address atomics): each
// block of a producer kernel writes its slot, set_dt reduces as many slots as the producer had
// blocks.  Staged primitives: cfl_blocks(p) blocks (grid-stride); fused update and fused CFL:
// one block per brick of the padded box, fused_cfl_parts(p).
constexpr int kCflBlock = 256;
constexpr int kCflMaxBlocks = 4096;
inline int cfl_blocks(const DevParams &p) {
  long long cells = (long long)p.isize * p.jsize * p.ksize;
  long long g = (cells + kCflBlock - 1) / kCflBlock;
  if (g > kCflMaxBlocks) g = kCflMaxBlocks;
  return g < 1 ? 1 : (int)g;
}

// Bricks: the fused per-cell kernels give each block of 256 threads a brick of cells.
// Shape 0 (default) is a run of 256 consecutive cells of the flattened range (one wave = 64
// cells of one x row); its rows are numbered in patches of 4 x 4 (y, z) rows in 3D, so the
// rows a cell's y and z neighbours live in were visited a few rows earlier (L2 hits).
// Shapes 1-3 are 3D bricks 64 x 2 x 2, 16 x 4 x 4, 32 x 4 x 2 (2D: 64 x 4), among which the
// batch's autotuner picks; single grids use shape 0.
constexpr int kPatch = 4;
struct Brick {
  int bx, by, bz;  // brick extents; bx = 0: flattened runs, by x bz = row patch
  int nx, ny, nz;  // bricks per direction; flattened: patches per direction in ny, nz
  int mx, my, mz;  // cells covered per direction
  long long nblocks;
  long long count() const { return nblocks; }
};
inline Brick make_brick(int dim, int mx, int my, int mz, int shape) {
  Brick b;
  b.mx = mx;
  b.my = my;
  b.mz = mz;
  if (shape <= 0 || shape > 3) {
    b.bx = 0;
    b.by = dim == 3 ? kPatch : 1;
    b.bz = dim == 3 ? kPatch : 1;
    b.ny = (my + b.by - 1) / b.by;
    b.nz = (mz + b.bz - 1) / b.bz;
    const long long rows = (long long)b.ny * b.by * b.nz * b.bz;
    b.nx = 0;
    b.nblocks = (rows * mx + 255) / 256;
    return b;
  }
  static const int shp[4][3] = {{0, 0, 0}, {64, 2, 2}, {16, 4, 4}, {32, 4, 2}};
  b.bx = dim == 3 ? shp[shape][0] : 64;
  b.by = dim == 3 ? shp[shape][1] : 4;
  b.bz = dim == 3 ? shp[shape][2] : 1;
  b.nx = (mx + b.bx - 1) / b.bx;
  b.ny = (my + b.by - 1) / b.by;
  b.nz = (mz + b.bz - 1) / b.bz;
  b.nblocks = (long long)b.nx * b.ny * b.nz;
  return b;
}
// bricks of the padded box (fused update, fused CFL)
inline Brick padded_bricks(const DevParams &p) {
  return make_brick(p.dim, p.isize, p.jsize, p.ksize, p.brick);
}
inline int fused_cfl_parts(const DevParams &p) { return (int)padded_bricks(p).count(); }
// the sub-box [gw, size-gw] per direction of the face and edge kernels, in bricks
inline Brick sub_bricks(const DevParams &p) {
  return make_brick(p.dim, p.nx + 1, p.ny + 1, p.dim == 3 ? p.nz + 1 : 1, p.brick);
}

// The single-pass 3D step (march3d.hip): blocks of 16 x 12 output columns marching along z
// through equal shares of the grid's tile-planes; one CFL partial per block
constexpr int kMarchOutX = 16, kMarchOutY = 12;
// Blocks of the launch: one per CU (each block needs a whole CU's LDS), fewer only when there
// are fewer tile-planes.  Every segment starts with the work of about two planes more, but a CU
// without a block gains nothing: at least 16 tile-planes per block left 231 CUs idle on a
// 37 x 29 x 45 box (286 us per step, then 75).
inline int march_nblk(const DevParams &p, int cus) {
  const long long total =
      (long long)((p.nx + kMarchOutX - 1) / kMarchOutX) * ((p.ny + kMarchOutY - 1) / kMarchOutY) *
      p.nz;
  long long b = cus > 0 ? cus : 256;
  if (b > total) b = total;
  return (int)(b < 1 ? 1 : b);
}
// PPK_PATH_AUTO: whether the single-pass 3D step is the faster form.  Its time is that of the
// tile-planes of one block, 15 us each, two more per segment (a second segment where the ranges
// cut tiles); the three-kernel form takes 0.43 us per 1000 cells once its launches are paid.
// Measured us per step, single-pass / three-kernel: 16^3 41 / 32, 32^3 45 / 42, 37x29x45 76 / 45,
// 48^3 74 / 75, 64^3 133 / 130, 72^3 153 / 162, 80^3 194 / 242, 96^3 284 / 398, 160x20x20 57 / 60.
// Near the crossing the estimate can take the slower form by a few percent (64^3: the single pass).
inline bool march_pays(const DevParams &p, int cus) {
  const double tiles =
      (double)((p.nx + kMarchOutX - 1) / kMarchOutX) * ((p.ny + kMarchOutY - 1) / kMarchOutY);
  const int b = march_nblk(p, cus);
  const int planes = (int)((tiles * p.nz + b - 1) / b);
  const double march = 28.0 + 15.2 * planes + (p.nz % planes ? 16.0 : 0.0);
  return march < 27.0 + 0.43e-3 * p.nx * p.ny * (double)p.nz;
}
// The single-pass 2D step (march2d.hip): strips of lw - 4 output columns (lw = 64 or 32 lanes)
// by `rows` output rows, 64 / lw strips per wave; one CFL partial per wave
inline long long march2d_waves(const DevParams &p, int lw, int rows) {
  const long long strips = (long long)((p.nx + lw - 5) / (lw - 4)) * ((p.ny + rows - 1) / rows);
  return (strips + 64 / lw - 1) / (64 / lw);
}
// Relative time of a launch of `waves` strips of `rows` output rows.  A strip takes rows + 2
// passes and a start of about one more.  One wave per SIMD issues instructions in 9 of 10
// cycles, so a second wave on the same SIMD hides the start but little else: two take 1.9 times
// as long as one, and so on per further wave.  Few rows give many waves but more passes per
// row.  Measured (us per launch, MI355X, Orszag-Tang; strips of 64 columns; the leaner solvers
// since took 10 to 13 % off each):
//   64^2    1 row 17.7, 2 rows 22.8, 3 rows 27.8        (128, 64, 44 waves)
//   256^2   1 row 27.4, 2 rows 24.3, 4 rows 34.1        (1280, 640, 320)
//   1024^2  8 rows 130, 10 rows 108, 20 rows 121, 32 rows 179  (2304, 1854, 936, 576)
//   2048^2  24 rows 362, 32 rows 448, 36 rows 361, 64 rows 563 (3010, 2240, 1995, 1120)
// 32-column strips (two per wave) were within 3 % of these; they pay where 64 columns leave
// lanes idle, which the wave count shows.
inline double march2d_time(double waves, int rows, int cus) {
  const double simds = 4.0 * (cus > 0 ? cus : 256);
  const double per = waves <= simds ? 1.0 : (double)(long long)((waves + simds - 1.0) / simds);
  return per <= 1.0 ? rows + 3.1 : 0.93 * per * (rows + 1.6);
}
// sets march_lw, march_rows and march
inline void march2d_shape(DevParams &p, int cus) {
  double best = 0.0;
  for (int lw = 64; lw >= 32; lw /= 2)
    for (int rows = 1; rows <= p.ny; ++rows) {
      if (best > 0.0 && rows + 2.9 > best) break;  // no launch takes less than its rows + 2.9
      const double t = march2d_time((double)march2d_waves(p, lw, rows), rows, cus);
      if (best == 0.0 || t < best * 0.999) {
        best = t;
        p.march_lw = lw;
        p.march_rows = rows;
      }
    }
  p.march = (int)march2d_waves(p, p.march_lw, p.march_rows);
}
// PPK_PATH_AUTO: whether the single-pass 2D step is the faster form (shape set by march2d_shape).
// Times of a step in us: the single pass by the rows of a strip and the waves per SIMD, the
// three-kernel form by the padded cells, dearer per cell once its records leave the caches.
// Measured single-pass / three-kernel, default build: 64^2 19 / 24, 256^2 27 / 31, 2048^2 299 / 880,
// 16x4096 31 / 34, 5x20000 65 / 57, 5x200000 438 / 577; strict build: 64^2 30 / 29, 256^2 48 / 40,
// 400^2 55 / 59, 2048^2 665 / 1008, 16x4096 52 / 42, 67x1272 52 / 41, 5x20000 129 / 72, 30x30000
// 303 / 280.  Strips of a narrow grid leave most lanes idle; the strict build's exact quotients
// cost the single pass, bound by issue at few waves, more than the other form.
inline bool march2d_pays(const DevParams &p, int cus, bool strict) {
  const double simds = 4.0 * (cus > 0 ? cus : 256);
  const double per = p.march <= simds ? 1.0 : (double)(long long)((p.march + simds - 1.0) / simds);
  const double rows = p.march_rows * (p.march_lw == 32 ? 1.12 : 1.0);
  const double k = (double)p.isize * p.jsize * 1e-3, far = k > 700.0 ? k - 700.0 : 0.0;
  if (strict)
    return (per <= 1.0 ? 18.5 + 11.3 * rows : 34.0 + 8.75 * per * rows) <
           25.0 + 0.2 * k + 0.045 * far;
  return (per <= 1.0 ? 14.5 + 5.0 * rows : 22.0 + 3.9 * per * rows) <
         22.0 + 0.14 * k + 0.1 * far;
}
// Whether the single-pass steps can give the CFL maxima of the state they write.  Behind the last
// cell of a direction they take the new face field of the ghost cell as computed from that last
// cell.  With both faces periodic this is what the next ghost fill puts there; with only the upper
// face periodic the fill copies the first cell's value, which the lower ghosts went into: dt then
// comes from a CFL pass of its own over the filled state (per step, with / without: 64^2 25 / 19 us,
// 2048^2 368 / 335 us, 256^3 4.72 / 4.61 ms).
inline bool march_folds_cfl(const DevParams &p) {
  for (int d = 0; d < p.dim; ++d)
    if (p.bc[2 * d + 1] == PPK_BC_PERIODIC && p.bc[2 * d] != PPK_BC_PERIODIC) return false;
  return true;
}
inline long long march_blocks(const DevParams &p) { return p.march > 0 ? p.march : 0; }

// half-step tile shapes of a batch (batch_block_counts / batch_step `tile`): 2D 32x8, 64x4,
// 16x16; 3D 16x4x4, 8x8x4, 32x4x2
constexpr int kBatchTiles = 3;

// ---- batched ensembles: many independent grids of one dimension advanced by the same
// launches.  Each batched launch covers the blocks of every member back to back; a member
// owns blocks [begin[stage], begin[stage] + its count) of that stage.
enum BatchStage {
  BS_BND = 0,                      // ghost fill of every face, edge and corner (one pass)
  BS_CFL,                          // standalone CFL of the current state (first step)
  BS_HALF, BS_RIEMANN, BS_UPDATE,  // the three fused stages
  BS_COUNT
};
struct BatchMember {
  DevParams p;
  double *U[2];        // ping-pong states; the current one is U[iteration & 1]
  void *rec, *flux, *emf;
  double *ctrl;        // the member's control block (CTRL_SLOTS)
  double *parts;       // the member's CFL partial maxima
  Brick pad, sub;      // bricks of the padded box and of the face/edge sub-box
  long long begin[BS_COUNT];
  int nparts;
  int unused;
};

#define PPK_DECLARE_KERNELS(NS)                                                                  \
  namespace NS {                                                                                 \
  /* ghost fill of U */                                                                          \
  hipError_t staged_boundaries(const DevParams &p, double *U, const double *ctrl,                \
                               hipStream_t s, StageTimer *tm);                                   \
  /* the finished test, the ghost fill of U and dt in one launch; copy (may be null) receives    \
     the same ghost values; nparts at most kPrologueParts unless mode is SETDT_FIXED or          \
     SETDT_LATER */                                                                              \
  hipError_t staged_prologue(const DevParams &p, double *U, double *copy, double *ctrl,          \
                             const double *parts, int nparts, double fixed_dt, int mode,         \
                             double cfl, int check_finished, hipStream_t s, StageTimer *tm);     \
  hipError_t staged_prim_dt(const DevParams &p, const double *U, double *Q, double *parts,       \
                            const double *ctrl, int do_dt, hipStream_t s, StageTimer *tm);       \
  hipError_t staged_begin(double *ctrl, int check_finished, hipStream_t s);                      \
  hipError_t staged_set_dt(double *ctrl, const double *parts, int nparts, double fixed_dt,       \
                           int mode, double cfl, hipStream_t s);                                 \
  hipError_t staged_end(double *ctrl, hipStream_t s);                                            \
  hipError_t staged_godunov(const DevParams &p, const double *Uin, double *Uout,                 \
                            const double *Q, StagedScratch &w, const double *ctrl,               \
                            hipStream_t s, StageTimer *tm);                                      \
  /* the fused steps: their last kernel ends the step (step_end, `host` its pinned copy) */      \
  hipError_t fused_godunov(const DevParams &p, const double *Uin, double *Uout,                  \
                           FusedScratch &w, double *parts, double *ctrl, double *host,           \
                           int fold_cfl, hipStream_t s, StageTimer *tm);                         \
  hipError_t fused_cfl(const DevParams &p, const double *U, double *parts, const double *ctrl,   \
                       hipStream_t s, StageTimer *tm);                                           \
  hipError_t fused_half(const DevParams &p, const double *U, void *rec, const double *ctrl,      \
                        hipStream_t s);                                                          \
  /* surrogate form: face solves, and the training-sample dump of the current records */        \
  hipError_t surrogate_faces(const DevParams &p, const void *rec, void *flux,                    \
                             const double *ctrl, const SurrogateCfg &cfg, hipStream_t s,         \
                             StageTimer *tm);                                                    \
  hipError_t surrogate_dump(const DevParams &p, const void *rec, const double *ctrl, float *X,   \
                            float *T, long long stride, long long phase, hipStream_t s);         \
  long long surrogate_dump_slots(const DevParams &p, long long stride, long long phase);         \
  /* single-pass 3D step (p.march > 0): the interior of Uout (its ghosts come from the ghost   \
     fill's copy target); CFL partials, one per block, when fold_cfl */                         \
  hipError_t march_godunov(const DevParams &p, const double *Uin, double *Uout, double *parts,   \
                           double *ctrl, double *host, int fold_cfl, hipStream_t s,              \
                           StageTimer *tm);                                                      \
  /* the same in 2D: CFL partials, one per wave */                                             \
  hipError_t march2d_godunov(const DevParams &p, const double *Uin, double *Uout, double *parts, \
                             double *ctrl, double *host, int fold_cfl, hipStream_t s,            \
                             StageTimer *tm);                                                    \
  /* batched ensemble: counts of blocks per stage for one member, then the batched step */      \
  void batch_block_counts(const DevParams &p, int tile, long long counts[BS_COUNT]);            \
  hipError_t batch_step(const BatchMember *members, int nmembers, int dim, int bulk32, int tile, \
                        const long long totals[BS_COUNT], int with_cfl, hipStream_t s);         \
  }

PPK_DECLARE_KERNELS(fast)
PPK_DECLARE_KERNELS(strict)

// entry-point table of one arithmetic variant
struct KernelTable {
  decltype(&fast::staged_boundaries) boundaries;
  decltype(&fast::staged_prologue) prologue;
  decltype(&fast::staged_prim_dt) prim_dt;
  decltype(&fast::staged_begin) begin;
  decltype(&fast::staged_set_dt) set_dt;
  decltype(&fast::staged_end) end;
  decltype(&fast::staged_godunov) godunov;
  decltype(&fast::fused_godunov) fused_godunov;
  decltype(&fast::fused_cfl) fused_cfl;
  decltype(&fast::fused_half) fused_half;
  decltype(&fast::surrogate_dump) surrogate_dump;
  decltype(&fast::surrogate_dump_slots) surrogate_dump_slots;
  decltype(&fast::march_godunov) march_godunov;
  decltype(&fast::march2d_godunov) march2d_godunov;
  decltype(&fast::batch_block_counts) batch_block_counts;
  decltype(&fast::batch_step) batch_step;
};

// entry-point tables of the two arithmetic variants (capi.cpp)
extern const KernelTable kFast;
extern const KernelTable kStrict;

// The ghost fill in one pass.  The reference fills x, then y, then z ghosts over the whole
// transverse range (src/shared/BoundariesFunctors.h:534-1057, SolverBase.cpp:339-537;
// Dirichlet flips the normal velocity and normal field), so a corner or edge ghost ends with
// the value its last pass reads from a ghost the earlier passes filled: the interior cell
// reached by mapping each of its ghost coordinates, times the product of the directions'
// Dirichlet signs (exact, each sign is +-1).  ghost_shell_element computes that composition
// directly: the same values, one write per ghost cell (copy, optional: a second state that
// receives the same ghost values, the single-pass step's output whose ghosts are the
// reference's U2 = U copy of the filled input).
// source coordinate of c in [0, n + 2 gw) along one direction; flip: a Dirichlet face mapped it
template <class P>
PPK_HD int ghost_src(const P &p, int d, int c, bool &flip) {
  const int gw = p.gw, n = d == 0 ? p.nx : (d == 1 ? p.ny : p.nz);
  flip = false;
  if (c >= gw && c < n + gw) return c;
  const bool upper = c >= n + gw;
  const int bc = p.bc[2 * d + (upper ? 1 : 0)];
  if (bc == PPK_BC_DIRICHLET) {
    flip = true;
    return upper ? 2 * n + 2 * gw - 1 - c : 2 * gw - 1 - c;
  }
  if (bc == PPK_BC_NEUMANN) return upper ? n + gw - 1 : gw;
  return upper ? c - n : n + c;
}
// ghost cells of the padded box: the 2 gw z planes (3D), then per interior plane the 2 gw y
// rows, then per interior row the 2 gw x cells
template <class P>
PPK_HD long long ghost_shell_cells(const P &p) {
  const long long gw2 = 2LL * p.gw, kin = p.dim == 3 ? p.nz : 1;
  return (p.dim == 3 ? gw2 * p.jsize * p.isize : 0) + kin * gw2 * p.isize + kin * p.ny * gw2;
}
template <int NV = 8, class P>
PPK_HD void ghost_shell_element(double *__restrict__ U, const P &p, long long cell,
                                double *__restrict__ copy) {
  // grids have at most 2^31 padded cells: 32-bit arithmetic
  const unsigned t = (unsigned)cell, gw = (unsigned)p.gw, gw2 = 2 * gw;
  const unsigned is = (unsigned)p.isize, js = (unsigned)p.jsize, ny = (unsigned)p.ny;
  const unsigned nA = p.dim == 3 ? gw2 * js * is : 0u;
  const unsigned nB = (p.dim == 3 ? (unsigned)p.nz : 1u) * gw2 * is;
  const int koff = p.dim == 3 ? p.gw : 0;
  int i, j, k;
  if (t < nA) {
    const unsigned row = t / is, kk = row / js;
    k = (int)(kk < gw ? kk : (unsigned)p.nz + kk);
    j = (int)(row - kk * js);
    i = (int)(t - row * is);
  } else if (t < nA + nB) {
    const unsigned u = t - nA, row = u / is, kk = row / gw2, jj = row - kk * gw2;
    k = (int)kk + koff;
    j = (int)(jj < gw ? jj : ny + jj);
    i = (int)(u - row * is);
  } else {
    const unsigned u = t - nA - nB, row = u / gw2, kk = row / ny, ii = u - row * gw2;
    k = (int)kk + koff;
    j = (int)(gw + (row - kk * ny));
    i = (int)(ii < gw ? ii : (unsigned)p.nx + ii);
  }
  bool fx, fy, fz = false;
  const int i0 = ghost_src(p, 0, i, fx), j0 = ghost_src(p, 1, j, fy);
  const int k0 = p.dim == 3 ? ghost_src(p, 2, k, fz) : k;
  const long long dst = ((long long)k * p.jsize + j) * p.isize + i;
  const long long src = ((long long)k0 * p.jsize + j0) * p.isize + i0;
#pragma unroll
  for (int v = 0; v < NV; ++v) {  // NV < 8: the Euler solvers, no field
    const bool neg = ((v == IU || v == IA) && fx) != (((v == IV || v == IB) && fy) !=
                                                      ((v == IW || v == IC) && fz));
    const double x = U[src + v * p.vstride] * (neg ? -1.0 : 1.0);
    U[dst + v * p.vstride] = x;
    if (copy) copy[dst + v * p.vstride] = x;
  }
}

// block-wide maximum of one double per thread (any block size that is a multiple of 64, up
// to 1024); every thread gets the result
__device__ __forceinline__ double block_max(double v, double *smem32) {
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
  const int wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if ((threadIdx.x & 63) == 0) smem32[wave] = v;
  __syncthreads();
  double m = smem32[0];
  for (int w = 1; w < nw; ++w) m = fmax(m, smem32[w]);
  __syncthreads();
  return m;
}

// ---- time-loop control, shared by the MHD and Euler steps ----------------------------------
// SolverBase::finished() (src/shared/SolverBase.cpp:195-201), if the step was asked to check
__device__ __forceinline__ bool step_wanted(const double *ctrl, int check_finished) {
  return !check_finished || !(ctrl[CTRL_T] >= (ctrl[CTRL_TEND] - 1e-14) ||
                              ctrl[CTRL_ITER] >= ctrl[CTRL_NSTEPMAX]);
}
// dt from the CFL partial maxima or the fixed value, clamped to tEnd - t,
// src/muscl/SolverMHDMuscl.h:737 and src/shared/SolverBase.cpp:173-177.  One block of NT
// threads; red: NT / 64 doubles of LDS.
template <int NT>
__device__ __forceinline__ void step_dt(double *ctrl, const double *__restrict__ parts,
                                        int nparts, double fixed_dt, int mode, double cfl,
                                        double *red) {
  if (mode == SETDT_FIXED) {
    // a fixed dt is clamped to tEnd like the CFL one (SolverBase.cpp:173-177), so a run of
    // fixed steps stops exactly at tEnd
    if (threadIdx.x == 0) {
      double dt = fixed_dt;
      if (ctrl[CTRL_T] + dt > ctrl[CTRL_TEND]) dt = ctrl[CTRL_TEND] - ctrl[CTRL_T];
      ctrl[CTRL_DT] = dt;
    }
    return;
  }
  // eight independent loads in flight per thread: the partials can number ~10^5
  double m[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  int b = threadIdx.x;
  for (; b + 7 * NT < nparts; b += 8 * NT) {
#pragma unroll
    for (int u = 0; u < 8; ++u) m[u] = fmax(m[u], parts[b + u * NT]);
  }
#pragma unroll
  for (int u = 0; u < 8; ++u)
    if (b + u * NT < nparts) m[u] = fmax(m[u], parts[b + u * NT]);
#pragma unroll
  for (int u = 1; u < 8; ++u) m[0] = fmax(m[0], m[u]);
  const double mx = block_max(m[0], red);
  if (threadIdx.x != 0) return;
  ctrl[CTRL_INVDT] = mx;
  if (mode == SETDT_CFL) {
    double dt = cfl / mx;
    if (ctrl[CTRL_T] + dt > ctrl[CTRL_TEND]) dt = ctrl[CTRL_TEND] - ctrl[CTRL_T];
    ctrl[CTRL_DT] = dt;
  }
}
// The prologue of a step in one launch: block 0 decides whether the step runs and sets its dt,
// the others fill the ghosts (they decide for themselves from t and the iteration, which no
// block of this launch writes).  Three launches (finished test, ghost fill, dt) took 14 us
// between them on grids too small to hide them, this one 6.
template <int NV, class P>
__device__ __forceinline__ void step_prologue(double *__restrict__ U, double *__restrict__ copy,
                                              const P &p, double *ctrl,
                                              const double *__restrict__ parts, int nparts,
                                              double fixed_dt, int mode, double cfl,
                                              int check_finished, double *red) {
  const bool on = step_wanted(ctrl, check_finished);
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) ctrl[CTRL_ACTIVE] = on ? 1.0 : 0.0;
    if (on && mode != SETDT_LATER) step_dt<256>(ctrl, parts, nparts, fixed_dt, mode, cfl, red);
    return;
  }
  if (!on) return;
  const long long total = ghost_shell_cells(p), stride = (long long)(gridDim.x - 1) * 256;
  for (long long t = (blockIdx.x - 1) * 256LL + threadIdx.x; t < total; t += stride)
    ghost_shell_element<NV>(U, p, t, copy);
}
inline unsigned prologue_blocks(long long ghost_cells) {
  const long long g = (ghost_cells + 255) / 256;
  return (unsigned)(1 + (g > 65536 ? 65536 : g));
}
// after a step: ++iteration; t += dt (src/shared/SolverBase.cpp:216-218), by one thread of the
// step's last kernel, whose blocks read only dt and the active flag of the control block.
// `host` (may be null): the pinned copy that the host reads after a synchronization.
__device__ __forceinline__ void step_end(double *ctrl, double *host) {
  const double it = ctrl[CTRL_ITER] + 1.0, t = ctrl[CTRL_T] + ctrl[CTRL_DT];
  ctrl[CTRL_ITER] = it;
  ctrl[CTRL_T] = t;
  if (host) {
    host[CTRL_ITER] = it;
    host[CTRL_T] = t;
    host[CTRL_DT] = ctrl[CTRL_DT];
    host[CTRL_INVDT] = ctrl[CTRL_INVDT];
  }
}

}  // namespace ppk
