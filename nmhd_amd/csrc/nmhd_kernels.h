// nmhd_kernels.h -- internal interface between the C ABI (capi.hip) and the
// kernel translation units.  Not installed; the public ABI is include/nmhd.h.
#pragma once

#include <functional>

#include "nmhd_device.h"

namespace nmhd {

struct FieldPtrs {
  float *f[8];  // rho, vx, vy, vz, p, Bx, By, Bz
};
struct FluxIn {
  const float *f[15];
};
struct FluxOut {
  float *f[7];
};
// Face fluxes of the three sweeps: dir[d].f[k], k = rho, m_x, m_y, m_z, E,
// B_next(d), B_prev(d) (the reference's flux buffers, INL:26-27).
struct FluxSet {
  FluxOut dir[3];
};

// Which stage step a stage kernel uses: StepState::h, ::dt or ::h_diag, or
// one given by value (StageStep::h).
enum HSel { H_HALF = 0, H_FULL = 1, H_DIAG = 2, H_FIXED = 3 };

// relative_displacement (INL:288-295) with D0 = 0 and
// relvel = -q*Omega*kLocalExtentY (application/kepler_disk_demo/
// mhd_solver.curb:46-52), in FP64 as the reference evaluates it.
__host__ __device__ inline void displacement(const Box &b, double t, float *normalized,
                                             int *n, float *minor) {
  const float relvel = -b.qshear * b.omega * b.local_ext[1];
  const double d0 = 0.0 + t * (double)relvel;
  const int fold = (int)floor(d0 / (double)b.ext[0]);
  const double d1 = d0 - (double)((float)fold * b.ext[0]);
  *normalized = (float)d1;
  *n = (int)floor(d1 / (double)b.d[0]);
  *minor = (float)(d1 / (double)b.d[0] - *n);
}

// The shear of a Y ghost fill: lower ghost row j takes the top interior row j
// shifted by +n along X, the upper ghost row the bottom interior row shifted
// by -n-1, v_X offset by -/+ relvel.  With fix_interp the shifted values are
// interpolated between the cells at +n and +n+1 (-n-1 and -n) with the gather
// kernel's weights (INL:100-110): part is the fractional displacement.
struct GhostShear {
  int n;  // |n| < nx
  float part;
};
// t: the box's committed time
__device__ __forceinline__ GhostShear ghost_shear(const Box &b, double t) {
  GhostShear g = {0, 0.0f};
  if (b.shear_y) {
    float nd;
    displacement(b, t, &nd, &g.n, &g.part);
    g.n %= b.n[0];  // same shift, and no int overflow in x + n for huge t
  }
  return g;
}

// The step record of a context with the CFL minimum of the state the step
// produces, spread over slots a cache line apart: the atomics of a few
// hundred workgroups on one word serialise (about 11 ns each, 6 us at 64^3),
// on 64 lines they do not.
constexpr int kCflSlots = 64, kCflStride = 32;
struct alignas(128) StepRec {
  StepState s;
  GhostShear shear;  // of the ghost fill that follows the step
  alignas(128) unsigned cfl[kCflSlots * kCflStride];  // float bits, +inf when empty
};
__device__ __forceinline__ unsigned *cfl_slot(StepRec *r, int block) {
  return &r->cfl[(block & (kCflSlots - 1)) * kCflStride];
}

// The step a stage kernel belongs to: its record, or (H_FIXED) a step of
// size h that is always taken.
struct StageStep {
  StepRec *rec;
  int hsel;
  float h;
};

// The bookkeeping between two steps, done by the first kernel of a step (every
// wave computes it, one writes it): commit the step in `in`, decide the next
// one from its CFL minimum, write it to `out`.  reset: `in` ends a run, start
// a new one.  in == NULL: the kernel opens no step.
struct OpenStep {
  const StepRec *in;
  StepRec *out;
  float goal;
  int reset;
};

constexpr int kBlock = 256;

inline unsigned grid_for(long n, int block = kBlock) {
  return (unsigned)((n + block - 1) / block);
}

void host_displacement(const Box &b, double t, float *normalized, int *n, float *minor);

// (x, y, z) of the cell at linear index a (x fastest), in 32-bit unsigned
// arithmetic: a box holds fewer than 2^31 cells.
__device__ __forceinline__ void cell_coords(const Box &b, long a, int &x, int &y, int &z) {
  const unsigned u = (unsigned)a, n0 = (unsigned)b.n[0], n1 = (unsigned)b.n[1];
  const unsigned row = u / n0;
  x = (int)(u - row * n0);
  z = (int)(row / n1);
  y = (int)(row - (unsigned)z * n1);
}

// ------------------------------------------------ step record transitions
// (shared by the single-box and the multi-box kernels)

// Decide the step: dt = CFL minimum, clipped so that t + dt <= goal
// (proceed(), INL:1126-1137).
__device__ __forceinline__ void step_dt(StepState &s, float goal) {
  if (s.finished) {
    s.active = 0;
    return;
  }
  float dt = fminf(goal, __uint_as_float(s.cfl_bits));
  const double next = s.t + (double)dt;
  if (next > (double)goal) {
    dt = (float)((double)goal - s.t);
    s.finished = 1;
    s.goal_reached = 1;
  }
  s.dt = dt;
  s.h = dt / 2;
  s.t_next = s.t + (double)dt;
  s.active = 1;
}

// GlobalSetup::proceed (mhd_solver.hrb:56-59)
__device__ __forceinline__ void step_commit(StepState &s) {
  if (!s.active) return;
  s.t = s.t_next;
  s.generation += 1;
  s.steps_done += 1;
  s.active = 0;
}

// The time of the state that the step in s leaves behind, and whether the
// run that it belongs to ended there.
__device__ __forceinline__ double committed_time(const StepState &s) {
  return s.active ? s.t_next : s.t;
}
__device__ __forceinline__ bool run_ended(const StepState &s, int reset) {
  return s.finished && !reset;
}

__device__ __forceinline__ float wave_min64(float v) {
  for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
  return v;
}

// OpenStep by a full wave; every wave of the launch gets the step in flight,
// the wave with `write` set records it.
__device__ __forceinline__ StepState open_step(const Box &b, const OpenStep &o, bool write) {
  const int slot = (threadIdx.x & 63) * kCflStride;
  const unsigned mine = o.in->cfl[slot];
  StepState s = o.in->s;
  step_commit(s);
  if (o.reset) s.finished = s.goal_reached = s.steps_done = 0;
  const bool ended = s.finished;
  s.cfl_bits = __float_as_uint(wave_min64(__uint_as_float(mine)));
  step_dt(s, o.goal);
  if (write) {
    o.out->cfl[slot] = ended ? mine : 0x7f800000u;
    const GhostShear g = ghost_shear(b, committed_time(s));
    if ((threadIdx.x & 63) == 0) {
      o.out->s = s;
      o.out->shear = g;
    }
  }
  return s;
}

// CFL time of one cell (cfl_condition_inner, INL:714-720):
// min_d C*d_d/|v_d + sqrt((gamma p + b2)/rho)|, b2 = sum_d max(B_lo^2, B_hi^2)
// (|v_d| + sqrt(..) with fix_cfl), without FMA contraction so that every CFL
// pass rounds the same way.  w: rho, v, p; lo, hi: the six face fields.
__device__ __forceinline__ float cfl_time(const Box &b, const float (&w)[5], const float (&lo)[3],
                                          const float (&hi)[3]) {
#pragma clang fp contract(off)
  const float b2 = fmaxf(lo[0] * lo[0], hi[0] * hi[0]) + fmaxf(lo[1] * lo[1], hi[1] * hi[1]) +
                   fmaxf(lo[2] * lo[2], hi[2] * hi[2]);
  const float c = sqrtf((b.gamma * w[4] + b2) / w[0]);
  float t = 3.0e38f;
  for (int d = 0; d < 3; ++d) t = fminf(t, b.cfl * b.d[d] / cfl_speed(b, w[1 + d], c));
  return t;
}

// Whether a ghost fill changes the CFL time of a cell of row y, plane z: it
// rewrites the ghost cells, and the upper B_z face of the last interior plane.
// The minimum that a step carries to the next leaves these cells out.
__device__ __forceinline__ bool refilled(const Box &b, int y, int z) {
  return y < b.m[1] || y >= b.n[1] - b.m[1] ||
         (b.m[2] > 0 && (z < b.m[2] || z >= b.n[2] - b.m[2] - 1));
}

__device__ __forceinline__ float cell_cfl(const Box &b, const FieldPtrs &W, long a, int x, int y,
                                          int z) {
  const float w[5] = {W.f[0][a], W.f[1][a], W.f[2][a], W.f[3][a], W.f[4][a]};
  const float lo[3] = {W.f[5][a], W.f[6][a], W.f[7][a]};
  const float hi[3] = {W.f[5][addr(b, wrap(x + 1, b.n[0]), y, z)],
                       W.f[6][addr(b, x, wrap(y + 1, b.n[1]), z)],
                       W.f[7][addr(b, x, y, wrap(z + 1, b.n[2]))]};
  return cfl_time(b, w, lo, hi);
}

// ------------------------------------------------------- multi-box batches

// One box of a batch: its parameters and the offsets (in floats) of its
// 8 state fields and 21 face-flux arrays in the batch's pools.
struct BatchBox {
  Box b;
  long off8;
  long off21;
};

__host__ __device__ inline FieldPtrs box_fields(float *pool, const BatchBox &bb) {
  FieldPtrs p;
  for (int f = 0; f < 8; ++f) p.f[f] = pool + bb.off8 + (long)f * bb.b.ncell;
  return p;
}

__host__ __device__ inline FluxSet box_fluxes(float *pool, const BatchBox &bb) {
  FluxSet F;
  for (int d = 0; d < 3; ++d)
    for (int k = 0; k < 7; ++k) F.dir[d].f[k] = pool + bb.off21 + (long)(d * 7 + k) * bb.b.ncell;
  return F;
}

// One tile of a batch launch: box, tile origin, z range, tile shape.
struct WorkItem {
  int box;
  int xy;       // x0 | y0 << 16
  int z;        // z0 | zend << 16
  int variant;  // TileVariant
};

// Tile shapes of the z-marching kernels (TX x TY, 256 threads each).
enum TileVariant { TV_64x4 = 0, TV_32x8 = 1, TV_16x16 = 2, TV_COUNT = 3 };
constexpr int kTileAuto = -1;  // NMHD_TILE_AUTO: kernel and tile shape by the box
constexpr int kTileTX[TV_COUNT] = {64, 32, 16};
constexpr int kTileTY[TV_COUNT] = {4, 8, 16};

// kernels_common.hip
// empty the CFL minimum of rec before a full pass
void launch_clear_cfl(hipStream_t s, StepRec *rec);
void launch_open_step(hipStream_t s, const Box &b, const OpenStep &open);
// the ghost fills and CFL passes of the step that follows rec's
void launch_cfl_ghosts(hipStream_t s, const Box &b, FieldPtrs W, StepRec *rec, bool reset);
void launch_ghost_y(hipStream_t s, const Box &b, FieldPtrs W, const StepRec *rec, bool reset);
// the Y fill and the CFL minimum of the rows it writes (boxes without Z ghosts)
void launch_ghost_y_cfl(hipStream_t s, const Box &b, FieldPtrs W, StepRec *rec, bool reset);
void launch_ghost_z(hipStream_t s, const Box &b, FieldPtrs W, const StepRec *rec, bool reset);
// the full pass; for a step that is not taken (the run that rec ends is
// finished and goes on) it does nothing, or with carry it leaves the minimum
// that the step is to hand on: without the cells that the next fill rewrites
// and without the goal
void launch_cfl(hipStream_t s, const Box &b, FieldPtrs W, float goal, StepRec *rec, bool reset,
                bool carry = false);
void launch_copy_state(hipStream_t s, const Box &b, FieldPtrs src, FieldPtrs dst,
                       const StepState *st);
void launch_copy_fields(hipStream_t s, long ncell, const FieldPtrs &src, const FieldPtrs &dst);
void launch_set_time(hipStream_t s, const Box &b, StepRec *rec, double t, int generation);
void launch_hlld_batch(hipStream_t s, long n, float gamma, bool strict, FluxIn in,
                       FluxOut out);
void launch_diag_prepare(hipStream_t s, StepRec *diag, const StepRec *rec, float h);

// kernels_unfused.hip (fast arithmetic) and kernels_strict.hip (reference
// rounding, bit-exact against the CPU oracle)
void launch_flux_strict(hipStream_t s, int dir, const Box &b, FieldPtrs W, FluxOut F,
                        const StepState *st, int hsel);
void launch_update_strict(hipStream_t s, const Box &b, FieldPtrs Win, const FluxSet &F,
                          FieldPtrs Wbase, FieldPtrs Wout, const StepState *st, int hsel,
                          bool pace_only);
void launch_hlld_batch_strict(hipStream_t s, long n, float gamma, FluxIn in, FluxOut out);
void launch_flux(hipStream_t s, int dir, const Box &b, FieldPtrs W, FluxOut F,
                 const StepState *st, int hsel);
void launch_update(hipStream_t s, const Box &b, FieldPtrs Win, const FluxSet &F,
                   FieldPtrs Wbase, FieldPtrs Wout, const StepState *st, int hsel,
                   bool pace_only);

// The step a stage launch over a batch belongs to.  rec[box] is its record,
// whose cfl_next_bits collects the CFL minimum of the state it produces.  The
// step's first launch opens it from the records `in` of the step before (open_step's
// transitions, per box; *goal in device memory, so that a captured step serves
// any); in == NULL: the launch opens no step.
struct BatchStep {
  StepState *rec;
  const StepState *in;
  const float *goal;
  int hsel;
};

// kernels_batch.hip (multi-box launches over a work table)
void launch_batch_cfl(hipStream_t s, const BatchBox *boxes, int nbox, float *state, float goal,
                      StepState *rec);
// ghost fills of the step that follows rec's, and their CFL minimum, for the
// boxes with ghost layers (grid blocks per box, blockIdx.y the box; boxes
// without return at once)
void launch_batch_ghost_y(hipStream_t s, const BatchBox *boxes, int nbox, int grid, float *state,
                          const StepState *rec);
void launch_batch_ghost_z(hipStream_t s, const BatchBox *boxes, int nbox, int grid, float *state,
                          const StepState *rec);
void launch_batch_cfl_ghosts(hipStream_t s, const BatchBox *boxes, int nbox, int grid,
                             float *state, StepState *rec);
// grid: workgroups that walk the table, 0: one per item.  wide: items of
// 64x4 tiles among them; nt: streamed() of all boxes together
void launch_batch_faces(hipStream_t s, int grid, const BatchBox *boxes, const WorkItem *items,
                        int nitems, float *state, float *flux, const BatchStep &step, bool wide,
                        bool nt);
void launch_batch_update(hipStream_t s, int grid, const BatchBox *boxes, const WorkItem *items,
                         int nitems, float *state_in, float *flux, float *state_base,
                         float *state_out, const BatchStep &step, bool cfl,
                         bool nt);

// kernels_diag.hip (run diagnostics: 12 FP64 values, see k_diag_partial)
constexpr int kDiagVals = 12;
int diag_blocks(const Box &b);
void launch_diag(hipStream_t s, const Box &b, FieldPtrs W, double *part, double *out);

// kernels_adjoint.hip (reverse of one RK stage of the periodic step)
struct AdjStageArgs {
  FieldPtrs Win, Wbase, Wout;  // stage input, conserved base, stage output
  FieldPtrs lam_out;           // dL/dW_out
  FieldPtrs lam_base;          // dL/dW_base (written, or added to with acc_base)
  FieldPtrs lam_in;            // dL/dW_in through P (written, or added to with acc_in)
  float h;
  bool acc_base, acc_in;
  // work arrays (ncell floats each); face: 15 per direction, the adjoints
  // of a face's left and right states (7 + 7) and its limiter branches
  // (one 32-bit word per face)
  float *gU[5], *lE[3], *lbb[3], *abn[3], *face[45];
};
void launch_adj_stage(hipStream_t s, const Box &b, const AdjStageArgs &A);

// kernels_tiny.hip (a whole stage of a very small box in one launch; it may
// not both open a step and reduce its CFL minimum, as the record is emptied
// by the launch that opens it)
bool tiny_stage(const Box &b);
void launch_tiny_stage(hipStream_t s, const Box &b, FieldPtrs Win, FieldPtrs Wbase, FieldPtrs Wout,
                       const StageStep &ss, const OpenStep &open, bool cfl);

// kernels_direct.hip (the stage of a small box: a thread per face, a thread
// per cell; all 21 flux arrays are used)
bool direct_stage(const Box &b);
void launch_direct_faces(hipStream_t s, const Box &b, FieldPtrs W, const FluxSet &F,
                         const StageStep &ss, const OpenStep &open);

// kernels_tiled.hip
// Planes per march of the face or update kernel: the chunk of the least
// estimated time, groups_at(zc) the workgroups of the launch with chunks of zc,
// per_cu how many of them a CU holds (march_per_cu).
// whether the stage kernels over that many cells store past the caches
bool streamed(long cells);
int march_chunk(bool faces, int nz, int per_cu, const std::function<long(int)> &groups_at);
int march_per_cu(bool faces, bool wide);  // wide: 64x4 tiles in the launch
// Tile shape (TileVariant) of the face or update kernel for a box.
int tiled_shape(int nx, int ny, bool faces);
// tile: TileVariant of the z-marching tiles, or kTileAuto (both launches of a
// stage then take the same route, direct_stage)
// open: the bookkeeping of the step that this launch begins (in == NULL: none)
void launch_faces(hipStream_t s, const Box &b, FieldPtrs W, const FluxSet &F, const StageStep &ss,
                  const OpenStep &open = {}, int tile = kTileAuto);
void launch_update_tiled(hipStream_t s, const Box &b, FieldPtrs Win, const FluxSet &F,
                         FieldPtrs Wbase, FieldPtrs Wout, const StageStep &ss, bool pace_only,
                         bool cfl, int tile = kTileAuto);

}  // namespace nmhd
