// kernels_common.hip -- kernels shared by every path: step bookkeeping on the
// device, the shearing-periodic ghost fill, the periodic Z ghost copy, the
// CFL reduction and the HLLD diagnostic.
//
// Reference correspondence (INL = library/mhd_solver.inl):
//   k_ghost_y   communicate_gather_kernel_y + communicate_scatter_kernel_y
//               (INL:90-286) with relative_displacement (INL:288-295)
//   k_ghost_z   the Z halo copies of communicate() (INL:446-708)
//   k_cfl       cfl_condition_kernel (INL:714-739) + thrust::min_element
//               (INL:1111-1116), as one pass with a wave/block/grid min
//   open_step   dt clipping of proceed() (INL:1126-1137) and
//               GlobalSetup::proceed (mhd_solver.hrb:56-59)
#include "ghost_fill.h"

namespace nmhd {

// Bookkeeping as a launch of its own, for the paths whose first kernel does
// not do it.
__global__ void k_open_step(Box b, OpenStep o) { (void)open_step(b, o, true); }

__global__ void k_clear_cfl(StepRec *rec) { rec->cfl[threadIdx.x * kCflStride] = 0x7f800000u; }

void host_displacement(const Box &b, double t, float *normalized, int *n, float *minor) {
  displacement(b, t, normalized, n, minor);
}

// Z ghost planes (ghost_z_cell).
__global__ void k_ghost_z(Box b, FieldPtrs W, const StepRec *rec, int reset) {
  if (run_ended(rec->s, reset)) return;
  const long unit = (long)b.n[0] * b.n[1] * b.m[2];
  const long a = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= unit) return;
  ghost_z_cell(b, W, a);
}

// Per-cell CFL time min(goal, C*d/|v_d + sqrt((gamma p + b2)/rho)|) with
// b2 = sum_d max(B_d,lo^2, B_d,hi^2), reduced with a wave shuffle min, an LDS
// block min and one atomic min per block on the float bits of the block's
// slot (valid: all candidates are >= 0).
__device__ __forceinline__ void cfl_block_fold(float t, StepRec *rec) {
  __shared__ float red[4];
  t = wave_min64(t);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) red[wid] = t;
  __syncthreads();
  if (threadIdx.x == 0) {
    float m = red[0];
    for (int i = 1; i < (int)(blockDim.x >> 6); ++i) m = fminf(m, red[i]);
    atomicMin(cfl_slot(rec, blockIdx.x), __float_as_uint(m));
  }
}

// Y ghost rows (ghost_y_cell), one thread per ghost cell; with
// Cfl also the CFL minimum of the rows, from the values just formed.  Bound by
// latency: as two launches, each thread a lower and an upper cell and the FP64
// displacement before its loads, a shearing step took 68.4 us at 64^3 and 33.0
// at 32^3; in one, a thread per cell and the displacement read from the record
// (the launch that opens a step computes the next fill's), 63.5 and 28.9.
template <bool Cfl>
__global__ void __launch_bounds__(256) k_ghost_y(Box b, FieldPtrs W, StepRec *rec, int reset) {
  if (run_ended(rec->s, reset)) return;
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const GhostShear g = rec->shear;
  float t = __uint_as_float(0x7f800000u);
  if (i < ghost_y_count(b)) t = ghost_y_cell<Cfl>(b, W, g, i);
  if (Cfl) cfl_block_fold(t, rec);
}

// The least CFL time of the thread's cells and t; Carried: of those that a step
// hands on (a loop of its own: the test in the other one's held back its loads,
// 69 us for 160^3 against 53).
template <bool Carried>
__device__ __forceinline__ float least_cfl(const Box &b, const FieldPtrs &W, float t) {
  for (long a = (long)blockIdx.x * blockDim.x + threadIdx.x; a < b.ncell;
       a += (long)gridDim.x * blockDim.x) {
    int x, y, z;
    cell_coords(b, a, x, y, z);
    if (Carried && refilled(b, y, z)) continue;
    t = fminf(t, cell_cfl(b, W, a, x, y, z));
  }
  return t;
}

// Grid-stride over the cells with a capped grid.
__global__ void __launch_bounds__(256) k_cfl(Box b, FieldPtrs W, float goal, StepRec *rec,
                                             int reset, int carry) {
  const bool ended = run_ended(rec->s, reset);
  if (ended && !carry) return;
  cfl_block_fold(ended ? least_cfl<true>(b, W, 3.0e38f) : least_cfl<false>(b, W, goal), rec);
}

// CFL over the cells a ghost fill rewrites (ghost_cfl_cell), slab 0 or 1.
__global__ void __launch_bounds__(256) k_cfl_ghosts(Box b, FieldPtrs W, int slab, StepRec *rec,
                                                    int reset) {
  if (run_ended(rec->s, reset)) return;
  const long n = ghost_cfl_count(b, slab);
  float t = 3.0e38f;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long)gridDim.x * blockDim.x)
    t = fminf(t, ghost_cfl_cell(b, W, slab, i));
  cfl_block_fold(t, rec);
}

__global__ void k_hlld_batch(long n, float gamma, FluxIn in, FluxOut out) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float inv_gm1 = (float)(1.0 / (double)(gamma - 1.0f));
  Flux7 F = hlld(gamma, inv_gm1, in.f[0][i], in.f[1][i], in.f[2][i], in.f[3][i], in.f[4][i],
                 in.f[5][i], in.f[6][i], in.f[7][i], in.f[8][i], in.f[9][i], in.f[10][i],
                 in.f[11][i], in.f[12][i], in.f[13][i], in.f[14][i]);
  out.f[0][i] = F.rho;
  out.f[1][i] = F.mn;
  out.f[2][i] = F.mt1;
  out.f[3][i] = F.mt2;
  out.f[4][i] = F.e;
  out.f[5][i] = F.bt1;
  out.f[6][i] = F.bt2;
}

// Copy the state (used when an enqueued step is inactive: the rotation of
// the state buffers still has to carry the state forward).  A small grid
// strides over the box, so that the usual case (the step was active and the
// kernel returns at once) costs one short launch.
__global__ void k_copy_state(Box b, FieldPtrs src, FieldPtrs dst, const StepState *st) {
  if (st->active) return;
  for (long a = (long)blockIdx.x * blockDim.x + threadIdx.x; a < b.ncell;
       a += (long)gridDim.x * blockDim.x)
    for (int f = 0; f < 8; ++f) dst.f[f][a] = src.f[f][a];
}

// All eight fields of a box in one launch (blockIdx.y the field): eight
// copies one after another cost a launch each, which is what a small box's
// transfer consists of.  Vec: every pointer is 16-byte aligned.
template <bool Vec>
__global__ void __launch_bounds__(256) k_copy_fields(long n, FieldPtrs src, FieldPtrs dst) {
  const float *__restrict__ a = src.f[blockIdx.y];
  float *__restrict__ d = dst.f[blockIdx.y];
  const long i0 = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long step = (long)gridDim.x * blockDim.x;
  long done = 0;
  if (Vec) {
    const long n4 = n / 4;
    for (long i = i0; i < n4; i += step)
      reinterpret_cast<float4 *>(d)[i] = reinterpret_cast<const float4 *>(a)[i];
    done = 4 * n4;
  }
  for (long i = done + i0; i < n; i += step) d[i] = a[i];
}

__global__ void k_set_time(Box b, StepRec *rec, double t, int generation) {
  rec->cfl[threadIdx.x * kCflStride] = 0x7f800000u;
  if (threadIdx.x != 0) return;
  StepState s = {};
  s.t = s.t_next = t;
  s.generation = generation;
  s.cfl_bits = s.cfl_next_bits = 0x7f800000u;
  rec->s = s;
  rec->shear = ghost_shear(b, t);
}

// Diagnostic entry points run on their own step record: current time of the
// run, active, not finished, explicit step h.
__global__ void k_diag_prepare(StepRec *diag, const StepRec *rec, float h) {
  diag->cfl[threadIdx.x * kCflStride] = 0x7f800000u;
  if (threadIdx.x != 0) return;
  StepState d = {};
  d.t = d.t_next = committed_time(rec->s);
  d.dt = d.h = d.h_diag = h;
  d.active = 1;
  d.cfl_bits = d.cfl_next_bits = 0x7f800000u;
  diag->s = d;
  diag->shear = rec->shear;
}

// ------------------------------------------------------------- launchers

void launch_clear_cfl(hipStream_t s, StepRec *rec) {
  hipLaunchKernelGGL(k_clear_cfl, dim3(1), dim3(kCflSlots), 0, s, rec);
}
void launch_open_step(hipStream_t s, const Box &b, const OpenStep &open) {
  hipLaunchKernelGGL(k_open_step, dim3(1), dim3(64), 0, s, b, open);
}
// Blocks of a reduction kernel: one per 1024 cells, at most 512.
unsigned reduce_grid(long n) {
  const unsigned g = grid_for(n, 4 * kBlock);
  return g < 1 ? 1 : (g > 512 ? 512 : g);
}

void launch_cfl_ghosts(hipStream_t s, const Box &b, FieldPtrs W, StepRec *rec, bool reset) {
  if (b.m[1] > 0) {
    const long n = (long)b.n[0] * 2 * b.m[1] * b.n[2];
    hipLaunchKernelGGL(k_cfl_ghosts, dim3(reduce_grid(n)), dim3(kBlock), 0, s, b, W, 0, rec,
                       (int)reset);
  }
  if (b.m[2] > 0) {
    const long n = (long)b.n[0] * b.n[1] * (2 * b.m[2] + 1);
    hipLaunchKernelGGL(k_cfl_ghosts, dim3(reduce_grid(n)), dim3(kBlock), 0, s, b, W, 1, rec,
                       (int)reset);
  }
}
void launch_ghost_y(hipStream_t s, const Box &b, FieldPtrs W, const StepRec *rec, bool reset) {
  const long unit = (long)b.n[0] * 2 * b.m[1] * b.n[2];
  hipLaunchKernelGGL(k_ghost_y<false>, dim3(grid_for(unit)), dim3(kBlock), 0, s, b, W,
                     const_cast<StepRec *>(rec), (int)reset);
}
void launch_ghost_y_cfl(hipStream_t s, const Box &b, FieldPtrs W, StepRec *rec, bool reset) {
  const long unit = (long)b.n[0] * 2 * b.m[1] * b.n[2];
  hipLaunchKernelGGL(k_ghost_y<true>, dim3(grid_for(unit)), dim3(kBlock), 0, s, b, W, rec,
                     (int)reset);
}
void launch_ghost_z(hipStream_t s, const Box &b, FieldPtrs W, const StepRec *rec, bool reset) {
  const long unit = (long)b.n[0] * b.n[1] * b.m[2];
  hipLaunchKernelGGL(k_ghost_z, dim3(grid_for(unit)), dim3(kBlock), 0, s, b, W, rec, (int)reset);
}
void launch_cfl(hipStream_t s, const Box &b, FieldPtrs W, float goal, StepRec *rec, bool reset,
                bool carry) {
  hipLaunchKernelGGL(k_cfl, dim3(reduce_grid(b.ncell)), dim3(kBlock), 0, s, b, W, goal, rec,
                     (int)reset, (int)carry);
}
void launch_copy_state(hipStream_t s, const Box &b, FieldPtrs src, FieldPtrs dst,
                       const StepState *st) {
  const unsigned g = grid_for(b.ncell);
  hipLaunchKernelGGL(k_copy_state, dim3(g < 2048 ? g : 2048), dim3(kBlock), 0, s, b, src, dst,
                     st);
}
void launch_copy_fields(hipStream_t s, long ncell, const FieldPtrs &src, const FieldPtrs &dst) {
  bool vec = true;
  for (int f = 0; f < 8; ++f)
    vec = vec && ((uintptr_t)src.f[f] | (uintptr_t)dst.f[f]) % sizeof(float4) == 0;
  const unsigned g = grid_for(ncell, 4 * kBlock);
  const dim3 grid(g < 1024 ? g : 1024, 8);
  if (vec)
    hipLaunchKernelGGL(k_copy_fields<true>, grid, dim3(kBlock), 0, s, ncell, src, dst);
  else
    hipLaunchKernelGGL(k_copy_fields<false>, grid, dim3(kBlock), 0, s, ncell, src, dst);
}
void launch_set_time(hipStream_t s, const Box &b, StepRec *rec, double t, int generation) {
  hipLaunchKernelGGL(k_set_time, dim3(1), dim3(kCflSlots), 0, s, b, rec, t, generation);
}
void launch_hlld_batch(hipStream_t s, long n, float gamma, bool strict, FluxIn in,
                       FluxOut out) {
  if (strict)
    launch_hlld_batch_strict(s, n, gamma, in, out);
  else
    hipLaunchKernelGGL(k_hlld_batch, dim3(grid_for(n)), dim3(kBlock), 0, s, n, gamma, in, out);
}
void launch_diag_prepare(hipStream_t s, StepRec *diag, const StepRec *rec, float h) {
  hipLaunchKernelGGL(k_diag_prepare, dim3(1), dim3(kCflSlots), 0, s, diag, rec, h);
}

}  // namespace nmhd
