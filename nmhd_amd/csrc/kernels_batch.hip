// kernels_batch.hip -- many independent boxes of uneven sizes
// advanced together.  Each RK stage runs the face fluxes, then the update,
// over a work table of tiles from every box, one launch each with a workgroup
// per work item (or, on request, a few workgroups per CU that walk the table);
// a tile's box record gives its sizes, its per-box step (own dt) and the
// offsets of its fields in the batch's pools.  The tile functions are the
// single-box path's (tiled_tiles.h), so a box advanced in a batch is
// bit-identical to the same box advanced alone.  As there, the bookkeeping
// between two steps is done by the first face launch, and an inactive box is
// carried along by the last update; boxes with ghost layers
// (the shearing box) are filled, and their ghost cells' CFL reduced, by
// per-box grids over the single-box cell functions (ghost_fill.h).
//
// Bound by the march's latency and issue as a single box of as many cells
// (faces 45 us, update 37 us a stage for 14 boxes of 16..96 cells per edge,
// 1.02M cells).  One launch per tile shape on streams side by side, with
// launches of their own for the bookkeeping and for the copy of inactive
// boxes, made a step a graph of 14 nodes with forks and joins: 193 us there at
// the same chunks, against 163 in four.
//
// The reference advances one compile-time-sized box per process and has no
// counterpart of this path; its per-box arithmetic is that of proceed()
// (library/mhd_solver.inl:1086-1204).
#include "ghost_fill.h"
#include "tiled_tiles.h"

namespace nmhd {

namespace {

constexpr int cmax(int a, int b) { return a > b ? a : b; }
template <bool Wide>
constexpr int kFacesLds = cmax(Wide ? tiled::FacesShape<64, 4>::kLds : 0,
                               cmax(tiled::FacesShape<32, 8>::kLds,
                                    tiled::FacesShape<16, 16>::kLds));
constexpr int kUpdateLds =
    cmax(cmax(tiled::UpdateShape<64, 4>::kLds, tiled::UpdateShape<32, 8>::kLds),
         tiled::UpdateShape<16, 16>::kLds);

__device__ __forceinline__ void item_tile(const WorkItem &w, int &x0, int &y0, int &z0,
                                          int &zend) {
  x0 = w.xy & 0xffff;
  y0 = (w.xy >> 16) & 0xffff;
  z0 = w.z & 0xffff;
  zend = (w.z >> 16) & 0xffff;
}

// The step that a launch opens for a box.
__device__ __forceinline__ StepState batch_open(const BatchStep &step, int box) {
  StepState s = step.in[box];
  step_commit(s);
  if (!s.finished) {
    s.cfl_bits = s.cfl_next_bits;
    s.cfl_next_bits = 0x7f800000u;  // +inf
  }
  step_dt(s, *step.goal);
  return s;
}

// The stage step of a box; false: the box takes no step.
__device__ __forceinline__ bool batch_begin(const BatchStep &step, int box, float &h) {
  if (step.in) {
    const StepState s = batch_open(step, box);
    h = __uint_as_float(
        __builtin_amdgcn_readfirstlane(__float_as_uint(tiled::opened_size(s, step.hsel))));
    return __builtin_amdgcn_readfirstlane(s.active);
  }
  const StepState *s = step.rec + box;
  h = tiled::stage_h(s, step.hsel);
  return s->active;
}

template <bool Wide, bool Nt>
__device__ __forceinline__ void faces_item(const BatchBox *boxes, const WorkItem &w, float *state,
                                           float *flux, const BatchStep &step, float *lds) {
  float h;
  const bool active = batch_begin(step, w.box, h);
  const BatchBox bb = boxes[w.box];
  const FieldPtrs W = box_fields(state, bb);
  const FluxSet F = box_fluxes(flux, bb);
  int x0, y0, z0, zend;
  item_tile(w, x0, y0, z0, zend);
  if (!active)
    ;
  else if (Wide && w.variant == TV_64x4)
    tiled::faces_tile_any<64, 4, Nt>(bb.b, W, F, h, x0, y0, z0, zend, lds);
  else if (w.variant == TV_32x8)
    tiled::faces_tile_any<32, 8, Nt>(bb.b, W, F, h, x0, y0, z0, zend, lds);
  else
    tiled::faces_tile_any<16, 16, Nt>(bb.b, W, F, h, x0, y0, z0, zend, lds);
  // the box's first item records the step it opened (after the tile: a store
  // before it would keep the box's parameters out of scalar registers)
  if (step.in && w.xy == 0 && z0 == 0 && threadIdx.x == 0) step.rec[w.box] = batch_open(step, w.box);
}

// A workgroup per item.  64x4 tiles need more registers and LDS than the other
// two shapes, of which four workgroups fit a CU: tables without them take the
// narrow instantiation.
template <bool Wide, bool Nt>
__global__ void __launch_bounds__(tiled::kTileThreads, Wide ? 3 : 4)
    k_batch_faces_items(const BatchBox *boxes, const WorkItem *items, float *state, float *flux,
                        BatchStep step) {
  __shared__ float lds[kFacesLds<Wide>];
  faces_item<Wide, Nt>(boxes, items[xcd_logical_block(blockIdx.x, gridDim.x)], state, flux, step,
                       lds);
}

// Workgroups that walk the table.  Nt by the rule of the others: 14 boxes of
// 1.02M cells, 4 workgroups per CU, 186 us a step past the caches against 169
// through them, 24 of 1.78M 314 / 282.
template <bool Nt>
__global__ void __launch_bounds__(tiled::kTileThreads)
    k_batch_faces(const BatchBox *boxes, const WorkItem *items, int nitems, float *state,
                  float *flux, BatchStep step) {
  __shared__ float lds[kFacesLds<true>];
  const int G = gridDim.x;
  for (int it = xcd_logical_block(blockIdx.x, G); it < nitems; it += G) {
    faces_item<true, Nt>(boxes, items[it], state, flux, step, lds);
    __syncthreads();  // the next tile's shape lays the LDS out anew
  }
}

template <int TX, int TY, bool Cfl, bool Nt>
__device__ __forceinline__ void update_tile_of(const Box &b, const WorkItem &w, bool active,
                                               const FieldPtrs &Win, const FluxSet &F,
                                               const FieldPtrs &Wb, const FieldPtrs &Wo, float h,
                                               float *lds, float &cfl_t) {
  int x0, y0, z0, zend;
  item_tile(w, x0, y0, z0, zend);
  if (active) {
    tiled::update_tile<TX, TY, false, Cfl, false, Nt>(b, Win, F, Wb, Wo, h, x0, y0, z0, zend, lds,
                                                      cfl_t);
    return;
  }
  // a box that takes no step: the last stage's output carries its state
  // through the buffer rotation
  const int x = x0 + (int)threadIdx.x % TX, y = y0 + (int)threadIdx.x / TX;
  if (Cfl && x < b.n[0] && y < b.n[1])
    for (int r = z0; r < zend; ++r) {
      const long a = ((long)r * b.n[1] + y) * b.n[0] + x;
      for (int f = 0; f < 8; ++f) Wo.f[f][a] = Wb.f[f][a];
    }
}

template <bool Cfl, bool Nt>
__device__ __forceinline__ void update_item(const BatchBox *boxes, const WorkItem &w,
                                            float *state_in, float *flux, float *state_base,
                                            float *state_out, const BatchStep &step, float *lds,
                                            float *red) {
  float h;
  const bool active = batch_begin(step, w.box, h);
  if (!Cfl && !active) return;
  const BatchBox bb = boxes[w.box];
  const FieldPtrs Win = box_fields(state_in, bb), Wb = box_fields(state_base, bb);
  const FieldPtrs Wo = box_fields(state_out, bb);
  const FluxSet F = box_fluxes(flux, bb);
  float cfl_t = 3.0e38f;
  if (w.variant == TV_64x4)
    update_tile_of<64, 4, Cfl, Nt>(bb.b, w, active, Win, F, Wb, Wo, h, lds, cfl_t);
  else if (w.variant == TV_32x8)
    update_tile_of<32, 8, Cfl, Nt>(bb.b, w, active, Win, F, Wb, Wo, h, lds, cfl_t);
  else
    update_tile_of<16, 16, Cfl, Nt>(bb.b, w, active, Win, F, Wb, Wo, h, lds, cfl_t);
  if (Cfl && active) tiled::block_min_into(cfl_t, &step.rec[w.box].cfl_next_bits, red);
}

template <bool Cfl, bool Nt>
__global__ void __launch_bounds__(tiled::kTileThreads, 4)
    k_batch_update_items(const BatchBox *boxes, const WorkItem *items, float *state_in,
                         float *flux, float *state_base, float *state_out, BatchStep step) {
  __shared__ float lds[kUpdateLds];
  __shared__ float red[4];
  update_item<Cfl, Nt>(boxes, items[xcd_logical_block(blockIdx.x, gridDim.x)], state_in, flux,
                   state_base, state_out, step, lds, red);
}

// 3 waves per SIMD (168 VGPRs; unbounded the second stage takes 172 and two):
// 64 boxes of 6.06M cells, 3 workgroups per CU, 866 us a step against 797; at 4
// waves it spills 33 and takes 903.
template <bool Cfl, bool Nt>
__global__ void __launch_bounds__(tiled::kTileThreads, 3)
    k_batch_update(const BatchBox *boxes, const WorkItem *items, int nitems, float *state_in,
                   float *flux, float *state_base, float *state_out, BatchStep step) {
  __shared__ float lds[kUpdateLds];
  __shared__ float red[4];
  const int G = gridDim.x;
  for (int it = xcd_logical_block(blockIdx.x, G); it < nitems; it += G) {
    update_item<Cfl, Nt>(boxes, items[it], state_in, flux, state_base, state_out, step, lds, red);
    __syncthreads();
  }
}

// Full CFL pass: blockIdx.y is the box, blocks stride over its cells.
__global__ void __launch_bounds__(256) k_batch_cfl(const BatchBox *boxes, float *state,
                                                   float goal, StepState *rec) {
  const int box = blockIdx.y;
  __shared__ float red[4];
  const BatchBox bb = boxes[box];
  const FieldPtrs W = box_fields(state, bb);
  const Box &b = bb.b;
  float t = goal;
  for (long a = (long)blockIdx.x * blockDim.x + threadIdx.x; a < b.ncell;
       a += (long)gridDim.x * blockDim.x) {
    int x, y, z;
    cell_coords(b, a, x, y, z);
    t = fminf(t, cell_cfl(b, W, a, x, y, z));
  }
  const float m = wave_min64(t);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    const float r = fminf(fminf(red[0], red[1]), fminf(red[2], red[3]));
    atomicMin(&rec[box].cfl_next_bits, __float_as_uint(r));
  }
}

// Ghost fills of the boxes that have ghost layers (shearing-periodic or
// periodic Y rows, periodic Z planes): blockIdx.y is the box, blocks stride
// over its slab; the cell operations are the single-box kernels'.
__global__ void k_batch_ghost_y(const BatchBox *boxes, float *state, const StepState *rec) {
  const int box = blockIdx.y;
  const BatchBox bb = boxes[box];
  if (bb.b.m[1] == 0 || rec[box].finished) return;
  const FieldPtrs W = box_fields(state, bb);
  const long unit = ghost_y_count(bb.b);
  const GhostShear g = ghost_shear(bb.b, committed_time(rec[box]));
  for (long a = (long)blockIdx.x * blockDim.x + threadIdx.x; a < unit;
       a += (long)gridDim.x * blockDim.x)
    (void)ghost_y_cell<false>(bb.b, W, g, a);
}

__global__ void k_batch_ghost_z(const BatchBox *boxes, float *state, const StepState *rec) {
  const int box = blockIdx.y;
  const BatchBox bb = boxes[box];
  if (bb.b.m[2] == 0 || rec[box].finished) return;
  const FieldPtrs W = box_fields(state, bb);
  const long unit = (long)bb.b.n[0] * bb.b.n[1] * bb.b.m[2];
  for (long a = (long)blockIdx.x * blockDim.x + threadIdx.x; a < unit;
       a += (long)gridDim.x * blockDim.x)
    ghost_z_cell(bb.b, W, a);
}

// CFL minimum over the cells the ghost fills rewrote, added to each box's
// running minimum (the stage-2 epilogue reduced the others).
__global__ void __launch_bounds__(256) k_batch_cfl_ghosts(const BatchBox *boxes, float *state,
                                                          StepState *rec) {
  const int box = blockIdx.y;
  const BatchBox bb = boxes[box];
  const long n0 = ghost_cfl_count(bb.b, 0), n1 = ghost_cfl_count(bb.b, 1);
  if ((n0 == 0 && n1 == 0) || rec[box].finished) return;
  __shared__ float red[4];
  const FieldPtrs W = box_fields(state, bb);
  float t = 3.0e38f;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n0;
       i += (long)gridDim.x * blockDim.x)
    t = fminf(t, ghost_cfl_cell(bb.b, W, 0, i));
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n1;
       i += (long)gridDim.x * blockDim.x)
    t = fminf(t, ghost_cfl_cell(bb.b, W, 1, i));
  const float m = wave_min64(t);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    const float r = fminf(fminf(red[0], red[1]), fminf(red[2], red[3]));
    atomicMin(&rec[box].cfl_next_bits, __float_as_uint(r));
  }
}

}  // namespace

void launch_batch_cfl(hipStream_t s, const BatchBox *boxes, int nbox, float *state, float goal,
                      StepState *rec) {
  hipLaunchKernelGGL(k_batch_cfl, dim3(64, nbox), dim3(256), 0, s, boxes, state, goal, rec);
}
void launch_batch_ghost_y(hipStream_t s, const BatchBox *boxes, int nbox, int grid, float *state,
                          const StepState *rec) {
  hipLaunchKernelGGL(k_batch_ghost_y, dim3(grid, nbox), dim3(256), 0, s, boxes, state, rec);
}
void launch_batch_ghost_z(hipStream_t s, const BatchBox *boxes, int nbox, int grid, float *state,
                          const StepState *rec) {
  hipLaunchKernelGGL(k_batch_ghost_z, dim3(grid, nbox), dim3(256), 0, s, boxes, state, rec);
}
void launch_batch_cfl_ghosts(hipStream_t s, const BatchBox *boxes, int nbox, int grid,
                             float *state, StepState *rec) {
  hipLaunchKernelGGL(k_batch_cfl_ghosts, dim3(grid, nbox), dim3(256), 0, s, boxes, state, rec);
}
void launch_batch_faces(hipStream_t s, int grid, const BatchBox *boxes, const WorkItem *items,
                        int nitems, float *state, float *flux, const BatchStep &step, bool wide,
                        bool nt) {
  const dim3 blk(tiled::kTileThreads);
  auto walk = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid), blk, 0, s, boxes, items, nitems, state, flux, step);
  };
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(nitems), blk, 0, s, boxes, items, state, flux, step);
  };
  if (grid)
    nt ? walk(k_batch_faces<true>) : walk(k_batch_faces<false>);
  else if (nt)
    wide ? go(k_batch_faces_items<true, true>) : go(k_batch_faces_items<false, true>);
  else
    wide ? go(k_batch_faces_items<true, false>) : go(k_batch_faces_items<false, false>);
}

template <bool Cfl>
void update_as(hipStream_t s, int grid, const BatchBox *boxes, const WorkItem *items, int nitems,
               float *state_in, float *flux, float *state_base, float *state_out,
               const BatchStep &step, bool nt) {
  const dim3 blk(tiled::kTileThreads);
  auto walk = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid), blk, 0, s, boxes, items, nitems, state_in, flux,
                       state_base, state_out, step);
  };
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(nitems), blk, 0, s, boxes, items, state_in, flux, state_base,
                       state_out, step);
  };
  if (grid)
    nt ? walk(k_batch_update<Cfl, true>) : walk(k_batch_update<Cfl, false>);
  else
    nt ? go(k_batch_update_items<Cfl, true>) : go(k_batch_update_items<Cfl, false>);
}

void launch_batch_update(hipStream_t s, int grid, const BatchBox *boxes, const WorkItem *items,
                         int nitems, float *state_in, float *flux, float *state_base,
                         float *state_out, const BatchStep &step, bool cfl, bool nt) {
  auto as = cfl ? update_as<true> : update_as<false>;
  as(s, grid, boxes, items, nitems, state_in, flux, state_base, state_out, step, nt);
}

}  // namespace nmhd
