// kernels_direct.hip -- the face fluxes of a box too small to fill the chip
// with marching tiles: one thread per face, no march, no staging, no barrier.
//
//  k_direct_faces   the seven fluxes of one face per thread, three threads
//                   per cell (x, y and z), into the stage's 21 flux arrays
//
// The tiled march solves three or four Riemann problems one after another per
// plane (3.8 us a plane whatever the box), so a box with few tiles is bound
// by that chain.  Here every face has its own thread and all its loads are in
// flight at once; the stencils come from L1 and L2, and the launch is bound by
// VALU issue from about 50^3 cells on.  It writes 21 arrays instead of the
// march's 11 (the update then differences the hydro fluxes), which a box this
// size does into the caches.  The arithmetic of a face is that of the tiles,
// expression by expression, so the two give the same bits.
//
// Reference correspondence: as tiled_tiles.h.
#include "tiled_tiles.h"

namespace nmhd {
namespace direct {

using tiled::at_byte;
using tiled::recon;
using tiled::recon_bsum;

constexpr int kThreads = 256;

// What a launch does with its step: opens it, follows the launch that did, or
// takes one of a given size.
enum Role { kFrozen, kOpens, kFollows };

// i (in [-2, n]) brought into [0, n)
__device__ __forceinline__ int wrap1(int i, int n) {
  const int j = i < 0 ? i + n : (i >= n ? i - n : i);
  return n == 1 ? 0 : j;
}

// One face per thread, the lower D-face of cell (x, y, z), and nothing of it
// (but the opening of the step) with skip, the step not being taken.  The loads
// come first: the size of the step is waited for with them, not before them.
template <int D, int Recon, int Role>
__device__ __forceinline__ void one_face(const Box &b, const FieldPtrs &W, const FluxOut &F,
                                         const StageStep &ss, const OpenStep &open, bool skip, int x,
                                         int y, int z, bool valid, float *hs) {
  constexpr int D1 = (D + 1) % 3, D2 = (D + 2) % 3;
  // byte offsets of the stencil cells c-2..c+1 along D, and of their upper
  // neighbours along the two transverse axes
  unsigned s[4], s1[4], s2[4];
  const unsigned row = b.n[0] * 4u, plane = row * (unsigned)b.n[1];
  const unsigned stride[3] = {4u, row, plane};
  auto at = [&](int d, int i) { return (unsigned)wrap1(i, b.n[d]) * stride[d]; };
  const int v[3] = {x, y, z};
  const unsigned o1 = v[D1] * stride[D1], o2 = v[D2] * stride[D2];
  const unsigned p1 = at(D1, v[D1] + 1), p2 = at(D2, v[D2] + 1);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const unsigned od = at(D, v[D] + k - 2);
    s[k] = od + (o1 + o2);
    s1[k] = od + (p1 + o2);
    s2[k] = od + (o1 + p2);
  }
  // the stencil of rho, v (normal first) and p, and the sums of the two
  // transverse B on the stencil cells' faces
  float q[5][4], e1[4], e2[4];
  auto ld = [&](int f, unsigned o) { return *at_byte((const float *)W.f[f], o); };
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    q[0][k] = ld(0, s[k]);
    q[1][k] = ld(1 + D, s[k]);
    q[2][k] = ld(1 + D1, s[k]);
    q[3][k] = ld(1 + D2, s[k]);
    q[4][k] = ld(4, s[k]);
    e1[k] = ld(5 + D1, s[k]) + ld(5 + D1, s1[k]);
    e2[k] = ld(5 + D2, s[k]) + ld(5 + D2, s2[k]);
  }
  const float bn = ld(5 + D, s[2]);
  float h = 0.0f;
  if (skip) {
    if (Role == kOpens && blockIdx.x == 0 && threadIdx.x < 64) (void)open_step(b, open, true);
    return;
  }
  if (Role == kOpens || (Role == kFrozen && open.in)) {
    // the launch that opens the step: only the face predictor needs its size,
    // so without a source term only the first wave forms it
    const bool src = D != 2 && b.source == 1;
    if (threadIdx.x < 64 && (src || blockIdx.x == 0)) {
      const StepState s = open_step(b, open, blockIdx.x == 0);
      if (threadIdx.x == 0) *hs = tiled::opened_size(s, ss.hsel);
    }
    if (src) {
      __syncthreads();
      h = *hs;
    }
  } else {
    if (Role == kFrozen && !tiled::stage_active(ss)) return;
    h = tiled::stage_size(ss);
  }
  float L[7], R[7];
  recon(Recon, q[0][0], q[0][1], q[0][2], q[0][3], L[0], R[0]);
  recon(Recon, q[1][0], q[1][1], q[1][2], q[1][3], L[1], R[1]);
  recon(Recon, q[2][0], q[2][1], q[2][2], q[2][3], L[2], R[2]);
  recon(Recon, q[3][0], q[3][1], q[3][2], q[3][3], L[3], R[3]);
  recon(Recon, q[4][0], q[4][1], q[4][2], q[4][3], L[4], R[4]);
  recon_bsum(Recon, e1[0], e1[1], e1[2], e1[3], L[5], R[5]);
  recon_bsum(Recon, e2[0], e2[1], e2[2], e2[3], L[6], R[6]);
  if (D != 2 && b.source == 1) {
    // the other in-plane velocity: v_y on an x-face, v_x on a y-face
    constexpr int o = D == 0 ? 2 : 3;
    const float va = 0.5f * (q[o][1] + q[o][2]);
    const float mbv = 0.5f * h * (D == 0 ? accel_x(b, va) : accel_y_face(b, va, y));
    L[1] += mbv;
    R[1] += mbv;
  }
  const Flux7 r = hlld(b.gamma, b.inv_gm1, bn, L[0], R[0], L[1], R[1], L[2], R[2], L[3], R[3],
                       L[4], R[4], L[5], R[5], L[6], R[6]);
  if (!valid) return;
  const unsigned o = (unsigned)((z * b.n[1] + y) * b.n[0] + x) * 4u;
  *at_byte(F.f[0], o) = r.rho;
  *at_byte(F.f[1 + D], o) = r.mn;
  *at_byte(F.f[1 + D1], o) = r.mt1;
  *at_byte(F.f[1 + D2], o) = r.mt2;
  *at_byte(F.f[4], o) = r.e;
  *at_byte(F.f[5], o) = r.bt1;
  *at_byte(F.f[6], o) = r.bt2;
}

// Consecutive workgroups take the three directions of the same cells, and
// each XCD a contiguous range of cells; a wave takes 64 cells in a row of the
// arrays (patches of narrower rows, which would spare the division below,
// touch more cache lines per load: 98 us against 50 at 130x109x75).  Threads
// past the last cell work on it and store nothing (a whole wave opens the
// step).
//
// The launches of a step that may not be taken (past the end of a run) find that
// out first and then do nothing: a run to a goal 4.5 steps away, whose other 27
// steps are such, takes 668 us at 64^3 and 1285 at 90^3, against 958 and 1945
// where they solved their first faces and loaded for the others.  One
// instantiation for all roles cost steps taken 1.4% at 64^3, these nothing.
// kFrozen keeps the branch on open.in though its launches open nothing: without
// it the compiler gives it 53 VGPRs instead of 73, and 30 frozen steps of 92^3
// take 3055 us against 3000.
template <int Recon, int Role>
__global__ void __launch_bounds__(kThreads)
    k_direct_faces(Box b, FieldPtrs W, FluxSet F, StageStep ss, OpenStep open) {
  __shared__ float hs;
  const bool skip = Role == kOpens     ? run_ended(open.in->s, open.reset)
                    : Role == kFollows ? !tiled::stage_active(ss)
                                       : false;
  const unsigned lb = xcd_logical_block(blockIdx.x, gridDim.x);
  const unsigned group = lb / 3, dir = lb - 3 * group;
  const unsigned i = group * kThreads + threadIdx.x, last = (unsigned)b.ncell - 1;
  const bool valid = i <= last;
  int x, y, z;
  cell_coords(b, valid ? i : last, x, y, z);
  if (dir == 0)
    one_face<0, Recon, Role>(b, W, F.dir[0], ss, open, skip, x, y, z, valid, &hs);
  else if (dir == 1)
    one_face<1, Recon, Role>(b, W, F.dir[1], ss, open, skip, x, y, z, valid, &hs);
  else
    one_face<2, Recon, Role>(b, W, F.dir[2], ss, open, skip, x, y, z, valid, &hs);
}

}  // namespace direct

// Up to 850,000 cells.  Step times, direct faces against the march: 32^3 26.0 /
// 33.7 us, 64^3 47.0 / 54.2, 75^3 69.7 / 79.6, 80^3 80.3 / 87.1, 90^3 103 / 116,
// 100x100x60 85 / 111, 64x64x192 (which the tiles fit) 96.4 / 101.2, shearing
// 64x64x150 98.9 / 108.4, first-order 64x64x192 90.4 / 96.2.  Past that the
// update's ten more arrays cost flat boxes that the tiles fit more than the
// tiles' prologues: 256x256x14 (0.92M) 121 / 118, 512x64x30 (0.98M) 125 / 118,
// 128x128x64 122.5 / 121.6, though ragged ones gain to 1.4M (112^3 167 / 178).
bool direct_stage(const Box &b) { return b.ncell <= 850000; }

void launch_direct_faces(hipStream_t s, const Box &b, FieldPtrs W, const FluxSet &F,
                         const StageStep &ss, const OpenStep &open) {
  const dim3 grid(3 * grid_for(b.ncell, direct::kThreads)), blk(direct::kThreads);
  auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, blk, 0, s, b, W, F, ss, open); };
  using namespace direct;
  if (open.in)
    b.recon == 1 ? go(k_direct_faces<1, kOpens>) : go(k_direct_faces<0, kOpens>);
  else if (ss.hsel == H_FIXED)
    b.recon == 1 ? go(k_direct_faces<1, kFrozen>) : go(k_direct_faces<0, kFrozen>);
  else
    b.recon == 1 ? go(k_direct_faces<1, kFollows>) : go(k_direct_faces<0, kFollows>);
}

}  // namespace nmhd
