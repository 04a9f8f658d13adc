// kernels_tiny.hip -- one RK stage of a box of a few hundred 4x4x4 tiles in a
// single launch.
//
//  k_tiny_stage   a workgroup of 512 threads stages the 8x8x8 cells around its
//                 4x4x4 tile in LDS (one cell per thread), solves the 480
//                 faces the tile needs (one per thread), upwinds its 300 edges
//                 and updates its 64 cells
//
// Such a box occupies the chip once, so a step takes as long as its launches'
// serial chains: a face launch and an update launch per stage cost their
// launch, the first loads and the write-back twice (24 us per step at 16^3 and
// at 32^3 alike).  Fused, the fluxes stay in LDS and a stage is one chain:
// load, one Riemann problem, edges, update.  The price is that a tile solves
// 480 faces for its 64 cells instead of 192, which costs nothing while the
// launch is bound by latency.  The arithmetic is that of the tiles, expression
// by expression, so the two give the same bits.
//
// Reference correspondence: as tiled_tiles.h.
#include "tiled_tiles.h"

namespace nmhd {
namespace tiny {

using tiled::recon;
using tiled::recon_bsum;
using tiled::upwind;

constexpr int T = 4;         // tile edge
constexpr int H = 8;         // staged edge: cells -2..5 of the tile
constexpr int kThreads = H * H * H;
// LDS strides of the staged cells: with planes 71 apart the 32 positions of a
// face plane, and the rows a thread group stages, fall into distinct banks in
// every direction (64 apart, the x-faces' reads would collide 8 ways)
constexpr int SY = H, SZ = 71, NS = 7 * SZ + 7 * SY + 7 + 1;
// faces per direction: 5 planes of the 32 positions (a, b) in [-1, 4]^2 with
// at most one of a, b outside the tile; B fluxes are kept on the 6x6 grid of
// positions, hydro fluxes on the tile's own 4x4
constexpr int NPOS = 32, NFACE = 5 * NPOS, NB = 5 * 36, NH = 5 * 16;
constexpr int NE = 5 * 5 * 4;  // edges of one orientation
static_assert(3 * NFACE <= kThreads && 3 * NE <= kThreads, "one face and one edge per thread");

struct Shared {
  float cell[8][NS];
  float hydro[3][5][NH];
  float b[3][2][NB];
  float edge[3][2][NE];
  float h;
  int active;
};

// LDS stride of axis d in cell[][]
__device__ __forceinline__ int stride_of(int d) { return d == 0 ? 1 : (d == 1 ? SY : SZ); }
__device__ __forceinline__ int next(int d) { return d == 2 ? 0 : d + 1; }

// i in [-2, n + 4] brought into [0, n): one wrap unless the box is tiny
__device__ __forceinline__ int into(int i, int n) {
  if (n < 5) return tiled::pmod(i, n);
  return i < 0 ? i + n : (i >= n ? i - n : i);
}

// One face of the tile: direction D, plane (0..4) along it, position (a, c)
// along the next two axes; y: the array row of the face's cell.
template <int Recon>
__device__ __forceinline__ void solve_face(const Box &b, Shared &S, int D, int plane, int pos,
                                           float h, int yrow) {
  const int D1 = next(D), D2 = next(D1);
  int a, c;  // positions 0..15 the tile's own, then the four sides
  const int side = (pos - 16) >> 2, along = pos & 3;
  if (pos < 16) {
    a = pos & 3;
    c = pos >> 2;
  } else {
    a = side == 0 ? -1 : (side == 1 ? T : along);
    c = side == 2 ? -1 : (side == 3 ? T : along);
  }
  const int sD = stride_of(D), s1 = stride_of(D1), s2 = stride_of(D2);
  const int at = (plane + 2) * sD + (a + 2) * s1 + (c + 2) * s2;
  const int i0 = at - 2 * sD, i1 = at - sD, i2 = at, i3 = at + sD;
  float L[7], R[7];
  const float *r = S.cell[0], *vn = S.cell[1 + D], *v1 = S.cell[1 + D1], *v2 = S.cell[1 + D2];
  const float *p = S.cell[4], *b1 = S.cell[5 + D1], *b2 = S.cell[5 + D2];
  recon(Recon, r[i0], r[i1], r[i2], r[i3], L[0], R[0]);
  recon(Recon, vn[i0], vn[i1], vn[i2], vn[i3], L[1], R[1]);
  recon(Recon, v1[i0], v1[i1], v1[i2], v1[i3], L[2], R[2]);
  recon(Recon, v2[i0], v2[i1], v2[i2], v2[i3], L[3], R[3]);
  recon(Recon, p[i0], p[i1], p[i2], p[i3], L[4], R[4]);
  recon_bsum(Recon, b1[i0] + b1[i0 + s1], b1[i1] + b1[i1 + s1], b1[i2] + b1[i2 + s1],
             b1[i3] + b1[i3 + s1], L[5], R[5]);
  recon_bsum(Recon, b2[i0] + b2[i0 + s2], b2[i1] + b2[i1 + s2], b2[i2] + b2[i2 + s2],
             b2[i3] + b2[i3 + s2], L[6], R[6]);
  if (b.source == 1 && D != 2) {
    const float *o = D == 0 ? S.cell[2] : S.cell[1];
    const float va = 0.5f * (o[i1] + o[i2]);
    const float mbv = 0.5f * h * (D == 0 ? accel_x(b, va) : accel_y_face(b, va, yrow));
    L[1] += mbv;
    R[1] += mbv;
  }
  const Flux7 f = hlld(b.gamma, b.inv_gm1, S.cell[5 + D][at], L[0], R[0], L[1], R[1], L[2], R[2],
                       L[3], R[3], L[4], R[4], L[5], R[5], L[6], R[6]);
  const int q = plane * 36 + (c + 1) * 6 + a + 1;
  S.b[D][0][q] = f.bt1;
  S.b[D][1][q] = f.bt2;
  if (pos < 16) {
    const int o = plane * 16 + pos;
    S.hydro[D][0][o] = f.rho;
    S.hydro[D][1 + D][o] = f.mn;
    S.hydro[D][1 + D1][o] = f.mt1;
    S.hydro[D][1 + D2][o] = f.mt2;
    S.hydro[D][4][o] = f.e;
  }
}

// B flux of the lower D-face of the tile's cell (coordinates t): component 0
// of B along the next axis, 1 along the one after
__device__ __forceinline__ float b_flux(const Shared &S, int D, int comp, const int (&t)[3]) {
  const int D1 = next(D), D2 = next(D1);
  auto get = [&](int d) { return d == 0 ? t[0] : (d == 1 ? t[1] : t[2]); };
  return S.b[D][comp][get(D) * 36 + (get(D2) + 1) * 6 + get(D1) + 1];
}

// The two sweeps' members of the edge on the lower P- and Q-faces of a cell
// (P < Q, R the edge's own axis): the P-face flux of B_Q upwinded along Q and
// the Q-face flux of B_P upwinded along P.
__device__ __forceinline__ void upwind_edge(Shared &S, int type, int i) {
  const int P = type == 2 ? 1 : 0, Q = type == 0 ? 1 : 2, R = 3 - P - Q;
  const int cP = i % 5, cQ = (i / 5) % 5, cR = i / 25;
  const int sP = stride_of(P), sQ = stride_of(Q);
  const int e = (cP + 2) * sP + (cQ + 2) * sQ + (cR + 2) * stride_of(R);
  const float *vP = S.cell[1 + P], *vQ = S.cell[1 + Q];
  const float sq = vQ[e] + vQ[e - sQ] + vQ[e - sP] + vQ[e - sP - sQ];
  const float sp = vP[e] + vP[e - sP] + vP[e - sQ] + vP[e - sP - sQ];
  auto coords = [&](int dP, int dQ, int (&t)[3]) {
    const int a = cP + dP, q = cQ + dQ;
    t[0] = P == 0 ? a : cR;               // x: P, or (type 2) the edge's axis
    t[1] = P == 1 ? a : (Q == 1 ? q : cR);
    t[2] = Q == 2 ? q : cR;
  };
  int here[3], loP[3], loQ[3];
  coords(0, 0, here);
  coords(-1, 0, loP);
  coords(0, -1, loQ);
  const int compP = Q == next(P) ? 0 : 1, compQ = P == next(Q) ? 0 : 1;
  S.edge[type][0][i] = upwind(sq, b_flux(S, P, compP, loQ), b_flux(S, P, compP, here));
  S.edge[type][1][i] = upwind(sp, b_flux(S, Q, compQ, loP), b_flux(S, Q, compQ, here));
}

template <int Recon, bool Cfl>
__global__ void __launch_bounds__(kThreads, 4)
    k_tiny_stage(Box b, FieldPtrs Win, FieldPtrs Wb, FieldPtrs Wo, StageStep ss, OpenStep open,
                 int gx, int gy) {
  __shared__ Shared S;
  const int tid = threadIdx.x;
  const int lb = xcd_logical_block(blockIdx.x, gridDim.x);
  const int x0 = lb % gx * T, y0 = lb / gx % gy * T, z0 = lb / gx / gy * T;
  const int nx = b.n[0], ny = b.n[1], nz = b.n[2];
  // the thread's staged cell
  float v[8];
  {
    const int x = into(x0 + (tid & 7) - 2, nx), y = into(y0 + (tid >> 3 & 7) - 2, ny);
    const int z = into(z0 + (tid >> 6) - 2, nz);
    const int a = (z * ny + y) * nx + x;
#pragma unroll
    for (int f = 0; f < 8; ++f) v[f] = Win.f[f][a];
  }
  // the first wave's threads update a cell each: its base values
  const int cx = tid & 3, cy = tid >> 2 & 3, cz = tid >> 4 & 3;
  const int x = x0 + cx, y = y0 + cy, z = z0 + cz;
  const bool mine = tid < 64 && x < nx && y < ny && z < nz;
  const int own = (z * ny + y) * nx + x;
  float wb[5] = {}, bb[6] = {};
  if (mine) {
#pragma unroll
    for (int f = 0; f < 5; ++f) wb[f] = Wb.f[f][own];
    bb[0] = Wb.f[5][own];
    bb[1] = Wb.f[5][(z * ny + y) * nx + wrap(x + 1, nx)];
    bb[2] = Wb.f[6][own];
    bb[3] = Wb.f[6][(z * ny + wrap(y + 1, ny)) * nx + x];
    bb[4] = Wb.f[7][own];
    bb[5] = Wb.f[7][(wrap(z + 1, nz) * ny + y) * nx + x];
  }
  if (tid < 64) {
    float h;
    const bool active = tiled::stage_begin(b, ss, open, h);
    if (tid == 0) {
      S.h = h;
      S.active = active;
    }
  }
#pragma unroll
  for (int f = 0; f < 8; ++f) S.cell[f][(tid & 7) + (tid >> 3 & 7) * SY + (tid >> 6) * SZ] = v[f];
  __syncthreads();
  if (!S.active) {
    // a step enqueued after the run reached its goal: the last stage carries
    // the state on
    if (Cfl && mine) {
      const float keep[8] = {wb[0], wb[1], wb[2], wb[3], wb[4], bb[0], bb[2], bb[4]};
#pragma unroll
      for (int f = 0; f < 8; ++f) Wo.f[f][own] = keep[f];
    }
    return;
  }
  const float h = S.h;
  if (tid < 3 * NFACE) {
    const int group = tid >> 5;  // 32 positions of one plane
    const int D = group / 5, plane = group - 5 * D;
    const int yf = y0 + plane;
    solve_face<Recon>(b, S, D, plane, tid & 31, h, yf < ny ? yf : yf - ny);
  }
  __syncthreads();
  if (tid < 3 * NE) {
    const int type = tid / NE;
    upwind_edge(S, type, tid - type * NE);
  }
  __syncthreads();
  if (tid >= 64) return;
  float cfl_t = 3.0e38f;
  if (mine) {
    float pc[5];
    const int fx = cx * 16 + cy + 4 * cz, fy = cy * 16 + cz + 4 * cx, fz = cz * 16 + cx + 4 * cy;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      float sacc = (S.hydro[0][k][fx] - S.hydro[0][k][fx + 16]) * b.inv_d[0];
      sacc += (S.hydro[1][k][fy] - S.hydro[1][k][fy + 16]) * b.inv_d[1];
      pc[k] = sacc + (S.hydro[2][k][fz] - S.hydro[2][k][fz + 16]) * b.inv_d[2];
    }
    tiled::CellEdges ce;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const int xy = cx + u + 5 * (cy + w) + 25 * cz, xz = cx + u + 5 * (cz + w) + 25 * cy;
        const int yz = cy + u + 5 * (cz + w) + 25 * cx;
        ce.XY[u][w] = S.edge[0][0][xy];
        ce.YX[u][w] = S.edge[0][1][xy];
        ce.XZ[u][w] = S.edge[1][0][xz];
        ce.ZX[u][w] = S.edge[1][1][xz];
        ce.YZ[u][w] = S.edge[2][0][yz];
        ce.ZY[u][w] = S.edge[2][1][yz];
      }
    tiled::finish_cell<false, Cfl, false>(b, ce, pc, wb, bb, h, y, z, own, Wo, cfl_t);
  }
  if (Cfl) {
    cfl_t = wave_min64(cfl_t);
    if (tid == 0) atomicMin(cfl_slot(ss.rec, blockIdx.x), __float_as_uint(cfl_t));
  }
}

}  // namespace tiny

// Up to 1024 tiles.  Step times, fused against one launch for the faces and
// one for the update: 16^3 (64 tiles) 13.5 / 24.2 us, 24^3 13.7 / 24.7, 32^3
// (512) 18.6 / 25.4, 40x36x33 (810) 25.5 / 28.2, 52x44x37 (1430) 33.1 / 29.8,
// 48^3 (1728) 35.7 / 32.8: with three workgroups on every CU the 480 solves
// per 64 cells are issue, no longer latency.
bool tiny_stage(const Box &b) {
  long tiles = 1;
  for (int d = 0; d < 3; ++d) tiles *= (b.n[d] + tiny::T - 1) / tiny::T;
  return tiles <= 1024;
}

void launch_tiny_stage(hipStream_t s, const Box &b, FieldPtrs Win, FieldPtrs Wbase, FieldPtrs Wout,
                       const StageStep &ss, const OpenStep &open, bool cfl) {
  const int gx = (b.n[0] + tiny::T - 1) / tiny::T, gy = (b.n[1] + tiny::T - 1) / tiny::T;
  const int gz = (b.n[2] + tiny::T - 1) / tiny::T;
  const dim3 grid(gx * gy * gz), blk(tiny::kThreads);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, blk, 0, s, b, Win, Wbase, Wout, ss, open, gx, gy);
  };
  if (b.recon == 1)
    cfl ? go(tiny::k_tiny_stage<1, true>) : go(tiny::k_tiny_stage<1, false>);
  else
    cfl ? go(tiny::k_tiny_stage<0, true>) : go(tiny::k_tiny_stage<0, false>);
}

}  // namespace nmhd
