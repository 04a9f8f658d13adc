// kernels_adjoint.hip -- the hand-written reverse (adjoint) of one RK stage
// of the periodic step, U_out = cons(W_base) + h P(W_in), W_out = prim(U_out),
// with dt frozen.  Given lam_out = dL/dW_out it produces dL/dW_base and
// dL/dW_in.  No reference counterpart: the reference has no derivatives; the
// forward it reverses is proceed()'s stage (library/mhd_solver.inl:
// 990-1071 for cons/prim/update, 760-897 for the fluxes and CT, HLLD
// library/hlld.inl:7-284).
//
// Kernels of one stage reverse (all gathers: every thread writes only its
// own cell, no atomics, results independent of scheduling):
//   k_adj_prim    adjoint of prim(U) and of cons(W_base): gU (5 per cell)
//                 and lam_base; and the adjoints of the 6 CT edge-EMF families
//                 (3 distinct values per cell: lamE_x, lamE_y, lamE_z) from the
//                 face-B adjoints of the cell and its lower neighbours, which
//                 the thread recomputes rather than reading them back
//   k_adj_faces   per face of the three directions: adjoint of
//                 the 7 fluxes (divergence + upwinded EMFs, with the forward's
//                 upwind choice recomputed), then the HLLD reverse sweep
//                 (adjoint_hlld.h) -> adjoints of the 7 left/right face states
//                 and of the normal field
//   k_adj_gather  per cell: the reconstruction adjoints of the three
//                 directions, gathered from the 4 faces whose stencils hold
//                 the cell (their state adjoints and the minmod branches the
//                 face reverse recorded) -> lam_in of rho, v, p and of the
//                 cell-averaged B
//   k_adj_bfinish face B: cell-average and normal-field adjoints -> lam_in B
//                 (in small boxes the gather does it)
#include "adjoint_hlld.h"
#include "nmhd_kernels.h"

namespace nmhd {

namespace {

// Cells by 32-bit byte offset from an array's start (the adjoint's arrays
// number over a hundred, so a box that fits the GPU has fewer than 2^30
// cells): loads and stores then take a scalar base and a 32-bit offset, and
// neighbours are sums of per-axis offsets, with no 64-bit or multiply
// arithmetic per access.
__device__ __forceinline__ float ld(const float *p, unsigned o) {
  return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(p) + o);
}
__device__ __forceinline__ float &at(float *p, unsigned o) {
  return *reinterpret_cast<float *>(reinterpret_cast<char *>(p) + o);
}

template <bool Nt>
__device__ __forceinline__ void put(float *p, float v) {
  if (Nt)
    __builtin_nontemporal_store(v, p);
  else
    *p = v;
}

// The thread's cell, and the offset contributions of its index along each
// axis and of the neighbours' (periodic).
struct Place {
  int v[3];           // x, y, z
  unsigned stride[3]; // bytes
  unsigned o[3];      // v * stride
  __device__ __forceinline__ unsigned own() const { return o[0] + o[1] + o[2]; }
  // contribution of index v[d] + s (s in -2..2; n: the box's cells along d)
  __device__ __forceinline__ unsigned to(int d, int s, int n) const {
    int i = v[d] + s;
    if (s < 0) i = i < 0 ? i + n : i;
    if (s > 0) i = i >= n ? i - n : i;
    // a shift of 2 in a box of one cell wraps twice
    return (unsigned)(n == 1 ? 0 : i) * stride[d];
  }
};

// The cell of a thread of workgroup `block` of the cells in order; false
// beyond the last one.
__device__ __forceinline__ bool place_of(const Box &b, unsigned block, Place &p) {
  const unsigned u = block * blockDim.x + threadIdx.x;
  if (u >= (unsigned)b.ncell) return false;
  cell_coords(b, u, p.v[0], p.v[1], p.v[2]);
  p.stride[0] = 4u;
  p.stride[1] = 4u * (unsigned)b.n[0];
  p.stride[2] = p.stride[1] * (unsigned)b.n[1];
  for (int d = 0; d < 3; ++d) p.o[d] = (unsigned)p.v[d] * p.stride[d];
  return true;
}

// weights of the two candidates of the upwind choice s > 0 ? f0 : s < 0 ? f1 : avg
__device__ __forceinline__ float w_lo(float s) { return s > 0.0f ? 1.0f : (s < 0.0f ? 0.0f : 0.5f); }
__device__ __forceinline__ float w_hi(float s) { return s > 0.0f ? 0.0f : (s < 0.0f ? 1.0f : 0.5f); }

// ------------------------------------------------------------- k_adj_prim

// Adjoint of the face value B_d at cell c (its lower d-face) from the stage
// output: its own adjoint, and through the pressure of the two cells that
// share the face (c and its lower d-neighbour m).
__device__ __forceinline__ float face_b_adj(const Box &b, const FieldPtrs &Wout,
                                            const FieldPtrs &lam, int d, unsigned c, unsigned m) {
  return ld(lam.f[5 + d], c) -
         b.gm1 * 0.5f * ld(Wout.f[5 + d], c) * (ld(lam.f[4], c) + ld(lam.f[4], m));
}

// lamE_z = adjoint of the z-edge EMF from the x-sweep (= minus that of the
// y-sweep's), at the edge on the lower x- and y-faces of the cell; likewise
// lamE_y (x-sweep / z-sweep pair on the lower x- and z-faces) and lamE_x
// (y-sweep / z-sweep pair on the lower y- and z-faces), scaled by h.
template <bool AccBase>
__global__ void __launch_bounds__(256) k_adj_prim(Box b, FieldPtrs Wout, FieldPtrs Wbase,
                                                  FieldPtrs lam, float *gU0, float *gU1,
                                                  float *gU2, float *gU3, float *gU4, float h,
                                                  float *lEx, float *lEy, float *lEz,
                                                  FieldPtrs lam_base) {
  Place p;
  if (!place_of(b, xcd_logical_block(blockIdx.x, gridDim.x), p)) return;
  const float gm1 = b.gm1, ig = b.inv_gm1;
  const unsigned a = p.own();
  const float rho = ld(Wout.f[0], a);
  const float v[3] = {ld(Wout.f[1], a), ld(Wout.f[2], a), ld(Wout.f[3], a)};
  const float lp = ld(lam.f[4], a);
  const float irho = frcp(rho);
  const float gE = gm1 * lp;
  float gm[3];
  float grho = ld(lam.f[0], a) + gm1 * lp * 0.5f * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
  for (int d = 0; d < 3; ++d) {
    const float lv = ld(lam.f[1 + d], a);
    gm[d] = lv * irho - gm1 * lp * v[d];
    grho -= lv * v[d] * irho;
  }
  // lower neighbours, one axis and two
  const unsigned lx = p.to(0, -1, b.n[0]), ly = p.to(1, -1, b.n[1]), lz = p.to(2, -1, b.n[2]);
  const unsigned xm = lx + (p.o[1] + p.o[2]), ym = p.o[0] + (ly + p.o[2]);
  const unsigned zm = p.o[0] + (p.o[1] + lz);
  const unsigned xym = lx + (ly + p.o[2]), xzm = lx + (p.o[1] + lz), yzm = p.o[0] + (ly + lz);
  const unsigned mm[3] = {xm, ym, zm};
  float gB[3];
  for (int d = 0; d < 3; ++d) gB[d] = face_b_adj(b, Wout, lam, d, a, mm[d]);
  at(gU0, a) = grho;
  at(gU1, a) = gm[0];
  at(gU2, a) = gm[1];
  at(gU3, a) = gm[2];
  at(gU4, a) = gE;
  // the edge-EMF adjoints: face-B adjoints of the lower x-, y- and
  // z-neighbours, each through its own lower neighbour along its face axis
  {
    const float idx = b.inv_d[0], idy = b.inv_d[1], idz = b.inv_d[2];
    const float gB0_ym = face_b_adj(b, Wout, lam, 0, ym, xym);
    const float gB0_zm = face_b_adj(b, Wout, lam, 0, zm, xzm);
    const float gB1_xm = face_b_adj(b, Wout, lam, 1, xm, xym);
    const float gB1_zm = face_b_adj(b, Wout, lam, 1, zm, yzm);
    const float gB2_xm = face_b_adj(b, Wout, lam, 2, xm, xzm);
    const float gB2_ym = face_b_adj(b, Wout, lam, 2, ym, yzm);
    at(lEz, a) = h * (0.5f * idy * (gB0_ym - gB[0]) + 0.5f * idx * (gB[1] - gB1_xm));
    at(lEy, a) = h * (0.5f * idz * (gB0_zm - gB[0]) + 0.5f * idx * (gB[2] - gB2_xm));
    at(lEx, a) = h * (0.5f * idz * (gB1_zm - gB[1]) + 0.5f * idy * (gB[2] - gB2_ym));
  }
  // cons(W_base): rho, m = rho v, E = p/(g-1) + rho v^2/2 + (B_lo^2 + B_hi^2)/4
  const float rho0 = ld(Wbase.f[0], a);
  const float v0[3] = {ld(Wbase.f[1], a), ld(Wbase.f[2], a), ld(Wbase.f[3], a)};
  float out[8];
  out[0] = grho + 0.5f * gE * (v0[0] * v0[0] + v0[1] * v0[1] + v0[2] * v0[2]);
  for (int d = 0; d < 3; ++d) {
    out[0] += gm[d] * v0[d];
    out[1 + d] = gm[d] * rho0 + gE * rho0 * v0[d];
  }
  out[4] = gE * ig;
  for (int d = 0; d < 3; ++d)
    out[5 + d] = gB[d] + 0.5f * ld(Wbase.f[5 + d], a) * (gE + gm1 * ld(lam.f[4], mm[d]));
  for (int f = 0; f < 8; ++f)
    at(lam_base.f[f], a) = AccBase ? ld(lam_base.f[f], a) + out[f] : out[f];
}

// ------------------------------------------------------------- k_adj_face
//
// Face = lower D-face of cell (x,y,z).  Flux components in the forward's
// order (rho, m_D, m_D+1, m_D+2, E, B_D+1, B_D+2).
//
// The face reverse hands the gather the adjoints of its two reconstructed
// states, aL[k] and aR[k] (variable k), and the limiter branches the
// forward took for them, 4 bits per variable in one word: bits 4k, 4k+1 the
// left state's limited slope, 4k+2, 4k+3 the right state's, each a two-bit
// signed number (limiter_branch).  The gather then spreads the adjoints over
// the stencil cells without reading the stencils again.
struct AdjFaceOut {
  float *aL[7];
  float *aR[7];
  unsigned *br;
  float *abn;
};

// The branch of minmod(a, b) that the forward took, as a two-bit signed
// number: 1 for a, -1 for b, 0 for a zero slope (ties and sign changes as
// minmod takes them).
__device__ __forceinline__ unsigned limiter_branch(float a, float b) {
  return a * b <= 0.0f ? 0u : (fabsf(a) < fabsf(b) ? 1u : 3u);
}

template <int D, bool Nt>
__device__ __forceinline__ void adj_face(const Box &b, const FieldPtrs &W, const float *gU0,
                                         const float *gU1, const float *gU2, const float *gU3,
                                         const float *gU4, const float *lEx, const float *lEy,
                                         const float *lEz, float h, const AdjFaceOut &out,
                                         const Place &pl) {
  constexpr int D1 = (D + 1) % 3, D2 = (D + 2) % 3;
  const float *gU[5] = {gU0, gU1, gU2, gU3, gU4};
  // stencil cells c-2..c+1 along D, and the cells next to them along the
  // transverse axes: s1, s2 above, r1, r2 (of c-1 and c) below
  const unsigned o1 = pl.o[D1], o2 = pl.o[D2];
  const unsigned up1 = pl.to(D1, 1, b.n[D1]), up2 = pl.to(D2, 1, b.n[D2]);
  const unsigned dn1 = pl.to(D1, -1, b.n[D1]), dn2 = pl.to(D2, -1, b.n[D2]);
  unsigned cs[4], s1[4], s2[4], r1[2], r2[2];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const unsigned od = pl.to(D, k - 2, b.n[D]);
    cs[k] = od + (o1 + o2);
    s1[k] = od + (up1 + o2);
    s2[k] = od + (o1 + up2);
    if (k == 1 || k == 2) {
      r1[k - 1] = od + (dn1 + o2);
      r2[k - 1] = od + (o1 + dn2);
    }
  }
  const unsigned a = cs[2], m1 = cs[1];
  // the stencil's variables in the face's order
  float q[7][4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    q[0][s] = ld(W.f[0], cs[s]);
    q[1][s] = ld(W.f[1 + D], cs[s]);
    q[2][s] = ld(W.f[1 + D1], cs[s]);
    q[3][s] = ld(W.f[1 + D2], cs[s]);
    q[4][s] = ld(W.f[4], cs[s]);
    // cell-centred transverse B: the average of the cell's two faces
    q[5][s] = 0.5f * (ld(W.f[5 + D1], cs[s]) + ld(W.f[5 + D1], s1[s]));
    q[6][s] = 0.5f * (ld(W.f[5 + D2], cs[s]) + ld(W.f[5 + D2], s2[s]));
  }
  const float id = b.inv_d[D];
  adj::HOut<float> aF;
  aF.rho = h * (ld(gU[0], a) - ld(gU[0], m1)) * id;
  aF.mn = h * (ld(gU[1 + D], a) - ld(gU[1 + D], m1)) * id;
  aF.mt1 = h * (ld(gU[1 + D1], a) - ld(gU[1 + D1], m1)) * id;
  aF.mt2 = h * (ld(gU[1 + D2], a) - ld(gU[1 + D2], m1)) * id;
  aF.e = h * (ld(gU[4], a) - ld(gU[4], m1)) * id;
  // B fluxes through the upwinded edge EMFs.  For the x-sweep: F(B_y) feeds
  // the z-edges on y-faces j (as the upper candidate) and j+1 (lower one),
  // upwinded by the y-velocity; F(B_z) the y-edges on z-faces k and k+1.
  {
    // adjoint of the edge on the lower D- and q-faces of a cell, with the sign
    // of the D-sweep's member of the pair: the x-sweep (or, for x-edges, the
    // y-sweep) member carries +lam, the other sweep's -lam
    auto edge_adj = [&](int q_, unsigned e) -> float {
      const int other = 3 - D - q_;  // the edge's axis
      const float *arr = other == 0 ? lEx : (other == 1 ? lEy : lEz);
      return D < q_ ? ld(arr, e) : -ld(arr, e);
    };
    // the forward's sums of the four cell velocities around the edge below
    // the face's row and above it, in its order, so that the sign decisions
    // are the same: v the velocity at c-1, c; lo, hi one row below, above
    auto below = [](float v1, float v2, float lo1, float lo2) { return v2 + lo2 + v1 + lo1; };
    auto above = [](float v1, float v2, float hi1, float hi2) { return hi2 + v2 + hi1 + v1; };
    const float *va = W.f[1 + D1], *vb = W.f[1 + D2];
    const float sa0 = below(q[2][1], q[2][2], ld(va, r1[0]), ld(va, r1[1]));
    const float sa1 = above(q[2][1], q[2][2], ld(va, s1[1]), ld(va, s1[2]));
    aF.bt1 = edge_adj(D1, a) * w_hi(sa0) + edge_adj(D1, s1[2]) * w_lo(sa1);
    const float sb0 = below(q[3][1], q[3][2], ld(vb, r2[0]), ld(vb, r2[1]));
    const float sb1 = above(q[3][1], q[3][2], ld(vb, s2[1]), ld(vb, s2[2]));
    aF.bt2 = edge_adj(D2, a) * w_hi(sb0) + edge_adj(D2, s2[2]) * w_lo(sb1);
  }
  // the face states (same reconstruction as the forward)
  float Lq[7], Rq[7];
  for (int k = 0; k < 7; ++k) {
    if (b.recon == 1) {
      Lq[k] = q[k][1];
      Rq[k] = q[k][2];
    } else {
      recon_minbee2_med3(q[k][0], q[k][1], q[k][2], q[k][3], Lq[k], Rq[k]);
    }
  }
  // the limiter branches of L = x1 + m(x1 - x0, x2 - x1)/2 and
  // R = x2 - m(x2 - x1, x3 - x2)/2 over the stencil x0..x3 (cells c-2..c+1),
  // for the gather
  unsigned br = 0u;
  if (b.recon != 1) {
#pragma unroll
    for (int k = 0; k < 7; ++k) {
      const float d01 = q[k][1] - q[k][0], d12 = q[k][2] - q[k][1], d23 = q[k][3] - q[k][2];
      br |= (limiter_branch(d01, d12) | limiter_branch(d12, d23) << 2) << (4 * k);
    }
  }
  adj::HIn<float> in;
  in.bx = ld(W.f[5 + D], a);
  in.rL = Lq[0], in.rR = Rq[0], in.unL = Lq[1], in.unR = Rq[1], in.u1L = Lq[2], in.u1R = Rq[2];
  in.u2L = Lq[3], in.u2R = Rq[3], in.pL = Lq[4], in.pR = Rq[4], in.b1L = Lq[5], in.b1R = Rq[5];
  in.b2L = Lq[6], in.b2R = Rq[6];
  adj::HTape<float> tape;
  adj::HOut<float> F;
  adj::hlld_forward(b.gamma, b.inv_gm1, in, tape, F);
  adj::HIn<float> g;
  adj::hlld_reverse(b.gamma, b.inv_gm1, in, tape, aF, g);
  const float gl[7] = {g.rL, g.unL, g.u1L, g.u2L, g.pL, g.b1L, g.b2L};
  const float gr[7] = {g.rR, g.unR, g.u1R, g.u2R, g.pR, g.b1R, g.b2R};
  for (int k = 0; k < 7; ++k) {
    put<Nt>(&at(out.aL[k], a), gl[k]);
    put<Nt>(&at(out.aR[k], a), gr[k]);
  }
  at(reinterpret_cast<float *>(out.br), a) = __uint_as_float(br);
  at(out.abn, a) = g.bx;
}

// Cells up to which the faces' 42 adjoint arrays (168 bytes a cell) are stored
// through the caches for the gather to find; past that they only displace the
// stencils' neighbours there.  One reverse step through / past the caches: 64^3
// 144 / 149 us, 72^3 200 / 207, 100x90x80 (720k cells) 371 / 387, 96^3 (885k)
// 443 / 430, 112^3 750 / 705, 128^3 1078 / 1019, 224^3 5690 / 5630.
constexpr long kAdjCached = 800000;

// All faces of the three directions in one launch: consecutive workgroups
// take the three directions of the same cells (a uniform branch each), and
// each XCD a contiguous range of them, so that neighbouring rows and planes
// share its L2.  VALU (about 990 instructions a face, 1330 with both sides of
// the fan reversed) and the traffic of 45 output arrays bound it about
// equally: 243 -> 213 us at 128^3, 198 past the caches.
struct AdjFaceOut3 {
  AdjFaceOut d[3];
};

template <bool Nt>
__global__ void __launch_bounds__(256) k_adj_faces(Box b, FieldPtrs W, const float *gU0,
                                                   const float *gU1, const float *gU2,
                                                   const float *gU3, const float *gU4,
                                                   const float *lEx, const float *lEy,
                                                   const float *lEz, float h, AdjFaceOut3 out) {
  const unsigned lb = xcd_logical_block(blockIdx.x, gridDim.x);
  const unsigned block = lb / 3, dir = lb - 3 * block;
  Place p;
  if (!place_of(b, block, p)) return;
  if (dir == 0)
    adj_face<0, Nt>(b, W, gU0, gU1, gU2, gU3, gU4, lEx, lEy, lEz, h, out.d[0], p);
  else if (dir == 1)
    adj_face<1, Nt>(b, W, gU0, gU1, gU2, gU3, gU4, lEx, lEy, lEz, h, out.d[1], p);
  else
    adj_face<2, Nt>(b, W, gU0, gU1, gU2, gU3, gU4, lEx, lEy, lEz, h, out.d[2], p);
}

// ------------------------------------------------------------ k_adj_gather
//
// Bound by memory: 42 adjoint and 3 branch arrays, most read twice.  Selecting
// by the two-bit numbers instead of four compares and selects per variable and
// taking 32-bit offsets: 141 -> 133 us at 128^3, 122 when the faces store past
// the caches.
//
// The reconstruction reverse of direction D at cell (x,y,z): res[0..6] =
// adjoints of rho, v_D, v_D+1, v_D+2, p, Bbar_D+1, Bbar_D+2 of the cell,
// gathered from the four faces whose stencils hold it: faces c+2, c+1, c
// and c-1 along D, where it is stencil cell 0, 1, 2 and 3.  A face's left
// state L = x1 + m/2 and right state R = x2 - m'/2 (m the limited slope of
// x0, x1, x2, m' that of x1, x2, x3) pass their adjoints aL, aR to the
// stencil cells through the branches the forward took:
//   cell 0: -aL/2 [m took x1 - x0]
//   cell 1:  aL + aL/2 ([m took x1 - x0] - [m took x2 - x1]) + aR/2 [m' took x2 - x1]
//   cell 2:  aR + aL/2 [m took x2 - x1] - aR/2 ([m' took x2 - x1] - [m' took x3 - x2])
//   cell 3: -aR/2 [m' took x3 - x2]

// The four faces along D around a cell, and their limiter branches.
struct GatherFaces {
  unsigned f[4], br[4];
};
template <int D>
__device__ __forceinline__ GatherFaces gather_faces(const Box &b, const AdjFaceOut &fa,
                                                    const Place &p) {
  const unsigned rest = p.o[(D + 1) % 3] + p.o[(D + 2) % 3];
  GatherFaces g;
  g.f[0] = p.to(D, 2, b.n[D]) + rest, g.f[1] = p.to(D, 1, b.n[D]) + rest;
  g.f[2] = p.o[D] + rest, g.f[3] = p.to(D, -1, b.n[D]) + rest;
  for (int q = 0; q < 4; ++q)
    g.br[q] = __float_as_uint(ld(reinterpret_cast<const float *>(fa.br), g.f[q]));
  return g;
}
__device__ __forceinline__ float gather_var(const AdjFaceOut &fa, const GatherFaces &g, int k) {
  const unsigned f0 = g.f[0], f1 = g.f[1], f2 = g.f[2], f3 = g.f[3];
  const unsigned b0 = g.br[0], b1 = g.br[1], b2 = g.br[2], b3 = g.br[3];
  // [m took the lower difference], [the upper], and their difference
  auto one = [](unsigned w, int i) { return (float)((w >> i) & 1u); };
  auto signed2 = [](unsigned w, int i) { return (float)((int)(w << (30 - i)) >> 30); };
  const int s = 4 * k;
  const float l0 = ld(fa.aL[k], f0), l1 = ld(fa.aL[k], f1), r1 = ld(fa.aR[k], f1);
  const float l2 = ld(fa.aL[k], f2), r2 = ld(fa.aR[k], f2), r3 = ld(fa.aR[k], f3);
  const float c0 = -0.5f * l0 * (float)((b0 >> s & 1u) & ~(b0 >> (s + 1)));
  const float r1_lo = (float)((b1 >> (s + 2) & 1u) & ~(b1 >> (s + 3)));
  const float c1 = l1 + 0.5f * l1 * signed2(b1, s) + 0.5f * r1 * r1_lo;
  const float c2 = r2 + 0.5f * l2 * one(b2, s + 1) - 0.5f * r2 * signed2(b2, s + 2);
  const float c3 = -0.5f * r3 * one(b3, s + 3);
  return c0 + c1 + c2 + c3;
}
template <int D>
__device__ __forceinline__ void adj_gather(const Box &b, const AdjFaceOut &fa, const Place &p,
                                           float (&res)[7]) {
  const GatherFaces g = gather_faces<D>(b, fa, p);
#pragma unroll
  for (int k = 0; k < 7; ++k) res[k] = gather_var(fa, g, k);
}

// The cell-average B_T adjoint of the cell below p along T, as k_adj_gather
// sums it for that cell.
template <int T>
__device__ __forceinline__ float lower_bbar(const Box &b, const AdjFaceOut3 &fa, const Place &p) {
  Place q = p;
  q.o[T] = p.to(T, -1, b.n[T]);
  // the sweeps along the other two axes, x before y before z; B_T is variable
  // 5 of the sweep along the axis before T, 6 of that after
  constexpr int A = T == 0 ? 1 : 0, C = T == 2 ? 1 : 2;
  float m = 0.0f;
  m += gather_var(fa.d[A], gather_faces<A>(b, fa.d[A], q), (A + 1) % 3 == T ? 5 : 6);
  m += gather_var(fa.d[C], gather_faces<C>(b, fa.d[C], q), (C + 1) % 3 == T ? 5 : 6);
  return m;
}

// lam_in of rho, v, p from the three directions' reconstruction reverses
// (written, or added to with accumulate), and the cell-average B adjoints
// lbb[t] (written), or with Finish the face B of lam_in (k_adj_bfinish), the
// lower neighbours' averages then gathered again.
template <bool Finish>
__global__ void __launch_bounds__(256) k_adj_gather(Box b, AdjFaceOut3 fa, FieldPtrs lam_in,
                                                    int accumulate, float *lbb0, float *lbb1,
                                                    float *lbb2) {
  Place p;
  if (!place_of(b, xcd_logical_block(blockIdx.x, gridDim.x), p)) return;
  const unsigned a = p.own();
  float rho = 0.0f, v[3] = {0.0f, 0.0f, 0.0f}, pr = 0.0f, bb[3] = {0.0f, 0.0f, 0.0f};
  float res[7];
  adj_gather<0>(b, fa.d[0], p, res);  // X: (rho, vx, vy, vz, p, Bby, Bbz)
  rho += res[0], v[0] += res[1], v[1] += res[2], v[2] += res[3], pr += res[4];
  bb[1] += res[5], bb[2] += res[6];
  adj_gather<1>(b, fa.d[1], p, res);  // Y: (rho, vy, vz, vx, p, Bbz, Bbx)
  rho += res[0], v[1] += res[1], v[2] += res[2], v[0] += res[3], pr += res[4];
  bb[2] += res[5], bb[0] += res[6];
  adj_gather<2>(b, fa.d[2], p, res);  // Z: (rho, vz, vx, vy, p, Bbx, Bby)
  rho += res[0], v[2] += res[1], v[0] += res[2], v[1] += res[3], pr += res[4];
  bb[0] += res[5], bb[1] += res[6];
  const float out[5] = {rho, v[0], v[1], v[2], pr};
  for (int f = 0; f < 5; ++f)
    at(lam_in.f[f], a) = accumulate ? ld(lam_in.f[f], a) + out[f] : out[f];
  if (Finish) {
    const float low[3] = {lower_bbar<0>(b, fa, p), lower_bbar<1>(b, fa, p),
                          lower_bbar<2>(b, fa, p)};
    for (int t = 0; t < 3; ++t) {
      const float f = 0.5f * (bb[t] + low[t]) + ld(fa.d[t].abn, a);
      at(lam_in.f[5 + t], a) = accumulate ? ld(lam_in.f[5 + t], a) + f : f;
    }
    return;
  }
  at(lbb0, a) = bb[0];
  at(lbb1, a) = bb[1];
  at(lbb2, a) = bb[2];
}

// Cells up to which the gather finishes the face B itself: it then reads 60
// values more a cell, mostly cached, and saves a launch and the averages' way
// through memory.  One reverse step folded / with k_adj_bfinish: 20^3 42 / 47
// us, 35x30x28 52 / 55, 48^3 88 / 92, 64^3 138 / 142, 72^3 192 / 191, 96^3 438 /
// 432, 128^3 1040 / 1027.
constexpr long kAdjFold = 300000;

// Face B_t of lam_in: half of each adjacent cell's cell-average adjoint plus
// the normal-field adjoint of the t-sweep's face.
__global__ void __launch_bounds__(256) k_adj_bfinish(Box b, const float *lbb0, const float *lbb1,
                                                     const float *lbb2, const float *abn0,
                                                     const float *abn1, const float *abn2,
                                                     FieldPtrs lam_in, int accumulate) {
  Place p;
  if (!place_of(b, xcd_logical_block(blockIdx.x, gridDim.x), p)) return;
  const unsigned a = p.own();
  const float *lbb[3] = {lbb0, lbb1, lbb2};
  const float *abn[3] = {abn0, abn1, abn2};
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    const unsigned m = p.to(t, -1, b.n[t]) + (p.o[(t + 1) % 3] + p.o[(t + 2) % 3]);
    const float v = 0.5f * (ld(lbb[t], a) + ld(lbb[t], m)) + ld(abn[t], a);
    at(lam_in.f[5 + t], a) = accumulate ? ld(lam_in.f[5 + t], a) + v : v;
  }
}

}  // namespace

// ------------------------------------------------------------- launchers

void launch_adj_stage(hipStream_t s, const Box &b, const AdjStageArgs &A) {
  const dim3 g(grid_for(b.ncell)), blk(kBlock);
  if (A.acc_base)
    hipLaunchKernelGGL(k_adj_prim<true>, g, blk, 0, s, b, A.Wout, A.Wbase, A.lam_out, A.gU[0],
                       A.gU[1], A.gU[2], A.gU[3], A.gU[4], A.h, A.lE[0], A.lE[1], A.lE[2],
                       A.lam_base);
  else
    hipLaunchKernelGGL(k_adj_prim<false>, g, blk, 0, s, b, A.Wout, A.Wbase, A.lam_out, A.gU[0],
                       A.gU[1], A.gU[2], A.gU[3], A.gU[4], A.h, A.lE[0], A.lE[1], A.lE[2],
                       A.lam_base);
  AdjFaceOut3 fo;
  for (int d = 0; d < 3; ++d) {
    for (int k = 0; k < 7; ++k) {
      fo.d[d].aL[k] = A.face[d * 15 + k];
      fo.d[d].aR[k] = A.face[d * 15 + 7 + k];
    }
    fo.d[d].br = reinterpret_cast<unsigned *>(A.face[d * 15 + 14]);
    fo.d[d].abn = A.abn[d];
  }
  const dim3 g3(3 * grid_for(b.ncell));
  auto faces = b.ncell > kAdjCached ? k_adj_faces<true> : k_adj_faces<false>;
  hipLaunchKernelGGL(faces, g3, blk, 0, s, b, A.Win, A.gU[0], A.gU[1], A.gU[2], A.gU[3], A.gU[4],
                     A.lE[0], A.lE[1], A.lE[2], A.h, fo);
  const bool fold = b.ncell <= kAdjFold;
  auto gather = fold ? k_adj_gather<true> : k_adj_gather<false>;
  hipLaunchKernelGGL(gather, g, blk, 0, s, b, fo, A.lam_in, A.acc_in ? 1 : 0, A.lbb[0], A.lbb[1],
                     A.lbb[2]);
  if (!fold)
    hipLaunchKernelGGL(k_adj_bfinish, g, blk, 0, s, b, A.lbb[0], A.lbb[1], A.lbb[2], A.abn[0],
                       A.abn[1], A.abn[2], A.lam_in, A.acc_in ? 1 : 0);
}

}  // namespace nmhd
