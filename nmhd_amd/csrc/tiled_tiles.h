// tiled_tiles.h -- the two stage kernels of the production path as tile
// functions, shared by the single-box launches (kernels_tiled.hip) and the
// multi-box launches (kernels_batch.hip).
//
//  faces_tile   all three face fluxes of every cell of a TX x TY column tile
//               over planes [z0, zend), one HLLD per face plus the tile's
//               upper boundary faces.  The x and y stencils (cells i-2..i+1)
//               are read from an LDS ring of two planes that the workgroup
//               stages cooperatively; the z stencil is the thread's own
//               column, carried in registers.  Differences the hydro fluxes in the tile (LDS
//               for x and y, registers for z) and writes the hydro
//               divergence of every cell (5 floats) and the six B fluxes the
//               CT needs (6 floats).
//  update_tile  per cell of the tile: the 24 upwinded edge EMFs of the
//               cell's six faces, the conserved update, primitive
//               recovery and the shearing-box kick, as a z march with the
//               neighbour data staged in LDS rings one plane ahead; in stage
//               2 it also returns the CFL time of the new state of the
//               thread's cells (interior cells only).
//
// Both run on 256-thread workgroups (TX * TY == 256, 1-D thread index) and
// take their LDS as a pointer so that one kernel can run tiles of
// several shapes out of one buffer.  The arithmetic of a cell does not depend
// on the tile shape or the z chunk, so every tiling gives bit-identical
// results.
//
// Reference correspondence (INL = library/mhd_solver.inl): calc_flux_kernel
// (INL:760-816) for the three sweeps -> faces_tile; add_flux_kernel x3
// (INL:851-897), corner_magnet_flux (INL:819-840), to_conserved
// (INL:990-1007), add_pace / update (INL:1029-1071), to_primitive
// (INL:1009-1027), external_acceleration_kernel (INL:1073-1084) and
// cfl_condition_kernel (INL:714-739) -> update_tile.
#pragma once

#include "nmhd_kernels.h"
#include <type_traits>

namespace nmhd {
namespace tiled {

__device__ __forceinline__ float stage_h(const StepState *st, int hsel) {
  return hsel == H_HALF ? st->h : (hsel == H_FULL ? st->dt : st->h_diag);
}

// The stage step of a step just opened (selected by value: a pointer into the
// record would keep it in memory).
__device__ __forceinline__ float opened_size(const StepState &s, int hsel) {
  const float half = s.h, full = s.dt;
  return hsel == H_HALF ? half : full;
}

// Whether the step that a stage kernel belongs to is taken, and its size.
__device__ __forceinline__ bool stage_active(const StageStep &ss) {
  return ss.hsel == H_FIXED || ss.rec->s.active;
}
__device__ __forceinline__ float stage_size(const StageStep &ss) {
  return ss.hsel == H_FIXED ? ss.h : stage_h(&ss.rec->s, ss.hsel);
}

// The stage step of a launch, opening the step first when it is the step's
// first kernel; false: the step is not taken.
__device__ __forceinline__ bool stage_begin(const Box &b, const StageStep &ss,
                                            const OpenStep &open, float &h) {
  if (open.in) {
    const StepState s = open_step(b, open, blockIdx.x == 0 && threadIdx.x < 64);
    h = opened_size(s, ss.hsel);
    return s.active;
  }
  h = stage_size(ss);
  return stage_active(ss);
}

// true modulo for staging coordinates, which may lie several box lengths
// outside [0, n) when a tile is wider than a small box
__device__ __forceinline__ int pmod(int i, int n) {
  const int r = i % n;
  return r < 0 ? r + n : r;
}

// Results that the next kernel reads, and values that only the loading thread
// reads.  Nt: past the caches, where they would displace the halo planes that
// neighbouring tiles re-read from L2; otherwise through them, where the next
// kernel finds them (streamed() decides).
template <bool Nt>
__device__ __forceinline__ void put(float *dst, float v) {
  if (Nt)
    __builtin_nontemporal_store(v, dst);
  else
    *dst = v;
}
template <bool Nt>
__device__ __forceinline__ float get(const float *src) {
  return Nt ? __builtin_nontemporal_load(src) : *src;
}

// The element at byte offset boff (32-bit) from a workgroup-uniform base:
// loads and stores through it take the scalar-base + 32-bit vector-offset
// form, with no 64-bit address arithmetic per lane.  The offsets used are
// in-plane (an XY plane holds fewer than 2^30 cells, checked at creation).
template <class T>
__device__ __forceinline__ T *at_byte(T *base, unsigned boff) {
  using C = typename std::conditional<std::is_const<T>::value, const char, char>::type;
  return reinterpret_cast<T *>(reinterpret_cast<C *>(base) + boff);
}

// A per-lane offset made opaque to the optimiser for the current plane (an
// empty asm operand, no instruction): otherwise the loop-invariant sum of
// an array base and the offset is hoisted out of the plane loop as a 64-bit
// per-lane pointer per array, which costs registers and 64-bit adds.
__device__ __forceinline__ unsigned opaque(unsigned v) {
  asm volatile("" : "+v"(v));
  return v;
}

__device__ __forceinline__ void recon(int mode, float x0, float x1, float x2, float x3, float &l,
                                      float &r) {
  if (mode == 1) {
    l = x1;
    r = x2;
  } else {
    recon_minbee2_med3(x0, x1, x2, x3, l, r);
  }
}

// Reconstruction of a cell-centred B component, the average of its cell's two
// faces, from the four stencil cells' face sums a + b instead of the
// averages 0.5 (a + b): every step of the reconstruction (differences,
// median of three, the half-slope multiply-add) commutes exactly with the
// scaling by 2, so halving the two face states gives the same bits as
// reconstructing the averages, with 4 multiplies fewer per variable.
__device__ __forceinline__ void recon_bsum(int mode, float s0, float s1, float s2, float s3,
                                           float &l, float &r) {
  recon(mode, s0, s1, s2, s3, l, r);
  l *= 0.5f;
  r *= 0.5f;
}

__device__ __forceinline__ float upwind(float s, float f0, float f1) {
  return s > 0.0f ? f0 : (s < 0.0f ? f1 : 0.5f * (f0 + f1));
}

// Minimum of v over the 256-thread workgroup, folded into *target (float
// bits, all candidates >= 0) by one atomic.  red: 4 floats of LDS.
__device__ __forceinline__ void block_min_into(float v, unsigned *target, float *red) {
  const float m = wave_min64(v);
  const int tid = threadIdx.x;
  if ((tid & 63) == 0) red[tid >> 6] = m;
  __syncthreads();
  if (tid == 0) {
    const float r = fminf(fminf(red[0], red[1]), fminf(red[2], red[3]));
    atomicMin(target, __float_as_uint(r));
  }
  __syncthreads();
}

constexpr int kTileThreads = 256;

// What the face kernel hands to the update kernel, in the 21-array flux
// storage of a stage: the hydro divergence of every cell (5 arrays, in the
// slots of the x-sweep's hydro fluxes) and the six face fluxes of B that
// the CT edge EMFs need.
struct StageBuf {
  float *pace[5];  // P_rho, P_mx, P_my, P_mz, P_E
  float *fb[6];    // x-face F(B_y), x-face F(B_z), y-face F(B_z), y-face F(B_x),
                   // z-face F(B_x), z-face F(B_y)
};

__host__ __device__ inline StageBuf stage_buf(const FluxSet &F) {
  StageBuf s;
  for (int k = 0; k < 5; ++k) s.pace[k] = F.dir[0].f[k];
  s.fb[0] = F.dir[0].f[5];
  s.fb[1] = F.dir[0].f[6];
  s.fb[2] = F.dir[1].f[5];
  s.fb[3] = F.dir[1].f[6];
  s.fb[4] = F.dir[2].f[5];
  s.fb[5] = F.dir[2].f[6];
  return s;
}

template <int TX, int TY>
struct FacesShape {
  static_assert(TX * TY == kTileThreads, "tiles have 256 threads");
  static_assert(TX <= 64 && TY <= 64, "a boundary face row or column fits one wave");
  static constexpr int LX = TX + 4, LY = TY + 4, LN = LX * LY;
  static constexpr int NS = (LN + kTileThreads - 1) / kTileThreads;  // slots per thread
  // LDS (floats): two staged planes of rho, v, p, B_x, B_y; one plane of the
  // sums of B_z on the lower and upper z-faces; then the hydro fluxes of the
  // plane's x-faces [5][TY][TX+1] and y-faces [5][TY+1][TX]
  static constexpr int kSz = 2 * 7 * LN;
  static constexpr int kFx = kSz + LN;
  static constexpr int kFy = kFx + 5 * TY * (TX + 1);
  // then the global in-plane offset of every staged slot (int), kept in LDS
  // rather than in registers (read once per plane by the slot's own thread)
  static constexpr int kGxy = kFy + 5 * (TY + 1) * TX;
  static constexpr int kLds = kGxy + LN;
  // waves per SIMD the LDS allows (4 workgroups of 4 waves per CU when 4
  // copies fit the 160 KiB, else 3): the kernels' occupancy target
  static constexpr int kWavesPerSimd = 4 * kLds * 4 <= 160 * 1024 ? 4 : 3;
};

// Face fluxes of a TX x TY column tile over planes [z0, zend), and the
// hydro divergence of its cells.  Per plane p the workgroup computes the
// x-faces i in [x0, x0+TX] and the y-faces j in [y0, y0+TY] (the upper
// boundary faces of the tile, i.e. one face column and one face row more
// than it owns, on the lanes of a rotating wave), keeps their hydro fluxes in
// LDS and differences them, and every thread its cell's lower z-face; one
// more pass computes the z-faces below plane zend.  Only the tile's own faces
// write their B fluxes to memory.  Recon is the box's reconstruction
// (b.recon: 0 minbee2, 1 piecewise constant) as a compile-time constant, so
// that the scheme costs no per-variable selects; faces_tile_any dispatches on
// it.
//
// Bound by VALU issue in large boxes, by the latency of a march in small
// ones.  The z stencil needs only the thread's own column, so its planes
// z0-2, z0-1 and zend+1 are loaded into registers and never staged: a chunk
// of zc planes takes zc passes, zc + 1 staged planes and one more z-face.
// Staging them too (zc + 4 passes over zc + 4 planes) took 496 us at 256^3
// (periodic) against 478, 20.2 against 18.3 at 64^3 and 13.3 against 11.4 at
// 32^3.  The column of plane zend+1 is loaded after the march: prefetching it
// during the last pass keeps the staging registers alive across the loop's
// end, which costs 14 VGPRs (11 spilled at 4 waves per SIMD).
template <int TX, int TY, int Recon, bool Nt>
__device__ __forceinline__ void faces_tile(const Box &b, const FieldPtrs &W, const FluxSet &Fs,
                                           float h, int x0, int y0, int z0, int zend,
                                           float *lds) {
  using S = FacesShape<TX, TY>;
  constexpr int NT = kTileThreads, LX = S::LX, LN = S::LN, NS = S::NS;
  const StageBuf SB = stage_buf(Fs);
  float *const FXL = lds + S::kFx;
  float *const FYL = lds + S::kFy;
  const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX;
  const int nx = b.n[0], ny = b.n[1], nz = b.n[2];
  const int plane = nx * ny;
  const int x = x0 + tx, y = y0 + ty;
  const bool valid = (x < nx) && (y < ny);
  constexpr int mode = Recon;
  const bool src = b.source == 1;
  const float idx = b.inv_d[0], idy = b.inv_d[1], idz = b.inv_d[2];

  float *const SZ = lds + S::kSz;  // B_z on the lower + upper z-face, plane p
  // global in-plane byte offset of every LDS slot this thread stages (each
  // thread writes and reads only its own slots)
  unsigned *const GXY = reinterpret_cast<unsigned *>(lds + S::kGxy);
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int li = tid + s * NT;
    const int lx = li % LX, ly = li / LX;
    if (li < LN) GXY[li] = (unsigned)(pmod(y0 - 2 + ly, ny) * nx + pmod(x0 - 2 + lx, nx)) * 4u;
  }
  // this thread's own cell: in-plane byte offset
  const unsigned own = (unsigned)(y * nx + x) * 4u;
  // start of plane p (wrapped) in an array
  auto plane_of = [&](auto *arr, int p) { return arr + (size_t)wrap(p, nz) * plane; };
  float stage[NS][8];
  auto load_plane = [&](int p, float (&dst)[NS][8]) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if (tid + s * NT < LN) {
        const unsigned g = opaque(GXY[tid + s * NT]);
#pragma unroll
        for (int f = 0; f < 8; ++f) dst[s][f] = *at_byte(plane_of(W.f[f], p), g);
      }
    }
  };
  // rho, v, p, B_x, B_y of a plane into buffer buf
  auto store_plane = [&](int buf, const float (&src)[NS][8]) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int li = tid + s * NT;
      if (li < LN) {
#pragma unroll
        for (int f = 0; f < 7; ++f) lds[(buf * 7 + f) * LN + li] = src[s][f];
      }
    }
  };
  // B_z of the newest staged plane at this thread's slots, and its sum with
  // the next plane's
  float bzs[NS];
  auto store_bzsum = [&](const float (&src)[NS][8]) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if (tid + s * NT < LN) SZ[tid + s * NT] = bzs[s] + src[s][7];
      bzs[s] = src[s][7];
    }
  };
  // the thread's own column of plane p, with the upper B_x and B_y faces:
  // rho, vx, vy, vz, p, B_x, B_y, B_z | B_x(x+1), B_y(y+1)
  const unsigned ownc = valid ? own : 0u;
  auto load_column = [&](int p, float (&dst)[NS][8]) {
    const unsigned ox = valid ? (unsigned)(y * nx + wrap(x + 1, nx)) * 4u : 0u;
    const unsigned oy = valid ? (unsigned)(wrap(y + 1, ny) * nx + x) * 4u : 0u;
#pragma unroll
    for (int f = 0; f < 7; ++f) dst[0][f] = *at_byte(plane_of(W.f[f], p), ownc);
    dst[1][0] = *at_byte(plane_of(W.f[5], p), ox);
    dst[1][1] = *at_byte(plane_of(W.f[6], p), oy);
  };
  // z-stencil values of a column: rho, vz, vx, vy, p, Bx_avg, By_avg
  auto column_vars = [&](const float (&cl)[NS][8], float (&q)[7]) {
    q[0] = cl[0][0];
    q[1] = cl[0][3];
    q[2] = cl[0][1];
    q[3] = cl[0][2];
    q[4] = cl[0][4];
    q[5] = 0.5f * (cl[0][5] + cl[1][0]);
    q[6] = 0.5f * (cl[0][6] + cl[1][1]);
  };

  // lower x-face of the cell at LDS index c of plane buffer cb
  auto face_x = [&](int cb, int c) -> Flux7 {
    const float *R = lds + (cb * 7 + 0) * LN, *VX = lds + (cb * 7 + 1) * LN;
    const float *VY = lds + (cb * 7 + 2) * LN, *VZ = lds + (cb * 7 + 3) * LN;
    const float *PR = lds + (cb * 7 + 4) * LN, *BX = lds + (cb * 7 + 5) * LN;
    const float *BY = lds + (cb * 7 + 6) * LN;
    float L[7], Rr[7];
    const int s0 = c - 2, s1 = c - 1, s2 = c, s3 = c + 1;
    recon(mode, R[s0], R[s1], R[s2], R[s3], L[0], Rr[0]);
    recon(mode, VX[s0], VX[s1], VX[s2], VX[s3], L[1], Rr[1]);
    recon(mode, VY[s0], VY[s1], VY[s2], VY[s3], L[2], Rr[2]);
    recon(mode, VZ[s0], VZ[s1], VZ[s2], VZ[s3], L[3], Rr[3]);
    recon(mode, PR[s0], PR[s1], PR[s2], PR[s3], L[4], Rr[4]);
    recon_bsum(mode, BY[s0] + BY[s0 + LX], BY[s1] + BY[s1 + LX], BY[s2] + BY[s2 + LX],
               BY[s3] + BY[s3 + LX], L[5], Rr[5]);
    recon_bsum(mode, SZ[s0], SZ[s1], SZ[s2], SZ[s3], L[6], Rr[6]);
    if (src) {
      const float mbv = 0.5f * h * accel_x(b, 0.5f * (VY[s1] + VY[s2]));
      L[1] += mbv;
      Rr[1] += mbv;
    }
    return hlld(b.gamma, b.inv_gm1, BX[c], L[0], Rr[0], L[1], Rr[1], L[2], Rr[2], L[3], Rr[3],
                L[4], Rr[4], L[5], Rr[5], L[6], Rr[6]);
  };
  // lower y-face of the cell at LDS index c; yrow = the face's array row
  auto face_y = [&](int cb, int c, int yrow) -> Flux7 {
    const float *R = lds + (cb * 7 + 0) * LN, *VX = lds + (cb * 7 + 1) * LN;
    const float *VY = lds + (cb * 7 + 2) * LN, *VZ = lds + (cb * 7 + 3) * LN;
    const float *PR = lds + (cb * 7 + 4) * LN, *BX = lds + (cb * 7 + 5) * LN;
    const float *BY = lds + (cb * 7 + 6) * LN;
    float L[7], Rr[7];
    const int s0 = c - 2 * LX, s1 = c - LX, s2 = c, s3 = c + LX;
    recon(mode, R[s0], R[s1], R[s2], R[s3], L[0], Rr[0]);
    recon(mode, VY[s0], VY[s1], VY[s2], VY[s3], L[1], Rr[1]);
    recon(mode, VZ[s0], VZ[s1], VZ[s2], VZ[s3], L[2], Rr[2]);
    recon(mode, VX[s0], VX[s1], VX[s2], VX[s3], L[3], Rr[3]);
    recon(mode, PR[s0], PR[s1], PR[s2], PR[s3], L[4], Rr[4]);
    recon_bsum(mode, SZ[s0], SZ[s1], SZ[s2], SZ[s3], L[5], Rr[5]);
    recon_bsum(mode, BX[s0] + BX[s0 + 1], BX[s1] + BX[s1 + 1], BX[s2] + BX[s2 + 1],
               BX[s3] + BX[s3 + 1], L[6], Rr[6]);
    if (src) {
      const float mbv = 0.5f * h * accel_y_face(b, 0.5f * (VX[s1] + VX[s2]), yrow);
      L[1] += mbv;
      Rr[1] += mbv;
    }
    return hlld(b.gamma, b.inv_gm1, BY[c], L[0], Rr[0], L[1], Rr[1], L[2], Rr[2], L[3], Rr[3],
                L[4], Rr[4], L[5], Rr[5], L[6], Rr[6]);
  };
  // the lower y-face (isy) or x-face of the cell at LDS index c, with the
  // stencil direction chosen per lane: the same expressions, in the same
  // order, as face_y / face_x, so the two give the same bits.  The five
  // hydro variables are reconstructed in the fixed order (rho, vx, vy, vz, p)
  // and the velocities then permuted into (normal, t1, t2); of the
  // transverse B averages, the one along z (the sums of B_z) is common to both and the other (B_y along y for an x-face, B_x along x
  // for a y-face) is read through a per-lane pointer.
  auto face_xy = [&](int cb, int c, bool isy, int yrow) -> Flux7 {
    const float *R = lds + (cb * 7 + 0) * LN, *VX = lds + (cb * 7 + 1) * LN;
    const float *VY = lds + (cb * 7 + 2) * LN, *VZ = lds + (cb * 7 + 3) * LN;
    const float *PR = lds + (cb * 7 + 4) * LN, *BX = lds + (cb * 7 + 5) * LN;
    const float *BY = lds + (cb * 7 + 6) * LN;
    const float *OA = isy ? BX : BY, *OB = isy ? BX + 1 : BY + LX;
    const int st = isy ? LX : 1;
    const int s0 = c - 2 * st, s1 = c - st, s2 = c, s3 = c + st;
    float L[7], Rr[7], lx, rx, ly, ry, lz, rz, lo, ro, lc, rc;
    recon(mode, R[s0], R[s1], R[s2], R[s3], L[0], Rr[0]);
    recon(mode, VX[s0], VX[s1], VX[s2], VX[s3], lx, rx);
    recon(mode, VY[s0], VY[s1], VY[s2], VY[s3], ly, ry);
    recon(mode, VZ[s0], VZ[s1], VZ[s2], VZ[s3], lz, rz);
    recon(mode, PR[s0], PR[s1], PR[s2], PR[s3], L[4], Rr[4]);
    recon_bsum(mode, OA[s0] + OB[s0], OA[s1] + OB[s1], OA[s2] + OB[s2], OA[s3] + OB[s3], lo, ro);
    recon_bsum(mode, SZ[s0], SZ[s1], SZ[s2], SZ[s3], lc, rc);
    // x-face: (vx, vy, vz), (B_y, B_z); y-face: (vy, vz, vx), (B_z, B_x)
    L[1] = isy ? ly : lx, Rr[1] = isy ? ry : rx;
    L[2] = isy ? lz : ly, Rr[2] = isy ? rz : ry;
    L[3] = isy ? lx : lz, Rr[3] = isy ? rx : rz;
    L[5] = isy ? lc : lo, Rr[5] = isy ? rc : ro;
    L[6] = isy ? lo : lc, Rr[6] = isy ? ro : rc;
    if (src) {
      const float *VA = isy ? VX : VY;
      const float va = 0.5f * (VA[s1] + VA[s2]);
      const float mbv = 0.5f * h * (isy ? accel_y_face(b, va, yrow) : accel_x(b, va));
      L[1] += mbv;
      Rr[1] += mbv;
    }
    return hlld(b.gamma, b.inv_gm1, isy ? BY[c] : BX[c], L[0], Rr[0], L[1], Rr[1], L[2], Rr[2],
                L[3], Rr[3], L[4], Rr[4], L[5], Rr[5], L[6], Rr[6]);
  };
  // hydro fluxes in the conserved order (rho, m_x, m_y, m_z, E)
  auto put_x = [&](int row, int col, const Flux7 &r) {
    float *d = FXL + row * (TX + 1) + col;
    constexpr int st = TY * (TX + 1);
    d[0] = r.rho;
    d[st] = r.mn;
    d[2 * st] = r.mt1;
    d[3 * st] = r.mt2;
    d[4 * st] = r.e;
  };
  auto put_y = [&](int row, int col, const Flux7 &r) {
    float *d = FYL + row * TX + col;
    constexpr int st = (TY + 1) * TX;
    d[0] = r.rho;
    d[st] = r.mt2;
    d[2 * st] = r.mn;
    d[3 * st] = r.mt1;
    d[4 * st] = r.e;
  };

  // own cell in the LDS tile
  const int c = (ty + 2) * LX + tx + 2;
  // z march: values of plane p, their difference to plane p-1, and the left
  // state of the z-face below plane p (all three carried from plane to plane)
  float qc[7], dm[7], Lz[7];
  float pxy[5] = {}, fzl[5] = {};  // x+y divergence and lower z-flux of plane p-1
  float bz;                        // B_z on the lower z-face of plane p, own cell

  // prologue, all loads in flight together: the own column of planes z0-2,
  // z0-1; planes z0 and z0+1 staged
  {
    float c0[NS][8], c1[NS][8], first[NS][8];
    load_plane(z0, first);
    load_plane(z0 + 1, stage);
    load_column(z0 - 2, c0);
    load_column(z0 - 1, c1);
    bz = *at_byte(plane_of(W.f[7], z0), ownc);
    store_plane(z0 & 1, first);
#pragma unroll
    for (int s = 0; s < NS; ++s) bzs[s] = first[s][7];
    store_plane((z0 + 1) & 1, stage);
    store_bzsum(stage);
    column_vars(c0, qc);
    column_vars(c1, Lz);
#pragma unroll
    for (int v = 0; v < 7; ++v) dm[v] = Lz[v] - qc[v];
  }
  __syncthreads();
  {
    const float *P0 = lds + (z0 & 1) * 7 * LN;
    qc[0] = P0[c];
    qc[1] = P0[3 * LN + c];
    qc[2] = P0[1 * LN + c];
    qc[3] = P0[2 * LN + c];
    qc[4] = P0[4 * LN + c];
    qc[5] = 0.5f * (P0[5 * LN + c] + P0[5 * LN + c + 1]);
    qc[6] = 0.5f * (P0[6 * LN + c] + P0[6 * LN + c + LX]);
#pragma unroll
    for (int v = 0; v < 7; ++v) {
      const float d = qc[v] - Lz[v];
      if (mode != 1) Lz[v] = Lz[v] + 0.5f * minmod_med3(dm[v], d);
      dm[v] = d;
    }
  }

  // the z-face below plane p: its left state was formed with plane p-1, the
  // right state needs qn, the values of plane p+1; completes plane p-1
  auto face_z = [&](int p, const float (&qn)[7], float (&fzn)[5], bool inner) {
    const unsigned ownp = opaque(own);
    float Rr[7], Ln[7];
#pragma unroll
    for (int v = 0; v < 7; ++v) {
      const float d = qn[v] - qc[v];
      if (mode == 1) {
        Rr[v] = qc[v];
        Ln[v] = qc[v];
      } else {
        const float sl = minmod_med3(dm[v], d);
        Rr[v] = qc[v] - 0.5f * sl;
        Ln[v] = qc[v] + 0.5f * sl;
      }
      dm[v] = d;
      qc[v] = qn[v];
    }
    if (valid) {
      // the z acceleration is zero: the face predictor adds nothing
      const Flux7 r = hlld(b.gamma, b.inv_gm1, bz, Lz[0], Rr[0], Lz[1], Rr[1], Lz[2], Rr[2],
                           Lz[3], Rr[3], Lz[4], Rr[4], Lz[5], Rr[5], Lz[6], Rr[6]);
      fzn[0] = r.rho;
      fzn[1] = r.mt1;
      fzn[2] = r.mt2;
      fzn[3] = r.mn;
      fzn[4] = r.e;
      if (inner) {
        put<Nt>(at_byte(plane_of(SB.fb[4], p), ownp), r.bt1);  // B_x
        put<Nt>(at_byte(plane_of(SB.fb[5], p), ownp), r.bt2);  // B_y
      }
      // plane p-1 complete: its lower z-face (fzl) and upper z-face (fzn)
      if (p > z0) {
#pragma unroll
        for (int k = 0; k < 5; ++k)
          put<Nt>(at_byte(plane_of(SB.pace[k], p - 1), ownp), pxy[k] + (fzl[k] - fzn[k]) * idz);
      }
    }
#pragma unroll
    for (int v = 0; v < 7; ++v) Lz[v] = Ln[v];
  };

  for (int p = z0; p < zend; ++p) {
    const int cb = p & 1, nb = (p + 1) & 1;
    const bool staged = p + 2 <= zend;   // plane p+2 is staged during this pass
    const unsigned ownp = opaque(own);
    if constexpr (TX + TY <= 64) {
      // the wave that also evaluates this plane's boundary faces sets the
      // workgroup's pace at the plane barrier: it issues first
      if (__builtin_amdgcn_readfirstlane(tid >> 6) == ((p + x0 / TX + y0 / TY) & 3))
        __builtin_amdgcn_s_setprio(1);
      else
        __builtin_amdgcn_s_setprio(0);
    }
    if (staged) load_plane(p + 2, stage);
    {
      const int yrow = y < ny ? y : y - ny;  // the face row y == ny is face 0
      if (y < ny && x <= nx) {
        const Flux7 r = face_x(cb, c);
        put_x(ty, tx, r);
        if (valid) {
          put<Nt>(at_byte(plane_of(SB.fb[0], p), ownp), r.bt1);  // B_y
          put<Nt>(at_byte(plane_of(SB.fb[1], p), ownp), r.bt2);  // B_z
        }
      }
      if (x < nx && y <= ny) {
        const Flux7 r = face_y(cb, c, yrow);
        put_y(ty, tx, r);
        if (valid) {
          put<Nt>(at_byte(plane_of(SB.fb[2], p), ownp), r.bt1);  // B_z
          put<Nt>(at_byte(plane_of(SB.fb[3], p), ownp), r.bt2);  // B_x
        }
      }
      // the tile's upper boundary faces, the y-faces of row y0+TY and the
      // x-faces of column x0+TX, on a wave that rotates with the plane and
      // starts at an offset given by the tile's position, so that the SIMDs
      // of a CU share the extra HLLD evaluations evenly also when the
      // workgroups on it march in step: when both fit one wave (TX + TY <=
      // 64), in one pass (lanes [0, TX) the y-faces, [TX, TX+TY) the
      // x-faces), else on two waves
      const int lane = tid & 63, wave = tid >> 6;
      const int rot = p + x0 / TX + y0 / TY;
      if constexpr (TX + TY <= 64) {
        if (wave == (rot & 3) && lane < TX + TY) {
          const bool isy = lane < TX;
          const int row = isy ? TY : lane - TX, col = isy ? lane : TX;
          const int yy = y0 + row;
          if (isy ? (x0 + lane < nx && yy <= ny) : (yy < ny && x0 + TX <= nx)) {
            const Flux7 r = face_xy(cb, (row + 2) * LX + col + 2, isy, yy < ny ? yy : yy - ny);
            if (isy)
              put_y(TY, lane, r);
            else
              put_x(row, TX, r);
          }
        }
      } else {
        if (wave == ((2 * rot) & 3) && lane < TY) {
          const int yy = y0 + lane;
          if (yy < ny && x0 + TX <= nx) put_x(lane, TX, face_x(cb, (lane + 2) * LX + TX + 2));
        } else if (wave == ((2 * rot + 1) & 3) && lane < TX) {
          const int yy = y0 + TY;
          if (x0 + lane < nx && yy <= ny)
            put_y(TY, lane, face_y(cb, (TY + 2) * LX + lane + 2, yy < ny ? yy : yy - ny));
        }
      }
    }
    const float bz_nx = *at_byte(plane_of(W.f[7], p + 1), opaque(ownc));
    float fzn[5] = {};
    {
      const float *P1 = lds + nb * 7 * LN;
      float qn[7];
      qn[0] = P1[c];
      qn[1] = P1[3 * LN + c];
      qn[2] = P1[1 * LN + c];
      qn[3] = P1[2 * LN + c];
      qn[4] = P1[4 * LN + c];
      qn[5] = 0.5f * (P1[5 * LN + c] + P1[5 * LN + c + 1]);
      qn[6] = 0.5f * (P1[6 * LN + c] + P1[6 * LN + c + LX]);
      face_z(p, qn, fzn, true);
    }
    bz = bz_nx;
    __syncthreads();
    // x + y divergence of plane p (X, Y order)
    if (valid) {
      constexpr int sx = TY * (TX + 1), sy = (TY + 1) * TX;
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        const float *fx = FXL + k * sx + ty * (TX + 1) + tx;
        const float *fy = FYL + k * sy + ty * TX + tx;
        float sacc = (fx[0] - fx[1]) * idx;
        sacc += (fy[0] - fy[TX]) * idy;
        pxy[k] = sacc;
      }
    }
#pragma unroll
    for (int k = 0; k < 5; ++k) fzl[k] = fzn[k];
    if (staged) {  // plane p is no longer needed
      store_plane(cb, stage);
      store_bzsum(stage);
    }
    __syncthreads();
  }
  // the z-faces below plane zend, the upper faces of the chunk's last plane
  {
    float qn[7], fzn[5];
    load_column(zend + 1, stage);
    column_vars(stage, qn);
    face_z(zend, qn, fzn, false);
  }
}

// faces_tile for the box's reconstruction (a uniform branch: two copies of
// the march, each without scheme selects).
template <int TX, int TY, bool Nt>
__device__ __forceinline__ void faces_tile_any(const Box &b, const FieldPtrs &W,
                                               const FluxSet &Fs, float h, int x0, int y0,
                                               int z0, int zend, float *lds) {
  if (b.recon == 1)
    faces_tile<TX, TY, 1, Nt>(b, W, Fs, h, x0, y0, z0, zend, lds);
  else
    faces_tile<TX, TY, 0, Nt>(b, W, Fs, h, x0, y0, z0, zend, lds);
}

template <int TX, int TY>
struct UpdateShape {
  static_assert(TX * TY == kTileThreads, "tiles have 256 threads");
  static_assert(TX <= 64 && TY < 64, "an edge row or column fits one wave");
  static constexpr int RX = TX + 2, RN = RX * (TY + 2);
  static constexpr int NR = (RN + kTileThreads - 1) / kTileThreads;  // ring slots per thread
  static constexpr int EX = TX + 1, EN = EX * (TY + 1);              // edges of the tile
  // LDS layout (floats): S3[5][2][RN] | SZ[2][RN] | SP[4][RN] | E[10][EN]
  static constexpr int kS3 = 0, kSZ = 10 * RN, kSP = 12 * RN, kE = 16 * RN;
  static constexpr int kLds = 16 * RN + 10 * EN;
};

// The two sweeps' members of the twelve edges of a cell, u and v (0: lower,
// 1: upper) indexing the edge: XY / YX on x-face u and y-face v, XZ / ZX on
// x-face u and z-face v, YZ / ZY on y-face u and z-face v.
struct CellEdges {
  float XY[2][2], YX[2][2], XZ[2][2], ZX[2][2], YZ[2][2], ZY[2][2];
};

// The update of the cell at address a, row y, plane r: pc the hydro
// divergence, wb the base rho, v, p, bb its six base face fields (x lower,
// x upper, y.., z..).  cfl_t is lowered to the CFL time of the new state.
template <bool PaceOnly, bool Cfl, bool Nt>
__device__ __forceinline__ void finish_cell(const Box &b, const CellEdges &ce, const float (&pc)[5],
                                            const float (&wb)[5], const float (&bb)[6], float h,
                                            int y, int r, int a, const FieldPtrs &Wo,
                                            float &cfl_t) {
  const float idx_ = b.inv_d[0], idy_ = b.inv_d[1], idz_ = b.inv_d[2];
  float pbx[2], pby[2], pbz[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    pbx[u] = 0.5f * ((ce.XY[u][1] - ce.XY[u][0]) * idy_ + (ce.XZ[u][1] - ce.XZ[u][0]) * idz_) -
             0.5f * (ce.YX[u][1] - ce.YX[u][0]) * idy_ - 0.5f * (ce.ZX[u][1] - ce.ZX[u][0]) * idz_;
    pby[u] = -0.5f * (ce.XY[1][u] - ce.XY[0][u]) * idx_ +
             0.5f * ((ce.YZ[u][1] - ce.YZ[u][0]) * idz_ + (ce.YX[1][u] - ce.YX[0][u]) * idx_) -
             0.5f * (ce.ZY[u][1] - ce.ZY[u][0]) * idz_;
    pbz[u] = -0.5f * (ce.XZ[1][u] - ce.XZ[0][u]) * idx_ - 0.5f * (ce.YZ[1][u] - ce.YZ[0][u]) * idy_ +
             0.5f * ((ce.ZX[1][u] - ce.ZX[0][u]) * idx_ + (ce.ZY[1][u] - ce.ZY[0][u]) * idy_);
  }
  if (PaceOnly) {
#pragma unroll
    for (int k = 0; k < 5; ++k) put<Nt>(&Wo.f[k][a], pc[k]);
    put<Nt>(&Wo.f[5][a], pbx[0]);
    put<Nt>(&Wo.f[6][a], pby[0]);
    put<Nt>(&Wo.f[7][a], pbz[0]);
  } else {
    const float rho0 = wb[0];
    const float vx0 = wb[1], vy0 = wb[2], vz0 = wb[3];
    const float bxl0 = bb[0], bxh0 = bb[1], byl0 = bb[2], byh0 = bb[3];
    const float bzl0 = bb[4], bzh0 = bb[5];
    const float e0 = wb[4] * b.inv_gm1 + 0.5f * rho0 * (vx0 * vx0 + vy0 * vy0 + vz0 * vz0) +
                     0.25f * (bxl0 * bxl0 + bxh0 * bxh0 + byl0 * byl0 + byh0 * byh0 +
                              bzl0 * bzl0 + bzh0 * bzh0);
    const float rho = rho0 + h * pc[0];
    const float mx = rho0 * vx0 + h * pc[1];
    const float my = rho0 * vy0 + h * pc[2];
    const float mz = rho0 * vz0 + h * pc[3];
    const float e = e0 + h * pc[4];
    const float bxl = bxl0 + h * pbx[0], bxh = bxh0 + h * pbx[1];
    const float byl = byl0 + h * pby[0], byh = byh0 + h * pby[1];
    const float bzl = bzl0 + h * pbz[0], bzh = bzh0 + h * pbz[1];
    const float irho = frcp(rho);
    float ux = mx * irho, uy = my * irho;
    const float uz = mz * irho;
    const float eint = e - 0.5f * (mx * mx + my * my + mz * mz) * irho -
                       0.25f * (bxl * bxl + bxh * bxh + byl * byl + byh * byh + bzl * bzl +
                                bzh * bzh);
    const float pres = eint * b.gm1;
    if (b.source == 1) {
      const float ax_ = accel_x(b, uy);
      const float ay_ = accel_y(b, ux, y);
      ux += h * ax_;
      uy += h * ay_;
    }
    put<Nt>(&Wo.f[0][a], rho);
    put<Nt>(&Wo.f[1][a], ux);
    put<Nt>(&Wo.f[2][a], uy);
    put<Nt>(&Wo.f[3][a], uz);
    put<Nt>(&Wo.f[4][a], pres);
    put<Nt>(&Wo.f[5][a], bxl);
    put<Nt>(&Wo.f[6][a], byl);
    put<Nt>(&Wo.f[7][a], bzl);
    if (Cfl) {
      // CFL time of the new state for cells the next ghost fill leaves
      // untouched (interior rows/planes); the ghost cells are reduced
      // after the fill
      if (!refilled(b, y, r)) {
        // same rounding as the full CFL pass (no contraction), so an
        // incrementally reduced dt equals it bit for bit
#pragma clang fp contract(off)
        const float b2 = fmaxf(bxl * bxl, bxh * bxh) + fmaxf(byl * byl, byh * byh) +
                         fmaxf(bzl * bzl, bzh * bzh);
        const float cs = sqrtf((b.gamma * pres + b2) / rho);
        const float t = fminf(b.cfl * b.d[0] / cfl_speed(b, ux, cs),
                              fminf(b.cfl * b.d[1] / cfl_speed(b, uy, cs),
                                    b.cfl * b.d[2] / cfl_speed(b, uz, cs)));
        cfl_t = fminf(cfl_t, t);
      }
    }
  }
}

// The cell update as a z march: a TX x TY column tile plus a one-cell ring
// is staged in LDS, one plane ahead (prefetched into registers while the
// current plane is computed), so that each HBM value is fetched once per tile.
//   S3 (planes r, r+1): v_x, v_y, v_z, x-face F(B_z), y-face F(B_z);
//   SZ (face r+1): z-face F(B_x), F(B_y);
//   SP (plane r): x-face F(B_y), y-face F(B_x), base B_x, B_y;
//   E: the two sweeps' members of every edge of the tile, the edges along z
//      of plane r and those along x and y on the z-faces r and r+1.
// Per plane every thread first forms the edges on its cell's lower faces
// (two waves also those on the tile's upper x- and y-faces), then, after a
// barrier, its cell's update from the shared edges: 6 upwind choices per
// cell instead of the 24 on all its edges, 54 LDS reads instead of 85, and
// two planes of the 3-D ring instead of three.  Bound by HBM in large boxes
// (4.8 TB/s at 256^3) and by the latency of a plane (2.3 us) in small ones;
// with every cell choosing all 24 the first / second stage took 408 / 443 us
// at 256^3 against 400 / 432, and 39 / 49 against 35 / 42 at 96^3.
// The hydro divergence and the base cell values are the thread's own and
// stay in registers.  cfl_t is lowered to the CFL time of every interior
// cell the thread updates (stage 2 with Cfl).
// Raw: the hydro fluxes themselves are in Fs (k_direct_faces wrote them) and
// are differenced here, in the order of the face march.
template <int TX, int TY, bool PaceOnly, bool Cfl, bool Raw, bool Nt>
__device__ __forceinline__ void update_tile(const Box &b, const FieldPtrs &Win, const FluxSet &Fs,
                                            const FieldPtrs &Wb, const FieldPtrs &Wo, float h,
                                            int x0, int y0, int z0, int zend, float *lds,
                                            float &cfl_t) {
  using S = UpdateShape<TX, TY>;
  constexpr int NT = kTileThreads, RX = S::RX, RN = S::RN, NR = S::NR, EX = S::EX, EN = S::EN;
  const StageBuf SB = stage_buf(Fs);
  float *const S3 = lds + S::kS3;
  float *const SZ = lds + S::kSZ;
  float *const SP = lds + S::kSP;
  float *const E = lds + S::kE;

  const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX;
  const int nx = b.n[0], ny = b.n[1], nz = b.n[2];
  const int plane = nx * ny;
  const int x = x0 + tx, y = y0 + ty;
  const bool valid = x < nx && y < ny;

  int gxy[NR];
#pragma unroll
  for (int s = 0; s < NR; ++s) {
    const int li = tid + s * NT;
    gxy[s] = (li < RN) ? pmod(y0 - 1 + li / RX, ny) * nx + pmod(x0 - 1 + li % RX, nx) : 0;
  }
  const float *a3[5] = {Win.f[1], Win.f[2], Win.f[3], SB.fb[1], SB.fb[2]};
  const float *az[2] = {SB.fb[4], SB.fb[5]};
  const float *ap[4] = {SB.fb[0], SB.fb[3], Wb.f[5], Wb.f[6]};
  // staging registers
  float r3[NR][5], rz[NR][2], rp[NR][4];
  auto load3 = [&](int p, float (&dst)[NR][5]) {
    const int base = wrap(p, nz) * plane;
#pragma unroll
    for (int s = 0; s < NR; ++s)
      if (tid + s * NT < RN)
#pragma unroll
        for (int k = 0; k < 5; ++k) dst[s][k] = a3[k][base + gxy[s]];
  };
  auto store3 = [&](int p, const float (&src)[NR][5]) {
#pragma unroll
    for (int s = 0; s < NR; ++s)
      if (tid + s * NT < RN)
#pragma unroll
        for (int k = 0; k < 5; ++k) S3[(k * 2 + (p & 1)) * RN + tid + s * NT] = src[s][k];
  };
  auto loadz = [&](int p, float (&dst)[NR][2]) {
    const int base = wrap(p, nz) * plane;
#pragma unroll
    for (int s = 0; s < NR; ++s)
      if (tid + s * NT < RN)
#pragma unroll
        for (int k = 0; k < 2; ++k) dst[s][k] = az[k][base + gxy[s]];
  };
  auto storez = [&](const float (&src)[NR][2]) {
#pragma unroll
    for (int s = 0; s < NR; ++s)
      if (tid + s * NT < RN)
#pragma unroll
        for (int k = 0; k < 2; ++k) SZ[k * RN + tid + s * NT] = src[s][k];
  };
  auto loadp = [&](int p) {
    const int base = wrap(p, nz) * plane;
#pragma unroll
    for (int s = 0; s < NR; ++s)
      if (tid + s * NT < RN)
#pragma unroll
        for (int k = 0; k < 4; ++k) rp[s][k] = ap[k][base + gxy[s]];
  };
  auto storep = [&]() {
#pragma unroll
    for (int s = 0; s < NR; ++s)
      if (tid + s * NT < RN)
#pragma unroll
        for (int k = 0; k < 4; ++k) SP[k * RN + tid + s * NT] = rp[s][k];
  };
  // Edges on the lower faces of the cell at ring index e, written to edge
  // slot q.  EXY: x-flux of B_y upwinded in y; EYX: y-flux of B_x upwinded in
  // x (and likewise for the XZ and YZ pairs).
  // the edge along z at the lower x- and y-faces, in plane r
  auto edge_z = [&](int r, int e, int q) {
    const float *VX = S3 + (0 * 2 + (r & 1)) * RN, *VY = S3 + (1 * 2 + (r & 1)) * RN;
    const float *FX5 = SP, *FY6 = SP + RN;
    const float sy = VY[e] + VY[e - RX] + VY[e - 1] + VY[e - 1 - RX];
    const float sx = VX[e] + VX[e - 1] + VX[e - RX] + VX[e - 1 - RX];
    E[0 * EN + q] = upwind(sy, FX5[e - RX], FX5[e]);
    E[1 * EN + q] = upwind(sx, FY6[e - 1], FY6[e]);
  };
  // the edge along y at the lower x-face, on z-face f (planes f-1 and f)
  auto edge_y = [&](int f, int e, int q) {
    const int h = f & 1, l = h ^ 1;
    const float *VXl = S3 + (0 * 2 + l) * RN, *VXh = S3 + (0 * 2 + h) * RN;
    const float *VZl = S3 + (2 * 2 + l) * RN, *VZh = S3 + (2 * 2 + h) * RN;
    const float *FX6l = S3 + (3 * 2 + l) * RN, *FX6h = S3 + (3 * 2 + h) * RN;
    const float *FZ5 = SZ;
    const float sz = VZh[e] + VZl[e] + VZh[e - 1] + VZl[e - 1];
    const float sx = VXh[e] + VXh[e - 1] + VXl[e] + VXl[e - 1];
    E[(2 + 4 * h) * EN + q] = upwind(sz, FX6l[e], FX6h[e]);
    E[(3 + 4 * h) * EN + q] = upwind(sx, FZ5[e - 1], FZ5[e]);
  };
  // the edge along x at the lower y-face, on z-face f
  auto edge_x = [&](int f, int e, int q) {
    const int h = f & 1, l = h ^ 1;
    const float *VYl = S3 + (1 * 2 + l) * RN, *VYh = S3 + (1 * 2 + h) * RN;
    const float *VZl = S3 + (2 * 2 + l) * RN, *VZh = S3 + (2 * 2 + h) * RN;
    const float *FY5l = S3 + (4 * 2 + l) * RN, *FY5h = S3 + (4 * 2 + h) * RN;
    const float *FZ6 = SZ + RN;
    const float sz = VZh[e] + VZl[e] + VZh[e - RX] + VZl[e - RX];
    const float sy = VYh[e] + VYh[e - RX] + VYl[e] + VYl[e - RX];
    E[(4 + 4 * h) * EN + q] = upwind(sz, FY5l[e], FY5h[e]);
    E[(5 + 4 * h) * EN + q] = upwind(sy, FZ6[e - RX], FZ6[e]);
  };
  const int c = (ty + 1) * RX + tx + 1;  // own slot in the ring tile
  const int q0 = ty * EX + tx;           // own edge slot
  // the edges on the tile's upper y-faces (row TY) and x-faces (column TX):
  // one wave each, rotating with the plane
  const int lane = tid & 63, wave = tid >> 6;
  const int rot0 = x0 / TX + y0 / TY;
  auto edges = [&](int r, int f, bool along_z) {
    if (along_z) edge_z(r, c, q0);
    edge_y(f, c, q0);
    edge_x(f, c, q0);
    const int rot = rot0 + f;
    if (wave == (rot & 3)) {
      if (lane < TX) {
        const int e = (TY + 1) * RX + lane + 1, q = TY * EX + lane;
        if (along_z) edge_z(r, e, q);
        edge_x(f, e, q);
      }
    } else if (wave == ((rot + 2) & 3)) {
      if (lane <= TY) {
        const int e = (lane + 1) * RX + TX + 1, q = lane * EX + TX;
        if (along_z) edge_z(r, e, q);
        if (lane < TY) edge_y(f, e, q);
      }
    }
  };
  // own-column registers: hydro divergence and base cell values of plane r.
  // Values the rings already hold are read from LDS instead of memory: the
  // base B_x, B_y (SP) always, the base velocities (S3) when the stage input
  // is the base state (the first stage); the base B_z of plane r is the
  // upper B_z of the previous plane.
  const int own = valid ? y * nx + x : 0;
  const bool in_is_base = Win.f[1] == Wb.f[1] && Win.f[2] == Wb.f[2] && Win.f[3] == Wb.f[3];
  float pc[5], pc_nx[5], wb[5] = {}, wb_nx[5] = {}, bz_lo = 0.0f, bz_hi = 0.0f, bz_nx = 0.0f;
  auto load_own = [&](int p, float *dpc, float *dwb) {
    const int base = wrap(p, nz) * plane + own;
    if (!Raw) {
#pragma unroll
      for (int k = 0; k < 5; ++k) dpc[k] = get<Nt>(&SB.pace[k][base]);
    }
    dwb[0] = get<Nt>(&Wb.f[0][base]);
    dwb[4] = get<Nt>(&Wb.f[4][base]);
    if (!in_is_base) {
#pragma unroll
      for (int k = 1; k < 4; ++k) dwb[k] = get<Nt>(&Wb.f[k][base]);
    }
  };

  // raw hydro fluxes of plane r's cell: x- and y-faces, and the lower z-face,
  // which is the upper one of the plane before
  const int ownx = valid ? y * nx + wrap(x + 1, nx) : 0;
  const int owny = valid ? wrap(y + 1, ny) * nx + x : 0;
  float fxl[5], fxh[5], fyl[5], fyh[5], fzl[5], fzh[5];
  auto load_raw = [&](int r) {
    const int base = r * plane, up = wrap(r + 1, nz) * plane;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      fxl[k] = Fs.dir[0].f[k][base + own];
      fxh[k] = Fs.dir[0].f[k][base + ownx];
      fyl[k] = Fs.dir[1].f[k][base + own];
      fyh[k] = Fs.dir[1].f[k][base + owny];
      fzh[k] = Fs.dir[2].f[k][up + own];
    }
  };
  if (Raw) {
#pragma unroll
    for (int k = 0; k < 5; ++k) fzl[k] = Fs.dir[2].f[k][z0 * plane + own];
  }

  // prologue: every load in flight at once; the edges on z-face z0 from
  // planes z0-1 and z0, then plane z0+1 and face z0+1 over them
  {
    float m3[NR][5], c3[NR][5], cz[NR][2];
    load3(z0 - 1, m3);
    load3(z0, c3);
    loadz(z0, cz);
    load3(z0 + 1, r3);
    loadz(z0 + 1, rz);
    loadp(z0);
    load_own(z0, pc, wb);
    bz_lo = Wb.f[7][wrap(z0, nz) * plane + own];
    bz_hi = Wb.f[7][wrap(z0 + 1, nz) * plane + own];
    store3(z0 - 1, m3);
    store3(z0, c3);
    storez(cz);
  }
  __syncthreads();
  edges(z0, z0, false);
  storep();
  __syncthreads();
  store3(z0 + 1, r3);
  storez(rz);
  __syncthreads();

  for (int r = z0; r < zend; ++r) {
    const bool more = r + 1 < zend;
    if (Raw) load_raw(r);
    if (more) {  // prefetch the data of the next iteration
      load3(r + 2, r3);
      loadz(r + 2, rz);
      loadp(r + 1);
      load_own(r + 1, pc_nx, wb_nx);
      bz_nx = get<Nt>(&Wb.f[7][wrap(r + 2, nz) * plane + own]);
    }
    edges(r, r + 1, true);
    const float *BXB = SP + 2 * RN, *BYB = SP + 3 * RN;
    const float bxl0 = BXB[c], bxh0 = BXB[c + 1];
    const float byl0 = BYB[c], byh0 = BYB[c + RX];
    if (in_is_base) {
      wb[1] = S3[(0 * 2 + (r & 1)) * RN + c];
      wb[2] = S3[(1 * 2 + (r & 1)) * RN + c];
      wb[3] = S3[(2 * 2 + (r & 1)) * RN + c];
    }
    __syncthreads();

    if (valid) {
      const int a = r * plane + own;
      // E at x-face i+u, y-face j+v (plane r); x-face i+u, z-face r+v; y-face
      // j+u, z-face r+v
      CellEdges ce;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          ce.XY[u][v] = E[0 * EN + q0 + u + v * EX];
          ce.YX[u][v] = E[1 * EN + q0 + u + v * EX];
          const float *F = E + (2 + 4 * ((r + v) & 1)) * EN + q0;
          ce.XZ[u][v] = F[u];
          ce.ZX[u][v] = F[EN + u];
          ce.YZ[u][v] = F[2 * EN + u * EX];
          ce.ZY[u][v] = F[3 * EN + u * EX];
        }
      const float bb[6] = {bxl0, bxh0, byl0, byh0, bz_lo, bz_hi};
      if (Raw) {
#pragma unroll
        for (int k = 0; k < 5; ++k) {
          float sacc = (fxl[k] - fxh[k]) * b.inv_d[0];
          sacc += (fyl[k] - fyh[k]) * b.inv_d[1];
          pc[k] = sacc + (fzl[k] - fzh[k]) * b.inv_d[2];
          fzl[k] = fzh[k];
        }
      }
      finish_cell<PaceOnly, Cfl, Nt>(b, ce, pc, wb, bb, h, y, r, a, Wo, cfl_t);
    }
    if (more) {
      // the rings are not read between the barriers
      store3(r + 2, r3);
      storez(rz);
      storep();
      if (!Raw) {
#pragma unroll
        for (int k = 0; k < 5; ++k) pc[k] = pc_nx[k];
      }
#pragma unroll
      for (int k = 0; k < 5; ++k) wb[k] = wb_nx[k];
      bz_lo = bz_hi;
      bz_hi = bz_nx;
      __syncthreads();
    }
  }
}

}  // namespace tiled
}  // namespace nmhd
