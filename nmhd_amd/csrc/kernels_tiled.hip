// kernels_tiled.hip -- the production kernel path for one box: two kernels
// per RK stage, each a grid of z-marching column tiles (the tile functions
// are in tiled_tiles.h).
//
//  k_faces         all three face fluxes of every cell, differenced in the
//                  tile (k_direct_faces takes its place in small boxes)
//  k_update_march  divergence, CT, conserved update, primitive recovery, the
//                  shearing-box kick and (stage 2) the CFL minimum of the
//                  new state, one atomic per workgroup
//
// Tiles are mapped to workgroups XCD-aware (xcd_logical_block) so that
// neighbouring tiles, which re-read each other's halos, share an L2.
#include <algorithm>
#include <cmath>

#include "tiled_tiles.h"

namespace nmhd {
namespace tiled {

// Recon = b.recon (the launcher picks the instantiation)
template <int TX, int TY, int Recon, bool Nt>
__global__ void __launch_bounds__(kTileThreads, (FacesShape<TX, TY>::kWavesPerSimd))
    k_faces(Box b, FieldPtrs W, FluxSet F, StageStep ss, OpenStep open, int zc, int gx, int gy) {
  float h;
  if (!stage_begin(b, ss, open, h)) return;
  __shared__ float lds[FacesShape<TX, TY>::kLds];
  const int lb = xcd_logical_block(blockIdx.x, gridDim.x);
  const int x0 = (lb % gx) * TX, y0 = ((lb / gx) % gy) * TY, z0 = (lb / gx / gy) * zc;
  faces_tile<TX, TY, Recon, Nt>(b, W, F, h, x0, y0, z0, min(z0 + zc, b.n[2]), lds);
}

template <int TX, int TY, bool PaceOnly, bool Cfl, bool Raw, bool Nt>
__global__ void __launch_bounds__(kTileThreads, 4) k_update_march(Box b, FieldPtrs Win, FluxSet F,
                                                               FieldPtrs Wb, FieldPtrs Wo,
                                                               StageStep ss, int zc, int gx,
                                                               int gy) {
  const int lb = xcd_logical_block(blockIdx.x, gridDim.x);
  const int x0 = (lb % gx) * TX, y0 = ((lb / gx) % gy) * TY, z0 = (lb / gx / gy) * zc;
  float h;
  if (!stage_begin(b, ss, OpenStep{}, h)) {
    // a step enqueued after the run reached its goal: the last stage's
    // output carries the step's base state through the buffer rotation
    if (Cfl && !PaceOnly) {
      const int x = x0 + (int)threadIdx.x % TX, y = y0 + (int)threadIdx.x / TX;
      const int zend = min(z0 + zc, b.n[2]);
      if (x < b.n[0] && y < b.n[1])
        for (int r = z0; r < zend; ++r) {
          const long a = ((long)r * b.n[1] + y) * b.n[0] + x;
          for (int f = 0; f < 8; ++f) Wo.f[f][a] = Wb.f[f][a];
        }
    }
    return;
  }
  __shared__ float lds[UpdateShape<TX, TY>::kLds];
  __shared__ float red[4];
  float cfl_t = 3.0e38f;
  update_tile<TX, TY, PaceOnly, Cfl, Raw, Nt>(b, Win, F, Wb, Wo, h, x0, y0, z0,
                                              min(z0 + zc, b.n[2]), lds, cfl_t);
  if (Cfl && !PaceOnly) block_min_into(cfl_t, cfl_slot(ss.rec, blockIdx.x), red);
}

}  // namespace tiled

// ------------------------------------------------------------- launchers

// A stage reads and writes 27 arrays (35 in the second), of which the next
// kernel wants most at once: boxes whose hand-off and states the 256 MB
// last-level cache holds for a good part keep them there.  Step times through
// the caches / past them: 80^3 90 / 96 us, 112^3 184 / 211, 130x109x75 180 /
// 205, 128^3 220 / 240, 170x158x120 (3.2M cells) 429 / 477; from 160^3 (4.1M)
// on the halo planes matter more: 469 / 451, 192^3 800 / 759, 256x264x256
// 1888 / 1820.
bool streamed(long cells) { return cells > 3500000; }

namespace {

// Microseconds a workgroup takes per plane with 1..4 of them on its CU,
// measured at 16^3-256^3: latency alone, then more and more issue (faces) or
// bandwidth (update).
struct MarchCost {
  float plane[4];
  int most;  // longest chunk worth considering
};
constexpr MarchCost kFacesCost = {{3.75f, 4.4f, 5.45f, 6.9f}, 32};
constexpr MarchCost kUpdateCost = {{2.3f, 3.1f, 4.0f, 5.5f}, 16};

}  // namespace

// Counted as four, 64x4 face tiles (and all face tiles of a batch with any)
// took chunks with a second round: 64x4x2000 cells 35 us a face launch against
// 30, 640x12x400 130 / 117, a step of 18 boxes of 2.39M cells 382 / 352, of 17
// of 0.83M 188 / 167.
int march_per_cu(bool faces, bool wide) {
  return faces && wide ? tiled::FacesShape<64, 4>::kWavesPerSimd : 4;
}

int march_chunk(bool faces, int nz, int per_cu, const std::function<long(int)> &groups_at) {
  // A march of zc planes costs about one plane more (the prologue and the
  // last z-face); 256 per_cu workgroups are resident.  In one round a
  // CU's share decides; past it the rounds blend, except that a remainder of
  // the first ones costs more than its share, a small one nearly a round of its
  // own (1050 workgroups 1.5 rounds, 1216 1.4, 1408 1.5, 1664 1.7, 2112 2.3,
  // 4224 4.1).  With the remainders past 0.4 at their share alone, 16 boxes of
  // 16..96 cells per edge took 214 us a step against 203, 112^3 185 / 181,
  // 170x158x120 428 / 418; 144^3 377 / 381 is the one the other way.
  const MarchCost &c = faces ? kFacesCost : kUpdateCost;
  int best = 1;
  float least = 0.0f;
  for (int want = 1; want <= c.most && want <= nz; ++want) {
    const int chunks = (nz + want - 1) / want, zc = (nz + chunks - 1) / chunks;
    const float rounds = (float)groups_at(zc) / (256.0f * (float)per_cu);
    float cost;
    if (rounds <= 1.0f) {
      const int share = (int)std::ceil(rounds * (float)per_cu);
      cost = c.plane[share < 1 ? 0 : share - 1] * (float)(zc + 1);
    } else {
      const float whole = std::floor(rounds), part = rounds - whole;
      const float extra =
          part > 0.0f ? (0.4f * std::max(0.0f, 1.0f - part / 0.3f) + 0.15f * (1.0f - part)) / whole
                      : 0.0f;
      cost = c.plane[per_cu - 1] * (float)(zc + 1) * (rounds + extra);
    }
    if (best == 1 && want == 1) least = cost;
    if (cost < least) least = cost, best = zc;
  }
  return best;
}

namespace {

int tiled_zchunk(const Box &b, int tx, int ty, bool faces) {
  const long cols = (long)((b.n[0] + tx - 1) / tx) * ((b.n[1] + ty - 1) / ty);
  return march_chunk(faces, b.n[2], march_per_cu(faces, tx == 64),
                     [&](int zc) { return cols * ((b.n[2] + zc - 1) / zc); });
}

}  // namespace

int tiled_shape(int nx, int ny, bool faces) {
  // Cells that tiles of a shape cover, idle lanes included.  Per covered cell
  // the face march takes 1.15 times as long on 64x4 and 1.16 on 16x16 tiles
  // as on 32x8 (256^3: 511 / 444 / 520 us; 80^3, which 16x16 covers exactly:
  // 38 / 31 / 27).  The update is fastest on 64x4 (256^3: 412 us against 432
  // on 32x8 and 600 on 16x16), whose idle lanes cost it less: 32x8 wins from
  // a fifth more on (130x109x75: 36 against 34, 160x120x100: 58 / 53).
  auto covered = [&](int v) {
    const long tx = kTileTX[v], ty = kTileTY[v];
    return (float)((nx + tx - 1) / tx * tx) * (float)((ny + ty - 1) / ty * ty);
  };
  if (!faces) return covered(TV_64x4) >= 1.19f * covered(TV_32x8) ? TV_32x8 : TV_64x4;
  int v = TV_32x8;
  if (1.15f * covered(TV_64x4) < covered(v)) v = TV_64x4;
  if (1.16f * covered(TV_16x16) < (v == TV_32x8 ? 1.0f : 1.15f) * covered(v)) v = TV_16x16;
  return v;
}

namespace {

template <int TX, int TY>
void faces_as(hipStream_t s, const Box &b, FieldPtrs W, const FluxSet &F, const StageStep &ss,
              const OpenStep &open) {
  const int zc = tiled_zchunk(b, TX, TY, true);
  const int gx = (b.n[0] + TX - 1) / TX, gy = (b.n[1] + TY - 1) / TY, gz = (b.n[2] + zc - 1) / zc;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(gx * gy * gz), dim3(tiled::kTileThreads), 0, s, b, W, F, ss,
                       open, zc, gx, gy);
  };
  if (streamed(b.ncell))
    b.recon == 1 ? go(tiled::k_faces<TX, TY, 1, true>) : go(tiled::k_faces<TX, TY, 0, true>);
  else
    b.recon == 1 ? go(tiled::k_faces<TX, TY, 1, false>) : go(tiled::k_faces<TX, TY, 0, false>);
}

template <int TX, int TY, bool Raw>
void update_as(hipStream_t s, const Box &b, FieldPtrs Win, const FluxSet &F, FieldPtrs Wbase,
               FieldPtrs Wout, const StageStep &ss, bool pace_only, bool cfl) {
  const int zc = tiled_zchunk(b, TX, TY, false);
  const int gx = (b.n[0] + TX - 1) / TX, gy = (b.n[1] + TY - 1) / TY, gz = (b.n[2] + zc - 1) / zc;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(gx * gy * gz), dim3(tiled::kTileThreads), 0, s, b, Win, F,
                       Wbase, Wout, ss, zc, gx, gy);
  };
  if (pace_only)
    go(tiled::k_update_march<TX, TY, true, false, false, false>);
  else if (!Raw && streamed(b.ncell))
    cfl ? go(tiled::k_update_march<TX, TY, false, true, false, true>)
        : go(tiled::k_update_march<TX, TY, false, false, false, true>);
  else
    cfl ? go(tiled::k_update_march<TX, TY, false, true, Raw, false>)
        : go(tiled::k_update_march<TX, TY, false, false, Raw, false>);
}

}  // namespace

void launch_faces(hipStream_t s, const Box &b, FieldPtrs W, const FluxSet &F, const StageStep &ss,
                  const OpenStep &open, int tile) {
  if (tile == kTileAuto && direct_stage(b)) return launch_direct_faces(s, b, W, F, ss, open);
  if (tile == kTileAuto) tile = tiled_shape(b.n[0], b.n[1], true);
  if (tile == TV_64x4)
    faces_as<64, 4>(s, b, W, F, ss, open);
  else if (tile == TV_16x16)
    faces_as<16, 16>(s, b, W, F, ss, open);
  else
    faces_as<32, 8>(s, b, W, F, ss, open);
}

void launch_update_tiled(hipStream_t s, const Box &b, FieldPtrs Win, const FluxSet &F,
                         FieldPtrs Wbase, FieldPtrs Wout, const StageStep &ss, bool pace_only, bool cfl,
                         int tile) {
  const bool raw = tile == kTileAuto && direct_stage(b);
  if (tile == kTileAuto) tile = tiled_shape(b.n[0], b.n[1], false);
  if (raw && tile == TV_64x4)
    update_as<64, 4, true>(s, b, Win, F, Wbase, Wout, ss, false, cfl);
  else if (raw)
    update_as<32, 8, true>(s, b, Win, F, Wbase, Wout, ss, false, cfl);
  else if (tile == TV_64x4)
    update_as<64, 4, false>(s, b, Win, F, Wbase, Wout, ss, pace_only, cfl);
  else if (tile == TV_16x16)
    update_as<16, 16, false>(s, b, Win, F, Wbase, Wout, ss, pace_only, cfl);
  else
    update_as<32, 8, false>(s, b, Win, F, Wbase, Wout, ss, pace_only, cfl);
}

}  // namespace nmhd
