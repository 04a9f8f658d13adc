// capi_adjoint.hip -- the nmhd_adj_* entry points of include/nmhd.h: the
// forward step with a frozen dt and its hand-written reverse, on caller-owned
// device state arrays (e.g. torch tensors), launched on a caller-chosen
// stream.  The reverse step needs the step's stage states (W*, W^{n+1}):
// nmhd_adj_reverse recomputes them from W^n with the forward kernels,
// nmhd_adj_reverse_stages takes them from the caller (as
// nmhd_adj_forward_stages stored them); both then run the stage reverses
// (kernels_adjoint.hip) from the last stage to the first.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include "capi_internal.h"

using namespace nmhd;

namespace nmhd {

void enqueue_frozen_step(hipStream_t s, const Box &b, int integrator, FieldPtrs Win,
                         FieldPtrs Wstar, FieldPtrs Wout, const FluxSet &F, float dt) {
  const StageStep full{nullptr, H_FIXED, dt}, half{nullptr, H_FIXED, dt / 2};
  bool all = true;  // 21 arrays
  for (const FluxOut &d : F.dir)
    for (const float *p : d.f) all = all && p;
  const int ftile = all ? kTileAuto : tiled_shape(b.n[0], b.n[1], true);
  const int utile = all ? kTileAuto : tiled_shape(b.n[0], b.n[1], false);
  auto stage = [&](FieldPtrs in, FieldPtrs out, const StageStep &ss) {
    if (tiny_stage(b)) return launch_tiny_stage(s, b, in, Win, out, ss, OpenStep{}, false);
    launch_faces(s, b, in, F, ss, OpenStep{}, ftile);
    launch_update_tiled(s, b, in, F, Win, out, ss, false, false, utile);
  };
  if (integrator == NMHD_EULER1) return stage(Win, Wout, full);
  stage(Win, Wstar, half);
  stage(Wstar, Wout, full);
}

}  // namespace nmhd

namespace {
// per thread: the message of the calling thread's last object-less failure
thread_local std::string g_adj_create_error;
constexpr int kWork = 5 + 3 + 3 + 3 + 45;  // gU, lE, lbb, abn, face
}  // namespace

struct nmhd_adj {
  nmhd_desc desc;
  Box box;
  nmhd_geometry geo;
  hipStream_t own = nullptr;
  hipStream_t stream = nullptr;
  std::vector<float *> blocks;  // that hold the arrays below
  float *wstar[8] = {};     // recomputed stage-1 state
  float *wnext[8] = {};     // recomputed stage-2 state
  float *lstar[8] = {};     // dL/dW*
  float *flux[21] = {};     // face fluxes of the forward stages
  float *work[kWork] = {};
  StepRec *rec = nullptr;  // of nmhd_adj_cfl_dt
  std::string err;
};

namespace {

int afail(nmhd_adj *a, int code, const std::string &msg) {
  if (a)
    a->err = msg;
  else
    g_adj_create_error = msg;
  return code;
}

#define AHIP(a, call)                                                                  \
  do {                                                                                 \
    hipError_t e_ = (call);                                                            \
    if (e_ != hipSuccess)                                                              \
      return afail((a), NMHD_EHIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

FieldPtrs to_fields(float *const p[8]) {
  FieldPtrs f;
  for (int i = 0; i < 8; ++i) f.f[i] = p[i];
  return f;
}

FieldPtrs to_fields_c(const float *const p[8]) {
  FieldPtrs f;
  for (int i = 0; i < 8; ++i) f.f[i] = const_cast<float *>(p[i]);
  return f;
}

FluxSet flux_set(nmhd_adj *a) {
  FluxSet F;
  for (int d = 0; d < 3; ++d)
    for (int k = 0; k < 7; ++k) F.dir[d].f[k] = a->flux[d * 7 + k];
  return F;
}

// W_out = S(W_in; dt) with the production stage kernels.
void enqueue_forward(nmhd_adj *a, FieldPtrs Win, FieldPtrs Wstar, FieldPtrs Wout, float dt) {
  enqueue_frozen_step(a->stream, a->box, a->desc.integrator, Win, Wstar, Wout, flux_set(a), dt);
}

AdjStageArgs stage_args(nmhd_adj *a) {
  AdjStageArgs A;
  std::memset(&A, 0, sizeof(A));
  float **w = a->work;
  for (int i = 0; i < 5; ++i) A.gU[i] = *w++;
  for (int i = 0; i < 3; ++i) A.lE[i] = *w++;
  for (int i = 0; i < 3; ++i) A.lbb[i] = *w++;
  for (int i = 0; i < 3; ++i) A.abn[i] = *w++;
  for (int i = 0; i < 45; ++i) A.face[i] = *w++;
  return A;
}

void free_adj(nmhd_adj *a) {
  for (float *p : a->blocks) (void)hipFree(p);
  a->blocks.clear();
  if (a->rec) (void)hipFree(a->rec), a->rec = nullptr;
  if (a->own) (void)hipStreamDestroy(a->own), a->own = nullptr;
}

bool ptrs_ok(const float *const p[8]) {
  if (!p) return false;
  for (int i = 0; i < 8; ++i)
    if (!p[i]) return false;
  return true;
}

}  // namespace

namespace nmhd {
void set_adj_global_error(const std::string &msg) { g_adj_create_error = msg; }
}  // namespace nmhd

extern "C" {

const char *nmhd_adj_last_error(const nmhd_adj *a) {
  return a ? a->err.c_str() : g_adj_create_error.c_str();
}

int nmhd_adj_create(const nmhd_desc *desc, nmhd_adj **out) {
  if (!desc || !out) return afail(nullptr, NMHD_EINVAL, "null argument");
  *out = nullptr;
  std::string why;
  if (!desc_valid(desc, why)) return afail(nullptr, NMHD_EINVAL, why);
  if (desc->margin[0] || desc->margin[1] || desc->margin[2] ||
      desc->source != NMHD_SOURCE_NONE || desc->shear_y)
    return afail(nullptr, NMHD_EINVAL,
                 "the adjoint step is for periodic boxes (margin 0, source NONE, shear_y 0)");
  nmhd_adj *a = new nmhd_adj();
  a->desc = *desc;
  derive_box(desc, a->box, a->geo);
  auto bail = [&](int code, const std::string &msg) {
    free_adj(a);
    delete a;
    return afail(nullptr, code, msg);
  };
  if (hipStreamCreateWithFlags(&a->own, hipStreamNonBlocking) != hipSuccess)
    return bail(NMHD_EHIP, "hipStreamCreate failed");
  a->stream = a->own;
  const size_t stride = array_stride(a->box.ncell);
  // One block for all arrays, but pieces of under 2 MB where they come to less
  // than 32 MB: hipMalloc keeps chunks for those (12 us a piece), while a
  // block of 4 to 30 MB is mapped afresh each time (300 to 700 us).
  size_t left = 3 * 8 + 21 + kWork, room = 0;
  const size_t piece = left * stride > (8u << 20) ? left : std::max<size_t>(1, 500000 / stride);
  float *next = nullptr;
  auto take = [&](float **p, int n) {
    for (int i = 0; i < n; ++i, --left, --room, next += stride) {
      if (!room) {
        room = std::min(piece, left);
        if (hipMalloc(&next, room * stride * sizeof(float)) != hipSuccess) return false;
        a->blocks.push_back(next);
      }
      p[i] = next;
    }
    return true;
  };
  if (!take(a->wstar, 8) || !take(a->wnext, 8) || !take(a->lstar, 8) || !take(a->flux, 21) ||
      !take(a->work, kWork))
    return bail(NMHD_ENOMEM, "allocation failed");
  if (hipMalloc(&a->rec, sizeof(StepRec)) != hipSuccess)
    return bail(NMHD_ENOMEM, "allocation failed");
  *out = a;
  return NMHD_OK;
}

int nmhd_adj_destroy(nmhd_adj *a) {
  if (!a) return NMHD_OK;
  if (a->stream) (void)hipStreamSynchronize(a->stream);
  free_adj(a);
  delete a;
  return NMHD_OK;
}

int nmhd_adj_get_geometry(const nmhd_adj *a, nmhd_geometry *geo) {
  if (!a || !geo) return NMHD_EINVAL;
  *geo = a->geo;
  return NMHD_OK;
}

int nmhd_adj_set_stream(nmhd_adj *a, void *stream) {
  if (!a) return NMHD_EINVAL;
  if (a->stream != (hipStream_t)stream) AHIP(a, hipStreamSynchronize(a->stream));
  a->stream = (hipStream_t)stream;  // NULL: HIP's null stream
  // the object's own stream is used only until the caller names one: release
  // it, so that it does not share the process's few hardware queues with
  // the caller's streams (streams beyond them share a queue and serialise)
  if (a->own && a->own != a->stream) {
    AHIP(a, hipStreamDestroy(a->own));
    a->own = nullptr;
  }
  return NMHD_OK;
}

int nmhd_adj_synchronize(nmhd_adj *a) {
  if (!a) return NMHD_EINVAL;
  AHIP(a, hipGetLastError());
  AHIP(a, hipStreamSynchronize(a->stream));
  return NMHD_OK;
}

int nmhd_adj_cfl_dt(nmhd_adj *a, const float *const w[8], float goal_time, float *dt) {
  if (!a || !ptrs_ok(w) || !dt) return afail(a, NMHD_EINVAL, "bad argument");
  launch_clear_cfl(a->stream, a->rec);
  launch_cfl(a->stream, a->box, to_fields_c(w), goal_time, a->rec, true);
  StepRec h;
  AHIP(a, hipMemcpyAsync(&h, a->rec, sizeof(h), hipMemcpyDeviceToHost, a->stream));
  AHIP(a, hipStreamSynchronize(a->stream));
  *dt = cfl_minimum(h);
  return NMHD_OK;
}

int nmhd_adj_forward(nmhd_adj *a, const float *const w_in[8], float dt, float *const w_out[8]) {
  if (!a || !ptrs_ok(w_in) || !w_out || !ptrs_ok(w_out)) return afail(a, NMHD_EINVAL, "bad argument");
  for (int i = 0; i < 8; ++i)
    if (w_in[i] == w_out[i]) return afail(a, NMHD_EINVAL, "w_out must not alias w_in");
  enqueue_forward(a, to_fields_c(w_in), to_fields(a->wstar), to_fields(w_out), dt);
  AHIP(a, hipGetLastError());
  return NMHD_OK;
}

int nmhd_adj_forward_stages(nmhd_adj *a, const float *const w_in[8], float dt,
                            float *const w_stage[8], float *const w_out[8]) {
  if (!a || !ptrs_ok(w_in) || !w_out || !ptrs_ok(w_out)) return afail(a, NMHD_EINVAL, "bad argument");
  const bool two = a->desc.integrator != NMHD_EULER1;
  if (two && (!w_stage || !ptrs_ok(w_stage))) return afail(a, NMHD_EINVAL, "bad argument");
  for (int i = 0; i < 8; ++i)
    for (int j = 0; j < 8; ++j)
      if (w_in[i] == w_out[j] || (two && (w_stage[i] == w_in[j] || w_stage[i] == w_out[j])))
        return afail(a, NMHD_EINVAL, "w_in, w_stage and w_out must not alias");
  enqueue_forward(a, to_fields_c(w_in), two ? to_fields(w_stage) : to_fields(a->wstar),
                  to_fields(w_out), dt);
  AHIP(a, hipGetLastError());
  return NMHD_OK;
}

namespace {

// lam_in = (dS/dW at Wn)^T lam_out given the step's stage states Ws, Wnext.
void enqueue_reverse(nmhd_adj *a, FieldPtrs Wn, FieldPtrs Ws, FieldPtrs Wnext, float dt,
                     FieldPtrs lam_out, FieldPtrs lam_in) {
  AdjStageArgs A = stage_args(a);
  if (a->desc.integrator == NMHD_EULER1) {
    A.Win = Wn, A.Wbase = Wn, A.Wout = Wnext;
    A.lam_out = lam_out;
    A.lam_base = lam_in;
    A.lam_in = lam_in;
    A.h = dt, A.acc_base = false, A.acc_in = true;
    launch_adj_stage(a->stream, a->box, A);
    return;
  }
  // stage 2: W^{n+1} = prim(cons(W^n) + dt P(W*))
  A.Win = Ws, A.Wbase = Wn, A.Wout = Wnext;
  A.lam_out = lam_out;
  A.lam_base = lam_in;
  A.lam_in = to_fields(a->lstar);
  A.h = dt, A.acc_base = false, A.acc_in = false;
  launch_adj_stage(a->stream, a->box, A);
  // stage 1: W* = prim(cons(W^n) + dt/2 P(W^n))
  A.Win = Wn, A.Wbase = Wn, A.Wout = Ws;
  A.lam_out = to_fields(a->lstar);
  A.lam_base = lam_in;
  A.lam_in = lam_in;
  A.h = dt / 2, A.acc_base = true, A.acc_in = true;
  launch_adj_stage(a->stream, a->box, A);
}

}  // namespace

int nmhd_adj_reverse(nmhd_adj *a, const float *const w_in[8], float dt,
                     const float *const lam_out[8], float *const lam_in[8]) {
  if (!a || !ptrs_ok(w_in) || !ptrs_ok(lam_out) || !lam_in || !ptrs_ok(lam_in))
    return afail(a, NMHD_EINVAL, "bad argument");
  for (int i = 0; i < 8; ++i)
    for (int j = 0; j < 8; ++j)
      if (lam_in[i] == lam_out[j] || lam_in[i] == w_in[j])
        return afail(a, NMHD_EINVAL, "lam_in must not alias w_in or lam_out");
  const FieldPtrs Wn = to_fields_c(w_in);
  const FieldPtrs Ws = to_fields(a->wstar);
  const FieldPtrs Wnext = to_fields(a->wnext);
  enqueue_forward(a, Wn, Ws, Wnext, dt);
  enqueue_reverse(a, Wn, Ws, Wnext, dt, to_fields_c(lam_out), to_fields(lam_in));
  AHIP(a, hipGetLastError());
  return NMHD_OK;
}

int nmhd_adj_reverse_stages(nmhd_adj *a, const float *const w_in[8],
                            const float *const w_stage[8], const float *const w_out[8],
                            float dt, const float *const lam_out[8], float *const lam_in[8]) {
  const bool two = a && a->desc.integrator != NMHD_EULER1;
  if (!a || !ptrs_ok(w_in) || !ptrs_ok(w_out) || (two && !ptrs_ok(w_stage)) ||
      !ptrs_ok(lam_out) || !lam_in || !ptrs_ok(lam_in))
    return afail(a, NMHD_EINVAL, "bad argument");
  for (int i = 0; i < 8; ++i)
    for (int j = 0; j < 8; ++j)
      if (lam_in[i] == lam_out[j] || lam_in[i] == w_in[j] || lam_in[i] == w_out[j] ||
          (two && lam_in[i] == w_stage[j]))
        return afail(a, NMHD_EINVAL, "lam_in must not alias a state or lam_out");
  enqueue_reverse(a, to_fields_c(w_in), two ? to_fields_c(w_stage) : to_fields(a->wstar),
                  to_fields_c(w_out), dt, to_fields_c(lam_out), to_fields(lam_in));
  AHIP(a, hipGetLastError());
  return NMHD_OK;
}

}  // extern "C"
