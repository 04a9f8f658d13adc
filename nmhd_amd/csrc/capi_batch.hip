// capi_batch.hip -- the nmhd_batch_* entry points of include/nmhd.h: many
// independent boxes (periodic or shearing) in shared pools, per-box step
// records, per-box ghost fills, a work
// table of tiles for the stage kernels (a workgroup per tile, or workgroups
// that walk the table), HIP-graph replay of the step, and the autotuner of
// tile shapes and launch parameters.
//
// Pools: state[k] (k = 0..2, the rotating W^n / W* / W^{n+1} copies) holds
// the 8 fields of every box back to back (box b at BatchBox::off8, field f at
// off8 + f*ncell_b); flux holds the 21 face-flux arrays of every box.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <map>
#include <sstream>
#include <string>
#include <sys/stat.h>
#include <vector>

#include "capi_internal.h"

using namespace nmhd;

namespace {

// per thread: the message of the calling thread's last failed create
thread_local std::string g_batch_create_error;

constexpr int kZChunks[6] = {0, 2, 4, 8, 16, 32};  // 0: by default_chunk
constexpr int kWgPerCu[5] = {0, 1, 2, 3, 4};  // 0: one workgroup per item
constexpr size_t kStage = 1 << 18;  // floats of a half of the copy-out buffer
// Raised with any change of the batch kernels or of the default tiling, so that
// entries of other kernels are not found.
constexpr int kTuneVersion = 2;
constexpr int kTuneItems = 48;  // work items timed per shape and tile shape

}  // namespace

struct nmhd_batch {
  int nbox = 0;
  int device = 0;
  int cus = 256;
  std::string arch;
  hipStream_t stream = nullptr;
  std::vector<nmhd_desc> desc;
  std::vector<nmhd_geometry> geo;
  std::vector<BatchBox> boxes;
  BatchBox *d_boxes = nullptr;
  long total8 = 0, total21 = 0;
  float *state[3] = {};
  float *flux = nullptr;
  // step records: rec + k * nbox holds those of the steps that left state[k]
  StepState *rec = nullptr;
  StepState *st_tune = nullptr;
  float *d_goal = nullptr;
  int cur = 0;
  int integrator = NMHD_MIDPOINT2;
  std::vector<int> ftile, utile;
  // z chunks (0: by default_chunk) and workgroups per CU that walk the table
  // (0: one workgroup per work item)
  int fzc = 0, uzc = 0, fwg = 0, uwg = 0;
  WorkItem *d_fitems = nullptr, *d_uitems = nullptr, *d_titems = nullptr;
  int nf = 0, nu = 0;
  bool fwide = false;  // 64x4 tiles among the face items
  size_t cap_f = 0, cap_u = 0, cap_t = 0;
  bool items_dirty = true;
  bool cfl_valid = false;
  // blocks per box of the ghost fills and their CFL pass (0: no box has
  // that ghost layer)
  int grid_gy = 0, grid_gz = 0, grid_gcfl = 0;
  hipGraphExec_t exec[3] = {};
  // pinned halves through which get_state copies, with an event each (made by
  // its first call)
  float *stage[2] = {};
  hipEvent_t staged[2] = {};
  std::string err;
};

namespace {

int bfail(nmhd_batch *b, int code, const std::string &msg) {
  if (b)
    b->err = msg;
  else
    g_batch_create_error = msg;
  return code;
}

#define BHIP(b, call)                                                                   \
  do {                                                                                  \
    hipError_t e_ = (call);                                                             \
    if (e_ != hipSuccess)                                                               \
      return bfail((b), NMHD_EHIP, std::string(#call) + ": " + hipGetErrorString(e_));  \
  } while (0)

// Work items of the given boxes: tiles of tile shape tile[box], z chunks of
// zc planes, grouped by tile shape, then box by box, x fastest, then y, then z.
std::vector<WorkItem> make_items(const nmhd_batch *b, const std::vector<int> &tile, int zc,
                                 const std::vector<int> &which) {
  std::vector<WorkItem> out;
  for (int v = 0; v < TV_COUNT; ++v) {
    const int TX = kTileTX[v], TY = kTileTY[v];
    for (int box : which) {
      if (tile[box] != v) continue;
      const Box &bx = b->boxes[box].b;
      for (int z0 = 0; z0 < bx.n[2]; z0 += zc)
        for (int y0 = 0; y0 < bx.n[1]; y0 += TY)
          for (int x0 = 0; x0 < bx.n[0]; x0 += TX) {
            WorkItem w;
            w.box = box;
            w.xy = x0 | (y0 << 16);
            w.z = z0 | (std::min(z0 + zc, bx.n[2]) << 16);
            w.variant = v;
            out.push_back(w);
          }
    }
  }
  return out;
}

bool has_wide(const std::vector<WorkItem> &items) {
  for (const WorkItem &w : items)
    if (w.variant == TV_64x4) return true;
  return false;
}

// The chunk at which march_chunk expects a launch over every box's tiles to
// end first.  Chunks of 16 planes, as a large box would take, left 14 boxes of
// 16..96 cells per edge with one workgroup per CU: 291 us a step against 169;
// 64 such boxes, which fill the GPU either way, get them still.
int default_chunk(const nmhd_batch *b, bool faces) {
  const std::vector<int> &tile = faces ? b->ftile : b->utile;
  int nz = 1;
  for (const BatchBox &bb : b->boxes) nz = std::max(nz, bb.b.n[2]);
  const bool wide = std::find(tile.begin(), tile.end(), (int)TV_64x4) != tile.end();
  return march_chunk(faces, nz, march_per_cu(faces, wide), [&](int zc) {
    long n = 0;
    for (int i = 0; i < b->nbox; ++i) {
      const Box &x = b->boxes[i].b;
      const long tx = kTileTX[tile[i]], ty = kTileTY[tile[i]];
      n += (x.n[0] + tx - 1) / tx * ((x.n[1] + ty - 1) / ty) * ((x.n[2] + zc - 1) / zc);
    }
    return n;
  });
}
int faces_chunk(const nmhd_batch *b) { return b->fzc ? b->fzc : default_chunk(b, true); }
int update_chunk(const nmhd_batch *b) { return b->uzc ? b->uzc : default_chunk(b, false); }

void set_tiles(nmhd_batch *b, int box, int faces, int update) {
  const Box &x = b->boxes[box].b;
  b->ftile[box] = faces == kTileAuto ? tiled_shape(x.n[0], x.n[1], true) : faces;
  b->utile[box] = update == kTileAuto ? tiled_shape(x.n[0], x.n[1], false) : update;
}

std::vector<int> all_boxes(const nmhd_batch *b) {
  std::vector<int> v(b->nbox);
  for (int i = 0; i < b->nbox; ++i) v[i] = i;
  return v;
}

int upload_items(nmhd_batch *b, const std::vector<WorkItem> &items, WorkItem **dst,
                 size_t *cap) {
  if (items.size() > *cap) {
    if (*dst) BHIP(b, hipFree(*dst));
    *dst = nullptr;
    *cap = 0;
    BHIP(b, hipMalloc(dst, sizeof(WorkItem) * items.size()));
    *cap = items.size();
  }
  if (!items.empty())
    BHIP(b, hipMemcpyAsync(*dst, items.data(), sizeof(WorkItem) * items.size(),
                           hipMemcpyHostToDevice, b->stream));
  BHIP(b, hipStreamSynchronize(b->stream));
  return NMHD_OK;
}

void drop_graphs(nmhd_batch *b) {
  for (auto &e : b->exec)
    if (e) (void)hipGraphExecDestroy(e), e = nullptr;
}

int refresh_items(nmhd_batch *b) {
  if (!b->items_dirty) return NMHD_OK;
  const std::vector<int> all = all_boxes(b);
  const std::vector<WorkItem> f = make_items(b, b->ftile, faces_chunk(b), all);
  const std::vector<WorkItem> u = make_items(b, b->utile, update_chunk(b), all);
  int r = upload_items(b, f, &b->d_fitems, &b->cap_f);
  if (r) return r;
  r = upload_items(b, u, &b->d_uitems, &b->cap_u);
  if (r) return r;
  b->nf = (int)f.size();
  b->nu = (int)u.size();
  b->fwide = has_wide(f);
  drop_graphs(b);
  b->items_dirty = false;
  return NMHD_OK;
}

// workgroups that walk a table of nitems; 0 (wg_per_cu == 0): one per item
int grid_of(const nmhd_batch *b, int nitems, int wg_per_cu) {
  return std::min(nitems, wg_per_cu * b->cus);
}

// The two launches of a stage over the work tables, the states by their slots.
void enqueue_faces(nmhd_batch *b, int from, const BatchStep &step) {
  launch_batch_faces(b->stream, grid_of(b, b->nf, b->fwg), b->d_boxes, b->d_fitems, b->nf,
                     b->state[from], b->flux, step, b->fwide, streamed(b->total8 / 8));
}
void enqueue_update(nmhd_batch *b, int from, int base, int to, const BatchStep &step, bool last) {
  launch_batch_update(b->stream, grid_of(b, b->nu, b->uwg), b->d_boxes, b->d_uitems, b->nu,
                      b->state[from], b->flux, b->state[base], b->state[to], step, last,
                      streamed(b->total8 / 8));
}

// One iteration of the proceed() loop for every box.
void enqueue_step(nmhd_batch *b, bool full_cfl, float goal) {
  hipStream_t s = b->stream;
  const int A = b->cur, n = b->nbox;
  const int B = (A + 1) % 3, next = b->integrator == NMHD_EULER1 ? B : (A + 2) % 3;
  StepState *const in = b->rec + A * n, *const rec = b->rec + next * n;
  // ghost fills of the boxes that have ghost layers, then the CFL minimum:
  // a full pass, or the ghost cells added to the stage-2 epilogue's minimum
  if (b->grid_gy) launch_batch_ghost_y(s, b->d_boxes, n, b->grid_gy, b->state[A], in);
  if (b->grid_gz) launch_batch_ghost_z(s, b->d_boxes, n, b->grid_gz, b->state[A], in);
  if (full_cfl)
    launch_batch_cfl(s, b->d_boxes, n, b->state[A], goal, in);
  else if (b->grid_gcfl)
    launch_batch_cfl_ghosts(s, b->d_boxes, n, b->grid_gcfl, b->state[A], in);
  auto stage = [&](int from, int base, int to, int hsel, bool first, bool last) {
    enqueue_faces(b, from, BatchStep{rec, first ? in : nullptr, b->d_goal, hsel});
    enqueue_update(b, from, base, to, BatchStep{rec, nullptr, nullptr, hsel}, last);
  };
  if (b->integrator == NMHD_EULER1) {
    stage(A, A, next, H_FULL, true, true);
  } else {
    stage(A, A, B, H_HALF, true, false);
    stage(B, A, next, H_FULL, false, true);
  }
  b->cur = next;
}

int ensure_graph(nmhd_batch *b) {
  const int phase = b->cur;
  if (b->exec[phase]) return NMHD_OK;
  hipGraph_t g = nullptr;
  BHIP(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
  enqueue_step(b, false, 0.0f);
  const hipError_t e = hipStreamEndCapture(b->stream, &g);
  b->cur = phase;  // capture records; it does not advance the state
  if (e != hipSuccess)
    return bfail(b, NMHD_EHIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
  const hipError_t ei = hipGraphInstantiate(&b->exec[phase], g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (ei != hipSuccess) {
    b->exec[phase] = nullptr;
    return bfail(b, NMHD_EHIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(ei));
  }
  return NMHD_OK;
}

// The records as the last enqueued step leaves them, committed.
int read_records(nmhd_batch *b, std::vector<StepState> &h) {
  h.resize(b->nbox);
  BHIP(b, hipMemcpyAsync(h.data(), b->rec + b->cur * b->nbox, sizeof(StepState) * b->nbox,
                         hipMemcpyDeviceToHost, b->stream));
  BHIP(b, hipStreamSynchronize(b->stream));
  for (StepState &s : h)
    if (s.active) {
      s.t = s.t_next;
      s.generation += 1;
      s.steps_done += 1;
      s.active = 0;
    }
  return NMHD_OK;
}

int write_records(nmhd_batch *b, const std::vector<StepState> &h) {
  BHIP(b, hipMemcpyAsync(b->rec + b->cur * b->nbox, h.data(), sizeof(StepState) * b->nbox,
                         hipMemcpyHostToDevice, b->stream));
  BHIP(b, hipStreamSynchronize(b->stream));
  return NMHD_OK;
}

void free_batch(nmhd_batch *b) {
  drop_graphs(b);
  for (auto &p : b->state)
    if (p) (void)hipFree(p), p = nullptr;
  void *ptrs[] = {b->flux, b->rec, b->st_tune, b->d_goal, b->d_boxes,
                  b->d_fitems, b->d_uitems, b->d_titems};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  b->flux = nullptr;
  b->rec = b->st_tune = nullptr;
  b->d_goal = nullptr;
  b->d_boxes = nullptr;
  b->d_fitems = b->d_uitems = b->d_titems = nullptr;
  for (int i = 0; i < 2; ++i) {
    if (b->stage[i]) (void)hipHostFree(b->stage[i]), b->stage[i] = nullptr;
    if (b->staged[i]) (void)hipEventDestroy(b->staged[i]), b->staged[i] = nullptr;
  }
  if (b->stream) (void)hipStreamDestroy(b->stream), b->stream = nullptr;
}

// ------------------------------------------------------------ autotuner

std::string shape_key(const nmhd_batch *b, int box) {
  const Box &x = b->boxes[box].b;
  std::ostringstream o;
  o << x.n[0] << " " << x.n[1] << " " << x.n[2] << " " << x.recon << " " << x.source;
  return o.str();
}

std::string kernels_key(const nmhd_batch *b) {
  return b->arch + "/" + std::to_string(kTuneVersion) + " ";
}

std::string cache_file(const char *path) {
  if (path && *path) return path;
  const char *env = std::getenv("NMHD_TUNE_CACHE");
  if (env && *env) return env;
  const char *home = std::getenv("HOME");
  return std::string(home && *home ? home : ".") + "/.cache/nmhd_amd/batch_tuning.txt";
}

void make_parent_dirs(const std::string &file) {
  for (size_t i = 1; i < file.size(); ++i)
    if (file[i] == '/') (void)mkdir(file.substr(0, i).c_str(), 0755);
}

// Cache lines: "shape <arch> <nx> <ny> <nz> <recon> <source> : <faces> <update>"
// and "launch <arch> <hash> : <fzc> <uzc> <fwg> <uwg> <ftuned> <utuned>", the
// last two whether a kernel takes the tuned tile shapes (1) or the default ones;
// <arch> ends in the version of the kernels timed (kTuneVersion).
// Whether an entry read back holds as many values, each in 0..most.
bool within(const std::vector<int> &v, const std::vector<int> &most) {
  if (v.size() != most.size()) return false;
  for (size_t i = 0; i < v.size(); ++i)
    if (v[i] < 0 || v[i] > most[i]) return false;
  return true;
}
struct TuneCache {
  std::map<std::string, std::vector<int>> entries;
  void load(const std::string &file) {
    std::ifstream in(file);
    std::string line;
    while (std::getline(in, line)) {
      const size_t colon = line.find(" : ");
      if (line.empty() || line[0] == '#' || colon == std::string::npos) continue;
      std::istringstream vals(line.substr(colon + 3));
      std::vector<int> v;
      int x;
      while (vals >> x) v.push_back(x);
      entries[line.substr(0, colon)] = v;
    }
  }
  bool save(const std::string &file) const {
    make_parent_dirs(file);
    std::ofstream out(file, std::ios::trunc);
    if (!out) return false;
    out << "# nmhd batch autotuner cache (tile shapes per box shape, launch parameters)\n";
    for (auto &kv : entries) {
      out << kv.first << " :";
      for (int v : kv.second) out << " " << v;
      out << "\n";
    }
    return (bool)out;
  }
};

std::string launch_key(const nmhd_batch *b) {
  std::vector<std::string> shapes;
  for (int i = 0; i < b->nbox; ++i) shapes.push_back(shape_key(b, i));
  std::sort(shapes.begin(), shapes.end());
  unsigned long long h = 1469598103934665603ull;  // FNV-1a over the sorted shapes
  for (auto &s : shapes)
    for (char c : s + ";") h = (h ^ (unsigned char)c) * 1099511628211ull;
  char buf[64];
  std::snprintf(buf, sizeof(buf), "%016llx", h);
  return "launch " + kernels_key(b) + buf;
}

// Milliseconds of one launch of fn (after one untimed warm-up launch), the
// least of reps.
template <class F>
int time_launch(nmhd_batch *b, F &&fn, float *ms, int reps = 1) {
  hipEvent_t e0 = nullptr, e1 = nullptr;
  BHIP(b, hipEventCreate(&e0));
  BHIP(b, hipEventCreate(&e1));
  fn();
  *ms = 1e30f;
  for (int i = 0; i < reps; ++i) {
    float t = 0.0f;
    BHIP(b, hipEventRecord(e0, b->stream));
    fn();
    BHIP(b, hipEventRecord(e1, b->stream));
    BHIP(b, hipEventSynchronize(e1));
    BHIP(b, hipGetLastError());
    BHIP(b, hipEventElapsedTime(&t, e0, e1));
    *ms = std::min(*ms, t);
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return NMHD_OK;
}

const std::vector<int> kLaunchMost = {32767, 32767, 64, 64, 1, 1};

// How a batch is tiled (nmhd_batch's members of these names).
struct Tiling {
  std::vector<int> ftile, utile;
  int fzc = 0, uzc = 0, fwg = 0, uwg = 0;
  int ftuned = 0, utuned = 0;  // tile shapes: the timed ones
};

void set_tiling(nmhd_batch *b, const Tiling &t) {
  b->ftile = t.ftile;
  b->utile = t.utile;
  b->fzc = t.fzc;
  b->uzc = t.uzc;
  b->fwg = t.fwg;
  b->uwg = t.uwg;
  b->items_dirty = true;
}

int prepare_tune_records(nmhd_batch *b) {
  // every box active with a zero step: the update kernels then reproduce
  // the base state into the scratch rotation slot
  std::vector<StepState> h(b->nbox);
  std::memset(h.data(), 0, sizeof(StepState) * h.size());
  for (auto &s : h) {
    s.active = 1;
    s.cfl_bits = s.cfl_next_bits = 0x7f800000u;
  }
  BHIP(b, hipMemcpyAsync(b->st_tune, h.data(), sizeof(StepState) * h.size(),
                         hipMemcpyHostToDevice, b->stream));
  BHIP(b, hipStreamSynchronize(b->stream));
  return NMHD_OK;
}

int tune(nmhd_batch *b, const char *path, int *timed) {
  const std::string file = cache_file(path);
  TuneCache cache;
  cache.load(file);
  int r = prepare_tune_records(b);
  if (r) return r;
  float *in = b->state[b->cur];
  float *scratch = b->state[(b->cur + 1) % 3];
  const BatchStep step{b->st_tune, nullptr, nullptr, H_HALF};
  const bool nt = streamed(b->total8 / 8);
  int ntimed = 0;

  // the default tiling, and the tile shapes timed as the best
  Tiling plain, tuned;
  for (int i = 0; i < b->nbox; ++i) set_tiles(b, i, kTileAuto, kTileAuto);
  plain.ftile = tuned.ftile = b->ftile;
  plain.utile = tuned.utile = b->utile;
  tuned.ftuned = tuned.utuned = 1;

  // per shape: the workgroup-time of each tile shape
  std::map<std::string, std::vector<int>> groups;
  for (int i = 0; i < b->nbox; ++i) groups[shape_key(b, i)].push_back(i);
  for (auto &g : groups) {
    const std::string key = "shape " + kernels_key(b) + g.first;
    auto hit = cache.entries.find(key);
    if (hit == cache.entries.end() || !within(hit->second, {TV_COUNT - 1, TV_COUNT - 1})) {
      float best_f = 1e30f, best_u = 1e30f;
      int vf = TV_16x16, vu = TV_16x16;
      for (int v = 0; v < TV_COUNT; ++v) {
        std::vector<int> tile(b->nbox, v);
        std::vector<WorkItem> items = make_items(b, tile, 16, g.second);
        const double total = (double)items.size();
        if ((int)items.size() > kTuneItems) items.resize(kTuneItems);
        r = upload_items(b, items, &b->d_titems, &b->cap_t);
        if (r) return r;
        const int n = (int)items.size();
        float msf = 0.0f, msu = 0.0f;
        r = time_launch(
            b,
            [&] {
              launch_batch_faces(b->stream, 1, b->d_boxes, b->d_titems, n, in, b->flux, step,
                                 true, nt);
            },
            &msf);
        if (r) return r;
        r = time_launch(
            b,
            [&] {
              launch_batch_update(b->stream, 1, b->d_boxes, b->d_titems, n, in, b->flux, in,
                                  scratch, step, false, nt);
            },
            &msu);
        if (r) return r;
        const float cf = (float)(msf * total / n), cu = (float)(msu * total / n);
        if (cf < best_f) best_f = cf, vf = v;
        if (cu < best_u) best_u = cu, vu = v;
      }
      cache.entries[key] = {vf, vu};
      ++ntimed;
    }
    for (int box : g.second) {
      tuned.ftile[box] = cache.entries[key][0];
      tuned.utile[box] = cache.entries[key][1];
    }
  }

  // whole batch: tile shapes, z chunk and workgroups per CU of each kernel, the
  // faces' first, then the update's.  Each is timed as a step runs it: the
  // stages' launches, the last update with its CFL epilogue.  The default tiling
  // is kept unless another takes less than 0.99 of its time, of the kernel and
  // then of the whole step (timings of one tiling differ by that).
  const std::string lkey = launch_key(b);
  auto hit = cache.entries.find(lkey);
  if (hit == cache.entries.end() || !within(hit->second, kLaunchMost)) {
    const int cur = b->cur, one = (cur + 1) % 3, two = (cur + 2) % 3;
    const bool euler = b->integrator == NMHD_EULER1;
    auto faces = [&] {
      enqueue_faces(b, cur, step);
      if (!euler) enqueue_faces(b, one, step);
    };
    auto update = [&] {
      if (!euler) enqueue_update(b, cur, cur, one, step, false);
      enqueue_update(b, euler ? cur : one, cur, two, step, true);
    };
    auto whole = [&] {
      enqueue_faces(b, cur, step);
      enqueue_update(b, cur, cur, one, step, euler);
      if (euler) return;
      enqueue_faces(b, one, step);
      enqueue_update(b, one, cur, two, step, true);
    };
    auto time_tiling = [&](const Tiling &t, auto &&launches, float *ms) {
      set_tiling(b, t);
      const int rc = refresh_items(b);
      return rc ? rc : time_launch(b, launches, ms, 3);
    };
    Tiling best = plain;
    float whole_plain, whole_best, least;
    r = time_tiling(plain, whole, &whole_plain);
    if (r) return r;
    for (int kernel = 0; kernel < 2; ++kernel) {
      auto time_kernel = [&](const Tiling &t, float *ms) {
        return kernel == 0 ? time_tiling(t, faces, ms) : time_tiling(t, update, ms);
      };
      r = time_kernel(best, &least);
      if (r) return r;
      least *= 0.99f;
      for (const Tiling *tiles : {&plain, &tuned})
        for (int zc : kZChunks) {
          if (tiles == &tuned && (kernel == 0 ? tuned.ftile == plain.ftile
                                              : tuned.utile == plain.utile))
            break;
          for (int wg : kWgPerCu) {
            Tiling t = best;
            if (kernel == 0)
              t.ftile = tiles->ftile, t.fzc = zc, t.fwg = wg, t.ftuned = tiles->ftuned;
            else
              t.utile = tiles->utile, t.uzc = zc, t.uwg = wg, t.utuned = tiles->utuned;
            float ms;
            r = time_kernel(t, &ms);
            if (r) return r;
            if (ms < least) least = ms, best = t;
          }
        }
    }
    r = time_tiling(best, whole, &whole_best);
    if (r) return r;
    if (!(whole_best < 0.99f * whole_plain)) best = plain;
    cache.entries[lkey] = {best.fzc, best.uzc, best.fwg, best.uwg, best.ftuned, best.utuned};
  }
  const std::vector<int> &lp = cache.entries[lkey];
  set_tiling(b, Tiling{lp[4] ? tuned.ftile : plain.ftile, lp[5] ? tuned.utile : plain.utile,
                       lp[0], lp[1], lp[2], lp[3], lp[4], lp[5]});
  (void)cache.save(file);  // a read-only cache location only costs a re-tune
  if (timed) *timed = ntimed;
  return NMHD_OK;
}

// Whether a field is memory that the CPU reaches like any other, and whether it
// is pinned (its copies then need no buffer between).
struct HostMemory {
  bool plain, pinned;
};
HostMemory host_memory(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return {true, false};
  }
  if (a.type == hipMemoryTypeUnregistered) return {true, false};
  return {a.type == hipMemoryTypeHost, a.type == hipMemoryTypeHost};
}

bool box_ok(const nmhd_batch *b, int box) { return b && box >= 0 && box < b->nbox; }

}  // namespace

extern "C" {

const char *nmhd_batch_last_error(const nmhd_batch *b) {
  return b ? b->err.c_str() : g_batch_create_error.c_str();
}

int nmhd_batch_create(const nmhd_desc *descs, int nbox, nmhd_batch **out) {
  if (!descs || !out || nbox <= 0) return bfail(nullptr, NMHD_EINVAL, "bad argument");
  *out = nullptr;
  for (int i = 0; i < nbox; ++i) {
    std::string why;
    const nmhd_desc &d = descs[i];
    if (!desc_valid(&d, why)) return bfail(nullptr, NMHD_EINVAL, "box " + std::to_string(i) + ": " + why);
    if (d.integrator != descs[0].integrator)
      return bfail(nullptr, NMHD_EINVAL, "all boxes of a batch share one integrator");
    for (int a = 0; a < 3; ++a)
      if (d.global_size[a] + 2 * d.margin[a] > 32767)
        return bfail(nullptr, NMHD_EINVAL,
                     "batched boxes are at most 32767 cells per axis (ghosts included)");
  }
  nmhd_batch *b = new nmhd_batch();
  auto bail = [&](int code, const std::string &msg) {
    free_batch(b);
    delete b;
    return bfail(nullptr, code, msg);
  };
  b->nbox = nbox;
  b->integrator = descs[0].integrator;
  b->desc.assign(descs, descs + nbox);
  b->geo.resize(nbox);
  b->boxes.resize(nbox);
  b->ftile.resize(nbox);
  b->utile.resize(nbox);
  long off8 = 0, off21 = 0;
  for (int i = 0; i < nbox; ++i) {
    derive_box(&descs[i], b->boxes[i].b, b->geo[i]);
    b->boxes[i].off8 = off8;
    b->boxes[i].off21 = off21;
    off8 += 8 * b->boxes[i].b.ncell;
    off21 += 21 * b->boxes[i].b.ncell;
    set_tiles(b, i, kTileAuto, kTileAuto);
  }
  b->total8 = off8;
  b->total21 = off21;
  // ghost grids: blocks of 256 for the largest slab, at most 512 per box
  {
    long gy = 0, gz = 0, gc = 0;
    for (const BatchBox &bb : b->boxes) {
      const Box &x = bb.b;
      gy = std::max(gy, (long)x.n[0] * x.m[1] * x.n[2]);
      gz = std::max(gz, (long)x.n[0] * x.n[1] * x.m[2]);
      long c = 0;
      if (x.m[1]) c += (long)x.n[0] * 2 * x.m[1] * x.n[2];
      if (x.m[2]) c += (long)x.n[0] * x.n[1] * (2 * x.m[2] + 1);
      gc = std::max(gc, c);
    }
    auto blocks = [](long cells, long cap) {
      return cells == 0 ? 0 : (int)std::min(cap, (cells + 255) / 256);
    };
    b->grid_gy = blocks(gy, 512);
    b->grid_gz = blocks(gz, 512);
    // each block of the CFL pass ends in one atomic on its box's record
    b->grid_gcfl = blocks(gc / 4, 128);
  }
  if (hipGetDevice(&b->device) != hipSuccess) return bail(NMHD_EHIP, "no HIP device");
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, b->device) != hipSuccess)
    return bail(NMHD_EHIP, "hipGetDeviceProperties failed");
  b->cus = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
  b->arch = prop.gcnArchName;
  const size_t colon = b->arch.find(':');
  if (colon != std::string::npos) b->arch = b->arch.substr(0, colon);
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess)
    return bail(NMHD_EHIP, "hipStreamCreate failed");
  for (auto &p : b->state)
    if (hipMalloc(&p, sizeof(float) * (size_t)off8) != hipSuccess)
      return bail(NMHD_ENOMEM, "state pool allocation failed");
  if (hipMalloc(&b->flux, sizeof(float) * (size_t)off21) != hipSuccess)
    return bail(NMHD_ENOMEM, "flux pool allocation failed");
  if (hipMalloc(&b->rec, 3 * sizeof(StepState) * nbox) != hipSuccess ||
      hipMalloc(&b->st_tune, sizeof(StepState) * nbox) != hipSuccess ||
      hipMalloc(&b->d_goal, sizeof(float)) != hipSuccess ||
      hipMalloc(&b->d_boxes, sizeof(BatchBox) * nbox) != hipSuccess)
    return bail(NMHD_ENOMEM, "batch record allocation failed");
  for (auto &p : b->state)
    if (hipMemsetAsync(p, 0, sizeof(float) * (size_t)off8, b->stream) != hipSuccess)
      return bail(NMHD_EHIP, "state clear failed");
  std::vector<StepState> h(nbox);
  std::memset(h.data(), 0, sizeof(StepState) * nbox);
  for (auto &s : h) s.cfl_bits = s.cfl_next_bits = 0x7f800000u;
  if (hipMemcpyAsync(b->rec, h.data(), sizeof(StepState) * nbox, hipMemcpyHostToDevice,
                     b->stream) != hipSuccess ||
      hipMemcpyAsync(b->d_boxes, b->boxes.data(), sizeof(BatchBox) * nbox,
                     hipMemcpyHostToDevice, b->stream) != hipSuccess ||
      hipStreamSynchronize(b->stream) != hipSuccess)
    return bail(NMHD_EHIP, "batch record init failed");
  *out = b;
  return NMHD_OK;
}

int nmhd_batch_destroy(nmhd_batch *b) {
  if (!b) return NMHD_OK;
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  free_batch(b);
  delete b;
  return NMHD_OK;
}

int nmhd_batch_get_geometry(const nmhd_batch *b, int box, nmhd_geometry *geo) {
  if (!box_ok(b, box) || !geo) return NMHD_EINVAL;
  *geo = b->geo[box];
  return NMHD_OK;
}

int nmhd_batch_set_state(nmhd_batch *b, int box, const float *const fields[8]) {
  if (!box_ok(b, box) || !fields) return bfail(b, NMHD_EINVAL, "bad argument");
  for (int f = 0; f < 8; ++f)
    if (!fields[f]) return bfail(b, NMHD_EINVAL, "null field pointer");
  BHIP(b, hipStreamSynchronize(b->stream));
  const FieldPtrs W = box_fields(b->state[b->cur], b->boxes[box]);
  const size_t bytes = sizeof(float) * (size_t)b->boxes[box].b.ncell;
  for (int f = 0; f < 8; ++f)
    BHIP(b, hipMemcpyAsync(W.f[f], fields[f], bytes, hipMemcpyHostToDevice, b->stream));
  BHIP(b, hipStreamSynchronize(b->stream));
  b->cfl_valid = false;
  return NMHD_OK;
}

int nmhd_batch_get_state(nmhd_batch *b, int box, float *const fields[8]) {
  if (!box_ok(b, box) || !fields) return bfail(b, NMHD_EINVAL, "bad argument");
  for (int f = 0; f < 8; ++f)
    if (!fields[f]) return bfail(b, NMHD_EINVAL, "null field pointer");
  // Copies straight into the caller's arrays: where the CPU may not write them
  // and, from half a megabyte a field, where they are pinned (96^3 580 us against
  // 992 through the buffer, 256^3 9.5 ms against 18.2; 48^3 143 against 134).
  const size_t cells = (size_t)b->boxes[box].b.ncell;
  bool plain = true, pinned = true;
  for (int f = 0; f < 8; ++f) {
    const HostMemory m = host_memory(fields[f]);
    plain = plain && m.plain;
    pinned = pinned && m.pinned;
  }
  if (!plain || (pinned && 8 * cells > 4 * kStage)) {
    const FieldPtrs W = box_fields(b->state[b->cur], b->boxes[box]);
    for (int f = 0; f < 8; ++f)
      BHIP(b, hipMemcpyAsync(fields[f], W.f[f], sizeof(float) * cells, hipMemcpyDeviceToHost,
                             b->stream));
    BHIP(b, hipStreamSynchronize(b->stream));
    return NMHD_OK;
  }
  for (int i = 0; i < 2; ++i) {
    if (!b->stage[i]) BHIP(b, hipHostMalloc(&b->stage[i], kStage * sizeof(float)));
    if (!b->staged[i]) BHIP(b, hipEventCreateWithFlags(&b->staged[i], hipEventDisableTiming));
  }
  // The eight fields lie back to back: they come over in pieces, the next one
  // in flight while the last is spread over the caller's arrays.  A copy per
  // field into pageable memory took 30 us each whatever its size, 3.4 ms for
  // 14 boxes of 1.02M cells together; this takes 1.8 ms.
  const size_t n = cells, total = 8 * n;
  const float *src = b->state[b->cur] + b->boxes[box].off8;
  auto piece = [&](size_t k) { return std::min(kStage, total - k * kStage); };
  auto fetch = [&](size_t k) {
    const hipError_t e = hipMemcpyAsync(b->stage[k & 1], src + k * kStage,
                                        piece(k) * sizeof(float), hipMemcpyDeviceToHost, b->stream);
    return e == hipSuccess ? hipEventRecord(b->staged[k & 1], b->stream) : e;
  };
  const size_t pieces = (total + kStage - 1) / kStage;
  for (size_t k = 0; k < pieces && k < 2; ++k) BHIP(b, fetch(k));
  for (size_t k = 0; k < pieces; ++k) {
    BHIP(b, hipEventSynchronize(b->staged[k & 1]));
    const float *from = b->stage[k & 1];
    for (size_t at = k * kStage, end = at + piece(k); at < end;) {
      const size_t f = at / n, len = std::min((f + 1) * n, end) - at;
      std::memcpy(fields[f] + (at - f * n), from, len * sizeof(float));
      from += len, at += len;
    }
    if (k + 2 < pieces) BHIP(b, fetch(k + 2));
  }
  return NMHD_OK;
}

int nmhd_batch_set_time(nmhd_batch *b, int box, double t, int generation) {
  if (!box_ok(b, box)) return bfail(b, NMHD_EINVAL, "bad box");
  std::vector<StepState> h;
  int r = read_records(b, h);
  if (r) return r;
  StepState &s = h[box];
  std::memset(&s, 0, sizeof(s));
  s.t = t;
  s.t_next = t;
  s.generation = generation;
  s.cfl_bits = s.cfl_next_bits = 0x7f800000u;
  b->cfl_valid = false;
  return write_records(b, h);
}

int nmhd_batch_get_time(nmhd_batch *b, int box, double *t, int *generation) {
  if (!box_ok(b, box)) return bfail(b, NMHD_EINVAL, "bad box");
  std::vector<StepState> h;
  int r = read_records(b, h);
  if (r) return r;
  if (t) *t = h[box].t;
  if (generation) *generation = h[box].generation;
  return NMHD_OK;
}

int nmhd_batch_get_status(nmhd_batch *b, int box, int *steps_taken, int *goal_reached,
                          float *last_dt) {
  if (!box_ok(b, box)) return bfail(b, NMHD_EINVAL, "bad box");
  std::vector<StepState> h;
  int r = read_records(b, h);
  if (r) return r;
  if (steps_taken) *steps_taken = h[box].steps_done;
  if (goal_reached) *goal_reached = h[box].goal_reached;
  if (last_dt) *last_dt = h[box].dt;
  return NMHD_OK;
}

int nmhd_batch_set_tiles(nmhd_batch *b, int box, int faces_tile, int update_tile) {
  if (!b || box < -1 || box >= b->nbox || faces_tile < kTileAuto || faces_tile >= TV_COUNT ||
      update_tile < kTileAuto || update_tile >= TV_COUNT)
    return bfail(b, NMHD_EINVAL, "bad tile selection");
  for (int i = 0; i < b->nbox; ++i)
    if (box == -1 || box == i) set_tiles(b, i, faces_tile, update_tile);
  b->items_dirty = true;
  return NMHD_OK;
}

int nmhd_batch_set_launch(nmhd_batch *b, int fzc, int uzc, int fwg, int uwg) {
  if (!b || fzc < 0 || uzc < 0 || fzc > 32767 || uzc > 32767 || fwg < 0 || uwg < 0 || fwg > 64 ||
      uwg > 64)
    return bfail(b, NMHD_EINVAL, "bad launch parameters");
  b->fzc = fzc;
  b->uzc = uzc;
  b->fwg = fwg;
  b->uwg = uwg;
  b->items_dirty = true;
  return NMHD_OK;
}

int nmhd_batch_get_launch(const nmhd_batch *b, int *fzc, int *uzc, int *fwg, int *uwg) {
  if (!b) return NMHD_EINVAL;
  if (fzc) *fzc = faces_chunk(b);
  if (uzc) *uzc = update_chunk(b);
  if (fwg) *fwg = b->fwg;
  if (uwg) *uwg = b->uwg;
  return NMHD_OK;
}

int nmhd_batch_autotune(nmhd_batch *b, const char *cache_path, int *timed_shapes) {
  if (!b) return NMHD_EINVAL;
  BHIP(b, hipStreamSynchronize(b->stream));
  return tune(b, cache_path, timed_shapes);
}

int nmhd_batch_run(nmhd_batch *b, float goal_time, int nsteps, int use_graph, int *min_steps,
                   int *all_reached) {
  if (!b || nsteps < 0) return bfail(b, NMHD_EINVAL, "bad argument");
  std::vector<StepState> h;
  int r = read_records(b, h);
  if (r) return r;
  for (auto &s : h) {
    s.finished = s.goal_reached = s.steps_done = 0;
    if (!b->cfl_valid) s.cfl_next_bits = 0x7f800000u;  // for the full pass
  }
  r = write_records(b, h);
  if (r) return r;
  r = refresh_items(b);
  if (r) return r;
  BHIP(b, hipMemcpyAsync(b->d_goal, &goal_time, sizeof(float), hipMemcpyHostToDevice,
                         b->stream));
  for (int k = 0; k < nsteps; ++k) {
    if (!b->cfl_valid) {
      enqueue_step(b, true, goal_time);
      b->cfl_valid = true;
    } else if (use_graph) {
      r = ensure_graph(b);
      if (r) return r;
      BHIP(b, hipGraphLaunch(b->exec[b->cur], b->stream));
      b->cur = b->integrator == NMHD_EULER1 ? (b->cur + 1) % 3 : (b->cur + 2) % 3;
    } else {
      enqueue_step(b, false, goal_time);
    }
  }
  BHIP(b, hipGetLastError());
  r = read_records(b, h);
  if (r) return r;
  int mn = nsteps, all = 1;
  for (auto &s : h) {
    mn = std::min(mn, s.steps_done);
    all = all && s.goal_reached;
  }
  if (min_steps) *min_steps = mn;
  if (all_reached) *all_reached = all;
  return NMHD_OK;
}

}  // extern "C"
