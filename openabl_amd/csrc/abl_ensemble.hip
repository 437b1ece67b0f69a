// abl_ensemble.hip -- many independent runs of one program batched into one
// launch per kernel, with one timestep captured as a HIP graph.
//
// Members (uneven agent counts, per-member parameters such as box size and
// flocking weights) are stored back to back in one set of columns; member m
// owns slots [off[m], off[m+1]) and the grid cells [cell_base[m],
// cell_base[m+1]), laid out member-major, so one counting sort over all cells
// keeps every member cell-sorted inside its own slot range.  The neighbour
// kernel is the program's LDS-tiled kernel over the concatenated tile list
// (tiled_step_multi); each block finds its member and reads that member's
// arguments through the scalar cache.  A member's agents are ordered, and its
// neighbours visited, exactly as in a run of it alone, so each member's result
// is bit-identical to that run.
//
// Neighbour lists ("hip.nlist", default on when the members share the near
// radius): one set of lists over the concatenated slots, built after a sort
// and walked while no agent of the member has moved more than skin / 2 since
// (abl_tile.hpp).  Each member has its own rebuild gate, set by its own
// agents, and its own list capacity, so it rebuilds, and enters its lists anew with
// more room, on exactly the timesteps a run of it alone would.
// Re-sort and list build are one launch that returns at once when no member is
// due (tiled_rebuild_multi); it re-sorts the agents of the members due by the
// delta method into the other buffers, and the list build copies them back, so
// the step always reads the current buffers.
//
// With static populations every timestep issues the same kernels on the same
// buffers (without lists the grid gather and the step each flip the columns;
// with lists the step flips them, and two timesteps return to the start): two
// timesteps are captured once as a graph and replayed.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/abl_hip.h"
#include "abl_pipeline.hpp"
#include "abl_runtime.hpp"

using namespace abl;

namespace {

thread_local std::string g_ens_error;

int ens_fail(int code, const std::string &msg) {
  g_ens_error = msg;
  return code;
}

#define ENS_TRY(call)                                                              \
  do {                                                                             \
    hipError_t e_ = (call);                                                        \
    if (e_ != hipSuccess) {                                                        \
      return ens_fail(ABL_ERR_DEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
    }                                                                              \
  } while (0)

struct Member {
  int n = 0;
  uint32_t off = 0;
  std::vector<double> params;
  GridView g{};
  uint32_t cell_base = 0, tile_base = 0, ntiles = 0;
  double cell = 0.0;
  float near_t = 0.f, rc = 0.f;
  // lists: estimated entries per agent, the capacity, and when to look at them
  int est = 0, cap = 0;
  ListWatch watch;
};

// Every slot's cell key.
template <typename P>
__global__ void k_ens_bin(const P *__restrict__ px, const P *__restrict__ py, EnsTiles e,
                          uint32_t *__restrict__ key, uint32_t *__restrict__ count, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int m = member_of(e.off, e.members, (uint32_t) i);
  const uint32_t k = e.cell_base[m] + cell_key<P>(e.grids[m], px, py, (const P *) nullptr, i);
  key[i] = k;
  atomicAdd(&count[k], 1u);
}

// The phases of the gated re-sort as launches of their own (issue_rebuild): the
// slots of the members due are binned, and placed.
template <typename P>
__global__ __launch_bounds__(256) void k_ens_delta(DeltaArgs d, EnsTiles e, const uint32_t *gate,
                                                   int parity, int phase) {
  if (gate[parity] == 0u) return;
  const int i = (int) (blockIdx.x * 256u + threadIdx.x);
  if (i >= d.n) return;
  const int m = member_of(e.off, e.members, (uint32_t) i);
  if (e.mgate[parity * e.members + m] == 0u) return;
  const uint32_t gen = gate[kGateGen];
  if (phase == 0)
    bin_delta_item(i, e.cell_base[m] + cell_key<P>(e.grids[m], (const P *) d.px, (const P *) d.py,
                                                   (const P *) nullptr, i),
                   d.skey, d.key, d.count, d.bsum, d.ml, gen);
  else
    place_item(i, d.key, d.skey, d.skey_out, d.start_old, d.start_new, d.ml, gen, d.gc, d.id_in,
               d.id_out, d.n);
}

// slot s of member m back to record id within that member's output block
__global__ void k_ens_unpermute(char *__restrict__ aos, ColSet cols, int elem, int ncols,
                                const int32_t *__restrict__ id, uint32_t begin, int n) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const uint32_t s = begin + (uint32_t) k;
  char *rec = aos + (size_t) id[s] * (size_t) (elem * ncols);
  for (int c = 0; c < ncols; c++) {
    if (elem == 8) ((double *) rec)[c] = ((const double *) cols.c[c])[s];
    else ((float *) rec)[c] = ((const float *) cols.c[c])[s];
  }
}

}  // namespace

struct abl_ensemble {
  const ProgramDesc *prog = nullptr;
  const EnsembleHooks *hooks = nullptr;
  int precision = 0;
  std::vector<Member> mem;
  size_t n = 0;
  int ncols = 0, elem = 8;
  void *col[2][kMaxCols] = {};
  int cur = 0;
  int32_t *id[2] = {nullptr, nullptr};
  int id_cur = 0;
  uint32_t *d_off = nullptr, *d_cell_base = nullptr;
  uint2 *d_tile_of = nullptr;
  GridView *d_grids = nullptr;
  void *d_args[2] = {nullptr, nullptr};  // member arguments for cur = 0 / cur = 1
  void *d_build[2] = {nullptr, nullptr};  // lists: the same on the rebuild's cell offsets
  uint32_t *key = nullptr, *count = nullptr, *start = nullptr, *bsum = nullptr, *tmp_idx = nullptr;
  int32_t *tmp_id = nullptr;
  size_t ncells = 0;
  unsigned total_tiles = 0;
  int reach = 1;
  float occupancy = 0.f;
  int cell_scale = 2, tile = 1, block = 256;
  bool use_graph = true;
  bool ready = false;
  uint64_t timestep = 0;       // timesteps issued (the lists' gates go by its parity)
  // neighbour lists
  bool nlist = true;           // "hip.nlist": lists when the members share the near radius
  double skin = kDefaultSkin;  // "hip.skin": list skin as a fraction of the near radius
  int list_cap = 0;            // "hip.list_cap": entries per list (0: sized from the data)
  bool lists = false;          // in use (decided by abl_ens_init)
  double r = 0.0, rl = 0.0, cell = 0.0;
  int nl_cap = 0;              // entries per agent allocated, at least the largest member's capacity
  uint16_t *nl_idx = nullptr, *nl_len = nullptr;
  uint32_t *nl_perm = nullptr;
  uint4 *nl_prow0 = nullptr;
  double *nl_pos0 = nullptr;
  uint32_t *nl_gate = nullptr;   // [0..1] some member due, by parity; error flag, generation
                                 // and queues (abl_pipeline.hpp)
  uint32_t *nl_mgate = nullptr;  // [2][members] member due, by parity
  uint32_t *nl_mcap = nullptr;   // [members] capacities; [members] lists to be entered anew
  uint32_t *nl_mlong = nullptr;  // [members] EnsTiles::mlong
  uint32_t *skey[2] = {nullptr, nullptr};  // each slot's cell key at the last sort; the rebuild's
  uint32_t *start_new = nullptr;           // the rebuild's cell offsets
  uint32_t *dirty = nullptr;               // MoverLists
  unsigned long long *mhead = nullptr, *mnext = nullptr;
  uint32_t *h_error = nullptr;   // pinned copy of the error flag as of the last simulate()
  // what look() asked for: pinned copies of the generation and of nl_mlong after a
  // timestep, in the slot of that timestep (answers are read kListSample later)
  static constexpr uint64_t kSlots = 2 * kListSample;
  uint32_t *h_look = nullptr;    // [kSlots][1 + members]
  hipEvent_t look_ev[kSlots] = {};
  uint64_t next_look = 0;        // the timestep after which look() has something to do
  ListWatch watch;               // the ensemble's own: the number of rebuilds
  std::vector<int> entering;     // members whose lists are entered anew at the next timestep
  // four launches per rebuild instead of one: many timesteps rebuild
  bool split = false;
  uint32_t gen_seen = 1;
  // download workspace: one member's records, grown to the largest asked for
  std::mutex dl_lock;
  void *dl = nullptr;
  size_t dl_bytes = 0;
  hipStream_t stream = nullptr;
  // two timesteps, captured with one launch per rebuild and with four
  hipGraphExec_t exec[2] = {nullptr, nullptr};
  hipGraph_t graph[2] = {nullptr, nullptr};
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  double last_ms = 0.0;
};

extern "C" const char *abl_ens_last_error(void) { return g_ens_error.c_str(); }

// Member m's generator start state: the base state with its first word mixed
// with m, so members draw independent, reproducible streams.
extern "C" int abl_ens_member_seed(uint64_t s0, uint64_t s1, int member, uint64_t out[2]) {
  if (!out || member < 0) return ens_fail(ABL_ERR_ARG, "bad argument");
  out[0] = s0 ^ (0x9E3779B97F4A7C15ULL * (uint64_t) (member + 1));
  out[1] = s1;
  if (out[0] == 0 && out[1] == 0) out[1] = 1;
  return ABL_OK;
}

extern "C" int abl_ens_create(const char *program, int precision, int members,
                              const int *counts, int num_params, const char *const *names,
                              const double *values, abl_ensemble **out) {
  if (!program || !out || members < 1 || !counts || (num_params && (!names || !values)))
    return ens_fail(ABL_ERR_ARG, "bad argument");
  *out = nullptr;
  const ProgramDesc *prog = find_program(program);
  if (!prog) return ens_fail(ABL_ERR_ARG, no_program(program));
  if (!prog->ensemble) return ens_fail(ABL_ERR_UNSUPPORTED, "program has no ensemble support");
  if (precision != ABL_PREC_F64 && precision != ABL_PREC_F32)
    return ens_fail(ABL_ERR_UNSUPPORTED, "precision not supported");
  abl_ensemble *e = new abl_ensemble();
  e->prog = prog;
  e->hooks = prog->ensemble;
  e->precision = precision;
  e->mem.resize((size_t) members);
  for (int m = 0; m < members; m++) {
    Member &mb = e->mem[(size_t) m];
    for (const ParamDesc &p : prog->params) mb.params.push_back(p.value);
    for (int k = 0; k < num_params; k++) {
      bool found = false;
      for (size_t p = 0; p < prog->params.size(); p++) {
        if (std::strcmp(prog->params[p].name, names[k]) == 0) {
          mb.params[p] = values[(size_t) m * (size_t) num_params + (size_t) k];
          found = true;
        }
      }
      if (!found) {
        delete e;
        return ens_fail(ABL_ERR_ARG, std::string("Unknown parameter \"") + names[k] + "\"");
      }
    }
    mb.n = counts[m];
  }
  e->elem = precision == ABL_PREC_F64 ? 8 : 4;
  int ncols = 0;
  for (const MemberDesc &md : prog->agents[0].members) ncols += kind_components(md.kind);
  e->ncols = ncols;
  if (hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&e->ev0) != hipSuccess || hipEventCreate(&e->ev1) != hipSuccess) {
    delete e;
    return ens_fail(ABL_ERR_DEVICE, "stream/event creation failed");
  }
  *out = e;
  return ABL_OK;
}

extern "C" int abl_ens_set_config(abl_ensemble *e, const char *key, const char *value) {
  if (!e || !key || !value) return ens_fail(ABL_ERR_ARG, "bad argument");
  if (e->ready) return ens_fail(ABL_ERR_STATE, "configure before abl_ens_init");
  std::string k(key), v(value);
  if (k == "hip.cell_scale") {
    e->cell_scale = std::max(1, std::min(4, std::atoi(value)));
  } else if (k == "hip.tile") {
    e->tile = std::max(1, std::min(3, std::atoi(value)));
  } else if (k == "hip.block") {
    int b = std::atoi(value);
    if (b < 64 || b > 256 || b % 64) return ens_fail(ABL_ERR_ARG, "hip.block must be 64..256");
    e->block = b;
  } else if (k == "hip.graph") {
    e->use_graph = v == "1" || v == "true";
  } else if (k == "hip.nlist") {
    if (v != "0" && v != "1") return ens_fail(ABL_ERR_ARG, "hip.nlist must be 0 or 1");
    e->nlist = v == "1";
  } else if (k == "hip.skin") {
    const double f = std::atof(value);
    if (!(f > 0.0 && f <= 1.0)) return ens_fail(ABL_ERR_ARG, "hip.skin must be in (0, 1]");
    e->skin = f;
  } else if (k == "hip.list_cap") {
    const int c = std::atoi(value);
    if (c < 0 || c > 65528) return ens_fail(ABL_ERR_ARG, "hip.list_cap must be 0..65528");
    e->list_cap = c;
  } else {
    return ens_fail(ABL_ERR_ARG, "unknown config key " + k);
  }
  return ABL_OK;
}

static void drop_graphs(abl_ensemble *e) {
  for (int k = 0; k < 2; k++) {
    if (e->exec[k]) (void) hipGraphExecDestroy(e->exec[k]);
    if (e->graph[k]) (void) hipGraphDestroy(e->graph[k]);
    e->exec[k] = nullptr;
    e->graph[k] = nullptr;
  }
}

static void free_all(abl_ensemble *e) {
  for (int b = 0; b < 2; b++) {
    for (int c = 0; c < kMaxCols; c++) {
      if (e->col[b][c]) (void) hipFree(e->col[b][c]);
      e->col[b][c] = nullptr;
    }
    if (e->id[b]) (void) hipFree(e->id[b]);
    if (e->d_args[b]) (void) hipFree(e->d_args[b]);
    if (e->d_build[b]) (void) hipFree(e->d_build[b]);
    e->id[b] = nullptr;
    e->d_args[b] = e->d_build[b] = nullptr;
  }
  auto drop = [](auto &q) {
    if (q) (void) hipFree(q);
    q = nullptr;
  };
  drop(e->d_off);
  drop(e->d_cell_base);
  drop(e->d_tile_of);
  drop(e->d_grids);
  drop(e->key);
  drop(e->count);
  drop(e->start);
  drop(e->bsum);
  drop(e->tmp_idx);
  drop(e->tmp_id);
  drop(e->nl_idx);
  drop(e->nl_len);
  drop(e->nl_perm);
  drop(e->nl_prow0);
  drop(e->nl_pos0);
  drop(e->nl_gate);
  drop(e->nl_mgate);
  drop(e->nl_mcap);
  drop(e->nl_mlong);
  drop(e->skey[0]);
  drop(e->skey[1]);
  drop(e->start_new);
  drop(e->dirty);
  drop(e->mhead);
  drop(e->mnext);
  drop(e->dl);
  e->dl_bytes = 0;
  if (e->h_error) (void) hipHostFree(e->h_error);
  if (e->h_look) (void) hipHostFree(e->h_look);
  e->h_error = e->h_look = nullptr;
  for (hipEvent_t &ev : e->look_ev) {
    if (ev) (void) hipEventDestroy(ev);
    ev = nullptr;
  }
  drop_graphs(e);
}

// The list arguments of the current timestep (as a run alone forms them).
static NListArgs ens_list_args(const abl_ensemble *e) {
  NListArgs nl{};
  nl.idx = e->nl_idx;
  nl.len = e->nl_len;
  nl.perm = e->nl_perm;
  nl.prow0 = e->nl_prow0;
  nl.pos0 = e->nl_pos0;
  nl.gate = e->nl_gate;
  nl.stats = e->nl_gate + 2;
  nl.n = (int) e->n;
  nl.cap = e->nl_cap;
  nl.stride = (int) e->n;
  nl.parity = (int) (e->timestep & 1u);
  nl.rc_list = (float) (e->rl / e->cell * (1.0 + 1.0 / 1048576.0));
  const double rw = e->rl * (1.0 + 1e-6) + 1e-5 * e->r;
  nl.r2_list = rw * rw;
  const double h = 0.5 * (e->rl - e->r);
  nl.half_skin2 = h * h;
  nl.ncells = (int) e->ncells;
  return nl;
}

static EnsTiles ens_tiles(const abl_ensemble *e) {
  EnsTiles t{};
  t.tile_of = e->d_tile_of;
  t.off = e->d_off;
  t.cell_base = e->d_cell_base;
  t.grids = e->d_grids;
  t.mgate = e->nl_mgate;
  t.mcap = e->nl_mcap;
  t.mlong = e->nl_mlong;
  t.members = (int) e->mem.size();
  t.total = e->total_tiles;
  return t;
}

static GatherCols ens_gather(const abl_ensemble *e, int from) {
  GatherCols gc{};
  gc.ncols = e->ncols;
  for (int c = 0; c < e->ncols; c++) {
    gc.src[c] = e->col[from][c];
    gc.dst[c] = e->col[1 - from][c];
    gc.elem[c] = e->elem;
  }
  return gc;
}

// The full sort of every slot into the other buffers: cell offsets to `start`;
// keys and restored counts where asked for.
static void issue_sort(abl_ensemble *e, uint32_t *start, uint32_t *skey_out, uint32_t *count_out) {
  const int n = (int) e->n;
  const int nc = (int) e->ncells;
  hipStream_t st = e->stream;
  const int b = e->cur;
  const EnsTiles t = ens_tiles(e);
  if (n > 0) {
    if (e->elem == 8)
      hipLaunchKernelGGL(k_ens_bin<double>, grid_blocks(n, 256), 256, 0, st,
                         (const double *) e->col[b][0], (const double *) e->col[b][1], t, e->key,
                         e->count, n);
    else
      hipLaunchKernelGGL(k_ens_bin<float>, grid_blocks(n, 256), 256, 0, st,
                         (const float *) e->col[b][0], (const float *) e->col[b][1], t, e->key,
                         e->count, n);
  }
  const int ntiles = (nc + kScanTile - 1) / kScanTile;
  hipLaunchKernelGGL(k_scan_tiles, ntiles, kScanBlock, 0, st, e->count, start, e->bsum, nc);
  hipLaunchKernelGGL(k_scan_totals, 1, 1024, 0, st, e->bsum, ntiles, start, nc);
  hipLaunchKernelGGL(k_scan_add, grid_blocks(nc, 256), 256, 0, st, start, e->bsum, nc);
  if (n > 0) {
    hipLaunchKernelGGL(k_scatter, grid_blocks(n, 256), 256, 0, st, e->key, e->count, start,
                       e->id[e->id_cur], e->tmp_idx, e->tmp_id, n);
    hipLaunchKernelGGL(k_rank_gather, grid_blocks(n, 256), 256, 0, st, e->tmp_idx, e->tmp_id,
                       e->key, start, ens_gather(e, b), e->id[1 - e->id_cur], n, skey_out,
                       count_out);
  }
}

// The list build's arguments: from the rebuild's buffers, its agents copied back
// to the current ones.
static NListArgs ens_build_args(const abl_ensemble *e) {
  NListArgs nl = ens_list_args(e);
  nl.copy = ens_gather(e, 1 - e->cur);
  nl.id_src = e->id[1 - e->id_cur];
  nl.id_dst = e->id[e->id_cur];
  nl.skey_src = e->skey[1];
  nl.skey_dst = e->skey[0];
  nl.start_src = e->start_new;
  nl.start_dst = e->start;
  return nl;
}

// The gated list build of the members due, their agents sorted already.
static int issue_build(abl_ensemble *e) {
  NListArgs nl = ens_build_args(e);
  nl.gated = 1;
  const int rc = e->hooks->launch_multi_list(e->precision, e->d_build[e->cur], ens_tiles(e), e->reach,
                                             e->occupancy, e->tile, e->block, e->stream, nl, nullptr, 1);
  return rc ? ens_fail(rc, "list build") : ABL_OK;
}

// The gated rebuild of the current timestep: one launch (tiled_rebuild_multi), or
// four (look), which cost a timestep without a rebuild about 10 us more and one
// on which all members rebuild half (tiled_rebuild_multi); the same results.
static int issue_rebuild(abl_ensemble *e) {
  DeltaArgs d{};
  const int b = e->cur;
  d.px = e->col[b][0];
  d.py = e->col[b][1];
  d.pos_elem = e->elem;
  d.skey = e->skey[0];
  d.key = e->key;
  d.count = e->count;
  d.bsum = e->bsum;
  d.ml = MoverLists{e->dirty, e->mhead, e->mnext};
  d.n = (int) e->n;
  d.start_old = e->start;
  d.start_new = e->start_new;
  d.ncells = (int) e->ncells;
  d.nscan = ((int) e->ncells + kScanTile - 1) / kScanTile;
  d.skey_out = e->skey[1];
  d.gc = ens_gather(e, b);
  d.id_in = e->id[e->id_cur];
  d.id_out = e->id[1 - e->id_cur];
  RebuildQueue *queues = reinterpret_cast<RebuildQueue *>(e->nl_gate + kGateQueue);
  d.q = queues + (e->timestep & 1u);
  d.q_other = queues + (~e->timestep & 1u);
  d.error = e->nl_gate + kGateError;
  d.spins = kPhaseSpins;
  NListArgs nl = ens_build_args(e);
  nl.gated = 1;
  const EnsTiles t = ens_tiles(e);
  if (e->split) {
    const auto delta = e->elem == 8 ? k_ens_delta<double> : k_ens_delta<float>;
    hipLaunchKernelGGL(delta, grid_blocks(d.n, 256), 256, 0, e->stream, d, t, nl.gate, nl.parity, 0);
    hipLaunchKernelGGL(k_scan_apply, d.nscan, kScanBlock, 0, e->stream, e->count, e->bsum,
                       e->start_new, d.ncells, nl.gate + nl.parity);
    hipLaunchKernelGGL(delta, grid_blocks(d.n, 256), 256, 0, e->stream, d, t, nl.gate, nl.parity, 2);
    return issue_build(e);
  }
  const int rc = e->hooks->launch_multi_list(e->precision, e->d_build[b], t, e->reach, e->occupancy,
                                             e->tile, e->block, e->stream, nl, &d, 3);
  return rc ? ens_fail(rc, "list rebuild: no launch size") : ABL_OK;
}

// Entry lists for the largest capacity; those of members that keep theirs stay
// (rows of eight entries of all agents, so more rows go behind).  Twice the rows
// asked for, where lists may grow: an allocation and captures anew, since the
// captured timesteps hold the address, cost 4 ms for 470,000 agents, as much as
// 100 timesteps.
static int reserve_entries(abl_ensemble *e) {
  int cap = 0;
  for (const Member &mb : e->mem) cap = std::max(cap, mb.cap);
  if (cap <= e->nl_cap) return ABL_OK;
  if (!e->list_cap) cap = list_capacity(2 * cap);
  uint16_t *idx = nullptr;
  ENS_TRY(hipMalloc(&idx, (size_t) cap * e->n * 2));
  if (e->nl_idx) {
    hipError_t err = hipMemcpyAsync(idx, e->nl_idx, (size_t) e->nl_cap * e->n * 2,
                                    hipMemcpyDeviceToDevice, e->stream);
    if (err == hipSuccess) err = hipStreamSynchronize(e->stream);
    if (err != hipSuccess) {
      (void) hipFree(idx);
      ENS_TRY(err);
    }
    ENS_TRY(hipFree(e->nl_idx));
  }
  e->nl_idx = idx;
  e->nl_cap = cap;
  drop_graphs(e);
  return ABL_OK;
}

// The capacities, and which members enter their lists anew, to the device.
static int put_capacities(abl_ensemble *e) {
  const size_t M = e->mem.size();
  std::vector<uint32_t> words(2 * M, 0u);
  for (size_t m = 0; m < M; m++) words[m] = (uint32_t) e->mem[m].cap;
  for (const int m : e->entering) words[M + (size_t) m] = 1u;
  ENS_TRY(hipMemcpyAsync(e->nl_mcap, words.data(), 2 * M * 4, hipMemcpyHostToDevice, e->stream));
  ENS_TRY(hipStreamSynchronize(e->stream));
  return ABL_OK;
}

// More room for the lists of member m, as a run alone makes it (enter_lists);
// whether there is any.
static bool grow_lists(const abl_ensemble *e, Member &mb, uint32_t longest) {
  const int room = list_room(mb.est, longest);
  if (e->list_cap || (int64_t) longest <= mb.cap || room <= mb.cap || mb.cap >= kListMost) return false;
  mb.cap = list_capacity(room);
  return true;
}

// Sets the members entering their lists due, nothing counted of them yet.
__global__ void k_ens_enter(const uint32_t *__restrict__ enter, int members, int parity,
                            uint32_t *__restrict__ gate, uint32_t *__restrict__ mgate,
                            uint32_t *__restrict__ mlong) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= members || !enter[m]) return;
  gate[parity] = 1u;
  mgate[parity * members + m] = 1u;
  mlong[m] = 0u;
}

// The rebuild of the current timestep where some members enter their lists anew
// (look): those are due whatever their agents did, get the capacity that look()
// gave them, and once more room if their lists have outgrown that meanwhile.  A
// run alone enters list mode like that, so its lists, and the order it adds its
// neighbours in, stay the member's.
static int enter_members(abl_ensemble *e) {
  const int M = (int) e->mem.size();
  int rc = reserve_entries(e);
  if (!rc) rc = put_capacities(e);
  if (rc) return rc;
  const int parity = (int) (e->timestep & 1u);
  hipLaunchKernelGGL(k_ens_enter, grid_blocks(M, 256), 256, 0, e->stream, e->nl_mcap + M, M, parity,
                     e->nl_gate, e->nl_mgate, e->nl_mlong);
  rc = issue_rebuild(e);
  if (rc) return rc;
  std::vector<uint32_t> longest((size_t) M);
  ENS_TRY(hipMemcpyAsync(longest.data(), e->nl_mlong, (size_t) M * 4, hipMemcpyDeviceToHost, e->stream));
  ENS_TRY(hipStreamSynchronize(e->stream));
  bool again = false;
  for (const int m : e->entering) {
    Member &mb = e->mem[(size_t) m];
    again = grow_lists(e, mb, longest[(size_t) m]) || again;
    mb.watch.entered(e->timestep);
    e->next_look = std::min(e->next_look, mb.watch.next());
  }
  if (again) {
    rc = reserve_entries(e);
    if (!rc) rc = put_capacities(e);
    if (!rc) rc = issue_build(e);
  }
  e->entering.clear();
  return rc;
}

// The generation and the members' longest lists to pinned memory: a copy command
// between kernels holds the stream up for some 20 us, twice what this launch takes.
__global__ void k_ens_tell(const uint32_t *__restrict__ gen, const uint32_t *__restrict__ mlong,
                           int members, uint32_t *__restrict__ out) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m == 0) __hip_atomic_store(out, *gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  if (m < members) __hip_atomic_store(out + 1 + m, mlong[m], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// List buffers, and every member's first sort and lists, as a run alone enters
// list mode: capacity "hip.list_cap", or from the expected population of the
// list radius, grown once to the longest list.
static int init_lists(abl_ensemble *e) {
  const size_t N = e->n;
  const size_t M = e->mem.size();
  for (Member &mb : e->mem) {
    mb.est = list_estimate(2, (size_t) mb.g.n[0] * (size_t) mb.g.n[1], mb.cell, (size_t) mb.n, e->rl);
    mb.cap = list_capacity(e->list_cap ? e->list_cap : mb.est);
    mb.watch.entered(0);
  }
  e->watch.entered(0);
  e->next_look = e->watch.next();
  e->entering.clear();
  e->nl_cap = 0;
  ENS_TRY(hipMalloc(&e->nl_len, N * 2));
  ENS_TRY(hipMalloc(&e->nl_perm, N * 4));
  ENS_TRY(hipMalloc(&e->nl_prow0, N * 16));
  ENS_TRY(hipMalloc(&e->nl_pos0, 2 * N * 8));
  ENS_TRY(hipMalloc(&e->nl_gate, kGateWords * 4));
  ENS_TRY(hipMalloc(&e->nl_mgate, 2 * M * 4));
  ENS_TRY(hipMalloc(&e->nl_mcap, 2 * M * 4));
  ENS_TRY(hipMalloc(&e->nl_mlong, M * 4));
  for (uint32_t *&k : e->skey) ENS_TRY(hipMalloc(&k, N * 4));
  ENS_TRY(hipMalloc(&e->dirty, e->ncells * 4));
  ENS_TRY(hipMalloc(&e->mhead, e->ncells * 8));
  ENS_TRY(hipMalloc(&e->mnext, N * 8));
  ENS_TRY(hipMemsetAsync(e->dirty, 0, e->ncells * 4, e->stream));
  ENS_TRY(hipMemsetAsync(e->mhead, 0, e->ncells * 8, e->stream));
  ENS_TRY(hipHostMalloc((void **) &e->h_error, 4, hipHostMallocDefault));
  ENS_TRY(hipHostMalloc((void **) &e->h_look, e->kSlots * (1 + M) * 4, hipHostMallocDefault));
  for (hipEvent_t &ev : e->look_ev) ENS_TRY(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
  *e->h_error = 0u;
  e->gen_seen = 1u;
  e->split = false;
  // The lists below are those of the initial state: no member is due at the
  // first timestep (an overflowed list sets its member's gate at that step).
  std::vector<uint32_t> words(kGateWords, 0u), longest(M), none(2 * M, 0u);
  words[kGateGen] = 1u;
  ENS_TRY(hipMemcpy(e->nl_mgate, none.data(), 2 * M * 4, hipMemcpyHostToDevice));
  ENS_TRY(hipMemcpy(e->nl_mlong, none.data(), M * 4, hipMemcpyHostToDevice));
  ENS_TRY(hipMemcpy(e->nl_gate, words.data(), kGateWords * 4, hipMemcpyHostToDevice));
  const int ntiles = ((int) e->ncells + kScanTile - 1) / kScanTile;
  ENS_TRY(hipMemsetAsync(e->count, 0, (e->ncells + 1) * 4, e->stream));
  issue_sort(e, e->start_new, e->skey[1], e->count);
  hipLaunchKernelGGL(k_tile_totals, ntiles, kScanBlock, 0, e->stream, e->count, e->bsum,
                     (int) e->ncells);
  for (bool again = true; again;) {
    int rc = reserve_entries(e);
    if (!rc) rc = put_capacities(e);
    if (rc) return rc;
    e->hooks->launch_multi_list(e->precision, e->d_build[e->cur], ens_tiles(e), e->reach,
                                e->occupancy, e->tile, e->block, e->stream, ens_build_args(e),
                                nullptr, 1);
    ENS_TRY(hipGetLastError());
    ENS_TRY(hipStreamSynchronize(e->stream));
    ENS_TRY(hipMemcpy(longest.data(), e->nl_mlong, M * 4, hipMemcpyDeviceToHost));
    again = false;
    for (size_t m = 0; m < M; m++) again = grow_lists(e, e->mem[m], longest[m]) || again;
  }
  return ABL_OK;
}

// Initial state of every member (main()'s agent creation from the member's
// generator state), the grids, and the per-member kernel arguments.
extern "C" int abl_ens_init(abl_ensemble *e, uint64_t s0, uint64_t s1) {
  if (!e) return ens_fail(ABL_ERR_ARG, "bad argument");
  free_all(e);
  const int M = (int) e->mem.size();
  std::vector<char> host;
  size_t total = 0, cells = 0;
  unsigned tiles = 0;
  int tx = 16, ty = 8, tz = 1;
  e->hooks->tile_shape(e->tile, &tx, &ty, &tz);
  e->reach = 1;
  double occ_max = 0.0;
  // the near radius of member m (under use_float the parameter is a float
  // global, as in a run alone)
  auto radius_of = [&](const Member &mb) {
    const StepDesc &sd = e->prog->steps[0];
    double r = 0.0;
    for (size_t p = 0; p < e->prog->params.size(); p++) {
      if (std::strcmp(e->prog->params[p].name, sd.radius_param) == 0) {
        double v = mb.params[p];
        if (e->precision != ABL_PREC_F64) v = (double) (float) v;
        r = sd.radius_scale * v;
      }
    }
    return r;
  };
  // neighbour lists when every member has the same near radius and cell size
  // and the list radius needs no more than four cells of reach (as for a run
  // alone); their cells are widened by 1 + skin, as a run alone's are
  e->lists = e->nlist && e->hooks->launch_multi_list && M > 0;
  double gran0 = 0.0;
  for (int m = 0; m < M && e->lists; m++) {
    double lo[3], hi[3], gran;
    e->prog->env(e->mem[(size_t) m].params.data(), lo, hi, &gran);
    const double r = radius_of(e->mem[(size_t) m]);
    if (m == 0) {
      gran0 = gran;
      e->r = r;
    } else if (gran != gran0 || r != e->r) {
      e->lists = false;
    }
  }
  if (e->lists) {
    e->rl = e->r * (1.0 + e->skin);
    const double cell = gran0 / (double) e->cell_scale * (1.0 + 1.0 / 1048576.0) * (1.0 + e->skin);
    if (!(e->r > 0.0) || std::ceil(e->rl / cell * (1.0 + 1.0 / 2097152.0)) > 4.0) e->lists = false;
  }
  const double inflate = e->lists ? 1.0 + e->skin : 1.0;
  for (int m = 0; m < M; m++) {
    Member &mb = e->mem[(size_t) m];
    uint64_t st[2];
    abl_ens_member_seed(s0, s1, m, st);
    abl_rng_seed(st[0], st[1]);
    std::vector<char> recs;
    size_t cnt = 0;
    int rc = e->hooks->host_records(mb.params.data(), e->precision, recs, &cnt);
    if (rc) return ens_fail(rc, "host initialisation failed");
    mb.n = (int) cnt;
    mb.off = (uint32_t) total;
    total += cnt;
    host.insert(host.end(), recs.begin(), recs.end());
    double lo[3], hi[3], gran;
    e->prog->env(mb.params.data(), lo, hi, &gran);
    const double cell = gran / (double) e->cell_scale * (1.0 + 1.0 / 1048576.0) * inflate;
    GridView g{};
    g.dim = 2;
    for (int d = 0; d < 3; d++) {
      g.lo[d] = d < 2 ? lo[d] : 0.0;
      g.n[d] = d < 2 ? std::max(1, (int) std::ceil((hi[d] - lo[d]) / cell)) : 1;
    }
    g.inv_cell = 1.0 / cell;
    const double r = radius_of(mb);
    // the stencil reaches the list radius in list mode
    const double reach_r = e->lists ? e->rl : r;
    g.reach = std::max(1, (int) std::ceil(reach_r / cell * (1.0 + 1.0 / 2097152.0)));
    e->reach = std::max(e->reach, g.reach);
    mb.g = g;
    mb.cell = cell;
    mb.near_t = sqrtf_le_threshold(r);
    mb.rc = (float) (r / cell * (1.0 + 1.0 / 1048576.0));
    mb.cell_base = (uint32_t) cells;
    cells += (size_t) g.n[0] * (size_t) g.n[1];
    mb.tile_base = tiles;
    mb.ntiles = (unsigned) (((g.n[0] + tx - 1) / tx) * ((g.n[1] + ty - 1) / ty));
    tiles += mb.ntiles;
    occ_max = std::max(occ_max, (double) cnt / ((double) g.n[0] * g.n[1]));
  }
  for (Member &mb : e->mem) mb.g.reach = e->reach;  // one kernel instance for all members
  if (e->lists) e->cell = e->mem[0].cell;
  e->n = total;
  e->ncells = cells;
  e->total_tiles = tiles;
  e->occupancy = (float) occ_max;
  const size_t N = std::max<size_t>(total, 1);
  for (int b = 0; b < 2; b++) {
    for (int c = 0; c < e->ncols; c++) ENS_TRY(hipMalloc(&e->col[b][c], N * (size_t) e->elem));
    ENS_TRY(hipMalloc(&e->id[b], N * 4));
  }
  ENS_TRY(hipMalloc(&e->key, N * 4));
  ENS_TRY(hipMalloc(&e->tmp_idx, N * 4));
  ENS_TRY(hipMalloc(&e->tmp_id, N * 4));
  ENS_TRY(hipMalloc(&e->count, (cells + 1) * 4));
  ENS_TRY(hipMalloc(&e->start, (cells + 1) * 4));
  ENS_TRY(hipMalloc(&e->bsum, ((cells + kScanTile - 1) / kScanTile + 1) * 4));
  ENS_TRY(hipMemsetAsync(e->count, 0, (cells + 1) * 4, e->stream));
  // transpose host records (AoS of ncols floats) into columns, ids = index in member
  std::vector<char> colbuf(N * (size_t) e->elem);
  std::vector<int32_t> ids(N);
  for (int c = 0; c < e->ncols; c++) {
    for (size_t i = 0; i < total; i++) {
      std::memcpy(&colbuf[i * (size_t) e->elem], &host[(i * (size_t) e->ncols + (size_t) c) * (size_t) e->elem],
                  (size_t) e->elem);
    }
    ENS_TRY(hipMemcpy(e->col[0][c], colbuf.data(), total * (size_t) e->elem, hipMemcpyHostToDevice));
  }
  for (const Member &mb : e->mem) {
    for (int i = 0; i < mb.n; i++) ids[mb.off + (uint32_t) i] = i;
  }
  ENS_TRY(hipMemcpy(e->id[0], ids.data(), total * 4, hipMemcpyHostToDevice));
  e->cur = 0;
  e->id_cur = 0;
  // device tables
  std::vector<uint32_t> off(M + 1), cb(M + 1);
  std::vector<uint2> tile_of;
  std::vector<GridView> grids(M);
  for (int m = 0; m < M; m++) {
    off[m] = e->mem[m].off;
    cb[m] = e->mem[m].cell_base;
    tile_of.insert(tile_of.end(), e->mem[m].ntiles, make_uint2((uint32_t) m, e->mem[m].tile_base));
    grids[m] = e->mem[m].g;
  }
  off[M] = (uint32_t) total;
  cb[M] = (uint32_t) cells;
  ENS_TRY(hipMalloc(&e->d_off, (M + 1) * 4));
  ENS_TRY(hipMalloc(&e->d_cell_base, (M + 1) * 4));
  ENS_TRY(hipMalloc(&e->d_tile_of, tile_of.size() * sizeof(uint2)));
  ENS_TRY(hipMalloc(&e->d_grids, M * sizeof(GridView)));
  ENS_TRY(hipMemcpy(e->d_off, off.data(), (M + 1) * 4, hipMemcpyHostToDevice));
  ENS_TRY(hipMemcpy(e->d_cell_base, cb.data(), (M + 1) * 4, hipMemcpyHostToDevice));
  ENS_TRY(hipMemcpy(e->d_tile_of, tile_of.data(), tile_of.size() * sizeof(uint2),
                    hipMemcpyHostToDevice));
  ENS_TRY(hipMemcpy(e->d_grids, grids.data(), M * sizeof(GridView), hipMemcpyHostToDevice));
  // member kernel arguments: after the grid gather the columns sit in buffer
  // 1 - cur; the step reads them and writes buffer cur
  const size_t asz = e->hooks->args_size(e->precision);
  if (e->lists) ENS_TRY(hipMalloc(&e->start_new, (cells + 1) * 4));
  for (int b = 0; b < 2; b++) {
    auto args_on = [&](const uint32_t *start, void **d_args) -> int {
      std::vector<char> args((size_t) M * asz);
      for (int m = 0; m < M; m++) {
        ColSet in{}, outc{};
        for (int c = 0; c < e->ncols; c++) {
          in.c[c] = e->col[1 - b][c];
          outc.c[c] = e->col[b][c];
        }
        GridView g = e->mem[m].g;
        g.start = start + e->mem[m].cell_base;
        e->hooks->fill_args(e->precision, &args[(size_t) m * asz], e->mem[m].params.data(), in, outc,
                            g, e->mem[m].near_t, e->mem[m].rc, e->mem[m].n, e->occupancy, e->tile);
      }
      ENS_TRY(hipMalloc(d_args, args.size()));
      ENS_TRY(hipMemcpy(*d_args, args.data(), args.size(), hipMemcpyHostToDevice));
      return ABL_OK;
    };
    int rc = args_on(e->start, &e->d_args[b]);
    if (!rc && e->lists) rc = args_on(e->start_new, &e->d_build[b]);
    if (rc) return rc;
  }
  e->timestep = 0;
  if (e->lists && total > 0) {
    int rc = init_lists(e);
    if (rc) return rc;
  }
  ENS_TRY(hipStreamSynchronize(e->stream));
  e->ready = true;
  return ABL_OK;
}

// One timestep: rebuild every member's grid (one sort over all cells), then
// the program's tiled step over all members' tiles.  With lists: the gated
// rebuild, then the step through the lists from the current buffers into the
// other ones.
static int issue_step(abl_ensemble *e) {
  const int n = (int) e->n;
  const int b = e->cur;
  if (e->lists) {
    if (n > 0) {
      const int rc = e->entering.empty() ? issue_rebuild(e) : enter_members(e);
      if (rc) return rc;
      // the step reads buffer b: the arguments whose input is 1 - (1 - b)
      e->hooks->launch_multi_list(e->precision, e->d_args[1 - b], ens_tiles(e), e->reach,
                                  e->occupancy, e->tile, e->block, e->stream, ens_list_args(e),
                                  nullptr, 2);
      e->cur ^= 1;
    }
    e->timestep += 1;
    ENS_TRY(hipGetLastError());
    return ABL_OK;
  }
  e->timestep += 1;
  issue_sort(e, e->start, nullptr, nullptr);
  if (n > 0) {
    e->id_cur ^= 1;
    // the step reads buffer 1 - b and writes buffer b: columns end where they began
    e->hooks->launch_multi(e->precision, e->d_args[b], ens_tiles(e), e->reach, e->occupancy, e->tile,
                           e->block, e->stream);
  }
  ENS_TRY(hipGetLastError());
  return ABL_OK;
}

// What follows from how the lists fare, after the timestep that next_look names has
// been issued.  Asked and read at fixed timesteps (ListWatch), whatever the pace of
// host and device and however simulate() is called.
//
// Lists grown: a member whose lists have outgrown their capacity enters them anew
// at the next timestep, which is the one a run of it alone does that at
// (list_watch, enter_lists).  One overflowed list makes its member rebuild on
// every timestep: 30 members of up to 8,192 boids, FP32, 18 us per timestep, and
// 90 from the first list that outgrew its capacity on.
//
// One launch per rebuild or four: four from a quarter of the timesteps on, back
// below an eighth, so that a rate in between does not switch to and fro.
static int look(abl_ensemble *e) {
  const uint64_t t = e->timestep - 1;
  const size_t M = e->mem.size();
  bool ask = false;
  auto slot = [&](uint64_t t_req) { return e->h_look + (t_req % e->kSlots) * (1 + M); };
  // an answer is there: waits, for what was asked kListSample timesteps ago
  auto answer = [&](ListWatch &w, const uint32_t **words) -> hipError_t {
    const hipError_t err = hipEventSynchronize(e->look_ev[w.t_req % e->kSlots]);
    *words = slot(w.t_req);
    w.read();
    return err;
  };
  const uint32_t *words = nullptr;
  uint64_t next = ~0ull;
  for (size_t m = 0; m < M; m++) {
    Member &mb = e->mem[m];
    if (mb.watch.next() == t) {
      if (mb.watch.pending) {
        ENS_TRY(answer(mb.watch, &words));
        if (grow_lists(e, mb, words[1 + m])) e->entering.push_back((int) m);
      } else {
        ask = true;
        mb.watch.asked(t);
      }
    }
    next = std::min(next, mb.watch.next());
  }
  if (e->watch.next() == t) {
    if (e->watch.pending) {
      const uint64_t steps = e->watch.t_req - e->watch.t_prev;
      ENS_TRY(answer(e->watch, &words));
      const uint64_t rebuilt = words[0] - e->gen_seen;
      e->gen_seen = words[0];
      const bool split = e->split ? rebuilt * 8u >= steps : rebuilt * 4u > steps;
      if (split != e->split) {
        e->split = split;
        ENS_TRY(hipMemsetAsync(e->nl_gate + kGateQueue, 0, (kGateWords - kGateQueue) * 4, e->stream));
      }
    } else {
      ask = true;
      e->watch.asked(t);
    }
  }
  e->next_look = std::min(next, e->watch.next());
  if (ask) {
    uint32_t *w = slot(t);
    hipLaunchKernelGGL(k_ens_tell, grid_blocks((int) M, 256), 256, 0, e->stream, e->nl_gate + kGateGen,
                       e->nl_mlong, (int) M, w);
    ENS_TRY(hipGetLastError());
    ENS_TRY(hipEventRecord(e->look_ev[t % e->kSlots], e->stream));
  }
  return ABL_OK;
}

// Two timesteps as a graph, in the form the rebuilds have.
static int capture(abl_ensemble *e) {
  const int k = e->split ? 1 : 0;
  if (e->exec[k]) return ABL_OK;
  const uint64_t t0 = e->timestep;
  ENS_TRY(hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal));
  int rc = issue_step(e);
  if (!rc) rc = issue_step(e);
  hipError_t ce = hipStreamEndCapture(e->stream, &e->graph[k]);
  e->timestep = t0;  // captured, not run
  if (rc) return rc;
  ENS_TRY(ce);
  ENS_TRY(hipGraphInstantiate(&e->exec[k], e->graph[k], nullptr, nullptr, 0));
  return ABL_OK;
}

extern "C" int abl_ens_simulate(abl_ensemble *e, int steps) {
  if (!e || steps < 0) return ens_fail(ABL_ERR_ARG, "bad argument");
  if (!e->ready) return ens_fail(ABL_ERR_STATE, "abl_ens_init first");
  ENS_TRY(hipEventRecord(e->ev0, e->stream));
  const uint64_t end = e->timestep + (uint64_t) steps;
  const bool watched = e->lists && e->n > 0;
  while (e->timestep < end) {
    // the id buffer (without lists) or the column buffers and the gates'
    // parity (with lists) alternate per step: two timesteps, captured from
    // an even start, end where they start
    const bool even = e->lists ? (e->timestep & 1u) == 0 : (e->id_cur & 1) == 0;
    const bool plain = !watched || (e->entering.empty() && e->next_look != e->timestep);
    if (e->use_graph && even && plain && e->timestep + 2 <= end) {
      const int rc = capture(e);
      if (rc) return rc;
      ENS_TRY(hipGraphLaunch(e->exec[e->split ? 1 : 0], e->stream));
      e->timestep += 2;
    } else {
      const int rc = issue_step(e);
      if (rc) return rc;
    }
    if (watched && e->next_look == e->timestep - 1) {
      const int rc = look(e);
      if (rc) return rc;
    }
  }
  ENS_TRY(hipEventRecord(e->ev1, e->stream));
  if (e->h_error)
    ENS_TRY(hipMemcpyAsync(e->h_error, e->nl_gate + kGateError, 4, hipMemcpyDeviceToHost, e->stream));
  return ABL_OK;
}

// After a synchronisation: no rebuild of the timesteps so far gave up waiting.
static int ens_check(const abl_ensemble *e) {
  if (e->h_error && *(const volatile uint32_t *) e->h_error)
    return ens_fail(ABL_ERR_DEVICE, "list rebuild: a phase did not finish");
  return ABL_OK;
}

extern "C" int abl_ens_synchronize(abl_ensemble *e, double *ms) {
  if (!e) return ens_fail(ABL_ERR_ARG, "bad argument");
  ENS_TRY(hipStreamSynchronize(e->stream));
  float f = 0.f;
  if (hipEventElapsedTime(&f, e->ev0, e->ev1) == hipSuccess) e->last_ms = f;
  if (ms) *ms = e->last_ms;
  return ens_check(e);
}

extern "C" int abl_ens_member_count(abl_ensemble *e, int member, size_t *count) {
  if (!e || member < 0 || member >= (int) e->mem.size() || !count)
    return ens_fail(ABL_ERR_ARG, "bad argument");
  *count = (size_t) e->mem[(size_t) member].n;
  return ABL_OK;
}

// Member's agents in its own id order (as a run of it alone downloads them).
extern "C" int abl_ens_download(abl_ensemble *e, int member, void *aos, size_t capacity,
                                size_t *count) {
  if (!e || member < 0 || member >= (int) e->mem.size()) return ens_fail(ABL_ERR_ARG, "bad argument");
  if (!e->ready) return ens_fail(ABL_ERR_STATE, "abl_ens_init first");
  const Member &mb = e->mem[(size_t) member];
  if (count) *count = (size_t) mb.n;
  if (mb.n == 0) return ABL_OK;
  if (!aos || capacity < (size_t) mb.n) return ens_fail(ABL_ERR_ARG, "buffer too small");
  const size_t rec = (size_t) e->ncols * (size_t) e->elem;
  const size_t bytes = (size_t) mb.n * rec;
  std::lock_guard<std::mutex> hold(e->dl_lock);
  if (e->dl_bytes < bytes) {
    ENS_TRY(hipStreamSynchronize(e->stream));
    if (e->dl) ENS_TRY(hipFree(e->dl));
    e->dl = nullptr;
    e->dl_bytes = 0;
    size_t most = 0;
    for (const Member &k : e->mem) most = std::max(most, (size_t) k.n * rec);
    ENS_TRY(hipMalloc(&e->dl, most));
    e->dl_bytes = most;
  }
  ColSet cols{};
  for (int c = 0; c < e->ncols; c++) cols.c[c] = e->col[e->cur][c];
  hipLaunchKernelGGL(k_ens_unpermute, grid_blocks(mb.n, 256), 256, 0, e->stream, (char *) e->dl,
                     cols, e->elem, e->ncols, e->id[e->id_cur], mb.off, mb.n);
  ENS_TRY(hipGetLastError());
  ENS_TRY(hipMemcpyAsync(aos, e->dl, bytes, hipMemcpyDeviceToHost, e->stream));
  ENS_TRY(hipStreamSynchronize(e->stream));
  return ens_check(e);
}

// What the ensemble has decided for a member.
extern "C" int abl_ens_inspect(abl_ensemble *e, int member, const char *what, double *value) {
  if (!e || member < 0 || member >= (int) e->mem.size() || !what || !value)
    return ens_fail(ABL_ERR_ARG, "bad argument");
  const Member &mb = e->mem[(size_t) member];
  const std::string k(what);
  if (k == "lists") *value = e->lists && mb.n > 0;
  else if (k == "list_capacity") *value = mb.cap;
  else if (k == "rebuild_launches") *value = e->split ? 4 : 1;
  else if (k == "rebuilds") *value = e->gen_seen - 1u;
  else return ens_fail(ABL_ERR_ARG, "unknown quantity " + k);
  return ABL_OK;
}

extern "C" int abl_ens_agents(abl_ensemble *e, size_t *total) {
  if (!e || !total) return ens_fail(ABL_ERR_ARG, "bad argument");
  *total = e->n;
  return ABL_OK;
}

extern "C" int abl_ens_destroy(abl_ensemble *e) {
  if (!e) return ens_fail(ABL_ERR_ARG, "bad argument");
  (void) hipStreamSynchronize(e->stream);
  free_all(e);
  if (e->ev0) (void) hipEventDestroy(e->ev0);
  if (e->ev1) (void) hipEventDestroy(e->ev1);
  if (e->stream) (void) hipStreamDestroy(e->stream);
  delete e;
  return ABL_OK;
}
