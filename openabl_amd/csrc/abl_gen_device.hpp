// abl_gen_device.hpp -- what step programs generated by the -b hip code
// generator (openabl_amd/compiler) build on, on the device.
//
// Generated device code is a template on F, the program's float type
// (double, or float under use_float), and reads like the C backend's
// program: vector values are vec2<F>/vec3<F>, operators are the helper
// functions below with the C runtime's argument and result types
// (asset/c/libabl.h:65-175: a scalar operand is converted to abl_float,
// length() is sqrtf of the abl_float sum of squares, min/max are fmin/fmax
// in double), so every operation rounds as the C backend's does.  Host-side
// only literals that C writes as double stay double (C's usual arithmetic
// conversions apply identically in C++).
#pragma once

#include <math.h>
#include <stdint.h>
#include <stdio.h>

#include "abl_root_bounds.hpp"
#include "abl_runtime.hpp"
#include "abl_tile.hpp"

namespace abl {
namespace gen {

template <typename F>
struct vec2 {
  F x, y;
};
template <typename F>
struct vec3 {
  F x, y, z;
};

// ---- vectors (asset/c/libabl.h:80-175 semantics) ----------------------------------
template <typename F>
__host__ __device__ inline vec2<F> v2_create(F x, F y) { return {x, y}; }
template <typename F>
__host__ __device__ inline vec2<F> v2_fill(F x) { return {x, x}; }
template <typename F>
__host__ __device__ inline vec2<F> v2_add(vec2<F> a, vec2<F> b) { return {a.x + b.x, a.y + b.y}; }
template <typename F>
__host__ __device__ inline vec2<F> v2_sub(vec2<F> a, vec2<F> b) { return {a.x - b.x, a.y - b.y}; }
template <typename F>
__host__ __device__ inline vec2<F> v2_mul(vec2<F> a, F s) { return {a.x * s, a.y * s}; }
template <typename F>
__host__ __device__ inline vec2<F> v2_div(vec2<F> a, F s) { return {a.x / s, a.y / s}; }
template <typename F>
__host__ __device__ inline bool v2_eq(vec2<F> a, vec2<F> b) { return a.x == b.x && a.y == b.y; }
template <typename F>
__host__ __device__ inline bool v2_ne(vec2<F> a, vec2<F> b) { return a.x != b.x || a.y != b.y; }

template <typename F>
__host__ __device__ inline vec3<F> v3_create(F x, F y, F z) { return {x, y, z}; }
template <typename F>
__host__ __device__ inline vec3<F> v3_fill(F x) { return {x, x, x}; }
template <typename F>
__host__ __device__ inline vec3<F> v3_add(vec3<F> a, vec3<F> b) {
  return {a.x + b.x, a.y + b.y, a.z + b.z};
}
template <typename F>
__host__ __device__ inline vec3<F> v3_sub(vec3<F> a, vec3<F> b) {
  return {a.x - b.x, a.y - b.y, a.z - b.z};
}
template <typename F>
__host__ __device__ inline vec3<F> v3_mul(vec3<F> a, F s) { return {a.x * s, a.y * s, a.z * s}; }
template <typename F>
__host__ __device__ inline vec3<F> v3_div(vec3<F> a, F s) { return {a.x / s, a.y / s, a.z / s}; }
template <typename F>
__host__ __device__ inline bool v3_eq(vec3<F> a, vec3<F> b) {
  return a.x == b.x && a.y == b.y && a.z == b.z;
}
template <typename F>
__host__ __device__ inline bool v3_ne(vec3<F> a, vec3<F> b) {
  return a.x != b.x || a.y != b.y || a.z != b.z;
}

// correctly rounded sqrtf on the host and on the device
__host__ __device__ inline float sqrtf_rn(float f) {
#if defined(__HIP_DEVICE_COMPILE__)
  return sqrt_rn_f32(f);
#else
  return ::sqrtf(f);
#endif
}

template <typename F>
__host__ __device__ inline F dot2(vec2<F> a, vec2<F> b) { return a.x * b.x + a.y * b.y; }
template <typename F>
__host__ __device__ inline F dot3(vec3<F> a, vec3<F> b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
template <typename F>
__host__ __device__ inline F length2(vec2<F> v) { return (F) sqrtf_rn((float) (v.x * v.x + v.y * v.y)); }
template <typename F>
__host__ __device__ inline F length3(vec3<F> v) {
  return (F) sqrtf_rn((float) (v.x * v.x + v.y * v.y + v.z * v.z));
}
// A distance or length that the step only compares with constants: the
// float square sum it is the correctly rounded root of, compared against
// exact bounds (abl_root_bounds.hpp), with the same sums as length2/length3.
template <typename F>
struct SqLen {
  float s;
};
template <typename F>
__host__ __device__ inline SqLen<F> sq_length2(vec2<F> v) { return {(float) (v.x * v.x + v.y * v.y)}; }
template <typename F>
__host__ __device__ inline SqLen<F> sq_length3(vec3<F> v) {
  return {(float) (v.x * v.x + v.y * v.y + v.z * v.z)};
}
template <typename F>
__host__ __device__ inline SqLen<F> sq_dist2(vec2<F> a, vec2<F> b) { return sq_length2<F>(v2_sub<F>(a, b)); }
template <typename F>
__host__ __device__ inline SqLen<F> sq_dist3(vec3<F> a, vec3<F> b) { return sq_length3<F>(v3_sub<F>(a, b)); }
template <typename F>
__host__ __device__ inline bool len_lt(SqLen<F> q, double c) { return rootb::root_lt(q.s, c); }
template <typename F>
__host__ __device__ inline bool len_le(SqLen<F> q, double c) { return rootb::root_le(q.s, c); }
template <typename F>
__host__ __device__ inline bool len_gt(SqLen<F> q, double c) { return rootb::root_gt(q.s, c); }
template <typename F>
__host__ __device__ inline bool len_ge(SqLen<F> q, double c) { return rootb::root_ge(q.s, c); }

template <typename F>
__host__ __device__ inline F dist2(vec2<F> a, vec2<F> b) { return length2<F>(v2_sub<F>(a, b)); }
template <typename F>
__host__ __device__ inline F dist3(vec3<F> a, vec3<F> b) { return length3<F>(v3_sub<F>(a, b)); }
template <typename F>
__host__ __device__ inline vec2<F> normalize2(vec2<F> v) { return v2_div<F>(v, length2<F>(v)); }
template <typename F>
__host__ __device__ inline vec3<F> normalize3(vec3<F> v) { return v3_div<F>(v, length3<F>(v)); }

// min/max of libabl.h: fmin/fmax of the arguments as abl_float
template <typename F>
__host__ __device__ inline F fmin_c(F a, F b) { return (F) ::fmin((double) a, (double) b); }
template <typename F>
__host__ __device__ inline F fmax_c(F a, F b) { return (F) ::fmax((double) a, (double) b); }

// ---- kernel arguments and per-agent context -----------------------------------------

struct GenArgs {
  void *in[kMaxCols];
  void *out[kMaxCols];
  void *nb[kMaxCols];
  void *birth[kMaxCols];
  const int32_t *nb_id;
  const int32_t *self_id;
  uint8_t *dead;
  uint8_t *born;
  GridView g;
  float near_t;
  int n;
  uint64_t seed, t;
  uint32_t ordinal;
};

inline GenArgs make_args(const StepLaunch &L) {
  GenArgs a{};
  for (int c = 0; c < kMaxCols; c++) {
    a.in[c] = L.in.c[c];
    a.out[c] = L.out.c[c];
    a.nb[c] = L.nb.c[c];
    a.birth[c] = L.birth.c[c];
  }
  a.nb_id = L.nb_id;
  a.self_id = L.self_id;
  a.dead = L.dead;
  a.born = L.born;
  a.g = L.grid;
  a.near_t = L.near_t;
  a.n = L.n;
  a.seed = L.seed;
  a.t = L.timestep;
  a.ordinal = L.step_ordinal;
  return a;
}

template <typename T>
__device__ __forceinline__ T col_at(void *const *cols, int c, int i);

// A near-loop candidate as the generated loop body reads it: column `col` of
// the near agent type, held at position `slot` of a staged record.  From the
// columns in global memory (candidate j) ...
struct ColRec {
  void *const *cols;
  uint32_t j;
  template <typename T>
  __device__ __forceinline__ T get(int col, int) const {
    return col_at<T>(cols, col, (int) j);
  }
};
// ... or from a record of the float columns the loop reads, staged in LDS
// (abl_tile.hpp's records: the position's components first).
template <typename F>
struct StagedRec {
  const F *r;
  template <typename T>
  __device__ __forceinline__ T get(int, int slot) const {
    return (T) r[slot];
  }
};

// random() inside a step: the k-th call of this agent in this step draws
// counter_bits(seed, timestep, step, id, k).
template <typename F>
struct CtxBase {
  const GenArgs &a;
  int i;
  uint32_t k = 0;
  __device__ CtxBase(const GenArgs &args, int slot) : a(args), i(slot) {}

  __device__ F random_float(F lo, F hi) {
    const uint64_t bits = counter_bits(a.seed, a.t, a.ordinal, (uint64_t) a.self_id[i], k++);
    return counter_random<F>(lo, hi, bits);
  }
  // random_int(lo, hi) on one draw: the C runtime's power-of-two branch
  // (asset/c/libabl.c:26-30, the low bits masked, lo not added), otherwise
  // lo + the draw's low 32 bits modulo the span
  __device__ int random_int(int lo, int hi) {
    const uint64_t bits = counter_bits(a.seed, a.t, a.ordinal, (uint64_t) a.self_id[i], k++);
    const unsigned n = (unsigned) (hi - lo + 1);
    if ((n & (n - 1)) == 0) return (int) ((unsigned) bits & (n - 1));
    return lo + (int) ((unsigned) bits % n);
  }
  __device__ void remove_current() { a.dead[i] = 1; }
  // the C near test dist(nx.pos, centre) > r, on the square sum against the
  // host threshold T (T = max{f : sqrtf(f) <= r})
  __device__ bool outside(vec2<F> q, vec2<F> p) const {
    return dist_sq_f32<F>(q.x, q.y, p.x, p.y) > a.near_t;
  }
  __device__ bool outside(vec3<F> q, vec3<F> p) const {
    return dist_sq_f32<F>(q.x, q.y, q.z, p.x, p.y, p.z) > a.near_t;
  }
  // the same test on the square sum sq_dist2/3(q, p) (the sums are the same)
  __device__ bool outside_sq(SqLen<F> q) const { return q.s > a.near_t; }
};

// One agent's view of a step walking the grid: its slot, random(), and the
// near loop's candidates read from the columns.
template <typename F, bool BY_ID>
struct Ctx : CtxBase<F> {
  using CtxBase<F>::a;
  __device__ Ctx(const GenArgs &args, int slot) : CtxBase<F>(args, slot) {}

  // Candidates of the near loop around `pos`: the stencil of cells in cell
  // order, or merged into ascending id order (the reference's); `visit(rec)`
  // returns false to stop (break).
  template <typename P, typename Visit>
  __device__ void near(P x, P y, P z, Visit &&visit) const {
    const GridView &g = a.g;
    const int3 c = cell_of<P>(g, x, y, z);
    const int reach = g.reach;
    const int x0 = c.x - reach < 0 ? 0 : c.x - reach;
    const int x1 = c.x + reach > g.n[0] - 1 ? g.n[0] - 1 : c.x + reach;
    const int y0 = c.y - reach < 0 ? 0 : c.y - reach;
    const int y1 = c.y + reach > g.n[1] - 1 ? g.n[1] - 1 : c.y + reach;
    int z0 = 0, z1 = 0;
    if (g.dim == 3) {
      z0 = c.z - reach < 0 ? 0 : c.z - reach;
      z1 = c.z + reach > g.n[2] - 1 ? g.n[2] - 1 : c.z + reach;
    }
    if (!BY_ID) {
      for (int zz = z0; zz <= z1; zz++) {
        for (int yy = y0; yy <= y1; yy++) {
          const uint32_t row = ((uint32_t) zz * (uint32_t) g.n[1] + (uint32_t) yy) * (uint32_t) g.n[0];
          const uint32_t s = g.start[row + x0], e = g.start[row + x1 + 1];
          for (uint32_t j = s; j < e; j++)
            if (!visit(ColRec{a.nb, j})) return;
        }
      }
      return;
    }
    constexpr int kMaxRuns = 27;
    uint32_t cur[kMaxRuns], end[kMaxRuns];
    int32_t head[kMaxRuns];
    int nr = 0;
    for (int zz = z0; zz <= z1; zz++) {
      for (int yy = y0; yy <= y1; yy++) {
        const uint32_t row = ((uint32_t) zz * (uint32_t) g.n[1] + (uint32_t) yy) * (uint32_t) g.n[0];
        for (int xx = x0; xx <= x1 && nr < kMaxRuns; xx++) {
          const uint32_t s = g.start[row + xx], e = g.start[row + xx + 1];
          if (s < e) {
            cur[nr] = s;
            end[nr] = e;
            head[nr] = a.nb_id[s];
            nr++;
          }
        }
      }
    }
    while (nr > 0) {
      int best = 0;
      for (int r = 1; r < nr; r++) best = head[r] < head[best] ? r : best;
      const uint32_t j = cur[best];
      if (!visit(ColRec{a.nb, j})) return;
      cur[best] = j + 1;
      if (j + 1 < end[best]) {
        head[best] = a.nb_id[j + 1];
      } else {
        nr--;
        cur[best] = cur[nr];
        end[best] = end[nr];
        head[best] = head[nr];
      }
    }
  }
};

template <typename T>
__device__ __forceinline__ T col_at(void *const *cols, int c, int i) {
  return ((const T *) cols[c])[i];
}

// ---- a generated step on the LDS-tiled kernels (abl_tile.hpp) ----------------------
// The tiled stencil walk (launch_gen_tiles), and for programs generated with
// -C hip.lists=1 the neighbour lists (launch_gen_lists).
// S describes one step of the program (generated): F, the agent struct
// Agent, DIM, the NS float columns its near loop reads (kCols, the
// position's components first), and load / store / pos / run.  Its near loop
// is over the stepping agent's own type and centred on the agent, so the
// agent's neighbour list holds every candidate of the loop within the
// list radius, in the stencil's order of the list build.

struct GenTileArgs : GenArgs {
  int cap;   // LDS records per tile
  float rc;  // near radius in cell units (the stencil of an overflowed list)
};

// One agent's view of a step walking its list: `walk(visit)` calls visit
// with every candidate record, in order, until visit returns false.
template <typename F, class Walk>
struct ListCtx : CtxBase<F> {
  Walk &walk;
  __device__ ListCtx(const GenArgs &args, int slot, Walk &w) : CtxBase<F>(args, slot), walk(w) {}
  template <typename P, typename Visit>
  __device__ void near(P, P, P, Visit &&visit) {
    walk([&](const F *r) { return visit(StagedRec<F>{r}); });
  }
};

template <class S>
struct GenPolicy {
  using F = typename S::F;
  static constexpr int DIM = S::DIM;
  static constexpr int NS = S::NS;
  static constexpr bool kAgentStep = true;
  static constexpr int kListWaves = 4;
  using Args = GenTileArgs;
  // the records of the stepping (= near) type from the step's input columns:
  // the rebuild launches point those at the freshly sorted buffers
  __device__ static void load(const Args &a, uint32_t j, F *r) {
#pragma unroll
    for (int v = 0; v < NS; v++) r[v] = col_at<F>(a.in, S::kCols[v], (int) j);
  }
  template <class Walk>
  __device__ static void agent(const Args &a, uint32_t gi, Walk &walk, double *np) {
    ListCtx<F, Walk> c((const GenArgs &) a, (int) gi, walk);
    const typename S::Agent in = S::load(a, (int) gi);
    typename S::Agent out = in;
    S::run(c, in, out);
    S::store(a, (int) gi, out);
    S::pos(out, np);
  }
};

// Launch step S on the LDS tiles of its dimension: its near loop walking each
// agent's stencil (cell order; the grid walk's candidates in its order), or
// what StepLaunch::nl_mode says.  LISTS: programs generated with lists.
template <class S, bool LISTS, int TX, int TY, int TZ, int RM>
inline void launch_gen_tile(const StepLaunch &L, const GenTileArgs &a) {
  using M = GenPolicy<S>;
  if (L.nl_mode == 4) {
    launch_probe<M, TX, TY, TZ, RM>(L);
  } else if constexpr (LISTS) {
    if (L.nl_mode)
      launch_list<M, TX, TY, TZ, RM>(a, L.grid, L.occupancy, L.block, L.stream, L.lds_slack, *L.nl,
                                     L.nl_mode, L.delta);
    else launch_tiled<M, TX, TY, TZ, RM>(a, L);
  } else {
    launch_tiled<M, TX, TY, TZ, RM>(a, L);
  }
}
template <class S, bool LISTS, int TX, int TY, int TZ>
inline void launch_gen_reach(const StepLaunch &L, const GenTileArgs &a) {
  if (L.grid.reach <= 1) launch_gen_tile<S, LISTS, TX, TY, TZ, 1>(L, a);
  else if (L.grid.reach == 2) launch_gen_tile<S, LISTS, TX, TY, TZ, 2>(L, a);
  else launch_gen_tile<S, LISTS, TX, TY, TZ, 4>(L, a);
}
template <class S, bool LISTS = false>
inline void launch_gen_tiles(const StepLaunch &L) {
  GenTileArgs a{};
  static_cast<GenArgs &>(a) = make_args(L);
  a.rc = L.rc;
  if constexpr (S::DIM == 3) {
    launch_gen_reach<S, LISTS, 8, 4, 4>(L, a);
  } else {
    const int t = tile_cells(L);
    if (t == 2) launch_gen_reach<S, LISTS, 8, 8, 1>(L, a);
    else if (t == 4) launch_gen_tile<S, LISTS, 8, 4, 1, 1>(L, a);
    else launch_gen_reach<S, LISTS, 16, 8, 1>(L, a);
  }
}

// The same for programs with lists: the list build (mode 1), the step through
// the lists (2) or the one-launch gated rebuild (3).
template <class S>
inline void launch_gen_lists(const StepLaunch &L) {
  launch_gen_tiles<S, true>(L);
}
template <typename T>
__device__ __forceinline__ void col_put(void *const *cols, int c, int i, T v) {
  ((T *) cols[c])[i] = v;
}

// ---- the sequential step's builtins (host; src/main.cpp:66-130) ----------------------
// count(T), count(T.m, v), sum(T.m), getLastExecTime() and log_csv(...) on the
// runtime's reductions.  A failing call records its status, which the
// generated sequential step returns after the step's statements.
inline int &seq_rc() {
  static thread_local int rc = 0;
  return rc;
}
inline void seq_reset() { seq_rc() = 0; }
inline int seq_status() { return seq_rc(); }
inline void seq_note(int rc) {
  if (rc && !seq_rc()) seq_rc() = rc;
}
inline int seq_count(abl_sim *sim, int type) {
  size_t n = 0;
  seq_note(abl_hip_count(sim, type, &n));
  return (int) n;
}
inline int seq_count_eq(abl_sim *sim, int type, const char *member, double v) {
  size_t n = 0;
  seq_note(abl_hip_reduce_count_eq(sim, type, member, v, &n));
  return (int) n;
}
inline double seq_sum(abl_sim *sim, int type, const char *member) {
  double o[3] = {0, 0, 0};
  seq_note(abl_hip_reduce_sum(sim, type, member, o));
  return o[0];
}
template <typename F>
inline vec2<F> seq_sum2(abl_sim *sim, int type, const char *member) {
  double o[3] = {0, 0, 0};
  seq_note(abl_hip_reduce_sum(sim, type, member, o));
  return {(F) o[0], (F) o[1]};
}
template <typename F>
inline vec3<F> seq_sum3(abl_sim *sim, int type, const char *member) {
  double o[3] = {0, 0, 0};
  seq_note(abl_hip_reduce_sum(sim, type, member, o));
  return {(F) o[0], (F) o[1], (F) o[2]};
}
inline double seq_last_exec(abl_sim *sim) {
  double t = 0.0;
  seq_note(abl_hip_last_exec_time(sim, &t));
  return t;
}
// log_csv: "%d"/"%f" joined by ',' (src/backend/FlameGPUPrinter.cpp:226-245)
template <typename... A>
inline void seq_log(abl_sim *sim, const char *fmt, A... args) {
  char row[1024];
  snprintf(row, sizeof row, fmt, args...);
  seq_note(abl_hip_log_csv(sim, row));
}

}  // namespace gen

// What a step library and the runtime have to agree on: the structures they
// hand each other (their sizes, taken when either is compiled) and what the
// members mean (kStepContract, counted up with every change that sizes do not
// show).
constexpr uint64_t kStepContract = 2;
constexpr uint64_t program_abi() {
  uint64_t h = kStepContract;
  for (const uint64_t size : {(uint64_t) sizeof(ProgramDesc), (uint64_t) sizeof(StepDesc),
                              (uint64_t) sizeof(StepLaunch), (uint64_t) sizeof(NListArgs),
                              (uint64_t) sizeof(DeltaArgs)})
    h = (h ^ size) * 0x100000001B3ull;
  return h;
}

// Register a generated step program with the runtime (abl_runtime.hip); a
// generated library calls it from a static initialiser.  `abi` as the library was
// compiled: a library built for other structures is refused, and creating its
// program fails saying so.  `writes_flags`: steps that remove or add write every
// agent's flag (StepLaunch::dead); for others the runtime clears the flags before
// each step.
bool register_program(const ProgramDesc *desc, uint64_t abi, bool writes_flags);

// The form of step programs emitted earlier, which write a flag only to set it.
static inline bool register_program(const ProgramDesc *desc) {
  return register_program(desc, program_abi(), false);
}

}  // namespace abl
