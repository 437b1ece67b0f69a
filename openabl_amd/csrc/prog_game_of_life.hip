// prog_game_of_life.hip -- step program for examples/game_of_life.abl: the
// device code `-b hip` emits for step_move.
//
//   living = 0
//   for nx in near(in, radius): living += nx.alive ? 1 : 0   (includes self)
//   alive: living -= 1; out.alive = living >= 2 && living <= 3
//   dead:  out.alive = living == 3
//   out.pos = in.pos
// The assignment out.pos = in.pos copies a member onto itself, so the
// program does not write the position columns at all (the step's write mask
// holds only `alive`): positions never change, the grid is built once, and a
// step moves 1 byte per cell plus the neighbours' flags.  Integer arithmetic:
// results are bit-exact whatever the visiting order.
#include <vector>

#include "abl_runtime.hpp"
#include "abl_pipeline.hpp"

namespace abl {
namespace {

enum { P_RADIUS, P_DEBUG, P_ALIVE_FRACTION, P_NUM_AGENTS, P_NUM_TIMESTEPS, P_SIZE };

template <typename F>
struct LifeArgs {
  const F *px, *py;
  const uint8_t *alive;
  uint8_t *out_alive;
  GridView g;
  float near_t;
  int n;
  FixedNeighbours fx;
};

__device__ __forceinline__ uint8_t life_rule(bool alive, int living) {
  bool out;
  if (alive) {
    living -= 1;
    out = living >= 2 && living <= 3;
  } else {
    out = living == 3;
  }
  return out ? 1 : 0;
}

// Cells within the radius of agent i that are alive, by the stencil.
template <typename F>
__device__ __forceinline__ int life_walk(const LifeArgs<F> &a, int i) {
  const F x = a.px[i], y = a.py[i];
  const int3 c = cell_of<F>(a.g, x, y, (F) 0);
  int living = 0;
  for_each_candidate(a.g, c.x, c.y, 0, a.g.reach, [&](uint32_t j) {
    const float f = dist_sq_f32<F>(a.px[j], a.py[j], x, y);
    if (f > a.near_t) return;
    living += a.alive[j] ? 1 : 0;
  });
  return living;
}

template <typename F>
__global__ __launch_bounds__(1024) void life_step(LifeArgs<F> a) {
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const int i = (int) (blk * blockDim.x + threadIdx.x);
  if (i >= a.n) return;
  a.out_alive[i] = life_rule(a.alive[i] != 0, life_walk(a, i));
}

// Positions never change, so neither does who is whose neighbour: up to eight of
// them, as signed 16-bit distances in slots, are kept for as long as the stored
// order stands, with their number and whether the agent counts itself
// (kLifeSelf).  An agent with more neighbours, or one further off, walks the
// stencil.  A timestep is then 19 bytes per agent and eight reads of a byte, where
// the walk tests some 20 candidates (1,048,576 cells, FP64: 8.9 us per timestep
// against 31.8 with the walk by a thread per agent and 38.7 on LDS tiles; FP32 8.6,
// 25.8 and 29.2).
constexpr int kLifeKept = 8;
constexpr uint8_t kLifeSelf = 0x80, kLifeWalk = 0x7F;

template <typename F>
__global__ __launch_bounds__(1024) void life_neighbours(LifeArgs<F> a) {
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const int i = (int) (blk * blockDim.x + threadIdx.x);
  if (i >= a.n) return;
  const F x = a.px[i], y = a.py[i];
  const int3 c = cell_of<F>(a.g, x, y, (F) 0);
  uint64_t lo = 0, hi = 0;
  uint32_t count = 0;
  uint8_t self = 0;
  bool fits = true;
  for_each_candidate(a.g, c.x, c.y, 0, a.g.reach, [&](uint32_t j) {
    const float f = dist_sq_f32<F>(a.px[j], a.py[j], x, y);
    if (f > a.near_t) return;
    if ((int) j == i) {
      self = kLifeSelf;
      return;
    }
    const int d = (int) j - i;
    fits = fits && d >= -32768 && d <= 32767;
    const uint64_t v = (uint64_t) ((uint32_t) d & 0xFFFFu) << (16u * (count & 3u));
    if (count < 4u) lo |= v;
    else if (count < (uint32_t) kLifeKept) hi |= v;
    count++;
  });
  fits = fits && count <= (uint32_t) kLifeKept;
  a.fx.len[i] = fits ? (uint8_t) (count | self) : kLifeWalk;
  a.fx.nb[i] = make_uint4((uint32_t) lo, (uint32_t) (lo >> 32), (uint32_t) hi, (uint32_t) (hi >> 32));
}

template <typename F>
__global__ __launch_bounds__(1024) void life_step_fixed(LifeArgs<F> a) {
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const int i = (int) (blk * blockDim.x + threadIdx.x);
  if (i >= a.n) return;
  const uint8_t len = a.fx.len[i];
  const bool alive = a.alive[i] != 0;
  int living;
  if (len == kLifeWalk) {
    living = life_walk(a, i);
  } else {
    const uint4 e = a.fx.nb[i];
    const uint32_t w[4] = {e.x, e.y, e.z, e.w};
    const int count = len & 0x0F;
    uint8_t v[kLifeKept];
#pragma unroll
    for (int k = 0; k < kLifeKept; k++) {  // all in flight; unused entries read the agent's own
      const int d = (int) (int16_t) (w[k / 2] >> (16 * (k & 1)));
      v[k] = a.alive[k < count ? i + d : i];
    }
    living = (len & kLifeSelf) && alive ? 1 : 0;
#pragma unroll
    for (int k = 0; k < kLifeKept; k++) living += k < count && v[k] ? 1 : 0;
  }
  a.out_alive[i] = life_rule(alive, living);
}

template <typename F>
void launch_typed(const StepLaunch &L) {
  LifeArgs<F> a{};
  a.px = (const F *) L.in.c[0];
  a.py = (const F *) L.in.c[1];
  a.alive = (const uint8_t *) L.in.c[2];
  a.out_alive = (uint8_t *) L.out.c[2];
  a.g = L.grid;
  a.near_t = L.near_t;
  a.n = L.n;
  a.fx = L.fixed;
  const unsigned nb = grid_blocks(L.n, L.block);
  if (!L.fixed.nb) {
    hipLaunchKernelGGL(life_step<F>, nb, L.block, 0, L.stream, a);
    return;
  }
  if (L.fixed.build) hipLaunchKernelGGL(life_neighbours<F>, nb, L.block, 0, L.stream, a);
  hipLaunchKernelGGL(life_step_fixed<F>, nb, L.block, 0, L.stream, a);
}

// main() of game_of_life.abl before simulate:
//   for x in 0..size: for y in 0..size:
//     add(Cell { pos: float2(x + 0.5, y + 0.5), alive: getInit(x, y) })
// getInit = debug ? glider-ish pattern : random(0, 1) < alive_fraction.
// Record layout: {F x, F y, bool alive} padded to the float alignment.
template <typename F>
int init_typed(abl_sim *sim, const double *p) {
  const int size = (int) p[P_SIZE];
  const bool debug = p[P_DEBUG] != 0.0;
  const F alive_fraction = (F) p[P_ALIVE_FRACTION];
  struct Rec {
    F x, y;
    bool alive;
  };
  std::vector<Rec> aos;
  aos.reserve((size_t) size * (size_t) (size > 0 ? size : 0));
  for (int x = 0; x < size; x++) {
    for (int y = 0; y < size; y++) {
      Rec r{};
      r.x = (F) (((F) x) + 0.5);
      r.y = (F) (((F) y) + 0.5);
      if (debug) {
        r.alive = (x == 10 || x == 11 || x == 12) && y == 10;
      } else {
        r.alive = host_random<F>((F) 0, (F) 1) < alive_fraction;
      }
      aos.push_back(r);
    }
  }
  if (abl_hip_agent_size(sim, 0) != sizeof(Rec)) return ABL_ERR_ARG;
  return abl_hip_upload(sim, 0, aos.data(), aos.size());
}

int host_init(abl_sim *sim, const double *p, int precision) {
  return precision == 0 ? init_typed<double>(sim, p) : init_typed<float>(sim, p);
}

void launch_step_move(const StepLaunch &L) {
  if (L.precision == 0) launch_typed<double>(L);
  else launch_typed<float>(L);
}

void env(const double *p, double lo[3], double hi[3], double *g) {
  lo[0] = lo[1] = lo[2] = 0.0;
  hi[0] = hi[1] = p[P_SIZE];
  hi[2] = 0.0;
  *g = p[P_RADIUS];
}

}  // namespace

const ProgramDesc *program_game_of_life() {
  static const ProgramDesc d = {
      "game_of_life",
      {{"Cell", {{"pos", K_FLOAT2, true}, {"alive", K_BOOL, false}}}},
      {{"radius", 1.5}, {"debug", 0}, {"alive_fraction", 0.1}, {"num_agents", 400},
       {"num_timesteps", 100}, {"size", 20}},
      {{"step_move", 0, 0, "radius", 1.0, 0x4u, launch_step_move, false, 0, false,
        nullptr, false, true}},
      env,
      host_init,
  };
  return &d;
}

}  // namespace abl
