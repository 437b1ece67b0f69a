// prog_circle.hpp -- step move_point of examples/circle.abl (2-D, registered by
// prog_circle.hip) and circle3d.abl / circle3d_clustered.abl (3-D, registered
// by prog_circle3d.hip): the device code `-b hip` emits for it.
//
// Arithmetic follows the C backend's generated expression, operation by
// operation and in the same types (src/backend/CPrinter.cpp:148-173,
// GenericCPrinter.cpp:20-75, AnalysisVisitor.cpp:89-112, 971-974):
//   new_pos = in.pos
//   for nx in near(in, 2.0*r):            dist(nx.pos, in.pos) <= 2.0*r
//     pos_dist = dist(in.pos, nx.pos)     (abl_float) sqrtf((float) sum of squares)
//     if (pos_dist == 0) continue
//     sep_dist = pos_dist - r
//     force = sep_dist > 0.0
//       ? ((nx.pos - in.pos) * (abl_float)(k_att * ((2.0*r) - pos_dist))) / pos_dist
//       : (in.pos - nx.pos) * k_rep
//     new_pos = new_pos + force
//   out.pos = clamp(new_pos, float(1), float(W - 1.0))
// The literals 2.0, 0.0 and 1.0 are C doubles, so under use_float the
// bracketed scalar expressions are evaluated in double and rounded to float
// where they are passed on, exactly as the C compiler does.
// Neighbour state is read through the cell-sorted columns; one thread per
// agent, the 3x3 (3x3x3) stencil of cells visited row by row.
#pragma once

#include <math.h>

#include <cmath>
#include <vector>

#include "abl_runtime.hpp"
#include "abl_tile.hpp"

namespace abl {
namespace {

enum { P_NUM_TIMESTEPS, P_NUM_AGENTS, P_RHO, P_K_REP, P_K_ATT, P_R, P_W, P_NUM_CLUSTERS,
       P_CLUSTER_SIGMA, P_BACKGROUND_FRACTION };

// Candidates of a stencil row read at once by the thread-per-agent kernels:
// the walk waits on each read in turn, so a lane's reads are issued in batches.
constexpr uint32_t kRowBatch = 4;

template <typename F, int DIM>
struct CircleArgs {
  const F *p[3];   // in.pos columns (cell-sorted)
  F *o[3];         // out.pos columns
  const int32_t *id;
  GridView g;
  float near_t;
  float rc;        // radius in cell units (row narrowing)
  int cap;         // LDS records per tile
  int n;
  F r, k_rep, k_att, W;
  bool quick;      // circle_quick
};

// One candidate of the near loop: new_pos += force (or skip).
//
// The walks run this for nearly every candidate (some lane of the wave accepts
// it), so they are bound by its VALU issue.  The root by float arithmetic
// instead of a double root, one reciprocal by two Newton steps instead of an
// IEEE division, and one range check for all quotients: FP64 clustered
// circle3d, 1,048,576 agents, thread per agent 1,600 -> 1,190 us per timestep,
// FP32 1,155 -> 910 us; 1,000,003 circle agents on tiles 164 -> 136 us (FP64).
template <typename F, int DIM>
__device__ __forceinline__ void circle_visit(const CircleArgs<F, DIM> &a, const F *x, const F *q,
                                             F *np) {
  // near test: dist(nx.pos, in.pos) > 2.0*r -> continue
  F e[3];
  F s2 = 0;
#pragma unroll
  for (int d = 0; d < DIM; d++) {
    e[d] = q[d] - x[d];
    s2 = d == 0 ? e[d] * e[d] : s2 + e[d] * e[d];
  }
  const float f = (float) s2;
  if (f > a.near_t) return;
  // pos_dist = dist(in.pos, nx.pos): same sum of squares (negated terms)
  const float df = sqrt_rn_f32(f);
  if (df == 0.f) return;
  const F pos_dist = (F) df;
  const F sep_dist = pos_dist - a.r;
  if ((double) sep_dist > 0.0) {
    const F s = (F) ((double) a.k_att * ((2.0 * (double) a.r) - (double) pos_dist));
    // the DIM quotients by pos_dist through one reciprocal (IEEE results):
    // a.quick says that pos_dist and the numerators are in div_ok's range but
    // for numerators near zero
    F num[3];
    F least = DivRange<F>::hi;
    const F y = rcp_rn<F>(df);
#pragma unroll
    for (int d = 0; d < DIM; d++) {
      num[d] = e[d] * s;
      least = least_mag(least, num[d]);
    }
    if (__builtin_expect(a.quick && least >= DivRange<F>::lo, 1)) {
#pragma unroll
      for (int d = 0; d < DIM; d++) np[d] = np[d] + div_by_recip(num[d], pos_dist, y);
    } else {
#pragma unroll
      for (int d = 0; d < DIM; d++) np[d] = np[d] + num[d] / pos_dist;
    }
  } else {
    // (in.pos - nx.pos) * k_rep: the negated difference, exactly
#pragma unroll
    for (int d = 0; d < DIM; d++) np[d] = np[d] + -e[d] * a.k_rep;
  }
}

// Whether every quotient of the attracting force has pos_dist and numerators
// within div_ok's range, numerators near zero aside: accepted pairs are at most
// 2r apart, attracted ones more than r, and |nx.pos - in.pos| <= 2r bounds the
// numerator.  (Factors of two allow for roundings.)
template <typename F>
bool circle_quick(double r, double k_att) {
  const double hi = (double) DivRange<F>::hi, lo = (double) DivRange<F>::lo;
  return r >= 2.0 * lo && r <= hi / 8.0 && std::fabs(k_att) * r * r <= hi / 64.0;
}

// out.pos = clamp(new_pos, float(1), float(W - 1.0))
template <typename F, int DIM>
__device__ __forceinline__ void circle_finish(const CircleArgs<F, DIM> &a, const F *np, uint32_t i,
                                              double *np_out = nullptr) {
  const F lo = (F) 1;
  const F hi = (F) ((double) a.W - 1.0);
#pragma unroll
  for (int d = 0; d < DIM; d++) {
    const F v = np[d];
    const F c = v < lo ? lo : (v > hi ? hi : v);
    a.o[d][i] = c;
    if (np_out) np_out[d] = (double) c;
  }
}

template <typename F, int DIM, bool BY_ID>
__global__ __launch_bounds__(1024) void circle_step(CircleArgs<F, DIM> a) {
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const int i = (int) (blk * blockDim.x + threadIdx.x);
  if (i >= a.n) return;
  F x[3] = {0, 0, 0};
  F np[3] = {0, 0, 0};
#pragma unroll
  for (int d = 0; d < DIM; d++) {
    x[d] = a.p[d][i];
    np[d] = x[d];
  }
  if (BY_ID) {
    const int3 c = cell_of<F>(a.g, x[0], x[1], DIM == 3 ? x[2] : (F) 0);
    auto body = [&](uint32_t j) {
      F q[3] = {0, 0, 0};
#pragma unroll
      for (int d = 0; d < DIM; d++) q[d] = a.p[d][j];
      circle_visit<F, DIM>(a, x, q, np);
    };
    for_each_candidate_by_id(a.g, c.x, c.y, c.z, a.g.reach, a.id, body);
  } else {
    // stencil rows narrowed to the cells within reach; candidates read
    // through buffer resources at one 32-bit offset (a.n * sizeof(F) < 2^31,
    // checked at launch)
    ColBuf cb[3];
#pragma unroll
    for (int d = 0; d < DIM; d++) cb[d] = col_buf(a.p[d], (uint32_t) a.n * (uint32_t) sizeof(F));
    // kRowBatch candidates of a row are read together (their loads in flight
    // at once) and then visited in order; reads past the row's end are not
    // visited, and past the column's end the buffer returns zero
    constexpr uint32_t S = (uint32_t) sizeof(F);
    for_each_candidate_row(a.g, (double) x[0], (double) x[1], DIM == 3 ? (double) x[2] : 0.0, a.rc,
                           [&](uint32_t j0, uint32_t j1) {
                             const uint32_t end = j1 * S;
                             for (uint32_t off = j0 * S; off < end; off += kRowBatch * S) {
                               F q[kRowBatch][3] = {};
#pragma unroll
                               for (int u = 0; u < kRowBatch; u++)
#pragma unroll
                                 for (int d = 0; d < DIM; d++) q[u][d] = col_load<F>(cb[d], off + u * S);
#pragma unroll
                               for (int u = 0; u < kRowBatch; u++)
                                 if (off + u * S < end) circle_visit<F, DIM>(a, x, q[u], np);
                             }
                           });
  }
  circle_finish<F, DIM>(a, np, (uint32_t) i);
}

// LDS-tiled policy (abl_tile.hpp): records are the positions.
template <typename F_, int DIM_>
struct CirclePolicy {
  using F = F_;
  static constexpr int DIM = DIM_, NS = DIM_;
  using Args = CircleArgs<F, DIM>;
  __device__ static void load(const Args &a, uint32_t j, F *r) {
#pragma unroll
    for (int d = 0; d < DIM; d++) r[d] = a.p[d][j];
  }
  struct Acc {
    F np[DIM];
    __device__ void visit(const Args &a, const F *own, const F *nb) {
      circle_visit<F, DIM>(a, own, nb, np);
    }
  };
  __device__ static void begin(const Args &, Acc &s, const F *own) {
#pragma unroll
    for (int d = 0; d < DIM; d++) s.np[d] = own[d];
  }
  __device__ static void finish(const Args &a, Acc &s, const F *, uint32_t i, double *np) {
    circle_finish<F, DIM>(a, s.np, i, np);
  }
};

// ---- FP32-compensated precision (ABL_PREC_F32C) -----------------------------
// Positions stay FP64 in HBM and the step's sum of forces is added to them in
// FP64.  The near loop runs in float on offsets nx.pos - in.pos (LDS records
// are positions relative to the tile centre): float square sum against the
// same threshold, fast float sqrt and reciprocal, and a Kahan-compensated
// float sum of the forces (up to a few hundred neighbours in dense clusters).
template <int DIM>
struct CircleArgsC {
  const double *p[3];
  double *o[3];
  const int32_t *id;
  GridView g;
  float near_t, rc;
  int cap, n;
  float r, k_rep, att_r2;  // att_r2 = 2.0 * r (folded in double, rounded)
  float k_att;
  double hi;                // W - 1.0
};

template <int DIM>
struct CircleAccC {
  KahanF f[DIM];
  // o = nx.pos - in.pos
  __device__ __forceinline__ void visit(const CircleArgsC<DIM> &a, const float *o) {
    float s2 = o[0] * o[0] + o[1] * o[1];
    if (DIM == 3) s2 = s2 + o[2] * o[2];
    if (s2 > a.near_t) return;
    if (s2 == 0.f) return;  // pos_dist == 0
    const float pos_dist = __builtin_amdgcn_sqrtf(s2);
    if (pos_dist - a.r > 0.f) {
      const float s = a.k_att * (a.att_r2 - pos_dist) * rcp_f32(pos_dist);
#pragma unroll
      for (int d = 0; d < DIM; d++) f[d].add(o[d] * s);
    } else {
#pragma unroll
      for (int d = 0; d < DIM; d++) f[d].add(-o[d] * a.k_rep);
    }
  }
};

template <int DIM>
__device__ __forceinline__ void circle_finish_c(const CircleArgsC<DIM> &a, const CircleAccC<DIM> &s,
                                                const double *x, uint32_t i,
                                                double *np_out = nullptr) {
#pragma unroll
  for (int d = 0; d < DIM; d++) {
    const double v = x[d] + s.f[d].value();
    const double c = v < 1.0 ? 1.0 : (v > a.hi ? a.hi : v);
    a.o[d][i] = c;
    if (np_out) np_out[d] = c;
  }
}

template <int DIM, bool BY_ID>
__global__ __launch_bounds__(1024) void circle_step_c(CircleArgsC<DIM> a) {
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const int i = (int) (blk * blockDim.x + threadIdx.x);
  if (i >= a.n) return;
  double x[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int d = 0; d < DIM; d++) x[d] = a.p[d][i];
  CircleAccC<DIM> s;
  if (BY_ID) {
    const int3 c = cell_of<double>(a.g, x[0], x[1], x[2]);
    auto body = [&](uint32_t j) {
      float o[3] = {0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < DIM; d++) o[d] = (float) (a.p[d][j] - x[d]);
      s.visit(a, o);
    };
    for_each_candidate_by_id(a.g, c.x, c.y, c.z, a.g.reach, a.id, body);
  } else {
    ColBuf cb[3];
#pragma unroll
    for (int d = 0; d < DIM; d++) cb[d] = col_buf(a.p[d], (uint32_t) a.n * 8u);
    // batches of kRowBatch reads, as circle_step
    for_each_candidate_row(a.g, x[0], x[1], x[2], a.rc, [&](uint32_t j0, uint32_t j1) {
      const uint32_t end = j1 * 8u;
      for (uint32_t off = j0 * 8u; off < end; off += kRowBatch * 8u) {
        double q[kRowBatch][3] = {};
#pragma unroll
        for (int u = 0; u < kRowBatch; u++)
#pragma unroll
          for (int d = 0; d < DIM; d++) q[u][d] = col_load<double>(cb[d], off + u * 8u);
#pragma unroll
        for (int u = 0; u < kRowBatch; u++) {
          if (off + u * 8u >= end) break;
          float o[3] = {0.f, 0.f, 0.f};
#pragma unroll
          for (int d = 0; d < DIM; d++) o[d] = (float) (q[u][d] - x[d]);
          s.visit(a, o);
        }
      }
    });
  }
  circle_finish_c<DIM>(a, s, x, (uint32_t) i);
}

template <int DIM_>
struct CirclePolicyC {
  using F = float;
  static constexpr int DIM = DIM_, NS = DIM_;
  static constexpr bool kRelative = true;
  using Args = CircleArgsC<DIM>;
  __device__ static void load(const Args &a, uint32_t j, float *r, const double *org) {
#pragma unroll
    for (int d = 0; d < DIM; d++) r[d] = (float) (a.p[d][j] - org[d]);
  }
  __device__ static void position(const Args &a, uint32_t j, double *p) {
#pragma unroll
    for (int d = 0; d < DIM; d++) p[d] = a.p[d][j];
  }
  struct Acc : CircleAccC<DIM> {
    float res[DIM];  // own record's rounding: (pos - org) - own, exact in double
    __device__ void visit(const Args &a, const float *own, const float *nb) {
      float o[3] = {0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < DIM; d++) o[d] = (nb[d] - own[d]) - res[d];
      CircleAccC<DIM>::visit(a, o);
    }
  };
  __device__ static void begin(const Args &, Acc &s, const float *own, const double *p,
                               const double *org) {
#pragma unroll
    for (int d = 0; d < DIM; d++) s.res[d] = (float) ((p[d] - org[d]) - (double) own[d]);
  }
  __device__ static void finish(const Args &a, Acc &s, const float *, uint32_t i, const double *p,
                                double *np) {
    circle_finish_c<DIM>(a, s, p, i, np);
  }
};

template <int DIM>
void launch_c(const StepLaunch &L) {
  CircleArgsC<DIM> a{};
  for (int d = 0; d < DIM; d++) {
    a.p[d] = (const double *) L.in.c[d];
    a.o[d] = (double *) L.out.c[d];
  }
  a.id = L.nb_id;
  a.g = L.grid;
  a.near_t = L.near_t;
  a.rc = L.rc;
  a.n = L.n;
  a.r = (float) L.params[P_R];
  a.k_rep = (float) L.params[P_K_REP];
  a.k_att = (float) L.params[P_K_ATT];
  a.att_r2 = (float) (2.0 * L.params[P_R]);
  a.hi = L.params[P_W] - 1.0;
  using M = CirclePolicyC<DIM>;
  const unsigned nb = grid_blocks(L.n, L.block);
  if (L.order == 1) {
    hipLaunchKernelGGL((circle_step_c<DIM, true>), nb, L.block, 0, L.stream, a);
  } else if (L.tile != 0 && L.grid.reach <= 4) {
    if constexpr (DIM == 3) launch_tiles<M, 8, 4, 4>(L, a);
    else launch_tiles_2d<M>(L, a);
  } else if ((size_t) L.n * 8u < ((size_t) 1 << 31)) {
    hipLaunchKernelGGL((circle_step_c<DIM, false>), nb, L.block, 0, L.stream, a);
  } else {
    hipLaunchKernelGGL((circle_step_c<DIM, true>), nb, L.block, 0, L.stream, a);
  }
}

// By default the LDS tiles serve the lists alone and the stencil is walked by the
// untiled kernel, which is the faster one at every size measured: a force per
// candidate hides its reads, and it has as many blocks as the agents fill.  FP64,
// circle with 1,000 / 64,000 / 1,000,003 agents 26.6 / 37.5 / 107 us per timestep
// with its re-sort (tiles 27.5 / 40.8 / 130), FP32 with 1,000,003 91 (110), circle3d
// with 2,000 agents 387 us (1,867).  (Its buffer offsets end at 2^31 bytes.)  A caller that
// asks for a tile shape gets it.  Not for FP32-compensated, whose tiles round
// offsets from the tile's own origin: lists and stencil would no longer agree to
// the bit.
inline bool on_tiles(const StepLaunch &L, size_t elem) {
  return L.tile != 0 && L.grid.reach <= 4 &&
         (L.nl_mode != 0 || L.tile_given || (size_t) L.n * elem >= ((size_t) 1 << 31));
}

// StepDesc::walks_tiles
inline bool walks_tiles(const StepLaunch &L) {
  if (L.precision == ABL_PREC_F32C) return true;
  return on_tiles(L, L.precision == ABL_PREC_F64 ? sizeof(double) : sizeof(float));
}

template <typename F, int DIM>
void launch_typed(const StepLaunch &L) {
  CircleArgs<F, DIM> a{};
  for (int d = 0; d < DIM; d++) {
    a.p[d] = (const F *) L.in.c[d];
    a.o[d] = (F *) L.out.c[d];
  }
  a.id = L.nb_id;
  a.g = L.grid;
  a.near_t = L.near_t;
  a.rc = L.rc;
  a.n = L.n;
  a.r = (F) L.params[P_R];
  a.k_rep = (F) L.params[P_K_REP];
  a.k_att = (F) L.params[P_K_ATT];
  a.W = (F) L.params[P_W];
  a.quick = circle_quick<F>((double) a.r, (double) a.k_att);
  const unsigned nb = grid_blocks(L.n, L.block);
  // buffer offsets of the untiled cell-order kernel are 32-bit (beyond
  // 2^31 bytes of a column the index-order kernel runs instead)
  const bool untiled_ok = (size_t) L.n * sizeof(F) < ((size_t) 1 << 31);
  if (L.order == 1) {
    hipLaunchKernelGGL((circle_step<F, DIM, true>), nb, L.block, 0, L.stream, a);
  } else if (on_tiles(L, sizeof(F))) {
    if constexpr (DIM == 3) launch_tiles<CirclePolicy<F, DIM>, 8, 4, 4>(L, a);
    else launch_tiles_2d<CirclePolicy<F, DIM>>(L, a);
  } else if (untiled_ok) {
    hipLaunchKernelGGL((circle_step<F, DIM, false>), nb, L.block, 0, L.stream, a);
  } else {
    hipLaunchKernelGGL((circle_step<F, DIM, true>), nb, L.block, 0, L.stream, a);
  }
}

template <int DIM>
void launch_move_point(const StepLaunch &L) {
  if (L.precision == ABL_PREC_F32C) launch_c<DIM>(L);
  else if (L.precision == ABL_PREC_F64) launch_typed<double, DIM>(L);
  else launch_typed<float, DIM>(L);
}

}  // namespace
}  // namespace abl
