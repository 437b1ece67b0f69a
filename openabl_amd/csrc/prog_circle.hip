// prog_circle.hip -- the circle program (examples/circle.abl): host
// initialisation and registration; the step is in prog_circle.hpp.
#include "prog_circle.hpp"

namespace abl {
namespace {

// main() of circle.abl before simulate: num_agents times
//   add(Point { pos: random(float2(W)) })
// random(float2 max) = float2(random(0, max.x), random(0, max.y)) from
// asset/lib.abl; the C backend's gcc evaluates the two calls right to left,
// so y takes the first draw and x the second.
template <typename F>
int init2(abl_sim *sim, const double *p) {
  const int n = (int) p[P_NUM_AGENTS];
  const F W = (F) p[P_W];
  std::vector<F> aos(2 * (size_t) (n > 0 ? n : 0));
  for (int i = 0; i < n; i++) {
    const F y = host_random<F>((F) 0, W);
    const F x = host_random<F>((F) 0, W);
    aos[2 * (size_t) i] = x;
    aos[2 * (size_t) i + 1] = y;
  }
  return abl_hip_upload(sim, 0, aos.data(), (size_t) n);
}

int host_init2(abl_sim *sim, const double *p, int precision) {
  return precision == ABL_PREC_F32 ? init2<float>(sim, p) : init2<double>(sim, p);
}

void env2(const double *p, double lo[3], double hi[3], double *g) {
  lo[0] = lo[1] = lo[2] = 0.0;
  hi[0] = hi[1] = p[P_W];
  hi[2] = 0.0;
  *g = 2.0 * p[P_R];
}

}  // namespace

const ProgramDesc *program_circle() {
  static const ProgramDesc d = {
      "circle",
      {{"Point", {{"pos", K_FLOAT2, true}}}},
      {{"num_timesteps", 100}, {"num_agents", 1000}, {"rho", 0.05}, {"k_rep", 0.05},
       {"k_att", 0.01}, {"r", 5.0}, {"W", 141.421}},
      {{"move_point", 0, 0, "r", 2.0, 0x3u, launch_move_point<2>, false, 0, true, nullptr,
        false, false, walks_tiles}},
      env2,
      host_init2,
      nullptr,
      nullptr,
      true,
  };
  return &d;
}

}  // namespace abl
