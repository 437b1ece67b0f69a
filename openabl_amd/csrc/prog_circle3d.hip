// prog_circle3d.hip -- the circle3d program (examples/circle3d.abl,
// circle3d_clustered.abl): host initialisation and registration; the step is
// in prog_circle.hpp.
#include "prog_circle.hpp"

namespace abl {
namespace {

// main() of circle3d_clustered.abl before simulate (num_clusters = 0 gives
// circle3d.abl's plain random(environment.max)):
//   per_cluster = num_clusters > 0 ? int((1.0 - bg) * float(N)) / num_clusters : 0
//   for each cluster: centre = random(env.max);
//     per_cluster times: dx, dy, dz = gaussian(sigma) (in that order)
//                        add(Point { pos: clamp(centre + float3(dx,dy,dz), env.max) })
//   N - per_cluster * num_clusters times: add(Point { pos: random(env.max) })
// gaussian(s) = s * sqrt(-2 * log(1.0 - u1)) * cos(2.0 * PI * u2), u1 drawn
// first; PI is the folded literal 3.14159.  float3 random draws run z, y, x
// (gcc's right-to-left argument order).
template <typename F>
F gaussian(F sigma) {
  const F pi = (F) 3.14159;
  const F u1 = host_random<F>((F) 0, (F) 1.0);
  const F u2 = host_random<F>((F) 0, (F) 1.0);
  return (F) ((sigma * sqrt(((F) (-2)) * log((1.0 - u1)))) * cos(((2.0 * pi) * u2)));
}

template <typename F>
void random3(F W, F out[3]) {
  const F z = host_random<F>((F) 0, W);
  const F y = host_random<F>((F) 0, W);
  const F x = host_random<F>((F) 0, W);
  out[0] = x;
  out[1] = y;
  out[2] = z;
}

template <typename F>
int init3(abl_sim *sim, const double *p) {
  const int n = (int) p[P_NUM_AGENTS];
  const int nclusters = (int) p[P_NUM_CLUSTERS];
  const F W = (F) p[P_W];
  const F sigma = (F) p[P_CLUSTER_SIGMA];
  const F bg = (F) p[P_BACKGROUND_FRACTION];
  const int per_cluster =
      nclusters > 0 ? ((int) ((1.0 - bg) * ((F) n))) / nclusters : 0;
  const int nbackground = n - per_cluster * nclusters;
  std::vector<F> aos;
  aos.reserve(3 * (size_t) (n > 0 ? n : 0));
  for (int c = 0; c < nclusters; c++) {
    F centre[3];
    random3<F>(W, centre);
    for (int i = 0; i < per_cluster; i++) {
      const F dx = gaussian<F>(sigma);
      const F dy = gaussian<F>(sigma);
      const F dz = gaussian<F>(sigma);
      const F d[3] = {dx, dy, dz};
      for (int k = 0; k < 3; k++) {
        const F v = centre[k] + d[k];
        aos.push_back(v < (F) 0 ? (F) 0 : (v > W ? W : v));
      }
    }
  }
  for (int i = 0; i < nbackground; i++) {
    F q[3];
    random3<F>(W, q);
    aos.insert(aos.end(), q, q + 3);
  }
  return abl_hip_upload(sim, 0, aos.data(), aos.size() / 3);
}

int host_init3(abl_sim *sim, const double *p, int precision) {
  return precision == ABL_PREC_F32 ? init3<float>(sim, p) : init3<double>(sim, p);
}

void env3(const double *p, double lo[3], double hi[3], double *g) {
  lo[0] = lo[1] = lo[2] = 0.0;
  hi[0] = hi[1] = hi[2] = p[P_W];
  *g = 2.0 * p[P_R];
}

}  // namespace

const ProgramDesc *program_circle3d() {
  static const ProgramDesc d = {
      "circle3d",
      {{"Point", {{"pos", K_FLOAT3, true}}}},
      {{"num_timesteps", 100}, {"num_agents", 1000}, {"rho", 0.05}, {"k_rep", 0.05},
       {"k_att", 0.01}, {"r", 5.0}, {"W", 27.1442}, {"num_clusters", 64},
       {"cluster_sigma", 20.0}, {"background_fraction", 0.2}},
      {{"move_point", 0, 0, "r", 2.0, 0x7u, launch_move_point<3>, false, 0, true, nullptr,
        false, false, walks_tiles}},
      env3,
      host_init3,
      nullptr,
      nullptr,
      true,
  };
  return &d;
}

}  // namespace abl
