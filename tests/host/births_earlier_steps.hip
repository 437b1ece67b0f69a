// steps.hip -- generated by openabl-hip (-b hip) from births.abl.
// Device program: one kernel per step function over the runtime's struct-of-arrays
// agents; registers program "births_earlier" with the runtime when loaded.
//
// Kept as an earlier version of the compiler wrote it (examples/births.abl): its
// steps write add() and removeCurrent() flags only to set them, and it registers
// without saying what it was built for.  tests/test_step_contract.py runs it.
#include <math.h>
#include <stdio.h>

#include "abl_gen_device.hpp"

namespace gen_births_earlier {
using namespace abl;
using namespace abl::gen;

template <typename F>
struct Cell {
  vec2<F> pos;
  int life;
  int age;
};

template <typename F>
__device__ inline Cell<F> load_Cell(void *const *cols, int i) {
  Cell<F> r;
  r.pos.x = col_at<F>(cols, 0, i); r.pos.y = col_at<F>(cols, 1, i); r.life = col_at<int32_t>(cols, 2, i); r.age = col_at<int32_t>(cols, 3, i); 
  return r;
}

template <typename F>
struct Prog {
  static constexpr F PI = (F) 3.14159;
  static constexpr int num_agents = (int) 3000;
  static constexpr int num_timesteps = (int) 12;
  template <typename C>
  static __device__ vec2<F> random_1(C &c_, vec2<F> min, vec2<F> max) {
    return v2_create<F>((F) (c_.random_float((F) (min.x), (F) (max.x))), (F) (c_.random_float((F) (min.y), (F) (max.y))));
  }
  template <typename C>
  static __device__ vec3<F> random_2(C &c_, vec3<F> min, vec3<F> max) {
    return v3_create<F>((F) (c_.random_float((F) (min.x), (F) (max.x))), (F) (c_.random_float((F) (min.y), (F) (max.y))), (F) (c_.random_float((F) (min.z), (F) (max.z))));
  }
  template <typename C>
  static __device__ F random_3(C &c_, F max) {
    return c_.random_float((F) (0), (F) (max));
  }
  template <typename C>
  static __device__ vec2<F> random_4(C &c_, vec2<F> max) {
    return random_1(c_, v2_fill<F>((F) (0)), max);
  }
  template <typename C>
  static __device__ vec3<F> random_5(C &c_, vec3<F> max) {
    return random_2(c_, v3_fill<F>((F) (0)), max);
  }
  template <typename C>
  static __device__ int randomInt_1(C &c_, int max) {
    return c_.random_int(0, max);
  }
  static __host__ __device__ F clamp(F pos, F min, F max) {
    return ((pos < min) ? min : ((pos > max) ? max : pos));
  }
  static __host__ __device__ vec2<F> clamp_1(vec2<F> pos, vec2<F> min, vec2<F> max) {
    return v2_create<F>((F) (((pos.x < min.x) ? min.x : ((pos.x > max.x) ? max.x : pos.x))), (F) (((pos.y < min.y) ? min.y : ((pos.y > max.y) ? max.y : pos.y))));
  }
  static __host__ __device__ vec3<F> clamp_2(vec3<F> pos, vec3<F> min, vec3<F> max) {
    return v3_create<F>((F) (((pos.x < min.x) ? min.x : ((pos.x > max.x) ? max.x : pos.x))), (F) (((pos.y < min.y) ? min.y : ((pos.y > max.y) ? max.y : pos.y))), (F) (((pos.z < min.z) ? min.z : ((pos.z > max.z) ? max.z : pos.z))));
  }
  static __host__ __device__ F clamp_3(F pos, F max) {
    return clamp(pos, 0, max);
  }
  static __host__ __device__ vec2<F> clamp_4(vec2<F> pos, vec2<F> max) {
    return clamp_1(pos, v2_fill<F>((F) (0)), max);
  }
  static __host__ __device__ vec3<F> clamp_5(vec3<F> pos, vec3<F> max) {
    return clamp_2(pos, v3_fill<F>((F) (0)), max);
  }
  static __host__ __device__ F wraparound(F pos, F max) {
    return ((pos < 0) ? (max + pos) : ((pos >= max) ? (pos - max) : pos));
  }
  static __host__ __device__ vec2<F> wraparound_1(vec2<F> pos, vec2<F> max) {
    return v2_create<F>((F) (((pos.x < 0) ? (max.x + pos.x) : ((pos.x >= max.x) ? (pos.x - max.x) : pos.x))), (F) (((pos.y < 0) ? (max.y + pos.y) : ((pos.y >= max.y) ? (pos.y - max.y) : pos.y))));
  }
  static __host__ __device__ vec3<F> wraparound_2(vec3<F> pos, vec3<F> max) {
    return v3_create<F>((F) (((pos.x < 0) ? (max.x + pos.x) : ((pos.x >= max.x) ? (pos.x - max.x) : pos.x))), (F) (((pos.y < 0) ? (max.y + pos.y) : ((pos.y >= max.y) ? (pos.y - max.y) : pos.y))), (F) (((pos.z < 0) ? (max.z + pos.z) : ((pos.z >= max.z) ? (pos.z - max.z) : pos.z))));
  }
  static __host__ __device__ bool is_inside(vec2<F> pos, vec2<F> max) {
    return ((((pos.x >= 0) && (pos.y >= 0)) && (pos.x <= max.x)) && (pos.y <= max.y));
  }
  // step age
  template <typename C>
  static __device__ void age(C &c_, const Cell<F> &in, Cell<F> &out) {
    out.age = (in.age + 1);
    out.life = (in.life - 1);
  }
  // step breed
  template <typename C>
  static __device__ void breed(C &c_, const Cell<F> &in, Cell<F> &out) {
    if (((in.age % 4) == 0)) {
      {
        Cell<F> t3_ = ({ Cell<F> t4_; t4_.pos = in.pos; t4_.life = (3 + in.age); t4_.age = 0; t4_; });
        col_put<F>(c_.a.birth, 0, c_.i, t3_.pos.x); col_put<F>(c_.a.birth, 1, c_.i, t3_.pos.y); col_put<int32_t>(c_.a.birth, 2, c_.i, t3_.life); col_put<int32_t>(c_.a.birth, 3, c_.i, t3_.age); 
        c_.a.born[c_.i] = 1;
      }
    }
    out.life = in.life;
  }
  // step starve
  template <typename C>
  static __device__ void starve(C &c_, const Cell<F> &in, Cell<F> &out) {
    if ((in.life < 1)) {
      c_.remove_current();
    }
    out.age = in.age;
  }
  // step renew
  template <typename C>
  static __device__ void renew(C &c_, const Cell<F> &in, Cell<F> &out) {
    if ((in.age > 9)) {
      {
        Cell<F> t5_ = ({ Cell<F> t6_; t6_.pos = in.pos; t6_.life = 6; t6_.age = 1; t6_; });
        col_put<F>(c_.a.birth, 0, c_.i, t5_.pos.x); col_put<F>(c_.a.birth, 1, c_.i, t5_.pos.y); col_put<int32_t>(c_.a.birth, 2, c_.i, t5_.life); col_put<int32_t>(c_.a.birth, 3, c_.i, t5_.age); 
        c_.a.born[c_.i] = 1;
      }
      c_.remove_current();
    }
    out.life = in.life;
  }
};

template <typename F, bool BY_ID>
__global__ __launch_bounds__(256) void k_age(GenArgs a) {
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const int i = (int) (blk * blockDim.x + threadIdx.x);
  if (i >= a.n) return;
  Ctx<F, BY_ID> c_(a, i);
  const Cell<F> in_ = load_Cell<F>(a.in, i);
  Cell<F> out_ = in_;
  Prog<F>::age(c_, in_, out_);
  col_put<int32_t>(a.out, 2, i, out_.life); col_put<int32_t>(a.out, 3, i, out_.age); 
}
template <typename F>
void launch_age_t(const StepLaunch &L) {
  const GenArgs a = make_args(L);
  const unsigned nb = grid_blocks(L.n, 256);
  if (L.order == 1) hipLaunchKernelGGL((k_age<F, true>), nb, 256, 0, L.stream, a);
  else hipLaunchKernelGGL((k_age<F, false>), nb, 256, 0, L.stream, a);
}
void launch_age(const StepLaunch &L) {
  if (L.precision == ABL_PREC_F32) launch_age_t<float>(L);
  else launch_age_t<double>(L);
}

template <typename F, bool BY_ID>
__global__ __launch_bounds__(256) void k_breed(GenArgs a) {
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const int i = (int) (blk * blockDim.x + threadIdx.x);
  if (i >= a.n) return;
  Ctx<F, BY_ID> c_(a, i);
  const Cell<F> in_ = load_Cell<F>(a.in, i);
  Cell<F> out_ = in_;
  Prog<F>::breed(c_, in_, out_);
  
}
template <typename F>
void launch_breed_t(const StepLaunch &L) {
  const GenArgs a = make_args(L);
  const unsigned nb = grid_blocks(L.n, 256);
  if (L.order == 1) hipLaunchKernelGGL((k_breed<F, true>), nb, 256, 0, L.stream, a);
  else hipLaunchKernelGGL((k_breed<F, false>), nb, 256, 0, L.stream, a);
}
void launch_breed(const StepLaunch &L) {
  if (L.precision == ABL_PREC_F32) launch_breed_t<float>(L);
  else launch_breed_t<double>(L);
}

template <typename F, bool BY_ID>
__global__ __launch_bounds__(256) void k_starve(GenArgs a) {
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const int i = (int) (blk * blockDim.x + threadIdx.x);
  if (i >= a.n) return;
  Ctx<F, BY_ID> c_(a, i);
  const Cell<F> in_ = load_Cell<F>(a.in, i);
  Cell<F> out_ = in_;
  Prog<F>::starve(c_, in_, out_);
  
}
template <typename F>
void launch_starve_t(const StepLaunch &L) {
  const GenArgs a = make_args(L);
  const unsigned nb = grid_blocks(L.n, 256);
  if (L.order == 1) hipLaunchKernelGGL((k_starve<F, true>), nb, 256, 0, L.stream, a);
  else hipLaunchKernelGGL((k_starve<F, false>), nb, 256, 0, L.stream, a);
}
void launch_starve(const StepLaunch &L) {
  if (L.precision == ABL_PREC_F32) launch_starve_t<float>(L);
  else launch_starve_t<double>(L);
}

template <typename F, bool BY_ID>
__global__ __launch_bounds__(256) void k_renew(GenArgs a) {
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const int i = (int) (blk * blockDim.x + threadIdx.x);
  if (i >= a.n) return;
  Ctx<F, BY_ID> c_(a, i);
  const Cell<F> in_ = load_Cell<F>(a.in, i);
  Cell<F> out_ = in_;
  Prog<F>::renew(c_, in_, out_);
  
}
template <typename F>
void launch_renew_t(const StepLaunch &L) {
  const GenArgs a = make_args(L);
  const unsigned nb = grid_blocks(L.n, 256);
  if (L.order == 1) hipLaunchKernelGGL((k_renew<F, true>), nb, 256, 0, L.stream, a);
  else hipLaunchKernelGGL((k_renew<F, false>), nb, 256, 0, L.stream, a);
}
void launch_renew(const StepLaunch &L) {
  if (L.precision == ABL_PREC_F32) launch_renew_t<float>(L);
  else launch_renew_t<double>(L);
}

void env(const double *, double lo[3], double hi[3], double *g) {
  lo[0] = 0.0; hi[0] = 100.0;
  lo[1] = 0.0; hi[1] = 100.0;
  lo[2] = 0.0; hi[2] = 0.0;
  *g = 10;
}

const ProgramDesc *program() {
  static const ProgramDesc d = {
    "births_earlier",
    {{"Cell", {{"pos", K_FLOAT2, true}, {"life", K_INT, false}, {"age", K_INT, false}}}},
    {},
    {{"age", 0, -1, nullptr, 0.0, 12u, launch_age, false, 0, false, nullptr},
     {"breed", 0, -1, nullptr, 0.0, 0u, launch_breed, false, 1, false, nullptr},
     {"starve", 0, -1, nullptr, 0.0, 0u, launch_starve, true, 0, false, nullptr},
     {"renew", 0, -1, nullptr, 0.0, 0u, launch_renew, true, 1, false, nullptr}},
    env,
    nullptr,
    nullptr,
    nullptr,
    false,
    nullptr,
  };
  return &d;
}

const bool registered = register_program(program());

}  // namespace gen_births_earlier
