// The emitted source of a step kernel compiled for the host: one workgroup of
// tvbx_step_split at a time, every lane a fiber that runs from barrier to
// barrier.  Between two barriers nothing orders the waves, so any order of
// the fibers is a legal one: what the results are must not depend on it.
// Compiled with -DKERNEL_SRC="<path of the emitted source>".
#include <ucontext.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <vector>

using std::isfinite;

#define __device__
#define __global__
#define __shared__ static
#define __forceinline__ inline
#define __noinline__
#define __launch_bounds__(...)
#define asm
#define volatile(...)

struct dim { unsigned x = 1, y = 1, z = 1; };
static dim threadIdx, blockIdx, blockDim, gridDim;
struct alignas(16) float4 { float x, y, z, w; };
struct uint2 { unsigned x, y; };
struct uint4 { unsigned x, y, z, w; };
static inline uint4 make_uint4(unsigned x, unsigned y, unsigned z, unsigned w) {
  return uint4{x, y, z, w};
}
static inline uint2 make_uint2(unsigned x, unsigned y) { return uint2{x, y}; }
static inline unsigned __umulhi(unsigned a, unsigned b) {
  return (unsigned)(((unsigned long long)a * b) >> 32);
}
template <typename T> static T min(T a, T b) { return b < a ? b : a; }
template <typename T> static T max(T a, T b) { return a < b ? b : a; }
static inline void sincospif(float v, float *s, float *c) {
  *s = sinf(3.14159265358979f * v);
  *c = cosf(3.14159265358979f * v);
}
static inline float __uint_as_float(unsigned v) {
  float f;
  memcpy(&f, &v, 4);
  return f;
}
static inline unsigned __float_as_uint(float v) {
  unsigned u;
  memcpy(&u, &v, 4);
  return u;
}
static inline int __float_as_int(float v) { return (int)__float_as_uint(v); }
static inline float __int_as_float(int v) { return __uint_as_float(v); }
static inline unsigned atomicAdd(unsigned *p, unsigned v) {
  const unsigned o = *p;
  *p += v;
  return o;
}
static inline unsigned atomicExch(unsigned *p, unsigned v) {
  const unsigned o = *p;
  *p = v;
  return o;
}
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_load(p, ...) (*(p))
#define __amdgpu_buffer_rsrc_t const char *
#define __builtin_amdgcn_make_buffer_rsrc(p, ...) ((const char *)(p))
#define __builtin_amdgcn_raw_buffer_load_b32(r, v, s, ...) \
  (*(const unsigned *)((r) + (unsigned)(v) + (unsigned)(s)))
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))
#define __builtin_amdgcn_readfirstlane(x) (x)  // of uniform values only
#define __builtin_amdgcn_readlane(x, l) (x)    // not reached here
#define __builtin_amdgcn_s_setprio(x)
#define __builtin_amdgcn_s_sleep(x)
#define __builtin_amdgcn_sched_barrier(x)
static void barrier();
#define __syncthreads() barrier()

#include KERNEL_SRC

#undef asm
#undef volatile

static ucontext_t g_main, g_ctx[192];
static int g_cur;
static bool g_done[192];
static int g_waits[192];
static tvbx_step_args g_args;

static void barrier() {
  ++g_waits[g_cur];
  swapcontext(&g_ctx[g_cur], &g_main);
}

static void lane_main() {
  tvbx_step_split(g_args);
  g_done[g_cur] = true;
  swapcontext(&g_ctx[g_cur], &g_main);
}

// One launch of n_steps steps from step 0 (slot 0) over all workgroups, the
// waves of a workgroup in `order` (lanes backwards when `back`).  Returns the
// number of lanes whose barrier count differs from their workgroup's.
extern "C" int split_launch(int N, int pitch, int H, int nnz, int steps,
                            float dt, const int *row, const unsigned *cd,
                            const float *w, float *state, float *ring,
                            const float *p_inst, const float *p_node,
                            unsigned *bad,
                            const int *order, int back) {
  const size_t stack = 256 << 10;
  static std::vector<char> mem(192 * stack);
  tvbx_step_args a;
  memset(&a, 0, sizeof a);
  a.n_node = N;
  a.n_inst = a.pitch = a.group_size = a.param_pitch = pitch;
  a.horizon = H;
  a.n_ring = 1;
  a.nnz = nnz;
  a.n_steps = steps;
  a.node_block = 1;
  a.dt = dt;
  a.sqrt_dt = sqrtf(dt);
  a.row = row;
  a.coldelay = cd;
  a.weight = w;
  a.state = state;
  a.ring = ring;
  a.p_inst = p_inst;
  a.p_node = p_node;
  a.bad = bad;
  a.ring_scale = a.ring_unscale = 1.0f;
  a.ring32 = 1;
  g_args = a;
  blockDim.x = 192;
  gridDim.x = pitch / 16;
  gridDim.y = N;
  int uneven = 0;
  for (blockIdx.y = 0; blockIdx.y < gridDim.y; ++blockIdx.y)
    for (blockIdx.x = 0; blockIdx.x < gridDim.x; ++blockIdx.x) {
      for (int t = 0; t < 192; ++t) {
        getcontext(&g_ctx[t]);
        g_ctx[t].uc_stack.ss_sp = mem.data() + t * stack;
        g_ctx[t].uc_stack.ss_size = stack;
        g_ctx[t].uc_link = nullptr;
        makecontext(&g_ctx[t], lane_main, 0);
        g_done[t] = false;
        g_waits[t] = 0;
      }
      for (int left = 192; left > 0;)
        for (int k = 0; k < 3; ++k)
          for (int l = 0; l < 64; ++l) {
            const int t = 64 * order[k] + (back ? 63 - l : l);
            if (g_done[t]) continue;
            g_cur = t;
            threadIdx.x = t;
            swapcontext(&g_main, &g_ctx[t]);
            left -= g_done[t];
          }
      for (int t = 1; t < 192; ++t) uneven += g_waits[t] != g_waits[0];
    }
  return uneven;
}
