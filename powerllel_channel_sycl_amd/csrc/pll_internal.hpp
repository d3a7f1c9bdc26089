// pll_internal.hpp -- shared definitions of the HIP library behind include/pll.h.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "pll.h"

namespace pll {

// Halo-padded field geometry: (nx+2)*(ny+2)*(nz+2), x fastest, logical 0..n+1.
struct Geom {
  int nx, ny, nz;
  long sx, sxy;
  __host__ __device__ long idx(int i, int j, int k) const { return i + sx * j + sxy * k; }
};

// Mesh coefficient arrays (length nz+2, index 0..nz+1) in the field precision.
template <typename T>
struct MeshT {
  const T* dzf;
  const T* dzf_inv;
  const T* dzc_inv;
  const T* dzflzi;
};

// Element k of a table that no kernel of the launch writes, k uniform over the
// wave: a scalar load.  Through an ordinary pointer the compiler cannot rule
// out that the kernel's stores change the table and loads it per lane, in order
// behind every plane load in flight, so that using the coefficient waits for
// all of them.
template <typename T>
__device__ __forceinline__ T uniform_load(const T* p, long k) {
  using C = const __attribute__((address_space(4))) T;
  return reinterpret_cast<C*>(reinterpret_cast<uintptr_t>(p))[k];
}

// Orders a wave's LDS writes before its lanes' later LDS reads of them.  A
// wave's LDS instructions execute in order, so this only has to keep the
// compiler from moving memory operations across it.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Stockham plan of a complex transform of length L held in LDS.
constexpr int kMaxPass = 8;
struct FftPlan {
  int L;
  int npass;
  int tps;  // threads per sequence: one butterfly of the smallest radix each
  int radix[kMaxPass];
  int ns[kMaxPass];        // span before the pass (product of earlier radices)
  int lr[kMaxPass];        // butterflies of the pass, L / radix
  int tws[kMaxPass];       // twiddle stride, L / (ns * radix)
  unsigned mns[kMaxPass];  // ceil(2^32 / ns): division by ns
};

// Blocks are dispatched round-robin over the 8 XCDs of the GPU; this gives each
// XCD a contiguous range of logical blocks, so neighbouring tiles share its L2.
__device__ __forceinline__ unsigned xcd_remap(unsigned b, unsigned n) {
  const unsigned q = n / 8, r = n % 8, x = b % 8, l = b / 8;
  return x * q + (x < r ? x : r) + l;
}

// Row chunks per plane of the bulk-mean reduction: the largest power of two
// <= ny with chunks*nz reaching 2048 partial sums (fewer when ny is small).
// Fewer than 4096 partials unless nz alone exceeds that (then nz).
inline int mean_chunks_for(int ny, int nz) {
  int chunks = 1;
  while (chunks * 2 <= ny && (long)chunks * nz < 2048) chunks *= 2;
  return chunks;
}

// Kernel identifiers for the per-kernel timers.
enum KernelId {
  K_RK1 = 0,
  K_RK2,
  K_RHS,
  K_FFT_X_FWD,
  K_FFT_Y_FWD,
  K_TRID,
  K_FFT_Y_BWD,
  K_FFT_X_BWD,
  K_CORRECT,
  K_MEAN_PARTIAL,
  K_MEAN_FINAL,
  K_FORCE,
  K_BC_VEL,
  K_BC_P,
  K_CHECK,
  K_INIT,
  K_MISC,
  K_FFT_X_FWD_RHS,  // calcRHS fused into the forward x transform
  K_RK_CLOSURE,     // RK stage with the learned eddy viscosity
  K_RK12,           // both RK stages of a step inside a run
  K_PLANE_FWD,      // calcRHS and both forward transforms of a small plane
  K_PLANE_BWD,      // both inverse transforms and p's boundary update
  K_COUNT
};
extern const char* const kKernelNames[K_COUNT];

// Orders the readers of a closure's weights (the stages of the contexts that it is
// attached to, on their streams) and its writers (training and set_params, on
// the closure's): a stage waits for the last writer, a writer for every stage
// enqueued before it.  Held by the closure and its contexts, whichever goes first.
struct ClosureOrder {
  std::mutex m;  // a stage's launch and a writer's, whole
  hipStream_t stream = nullptr;  // the closure's; null when it is gone
  std::vector<pll_context*> readers;
};

// Pending event pair of one timed launch.
struct PendingTimer {
  int kid;
  hipEvent_t start, stop;
};

}  // namespace pll

struct pll_context {
  pll_config cfg;
  pll::Geom g;
  long nfield;  // halo-padded element count
  long nspec;   // nx*ny*nz
  int prec;     // pll_precision
  size_t esz;   // field element size in bytes
  hipStream_t stream = nullptr;

  void* fld[PLL_NFIELD] = {};
  void* fld_alt[3] = {};  // spare u, v, w: the fused stages write here, then the roles swap
  void* spec = nullptr;

  // host mesh in FP64 (index 0..nz+1)
  std::vector<double> dzf_global, dzf, dzf_inv, dzc, dzc_inv, dzflzi, zc_global;
  double dx, dy, dx_inv, dy_inv, re_inv, dt, u_crf;
  double vel_force[3];
  int is_forced[3];

  void* d_mesh = nullptr;      // 4*(nz+2) in field precision: dzf, dzf_inv, dzc_inv, dzflzi
  void* d_rkcoef = nullptr;    // tendency_fast coefficients, nz+2 planes
  double* d_mesh64 = nullptr;  // same, FP64

  // tridiagonal solve: a, c (nz), pre-factored pivot table [k][cy][cx]
  int cxn = 0, cyn = 0;  // nx/2+1, ny/2+1
  double* d_a = nullptr;
  double* d_c = nullptr;
  double* d_piv = nullptr;  // FP64 pivots (FP32-mixed: their reciprocals), cxn*cyn*nz
  // the partitioned solve of the step: b (nz), compact eigenvalues (cxn, cyn)
  // and the pivots of the planes below its segments (k_trid.hip)
  double* d_seg = nullptr;
  int seg_pin = 0;  // the (0,0) column's last pivot is pinned to 0

  // FFT plans and twiddles (in field precision)
  pll::FftPlan plan_x;  // complex length nx/2
  pll::FftPlan plan_y;  // complex length ny
  void* d_rtw_x = nullptr;  // exp(-2 pi i k/nx), k = 0..nx/2
  void* d_twl_x = nullptr;  // exp(-2 pi i t/L), L = nx/2 
  void* d_twl_y = nullptr;  // exp(-2 pi i t/L), L = ny
  bool x_fixed = false, y_fixed = false;
  int rhs_bcfold = 0;  // calcRHS in the x transform reads halos through the boundary rules
  int x_batch = 1;  // rows per block of the run-time-plan x transforms
  int y_tile = 0;   // log2 of the column pairs per block of the y transforms
  int plane_threads = 0;  // threads of the whole-plane transforms (0: not used)

  // reductions
  double* d_partial = nullptr;
  long npartial = 0;
  int mean_chunks = 1;
  long mean_pending = 0;  // partials of the bulk mean that the next transform adds up
  double* d_scalar = nullptr;  // [0..2] means, [3..5] forces, [6..] scratch
  void* d_red = nullptr;       // check-reduction scratch
  long nred = 0;

  // statistics: FP64 per-point sums of the 11 sampled quantities (interior,
  // nz*ny*nx, x fastest); null when not selected
  double* d_stat[11] = {};

  // learned closure (not owned): when attached, the RK stages add the
  // eddy-viscosity stress with the network evaluated in the stage kernel
  pll_closure* closure = nullptr;
  long closure_version = -1;  // the closure's weight version this stream has waited for
  std::shared_ptr<pll::ClosureOrder> closure_order;
  hipEvent_t closure_read = nullptr;  // recorded behind the stages that a writer waits for
  bool closure_reading = false;       // stages enqueued since the last writer
  void* d_feat = nullptr;   // feature coefficients per plane (field precision), 3*(nz+2)
  float* d_nut = nullptr;   // eddy viscosity of the last closure stage, nx*ny*nz

  // device bytes allocated for this context (ctx_malloc)
  size_t dev_bytes = 0;

  // timers
  bool timing = false;
  std::vector<pll::PendingTimer> pending;
  std::vector<hipEvent_t> event_pool;
  double timer_ms[pll::K_COUNT] = {};
  long timer_launches[pll::K_COUNT] = {};
};

namespace pll {

// ---- error reporting --------------------------------------------------------
void set_error(const std::string& msg);
int fail(int code, const std::string& msg);
int hip_fail(hipError_t e, const char* what);
const char* last_error_cstr();

#define PLL_HIP_TRY(expr)                                  \
  do {                                                      \
    hipError_t _e = (expr);                                 \
    if (_e != hipSuccess) return ::pll::hip_fail(_e, #expr); \
  } while (0)

// hipMalloc of a buffer the context owns, counted in pll_device_bytes.
template <typename P>
hipError_t ctx_malloc(pll_context* c, P** p, size_t bytes) {
  hipError_t e = hipMalloc(reinterpret_cast<void**>(p), bytes);
  if (e == hipSuccess) c->dev_bytes += bytes;
  return e;
}

// ---- timers -------------------------------------------------------------------
void timer_begin(pll_context* c, int kid, PendingTimer* out);
void timer_end(pll_context* c, PendingTimer* t);
int timer_collect(pll_context* c);

struct TimerScope {
  pll_context* c;
  PendingTimer t;
  bool on;
  TimerScope(pll_context* ctx, int kid) : c(ctx), on(ctx->timing) {
    if (on) timer_begin(c, kid, &t);
  }
  ~TimerScope() {
    if (on) timer_end(c, &t);
  }
};

// ---- launchers (implemented in the .hip files) -------------------------------------
// stencils and pointwise kernels (k_stencil.hip)
// A stage on its own; with a closure attached, the closure's.  acc (stage 2): the
// bulk mean of the new u is left for the next transform (force_from_partials);
// bcload (plain stage 2): rebuild the source's halos on load (u1's boundary update
// not run)
int launch_rk(pll_context* c, int stage, int acc = 0, int bcload = 0);
// The stage of a context with an attached closure (k_closure.hip).  deferred (stage
// 1): the previous step's projection, forcing and boundary update first; halo
// (stage 1): u1's boundary update is written too; acc as above.
int launch_rk_closure(pll_context* c, int stage, int deferred, int acc, int halo);
// Takes the context off its closure's readers; a writer still waits for its stages.
int closure_detach(pll_context* c);
// the closure stages' bulk-mean partials fit d_partial (the fused step sequence)
bool closure_fused_available(const pll_context* c);
// forceVel's bulk mean of u and its force from n FP64 block partials in
// d_partial, into d_scalar[0] and d_scalar[3]: left to the forward x transform
// with calcRHS, which follows every stage 2 that sums partials
int force_from_partials(pll_context* c, long n);

int rk_setup(pll_context* c);  // per-plane coefficients of the stages
int launch_calc_rhs(pll_context* c);
// Both RK stages of a step inside a run, the previous step's projection,
// forcing and boundary update applied on load; u1out: u1 is left in its arrays.
int launch_rk12(pll_context* c, int acc, int u1out);
// with_force: the force that is on the device is added as well (forceVel)
int launch_correct_vel(pll_context* c, bool with_force);
int launch_mean(pll_context* c, int field, double nxg, double nyg, double* d_out);
int launch_force(pll_context* c);
// which: 0 u, v, w; 1 u1, v1, w1; 2 both
int launch_bc_vel(pll_context* c, int which, int walls_only = 0);
int launch_bc_p(pll_context* c);
int launch_add_scalar(pll_context* c, int field, double value);
int launch_init_flow(pll_context* c, const double* d_prof, int with_noise, double noise,
                     const uint32_t seeds[3]);
int launch_scale_by_inverse_mean(pll_context* c, int field, const double* d_mean, double u_ref);
int launch_max_div(pll_context* c, pll_value_index* out);
int launch_max_cfl(pll_context* c, pll_value_index* out);
int launch_check_nan(pll_context* c, int field, int* passed);

// transforms and the tridiagonal solve (k_fft.hip, k_trid.hip)
int fft_setup(pll_context* c);
// One pass of the transforms with a compiled-in length n (k_fft_fixed.hip).
enum class FftPass { x_fwd, x_bwd, y_fwd, y_bwd };
template <typename T, FftPass PASS>
int fft_fixed(pll_context* c, int n, bool step);
int launch_fft_x_fwd(pll_context* c);
// calcRHS fused into the forward x transform (reads u, v, w; p is not written);
// takes along the bulk mean that force_from_partials left
int launch_fft_x_fwd_rhs(pll_context* c);
// inverse x transform inside the step (p's boundary update included)
int launch_fft_x_bwd_step(pll_context* c);
int launch_fft_x_bwd(pll_context* c);
int launch_fft_y_fwd(pll_context* c);
int launch_fft_y_bwd(pll_context* c);
int trid_setup(pll_context* c);
int launch_trid(pll_context* c);
// the solve inside the step: columns partitioned into register-held segments
int launch_trid_step(pll_context* c);
// The pressure solve of the step (src/mod_poisson_solver.cc:454-510) from p
// (or, with rhs, from calcRHS computed in the x transform's loads) back to p
// with its boundary update.
int launch_poisson_step(pll_context* c, bool rhs);

}  // namespace pll
