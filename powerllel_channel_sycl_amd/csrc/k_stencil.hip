// k_stencil.hip -- momentum RK stages, Poisson RHS, projection, forcing, the
// boundary/halo update, the bulk-velocity reduction, the initial condition and
// the runtime checks.  All kernels are templated on the field type T (double
// for the FP64 path, float for the FP32-mixed path).
//
// FP64 parity: the library is compiled with -ffp-contract=off, and the separate
// stages and routines keep the association of the reference formulas they cite,
// so an FP64 launch of them reproduces the reference arithmetic bit for bit.
// Inside a run the two stages of a step are fused (k_rk12, tendency_fast), in
// another order of operations and as accurately.
#include "pll_internal.hpp"
#include "stencil_ops.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <utility>
#include <vector>

namespace pll {

namespace {

constexpr int kTx = 64;  // threads along x (one wavefront)
constexpr int kTy = 4;   // rows along y per block
constexpr int kRedBlocks = 1024;
constexpr int kRedThreads = 256;

// Stencil value (di, dj, dk) around the thread's cell, read from an LDS ring
// of three tile planes (k-1, k, k+1) of width SX.
template <typename T, int SX>
struct PlaneAcc {
  const T* m;
  const T* z;
  const T* p;
  int c;
  __device__ __forceinline__ T operator()(int di, int dj, int dk) const {
    const T* pl = dk < 0 ? m : (dk > 0 ? p : z);
    return pl[c + di + dj * SX];
  }
};

// The momentum operator with fewer operations, scaled by S = dt (stage 2 halves
// its result): algebraically equal to S*(visc - conv) of tendency_z, with the
// mesh factors gathered into per-plane coefficients (RkCoef) and products fused
// into FMAs: about 95 operations for the three components instead of 150 in
// FP64, 85 in FP32.  It rounds differently from the reference's order, so only
// the FP32-mixed stages and the fused stages inside a run use it; against 80-bit
// arithmetic a run's FP64 error is that of the reference's order.
template <typename T>
struct RkCoef {
  T a1, a2, b1, b2;  // (u,v) face interpolation to k+1/2 and k-1/2
  T zuv, cp, cm;     // S*0.25*dzf_inv(k); S*re_inv*dzc_inv(k|k-1)*dzf_inv(k)
  T zw, dp, dm;      // S*0.25*dzc_inv(k); S*re_inv*dzf_inv(k+1|k)*dzc_inv(k)
  T cdu, cdw;        // FP32's diagonal of the viscous operator: 2 vx + 2 vy + cp + cm (u, v), + dp + dm (w)
};
template <typename T>
__device__ __forceinline__ RkCoef<T> load_coef(const RkCoef<T>* p, int k) {
  static_assert(sizeof(RkCoef<T>) == 12 * sizeof(T), "twelve coefficients");
  const T* f = reinterpret_cast<const T*>(p + k);
  auto c = [&](int n) { return uniform_load(f, n); };
  return RkCoef<T>{c(0), c(1), c(2), c(3), c(4), c(5), c(6), c(7), c(8), c(9), c(10), c(11)};
}
template <typename T>
struct RkUniform {
  T cx, cy, vx, vy, crf;  // S*0.25*dxi, S*0.25*dyi, S*re_inv*dxi^2, S*re_inv*dyi^2, S*0.5*u_crf*dxi
};

// The z-face value of u or v between cells below and above the face, with the
// upper-face weights (a1, a2) of the lower cell, which are the lower-face
// weights (b2, b1) of the upper one: one expression for both.
__device__ __forceinline__ float zface_value(float below, float above, float wb, float wa) {
  return __builtin_fmaf(below, wb, above * wa);
}
__device__ __forceinline__ double zface_value(double below, double above, double wb, double wa) {
  return __builtin_fma(below, wb, above * wa);
}

// The lower z-face convective products of the three components: the
// upper-face products of the cell below, bit for bit, carried up a column like
// tendency_z's ZFace.
template <typename T>
struct ZConv {
  T u, v, w;
};

template <typename T, class A>
__device__ __forceinline__ ZConv<T> zconv_lower(const A& U, const A& V, const A& W,
                                                const RkCoef<T>& q) {
  ZConv<T> z;
  z.u = zface_value(U(0, 0, -1), U(0, 0, 0), q.b2, q.b1) * (W(0, 0, -1) + W(1, 0, -1));
  z.v = zface_value(V(0, 0, -1), V(0, 0, 0), q.b2, q.b1) * (W(0, 0, -1) + W(0, 1, -1));
  const T wb = W(0, 0, -1) + W(0, 0, 0);
  z.w = wb * wb;
  return z;
}

// The lower-face products come from zc, which then receives the upper ones.
template <bool CRF, typename T, class A>
__device__ __forceinline__ void tendency_fast(const A& U, const A& V, const A& W,
                                              const RkCoef<T>& q, const RkUniform<T>& cu, T& iu,
                                              T& iv, T& iw, ZConv<T>& zc) {
  // not held to the reference's rounding: let products fuse into FMAs
#pragma clang fp contract(fast)
  // The viscous part, in FP64 as second differences: they are exact where
  // neighbours are close, and leave a uniform field as it is.  FP32 takes the
  // neighbours' sums minus the diagonal, which is fewer operations (FP64 would gain
  // 1 % of a step by it).
  constexpr bool kDiff = sizeof(T) == 8;
  // FP64: one component at a time, or the compiler reads the LDS values of all
  // three ahead and the registers of a wave no longer fit three waves per SIMD
  // (k_rk12 at 768x384x384: 2442 us without the fence, 2348 us with it; FP32
  // loses 5 % to it)
  auto fence = [] {
    if constexpr (sizeof(T) == 8) __builtin_amdgcn_sched_barrier(0);
  };
  {
    const T q0 = U(0, 0, 0), qe = U(1, 0, 0), qw = U(-1, 0, 0), qn = U(0, 1, 0);
    const T qs = U(0, -1, 0), qt = U(0, 0, 1), qb = U(0, 0, -1);
    const T ae = q0 + qe, aw = qw + q0, an = q0 + qn, as = qs + q0;
    const T at = zface_value(q0, qt, q.a1, q.a2);
    const T vn = V(0, 0, 0) + V(1, 0, 0), vs = V(0, -1, 0) + V(1, -1, 0);
    const T wt = W(0, 0, 0) + W(1, 0, 0);
    const T ct = at * wt;
    const T cb = zc.u;
    zc.u = ct;
    T conv = cu.cx * (ae * ae - aw * aw) + cu.cy * (an * vn - as * vs) + q.zuv * (ct - cb);
    if (CRF) conv += cu.crf * (ae - aw);
    if constexpr (kDiff)
      iu = cu.vx * ((qe - q0) - (q0 - qw)) + cu.vy * ((qn - q0) - (q0 - qs)) +
           q.cp * (qt - q0) - q.cm * (q0 - qb) - conv;
    else
      iu = cu.vx * (qe + qw) + cu.vy * (qn + qs) + q.cp * qt + q.cm * qb - q.cdu * q0 - conv;
  }
  fence();
  {
    const T q0 = V(0, 0, 0), qe = V(1, 0, 0), qw = V(-1, 0, 0), qn = V(0, 1, 0);
    const T qs = V(0, -1, 0), qt = V(0, 0, 1), qb = V(0, 0, -1);
    const T ae = q0 + qe, aw = qw + q0, an = q0 + qn, as = qs + q0;
    const T at = zface_value(q0, qt, q.a1, q.a2);
    const T ue = U(0, 0, 0) + U(0, 1, 0), uw = U(-1, 0, 0) + U(-1, 1, 0);
    const T wt = W(0, 0, 0) + W(0, 1, 0);
    const T ct = wt * at;
    const T cb = zc.v;
    zc.v = ct;
    T conv = cu.cx * (ue * ae - uw * aw) + cu.cy * (an * an - as * as) + q.zuv * (ct - cb);
    if (CRF) conv += cu.crf * (ae - aw);
    if constexpr (kDiff)
      iv = cu.vx * ((qe - q0) - (q0 - qw)) + cu.vy * ((qn - q0) - (q0 - qs)) +
           q.cp * (qt - q0) - q.cm * (q0 - qb) - conv;
    else
      iv = cu.vx * (qe + qw) + cu.vy * (qn + qs) + q.cp * qt + q.cm * qb - q.cdu * q0 - conv;
  }
  fence();
  {
    const T q0 = W(0, 0, 0), qe = W(1, 0, 0), qw = W(-1, 0, 0), qn = W(0, 1, 0);
    const T qs = W(0, -1, 0), qt = W(0, 0, 1), qb = W(0, 0, -1);
    const T ae = q0 + qe, aw = qw + q0, an = q0 + qn, as = qs + q0;
    const T at = q0 + qt;
    const T ue = U(0, 0, 0) * q.a1 + U(0, 0, 1) * q.a2;
    const T uw = U(-1, 0, 0) * q.a1 + U(-1, 0, 1) * q.a2;
    const T vn = V(0, 0, 0) * q.a1 + V(0, 0, 1) * q.a2;
    const T vs = V(0, -1, 0) * q.a1 + V(0, -1, 1) * q.a2;
    const T ct = at * at;
    const T cb = zc.w;
    zc.w = ct;
    T conv = cu.cx * (ue * ae - uw * aw) + cu.cy * (vn * an - vs * as) + q.zw * (ct - cb);
    if (CRF) conv += cu.crf * (ae - aw);
    if constexpr (kDiff)
      iw = cu.vx * ((qe - q0) - (q0 - qw)) + cu.vy * ((qn - q0) - (q0 - qs)) +
           q.dp * (qt - q0) - q.dm * (q0 - qb) - conv;
    else
      iw = cu.vx * (qe + qw) + cu.vy * (qn + qs) + q.dp * qt + q.dm * qb - q.cdw * q0 - conv;
  }
}


constexpr int kRkTx = 64;  // tile width along x (one wavefront per row)
constexpr int kRkTy = 8;   // tile rows along y

// Tile rows of the projection kernel: 4 in FP64 (4-7 % faster than 8 at
// 768x384x384), 8 in FP32.
template <typename T>
constexpr int correct_ty() {
  return std::is_same<T, double>::value ? 4 : kRkTy;
}

// The stencil coefficients of both stages: the mesh and the uniform factors of
// the reference's formulas, and the per-plane tables of tendency_fast.
template <typename T>
struct RkParam {
  MeshT<T> m;
  T dxi, dyi, rei, dt, ucrf, dtdxi, dtdyi, bc_u;
  const RkCoef<T>* coef;  // tendency_fast's, scaled by dt
  RkUniform<T> cu;
};

// What a thread of k_rk12 carries up its column from one plane to the next:
// the lower convective products and the values of the plane below, which the
// viscous terms read.  With them a stage reads only the planes k and k+1.
template <typename T>
struct ZCarry {
  ZConv<T> z;
  T u, v, w;
};

template <typename T, class A>
__device__ __forceinline__ ZCarry<T> carry_start(const A& U, const A& V, const A& W,
                                                 const RkParam<T>& q, int k) {
  return ZCarry<T>{zconv_lower(U, V, W, load_coef(q.coef, k)), U(0, 0, -1), V(0, 0, -1), W(0, 0, -1)};
}

// A stencil accessor whose value below the centre is carried in a register.
template <typename T, int SX>
struct CarryAcc {
  PlaneAcc<T, SX> a;
  T below;
  __device__ __forceinline__ T operator()(int di, int dj, int dk) const {
    return dk < 0 ? below : a(di, dj, dk);
  }
};

// Stage 2's value from the source, dt*F and the old value.  FP64 adds in the
// reference's order (src/mod_calcVel.cc:194,216,238): s + old, added first, would
// round at twice the magnitude twice.  FP32, which its separate stage shares, does
// that: an rms error of the velocities 4-13 % above the other order's.
__device__ __forceinline__ double stage2_value(double s, double i, double old) {
  return ((s + i) + old) * 0.5;
}
__device__ __forceinline__ float stage2_value(float s, float i, float old) {
  return ((s + old) + i) * 0.5f;
}

// Stage 1: o = s + dt*F(s); stage 2: o = (s + dt*F(s) + old)/2, with the carry
// replaced by the next plane's.
template <typename T, int STAGE, bool CRF, int SX>
__device__ __forceinline__ void stage_update(const PlaneAcc<T, SX>& U, const PlaneAcc<T, SX>& V,
                                             const PlaneAcc<T, SX>& W, const RkParam<T>& q, int k,
                                             T ou, T ov, T ow, ZCarry<T>& z, T& o1, T& o2, T& o3) {
  const RkCoef<T> cq = load_coef(q.coef, k);
  const CarryAcc<T, SX> Uc{U, z.u}, Vc{V, z.v}, Wc{W, z.w};
  T iu, iv, iw;
  tendency_fast<CRF>(Uc, Vc, Wc, cq, q.cu, iu, iv, iw, z.z);
  z.u = U(0, 0, 0);
  z.v = V(0, 0, 0);
  z.w = W(0, 0, 0);
  if (STAGE == 1) {
    o1 = z.u + iu;
    o2 = z.v + iv;
    o3 = z.w + iw;
  } else {
    o1 = stage2_value(z.u, iu, ou);
    o2 = stage2_value(z.v, iv, ov);
    o3 = stage2_value(z.w, iw, ow);
  }
}

// The block's FP64 partial of the bulk mean into partial[b], through NT doubles
// of LDS that every thread is done with; the block size is folded onto its
// largest power of two first.
template <int NT>
__device__ __forceinline__ void block_partial(double* red, double s, double* partial, unsigned b) {
  constexpr int P2 = NT >= 1024 ? 1024 : (NT >= 512 ? 512 : 256);
  static_assert(NT >= P2 && NT < 2 * P2, "block size");
  const int t = threadIdx.x;
  red[t] = s;
  __syncthreads();
  if (t < NT - P2) red[t] += red[t + P2];
  __syncthreads();
  for (int h = P2 / 2; h > 0; h >>= 1) {
    if (t < h) red[t] += red[t + h];
    __syncthreads();
  }
  if (t == 0) partial[b] = red[0];
}

// One RK stage.  Stage 1: d = s + dt*F(s).  Stage 2: d = (s + dt*F(s) + d)/2.
// A block owns a 64 x 8 (i,j) tile and marches a chunk of k planes.  The three
// source fields of planes k-1, k, k+1 (tile plus a one-cell halo) sit in an
// LDS ring; plane k+2 is fetched into registers while plane k is computed and
// replaces plane k-1 afterwards, so every source value leaves HBM once per block.
// These stages run where u1 goes through HBM: the reference's routines one by
// one, the first step of a run (nothing of a previous step to apply) and steps
// that force v or w.
//
// With `bcload` every halo cell of the source is rebuilt on load from interior
// cells by the reference's closed-form rules, for a source whose boundary
// update was not run: x/y halos are periodic images, the z ghost planes are
// 2*bc - u for u, -v for v and 0 for w, and w on plane nz is 0
// (src/mod_updateBound.cc:11-144).  With `acc` stage 2 also sums its new u
// times dzflzi(k) in FP64 into partial[block]: the bulk mean of the next
// projected velocity, since the projection changes every x-row's sum only by
// p(nx+1) - p(1) = 0.
// k_rk is the FP32-mixed form (tendency_fast, per-plane coefficients): at up to
// 8 waves per SIMD the other waves cover the wait for a fetch's loads, and the
// late form's registers cost it 6-9 %.
template <typename T, int STAGE, bool CRF>
__global__ __launch_bounds__(kRkTx * kRkTy) void k_rk(Geom g, const T* __restrict__ su,
                                                     const T* __restrict__ sv,
                                                     const T* __restrict__ sw, T* __restrict__ du,
                                                     T* __restrict__ dv, T* __restrict__ dw,
                                                     RkParam<T> q0, int kchunk, int ntx, int nty,
                                                     int acc, const double* __restrict__ dzflzi,
                                                     double* __restrict__ partial, int bcload) {
  constexpr int TX = kRkTx, TY = kRkTy, SX = TX + 2, SY = TY + 2, PL = SX * SY,
                NT = TX * TY;
  constexpr int NPF = (PL + NT - 1) / NT;
  static_assert(std::is_same<T, float>::value, "the FP64 stages run k_rk_late");
  __shared__ T sh[3][3][PL];  // [field][ring slot][tile cell]
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const int ti = (int)(b % (unsigned)ntx), tj = (int)((b / (unsigned)ntx) % (unsigned)nty);
  const int kc = (int)(b / (unsigned)(ntx * nty));
  const int i0 = ti * TX, j0 = tj * TY;  // tile cell (0,0) is the halo corner (i0, j0)
  const int k0 = kc * kchunk + 1, k1 = min(k0 + kchunk - 1, g.nz);
  const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
  const int i = i0 + tx + 1, j = j0 + ty + 1;
  const bool active = i <= g.nx && j <= g.ny;

  long gaddr[NPF];  // plane-relative source address of this thread's tile cells (-1: outside)
#pragma unroll
  for (int n = 0; n < NPF; ++n) {
    const int e = threadIdx.x + n * NT;
    int gx = i0 + e % SX, gy = j0 + e / SX;
    const bool inside = e < PL && gx <= g.nx + 1 && gy <= g.ny + 1;
    if (bcload) {  // halo cells read their periodic image
      gx = gx == 0 ? g.nx : (gx == g.nx + 1 ? 1 : gx);
      gy = gy == 0 ? g.ny : (gy == g.ny + 1 ? 1 : gy);
    }
    gaddr[n] = inside ? gx + g.sx * gy : -1;
  }
  T pre[3][NPF];
  auto fetch = [&](int kk) {
    const bool ghost = bcload && (kk == 0 || kk == g.nz + 1);
    const int ks = ghost ? (kk == 0 ? 1 : g.nz) : kk;
    const bool wzero = bcload && (kk == 0 || kk >= g.nz);
#pragma unroll
    for (int n = 0; n < NPF; ++n)
      if (gaddr[n] >= 0) {
        const long a = gaddr[n] + g.sxy * ks;
        T qu = su[a], qv = sv[a];
        const T qw = wzero ? T(0) : sw[a];
        if (ghost) {
          qu = T(2) * q0.bc_u - qu;  // src/mod_updateBound.cc:92,123
          qv = T(2) * T(0) - qv;
        }
        pre[0][n] = qu;
        pre[1][n] = qv;
        pre[2][n] = qw;
      }
  };
  auto commit = [&](int slot) {
#pragma unroll
    for (int n = 0; n < NPF; ++n)
      if (gaddr[n] >= 0) {
        const int e = threadIdx.x + n * NT;
        sh[0][slot][e] = pre[0][n];
        sh[1][slot][e] = pre[1][n];
        sh[2][slot][e] = pre[2][n];
      }
  };
  if (k0 > k1) {
    if (acc && threadIdx.x == 0) partial[b] = 0.0;
    return;
  }
  double msum = 0.0;  // FP64 partial of the bulk mean (acc)
  fetch(k0 - 1);
  commit(0);
  fetch(k0);
  commit(1);
  fetch(k0 + 1);
  commit(2);
  __syncthreads();
  int sm = 0, s0 = 1, sp = 2;
  const int c = (ty + 1) * SX + tx + 1;
  ZConv<T> zc{};  // the carried lower-face convective products of the thread's column
  if (active) {
    const PlaneAcc<T, SX> U{sh[0][sm], sh[0][s0], sh[0][sp], c};
    const PlaneAcc<T, SX> V{sh[1][sm], sh[1][s0], sh[1][sp], c};
    const PlaneAcc<T, SX> W{sh[2][sm], sh[2][s0], sh[2][sp], c};
    zc = zconv_lower(U, V, W, load_coef(q0.coef, k0));
  }
  for (int k = k0; k <= k1; ++k) {
    const bool more = k + 2 <= k1 + 1;
    if (more) fetch(k + 2);
    if (active) {
      const long a = g.idx(i, j, k);
      T ou = T(0), ov = T(0), ow = T(0);
      if (STAGE == 2) {
        ou = du[a];
        ov = dv[a];
        ow = dw[a];
      }
      const PlaneAcc<T, SX> U{sh[0][sm], sh[0][s0], sh[0][sp], c};
      const PlaneAcc<T, SX> V{sh[1][sm], sh[1][s0], sh[1][sp], c};
      const PlaneAcc<T, SX> W{sh[2][sm], sh[2][s0], sh[2][sp], c};
      const RkCoef<T> q = load_coef(q0.coef, k);
      float iu, iv, iw;
      tendency_fast<CRF>(U, V, W, q, q0.cu, iu, iv, iw, zc);
      if (STAGE == 1) {
        du[a] = U(0, 0, 0) + iu;
        dv[a] = V(0, 0, 0) + iv;
        dw[a] = W(0, 0, 0) + iw;
      } else {
        const T nu = stage2_value(U(0, 0, 0), iu, ou);
        du[a] = nu;
        dv[a] = stage2_value(V(0, 0, 0), iv, ov);
        dw[a] = stage2_value(W(0, 0, 0), iw, ow);
        if (acc) msum += (double)nu * uniform_load(dzflzi, k);
      }
    }
    __syncthreads();
    if (more) commit(sm);
    __syncthreads();
    const int t = sm;
    sm = s0;
    s0 = sp;
    sp = t;
  }
  // the ring is free after the last barrier of the loop
  static_assert(sizeof(sh) >= NT * sizeof(double), "reduction scratch");
  if (acc) block_partial<NT>(reinterpret_cast<double*>(&sh[0][0][0]), msum, partial, b);
}

// The FP64 stages: k_rk's ring and loads in the reference's arithmetic and
// operation order (tendency_z, src/mod_calcVel.cc:81,103,125 and :194,216,238;
// bit-identical to the reference's stages), with the plane loads scheduled
// late.  A fetch only issues the loads of plane k+2 into registers; the
// boundary rules apply when that plane is committed to the ring, after plane k
// has been computed, and plane k's new values are stored after the commit.
// With that arithmetic inside the fetch (k_rk's form) every wave waits for its
// loads there, and a commit after the stores waits for their completion too:
// that form ran 4-5 % slower in FP64 at 768x384x384 (4 waves per SIMD).  Every
// plane load is unconditional (a thread without a tile cell loads the corner
// cell (0, 0) and writes LDS slot PL; w is loaded on every plane and replaced
// by the wall value where it applies): loads that some paths skip leave the
// compiler's wait counting unsure which are still in flight, and it then waits
// for them before the next fetch reuses their registers.  The FP64 tendency
// carries the lower z face, so plane k-1 is not read while plane k is computed
// and one barrier per plane suffices.  Stage 2 issues the point values of plane
// k before the fetch, so that waiting for them leaves the plane in flight.
// tile rows of k_rk_late: 8; 4 rows measured 9 % and 16 rows 5 % slower at
// 768x384x384
constexpr int kLateTy = 8;
template <int STAGE, bool CRF>
__global__ __launch_bounds__(kRkTx * kLateTy, 4) void k_rk_late(
    Geom g, const double* __restrict__ su, const double* __restrict__ sv,
    const double* __restrict__ sw, double* __restrict__ du, double* __restrict__ dv,
    double* __restrict__ dw, RkParam<double> q0, int kchunk, int ntx, int nty, int acc,
    const double* __restrict__ dzflzi, double* __restrict__ partial, int bcload) {
  using T = double;
  constexpr int TX = kRkTx, TY = kLateTy, SX = TX + 2, SY = TY + 2, PL = SX * SY,
                NT = TX * TY;
  constexpr int NPF = (PL + NT - 1) / NT;
  __shared__ T sh[3][3][PL + 1];  // [field][ring slot][tile cell]; slot PL: no cell
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const int ti = (int)(b % (unsigned)ntx), tj = (int)((b / (unsigned)ntx) % (unsigned)nty);
  const int kc = (int)(b / (unsigned)(ntx * nty));
  const int i0 = ti * TX, j0 = tj * TY;  // tile cell (0,0) is the halo corner (i0, j0)
  const int k0 = kc * kchunk + 1, k1 = min(k0 + kchunk - 1, g.nz);
  const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
  const int i = i0 + tx + 1, j = j0 + ty + 1;
  const bool active = i <= g.nx && j <= g.ny;

  long gaddr[NPF];  // plane-relative source address of this thread's tile cells
  int cell[NPF];
#pragma unroll
  for (int n = 0; n < NPF; ++n) {
    const int e = threadIdx.x + n * NT;
    int gx = i0 + e % SX, gy = j0 + e / SX;
    const bool inside = e < PL && gx <= g.nx + 1 && gy <= g.ny + 1;
    if (bcload) {  // halo cells read their periodic image
      gx = gx == 0 ? g.nx : (gx == g.nx + 1 ? 1 : gx);
      gy = gy == 0 ? g.ny : (gy == g.ny + 1 ? 1 : gy);
    }
    gaddr[n] = inside ? gx + g.sx * gy : 0;
    cell[n] = inside ? e : PL;
  }
  T ru[NPF], rv[NPF], rw[NPF];
  auto fetch = [&](int kk) {
    const bool ghost = bcload && (kk == 0 || kk == g.nz + 1);
    const long pofs = g.sxy * (ghost ? (kk == 0 ? 1 : g.nz) : kk);
#pragma unroll
    for (int n = 0; n < NPF; ++n) {
      const long a = gaddr[n] + pofs;
      ru[n] = su[a];
      rv[n] = sv[a];
      rw[n] = sw[a];
    }
  };
  auto commit = [&](int kk, int slot) {
    const bool ghost = bcload && (kk == 0 || kk == g.nz + 1);
    const bool wzero = bcload && (kk == 0 || kk >= g.nz);
#pragma unroll
    for (int n = 0; n < NPF; ++n) {
      T qu = ru[n], qv = rv[n], qw = rw[n];
      if (wzero) qw = T(0);
      if (ghost) {
        qu = T(2) * q0.bc_u - qu;  // src/mod_updateBound.cc:92,123
        qv = T(2) * T(0) - qv;
      }
      sh[0][slot][cell[n]] = qu;
      sh[1][slot][cell[n]] = qv;
      sh[2][slot][cell[n]] = qw;
    }
  };
  if (k0 > k1) {
    if (acc && threadIdx.x == 0) partial[b] = 0.0;
    return;
  }
  fetch(k0 - 1);
  commit(k0 - 1, 0);
  fetch(k0);
  commit(k0, 1);
  fetch(k0 + 1);
  commit(k0 + 1, 2);
  __syncthreads();
  int sm = 0, s0 = 1, sp = 2;
  const int c = (ty + 1) * SX + tx + 1;
  // stage 2's point values, loaded for every thread (a thread without a point
  // reads cell (1, 1))
  T qu0 = T(0), qv0 = T(0), qw0 = T(0);
  auto load_point = [&](int kk) {
    const long a = active ? g.idx(i, j, kk) : g.idx(1, 1, kk);
    qu0 = du[a];
    qv0 = dv[a];
    qw0 = dw[a];
  };
  // the lower z-face terms of the thread's cell, carried up the column
  ZFace<T> zf{};
  if (active) {
    const PlaneAcc<T, SX> U{sh[0][sm], sh[0][s0], sh[0][sp], c};
    const PlaneAcc<T, SX> V{sh[1][sm], sh[1][s0], sh[1][sp], c};
    const PlaneAcc<T, SX> W{sh[2][sm], sh[2][s0], sh[2][sp], c};
    zf = zface_lower<T>(U, V, W, q0.m, k0);
  }
  __syncthreads();  // plane k0-1 is read above and rewritten in the loop
  T nu = T(0), nv = T(0), nw = T(0);  // plane k's new values until they are stored
  double msum = 0.0;                  // FP64 partial of the bulk mean (acc)
  auto compute = [&](int k) {
    if (!active) return;
    const PlaneAcc<T, SX> U{sh[0][sm], sh[0][s0], sh[0][sp], c};
    const PlaneAcc<T, SX> V{sh[1][sm], sh[1][s0], sh[1][sp], c};
    const PlaneAcc<T, SX> W{sh[2][sm], sh[2][s0], sh[2][sp], c};
    // reference arithmetic, src/mod_calcVel.cc:81,103,125 and :194,216,238
    T tu, tv, tw;
    tendency_z<T, CRF, true>(U, V, W, q0.m, k, q0.dxi, q0.dyi, q0.rei, q0.ucrf, tu, tv, tw, zf);
    nu = U(0, 0, 0) + q0.dt * tu;
    nv = V(0, 0, 0) + q0.dt * tv;
    nw = W(0, 0, 0) + q0.dt * tw;
    if (STAGE == 2) {
      nu = (nu + qu0) * T(0.5);
      nv = (nv + qv0) * T(0.5);
      nw = (nw + qw0) * T(0.5);
    }
    if (STAGE == 2 && acc) msum += nu * uniform_load(dzflzi, k);
  };
  auto store = [&](int k) {
    if (active) {
      const long a = g.idx(i, j, k);
      du[a] = nu;
      dv[a] = nv;
      dw[a] = nw;
    }
  };
  // the last plane, whose k+2 lies beyond the chunk's ring, runs after the loop
  for (int k = k0; k < k1; ++k) {
    if (STAGE == 2) load_point(k);
    fetch(k + 2);
    compute(k);
    commit(k + 2, sm);
    store(k);
    __syncthreads();
    const int t = sm;
    sm = s0;
    s0 = sp;
    sp = t;
  }
  if (STAGE == 2) load_point(k1);
  compute(k1);
  store(k1);
  if (STAGE == 2 && acc) {
    __syncthreads();
    static_assert(sizeof(sh) >= NT * sizeof(double), "reduction scratch");
    block_partial<NT>(&sh[0][0][0], msum, partial, b);
  }
}

// Tile rows of k_rk12: one block of them fills a CU either way.  FP64 12 (160
// VGPRs: three waves per SIMD; 16 rows spill), FP32 16.  Measured with two barriers
// a plane: FP64 8 and 10 rows 3021 and 2679 against 2348 us at 768x384x384, FP32
// 8 and 12 rows 1312 and 1440 against 1302.
template <typename T>
constexpr int kRk12Ty() {
  return std::is_same<T, double>::value ? 12 : 16;
}
constexpr int kRk12Slots = 256;  // blocks of k_rk12 that run at once: one per CU

// Both RK stages of a step inside a run (src/mod_calcVel.cc:61-125 then
// :174-238) in one pass.  The stored velocity is the previous step's
// predictor u*; its projection, forcing and boundary update are applied on
// load as in the separate stage 1 (fold and corr).  A block owns a 64 x TY
// tile of stage-2 points and marches a chunk of k planes.  Stage 1 runs on the
// tile plus a one-cell ring (each thread its tile point, the first threads one
// ring cell more) from an LDS ring of the loaded source (tile plus two
// cells); its result u1 goes to a second LDS ring and, except on the
// last step of a run (U1OUT), never to HBM.  The u1 values on the ring are
// stage 1 at the periodic position -- the x/y boundary update of u1 -- and the
// planes 0 and nz+1 of u1 and w1 on plane nz follow the boundary rules
// (src/mod_updateBound.cc:92,123,137).  Stage 2's point values are the loaded
// source at the tile point.  Per point u, v, w and p are read once and the new
// u, v, w written once; the result goes to separate arrays, since other blocks
// still read the source.  With `acc` the block sums the new u times dzflzi(k)
// in FP64 into partial[block].
//
// One barrier per plane: in iteration q a wave runs stage 1 on plane q, stage 2
// on plane q-2 (its neighbours' u1 of q-1 is behind the last barrier) and the
// commit of source plane q+2, so the waves of a block drift apart within it and
// one's LDS reads overlap another's arithmetic.  The carry holds what plane k-1
// would be read for, so each ring is two planes and the one being written.  The
// projection, forcing and boundary rules apply at a plane's commit, and stage 2's
// results are stored after the commit: arithmetic on the loaded values in the
// fetch, or stores ahead of the commit, would make a wave wait there.
//
// What bounds it is the chain of a plane at one block per CU (leaving stage 2 out
// saved 3 % in FP64 and nothing in FP32 when the loads were issued after stage 1):
// so a plane's loads are issued first, each thread loads a pair of cells (6 or 7
// wide loads instead of up to 14), and the waves that load are not those with ring
// cells.  At 768x384x384 FP64 2261 -> 2010-2040 us, with the viscous terms as second
// differences 2040-2120 (3.3 TB/s of 61 B a point), FP32 1243 -> 1070; 256x192x128 FP64 128 -> 115, 384x256x192 FP32 213 -> 186,
// 1536x768x512 FP32 6850 -> 6040.  Loads two planes ahead in a second set of
// registers ran slower (FP32 1178: the registers are full and all waves load).
// The two kernels that it replaces took 1646 + 2331 us (FP64, 768x384x384).
template <typename T, int TY, bool U1OUT, bool CRF>
__global__ __launch_bounds__(kRkTx* TY) void k_rk12(
    Geom g, const T* __restrict__ su, const T* __restrict__ sv, const T* __restrict__ sw,
    const T* __restrict__ pp, T* __restrict__ du, T* __restrict__ dv, T* __restrict__ dw,
    T* __restrict__ u1, T* __restrict__ v1, T* __restrict__ w1, RkParam<T> q0,
    const double* __restrict__ force, int kchunk, int ntx, int nty, int acc,
    const double* __restrict__ dzflzi, double* __restrict__ partial) {
  constexpr int TX = kRkTx, NT = TX * TY;
  constexpr int RX = TX + 2, RY = TY + 2, RPL = RX * RY;  // u1 region: tile + 1
  constexpr int UX = TX + 4, UY = TY + 4, UPL = UX * UY;  // source: tile + 2
  constexpr int NRING = RPL - NT;  // region cells outside the tile
  static_assert(NRING == 2 * RX + 2 * TY && NRING <= NT, "one ring cell per thread");
  // the source is loaded in pairs of x neighbours by waves that have no ring cells
  constexpr int F0 = (NRING + 63) / 64 * 64;
  static_assert(F0 + UPL / 2 <= NT && UX % 2 == 0, "one pair of source cells per thread");
  using V2 = T __attribute__((ext_vector_type(2)));
  typedef V2 V2u __attribute__((aligned(sizeof(T))));
  __shared__ __align__(16) T ssrc[3][3][UPL];  // [field][plane % 3][cell]; cell (cx, cy) = (i0-1+cx, j0-1+cy)
  __shared__ ZCarry<T> szb[NRING];  // the ring cells' carry: few threads have one
  __shared__ T su1[3][3][RPL];   // [field][plane % 3][cell]; cell (rx, ry) = (i0+rx, j0+ry)
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const int ti = (int)(b % (unsigned)ntx), tj = (int)((b / (unsigned)ntx) % (unsigned)nty);
  const int kc = (int)(b / (unsigned)(ntx * nty));
  const int i0 = ti * TX, j0 = tj * TY;
  const int k0 = kc * kchunk + 1, k1 = min(k0 + kchunk - 1, g.nz);
  const int t = threadIdx.x, tx = t % TX, ty = t / TX;
  const int i = i0 + tx + 1, j = j0 + ty + 1;
  const bool active = i <= g.nx && j <= g.ny;
  const T f_u = force ? (T)force[0] : T(0);
  if (k0 > k1) {
    if (acc && t == 0) partial[b] = 0.0;
    return;
  }
  auto wrap = [](int x, int n) { return ((x - 1) % n + n) % n + 1; };
  // plane-relative address of the pair's periodic image: its first cell's x is
  // odd and nx even, so no pair straddles the wrap
  const int e = 2 * (t - F0);
  const bool loads = t >= F0 && e < UPL;
  const int gaddr =
      loads ? wrap(i0 - 1 + e % UX, g.nx) + (int)g.sx * wrap(j0 - 1 + e / UX, g.ny) : 0;
  V2 ru{}, rv{}, rw{}, rp{}, rpn{}, rpt{};
  T rpe = T(0);
  auto fetch = [&](int kk) {
    const bool ghost = kk == 0 || kk == g.nz + 1;
    const long o = g.sxy * (ghost ? (kk == 0 ? 1 : g.nz) : kk);
    if (loads) {
      auto at = [&](const T* f, long d) { return *reinterpret_cast<const V2u*>(f + (o + d) + gaddr); };
      ru = at(su, 0);
      rv = at(sv, 0);
      rw = at(sw, 0);
      rp = at(pp, 0);
      rpe = pp[o + 2 + gaddr];
      rpn = at(pp, g.sx);
      rpt = at(pp, g.sxy);
    }
  };
  auto commit = [&](int kk, int slot) {
    const bool ghost = kk == 0 || kk == g.nz + 1;
    const int ks = ghost ? (kk == 0 ? 1 : g.nz) : kk;
    const bool wzero = kk == 0 || kk >= g.nz;
    const T dzci = uniform_load(q0.m.dzc_inv, ks);
    if (loads) {
      V2 su2, sv2, sw2;
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        const T p0 = rp[n], pe = n ? rpe : rp[1];
        T qu = ru[n] - (pe - p0) * q0.dtdxi;
        T qv = rv[n] - (rpn[n] - p0) * q0.dtdyi;
        // same association as k_correct: ((p(k+1) - p(k)) * dt) * dzc_inv(k)
        T qw = rw[n] - (rpt[n] - p0) * q0.dt * dzci;
        qu = qu + f_u;
        if (wzero) qw = T(0);
        if (ghost) {
          qu = T(2) * q0.bc_u - qu;  // src/mod_updateBound.cc:92,123
          qv = T(2) * T(0) - qv;
        }
        su2[n] = qu;
        sv2[n] = qv;
        sw2[n] = qw;
      }
      *reinterpret_cast<V2*>(&ssrc[0][slot][e]) = su2;
      *reinterpret_cast<V2*>(&ssrc[1][slot][e]) = sv2;
      *reinterpret_cast<V2*>(&ssrc[2][slot][e]) = sw2;
    }
  };
  // this thread's stage-1 cells: A = its own tile point, B = one ring cell (t < NRING)
  const int ra = (ty + 1) * RX + tx + 1;
  int bx, by;
  if (t < RX) {
    bx = t;
    by = 0;
  } else if (t < 2 * RX) {
    bx = t - RX;
    by = RY - 1;
  } else if (t < 2 * RX + TY) {
    bx = 0;
    by = t - 2 * RX + 1;
  } else {
    bx = RX - 1;
    by = t - 2 * RX - TY + 1;
  }
  const bool has_b = t < NRING;
  const int rb = by * RX + bx;
  const int ca = (ty + 2) * UX + tx + 2, cb = (by + 1) * UX + bx + 1;  // in the source ring
  const int qs = max(k0 - 1, 1), qe = k1 + 1;  // u1 planes formed: stage 1 up to nz, rules at nz+1
  // stencil accessors: centre plane in slot z, the plane above in slot p
  auto src = [&](int f, int z, int p, int c) {
    return PlaneAcc<T, UX>{ssrc[f][z], ssrc[f][z], ssrc[f][p], c};
  };
  auto reg = [&](int f, int z, int p) {
    return PlaneAcc<T, RX>{su1[f][z], su1[f][z], su1[f][p], ra};
  };
  // slots of planes q, q+1 and q+2 (= q-1) of either ring, at q = qs
  int s0 = 0, s1 = 1, s2 = 2;
  fetch(qs - 1);
  commit(qs - 1, s2);
  fetch(qs);
  commit(qs, s0);
  fetch(qs + 1);
  commit(qs + 1, s1);
  __syncthreads();
  ZCarry<T> za{}, z2{};
  {
    auto below = [&](int f, int c) { return PlaneAcc<T, UX>{ssrc[f][s2], ssrc[f][s0], ssrc[f][s0], c}; };
    za = carry_start<T>(below(0, ca), below(1, ca), below(2, ca), q0, qs);
    if (has_b) szb[t] = carry_start<T>(below(0, cb), below(1, cb), below(2, cb), q0, qs);
  }
  __syncthreads();  // plane qs-1's slot is rewritten by the first commit
  // u1 of plane q (slot s0) at region cell r; with q == 1 also plane 0 by the rules
  auto put1 = [&](int q, int r, T o1, T o2, T o3) {
    if (q == g.nz) o3 = T(0);
    su1[0][s0][r] = o1;
    su1[1][s0][r] = o2;
    su1[2][s0][r] = o3;
    if (q == 1) {
      su1[0][s2][r] = T(2) * q0.bc_u - o1;
      su1[1][s2][r] = T(2) * T(0) - o2;
      su1[2][s2][r] = T(0);
    }
  };
  // plane nz+1 of u1 by the rules from plane nz (the same thread wrote cell r of it)
  auto ghost_top = [&](int r) {
    su1[0][s0][r] = T(2) * q0.bc_u - su1[0][s2][r];
    su1[1][s0][r] = T(2) * T(0) - su1[1][s2][r];
    su1[2][s0][r] = T(0);
  };
  double msum = 0.0;
  T nextu = T(0), nextv = T(0), nextw = T(0);  // the source at the tile point of plane q-2
  for (int q = qs; q <= qe + 1; ++q) {
    const int k = q - 2;  // stage-2 plane
    // the next iteration's stage 1 reads source planes q+1, q+2
    const bool more = q < qe && q < g.nz;
    if (more) fetch(q + 2);
    const T pu = nextu, pv = nextv, pw = nextw;
    nextu = za.u;
    nextv = za.v;
    nextw = za.w;
    if (q <= qe && q <= g.nz) {
      T o1, o2, o3;
      stage_update<T, 1, CRF, UX>(src(0, s0, s1, ca), src(1, s0, s1, ca), src(2, s0, s1, ca), q0,
                                  q, T(0), T(0), T(0), za, o1, o2, o3);
      put1(q, ra, o1, o2, o3);
      if (U1OUT && active && q >= k0 && q <= k1) {
        const long a = g.idx(i, j, q);
        u1[a] = o1;
        v1[a] = o2;
        w1[a] = o3;
      }
      if (has_b) {
        ZCarry<T> zb = szb[t];
        stage_update<T, 1, CRF, UX>(src(0, s0, s1, cb), src(1, s0, s1, cb), src(2, s0, s1, cb), q0,
                                    q, T(0), T(0), T(0), zb, o1, o2, o3);
        szb[t] = zb;
        put1(q, rb, o1, o2, o3);
      }
    } else if (q == g.nz + 1) {
      ghost_top(ra);
      if (has_b) ghost_top(rb);
    }
    T nu = T(0), nv = T(0), nw = T(0);
    if (k >= k0 && active) {
      // u1 planes k = q-2 and q-1 are in the slots of q+1 and q+2
      stage_update<T, 2, CRF, RX>(reg(0, s1, s2), reg(1, s1, s2), reg(2, s1, s2), q0, k, pu, pv,
                                  pw, z2, nu, nv, nw);
      if (acc) msum += (double)nu * uniform_load(dzflzi, k);
    } else if (k == k0 - 1 && active) {
      auto below = [&](int f) { return PlaneAcc<T, RX>{su1[f][s1], su1[f][s2], su1[f][s2], ra}; };
      z2 = carry_start<T>(below(0), below(1), below(2), q0, k0);
    }
    if (more) commit(q + 2, s2);
    if (k >= k0 && active) {
      const long a = g.idx(i, j, k);
      du[a] = nu;
      dv[a] = nv;
      dw[a] = nw;
    }
    __syncthreads();
    const int r = s0;
    s0 = s1;
    s1 = s2;
    s2 = r;
  }
  static_assert(sizeof(ssrc) >= NT * sizeof(double), "reduction scratch");
  if (acc) block_partial<NT>(reinterpret_cast<double*>(&ssrc[0][0][0]), msum, partial, b);
}

// calcRHS, src/mod_calcRHS.cc:27-29.  w(k-1) is carried from the previous plane.
template <typename T>
__global__ __launch_bounds__(kRkTx* kRkTy) void k_calc_rhs(Geom g, const T* __restrict__ u,
                                                           const T* __restrict__ v,
                                                           const T* __restrict__ w,
                                                           T* __restrict__ p,
                                                           const T* __restrict__ dzf_inv, T dti,
                                                           T dtidxi, T dtidyi, int kchunk,
                                                           int ntx, int nty) {
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const int ti = (int)(b % (unsigned)ntx), tj = (int)((b / (unsigned)ntx) % (unsigned)nty);
  const int kc = (int)(b / (unsigned)(ntx * nty));
  const int i = ti * kRkTx + (int)(threadIdx.x % kRkTx) + 1;
  const int j = tj * kRkTy + (int)(threadIdx.x / kRkTx) + 1;
  if (i > g.nx || j > g.ny) return;
  const int k0 = kc * kchunk + 1, k1 = min(k0 + kchunk - 1, g.nz);
  long c = g.idx(i, j, k0);
  T wb = k0 <= k1 ? w[c - g.sxy] : T(0);
  for (int k = k0; k <= k1; ++k, c += g.sxy) {
    const T w0 = w[c];
    p[c] = (u[c] - u[c - 1]) * dtidxi + (v[c] - v[c - g.sx]) * dtidyi + (w0 - wb) * dti * dzf_inv[k];
    wb = w0;
  }
}

// correctVel, src/mod_calcVel.cc:272-274.  p(k+1) becomes the next plane's p(k).
// With fmask the force that is on the device is added to those components
// (forceVel, :299-315), which saves the end of a run its pass over u.  The
// boundary update stays a launch of its own: written by the cells that the halo
// copies, in this loop, it took the loads of the next planes out of flight (one
// 128^3 step 183 us, 1536x768x512 FP32 4 steps 74.3 ms; as it is 132 us, 69.9 ms).
template <typename T>
__global__ __launch_bounds__(kRkTx* correct_ty<T>()) void k_correct(
    Geom g, const T* __restrict__ p, T* __restrict__ u, T* __restrict__ v, T* __restrict__ w,
    RkParam<T> q, const double* __restrict__ force, int fmask, int kchunk, int ntx, int nty) {
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const int ti = (int)(b % (unsigned)ntx), tj = (int)((b / (unsigned)ntx) % (unsigned)nty);
  const int kc = (int)(b / (unsigned)(ntx * nty));
  constexpr int TY = correct_ty<T>();
  const int i = ti * kRkTx + (int)(threadIdx.x % kRkTx) + 1;
  const int j = tj * TY + (int)(threadIdx.x / kRkTx) + 1;
  const int k0 = kc * kchunk + 1, k1 = min(k0 + kchunk - 1, g.nz);
  if (i > g.nx || j > g.ny || k0 > k1) return;
  const bool fu = fmask & 1, fv = fmask & 2, fw = fmask & 4;
  const T f_u = fu ? (T)force[0] : T(0), f_v = fv ? (T)force[1] : T(0),
          f_w = fw ? (T)force[2] : T(0);
  long c = g.idx(i, j, k0);
  T p0 = p[c];
  for (int k = k0; k <= k1; ++k, c += g.sxy) {
    const T pt = p[c + g.sxy];
    T nu = u[c] - (p[c + 1] - p0) * q.dtdxi;
    T nv = v[c] - (p[c + g.sx] - p0) * q.dtdyi;
    T nw = w[c] - (pt - p0) * q.dt * uniform_load(q.m.dzc_inv, k);
    if (fu) nu = nu + f_u;
    if (fv) nv = nv + f_v;
    if (fw) nw = nw + f_w;
    u[c] = nu;
    v[c] = nv;
    w[c] = nw;
    p0 = pt;
  }
}

// ---------------------------------------------------------------------------
// Bulk mean (Mean, src/mod_utils.cc:30-51) in FP64: per-block partial sums of
// f*dzflzi(k) over a chunk of rows of one plane, then one block combines the
// partials in a fixed order, so the result is the same on every run.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double block_sum(double s, double* sh) {
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int h = blockDim.x / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) sh[threadIdx.x] += sh[threadIdx.x + h];
    __syncthreads();
  }
  return sh[0];
}

template <typename T>
__global__ __launch_bounds__(kRedThreads) void k_mean_partial(Geom g, const T* __restrict__ f,
                                                              const double* __restrict__ dzflzi,
                                                              double* __restrict__ partial,
                                                              int rows_per_chunk) {
  __shared__ double sh[kRedThreads];
  const int k = blockIdx.y + 1;
  const int j0 = blockIdx.x * rows_per_chunk;
  const int j1 = min(j0 + rows_per_chunk, g.ny);
  const double wk = dzflzi[k];
  double s = 0.0;
  for (int j = j0; j < j1; ++j) {
    const T* row = f + g.idx(1, j + 1, k);
    for (int i = threadIdx.x; i < g.nx; i += blockDim.x) s += (double)row[i] * wk;
  }
  s = block_sum(s, sh);
  if (threadIdx.x == 0) partial[(long)blockIdx.y * gridDim.x + blockIdx.x] = s;
}

// out[0] = sum(partial)/nxg/nyg; when force_slot >= 0 also stores
// out[force_slot] = vel_force - mean (forceVel, src/mod_calcVel.cc:297).
__global__ __launch_bounds__(kRedThreads) void k_mean_final(const double* __restrict__ partial,
                                                            long n, double nxg, double nyg,
                                                            double* out, double vel_force,
                                                            double* force_out) {
  __shared__ double sh[kRedThreads];
  double s = 0.0;
  for (long t = threadIdx.x; t < n; t += blockDim.x) s += partial[t];
  s = block_sum(s, sh);
  if (threadIdx.x == 0) {
    const double mean = s / nxg / nyg;
    out[0] = mean;
    if (force_out) force_out[0] = vel_force - mean;
  }
}

// forceVel update (src/mod_calcVel.cc:299-315): interior += force.
template <typename T>
__global__ __launch_bounds__(kTx* kTy) void k_add_force(Geom g, T* __restrict__ f,
                                                        const double* __restrict__ force,
                                                        int kchunk) {
  const int i = blockIdx.x * kTx + threadIdx.x + 1;
  const int j = blockIdx.y * kTy + threadIdx.y + 1;
  if (i > g.nx || j > g.ny) return;
  const T fv = (T)force[0];
  const int k0 = blockIdx.z * kchunk + 1;
  const int k1 = min(k0 + kchunk - 1, g.nz);
  for (int k = k0; k <= k1; ++k) {
    const long c = g.idx(i, j, k);
    f[c] += fv;
  }
}

// transform2CRF and other uniform shifts: interior += value.
template <typename T>
__global__ __launch_bounds__(kTx* kTy) void k_add_value(Geom g, T* __restrict__ f, T value,
                                                        int kchunk) {
  const int i = blockIdx.x * kTx + threadIdx.x + 1;
  const int j = blockIdx.y * kTy + threadIdx.y + 1;
  if (i > g.nx || j > g.ny) return;
  const int k0 = blockIdx.z * kchunk + 1;
  const int k1 = min(k0 + kchunk - 1, g.nz);
  for (int k = k0; k <= k1; ++k) f[g.idx(i, j, k)] += value;
}

// ---------------------------------------------------------------------------
// Boundary update at one GPU.  The reference's sequence -- y self-exchange,
// x periodic copies over the whole y/z extent, then the z walls over the whole
// x/y extent (src/mod_updateBound.cc:229-296) -- leaves every halo cell equal
// to a closed form of interior values:
//   side halo (i or j in {0, n+1}, 1 <= k <= nz): f(wrap i, wrap j, k)
//   z planes: centred u, v: 2*bc - f(wrap i, wrap j, 1|nz); face w: bc on
//   planes 0, nz and nz+1 (src/mod_updateBound.cc:75-144); p: zero gradient.
// Each halo cell is written once from interior cells, so one launch covers
// all of them with no ordering hazard.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int wrap(int i, int n) { return i == 0 ? n : (i == n + 1 ? 1 : i); }

// Perimeter cell q of an (nx+2)x(ny+2) plane -> (i, j).
__device__ __forceinline__ void perimeter(int q, int nx, int ny, int& i, int& j) {
  const int xl = nx + 2;
  if (q < xl) {
    i = q;
    j = 0;
  } else if (q < 2 * xl) {
    i = q - xl;
    j = ny + 1;
  } else {
    const int r = q - 2 * xl;  // rows 1..ny, two cells each
    j = r / 2 + 1;
    i = (r & 1) ? nx + 1 : 0;
  }
}

// blockIdx.y 0 updates u, v, w, 1 the second set u2, v2, w2.
template <typename T>
__global__ __launch_bounds__(256) void k_bc_vel(Geom g, T* __restrict__ u, T* __restrict__ v,
                                                T* __restrict__ w, T* __restrict__ u2,
                                                T* __restrict__ v2, T* __restrict__ w2, T bc_u,
                                                int walls_only) {
  if (blockIdx.y) {
    u = u2;
    v = v2;
    w = w2;
  }
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int nper = 2 * (g.nx + 2) + 2 * g.ny;
  const long nside = walls_only ? 0 : (long)nper * g.nz;
  const long nplane = (long)(g.nx + 2) * (g.ny + 2);
  const T zero = T(0), two = T(2);
  if (t < nside) {
    const int k = (int)(t / nper) + 1;
    int i, j;
    perimeter((int)(t % nper), g.nx, g.ny, i, j);
    const long d = g.idx(i, j, k);
    const long s = g.idx(wrap(i, g.nx), wrap(j, g.ny), k);
    u[d] = u[s];
    v[d] = v[s];
    w[d] = (k == g.nz) ? zero : w[s];
  } else if (t < nside + nplane) {
    const long q = t - nside;
    const int i = (int)(q % (g.nx + 2));
    const int j = (int)(q / (g.nx + 2));
    // after the exchange the wall rows read the periodic image; alone
    // (imposeBCVel) they read the halo cells as they stand
    const int wi = walls_only ? i : wrap(i, g.nx), wj = walls_only ? j : wrap(j, g.ny);
    u[g.idx(i, j, 0)] = two * bc_u - u[g.idx(wi, wj, 1)];
    u[g.idx(i, j, g.nz + 1)] = two * bc_u - u[g.idx(wi, wj, g.nz)];
    v[g.idx(i, j, 0)] = two * zero - v[g.idx(wi, wj, 1)];
    v[g.idx(i, j, g.nz + 1)] = two * zero - v[g.idx(wi, wj, g.nz)];
    w[g.idx(i, j, 0)] = zero;
    w[g.idx(i, j, g.nz)] = zero;
    w[g.idx(i, j, g.nz + 1)] = zero;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_bc_p(Geom g, T* __restrict__ p) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int nper = 2 * (g.nx + 2) + 2 * g.ny;
  const long nside = (long)nper * g.nz;
  const long nplane = (long)(g.nx + 2) * (g.ny + 2);
  if (t < nside) {
    const int k = (int)(t / nper) + 1;
    int i, j;
    perimeter((int)(t % nper), g.nx, g.ny, i, j);
    p[g.idx(i, j, k)] = p[g.idx(wrap(i, g.nx), wrap(j, g.ny), k)];
  } else if (t < nside + nplane) {
    const long q = t - nside;
    const int i = (int)(q % (g.nx + 2));
    const int j = (int)(q / (g.nx + 2));
    const int wi = wrap(i, g.nx), wj = wrap(j, g.ny);
    p[g.idx(i, j, 0)] = p[g.idx(wi, wj, 1)];
    p[g.idx(i, j, g.nz + 1)] = p[g.idx(wi, wj, g.nz)];
  }
}

// ---------------------------------------------------------------------------
// Initial condition (src/mod_initFlow.cc:47-102): u = profile(k) + noise,
// v = w = noise.  Noise: std::minstd_rand (a = 48271, m = 2^31-1) seeded with
// seed and advanced L+1 steps, L the interior linear index.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t mulmod31(uint64_t a, uint64_t b) {
  return (a * b) % 2147483647ULL;
}

__device__ double noise_uniform(uint32_t seed, uint64_t offset) {
  uint64_t x = seed % 2147483647ULL;
  if (x == 0) x = 1;
  uint64_t base = 48271ULL, e = offset + 1, r = 1;
  while (e) {
    if (e & 1) r = mulmod31(r, base);
    base = mulmod31(base, base);
    e >>= 1;
  }
  x = mulmod31(x, r);
  return (double)(x - 1) / 2147483646.0;
}

template <typename T>
__global__ __launch_bounds__(kTx* kTy) void k_init(Geom g, const double* __restrict__ prof,
                                                   T* __restrict__ u, T* __restrict__ v,
                                                   T* __restrict__ w, uint32_t s0, uint32_t s1,
                                                   uint32_t s2, int with_noise, double noise,
                                                   int kchunk) {
  const int i = blockIdx.x * kTx + threadIdx.x + 1;
  const int j = blockIdx.y * kTy + threadIdx.y + 1;
  if (i > g.nx || j > g.ny) return;
  const int k0 = blockIdx.z * kchunk + 1;
  const int k1 = min(k0 + kchunk - 1, g.nz);
  for (int k = k0; k <= k1; ++k) {
    const long c = g.idx(i, j, k);
    double uu = prof[k], vv = 0.0, ww = 0.0;
    if (with_noise) {
      const uint64_t L = ((uint64_t)(k - 1) * g.ny + (j - 1)) * g.nx + (i - 1);
      uu += 2.0 * (noise_uniform(s0, L) - 0.5) * noise;
      vv += 2.0 * (noise_uniform(s1, L) - 0.5) * noise;
      ww += 2.0 * (noise_uniform(s2, L) - 0.5) * noise;
    }
    u[c] = (T)uu;
    v[c] = (T)vv;
    w[c] = (T)ww;
  }
}

// u *= 1/(mean*u_ref) when mean != 0 (src/mod_initFlow.cc:91-100).
template <typename T>
__global__ __launch_bounds__(kTx* kTy) void k_scale_inv_mean(Geom g, T* __restrict__ f,
                                                             const double* __restrict__ mean,
                                                             double u_ref, int kchunk) {
  const int i = blockIdx.x * kTx + threadIdx.x + 1;
  const int j = blockIdx.y * kTy + threadIdx.y + 1;
  if (i > g.nx || j > g.ny) return;
  const double m = mean[0];
  if (m == 0.0) return;
  const double mult = 1.0 / (m * u_ref);
  const int k0 = blockIdx.z * kchunk + 1;
  const int k1 = min(k0 + kchunk - 1, g.nz);
  for (int k = k0; k <= k1; ++k) {
    const long c = g.idx(i, j, k);
    f[c] = (T)((double)f[c] * mult);
  }
}

// ---------------------------------------------------------------------------
// Runtime checks (src/mod_utils.cc:77-217).  Max with location: a candidate
// replaces the running best only when strictly larger (NaN never does), and
// ties between threads go to the smaller linear index, which reproduces the
// reference's k-j-i loop's first maximum.
// ---------------------------------------------------------------------------
struct ValIdx {
  double v;
  long l;
};

__device__ __forceinline__ bool better(double va, long la, double vb, long lb) {
  return va > vb || (va == vb && la < lb);
}

template <typename T, int KIND>
__global__ __launch_bounds__(kRedThreads) void k_max_partial(Geom g, const T* __restrict__ u,
                                                             const T* __restrict__ v,
                                                             const T* __restrict__ w,
                                                             const T* __restrict__ dzf_inv,
                                                             T dxi, T dyi, ValIdx* out) {
  __shared__ double sv[kRedThreads];
  __shared__ long sl[kRedThreads];
  const long n = (long)g.nx * g.ny * g.nz;
  double best = 0.0;
  long bl = 0;
  for (long L = (long)blockIdx.x * blockDim.x + threadIdx.x; L < n;
       L += (long)gridDim.x * blockDim.x) {
    const int i = (int)(L % g.nx) + 1;
    const int j = (int)((L / g.nx) % g.ny) + 1;
    const int k = (int)(L / ((long)g.nx * g.ny)) + 1;
    const long c = g.idx(i, j, k);
    T val;
    if (KIND == 0) {  // divergence, src/mod_utils.cc:177-179
      val = fabs((u[c] - u[c - 1]) * dxi + (v[c] - v[c - g.sx]) * dyi +
                 (w[c] - w[c - g.sxy]) * dzf_inv[k]);
    } else {  // CFL, src/mod_utils.cc:121-123
      val = fabs((u[c] + u[c - 1]) * T(0.5)) * dxi + fabs((v[c] + v[c - g.sx]) * T(0.5)) * dyi +
            fabs((w[c] + w[c - g.sxy]) * T(0.5)) * dzf_inv[k];
    }
    const double dv = (double)val;
    if (dv > best) {
      best = dv;
      bl = L;
    }
  }
  sv[threadIdx.x] = best;
  sl[threadIdx.x] = bl;
  __syncthreads();
  for (int h = blockDim.x / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h &&
        better(sv[threadIdx.x + h], sl[threadIdx.x + h], sv[threadIdx.x], sl[threadIdx.x])) {
      sv[threadIdx.x] = sv[threadIdx.x + h];
      sl[threadIdx.x] = sl[threadIdx.x + h];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = ValIdx{sv[0], sl[0]};
}

__global__ __launch_bounds__(kRedThreads) void k_max_final(const ValIdx* __restrict__ in, int n,
                                                           ValIdx* out) {
  __shared__ double sv[kRedThreads];
  __shared__ long sl[kRedThreads];
  double best = 0.0;
  long bl = 0;
  for (int t = threadIdx.x; t < n; t += blockDim.x)
    if (better(in[t].v, in[t].l, best, bl)) {
      best = in[t].v;
      bl = in[t].l;
    }
  sv[threadIdx.x] = best;
  sl[threadIdx.x] = bl;
  __syncthreads();
  for (int h = blockDim.x / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h &&
        better(sv[threadIdx.x + h], sl[threadIdx.x + h], sv[threadIdx.x], sl[threadIdx.x])) {
      sv[threadIdx.x] = sv[threadIdx.x + h];
      sl[threadIdx.x] = sl[threadIdx.x + h];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = ValIdx{sv[0], sl[0]};
}

// NaN count over the whole halo-padded array.
template <typename T>
__global__ __launch_bounds__(kRedThreads) void k_nan_partial(const T* __restrict__ f, long n,
                                                             double* out) {
  __shared__ double sh[kRedThreads];
  double cnt = 0.0;
  for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n;
       t += (long)gridDim.x * blockDim.x)
    if (isnan(f[t])) cnt += 1.0;
  cnt = block_sum(cnt, sh);
  if (threadIdx.x == 0) out[blockIdx.x] = cnt;
}

// ---------------------------------------------------------------------------
// host-side helpers
// ---------------------------------------------------------------------------
inline int kchunk_for(const pll_context* c) {
  // enough blocks to fill 256 CUs several times over, k-chunks of >= 4 planes
  const long cols = (long)((c->g.nx + kTx - 1) / kTx) * ((c->g.ny + kTy - 1) / kTy);
  long want = 4096 / (cols > 0 ? cols : 1);
  if (want < 1) want = 1;
  long kc = (c->g.nz + want - 1) / want;
  if (kc < 4) kc = 4;
  if (kc > c->g.nz) kc = c->g.nz;
  return (int)kc;
}

inline dim3 col_grid(const pll_context* c, int kc) {
  return dim3((c->g.nx + kTx - 1) / kTx, (c->g.ny + kTy - 1) / kTy, (c->g.nz + kc - 1) / kc);
}

template <typename T>
inline MeshT<T> mesh_of(const pll_context* c) {
  const T* base = static_cast<const T*>(c->d_mesh);
  const long n = c->g.nz + 2;
  return MeshT<T>{base, base + n, base + 2 * n, base + 3 * n};
}

template <typename T>
inline T* F(pll_context* c, int f) {
  return static_cast<T*>(c->fld[f]);
}

// Tiled launch shape of the stencil kernels: ntx*nty tiles of 64 x ty columns,
// each marching a chunk of k planes; about 2048 blocks in total.
struct TileGrid {
  int ntx, nty, nkc, kchunk;
  unsigned blocks() const { return (unsigned)ntx * nty * nkc; }
};

inline TileGrid tile_grid(const pll_context* c, int ty = kRkTy) {
  TileGrid t;
  t.ntx = (c->g.nx + kRkTx - 1) / kRkTx;
  t.nty = (c->g.ny + ty - 1) / ty;
  const long cols = (long)t.ntx * t.nty;
  long want = (2048 + cols - 1) / cols;
  int kc = (int)((c->g.nz + want - 1) / want);
  if (kc < 4) kc = 4;
  if (kc > c->g.nz) kc = c->g.nz;
  t.kchunk = kc;
  t.nkc = (c->g.nz + kc - 1) / kc;
  return t;
}

inline int forced_mask(const pll_context* c) {
  return (c->is_forced[0] ? 1 : 0) | (c->is_forced[1] ? 2 : 0) | (c->is_forced[2] ? 4 : 0);
}

// Coefficients of tendency_fast (S = dt), computed in FP64 and rounded once.
template <typename T>
RkUniform<T> rk_uniform(const pll_context* c) {
  const double S = c->dt;
  return RkUniform<T>{(T)(S * 0.25 * c->dx_inv), (T)(S * 0.25 * c->dy_inv),
                      (T)(S * c->re_inv * c->dx_inv * c->dx_inv),
                      (T)(S * c->re_inv * c->dy_inv * c->dy_inv),
                      (T)(S * 0.5 * c->u_crf * c->dx_inv)};
}

template <typename T>
int rk_coef_setup(pll_context* c) {
  const int nz = c->g.nz;
  std::vector<RkCoef<T>> h((size_t)(nz + 2));
  const double S = c->dt, rei = c->re_inv;
  for (int k = 1; k <= nz; ++k) {
    const double* f = c->dzf.data();
    const double* fi = c->dzf_inv.data();
    const double* ci = c->dzc_inv.data();
    RkCoef<T>& q = h[k];
    q.a1 = (T)(f[k + 1] * ci[k]);
    q.a2 = (T)(f[k] * ci[k]);
    q.b1 = (T)(f[k - 1] * ci[k - 1]);
    q.b2 = (T)(f[k] * ci[k - 1]);
    q.zuv = (T)(S * 0.25 * fi[k]);
    q.cp = (T)(S * rei * ci[k] * fi[k]);
    q.cm = (T)(S * rei * ci[k - 1] * fi[k]);
    q.zw = (T)(S * 0.25 * ci[k]);
    q.dp = (T)(S * rei * fi[k + 1] * ci[k]);
    q.dm = (T)(S * rei * fi[k] * ci[k]);
    // the diagonal from the rounded coefficients (one rounding off their sum)
    const RkUniform<T> cu = rk_uniform<T>(c);
    const double vxy = 2.0 * (double)cu.vx + 2.0 * (double)cu.vy;
    q.cdu = (T)(vxy + (double)q.cp + (double)q.cm);
    q.cdw = (T)(vxy + (double)q.dp + (double)q.dm);
  }
  PLL_HIP_TRY(ctx_malloc(c, &c->d_rkcoef, h.size() * sizeof(RkCoef<T>)));
  PLL_HIP_TRY(hipMemcpy(c->d_rkcoef, h.data(), h.size() * sizeof(RkCoef<T>), hipMemcpyHostToDevice));
  return PLL_OK;
}

template <typename T>
RkParam<T> rk_param(const pll_context* c) {
  return RkParam<T>{mesh_of<T>(c), (T)c->dx_inv, (T)c->dy_inv, (T)c->re_inv, (T)c->dt, (T)c->u_crf,
                    (T)(c->dt * c->dx_inv), (T)(c->dt * c->dy_inv),  // src/mod_calcVel.cc:256-258
                    (T)(0.0 - c->u_crf),                             // src/mod_updateBound.cc:80
                    static_cast<const RkCoef<T>*>(c->d_rkcoef), rk_uniform<T>(c)};
}

template <typename T>
int rk_t(pll_context* c, int stage, int acc, int bcload) {
  constexpr bool kF64 = std::is_same<T, double>::value;
  const int ty = kF64 ? kLateTy : kRkTy;
  const TileGrid t = tile_grid(c, ty);
  if (acc && (long)t.blocks() > c->npartial)
    return fail(PLL_ERR_STATE, "reduction scratch smaller than the stencil grid");
  const double* dzflzi = c->d_mesh64 + 3 * (c->g.nz + 2);
  {
    TimerScope ts(c, stage == 1 ? K_RK1 : K_RK2);
    auto go = [&](auto kernel, int src, int dst) {
      hipLaunchKernelGGL(kernel, dim3(t.blocks()), dim3(kRkTx * ty), 0, c->stream, c->g,
                         F<T>(c, src), F<T>(c, src + 1), F<T>(c, src + 2), F<T>(c, dst),
                         F<T>(c, dst + 1), F<T>(c, dst + 2), rk_param<T>(c), t.kchunk, t.ntx,
                         t.nty, acc, dzflzi, c->d_partial, bcload);
    };
    // FP64 runs the late-commit form of the stages (k_rk_late), FP32 k_rk
    const bool crf = c->u_crf != 0.0;
    if constexpr (kF64)
      stage == 1 ? go(crf ? k_rk_late<1, true> : k_rk_late<1, false>, PLL_U, PLL_U1)
                 : go(crf ? k_rk_late<2, true> : k_rk_late<2, false>, PLL_U1, PLL_U);
    else
      stage == 1 ? go(crf ? k_rk<T, 1, true> : k_rk<T, 1, false>, PLL_U, PLL_U1)
                 : go(crf ? k_rk<T, 2, true> : k_rk<T, 2, false>, PLL_U1, PLL_U);
  }
  PLL_HIP_TRY(hipGetLastError());
  return acc ? force_from_partials(c, (long)t.blocks()) : PLL_OK;
}

// Launch shape of the fused stages: `slots` blocks run at once, and a block
// costs its chunk's planes and about three more (two of stage 1 alone and the
// ring's start), so the chunk is the one with the least rounds x (chunk + 3);
// of equal costs the shortest, whose last round is spread the most.  Against
// chunks for about 1024 blocks: 230 against 255 us at 384x256x192 (FP32), 30
// against 39 us at 160x96x96; against chunks of four planes and more 22 against 27
// us at 64x64x64, 17 against 26 at 24x20x12.
TileGrid rk12_grid(const pll_context* c, int ty, int slots) {
  TileGrid t;
  t.ntx = (c->g.nx + kRkTx - 1) / kRkTx;
  t.nty = (c->g.ny + ty - 1) / ty;
  const long cols = (long)t.ntx * t.nty;
  long best = 0;
  for (int kc = 1; kc <= c->g.nz; ++kc) {
    const long nkc = (c->g.nz + kc - 1) / kc;
    const long cost = ((cols * nkc + slots - 1) / slots) * (kc + 3);
    if (best && cost >= best) continue;
    best = cost;
    t.kchunk = kc;
    t.nkc = (int)nkc;
  }
  return t;
}

// Both stages of a step inside a run (the previous step's projection, forcing
// and boundary update applied on load) into the spare velocity buffers, then
// swapped in; u1out: u1 goes to its arrays as well; acc: the bulk mean of the
// new u and the force of u go to d_scalar[0], [3].
template <typename T>
int rk12_t(pll_context* c, int acc, int u1out) {
  constexpr int ty = kRk12Ty<T>();
  const TileGrid t = rk12_grid(c, ty, kRk12Slots);
  if (acc && (long)t.blocks() > c->npartial)
    return fail(PLL_ERR_STATE, "reduction scratch smaller than the stencil grid");
  if (!c->fld_alt[0] || !c->fld_alt[1] || !c->fld_alt[2])
    return fail(PLL_ERR_STATE, "no spare velocity buffers");
  {
    TimerScope ts(c, K_RK12);
    const auto kernel =
        c->u_crf != 0.0 ? (u1out ? k_rk12<T, ty, true, true> : k_rk12<T, ty, false, true>)
                        : (u1out ? k_rk12<T, ty, true, false> : k_rk12<T, ty, false, false>);
    hipLaunchKernelGGL(kernel, dim3(t.blocks()), dim3(kRkTx * ty), 0, c->stream, c->g, F<T>(c, PLL_U), F<T>(c, PLL_V),
                       F<T>(c, PLL_W), F<T>(c, PLL_P), static_cast<T*>(c->fld_alt[0]),
                       static_cast<T*>(c->fld_alt[1]), static_cast<T*>(c->fld_alt[2]),
                       F<T>(c, PLL_U1), F<T>(c, PLL_V1), F<T>(c, PLL_W1), rk_param<T>(c),
                       c->is_forced[0] ? c->d_scalar + 3 : nullptr, t.kchunk, t.ntx, t.nty, acc,
                       c->d_mesh64 + 3 * (c->g.nz + 2), c->d_partial);
  }
  PLL_HIP_TRY(hipGetLastError());
  for (int d = 0; d < 3; ++d) std::swap(c->fld[PLL_U + d], c->fld_alt[d]);
  return acc ? force_from_partials(c, (long)t.blocks()) : PLL_OK;
}

template <typename T>
int rhs_t(pll_context* c) {
  const TileGrid t = tile_grid(c);
  const double dti = 1.0 / c->dt;  // src/mod_calcRHS.cc:11-13
  const double dtidxi = dti * c->dx_inv;
  const double dtidyi = dti * c->dy_inv;
  TimerScope ts(c, K_RHS);
  hipLaunchKernelGGL((k_calc_rhs<T>), dim3(t.blocks()), dim3(kRkTx * kRkTy), 0, c->stream, c->g,
                     F<T>(c, PLL_U), F<T>(c, PLL_V), F<T>(c, PLL_W), F<T>(c, PLL_P),
                     mesh_of<T>(c).dzf_inv, (T)dti, (T)dtidxi, (T)dtidyi, t.kchunk, t.ntx, t.nty);
  PLL_HIP_TRY(hipGetLastError());
  return PLL_OK;
}

template <typename T>
int correct_t(pll_context* c, bool with_force) {
  constexpr int ty = correct_ty<T>();
  const TileGrid t = tile_grid(c, ty);
  TimerScope ts(c, K_CORRECT);
  hipLaunchKernelGGL((k_correct<T>), dim3(t.blocks()), dim3(kRkTx * ty), 0, c->stream, c->g,
                     F<T>(c, PLL_P), F<T>(c, PLL_U), F<T>(c, PLL_V), F<T>(c, PLL_W),
                     rk_param<T>(c), c->d_scalar + 3, with_force ? forced_mask(c) : 0, t.kchunk,
                     t.ntx, t.nty);
  PLL_HIP_TRY(hipGetLastError());
  return PLL_OK;
}

template <typename T>
int mean_t(pll_context* c, int field, double nxg, double nyg, double* d_out, double vel_force,
           double* d_force) {
  const int chunks = c->mean_chunks;
  const int rpc = (c->g.ny + chunks - 1) / chunks;
  if (chunks < 1 || (long)chunks * c->g.nz > c->npartial || !c->d_partial || !F<T>(c, field) || !d_out)
    return fail(PLL_ERR_STATE, "bulk-mean reduction scratch does not fit the grid");
  {
    TimerScope ts(c, K_MEAN_PARTIAL);
    hipLaunchKernelGGL((k_mean_partial<T>), dim3(chunks, c->g.nz), dim3(kRedThreads), 0,
                       c->stream, c->g, F<T>(c, field), c->d_mesh64 + 3 * (c->g.nz + 2),
                       c->d_partial, rpc);
  }
  {
    TimerScope ts(c, K_MEAN_FINAL);
    hipLaunchKernelGGL(k_mean_final, dim3(1), dim3(kRedThreads), 0, c->stream, c->d_partial,
                       (long)chunks * c->g.nz, nxg, nyg, d_out, vel_force, d_force);
  }
  PLL_HIP_TRY(hipGetLastError());
  return PLL_OK;
}

template <typename T>
int force_t(pll_context* c) {
  const int kc = kchunk_for(c);
  for (int d = 0; d < 3; ++d) {
    if (!c->is_forced[d]) continue;
    int rc = mean_t<T>(c, PLL_U + d, (double)c->g.nx, (double)c->g.ny, c->d_scalar + d,
                       c->vel_force[d], c->d_scalar + 3 + d);
    if (rc) return rc;
  }
  for (int d = 0; d < 3; ++d) {
    if (!c->is_forced[d]) continue;
    TimerScope ts(c, K_FORCE);
    hipLaunchKernelGGL((k_add_force<T>), col_grid(c, kc), dim3(kTx, kTy), 0, c->stream, c->g,
                       F<T>(c, PLL_U + d), c->d_scalar + 3 + d, kc);
  }
  PLL_HIP_TRY(hipGetLastError());
  return PLL_OK;
}

inline long bc_threads(const pll_context* c) {
  const long nper = 2L * (c->g.nx + 2) + 2L * c->g.ny;
  return nper * c->g.nz + (long)(c->g.nx + 2) * (c->g.ny + 2);
}

// which: 0 (u, v, w), 1 (u1, v1, w1), 2 both
template <typename T>
int bc_vel_t(pll_context* c, int which, int walls_only) {
  const long n = walls_only ? (long)(c->g.nx + 2) * (c->g.ny + 2) : bc_threads(c);
  const int a = which == 1 ? PLL_U1 : PLL_U, b = which == 0 ? PLL_U : PLL_U1;
  const double bc_u = 0.0 - c->u_crf;  // src/mod_updateBound.cc:80
  TimerScope ts(c, K_BC_VEL);
  hipLaunchKernelGGL((k_bc_vel<T>), dim3((unsigned)((n + 255) / 256), which == 2 ? 2 : 1),
                     dim3(256), 0, c->stream, c->g, F<T>(c, a), F<T>(c, a + 1), F<T>(c, a + 2),
                     F<T>(c, b), F<T>(c, b + 1), F<T>(c, b + 2), (T)bc_u, walls_only);
  PLL_HIP_TRY(hipGetLastError());
  return PLL_OK;
}

template <typename T>
int bc_p_t(pll_context* c) {
  const long n = bc_threads(c);
  TimerScope ts(c, K_BC_P);
  hipLaunchKernelGGL((k_bc_p<T>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream,
                     c->g, F<T>(c, PLL_P));
  PLL_HIP_TRY(hipGetLastError());
  return PLL_OK;
}

template <typename T>
int add_scalar_t(pll_context* c, int field, double value) {
  const int kc = kchunk_for(c);
  TimerScope ts(c, K_MISC);
  hipLaunchKernelGGL((k_add_value<T>), col_grid(c, kc), dim3(kTx, kTy), 0, c->stream, c->g,
                     F<T>(c, field), (T)value, kc);
  PLL_HIP_TRY(hipGetLastError());
  return PLL_OK;
}

template <typename T>
int init_t(pll_context* c, const double* d_prof, int with_noise, double noise,
           const uint32_t seeds[3]) {
  const int kc = kchunk_for(c);
  TimerScope ts(c, K_INIT);
  hipLaunchKernelGGL((k_init<T>), col_grid(c, kc), dim3(kTx, kTy), 0, c->stream, c->g, d_prof,
                     F<T>(c, PLL_U), F<T>(c, PLL_V), F<T>(c, PLL_W), seeds[0], seeds[1],
                     seeds[2], with_noise, noise, kc);
  PLL_HIP_TRY(hipGetLastError());
  return PLL_OK;
}

template <typename T>
int scale_inv_mean_t(pll_context* c, int field, const double* d_mean, double u_ref) {
  const int kc = kchunk_for(c);
  TimerScope ts(c, K_INIT);
  hipLaunchKernelGGL((k_scale_inv_mean<T>), col_grid(c, kc), dim3(kTx, kTy), 0, c->stream, c->g,
                     F<T>(c, field), d_mean, u_ref, kc);
  PLL_HIP_TRY(hipGetLastError());
  return PLL_OK;
}

template <typename T, int KIND>
int max_t(pll_context* c, pll_value_index* out) {
  ValIdx* red = static_cast<ValIdx*>(c->d_red);
  {
    TimerScope ts(c, K_CHECK);
    hipLaunchKernelGGL((k_max_partial<T, KIND>), dim3(kRedBlocks), dim3(kRedThreads), 0,
                       c->stream, c->g, F<T>(c, PLL_U), F<T>(c, PLL_V), F<T>(c, PLL_W),
                       mesh_of<T>(c).dzf_inv, (T)c->dx_inv, (T)c->dy_inv, red);
    hipLaunchKernelGGL(k_max_final, dim3(1), dim3(kRedThreads), 0, c->stream, red, kRedBlocks,
                       red + kRedBlocks);
  }
  PLL_HIP_TRY(hipGetLastError());
  ValIdx h;
  PLL_HIP_TRY(hipMemcpyAsync(&h, red + kRedBlocks, sizeof(ValIdx), hipMemcpyDeviceToHost,
                             c->stream));
  PLL_HIP_TRY(hipStreamSynchronize(c->stream));
  const long nxy = (long)c->g.nx * c->g.ny;
  out->value = (KIND == 1) ? h.v * (double)(T)c->dt : h.v;
  out->rank = 0;
  out->ig = (int)(h.l % c->g.nx) + 1;
  out->jg = (int)((h.l / c->g.nx) % c->g.ny) + 1;
  out->kg = (int)(h.l / nxy) + 1;
  return PLL_OK;
}

template <typename T>
int nan_t(pll_context* c, int field, int* passed) {
  double* red = static_cast<double*>(c->d_red);
  {
    TimerScope ts(c, K_CHECK);
    hipLaunchKernelGGL((k_nan_partial<T>), dim3(kRedBlocks), dim3(kRedThreads), 0, c->stream,
                       F<T>(c, field), c->nfield, red);
    hipLaunchKernelGGL(k_mean_final, dim3(1), dim3(kRedThreads), 0, c->stream, red,
                       (long)kRedBlocks, 1.0, 1.0, red + kRedBlocks, 0.0, (double*)nullptr);
  }
  PLL_HIP_TRY(hipGetLastError());
  double cnt = 0.0;
  PLL_HIP_TRY(hipMemcpyAsync(&cnt, red + kRedBlocks, sizeof(double), hipMemcpyDeviceToHost,
                             c->stream));
  PLL_HIP_TRY(hipStreamSynchronize(c->stream));
  *passed = (cnt == 0.0) ? 1 : 0;
  return PLL_OK;
}

}  // namespace

// ---- dispatch on the context precision ------------------------------------------
#define PLL_DISPATCH(c, call_fp64, call_fp32) \
  ((c)->prec == PLL_FP64 ? (call_fp64) : (call_fp32))

int rk_setup(pll_context* c) {
  return PLL_DISPATCH(c, rk_coef_setup<double>(c), rk_coef_setup<float>(c));
}

int launch_rk(pll_context* c, int stage, int acc, int bcload) {
  if (c->closure) return launch_rk_closure(c, stage, 0, acc, 0);
  return PLL_DISPATCH(c, rk_t<double>(c, stage, acc, bcload), rk_t<float>(c, stage, acc, bcload));
}
int launch_calc_rhs(pll_context* c) { return PLL_DISPATCH(c, rhs_t<double>(c), rhs_t<float>(c)); }
int force_from_partials(pll_context* c, long n) {
  if (n < 1 || n > c->npartial || !c->d_partial)
    return fail(PLL_ERR_STATE, "bulk-mean partials do not fit the scratch");
  c->mean_pending = n;
  return PLL_OK;
}
int launch_rk12(pll_context* c, int acc, int u1out) {
  return PLL_DISPATCH(c, rk12_t<double>(c, acc, u1out), rk12_t<float>(c, acc, u1out));
}
int launch_correct_vel(pll_context* c, bool with_force) {
  return PLL_DISPATCH(c, correct_t<double>(c, with_force), correct_t<float>(c, with_force));
}
int launch_mean(pll_context* c, int field, double nxg, double nyg, double* d_out) {
  return PLL_DISPATCH(c, mean_t<double>(c, field, nxg, nyg, d_out, 0.0, nullptr),
                      mean_t<float>(c, field, nxg, nyg, d_out, 0.0, nullptr));
}
int launch_force(pll_context* c) { return PLL_DISPATCH(c, force_t<double>(c), force_t<float>(c)); }
int launch_bc_vel(pll_context* c, int which, int walls_only) {
  return PLL_DISPATCH(c, bc_vel_t<double>(c, which, walls_only),
                      bc_vel_t<float>(c, which, walls_only));
}
int launch_bc_p(pll_context* c) { return PLL_DISPATCH(c, bc_p_t<double>(c), bc_p_t<float>(c)); }
int launch_add_scalar(pll_context* c, int field, double value) {
  return PLL_DISPATCH(c, add_scalar_t<double>(c, field, value),
                      add_scalar_t<float>(c, field, value));
}
int launch_init_flow(pll_context* c, const double* d_prof, int with_noise, double noise,
                     const uint32_t seeds[3]) {
  return PLL_DISPATCH(c, init_t<double>(c, d_prof, with_noise, noise, seeds),
                      init_t<float>(c, d_prof, with_noise, noise, seeds));
}
int launch_scale_by_inverse_mean(pll_context* c, int field, const double* d_mean, double u_ref) {
  return PLL_DISPATCH(c, scale_inv_mean_t<double>(c, field, d_mean, u_ref),
                      scale_inv_mean_t<float>(c, field, d_mean, u_ref));
}
int launch_max_div(pll_context* c, pll_value_index* out) {
  return PLL_DISPATCH(c, (max_t<double, 0>(c, out)), (max_t<float, 0>(c, out)));
}
int launch_max_cfl(pll_context* c, pll_value_index* out) {
  return PLL_DISPATCH(c, (max_t<double, 1>(c, out)), (max_t<float, 1>(c, out)));
}
int launch_check_nan(pll_context* c, int field, int* passed) {
  return PLL_DISPATCH(c, nan_t<double>(c, field, passed), nan_t<float>(c, field, passed));
}

}  // namespace pll
