// fft_fixed.hpp -- the transforms of compiled-in length (k_fft_fixed.hip) and what
// they share with those of a run-time plan (k_fft.hip, which describes both).
#pragma once

#include "fft_radix.hpp"
#include "pll_internal.hpp"

namespace pll {
namespace {

// ============================================================================
// Compile-time transforms: every product of 2, 3 and 5 up to kFixedMax but 625,
// which no three of the radices make (it runs from a run-time plan).  One
// padded LDS buffer per block; each pass reads its butterfly inputs into
// registers, synchronises, and writes the outputs back in place, so every
// thread does at most one radix-R butterfly per pass.  The first pass of the
// forward transforms and of the inverse x transform takes its inputs from the
// registers that they were loaded to (the smallest radix comes first, so every
// thread has a butterfly), the last pass of the inverse ones stores to HBM.
// Index arithmetic is constant-folded and radices up to 16 keep the pass count at
// 2-3.  Against run-time plans a step takes 151 instead of 172 us at 200x90x176,
// 136 instead of 156 at 128x128x128, 400 instead of 451 at 300x216x128 (FP64), 599
// instead of 684 at 640x300x128 (FP32).
// ============================================================================
constexpr int kFixedMax = 768;
struct Radices {
  int np = 0, r[3] = {0, 0, 0}, lo = 0, hi = 0;
};
// Fewest passes, then the largest smallest radix (fewest threads per sequence),
// then the smallest largest one (fewest registers); smallest first, the middle
// one last.  np = 0: no plan of three passes.  The rms error of a transform is that
// of radix 4, 2, 3 and 5 passes to -4 ... +20 % (FP64, 33 lengths, on average
// +3 %, the most at 216 = 6 6 6; FP32 +-5 %): fewer passes, and fewer of their
// twiddles are 1.
constexpr Radices radices(int L) {
  constexpr int R[] = {2, 3, 4, 5, 6, 8, 9, 10, 12, 15, 16};
  Radices best;
  for (int a : R)
    if (L == a) return Radices{1, {a, 0, 0}, a, a};
  for (int a : R)
    for (int b : R)
      if (a <= b && a * b == L && a > best.lo) best = Radices{2, {a, b, 0}, a, b};
  if (best.np) return best;
  for (int a : R)
    for (int b : R)
      for (int c : R)
        if (a <= b && b <= c && a * b * c == L &&
            (a > best.lo || (a == best.lo && c < best.hi)))
          best = Radices{3, {a, c, b}, a, c};
  return best;
}
constexpr bool fixed_length(int L) { return L >= 2 && L <= kFixedMax && radices(L).np > 0; }

template <int L>
struct Shape {
  static constexpr Radices plan = radices(L);
  static constexpr int np = plan.np;
};

template <class SH, int P>
constexpr int shape_span() {
  int s = 1;
  for (int p = 0; p < P; ++p) s *= SH::plan.r[p];
  return s;
}
// threads per sequence: every thread owns one butterfly of the smallest radix
template <int L>
constexpr int tps() {
  return L / Shape<L>::plan.lo;
}
// one pad slot per 16 complex values spreads strided accesses over the banks
__device__ __forceinline__ int pad(int x) { return x + (x >> 4); }
constexpr int padded(int n) { return n + (n >> 4) + 1; }
constexpr int kLdsMax = 64 * 1024;

// Rows per block of the x transforms: the fewest that fill one wave, or several
// (up to 256 threads), to nine tenths.  One wave a block needs no barrier and
// leaves small grids the most blocks; with one row of 96 threads a block (L = 768)
// the FP32 transforms ran 2549 + 1413 us at 1536x768x512, with two 2304 + 1261.
template <int L>
constexpr int x_rows() {
  constexpr int T = tps<L>();
  int best = 1, bw = 1 << 30;
  for (int n = T < 64 ? 64 / T : 1; n * T <= 256 || n == 1; ++n) {
    const int waste = ((n * T + 63) / 64 * 64 - n * T) * 1024 / (n * T);
    if (waste < bw) {
      best = n;
      bw = waste;
    }
    if (bw <= 102) break;
  }
  return best;
}
// sequences per block of the y transforms: 128-byte rows, at most 1024 threads
// and 64 KiB of LDS
template <typename T, int L>
constexpr int y_seqs() {
  int q = 128 / (2 * (int)sizeof(T));
  while (q > 1 && (q * tps<L>() > 1024 || padded(L * q) * 2 * (int)sizeof(T) > kLdsMax)) q /= 2;
  return q;
}


// Butterfly jj of pass P: from LDS, twiddled, into v.
template <typename T, int S, int L, int ES, int P>
__device__ __forceinline__ void pass_load(const cpx<T>* buf, const cpx<T>* __restrict__ twL,
                                          int soff, int jj, cpx<T>* v) {
  using SH = Shape<L>;
  constexpr int R = SH::plan.r[P], NS = shape_span<SH, P>(), LR = L / R;
  cpx<T> w[R];
  if (NS > 1) {
#pragma unroll
    for (int r = 1; r < R; ++r) w[r] = twL[r * (jj % NS) * (L / (NS * R))];
  }
#pragma unroll
  for (int r = 0; r < R; ++r) v[r] = buf[pad(soff + (jj + r * LR) * ES)];
  if (NS > 1) {
#pragma unroll
    for (int r = 1; r < R; ++r) {
      if (S > 0) w[r].im = -w[r].im;
      v[r] = cmul(v[r], w[r]);
    }
  }
}
// The results of butterfly jj of pass P to LDS.
template <typename T, int L, int ES, int P>
__device__ __forceinline__ void pass_store(cpx<T>* buf, int soff, int jj, const cpx<T>* v) {
  using SH = Shape<L>;
  constexpr int R = SH::plan.r[P], NS = shape_span<SH, P>();
  const int base = (jj / NS) * NS * R + jj % NS;
#pragma unroll
  for (int r = 0; r < R; ++r) buf[pad(soff + (base + r * NS) * ES)] = v[r];
}

// Passes P .. PE-1 in place; `buf` is whole when it starts and when it returns.
template <typename T, int S, int L, int ES, int P, int PE>
__device__ __forceinline__ void stockham(cpx<T>* buf, const cpx<T>* __restrict__ twL, int soff,
                                         int jj) {
  if constexpr (P < PE) {
    constexpr int R = Shape<L>::plan.r[P];
    cpx<T> v[R];
    const bool active = jj < L / R;
    if (active) pass_load<T, S, L, ES, P>(buf, twL, soff, jj, v);
    __syncthreads();
    if (active) {
      dft<T, R, S>(v);
      pass_store<T, L, ES, P>(buf, soff, jj, v);
    }
    __syncthreads();
    stockham<T, S, L, ES, P + 1, PE>(buf, twL, soff, jj);
  }
}

// The last pass: its results v[r] are elements jj + r L/R of the sequence, for
// jj < L/R.
template <typename T, int S, int L, int ES>
__device__ __forceinline__ bool last_pass(const cpx<T>* buf, const cpx<T>* __restrict__ twL,
                                          int soff, int jj, cpx<T>* v) {
  constexpr int P = Shape<L>::np - 1, R = Shape<L>::plan.r[P];
  if (jj >= L / R) return false;
  pass_load<T, S, L, ES, P>(buf, twL, soff, jj, v);
  dft<T, R, S>(v);
  return true;
}

template <typename T>
__device__ __forceinline__ T& real_at(cpx<T>* buf, int e) {
  return reinterpret_cast<T*>(buf)[2 * pad(e >> 1) + (e & 1)];
}

// the largest divisor of n that is at most m
constexpr int chunk_of(int n, int m) {
  int c = m < n ? m : n;
  while (n % c) --c;
  return c;
}

// The velocity divergence of calcRHS (src/mod_calcRHS.cc:7-33), for a forward
// x transform that reads it straight from u, v, w instead of from p.
template <typename T>
struct RhsSrc {
  const T* u;
  const T* v;
  const T* w;
  const T* dzf_inv;
  T dti, dtidxi, dtidyi;
  // the velocity's boundary update did not run: the backward neighbours in
  // the halo are read from their periodic images and w is the wall value 0
  // on planes 0 and nz (src/mod_updateBound.cc:32-144)
  int bcfold;
};

// forceVel's bulk mean and force of u (src/mod_calcVel.cc:287,297) from n block
// partials of stage 2, as a block of its own in the forward transform that
// follows: a launch of one block costs more than its work (5-6 us, of which a
// step of 256x192x128 has 284).  The sums are trees: a chain of 64 additions rounds
// the mean, and with it every u, to 2-4 times the error (64x64x64, rms of 24 runs
// 2.0e-16 against 7e-17).
struct MeanJob {
  const double* partial;
  long n;  // 0: nothing to do
  double nxg, nyg, vel_force;
  double* mean;
  double* force;
};
__device__ __forceinline__ double sum8(const double* s) {
  return ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
}
__device__ __forceinline__ void mean_job(const MeanJob& m) {
  __shared__ double red[64], top[8];
  const int W = blockDim.x < 64 ? (int)blockDim.x : 64, t = threadIdx.x;
  if (t < W) {
    double s = 0.0;
    for (long i = t; i < m.n; i += 8 * W) {
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = i + u * W < m.n ? m.partial[i + u * W] : 0.0;
      s += sum8(v);
    }
    red[t] = s;
    for (int i = t + W; i < 64; i += W) red[i] = 0.0;
  }
  __syncthreads();
  if (t < 8) top[t] = sum8(red + 8 * t);  // a block has at least 8 threads
  __syncthreads();
  if (t == 0) {
    const double mean = sum8(top) / m.nxg / m.nyg;
    *m.mean = mean;
    *m.force = m.vel_force - mean;
  }
}

template <typename T>
RhsSrc<T> rhs_src(const pll_context* c) {
  const double dti = 1.0 / c->dt;  // src/mod_calcRHS.cc:11-13
  return RhsSrc<T>{static_cast<const T*>(c->fld[PLL_U]), static_cast<const T*>(c->fld[PLL_V]),
                   static_cast<const T*>(c->fld[PLL_W]),
                   static_cast<const T*>(c->d_mesh) + (c->g.nz + 2),  // dzf_inv
                   (T)dti, (T)(dti * c->dx_inv), (T)(dti * c->dy_inv), c->rhs_bcfold};
}

// Two neighbouring values in one load or store, aligned to one value.
template <typename T>
struct alignas(sizeof(T)) Two {
  typedef T V __attribute__((ext_vector_type(2)));
  typedef V U __attribute__((aligned(sizeof(T))));
};
template <typename T>
__device__ __forceinline__ cpx<T> load_two(const T* p) {
  const typename Two<T>::V v = *reinterpret_cast<const typename Two<T>::U*>(p);
  return cpx<T>{v[0], v[1]};
}
template <typename T>
__device__ __forceinline__ void store_two(T* p, cpx<T> v) {
  *reinterpret_cast<typename Two<T>::U*>(p) = typename Two<T>::V{v.re, v.im};
}

// execute_fft_fwd_xpen (src/mod_fft.cc:60-88), L = nx/2 points per row.  With
// RHS the rows are calcRHS's output computed on load (nothing is stored in p).
// A row's TPS threads each load the pairs jj + u TPS, the inputs of their own
// first butterflies, so these go from registers: one pass through
// LDS less than with rows staged there first, and no table of rows.  With the step's
// loads, FP64: 57 -> 49 us at 256x192x128, 809 -> 772 at 768x384x384 (6.1 TB/s of
// 41 B a point).  In FP32 the pairs, which are aligned to one value, cost as much
// as single loads: 75 -> 74 us at 384x256x192, 410 -> 432 at 768x384x384.  Taking the
// rows plane after plane within groups of 32 read 24 % less from HBM (w of the
// plane below from the L2) in the same time and left the next pass its input
// in a worse order.
template <typename T, int L, bool RHS>
__global__ __launch_bounds__((x_rows<L>() * tps<L>())) void k_xf(Geom g, const T* __restrict__ p,
                                                               T* __restrict__ spec,
                                                               const cpx<T>* __restrict__ twL,
                                                               const cpx<T>* __restrict__ rtw,
                                                               long nrows, RhsSrc<T> rs,
                                                               MeanJob mj) {
  unsigned bid = blockIdx.x, nblk = gridDim.x;
  if (RHS && mj.n) {
    if (bid == 0) {
      mean_job(mj);
      return;
    }
    --bid;
    --nblk;
  }
  constexpr int TPS = tps<L>(), NB = x_rows<L>(), N = 2 * L, R0 = Shape<L>::plan.r[0];
  static_assert(R0 * TPS == L, "the first radix is the smallest");
  __shared__ cpx<T> buf[padded(NB * L)];
  const int s = threadIdx.x / TPS, jj = threadIdx.x % TPS;
  const long r = (long)xcd_remap(bid, nblk) * NB + s;
  const int rc = (int)(r < nrows ? r : nrows - 1), j = rc % g.ny, k = rc / g.ny;
  const long b = g.idx(1, j + 1, k + 1);
  cpx<T> v[R0];
  if constexpr (RHS) {
    const bool f = rs.bcfold != 0;
    const bool below0 = f && k == 0, top0 = f && k + 1 == g.nz;  // w is the wall 0
    const long vs = f && j == 0 ? (long)(g.ny - 1) * g.sx : -g.sx;   // the v row below, or its image
    const T dz = rs.dti * rs.dzf_inv[k + 1];
    const T *pu = rs.u + b, *pv = rs.v + b, *pw = rs.w + b;
    // the loads of CH pairs are all issued before the first is used
    constexpr int CH = chunk_of(R0, sizeof(T) == 8 ? 4 : 8);
#pragma unroll
    for (int u0 = 0; u0 < R0; u0 += CH) {
      T ul[CH];
      cpx<T> uu[CH], vv[CH], vb[CH], ww[CH], wb[CH];
#pragma unroll
      for (int u = 0; u < CH; ++u) {
        const int i = 2 * (jj + (u0 + u) * TPS);
        uu[u] = load_two(pu + i);
        ul[u] = pu[i == 0 && f ? N - 1 : i - 1];  // u(0) = u(nx)
        vv[u] = load_two(pv + i);
        vb[u] = load_two(pv + vs + i);
        ww[u] = load_two(pw + i);
        wb[u] = load_two(pw - g.sxy + i);
      }
#pragma unroll
      for (int u = 0; u < CH; ++u) {
        if (top0) ww[u] = cpx<T>{T(0), T(0)};
        if (below0) wb[u] = cpx<T>{T(0), T(0)};
        // src/mod_calcRHS.cc:21-28, same association as k_calc_rhs
        v[u0 + u] = cpx<T>{(uu[u].re - ul[u]) * rs.dtidxi + (vv[u].re - vb[u].re) * rs.dtidyi +
                               (ww[u].re - wb[u].re) * dz,
                           (uu[u].im - uu[u].re) * rs.dtidxi + (vv[u].im - vb[u].im) * rs.dtidyi +
                               (ww[u].im - wb[u].im) * dz};
      }
    }
  } else {
#pragma unroll
    for (int u = 0; u < R0; ++u) v[u] = load_two(p + b + 2 * (jj + u * TPS));
  }
  dft<T, R0, -1>(v);
  pass_store<T, L, 1, 0>(buf, s * L, jj, v);
  __syncthreads();
  stockham<T, -1, L, 1, 1, Shape<L>::np>(buf, twL, s * L, jj);
  if (r >= nrows) return;
  cpx<T>* out = reinterpret_cast<cpx<T>*>(spec + r * N);
#pragma unroll
  for (int u = 0; u < R0; ++u) {
    const int kk = jj + u * TPS;
    const cpx<T> zk = buf[pad(s * L + kk)];
    if (kk == 0) {
      out[0] = cpx<T>{zk.re + zk.im, zk.re - zk.im};  // X0, X(n/2)
    } else {
      const cpx<T> zm = buf[pad(s * L + (L - kk))];
      const T er = T(0.5) * (zk.re + zm.re), ei = T(0.5) * (zk.im - zm.im);
      const T orr = T(0.5) * (zk.im + zm.im), oi = T(-0.5) * (zk.re - zm.re);
      const cpx<T> w = rtw[kk];
      out[kk] = cpx<T>{er + (w.re * orr - w.im * oi), ei + (w.re * oi + w.im * orr)};
    }
  }
}

// execute_fft_bwd_xpen (src/mod_fft.cc:90-120): perm rows -> p interior * norm.
// With HALO (the step sequence, where updateBoundP follows at once) a row is
// stored as aligned pairs p(0..nx+1), the two x-halo cells holding their
// periodic values p(nx) and p(1), and a row whose copies updateBoundP puts on
// the y halo or a wall's ghost plane is stored there too (row_images), so that
// boundary update (src/mod_updateBound.cc:253-296) needs no pass of its own.
// Offsets of row (j, k)'s copies (0: none): y the periodic image on the y halo,
// z the zero-gradient ghost plane (src/mod_updateBound.cc:253-296).
struct RowImage {
  long y, z;
};
__device__ __forceinline__ RowImage row_images(const Geom& g, int j, int k) {
  return RowImage{j == 0 ? (long)g.ny * g.sx : (j == g.ny - 1 ? -(long)g.ny * g.sx : 0),
                  k == 0 ? -g.sxy : (k == g.nz - 1 ? g.sxy : 0)};
}
template <typename V>
__device__ __forceinline__ void store_images(V* at, long stride, const RowImage& im, V val) {
  at[0] = val;
  if (im.y) at[im.y / stride] = val;
  if (im.z) at[im.z / stride] = val;
  if (im.y && im.z) at[(im.y + im.z) / stride] = val;
}

// Elements 2n and 2n+1 of a row of p with interior at `out`, its x halos and images.
template <typename T>
__device__ __forceinline__ void store_halo(T* out, const RowImage& im, int n, int L, cpx<T> v) {
  auto at = [&](long d) {
    T* o = out + d;
    store_two(o + 2 * n, v);
    if (n == 0) o[2 * L] = v.re;   // p(nx+1) = p(1)
    if (n == L - 1) o[-1] = v.im;  // p(0) = p(nx)
  };
  at(0);
  if (im.y) at(im.y);
  if (im.z) at(im.z);
  if (im.y && im.z) at(im.y + im.z);
}

template <typename T, int L, bool HALO>
__global__ __launch_bounds__((x_rows<L>() * tps<L>())) void k_xb(Geom g, const T* __restrict__ spec,
                                                               T* __restrict__ p,
                                                               const cpx<T>* __restrict__ twL,
                                                               const cpx<T>* __restrict__ rtw,
                                                               long nrows, T norm) {
  constexpr int TPS = tps<L>(), NB = x_rows<L>(), N = 2 * L, NP = Shape<L>::np;
  constexpr int R0 = Shape<L>::plan.r[0], RE = Shape<L>::plan.r[NP - 1];
  __shared__ cpx<T> buf[padded(NB * L)];
  const int s = threadIdx.x / TPS, jj = threadIdx.x % TPS;
  const long r = (long)xcd_remap(blockIdx.x, gridDim.x) * NB + s;
  const int rc = (int)(r < nrows ? r : nrows - 1), j = rc % g.ny, k = rc / g.ny;
  // perm slot kk holds (Re Xkk, Im Xkk); slot 0 holds (X0, X(n/2)).  A thread
  // loads the slots jj + u TPS, merges them with the slots L - kk (through LDS)
  // and has the inputs of its first butterfly.
  const cpx<T>* in = reinterpret_cast<const cpx<T>*>(spec) + (long)rc * L;
  cpx<T> z[R0];
#pragma unroll
  for (int u = 0; u < R0; ++u) z[u] = in[jj + u * TPS];
#pragma unroll
  for (int u = 0; u < R0; ++u) buf[pad(s * L + jj + u * TPS)] = z[u];
  __syncthreads();
#pragma unroll
  for (int u = 0; u < R0; ++u) {
    const int kk = jj + u * TPS;
    const cpx<T> a = z[u];
    cpx<T> xk = a, xm;
    if (kk == 0) {
      xk = cpx<T>{a.re, T(0)};
      xm = cpx<T>{a.im, T(0)};
    } else {
      xm = buf[pad(s * L + (L - kk))];
    }
    const cpx<T> sm{xk.re + xm.re, xk.im - xm.im};  // Xk + conj(X(h-k))
    const cpx<T> d{xk.re - xm.re, xk.im + xm.im};   // Xk - conj(X(h-k))
    const cpx<T> w{rtw[kk].re, -rtw[kk].im};        // exp(+2 pi i k/n)
    const cpx<T> wd = cmul(w, d);
    z[u] = cpx<T>{sm.re - wd.im, sm.im + wd.re};
  }
  dft<T, R0, +1>(z);
  // the last pass stores its results, elements 2n and 2n+1 of the row
  T* out = p + g.idx(1, j + 1, k + 1);
  const RowImage im = row_images(g, j, k);
  auto store = [&](int n, cpx<T> v) {
    v = cpx<T>{norm * v.re, norm * v.im};
    if (!HALO) {
      store_two(out + 2 * n, v);
      return;
    }
    store_halo(out, im, n, L, v);
  };
  if constexpr (NP == 1) {
    if (r >= nrows) return;
#pragma unroll
    for (int u = 0; u < R0; ++u) store(jj + u * (L / R0), z[u]);
  } else {
    __syncthreads();
    pass_store<T, L, 1, 0>(buf, s * L, jj, z);
    __syncthreads();
    stockham<T, +1, L, 1, 1, NP - 1>(buf, twL, s * L, jj);
    cpx<T> v[RE];
    if (r >= nrows || !last_pass<T, +1, L, 1>(buf, twL, s * L, jj, v)) return;
#pragma unroll
    for (int u = 0; u < RE; ++u) store(jj + u * (L / RE), v[u]);
  }
}

// execute_fft_fwd_ypen (src/mod_fft.cc:122-153) on a tile of 2Q perm columns: slot
// (j, q) is the pair of columns (2q, 2q+1) of row j.  A thread loads the rows
// jj + u TPS of its pair, the inputs of its first butterfly.
template <typename T, int L>
__global__ __launch_bounds__((y_seqs<T, L>() * tps<L>())) void k_yf(Geom g, T* __restrict__ spec,
                                                                  const cpx<T>* __restrict__ twL,
                                                                  int ntiles) {
  constexpr int TPS = tps<L>(), Q = y_seqs<T, L>(), W = 2 * Q, R0 = Shape<L>::plan.r[0];
  __shared__ cpx<T> buf[padded(L * Q)];
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const int tile = (int)(b % (unsigned)ntiles), k = (int)(b / (unsigned)ntiles);
  T* plane = spec + (long)k * g.nx * g.ny + (long)tile * W;
  const int q = threadIdx.x % Q, jj = threadIdx.x / Q;
  const bool on = tile * Q + q < g.nx / 2;  // the last tile of a plane may be ragged
  cpx<T> v[R0] = {};
  if (on) {
#pragma unroll
    for (int u = 0; u < R0; ++u)
      v[u] = reinterpret_cast<const cpx<T>*>(plane + (long)(jj + u * TPS) * g.nx)[q];
  }
  dft<T, R0, -1>(v);
  pass_store<T, L, Q, 0>(buf, q, jj, v);
  __syncthreads();
  stockham<T, -1, L, Q, 1, Shape<L>::np>(buf, twL, q, jj);
  if (!on) return;
#pragma unroll
  for (int mu = 0; mu <= L / 2 / TPS; ++mu) {
    const int m = jj + mu * TPS;
    if (m > L / 2) break;
    const cpx<T> zm = buf[pad(m * Q + q)];
    const cpx<T> zc = buf[pad(((L - m) % L) * Q + q)];
    const T ar = T(0.5) * (zm.re + zc.re), ai = T(0.5) * (zm.im - zc.im);
    const T br = T(0.5) * (zm.im + zc.im), bi = T(-0.5) * (zm.re - zc.re);
    if (m == 0) {
      reinterpret_cast<cpx<T>*>(plane)[q] = cpx<T>{ar, br};
    } else if (m == L / 2) {
      reinterpret_cast<cpx<T>*>(plane + g.nx)[q] = cpx<T>{ar, br};
    } else {
      reinterpret_cast<cpx<T>*>(plane + (long)(2 * m) * g.nx)[q] = cpx<T>{ar, br};
      reinterpret_cast<cpx<T>*>(plane + (long)(2 * m + 1) * g.nx)[q] = cpx<T>{ai, bi};
    }
  }
}

// execute_fft_bwd_ypen (src/mod_fft.cc:155-187), unscaled.
template <typename T, int L>
__global__ __launch_bounds__((y_seqs<T, L>() * tps<L>())) void k_yb(Geom g, T* __restrict__ spec,
                                                                  const cpx<T>* __restrict__ twL,
                                                                  int ntiles) {
  constexpr int TPS = tps<L>(), Q = y_seqs<T, L>(), W = 2 * Q, NP = Shape<L>::np;
  constexpr int RE = Shape<L>::plan.r[NP - 1];
  __shared__ cpx<T> buf[padded(L * Q)];
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const int tile = (int)(b % (unsigned)ntiles), k = (int)(b / (unsigned)ntiles);
  T* plane = spec + (long)k * g.nx * g.ny + (long)tile * W;
  // Global row j, column pair q holds (perm_a[j], perm_b[j]) of columns 2q and
  // 2q+1.  Rows 2m and 2m+1 (m = 1..L/2-1) give the complex inputs Z[m] and
  // Z[L-m] of the pair's transform: with A = (e0.re, e1.re), B = (e0.im,
  // e1.im), Z = A + iB below L/2 and conj(A) + i conj(B) above; rows 0 and 1
  // hold Z[0] and Z[L/2].  Each thread loads its row pairs and writes the
  // unpacked values to LDS directly.
  const int q = threadIdx.x % Q, jj = threadIdx.x / Q;
  const bool on = tile * Q + q < g.nx / 2;
  {
    constexpr int NLD = (L / 2 + TPS - 1) / TPS;
    cpx<T> e0[NLD] = {}, e1[NLD] = {};
#pragma unroll
    for (int u = 0; u < NLD; ++u) {
      const int m = jj + u * TPS;
      if (on && m < L / 2) {
        e0[u] = reinterpret_cast<const cpx<T>*>(plane + (long)(2 * m) * g.nx)[q];
        e1[u] = reinterpret_cast<const cpx<T>*>(plane + (long)(2 * m + 1) * g.nx)[q];
      }
    }
#pragma unroll
    for (int u = 0; u < NLD; ++u) {
      const int m = jj + u * TPS;
      if (m == 0) {
        buf[pad(q)] = e0[u];
        buf[pad((L / 2) * Q + q)] = e1[u];
      } else if (m < L / 2) {
        buf[pad(m * Q + q)] = cpx<T>{e0[u].re - e1[u].im, e1[u].re + e0[u].im};
        buf[pad((L - m) * Q + q)] = cpx<T>{e0[u].re + e1[u].im, e0[u].im - e1[u].re};
      }
    }
  }
  __syncthreads();
  stockham<T, +1, L, Q, 0, NP - 1>(buf, twL, q, jj);
  cpx<T> v[RE];
  if (!last_pass<T, +1, L, Q>(buf, twL, q, jj, v) || !on) return;
#pragma unroll
  for (int u = 0; u < RE; ++u)
    reinterpret_cast<cpx<T>*>(plane + (long)(jj + u * (L / RE)) * g.nx)[q] = v[u];
}

// The bulk mean that stage 2 left partials of, for the transform that runs next.
inline MeanJob take_mean(pll_context* c) {
  const long n = c->mean_pending;
  c->mean_pending = 0;
  return MeanJob{c->d_partial, n, (double)c->g.nx, (double)c->g.ny, c->vel_force[0], c->d_scalar,
                 c->d_scalar + 3};
}

// step: calcRHS in the forward loads, p's boundary update in the inverse's stores
template <typename T, int L>
int launch_xf(pll_context* c, bool step) {
  constexpr int NB = x_rows<L>(), NT = NB * tps<L>();
  const long nrows = (long)c->g.ny * c->g.nz;
  const unsigned blocks = (unsigned)((nrows + NB - 1) / NB);
  const cpx<T>* tw = static_cast<const cpx<T>*>(c->d_twl_x);
  const cpx<T>* rtw = static_cast<const cpx<T>*>(c->d_rtw_x);
  if (step) {
    const MeanJob mj = take_mean(c);
    TimerScope ts(c, K_FFT_X_FWD_RHS);
    hipLaunchKernelGGL((k_xf<T, L, true>), dim3(blocks + (mj.n ? 1 : 0)), dim3(NT), 0, c->stream, c->g,
                       static_cast<const T*>(nullptr), static_cast<T*>(c->spec), tw, rtw, nrows,
                       rhs_src<T>(c), mj);
  } else {
    TimerScope ts(c, K_FFT_X_FWD);
    hipLaunchKernelGGL((k_xf<T, L, false>), dim3(blocks), dim3(NT), 0, c->stream, c->g,
                       static_cast<const T*>(c->fld[PLL_P]), static_cast<T*>(c->spec), tw, rtw,
                       nrows, RhsSrc<T>{}, MeanJob{});
  }
  PLL_HIP_TRY(hipGetLastError());
  return PLL_OK;
}

template <typename T, int L>
int launch_xb(pll_context* c, bool step) {
  constexpr int NB = x_rows<L>(), NT = NB * tps<L>();
  const long nrows = (long)c->g.ny * c->g.nz;
  const double norm = 1.0 / (c->g.nx * c->g.ny);  // src/mod_fft.cc:57
  TimerScope ts(c, K_FFT_X_BWD);
  hipLaunchKernelGGL((step ? k_xb<T, L, true> : k_xb<T, L, false>), dim3((unsigned)((nrows + NB - 1) / NB)),
                     dim3(NT), 0, c->stream, c->g, static_cast<const T*>(c->spec),
                     static_cast<T*>(c->fld[PLL_P]), static_cast<const cpx<T>*>(c->d_twl_x),
                     static_cast<const cpx<T>*>(c->d_rtw_x), nrows, (T)norm);
  PLL_HIP_TRY(hipGetLastError());
  return PLL_OK;
}

template <typename T, int L, bool FWD>
int launch_y(pll_context* c, bool) {
  constexpr int Q = y_seqs<T, L>(), NT = Q * tps<L>();
  const int ntiles = (c->g.nx / 2 + Q - 1) / Q;
  TimerScope ts(c, FWD ? K_FFT_Y_FWD : K_FFT_Y_BWD);
  hipLaunchKernelGGL((FWD ? k_yf<T, L> : k_yb<T, L>), dim3((unsigned)ntiles * c->g.nz), dim3(NT), 0,
                     c->stream, c->g, static_cast<T*>(c->spec),
                     static_cast<const cpx<T>*>(c->d_twl_y), ntiles);
  PLL_HIP_TRY(hipGetLastError());
  return PLL_OK;
}

}  // namespace
}  // namespace pll
