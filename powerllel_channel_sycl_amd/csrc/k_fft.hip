// k_fft.hip -- the pressure-Poisson transforms (src/mod_fft.cc:60-187) as
// hand-written LDS kernels.
//
// x direction: each row of nx reals is transformed as a complex sequence of
// nx/2 points (even samples real, odd samples imaginary) followed by the
// split step that yields the half spectrum; the result is written straight in
// the reference's perm packing [X0, X(n/2), Re X1, Im X1, ...].  The inverse
// runs the same steps backwards and folds in the 1/(nx*ny) scale.
//
// y direction: the work array keeps its [k][j][i] order (no transpose pass).
// A block loads a tile of adjacent perm columns of one k plane; columns
// (2q, 2q+1) form one complex sequence along j, whose DFT is split into the two
// real-column DFTs and written back in perm packing along j.  This is the
// reference's per-column real DFT (src/mod_fft.cc:122-187) computed two
// columns at a time.
//
// Complex transforms use the Stockham autosort formulation, in place in one
// LDS buffer with the butterflies in registers: products of 2, 3 and 5 up to 768
// (but 625) are compiled in (fft_fixed.hpp), others run from a plan.  Twiddles
// are computed on the host in long double and rounded to the field precision.
#include "fft_fixed.hpp"

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdlib>

namespace pll {

namespace {

// ============================================================================
// Run-time-plan transforms for every other length: the same one-buffer Stockham
// passes with the radices of an FftPlan (fft_plan in fft_radix.hpp: the fewest
// passes of radices 2..16, then the largest smallest radix), one butterfly per
// thread and pass, so L = 100 takes two passes (10, 10) and one LDS buffer.
// What matters is loads in flight: kGenChunk loads per thread are issued before
// the first LDS write, and blocks of about 256 threads and at most 32 KiB of LDS
// leave five or more of them on a CU.  Against radix 4/2/3/5 passes ping-ponging in
// 64 KiB blocks the FP64 step at 200x90x176 took 246 instead of 294 us (its four
// transforms 88 instead of 136; compiled in, 61).
// ============================================================================
// n / d by multiplication, m = ceil(2^32 / d): exact for n * d < 2^32, d > 1
__device__ __forceinline__ int div_by(int n, unsigned m) { return (int)__umulhi((unsigned)n, m); }

template <typename T, int S, int R>
__device__ __forceinline__ void plan_pass(cpx<T>* buf, const cpx<T>* __restrict__ twL, int soff,
                                          int es, int jj, bool on, int LR, int ns, unsigned mns,
                                          int tws) {
  cpx<T> v[R];
  const bool active = on && jj < LR;
  if (active) {
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = buf[pad(soff + (jj + r * LR) * es)];
  }
  __syncthreads();
  if (active) {
    int hi = jj, k = 0;
    if (ns > 1) {
      hi = div_by(jj, mns);
      k = jj - hi * ns;
#pragma unroll
      for (int r = 1; r < R; ++r) {
        cpx<T> w = twL[r * k * tws];
        if (S > 0) w.im = -w.im;
        v[r] = cmul(v[r], w);
      }
    }
    dft<T, R, S>(v);
    const int base = hi * ns * R + k;
#pragma unroll
    for (int r = 0; r < R; ++r) buf[pad(soff + (base + r * ns) * es)] = v[r];
  }
  __syncthreads();
}

// All passes in place; `on` is false for threads without a sequence.
template <typename T, int S>
__device__ __forceinline__ void plan_fft(cpx<T>* buf, const FftPlan& pl,
                                         const cpx<T>* __restrict__ twL, int soff, int es, int jj,
                                         bool on) {
  for (int p = 0; p < pl.npass; ++p) {
    const int LR = pl.lr[p], ns = pl.ns[p], tws = pl.tws[p];
    const unsigned mns = pl.mns[p];
#define PLL_PASS(R) \
  case R: plan_pass<T, S, R>(buf, twL, soff, es, jj, on, LR, ns, mns, tws); break;
    switch (pl.radix[p]) {
      PLL_PASS(2)
      PLL_PASS(3)
      PLL_PASS(4)
      PLL_PASS(5)
      PLL_PASS(6)
      PLL_PASS(8)
      PLL_PASS(9)
      PLL_PASS(10)
      PLL_PASS(12)
      PLL_PASS(15)
      default: plan_pass<T, S, 16>(buf, twL, soff, es, jj, on, LR, ns, mns, tws); break;
    }
#undef PLL_PASS
  }
}

constexpr int kGenChunk = 8;      // loads in flight per thread
constexpr int kGenRows = 64;      // most rows of an x block
constexpr int kGenThreads = 1024; // most threads of a block

// Launch shape of an x transform: nb rows per block, magic divisors.
struct XShape {
  int nb, tps;
  unsigned mN, mtps;  // dividing by nx and tps (tps = 1: unused)
};

// k_xf's transform (src/mod_fft.cc:60-88) with a run-time plan.
template <typename T, bool RHS>
__global__ __launch_bounds__(kGenThreads) void k_gxf(Geom g, const T* __restrict__ p,
                                                     T* __restrict__ spec, FftPlan pl, XShape xs,
                                                     const cpx<T>* __restrict__ twL,
                                                     const cpx<T>* __restrict__ rtw, long nrows,
                                                     RhsSrc<T> rs, MeanJob mj) {
  unsigned bid = blockIdx.x, nblk = gridDim.x;
  if (RHS && mj.n) {
    if (bid == 0) {
      mean_job(mj);
      return;
    }
    --bid;
    --nblk;
  }
  extern __shared__ __align__(16) unsigned char smem[];
  cpx<T>* buf = reinterpret_cast<cpx<T>*>(smem);
  __shared__ long rowbase[kGenRows];
  __shared__ T rowdz[kGenRows];
  __shared__ long rowvs[kGenRows];           // offset of the v row below (j-1, or its image)
  __shared__ unsigned char roww[kGenRows];   // bit 0: w below is the wall 0; bit 1: w is the wall 0
  const int N = g.nx, L = N / 2, NT = blockDim.x;
  const long row0 = (long)xcd_remap(bid, nblk) * xs.nb;
  if ((int)threadIdx.x < xs.nb) {
    const long r = row0 + threadIdx.x;
    const int j = (int)(r % g.ny), k = (int)(r / g.ny);
    rowbase[threadIdx.x] = r < nrows ? g.idx(1, j + 1, k + 1) : -1;
    if (RHS) {
      rowdz[threadIdx.x] = r < nrows ? rs.dti * rs.dzf_inv[k + 1] : T(0);
      const bool f = rs.bcfold != 0;
      rowvs[threadIdx.x] = (f && j == 0) ? (long)(g.ny - 1) * g.sx : -g.sx;
      roww[threadIdx.x] = (unsigned char)((f && k == 0 ? 1 : 0) | (f && k + 1 == g.nz ? 2 : 0));
    }
  }
  __syncthreads();
  constexpr int CH = RHS ? kGenChunk / 2 : kGenChunk;
  const int total = xs.nb * N;
  for (int e0 = threadIdx.x; e0 < total; e0 += CH * NT) {
    T a0[CH], a1[CH], a2[CH], a3[CH], a4[CH], a5[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int e = e0 + u * NT;
      a0[u] = a1[u] = a2[u] = a3[u] = a4[u] = a5[u] = T(0);
      if (e < total) {
        const int s = div_by(e, xs.mN), i = e - s * N;
        const long b = rowbase[s];
        if (b >= 0) {
          const long c = b + i;
          if (RHS) {
            const long cw = (i == 0 && rs.bcfold) ? b + (N - 1) : c - 1;  // u(0) = u(nx)
            const unsigned char wf = roww[s];
            a0[u] = rs.u[c];
            a1[u] = rs.u[cw];
            a2[u] = rs.v[c];
            a3[u] = rs.v[c + rowvs[s]];
            if (!(wf & 2)) a4[u] = rs.w[c];
            if (!(wf & 1)) a5[u] = rs.w[c - g.sxy];
          } else {
            a0[u] = p[c];
          }
        }
      }
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int e = e0 + u * NT;
      if (e < total) {
        T val = a0[u];
        if (RHS) {
          // src/mod_calcRHS.cc:21-28, same association as k_calc_rhs
          val = (a0[u] - a1[u]) * rs.dtidxi + (a2[u] - a3[u]) * rs.dtidyi +
                (a4[u] - a5[u]) * rowdz[div_by(e, xs.mN)];
        }
        real_at(buf, e) = val;  // row s starts at element s * N
      }
    }
  }
  __syncthreads();
  const int s = xs.tps > 1 ? div_by(threadIdx.x, xs.mtps) : (int)threadIdx.x;
  const int jj = (int)threadIdx.x - s * xs.tps;
  const bool on = s < xs.nb;
  plan_fft<T, -1>(buf, pl, twL, s * L, 1, jj, on);
  const long r = row0 + s;
  if (!on || r >= nrows) return;
  cpx<T>* out = reinterpret_cast<cpx<T>*>(spec + r * N);
  for (int kk = jj; kk < L; kk += xs.tps) {
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

// k_xb's transform (src/mod_fft.cc:90-120) with a run-time plan.  One thread
// merges slots kk and L - kk, so the merge runs in place without a barrier.
template <typename T, bool HALO>
__global__ __launch_bounds__(kGenThreads) void k_gxb(Geom g, const T* __restrict__ spec,
                                                     T* __restrict__ p, FftPlan pl, XShape xs,
                                                     const cpx<T>* __restrict__ twL,
                                                     const cpx<T>* __restrict__ rtw, long nrows,
                                                     unsigned mP, T norm) {
  extern __shared__ __align__(16) unsigned char smem[];
  cpx<T>* buf = reinterpret_cast<cpx<T>*>(smem);
  __shared__ long rowbase[kGenRows];
  __shared__ RowImage rowimg[kGenRows];
  const int N = g.nx, L = N / 2, NT = blockDim.x;
  const long row0 = (long)xcd_remap(blockIdx.x, gridDim.x) * xs.nb;
  if ((int)threadIdx.x < xs.nb) {
    const long r = row0 + threadIdx.x;
    const int j = (int)(r % g.ny), k = (int)(r / g.ny);
    rowbase[threadIdx.x] = r < nrows ? g.idx(HALO ? 0 : 1, j + 1, k + 1) : -1;
    if (HALO) rowimg[threadIdx.x] = row_images(g, j, k);
  }
  const cpx<T>* specc = reinterpret_cast<const cpx<T>*>(spec) + row0 * L;
  const int slots = xs.nb * L;
  const long have = (nrows - row0) * L;  // slots of rows that exist
  for (int e0 = threadIdx.x; e0 < slots; e0 += kGenChunk * NT) {
    cpx<T> t[kGenChunk];
#pragma unroll
    for (int u = 0; u < kGenChunk; ++u) {
      const int e = e0 + u * NT;
      t[u] = e < slots && e < have ? specc[e] : cpx<T>{T(0), T(0)};
    }
#pragma unroll
    for (int u = 0; u < kGenChunk; ++u) {
      const int e = e0 + u * NT;
      if (e < slots) buf[pad(e)] = t[u];
    }
  }
  __syncthreads();
  const int s = xs.tps > 1 ? div_by(threadIdx.x, xs.mtps) : (int)threadIdx.x;
  const int jj = (int)threadIdx.x - s * xs.tps;
  const bool on = s < xs.nb;
  // perm slot kk holds (Re Xkk, Im Xkk); slot 0 holds (X0, X(n/2))
  if (on) {
    auto merge = [&](cpx<T> xk, cpx<T> xm, int kk) {
      const cpx<T> sm{xk.re + xm.re, xk.im - xm.im};  // Xk + conj(X(h-k))
      const cpx<T> d{xk.re - xm.re, xk.im + xm.im};   // Xk - conj(X(h-k))
      const cpx<T> w{rtw[kk].re, -rtw[kk].im};        // exp(+2 pi i k/n)
      const cpx<T> wd = cmul(w, d);
      return cpx<T>{sm.re - wd.im, sm.im + wd.re};
    };
    for (int kk = jj; kk <= L / 2; kk += xs.tps) {
      cpx<T>& lo = buf[pad(s * L + kk)];
      const cpx<T> a = lo;
      if (kk == 0) {
        lo = merge(cpx<T>{a.re, T(0)}, cpx<T>{a.im, T(0)}, 0);
      } else {
        cpx<T>& hi = buf[pad(s * L + (L - kk))];
        const cpx<T> b = hi;
        lo = merge(a, b, kk);
        if (2 * kk != L) hi = merge(b, a, L - kk);
      }
    }
  }
  __syncthreads();
  plan_fft<T, +1>(buf, pl, twL, s * L, 1, jj, on);
  if (HALO) {
    // pair q = (p(2q), p(2q+1)); p(i) is element i-1 of the row, p(0) = p(nx), p(nx+1) = p(1)
    const int NP = L + 1;
    for (int e = threadIdx.x; e < xs.nb * NP; e += NT) {
      const int s2 = div_by(e, mP), q = e - s2 * NP;
      if (rowbase[s2] < 0) continue;
      const int i0 = q == 0 ? N - 1 : 2 * q - 1, i1 = q == L ? 0 : 2 * q;
      store_images(reinterpret_cast<cpx<T>*>(p + rowbase[s2]) + q, 2, rowimg[s2],
                   cpx<T>{norm * real_at(buf, s2 * N + i0), norm * real_at(buf, s2 * N + i1)});
    }
  } else {
    for (int e = threadIdx.x; e < xs.nb * N; e += NT) {
      const int s2 = div_by(e, xs.mN);
      if (rowbase[s2] >= 0) p[rowbase[s2] + (e - s2 * N)] = norm * real_at(buf, e);
    }
  }
}

// k_yf's transform (src/mod_fft.cc:122-153) with a run-time plan: a tile of
// 2^lq column pairs of one k plane, the last tile of a plane possibly ragged.
template <typename T>
__global__ __launch_bounds__(kGenThreads) void k_gyf(Geom g, T* __restrict__ spec, FftPlan pl,
                                                     const cpx<T>* __restrict__ twL, int lq,
                                                     int ntiles) {
  extern __shared__ __align__(16) unsigned char smem[];
  cpx<T>* buf = reinterpret_cast<cpx<T>*>(smem);
  const int L = g.ny, Q = 1 << lq, NT = blockDim.x;
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const int tile = (int)(b % (unsigned)ntiles), k = (int)(b / (unsigned)ntiles);
  T* plane = spec + (long)k * g.nx * g.ny + ((long)tile << (lq + 1));
  const int have = g.nx / 2 - (tile << lq);  // column pairs of this tile that exist
  const int total = L << lq;
  for (int e0 = threadIdx.x; e0 < total; e0 += kGenChunk * NT) {
    cpx<T> t[kGenChunk];
#pragma unroll
    for (int u = 0; u < kGenChunk; ++u) {
      const int e = e0 + u * NT, q = e & (Q - 1);
      t[u] = e < total && q < have ? reinterpret_cast<const cpx<T>*>(plane + (long)(e >> lq) * g.nx)[q]
                                   : cpx<T>{T(0), T(0)};
    }
#pragma unroll
    for (int u = 0; u < kGenChunk; ++u) {
      const int e = e0 + u * NT;
      if (e < total) buf[pad(e)] = t[u];
    }
  }
  __syncthreads();
  const int q = (int)threadIdx.x & (Q - 1), jj = (int)threadIdx.x >> lq;
  plan_fft<T, -1>(buf, pl, twL, q, Q, jj, jj < pl.tps);
  if (q >= have) return;
  for (int m = jj; m <= L / 2; m += NT >> lq) {
    const cpx<T> zm = buf[pad(m * Q + q)];
    const cpx<T> zc = buf[pad((m == 0 ? 0 : L - m) * Q + q)];
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

// k_yb's transform (src/mod_fft.cc:155-187, unscaled) with a run-time plan.
template <typename T>
__global__ __launch_bounds__(kGenThreads) void k_gyb(Geom g, T* __restrict__ spec, FftPlan pl,
                                                     const cpx<T>* __restrict__ twL, int lq,
                                                     int ntiles) {
  extern __shared__ __align__(16) unsigned char smem[];
  cpx<T>* buf = reinterpret_cast<cpx<T>*>(smem);
  const int L = g.ny, Q = 1 << lq, NT = blockDim.x;
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const int tile = (int)(b % (unsigned)ntiles), k = (int)(b / (unsigned)ntiles);
  T* plane = spec + (long)k * g.nx * g.ny + ((long)tile << (lq + 1));
  const int have = g.nx / 2 - (tile << lq);
  // rows 2m and 2m+1 unpack into the complex inputs Z[m] and Z[L-m] (k_yb)
  constexpr int CH = kGenChunk / 2;
  const int total = (L / 2) << lq;
  for (int e0 = threadIdx.x; e0 < total; e0 += CH * NT) {
    cpx<T> r0[CH], r1[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int e = e0 + u * NT, mm = e >> lq, q = e & (Q - 1);
      r0[u] = r1[u] = cpx<T>{T(0), T(0)};
      if (e < total && q < have) {
        r0[u] = reinterpret_cast<const cpx<T>*>(plane + (long)(2 * mm) * g.nx)[q];
        r1[u] = reinterpret_cast<const cpx<T>*>(plane + (long)(2 * mm + 1) * g.nx)[q];
      }
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int e = e0 + u * NT, mm = e >> lq, q = e & (Q - 1);
      if (e < total) {
        if (mm == 0) {
          buf[pad(q)] = r0[u];
          buf[pad((L / 2) * Q + q)] = r1[u];
        } else {
          buf[pad(mm * Q + q)] = cpx<T>{r0[u].re - r1[u].im, r1[u].re + r0[u].im};
          buf[pad((L - mm) * Q + q)] = cpx<T>{r0[u].re + r1[u].im, r0[u].im - r1[u].re};
        }
      }
    }
  }
  __syncthreads();
  const int q = (int)threadIdx.x & (Q - 1), jj = (int)threadIdx.x >> lq;
  plan_fft<T, +1>(buf, pl, twL, q, Q, jj, jj < pl.tps);
  if (q >= have) return;
  for (int j = jj; j < L; j += NT >> lq)
    reinterpret_cast<cpx<T>*>(plane + (long)j * g.nx)[q] = buf[pad(j * Q + q)];
}

// ============================================================================
// Whole planes: on the smallest x-y planes one kernel each way runs both transforms
// of the step (calcRHS in the loads, p's boundary update in the stores).  A step of
// such a grid is a chain of launches, 3-4 us each for the host: four instead of
// six.  24x20x12 (FP64, 10 steps): 172 against 237 us where several runs share the
// host's launches, 358 against 359 us for one run alone.
// Complex slot j Lx + q of the buffer is element q of row j to the x transforms and,
// after their split, the column pair (2q, 2q+1) of row j to the y transforms.
// ============================================================================
// The largest plane that they take, in complex slots nx/2 ny: one block a plane is a
// longer chain of passes than two kernels of many blocks, and beyond 512 slots a
// run alone loses more to it than the launches cost (FP64 32x32x64 37.4 -> 36.1 us a
// step, 48x48x32 34.3 -> 38.6, 64x64x64 41.7 -> 47.0).
constexpr int kPlaneSlots = 512;
struct PlaneShape {
  int bx, lby;            // rows, log2 of the column pairs that the block transforms at a time
  unsigned mtps, mL, mH;  // dividing by plan_x.tps (tps = 1: unused), Lx and Lx/2 + 1
};

// Both directions of x on the plane's rows, rows of a batch side by side.
template <typename T, int S>
__device__ __forceinline__ void plane_x(cpx<T>* buf, const Geom& g, const FftPlan& px,
                                        const PlaneShape& ps, const cpx<T>* __restrict__ tw) {
  const int s = px.tps > 1 ? div_by(threadIdx.x, ps.mtps) : (int)threadIdx.x;
  const int jj = (int)threadIdx.x - s * px.tps;
  for (int r0 = 0; r0 < g.ny; r0 += ps.bx)
    plan_fft<T, S>(buf, px, tw, (r0 + s) * px.L, 1, jj, s < ps.bx && r0 + s < g.ny);
}
template <typename T, int S>
__device__ __forceinline__ void plane_y(cpx<T>* buf, const FftPlan& px, const FftPlan& py,
                                        const PlaneShape& ps, const cpx<T>* __restrict__ tw) {
  const int by = 1 << ps.lby, q = (int)threadIdx.x & (by - 1), jj = (int)threadIdx.x >> ps.lby;
  for (int q0 = 0; q0 < px.L; q0 += by)
    plan_fft<T, S>(buf, py, tw, q0 + q, px.L, jj, jj < py.tps && q0 + q < px.L);
}

// src/mod_calcRHS.cc:7-33, then src/mod_fft.cc:60-88 and :122-153
template <typename T>
__global__ __launch_bounds__(kPlaneSlots / 2) void k_plane_fwd(
    Geom g, T* __restrict__ spec, FftPlan px, FftPlan py, PlaneShape ps,
    const cpx<T>* __restrict__ twx, const cpx<T>* __restrict__ rtw,
    const cpx<T>* __restrict__ twy, RhsSrc<T> rs, MeanJob mj) {
  int k = blockIdx.x;  // plane k+1
  if (mj.n) {
    if (k == 0) {
      mean_job(mj);
      return;
    }
    --k;
  }
  extern __shared__ __align__(16) unsigned char smem[];
  cpx<T>* buf = reinterpret_cast<cpx<T>*>(smem);
  const int L = px.L, N = 2 * L, NT = blockDim.x, total = g.ny * L;
  const bool f = rs.bcfold != 0;
  const bool below0 = f && k == 0, top0 = f && k + 1 == g.nz;  // w is the wall 0
  const T dz = rs.dti * rs.dzf_inv[k + 1];
  const long b0 = g.idx(1, 1, k + 1);
  constexpr int CH = 2;
  for (int e0 = threadIdx.x; e0 < total; e0 += CH * NT) {
    T ul[CH];
    cpx<T> uu[CH], vv[CH], vb[CH], ww[CH], wb[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int e = e0 + u * NT;
      if (e < total) {
        const int j = div_by(e, ps.mL), i = 2 * (e - j * L);
        const long c = b0 + (long)j * g.sx;
        uu[u] = load_two(rs.u + c + i);
        ul[u] = rs.u[c + (i == 0 && f ? N - 1 : i - 1)];  // u(0) = u(nx)
        vv[u] = load_two(rs.v + c + i);
        vb[u] = load_two(rs.v + c + (f && j == 0 ? (long)(g.ny - 1) * g.sx : -g.sx) + i);
        ww[u] = load_two(rs.w + c + i);
        wb[u] = load_two(rs.w + c - g.sxy + i);
      }
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int e = e0 + u * NT;
      if (e < total) {
        if (top0) ww[u] = cpx<T>{T(0), T(0)};
        if (below0) wb[u] = cpx<T>{T(0), T(0)};
        // src/mod_calcRHS.cc:21-28, same association as k_calc_rhs
        buf[pad(e)] = cpx<T>{(uu[u].re - ul[u]) * rs.dtidxi + (vv[u].re - vb[u].re) * rs.dtidyi +
                                 (ww[u].re - wb[u].re) * dz,
                             (uu[u].im - uu[u].re) * rs.dtidxi + (vv[u].im - vb[u].im) * rs.dtidyi +
                                 (ww[u].im - wb[u].im) * dz};
      }
    }
  }
  __syncthreads();
  plane_x<T, -1>(buf, g, px, ps, twx);
  // split the rows in place: one thread takes slots kk and L - kk
  const int H = L / 2 + 1;
  for (int e = threadIdx.x; e < g.ny * H; e += NT) {
    const int j = div_by(e, ps.mH), kk = e - j * H;
    auto half = [&](cpx<T> zk, cpx<T> zm, int n) {
      const T er = T(0.5) * (zk.re + zm.re), ei = T(0.5) * (zk.im - zm.im);
      const T orr = T(0.5) * (zk.im + zm.im), oi = T(-0.5) * (zk.re - zm.re);
      const cpx<T> w = rtw[n];
      return cpx<T>{er + (w.re * orr - w.im * oi), ei + (w.re * oi + w.im * orr)};
    };
    cpx<T>& lo = buf[pad(j * L + kk)];
    const cpx<T> a = lo;
    if (kk == 0) {
      lo = cpx<T>{a.re + a.im, a.re - a.im};  // X0, X(n/2)
    } else if (2 * kk <= L) {
      cpx<T>& hi = buf[pad(j * L + (L - kk))];
      const cpx<T> b = hi;
      lo = half(a, b, kk);
      if (2 * kk != L) hi = half(b, a, L - kk);
    }
  }
  __syncthreads();
  plane_y<T, -1>(buf, px, py, ps, twy);
  cpx<T>* out = reinterpret_cast<cpx<T>*>(spec + (long)k * g.nx * g.ny);
  for (int e = threadIdx.x; e < (g.ny / 2 + 1) * L; e += NT) {
    const int m = div_by(e, ps.mL), q = e - m * L;
    const cpx<T> zm = buf[pad(m * L + q)];
    const cpx<T> zc = buf[pad((m == 0 ? 0 : g.ny - m) * L + q)];
    const cpx<T> re{T(0.5) * (zm.re + zc.re), T(0.5) * (zm.im + zc.im)};
    const cpx<T> im{T(0.5) * (zm.im - zc.im), T(-0.5) * (zm.re - zc.re)};
    if (m == 0) {
      out[q] = re;
    } else if (2 * m == g.ny) {
      out[L + q] = re;
    } else {
      out[2 * m * L + q] = re;
      out[(2 * m + 1) * L + q] = im;
    }
  }
}

// src/mod_fft.cc:155-187 and :90-120, then src/mod_updateBound.cc:253-296
template <typename T>
__global__ __launch_bounds__(kPlaneSlots / 2) void k_plane_bwd(
    Geom g, const T* __restrict__ spec, T* __restrict__ p, FftPlan px, FftPlan py, PlaneShape ps,
    const cpx<T>* __restrict__ twx, const cpx<T>* __restrict__ rtw,
    const cpx<T>* __restrict__ twy, T norm) {
  extern __shared__ __align__(16) unsigned char smem[];
  cpx<T>* buf = reinterpret_cast<cpx<T>*>(smem);
  const int k = blockIdx.x, L = px.L, NT = blockDim.x;
  // rows 2m and 2m+1 unpack into the complex inputs Z[m] and Z[ny-m] (k_yb)
  const cpx<T>* in = reinterpret_cast<const cpx<T>*>(spec + (long)k * g.nx * g.ny);
  constexpr int CH = 2;
  const int half = g.ny / 2 * L;
  for (int e0 = threadIdx.x; e0 < half; e0 += CH * NT) {
    cpx<T> r0[CH], r1[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int e = e0 + u * NT;
      if (e < half) {
        const int m = div_by(e, ps.mL), q = e - m * L;
        r0[u] = in[2 * m * L + q];
        r1[u] = in[(2 * m + 1) * L + q];
      }
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int e = e0 + u * NT;
      if (e < half) {
        const int m = div_by(e, ps.mL), q = e - m * L;
        if (m == 0) {
          buf[pad(q)] = r0[u];
          buf[pad(g.ny / 2 * L + q)] = r1[u];
        } else {
          buf[pad(m * L + q)] = cpx<T>{r0[u].re - r1[u].im, r1[u].re + r0[u].im};
          buf[pad((g.ny - m) * L + q)] = cpx<T>{r0[u].re + r1[u].im, r0[u].im - r1[u].re};
        }
      }
    }
  }
  __syncthreads();
  plane_y<T, +1>(buf, px, py, ps, twy);
  // perm slot kk holds (Re Xkk, Im Xkk); slot 0 holds (X0, X(n/2)).  One thread
  // merges slots kk and L - kk.
  const int H = L / 2 + 1;
  for (int e = threadIdx.x; e < g.ny * H; e += NT) {
    const int j = div_by(e, ps.mH), kk = e - j * H;
    auto merge = [&](cpx<T> xk, cpx<T> xm, int n) {
      const cpx<T> sm{xk.re + xm.re, xk.im - xm.im};  // Xk + conj(X(h-k))
      const cpx<T> d{xk.re - xm.re, xk.im + xm.im};   // Xk - conj(X(h-k))
      const cpx<T> w{rtw[n].re, -rtw[n].im};          // exp(+2 pi i k/n)
      const cpx<T> wd = cmul(w, d);
      return cpx<T>{sm.re - wd.im, sm.im + wd.re};
    };
    cpx<T>& lo = buf[pad(j * L + kk)];
    const cpx<T> a = lo;
    if (kk == 0) {
      lo = merge(cpx<T>{a.re, T(0)}, cpx<T>{a.im, T(0)}, 0);
    } else if (2 * kk <= L) {
      cpx<T>& hi = buf[pad(j * L + (L - kk))];
      const cpx<T> b = hi;
      lo = merge(a, b, kk);
      if (2 * kk != L) hi = merge(b, a, L - kk);
    }
  }
  __syncthreads();
  plane_x<T, +1>(buf, g, px, ps, twx);
  for (int e = threadIdx.x; e < g.ny * L; e += NT) {
    const int j = div_by(e, ps.mL), n = e - j * L;
    const cpx<T> z = buf[pad(e)];
    store_halo(p + g.idx(1, j + 1, k + 1), row_images(g, j, k), n, L, cpx<T>{norm * z.re, norm * z.im});
  }
}

// ---- host side -------------------------------------------------------------------
unsigned magic(int d) { return (unsigned)((0x100000000ULL + (unsigned)d - 1) / (unsigned)d); }

bool build_plan(int L, FftPlan& pl) {
  int rad[kMaxPass];
  const int np = fft_plan(L, kGenThreads, rad);
  if (np < 1) return false;
  pl.L = L;
  pl.npass = np;
  int ns = 1, rmin = L;
  for (int p = 0; p < np; ++p) {
    const int R = rad[p];
    pl.radix[p] = R;
    pl.ns[p] = ns;
    pl.lr[p] = L / R;
    pl.tws[p] = L / (ns * R);
    pl.mns[p] = ns > 1 ? magic(ns) : 0;
    ns *= R;
    rmin = R < rmin ? R : rmin;
  }
  pl.tps = L / rmin;
  return true;
}

template <typename T>
int upload_table(pll_context* c, const std::vector<std::complex<long double>>& src, void** dst) {
  std::vector<cpx<T>> h(src.size());
  for (size_t t = 0; t < src.size(); ++t) h[t] = cpx<T>{(T)src[t].real(), (T)src[t].imag()};
  PLL_HIP_TRY(ctx_malloc(c, dst, h.size() * sizeof(cpx<T>)));
  PLL_HIP_TRY(hipMemcpy(*dst, h.data(), h.size() * sizeof(cpx<T>), hipMemcpyHostToDevice));
  return PLL_OK;
}

// The longest lengths taken: two complex rows (or column pairs) of 64 KiB.
constexpr size_t kLdsBudget = 64 * 1024;
// LDS of a run-time-plan block: several blocks per CU
constexpr size_t kGenLds = 32 * 1024;

template <typename T>
int setup_t(pll_context* c) {
  const int nx = c->g.nx, ny = c->g.ny;
  if ((size_t)nx * sizeof(T) * 2 > kLdsBudget)
    return fail(PLL_ERR_ARG, "nx too large for one LDS row transform");
  if ((size_t)ny * sizeof(T) * 4 > kLdsBudget)
    return fail(PLL_ERR_ARG, "ny too large for one LDS column transform");
  if (!build_plan(nx / 2, c->plan_x)) return fail(PLL_ERR_ARG, "nx/2 must factor into 2, 3, 5");
  if (!build_plan(ny, c->plan_y)) return fail(PLL_ERR_ARG, "ny must factor into 2, 3, 5");
  std::vector<std::complex<long double>> rtw;
  const long double two_pi = 6.283185307179586476925286766559005768L;
  for (int k = 0; k <= nx / 2; ++k) {
    const long double ang = -two_pi * (long double)k / (long double)nx;
    rtw.emplace_back(cosl(ang), sinl(ang));
  }
  int rc;
  if ((rc = upload_table<T>(c, rtw, &c->d_rtw_x))) return rc;
  // rows per block of the x transforms: about 256 threads within kGenLds, fewer
  // where that would leave the chip with under two blocks per CU
  const long nrows = (long)ny * c->g.nz;
  int nb = std::max(1, std::min(kGenRows, 256 / c->plan_x.tps));
  while (nb > 1 && (size_t)padded(nb * (nx / 2)) * 2 * sizeof(T) > kGenLds) --nb;
  while (nb > 1 && nrows / nb < 512) nb = (nb + 1) / 2;
  c->x_batch = nb;
  // column pairs per block of the y transforms: 128-byte rows within 1024
  // threads and kLdsBudget, no more than the plane has
  int lq = sizeof(T) == 8 ? 3 : 4;
  while (lq > 0 && ((c->plan_y.tps << lq) > kGenThreads ||
                    (size_t)padded(ny << lq) * 2 * sizeof(T) > kLdsBudget ||
                    (1 << (lq - 1)) >= nx / 2))
    --lq;
  c->y_tile = lq;
  return PLL_OK;
}

int round_wave(int n) { return (n + 63) / 64 * 64; }

XShape x_shape(const pll_context* c) {
  const int tps = c->plan_x.tps;
  return XShape{c->x_batch, tps, magic(c->g.nx), tps > 1 ? magic(tps) : 0};
}

template <typename T>
int x_generic(pll_context* c, bool fwd, bool step) {
  const long nrows = (long)c->g.ny * c->g.nz;
  const XShape xs = x_shape(c);
  const int L = c->g.nx / 2;
  const dim3 blocks((unsigned)((nrows + xs.nb - 1) / xs.nb)), threads(round_wave(xs.nb * xs.tps));
  const size_t sh = (size_t)padded(xs.nb * L) * 2 * sizeof(T);
  const cpx<T>* tw = static_cast<const cpx<T>*>(c->d_twl_x);
  const cpx<T>* rtw = static_cast<const cpx<T>*>(c->d_rtw_x);
  T* p = static_cast<T*>(c->fld[PLL_P]);
  T* spec = static_cast<T*>(c->spec);
  if (fwd && step) {
    const MeanJob mj = take_mean(c);
    TimerScope ts(c, K_FFT_X_FWD_RHS);
    hipLaunchKernelGGL((k_gxf<T, true>), dim3(blocks.x + (mj.n ? 1 : 0)), threads, sh, c->stream, c->g,
                       static_cast<const T*>(nullptr), spec, c->plan_x, xs, tw, rtw, nrows,
                       rhs_src<T>(c), mj);
  } else if (fwd) {
    TimerScope ts(c, K_FFT_X_FWD);
    hipLaunchKernelGGL((k_gxf<T, false>), blocks, threads, sh, c->stream, c->g,
                       static_cast<const T*>(p), spec, c->plan_x, xs, tw, rtw, nrows, RhsSrc<T>{},
                       MeanJob{});
  } else {
    const double norm = 1.0 / (c->g.nx * c->g.ny);  // src/mod_fft.cc:57
    TimerScope ts(c, K_FFT_X_BWD);
    hipLaunchKernelGGL((step ? k_gxb<T, true> : k_gxb<T, false>), blocks, threads, sh, c->stream,
                       c->g, static_cast<const T*>(spec), p, c->plan_x, xs, tw, rtw, nrows,
                       magic(L + 1), (T)norm);
  }
  PLL_HIP_TRY(hipGetLastError());
  return PLL_OK;
}

template <typename T>
int y_generic(pll_context* c, bool fwd) {
  const int lq = c->y_tile, ntiles = (c->g.nx / 2 + (1 << lq) - 1) >> lq;
  const dim3 blocks((unsigned)ntiles * c->g.nz), threads(round_wave(c->plan_y.tps << lq));
  const size_t sh = (size_t)padded(c->g.ny << lq) * 2 * sizeof(T);
  TimerScope ts(c, fwd ? K_FFT_Y_FWD : K_FFT_Y_BWD);
  hipLaunchKernelGGL((fwd ? k_gyf<T> : k_gyb<T>), blocks, threads, sh, c->stream, c->g,
                     static_cast<T*>(c->spec), c->plan_y, static_cast<const cpx<T>*>(c->d_twl_y),
                     lq, ntiles);
  PLL_HIP_TRY(hipGetLastError());
  return PLL_OK;
}

// step: calcRHS in the forward loads, periodic halos in the inverse's stores
template <typename T>
int x_t(pll_context* c, bool fwd, bool step = false) {
  if (c->x_fixed)
    return fwd ? fft_fixed<T, FftPass::x_fwd>(c, c->g.nx / 2, step)
               : fft_fixed<T, FftPass::x_bwd>(c, c->g.nx / 2, step);
  return x_generic<T>(c, fwd, step);
}

template <typename T>
int y_t(pll_context* c, bool fwd) {
  if (c->y_fixed)
    return fwd ? fft_fixed<T, FftPass::y_fwd>(c, c->g.ny, false)
               : fft_fixed<T, FftPass::y_bwd>(c, c->g.ny, false);
  return y_generic<T>(c, fwd);
}

// W_L^t = exp(-2 pi i t / L), t = 0..L-1, for the fixed-length kernels.
template <typename T>
int unit_table(pll_context* c, int L, void** dst) {
  const long double two_pi = 6.283185307179586476925286766559005768L;
  std::vector<std::complex<long double>> t;
  for (int k = 0; k < L; ++k) {
    const long double ang = -two_pi * (long double)k / (long double)L;
    t.emplace_back(cosl(ang), sinl(ang));
  }
  return upload_table<T>(c, t, dst);
}

void setup_plane(pll_context* c) {
  const long slots = (long)c->g.nx / 2 * c->g.ny;
  // two slots a thread; plans of so short rows and columns take no more threads
  c->plane_threads = slots <= kPlaneSlots
                         ? std::max(round_wave((int)(slots + 1) / 2),
                                    round_wave(std::max(c->plan_x.tps, c->plan_y.tps)))
                         : 0;
}
template <typename T>
int plane_t(pll_context* c, bool fwd) {
  const int L = c->g.nx / 2, nt = c->plane_threads;
  PlaneShape ps{nt / c->plan_x.tps, 0, c->plan_x.tps > 1 ? magic(c->plan_x.tps) : 0,
                magic(L), magic(L / 2 + 1)};
  while ((c->plan_y.tps << (ps.lby + 1)) <= nt && (1 << ps.lby) < L) ++ps.lby;
  const cpx<T>* twx = static_cast<const cpx<T>*>(c->d_twl_x);
  const cpx<T>* twy = static_cast<const cpx<T>*>(c->d_twl_y);
  const cpx<T>* rtw = static_cast<const cpx<T>*>(c->d_rtw_x);
  T* spec = static_cast<T*>(c->spec);
  const size_t lds = (size_t)padded(c->g.ny * L) * 2 * sizeof(T);
  if (fwd) {
    const MeanJob mj = take_mean(c);
    TimerScope ts(c, K_PLANE_FWD);
    hipLaunchKernelGGL((k_plane_fwd<T>), dim3(c->g.nz + (mj.n ? 1 : 0)), dim3(nt), lds,
                       c->stream, c->g, spec, c->plan_x, c->plan_y, ps, twx, rtw, twy, rhs_src<T>(c),
                       mj);
  } else {
    const double norm = 1.0 / (c->g.nx * c->g.ny);  // src/mod_fft.cc:57
    TimerScope ts(c, K_PLANE_BWD);
    hipLaunchKernelGGL((k_plane_bwd<T>), dim3(c->g.nz), dim3(nt), lds, c->stream, c->g,
                       static_cast<const T*>(spec), static_cast<T*>(c->fld[PLL_P]), c->plan_x,
                       c->plan_y, ps, twx, rtw, twy, (T)norm);
  }
  PLL_HIP_TRY(hipGetLastError());
  return PLL_OK;
}

template <typename T>
int setup_fixed(pll_context* c) {
  const char* env = std::getenv("PLL_FFT_GENERIC");
  const bool force_generic = env && env[0] == '1';
  c->x_fixed = !force_generic && fixed_length(c->g.nx / 2);
  c->y_fixed = !force_generic && fixed_length(c->g.ny);
  int rc;
  if ((rc = unit_table<T>(c, c->g.nx / 2, &c->d_twl_x))) return rc;
  if ((rc = unit_table<T>(c, c->g.ny, &c->d_twl_y))) return rc;
  if (!force_generic) setup_plane(c);
  return PLL_OK;
}

}  // namespace

int fft_setup(pll_context* c) {
  int rc = c->prec == PLL_FP64 ? setup_t<double>(c) : setup_t<float>(c);
  if (rc) return rc;
  return c->prec == PLL_FP64 ? setup_fixed<double>(c) : setup_fixed<float>(c);
}
int launch_fft_x_fwd(pll_context* c) { return c->prec == PLL_FP64 ? x_t<double>(c, true) : x_t<float>(c, true); }

int launch_fft_x_fwd_rhs(pll_context* c) {
  return c->prec == PLL_FP64 ? x_t<double>(c, true, true) : x_t<float>(c, true, true);
}
int launch_fft_x_bwd_step(pll_context* c) {
  return c->prec == PLL_FP64 ? x_t<double>(c, false, true) : x_t<float>(c, false, true);
}
int launch_fft_x_bwd(pll_context* c) { return c->prec == PLL_FP64 ? x_t<double>(c, false) : x_t<float>(c, false); }
int launch_fft_y_fwd(pll_context* c) { return c->prec == PLL_FP64 ? y_t<double>(c, true) : y_t<float>(c, true); }
int launch_fft_y_bwd(pll_context* c) { return c->prec == PLL_FP64 ? y_t<double>(c, false) : y_t<float>(c, false); }

int launch_poisson_step(pll_context* c, bool rhs) {
  int rc;
  if (rhs && c->plane_threads) {
    const bool f64 = c->prec == PLL_FP64;
    if ((rc = f64 ? plane_t<double>(c, true) : plane_t<float>(c, true))) return rc;
    if ((rc = launch_trid_step(c))) return rc;
    return f64 ? plane_t<double>(c, false) : plane_t<float>(c, false);
  }
  if ((rc = rhs ? launch_fft_x_fwd_rhs(c) : launch_fft_x_fwd(c))) return rc;
  if ((rc = launch_fft_y_fwd(c))) return rc;
  if ((rc = launch_trid_step(c))) return rc;
  if ((rc = launch_fft_y_bwd(c))) return rc;
  return launch_fft_x_bwd_step(c);
}

}  // namespace pll
