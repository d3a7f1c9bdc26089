// k_trid.hip -- the wall-normal tridiagonal solve of the pressure Poisson
// equation for every (kx, ky) mode (ssolve_trid, src/mod_poisson_solver.cc:317-357).
//
// The reference stores the forward-eliminated pivots as a full nx*ny*nz
// array (src/mod_poisson_solver.cc:255-282).  The pivots of a column depend
// only on its eigenvalue lambda_x(i) + lambda_y(j), and the perm packing gives
// the real and imaginary parts of a mode the same eigenvalue, so four columns
// share each pivot column.  The table here keeps one pivot column per
// distinct pair: (nx/2+1)*(ny/2+1)*nz values, built on the host with the
// reference's arithmetic, so every pivot is bit-identical to the reference's.
//
// One thread per (i,j) column, coalesced over i, sequential in k; many
// columns per CU hide the latency of the dependent sweeps.  (Staging whole
// columns in LDS saves the second pass over the work array but leaves a CU
// only ~50 FP64 columns of 384 planes: the sweeps then run latency-bound,
// 3x slower at 768x384x384.)  The arithmetic is FP64 in both precision modes
// (the FP32-mixed path stores the work array in FP32 but eliminates in FP64,
// which covers the kx=ky=0 and the near-singular low-wavenumber columns).
// FP64 keeps the reference's divisions (bit-exact); FP32-mixed stores
// reciprocal pivots and multiplies (RECIP).
#include "pll_internal.hpp"

#include <cmath>
#include <type_traits>

namespace pll {

namespace {

constexpr int kTx = 64;
constexpr int kTy = 4;

// perm index -> compact eigenvalue index: 0 -> 0, 1 -> 1 (Nyquist), 2m/2m+1 -> m+1.
__host__ __device__ __forceinline__ int compact_index(int i) { return i <= 1 ? i : (i >> 1) + 1; }

// Loads are issued a chunk of D planes ahead of the sequential recurrence, so
// each sweep waits on HBM latency once per D planes rather than once per plane.
constexpr int kD = 8;

template <typename T, bool RECIP>
__global__ __launch_bounds__(kTx* kTy) void k_trid(int nx, int ny, int nz, T* __restrict__ var,
                                                   const double* __restrict__ a,
                                                   const double* __restrict__ c,
                                                   const double* __restrict__ piv, int cxn,
                                                   int cyn) {
  const int i = blockIdx.x * kTx + threadIdx.x;
  const int j = blockIdx.y * kTy + threadIdx.y;
  if (i >= nx || j >= ny) return;
  const long nxy = (long)nx * ny;
  const long P = (long)cxn * cyn;
  // plane bases are uniform across the block; each lane keeps one 32-bit offset
  const int off = j * nx + i;
  const int poff = compact_index(j) * cxn + compact_index(i);
  auto V = [&](int k) -> T& { return (var + (long)k * nxy)[off]; };
  auto B = [&](int k) -> double { return (piv + (long)k * P)[poff]; };

  // forward elimination, src/mod_poisson_solver.cc:334-339:
  // var[k] -= (a[k] / b[k-1]) * var[k-1], k = 1..nz-1
  double prev = (double)V(0);
  T xv[2][kD];
  double xb[2][kD];
  auto load_fwd = [&](int buf, int kb) {
#pragma unroll
    for (int d = 0; d < kD; ++d) {
      const int k = kb + d;
      if (k < nz) {
        xv[buf][d] = V(k);
        xb[buf][d] = B(k - 1);
      }
    }
  };
  auto run_fwd = [&](int buf, int kb) {
#pragma unroll
    for (int d = 0; d < kD; ++d) {
      const int k = kb + d;
      if (k < nz) {
        const double a_tmp = RECIP ? a[k] * xb[buf][d] : a[k] / xb[buf][d];
        const double cur = (double)xv[buf][d] - a_tmp * prev;
        V(k) = (T)cur;
        prev = cur;
      }
    }
  };
  load_fwd(0, 1);
  for (int kb = 1; kb < nz; kb += 2 * kD) {
    if (kb + kD < nz) load_fwd(1, kb + kD);
    run_fwd(0, kb);
    if (kb + 2 * kD < nz) load_fwd(0, kb + 2 * kD);
    if (kb + kD < nz) run_fwd(1, kb + kD);
  }
  // last row, src/mod_poisson_solver.cc:341-346
  const double b_val = B(nz - 1);
  if (RECIP)
    prev = prev * b_val;  // the reciprocal table holds 0 for a zero pivot
  else
    prev = (b_val != 0) ? prev / b_val : 0.0;
  V(nz - 1) = (T)prev;
  // back substitution, src/mod_poisson_solver.cc:348-354:
  // var[k] = (var[k] - c[k] * var[k+1]) / b[k], k = nz-2..0
  auto load_bwd = [&](int buf, int kt) {
#pragma unroll
    for (int d = 0; d < kD; ++d) {
      const int k = kt - d;
      if (k >= 0) {
        xv[buf][d] = V(k);
        xb[buf][d] = B(k);
      }
    }
  };
  auto run_bwd = [&](int buf, int kt) {
#pragma unroll
    for (int d = 0; d < kD; ++d) {
      const int k = kt - d;
      if (k >= 0) {
        const double r = (double)xv[buf][d] - c[k] * prev;
        const double cur = RECIP ? r * xb[buf][d] : r / xb[buf][d];
        V(k) = (T)cur;
        prev = cur;
      }
    }
  };
  load_bwd(0, nz - 2);
  for (int kt = nz - 2; kt >= 0; kt -= 2 * kD) {
    if (kt - kD >= 0) load_bwd(1, kt - kD);
    run_bwd(0, kt);
    if (kt - 2 * kD >= 0) load_bwd(0, kt - 2 * kD);
    if (kt - kD >= 0) run_bwd(1, kt - kD);
  }
}


// ---------------------------------------------------------------------------
// The same solve inside the step, partitioned so that the work array makes one
// HBM pass each way.  The columns (2m, 2m+1) x (2n, 2n+1) of the perm packing
// share one eigenvalue (m, n >= 1; columns and rows 0 and 1 are classes of their
// own), so a thread owns a whole eigenvalue class, up to four columns: the
// pivots, the multipliers and the coefficients' LDS reads are formed once for
// all four, the four recurrences overlap, and loads are pairs.  A class's columns
// are cut into S segments of M planes, one thread per segment, and the segment's
// values and reciprocal pivots stay in registers.  The pivots are not read from
// a table: each segment continues the elimination's pivot recurrence
// (init_poisson_solver, src/mod_poisson_solver.cc:273-282) from the pivot of the
// plane below it, which the table `pstart` holds, with the reference's
// operations (FP64 division), so every pivot is the one the full table holds,
// bit for bit; the reciprocal is 0 for a zero pivot:
//   A. forward elimination of the segment from a zero incoming value, with the
//      running product g of the negated multipliers (the segment end's
//      dependence on the incoming value);
//   exchange: the true segment-end values, sequentially over the S segments
//      (Y_s = yhat_s + g_s * Y_{s-1}), through LDS;
//   B. the forward elimination again from the true incoming value (the last
//      row divided by its pivot, src/mod_poisson_solver.cc:341-346);
//   C, exchange, D: the same for the back substitution (:348-354) from the top.
// The segment boundaries are combined with other roundings than the
// sequential sweep, and the pivots are applied as reciprocals, so the result
// differs from k_trid's by FP64 round-off (it is not bit-identical).
// FP32-mixed runs the recurrence without divisions: the multiplier is a[k] times
// the reciprocal of the pivot below (already formed), and the reciprocal is the
// hardware estimate refined by one Newton step (which squares its relative
// error: far below the 6e-8 rounding of the FP32 work array).
// One thread per column was bound by the pivots' arithmetic and the coefficients'
// LDS reads (FP32 2.0 TB/s).  One per class: FP32 1536x768x512 2377 -> 1420 us,
// 768x384x384 316 -> 249, 384x256x192 79 -> 53; FP64 768x384x384 474 -> 413,
// 256x192x128 34 -> 23 us.
__device__ __forceinline__ double rcp_newton(double q) {
  const double r = __builtin_amdgcn_rcp(q);
  return __builtin_fma(r, __builtin_fma(-q, r, 1.0), r);
}
constexpr int kSegPlanes = 768;  // the deepest column the segments hold
// Planes per segment M and most segments per column S.  Short segments keep the
// registers (4 M values, M+1 reciprocals) at four waves per SIMD; M = 12 where
// M = 8 would make blocks that leave a CU's wave slots idle (768x384x384: FP64 413
// against 464 us, FP32 249 against 299 us).  M = 12 takes 168 registers in FP64
// (three waves) and 134 in FP32, which is held to four waves all the same: 8
// registers spill, but two blocks of 512 threads fit a CU instead of one
// (768x384x384, 10 steps 25.3 against 25.6 ms).
constexpr int seg_planes(int nz) { return nz <= 256 || (nz > 384 && nz <= 512) ? 8 : 12; }
constexpr int seg_count_max(int nz) { return nz <= 128 ? 16 : (nz <= 384 ? 32 : 64); }
constexpr bool segs_hold(int nz) { return seg_planes(nz) * seg_count_max(nz) >= nz; }
static_assert(segs_hold(128) && segs_hold(256) && segs_hold(384) && segs_hold(512) &&
                  segs_hold(kSegPlanes),
              "the segments hold every column they take");
// Classes per block: 128 bytes of a row, or half that in FP32 columns of more than
// 32 segments (512 threads a block).
template <typename T, int S>
constexpr int seg_classes() {
  return std::is_same<T, float>::value && S <= 32 ? 16 : 8;
}

// The sequential combination of the segment-end values in place, Y_q = end_q +
// dep_q * Y_{q-1} (forward) or from the top (REV), by one thread per column
// (column t = component * CW + class); the LDS reads are issued four at a time
// ahead of the dependent chain.
template <int CW, int S, bool REV>
__device__ __forceinline__ void combine(double (*end)[4 * CW], const double (*dep)[CW], int nseg,
                                        int t) {
  double y = 0.0;
  for (int q0 = 0; q0 < nseg; q0 += 4) {
    double h[4], d[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int q = REV ? nseg - 1 - (q0 + u) : q0 + u;
      if (q0 + u < nseg) {
        h[u] = end[q][t];
        d[u] = dep[q][t % CW];
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int q = REV ? nseg - 1 - (q0 + u) : q0 + u;
      if (q0 + u < nseg) {
        y = __builtin_fma(d[u], y, h[u]);
        end[q][t] = y;
      }
    }
  }
}

// SegCoef: the diagonal before the eigenvalue b (nz), the compact eigenvalues
// of x (cxn) and y (cyn), and the pivots of the planes below the segments,
// pstart[s * cxn * cyn + cy * cxn + cx] = pivot of plane s*M - 1 (s >= 1).
struct SegCoef {
  const double* b;
  const double* elx;
  const double* ely;
  const double* pstart;
  int pin;  // the (0,0) column's last pivot is pinned to 0
};

// Hides where a register's value came from.
template <typename V>
__device__ __forceinline__ void pin(V& v) {
  asm volatile("" : "+v"(v));
}

// Blocks: tiles of CW column pairs for each row pair (pair 0 standing for the
// classes 0), then the same tiles of row 1, then tiles of CW row classes of
// column 1.
template <int CW>
__host__ __device__ constexpr unsigned seg_blocks(int nx, int ny) {
  return (unsigned)((nx / 2 + CW - 1) / CW) * (ny / 2 + 1) + (ny / 2 + CW) / CW;
}

template <typename T, int M, int CW, int S>
__global__ __launch_bounds__(CW* S, (sizeof(T) == 8 && M > 8 ? 3 : 4)) void k_trid_seg(int nx, int ny, int nz, int nseg,
                                                    T* __restrict__ var,
                                                    const double* __restrict__ a,
                                                    const double* __restrict__ c, SegCoef sg,
                                                    int cxn, int cyn) {
  struct alignas(2 * sizeof(T)) Pair {
    T x, y;
  };
  __shared__ double end[S][4 * CW];  // segment-end values: from a zero incoming value, then true
  __shared__ double dep[S][CW];      // their dependence on the incoming value
  __shared__ double sa[M * S], sb[M * S], sc[M * S];
  const int t = threadIdx.x, cl = t % CW, s = t / CW;
  for (int k = t; k < nseg * M; k += CW * nseg) {  // zero past the last plane
    sa[k] = k < nz ? a[k] : 0.0;
    sb[k] = k < nz ? sg.b[k] : 0.0;
    sc[k] = k < nz ? c[k] : 0.0;
  }
  // the thread's class (ci, cj) and its columns, i0 and i0+1 of rows j0 and
  // j0+1, of which it keeps those in `keep` (bit 2 dy + dx).  The others, of a
  // column or row 0 or 1, are another thread's: they are loaded, perhaps while
  // that thread stores them, and what becomes of them is not used.
  const int nxp = nx / 2, nyp = ny / 2, tpr = (nxp + CW - 1) / CW;
  const int b = (int)xcd_remap(blockIdx.x, gridDim.x);
  const bool col1 = b >= tpr * (nyp + 1);
  const int e = (b - tpr * (nyp + 1)) * CW + cl;
  const int xp = col1 ? 0 : (b % tpr) * CW + cl, yp = col1 ? e : b / tpr;
  const bool on = xp < nxp && yp <= nyp;
  const int i0 = 2 * xp, j0 = yp < nyp ? 2 * yp : 0;
  const int ci = col1 ? 1 : compact_index(on ? i0 : 0);
  const int cj = on ? (yp < nyp ? compact_index(j0) : 1) : 0;
  const int keep = ((col1 ? 2 : (xp ? 3 : 1)) & 3) * (yp == nyp ? 4 : (yp ? 5 : 1));
  const long nxy = (long)nx * ny;
  const int k0 = s * M;
  const int n = on ? min(M, nz - k0) : 0, last = nz - 1 - k0;  // planes; the last row
  long off = (long)k0 * nxy + (on ? (long)j0 * nx + i0 : 0);
  // the segment's values (in the field precision: FP32-mixed rounds the
  // forward-eliminated values to FP32 between the sweeps, as k_trid does),
  // loaded first; 0 past the last plane
  T x[4][M];
  {
    const T* q = var + off;
#pragma unroll
    for (int m = 0; m < M; ++m, q += nxy) {
      Pair r0{T(0), T(0)}, r1{T(0), T(0)};
      if (m < n) {
        r0 = *reinterpret_cast<const Pair*>(q);
        r1 = *reinterpret_cast<const Pair*>(q + nx);
      }
      x[0][m] = r0.x;
      x[1][m] = r0.y;
      x[2][m] = r1.x;
      x[3][m] = r1.y;
    }
  }
  const double lxy = sg.elx[ci] + sg.ely[cj];
  double piv = k0 > 0 && n > 0 ? sg.pstart[(long)s * cxn * cyn + (long)cj * cxn + ci] : 1.0;
  double rb[M + 1];  // reciprocal pivots of planes k0-1 .. k0+M-1, 0 where there is no plane
  rb[0] = k0 > 0 && piv != 0.0 ? 1.0 / piv : 0.0;
  __syncthreads();  // sa, sb, sc
  // init_poisson_solver's recurrence (src/mod_poisson_solver.cc:273-282): a[0]
  // is 0, and a zero pivot only ends a column
  constexpr bool kMixed = std::is_same<T, float>::value;
  // the coefficients are read kAhead planes at a time, not all ahead
  constexpr int kAhead = 4;
  const auto step_fence = [] { __builtin_amdgcn_sched_barrier(0); };
  const int pinned = sg.pin && ci == 0 && cj == 0 ? last + 1 : 0;
#pragma unroll
  for (int m = 1; m <= M; ++m) {
    if (m % kAhead == 1) step_fence();
    const int k = k0 + m - 1;
    const double a_tmp = kMixed ? sa[k] * rb[m - 1] : sa[k] / piv;
    double q = sb[k] + lxy;
    q -= (a_tmp * sc[m > 1 ? k - 1 : max(k - 1, 0)]);
    if (m == pinned) q = 0.0;
    rb[m] = m <= n && q != 0.0 ? (kMixed ? rcp_newton(q) : 1.0 / q) : 0.0;
    piv = q;
  }
  // past the last plane the values, multipliers and reciprocals are 0, and a[0]
  // and c[nz-1] are 0: the sweeps need no test for a column's ends
  // between the sweeps the values stay in the field precision, not as the
  // doubles that the last sweep made of them
  const auto pin_values = [&] {
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int m = 0; m < M; ++m) pin(x[f][m]);
  };
  // A: forward elimination from a zero incoming value
  {
    double y[4] = {0.0, 0.0, 0.0, 0.0}, g = 1.0;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      if (m % kAhead == 0) step_fence();
      const double l = sa[k0 + m] * rb[m];
#pragma unroll
      for (int f = 0; f < 4; ++f) y[f] = __builtin_fma(-l, y[f], (double)x[f][m]);
      g = -l * g;
    }
#pragma unroll
    for (int f = 0; f < 4; ++f) end[s][f * CW + cl] = y[f];
    dep[s][cl] = g;
  }
  __syncthreads();
  if (t < 4 * CW) combine<CW, S, false>(end, dep, nseg, t);
  // few segments leave fewer threads than columns
  for (int u = t + CW * nseg; u < 4 * CW; u += CW * nseg) combine<CW, S, false>(end, dep, nseg, u);
  __syncthreads();
  pin_values();
  // B: forward elimination from the true incoming value; the last row
  {
    double y[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) y[f] = s > 0 ? end[s - 1][f * CW + cl] : 0.0;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      if (m % kAhead == 0) step_fence();
      const double l = sa[k0 + m] * rb[m];
#pragma unroll
      for (int f = 0; f < 4; ++f) y[f] = __builtin_fma(-l, y[f], (double)x[f][m]);
      if (m == last) {  // the reciprocal is 0 for a zero pivot
#pragma unroll
        for (int f = 0; f < 4; ++f) y[f] *= rb[m + 1];
        rb[m + 1] = 1.0;  // the back substitution takes the row as it is
      }
#pragma unroll
      for (int f = 0; f < 4; ++f) x[f][m] = (T)y[f];
    }
  }
  __syncthreads();  // end is rewritten below
  // C: back substitution from a zero value above the segment
  {
    double xv[4] = {0.0, 0.0, 0.0, 0.0}, h = 1.0;
#pragma unroll
    for (int m = M - 1; m >= 0; --m) {
      if (m % kAhead == kAhead - 1) step_fence();
      const double q = sc[k0 + m] * rb[m + 1];
#pragma unroll
      for (int f = 0; f < 4; ++f)
        xv[f] = __builtin_fma((double)x[f][m], rb[m + 1], -(q * xv[f]));
      h = -q * h;
    }
#pragma unroll
    for (int f = 0; f < 4; ++f) end[s][f * CW + cl] = xv[f];
    dep[s][cl] = h;
  }
  __syncthreads();
  if (t < 4 * CW) combine<CW, S, true>(end, dep, nseg, t);
  for (int u = t + CW * nseg; u < 4 * CW; u += CW * nseg) combine<CW, S, true>(end, dep, nseg, u);
  __syncthreads();
  pin_values();
  // D: back substitution from the true value above the segment
  {
    double xv[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) xv[f] = s + 1 < nseg ? end[s + 1][f * CW + cl] : 0.0;
#pragma unroll
    for (int m = M - 1; m >= 0; --m) {
      if (m % kAhead == kAhead - 1) step_fence();
      const double q = sc[k0 + m] * rb[m + 1];
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        xv[f] = __builtin_fma((double)x[f][m], rb[m + 1], -(q * xv[f]));
        x[f][m] = (T)xv[f];
      }
    }
  }
  pin(off);  // the addresses are formed again rather than kept from the loads
  T* q = var + off;
  if (keep == 15) {
#pragma unroll
    for (int m = 0; m < M; ++m, q += nxy)
      if (m < n) {
        *reinterpret_cast<Pair*>(q) = Pair{x[0][m], x[1][m]};
        *reinterpret_cast<Pair*>(q + nx) = Pair{x[2][m], x[3][m]};
      }
  } else {
#pragma unroll
    for (int m = 0; m < M; ++m, q += nxy)
      if (m < n) {
        if (keep & 1) q[0] = x[0][m];
        if (keep & 2) q[1] = x[1][m];
        if (keep & 4) q[nx] = x[2][m];
        if (keep & 8) q[nx + 1] = x[3][m];
      }
  }
}

}  // namespace

// init_poisson_solver's eigenvalue, coefficient and pivot set-up
// (src/mod_poisson_solver.cc:230-282, src/mod_fft.cc:196-222) at one GPU,
// boundary types "PP","PP","NN" (src/main.cc:55-57).
int trid_setup(pll_context* c) {
  const int nx = c->g.nx, ny = c->g.ny, nz = c->g.nz;
  std::vector<double> lx(nx), ly(ny);
  pll_eigen_values(nx, lx.data());
  for (int i = 0; i < nx; ++i) lx[i] /= (c->dx * c->dx);
  pll_eigen_values(ny, ly.data());
  for (int j = 0; j < ny; ++j) ly[j] /= (c->dy * c->dy);

  // set_trid_coeff('c', "NN") with dzf0[k] = dzf_global(k), k = 0..nz+1
  // (src/mod_poisson_solver.cc:35-98,258-264)
  const double* dzf0 = c->dzf_global.data();
  std::vector<double> a(nz), b(nz), cc(nz);
  for (int k = 0; k < nz; ++k) {
    a[k] = 2.0 / (dzf0[k + 1] * (dzf0[k] + dzf0[k + 1]));
    cc[k] = 2.0 / (dzf0[k + 1] * (dzf0[k + 2] + dzf0[k + 1]));
  }
  for (int k = 0; k < nz; ++k) b[k] = -a[k] - cc[k];
  const double factor = 1.0;  // 'N'
  b[0] += factor * a[0];
  a[0] *= std::fabs(factor) - 1.0;
  b[nz - 1] += factor * cc[nz - 1];
  cc[nz - 1] *= std::fabs(factor) - 1.0;

  c->cxn = nx / 2 + 1;
  c->cyn = ny / 2 + 1;
  const long P = (long)c->cxn * c->cyn;
  std::vector<double> piv((size_t)P * nz);
  auto rep = [](int ci) { return ci <= 1 ? ci : 2 * (ci - 1); };  // a perm index of that class
  for (int cy = 0; cy < c->cyn; ++cy)
    for (int cx = 0; cx < c->cxn; ++cx) {
      const double lxy = lx[rep(cx)] + ly[rep(cy)];
      double* col = piv.data() + (long)cy * c->cxn + cx;
      for (int k = 0; k < nz; ++k) col[k * P] = b[k] + lxy;
      for (int k = 1; k < nz; ++k) {
        const double a_tmp = a[k] / col[(k - 1) * P];
        col[k * P] -= (a_tmp * cc[k - 1]);
      }
    }
  // FP32-mixed always pins: the reference's round-off pivot would divide the
  // FP32 round-off of the mean right-hand side into a constant of ~1e6 in p,
  // which an FP32 p cannot carry next to O(1) pressure differences
  if (c->cfg.pin_singular || c->prec != PLL_FP64) piv[(size_t)(nz - 1) * P] = 0.0;
  // the partitioned solve of the step: b, the compact eigenvalues and the
  // pivots of the planes below its segments (it rebuilds the others)
  std::vector<double> seg;
  if (nz <= kSegPlanes) {
    const int M = seg_planes(nz), nseg = (nz + M - 1) / M;
    seg.assign(nz + c->cxn + c->cyn + (size_t)nseg * P, 0.0);
    for (int k = 0; k < nz; ++k) seg[k] = b[k];
    for (int cx = 0; cx < c->cxn; ++cx) seg[nz + cx] = lx[rep(cx)];
    for (int cy = 0; cy < c->cyn; ++cy) seg[nz + c->cxn + cy] = ly[rep(cy)];
    double* ps = seg.data() + nz + c->cxn + c->cyn;
    for (int s = 1; s < nseg; ++s)
      for (long q = 0; q < P; ++q) ps[s * P + q] = piv[(size_t)(s * M - 1) * P + q];
    c->seg_pin = (c->cfg.pin_singular || c->prec != PLL_FP64) ? 1 : 0;
  }
  // FP32-mixed multiplies by reciprocal pivots (0 stands for a zero pivot:
  // the reference's b == 0 branch gives 0, src/mod_poisson_solver.cc:341-346)
  if (c->prec != PLL_FP64)
    for (double& x : piv) x = x != 0.0 ? 1.0 / x : 0.0;

  PLL_HIP_TRY(ctx_malloc(c, &c->d_a, nz * sizeof(double)));
  PLL_HIP_TRY(ctx_malloc(c, &c->d_c, nz * sizeof(double)));
  PLL_HIP_TRY(ctx_malloc(c, &c->d_piv, piv.size() * sizeof(double)));
  PLL_HIP_TRY(hipMemcpy(c->d_a, a.data(), nz * sizeof(double), hipMemcpyHostToDevice));
  PLL_HIP_TRY(hipMemcpy(c->d_c, cc.data(), nz * sizeof(double), hipMemcpyHostToDevice));
  PLL_HIP_TRY(hipMemcpy(c->d_piv, piv.data(), piv.size() * sizeof(double), hipMemcpyHostToDevice));
  if (!seg.empty()) {
    PLL_HIP_TRY(ctx_malloc(c, &c->d_seg, seg.size() * sizeof(double)));
    PLL_HIP_TRY(hipMemcpy(c->d_seg, seg.data(), seg.size() * sizeof(double), hipMemcpyHostToDevice));
  }
  return PLL_OK;
}

int launch_trid(pll_context* c) {
  TimerScope ts(c, K_TRID);
  const dim3 grid((c->g.nx + kTx - 1) / kTx, (c->g.ny + kTy - 1) / kTy);
  if (c->prec == PLL_FP64)
    hipLaunchKernelGGL((k_trid<double, false>), grid, dim3(kTx, kTy), 0, c->stream, c->g.nx,
                       c->g.ny, c->g.nz, static_cast<double*>(c->spec), c->d_a, c->d_c, c->d_piv,
                       c->cxn, c->cyn);
  else
    hipLaunchKernelGGL((k_trid<float, true>), grid, dim3(kTx, kTy), 0, c->stream, c->g.nx,
                       c->g.ny, c->g.nz, static_cast<float*>(c->spec), c->d_a, c->d_c, c->d_piv,
                       c->cxn, c->cyn);
  PLL_HIP_TRY(hipGetLastError());
  return PLL_OK;
}

namespace {
template <typename T, int M, int S>
void trid_seg(pll_context* c) {
  constexpr int kCw = seg_classes<T, S>();
  const int nz = c->g.nz, nseg = (nz + M - 1) / M;
  const SegCoef sg{c->d_seg, c->d_seg + nz, c->d_seg + nz + c->cxn,
                   c->d_seg + nz + c->cxn + c->cyn, c->seg_pin};
  hipLaunchKernelGGL((k_trid_seg<T, M, kCw, S>), dim3(seg_blocks<kCw>(c->g.nx, c->g.ny)),
                     dim3(kCw * nseg), 0, c->stream, c->g.nx, c->g.ny, nz, nseg,
                     static_cast<T*>(c->spec), c->d_a, c->d_c, sg, c->cxn, c->cyn);
}
template <typename T>
void trid_seg_t(pll_context* c) {
  static_assert(seg_planes(256) == 8 && seg_planes(384) == 12 && seg_planes(512) == 8 &&
                    seg_planes(kSegPlanes) == 12,
                "the instances below");
  const int nz = c->g.nz;
  if (nz <= 128)
    trid_seg<T, 8, 16>(c);
  else if (nz <= 256)
    trid_seg<T, 8, 32>(c);
  else if (nz <= 384)
    trid_seg<T, 12, 32>(c);
  else if (nz <= 512)
    trid_seg<T, 8, 64>(c);
  else
    trid_seg<T, 12, 64>(c);
}
}  // namespace

int launch_trid_step(pll_context* c) {
  // columns deeper than the segments hold take the sequential kernel (2533 against
  // 1420 us in FP32-mixed at 1536x768x512)
  if (!c->d_seg || c->g.nz > kSegPlanes) return launch_trid(c);
  TimerScope ts(c, K_TRID);
  if (c->prec == PLL_FP64)
    trid_seg_t<double>(c);
  else
    trid_seg_t<float>(c);
  PLL_HIP_TRY(hipGetLastError());
  return PLL_OK;
}

}  // namespace pll
