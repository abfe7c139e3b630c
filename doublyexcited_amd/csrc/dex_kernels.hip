// HIP kernels for gfx950 (MI355X): the two-electron sinc-DVR matvec and the
// tall-skinny block kernels of the GPLMR eigensolver.
//
// Matvec.  A two-electron vector is the M x M matrix X[p + M q] (p: electron 1,
// q: electron 2, each p = i + NN j + NN^2 k).  With T = tau / delta^2 the real
// Toeplitz sinc-DVR matrix (tau(0) = pi^2/6, tau(m) = (-1)^m / m^2) the
// reference's HAMMULT (hammod.F90:19-67) is
//     Y = e^{-2 i theta} (T3D x I + I x T3D) X + e^{-i theta} Vr o X,
// Vr(p, q) = -Z/delta^3 (Tinv(r_p) + Tinv(r_q)) + Tinv(r_q - r_p)/delta^3.
// tau is a compile-time table, so the kinetic contraction is a stream of
// FMAs with scalar constants.  Two passes:
//   pass 1 (electron 1): Z[:, q] = s2 tau3D X[:, q] + w c1 Vr X[:, q]  (contiguous
//     cubes in LDS),
//   exchange-(anti)symmetric vectors (w = 1/2): Y = Z + sign Z^T, in place,
//   general ones (w = 1): Y[p, :] = Z[p, :] + s2 tau3D X[p, :]  (cubes at stride
//     M) on the smallest grids; on the others three passes of two axes each
//     (k_plane1, k_plane2) replace both.
// The kinetic operator is real, so the real and imaginary parts are contracted
// in turn through two LDS buffers of NN^3 reals each (148 KB at NN = 21 in FP64).
#include <atomic>
#include <cstdlib>
#include <mutex>

#include <hip/hip_runtime.h>

#include "dex_internal.h"

namespace dex {

namespace {

constexpr double kPi2over6 = 1.6449340668482264;  // pi^2 / 6

template <int M>
__device__ __forceinline__ constexpr double tau_c() {
  if constexpr (M == 0) {
    return kPi2over6;
  } else {
    return ((M & 1) ? -1.0 : 1.0) / double(M * M);
  }
}

__device__ __forceinline__ constexpr double tau_rt(int m) {
  m = m < 0 ? -m : m;
  return m == 0 ? kPi2over6 : ((m & 1) ? -1.0 : 1.0) / double(m * m);
}

template <typename R>
struct Cplx;
template <>
struct Cplx<double> {
  using type = double2;
};
template <>
struct Cplx<float> {
  using type = float2;
};

template <typename T>
struct Real;
template <>
struct Real<double2> {
  using type = double;
};
template <>
struct Real<float2> {
  using type = float;
};

constexpr int round_up(int a, int b) { return (a + b - 1) / b * b; }

template <int NN>
constexpr int cube_threads() {
  return round_up(NN * NN, 64) > 1024 ? 1024 : round_up(NN * NN, 64);
}

// emit(i, y_i) for y = tau x along one axis of NN = 2 H + 1 points.  tau is a
// symmetric Toeplitz matrix, so it maps the even and the odd part of a line (about
// its centre) to themselves: with s_m = x_{H+m} + x_{H-m} and d_m = x_{H+m} - x_{H-m},
//   y_{H+-n} = tau(n) x_H + sum_m (tau(n-m) + tau(n+m)) s_m / 2
//              +- sum_m (tau(n-m) - tau(n+m)) d_m / 2,
// (H + 1)^2 + H^2 multiply-adds and 4 H additions a line in place of NN^2
// multiply-adds (221 + 40 for 441 at NN = 21), with compile-time coefficients.
template <int NN, typename R, typename F>
__device__ __forceinline__ void line_apply(const R (&x)[NN], F &&emit) {
  constexpr int H = NN / 2;
  R s[H + 1], d[H + 1];
#pragma unroll
  for (int m = 1; m <= H; ++m) {
    s[m] = x[H + m] + x[H - m];
    d[m] = x[H + m] - x[H - m];
  }
  R y0 = R(tau_rt(0)) * x[H];
#pragma unroll
  for (int m = 1; m <= H; ++m) y0 += R(tau_rt(m)) * s[m];
  emit(H, y0);
#pragma unroll
  for (int n = 1; n <= H; ++n) {
    R e = R(tau_rt(n)) * x[H], o = R((tau_rt(n - 1) - tau_rt(n + 1)) / 2) * d[1];
#pragma unroll
    for (int m = 1; m <= H; ++m) {
      e += R((tau_rt(n - m) + tau_rt(n + m)) / 2) * s[m];
      if (m > 1) o += R((tau_rt(n - m) - tau_rt(n + m)) / 2) * d[m];
    }
    emit(H + n, e + o);
    emit(H - n, e - o);
  }
}

// The i and j axes of tau3D on one NN^3 cube of reals, one thread per line:
// thread c < NN^2 holds the k line through (i, j), c = i + NN j, in x (the order
// of the global loads, so the k axis costs no LDS access).  a is the cube; b
// collects the two axes' sums, which thread c then finds at b[c + NN^2 k].
template <int NN, typename R>
__device__ __forceinline__ void plane_axes(const R (&x)[NN], R *__restrict__ a, R *__restrict__ b, int c) {
  constexpr int N2 = NN * NN;
  const bool on = c < N2;
  if (on) {
#pragma unroll
    for (int k = 0; k < NN; ++k) a[c + N2 * k] = x[k];
  }
  __syncthreads();
  if (on) {  // axis i: line (j, k) = c
    R v[NN];
#pragma unroll
    for (int l = 0; l < NN; ++l) v[l] = a[c * NN + l];
    line_apply<NN, R>(v, [&](int i, R y) { b[c * NN + i] = y; });
  }
  __syncthreads();
  if (on) {  // axis j: line (i, k)
    const int base = c % NN + N2 * (c / NN);
    R v[NN];
#pragma unroll
    for (int l = 0; l < NN; ++l) v[l] = a[base + NN * l];
    line_apply<NN, R>(v, [&](int j, R y) { b[base + NN * j] += y; });
  }
  __syncthreads();
}

// a b, rounded by itself: of the two products of a potential term the compiler would fuse
// one into the addition, which one depending on the code around it.  Neither form is the
// more accurate.  Rounded, so that results do not move with that choice: their last bits
// decide where a solve ends whose last pair has a rival at nearly the same distance from
// sigma (NN = 11, theta 0.31: levels at 0.806 and 0.823; of four starts, two end warm and
// cold solves apart).
template <typename R>
__device__ __forceinline__ R rounded_product(R a, R b) {
#pragma clang fp contract(off)
  return a * b;
}

// Electron-1 pass on the cube of electron-2 index q = blockIdx.x (contiguous) of
// column blockIdx.y: Z = s2 tau3D X + w (c1 Vr - shift) o X.  w = 1/2 for
// exchange-(anti)symmetric vectors (Y = Z + sign Z^T follows, k_symfold), 1 for
// general ones (Y = Z + s2 K2 X follows, k_pass2).  A workgroup reads its whole
// cube before it writes, so Z may be X's own storage.
//
// One workgroup a cube: the LDS cube and the registers of three lines leave one
// workgroup (7 waves) on a CU at NN = 21 in FP64, two in FP32, and a new workgroup's
// loads need not wait for the last one's stores, as they do in a loop over cubes
// (a wave's memory operations complete in order).  The loop also let the compiler
// keep vn in registers, which cost the second workgroup: FP32 at NN = 19 ran 277 us
// a column looped and 175 us not, at NN = 21 487 and 354.
//
// SHIFT: H - shift (FP64 forms), each product of the potential term less that of the
// shift.  A variant of its own: with a zero shift the plain matvec took 1-2% more (one
// column at NN = 25 6.96 for 6.85 ms).
template <int NN, typename R, typename XT, typename ZT, bool SHIFT>
__global__ __launch_bounds__(cube_threads<NN>()) void k_pass1(ColPtrs xs, ColPtrsW zs, const double *__restrict__ vn,
                                                              const double *__restrict__ tinv, MatvecCoef cf,
                                                              double w) {
  constexpr int N2 = NN * NN;
  constexpr int N3 = NN * N2;
  constexpr int L = 2 * NN + 1;
  extern __shared__ __align__(16) unsigned char smem[];
  R *a = reinterpret_cast<R *>(smem);
  R *b = a + N3;
  const int c = threadIdx.x;
  const bool on = c < N2;
  const int q = blockIdx.x;
  const XT *xq = static_cast<const XT *>(xs.p[blockIdx.y]) + int64_t(q) * N3;
  R xr[NN], xi[NN], kr[NN];
  if (on) {
#pragma unroll
    for (int k = 0; k < NN; ++k) {
      const XT v = xq[c + N2 * k];
      xr[k] = R(v.x);
      xi[k] = R(v.y);
    }
  }
  plane_axes<NN, R>(xr, a, b, c);
  if (on) line_apply<NN, R>(xr, [&](int k, R y) { kr[k] = y + b[c + N2 * k]; });
  plane_axes<NN, R>(xi, a, b, c);
  if (on) {
    const R s2r = R(cf.s2_re), s2i = R(cf.s2_im), c1r = R(w * cf.c1_re), c1i = R(w * cf.c1_im);
    const R shr = R(w * cf.sh_re), shi = R(w * cf.sh_im);
    const int iq = q % NN, jq = (q / NN) % NN, kq = q / N2;
    const int t0 = (iq - c % NN + NN) + L * ((jq - c / NN + NN) + L * (kq + NN));
    const double vq = vn[q];
    ZT *zq = static_cast<ZT *>(zs.p[blockIdx.y]) + int64_t(q) * N3;
    line_apply<NN, R>(xi, [&](int k, R y) {
      const R ki = y + b[c + N2 * k];
      const R vr = R(vn[c + N2 * k] + vq + tinv[t0 - L * L * k] * cf.inv_d3);
      const R vxr = vr * xr[k], vxi = vr * xi[k];
      ZT o;
      if constexpr (SHIFT) {
        o.x = s2r * kr[k] - s2i * ki + (c1r * vxr - shr * xr[k]) - (c1i * vxi - shi * xi[k]);
        o.y = s2r * ki + s2i * kr[k] + (c1r * vxi - shr * xi[k]) + (c1i * vxr - shi * xr[k]);
      } else {
        o.x = s2r * kr[k] - s2i * ki + rounded_product(c1r, vxr) - rounded_product(c1i, vxi);
        o.y = s2r * ki + s2i * kr[k] + rounded_product(c1r, vxi) + rounded_product(c1i, vxr);
      }
      zq[c + N2 * k] = o;
    });
  }
}

// Workgroup -> electron-1 index p for pass 2: consecutive workgroups are
// dealt round-robin to the 8 XCDs, so the s-th workgroup on XCD x takes
// p = 8 (x + 8 (s / 8)) + s % 8, which puts 8 consecutive p (one 128-byte
// line of complex doubles per q) on the same XCD at nearly the same time.
__device__ __forceinline__ int64_t xcd_group_map(int64_t b, int64_t m) {
  const int64_t full = (m / 64) * 64;
  if (b >= full) return b;
  const int64_t x = b % 8, s = b / 8;
  return 8 * (x + 8 * (s / 8)) + (s % 8);
}

// Electron-2 pass for general vectors: Y = Z + s2 tau3D X on the stride-M cube
// of each electron-1 index p of column blockIdx.y (columns M^2 entries apart; Z from
// k_pass1 with w = 1).  Y may be X's or Z's storage (so none is __restrict__): a thread
// reads each entry of Z before it writes that of Y, and the workgroup's entries of X
// before any.
template <int NN, typename R, typename XT, typename YT>
__global__ __launch_bounds__(cube_threads<NN>()) void k_pass2(const XT *x, const typename Cplx<R>::type *z, YT *y,
                                                              MatvecCoef cf) {
  using C = typename Cplx<R>::type;
  constexpr int N2 = NN * NN;
  constexpr int N3 = NN * N2;
  extern __shared__ __align__(16) unsigned char smem[];
  R *a = reinterpret_cast<R *>(smem);
  R *b = a + N3;
  const int c = threadIdx.x;
  const bool on = c < N2;
  const int64_t p = xcd_group_map(blockIdx.x, N3) + int64_t(N3) * N3 * blockIdx.y;
  const int64_t M = N3;
  R xr[NN], xi[NN], kr[NN];
  if (on) {
#pragma unroll
    for (int k = 0; k < NN; ++k) {
      const XT v = x[p + M * (c + N2 * k)];
      xr[k] = R(v.x);
      xi[k] = R(v.y);
    }
  }
  plane_axes<NN, R>(xr, a, b, c);
  if (on) line_apply<NN, R>(xr, [&](int k, R y) { kr[k] = y + b[c + N2 * k]; });
  plane_axes<NN, R>(xi, a, b, c);
  if (on) {
    const R s2r = R(cf.s2_re), s2i = R(cf.s2_im);
    C zv[NN];  // ahead of the stores, behind which each load would wait in turn
#pragma unroll
    for (int k = 0; k < NN; ++k) zv[k] = z[p + M * (c + N2 * k)];
    line_apply<NN, R>(xi, [&](int k, R t) {
      const R ki = t + b[c + N2 * k];
      YT o;
      o.x = zv[k].x + (s2r * kr[k] - s2i * ki);
      o.y = zv[k].y + (s2r * ki + s2i * kr[k]);
      y[p + M * (c + N2 * k)] = o;
    });
  }
}

// ---- exchange-symmetric second pass ------------------------------------------
// For X = sign X^T (sign = +1 singlet, -1 triplet) electron 2's kinetic term is
// the transpose of electron 1's: (I x T3D) X = sign (T3D X)^T, and Vr = Vr^T.
// So after pass 1 (Z = s2 tau3D X + c1 Vr o X / 2, in Y's storage) the result is
// Y = Z + sign Z^T, in place: a workgroup owns the 32 x 32 tile (ta, tb),
// ta <= tb, and its mirror (tb, ta); all global accesses run along p (coalesced)
// and the transposes go through LDS.  Both members of a pair {(p, q), (q, p)} are
// the same two addends, so the output is exactly (anti)symmetric.
//
// M is odd, so a tile's 512-byte runs start at any multiple of 16 bytes and share
// their first and last 128-byte lines with the next tiles along p.  Tiles go to
// the XCDs (consecutive workgroups: round robin) in blocks of 4 x 4, so that most
// shared lines meet in one L2.  Bound by HBM (32 bytes an entry, 16 in complex64): 4.8
// TB/s at NN = 21 in FP64, 4.65 on complex64.  The form before, which read X and U = tau3D X
// and rebuilt the potential here, moved 48 bytes an entry (1.0 ms a vector at
// NN = 21 where this takes 0.58).
constexpr int kSymT = 32;
constexpr int kSymBlk = 4;

// Tile pair (ta, tb), ta <= tb, of this workgroup; false beyond the matrix.
__device__ __forceinline__ bool sym_tile(int m, int nblk, int &ta, int &tb) {
  const int xcd = blockIdx.x % 8, s = blockIdx.x / 8;
  const int blk = (s / (kSymBlk * kSymBlk)) * 8 + xcd, in = s % (kSymBlk * kSymBlk);
  // block (ba, bb), ba <= bb, from its index bb (bb + 1) / 2 + ba
  int bb = int((sqrtf(8.0f * float(blk) + 1.0f) - 1.0f) * 0.5f);
  while (bb * (bb + 1) / 2 > blk) --bb;
  while ((bb + 1) * (bb + 2) / 2 <= blk) ++bb;
  const int ba = blk - bb * (bb + 1) / 2;
  ta = ba * kSymBlk + in % kSymBlk;
  tb = bb * kSymBlk + in / kSymBlk;
  return bb < nblk && ta <= tb && tb * kSymT < m;
}

// Blocks along an axis, and workgroups of a launch over the tile pairs.
constexpr int sym_blocks(int m) { return ((m + kSymT - 1) / kSymT + kSymBlk - 1) / kSymBlk; }
constexpr int sym_grid(int m) { return round_up(sym_blocks(m) * (sym_blocks(m) + 1) / 2, 8) * kSymBlk * kSymBlk; }

template <typename T>
__global__ __launch_bounds__(256) void k_symfold(ColPtrsW ys, int m, int nblk, int sign) {
  using R = typename Real<T>::type;
  int ta, tb;
  if (!sym_tile(m, nblk, ta, tb)) return;
  T *__restrict__ y = static_cast<T *>(ys.p[blockIdx.y]);
  __shared__ T s1[kSymT][kSymT + 1], s2[kSymT][kSymT + 1];
  const int tx = threadIdx.x, ty = threadIdx.y;
  const int pa = ta * kSymT, qb = tb * kSymT;
  constexpr int PER = kSymT / 8;
  T v1[PER], v2[PER];
  const bool okp = pa + tx < m, okq = qb + tx < m, diag = ta == tb;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int r = ty + 8 * u;
    // main element (pa + tx, qb + r), mirror element (qb + tx, pa + r)
    if (okp && qb + r < m) v1[u] = y[pa + tx + int64_t(m) * (qb + r)];
    if (okq && pa + r < m) v2[u] = y[qb + tx + int64_t(m) * (pa + r)];
  }
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    s1[ty + 8 * u][tx] = v1[u];
    s2[ty + 8 * u][tx] = v2[u];
  }
  __syncthreads();
  const R sg = R(sign);
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int r = ty + 8 * u;
    const T m1 = s2[tx][r], m2 = s1[tx][r];
    T o1, o2;
    o1.x = v1[u].x + sg * m1.x;
    o1.y = v1[u].y + sg * m1.y;
    o2.x = v2[u].x + sg * m2.x;
    o2.y = v2[u].y + sg * m2.y;
    if (okp && qb + r < m) y[pa + tx + int64_t(m) * (qb + r)] = o1;
    if (!diag && okq && pa + r < m) y[qb + tx + int64_t(m) * (pa + r)] = o2;
  }
}

// ---- two axes at a time --------------------------------------------------------
// General vectors in three passes of two axes each, for grids whose cube does not
// fit the LDS (FP64 at NN >= 23) and for those where the stride-M cubes of k_pass2
// cost more than a third pass: every access runs along a contiguous direction.
// A workgroup holds NN x NN lines of kPlaneRun entries: each thread keeps one line
// of the first axis in registers (contracted there), the second axis goes through
// the LDS buffers a (entries) and b (its sums), one real component at a time.
// 32 + 48 + 48 bytes an entry over the three passes, 4.5 TB/s of them at NN = 25 in
// FP64 (k_plane1 4.0, k_plane2 4.7; 6.9 ms a vector where six passes of one axis and the
// potential's take 16.8), with
// 8 waves a CU in flight (two workgroups: 80 KB of LDS, 205-240 registers).
template <typename XT>
constexpr int plane_run() {
  return int(128 / sizeof(XT));  // entries of a 128-byte run
}
constexpr int kPlane1Planes = 8;  // i1 x j1 planes of a workgroup

// Axes i1 and j1 and the potential: Z = s2 (tau x 1 + 1 x tau) X + (c1 Vr - shift) o X.
// blockIdx: electron-2 index q, group of kPlane1Planes planes k1.  Thread (i, g) keeps the
// j line of plane g.
template <int NN, typename R, typename XT, typename ZT, bool SHIFT>
__global__ __launch_bounds__(round_up(NN *kPlane1Planes, 64)) void k_plane1(
    const XT *__restrict__ x, ZT *__restrict__ z, const double *__restrict__ vn, const double *__restrict__ tinv,
    MatvecCoef cf) {
  constexpr int N2 = NN * NN, N3 = NN * N2, L = 2 * NN + 1, G = kPlane1Planes;
  extern __shared__ __align__(16) unsigned char smem[];
  const int i = threadIdx.x % NN, g = threadIdx.x / NN, k = int(blockIdx.y) * G + g;
  const bool on = g < G && k < NN;
  R *a = reinterpret_cast<R *>(smem) + g * N2;
  R *b = a + G * N2;
  const int q = blockIdx.x;
  const int64_t base = int64_t(q) * N3 + N2 * k + i;
  R xr[NN], xi[NN], kr[NN];
  if (on) {
#pragma unroll
    for (int j = 0; j < NN; ++j) {
      const XT v = x[base + NN * j];
      xr[j] = R(v.x);
      xi[j] = R(v.y);
    }
  }
  // i lines of one component through LDS, thread (line j = i, plane g)
  auto i_axis = [&](const R(&v)[NN]) {
    if (on) {
#pragma unroll
      for (int j = 0; j < NN; ++j) a[NN * j + i] = v[j];
    }
    __syncthreads();
    if (on) {
      R t[NN];
#pragma unroll
      for (int l = 0; l < NN; ++l) t[l] = a[NN * i + l];
      line_apply<NN, R>(t, [&](int l, R y) { b[NN * i + l] = y; });
    }
    __syncthreads();
  };
  i_axis(xr);
  if (on) line_apply<NN, R>(xr, [&](int j, R y) { kr[j] = y + b[NN * j + i]; });
  i_axis(xi);
  if (on) {
    const R s2r = R(cf.s2_re), s2i = R(cf.s2_im), c1r = R(cf.c1_re), c1i = R(cf.c1_im);
    const R shr = R(cf.sh_re), shi = R(cf.sh_im);
    const int iq = q % NN, jq = (q / NN) % NN, kq = q / N2;
    const int t0 = (iq - i + NN) + L * ((jq + NN) + L * (kq - k + NN));
    const double vq = vn[q];
    line_apply<NN, R>(xi, [&](int j, R y) {
      const R ki = y + b[NN * j + i];
      const R vr = R(vn[N2 * k + NN * j + i] + vq + tinv[t0 - L * j] * cf.inv_d3);
      const R vxr = vr * xr[j], vxi = vr * xi[j];
      ZT o;
      if constexpr (SHIFT) {
        o.x = s2r * kr[j] - s2i * ki + (c1r * vxr - shr * xr[j]) - (c1i * vxi - shi * xi[j]);
        o.y = s2r * ki + s2i * kr[j] + (c1r * vxi - shr * xi[j]) + (c1i * vxr - shi * xr[j]);
      } else {
        o.x = s2r * kr[j] - s2i * ki + rounded_product(c1r, vxr) - rounded_product(c1i, vxi);
        o.y = s2r * ki + s2i * kr[j] + rounded_product(c1r, vxi) + rounded_product(c1i, vxr);
      }
      z[base + NN * j] = o;
    });
  }
}

// Two more axes a, b at strides sa, sb: Y = Z + s2 (tau x 1 + 1 x tau) X on
// entries base + r + sa a + sb b, r < run.  A workgroup takes a run tile of
// blockIdx.x and the outer index blockIdx.y (stride so); thread (r, b) keeps the a
// line.  It reads its entries of X and Z before it writes them, so Y may be either.
// Runs start at any multiple of an entry (M is odd) and share lines with their
// neighbours: consecutive tiles go to one XCD (workgroups are dealt to the 8 XCDs
// in turn).  With NORMS nothing is written but each workgroup's sums of |Y - e X|^2 and
// |X|^2 in norms[2 blockIdx.x]: a residual needs no more of Y (112 bytes an entry over
// the three passes where writing Y and reading it back with X took 160; 8 pairs at
// NN = 17: 7.4 ms before).
//
// HBM-bound (48 bytes an entry), 4.7 TB/s at NN = 25 in FP64.  From NN = 17 on Z is read
// while the second component still has to go through LDS, and what is known of Y is
// summed onto it: read in the last loop, each entry's wait stood before its store
// (NN = 25 3.02 -> 2.48 ms a launch, NN = 21 1.13 -> 0.93).  On the smaller grids that
// costs a wave of each SIMD (registers) and 0-4%, as it would with NORMS from NN = 23 on.
template <int NN, typename R, typename XT, typename ZT, typename YT, bool NORMS = false>
__global__ __launch_bounds__(round_up(NN *plane_run<XT>(), 64)) void k_plane2(const XT *x, const ZT *z, YT *y,
                                                                             int64_t run, int64_t sa, int64_t sb,
                                                                             int64_t so, int64_t per_xcd,
                                                                             MatvecCoef cf, double e_re, double e_im,
                                                                             double *norms) {
  constexpr int P = plane_run<XT>(), N2 = NN * NN;
  extern __shared__ __align__(16) unsigned char smem[];
  const int r = threadIdx.x % P, bb = threadIdx.x / P;
  const int64_t r0 = ((blockIdx.x % 8) * per_xcd + blockIdx.x / 8) * P;
  const bool on = bb < NN && r0 + r < run;
  const int64_t base = r0 + r + so * blockIdx.y + sb * bb;
  R *a = reinterpret_cast<R *>(smem) + r;
  R *b = a + N2 * P;
  constexpr bool EARLY = NN >= 17 && !(NORMS && NN >= 23);
  R xr[NN], xi[NN], kr[NN];
  ZT o[NN];  // EARLY: Y's sum so far, in kr's place
  if (on) {
#pragma unroll
    for (int l = 0; l < NN; ++l) {
      const XT v = x[base + sa * l];
      xr[l] = R(v.x);
      xi[l] = R(v.y);
    }
  }
  // b lines of one component through LDS, thread (r, line a = bb)
  auto b_lines = [&](const R(&v)[NN]) {
    if (on) {
#pragma unroll
      for (int l = 0; l < NN; ++l) a[(l * NN + bb) * P] = v[l];
    }
    __syncthreads();
    if (on) {
      R t[NN];
#pragma unroll
      for (int l = 0; l < NN; ++l) t[l] = a[(bb * NN + l) * P];
      line_apply<NN, R>(t, [&](int l, R s) { b[(bb * NN + l) * P] = s; });
    }
  };
  const R s2r = R(cf.s2_re), s2i = R(cf.s2_im);
  double rr = 0.0, xx = 0.0;
  b_lines(xr);
  if constexpr (EARLY) {
    if (on) {
#pragma unroll
      for (int l = 0; l < NN; ++l) o[l] = z[base + sa * l];
    }
  }
  __syncthreads();
  if (on) {
    line_apply<NN, R>(xr, [&](int l, R s) {
      kr[l] = s + b[(l * NN + bb) * P];
      if constexpr (EARLY) {
        o[l].x += s2r * kr[l];
        o[l].y += s2i * kr[l];
        if constexpr (NORMS) {
          o[l].x -= e_re * xr[l];
          o[l].y -= e_im * xr[l];
          xx += double(xr[l]) * xr[l];
        }
      }
    });
  }
  b_lines(xi);
  __syncthreads();
  if (on) {
    line_apply<NN, R>(xi, [&](int l, R s) {
      const R ki = s + b[(l * NN + bb) * P];
      YT out;
      if constexpr (EARLY) {
        out.x = o[l].x - s2i * ki;
        out.y = o[l].y + s2r * ki;
      } else {
        const ZT zv = z[base + sa * l];
        out.x = zv.x + (s2r * kr[l] - s2i * ki);
        out.y = zv.y + (s2r * ki + s2i * kr[l]);
      }
      if constexpr (NORMS) {
        if constexpr (!EARLY) {
          out.x -= e_re * xr[l];
          out.y -= e_im * xr[l];
          xx += double(xr[l]) * xr[l];
        }
        const double dr = out.x + e_im * xi[l], di = out.y - e_re * xi[l];
        rr += dr * dr + di * di;
        xx += double(xi[l]) * xi[l];
      } else {
        y[base + sa * l] = out;
      }
    });
  }
  if constexpr (NORMS) {
    constexpr int W = round_up(NN * P, 64) / 64;
    __shared__ double red[W][2];
    for (int off = 32; off > 0; off >>= 1) {
      rr += __shfl_down(rr, off);
      xx += __shfl_down(xx, off);
    }
    if ((threadIdx.x & 63) == 0) {
      red[threadIdx.x >> 6][0] = rr;
      red[threadIdx.x >> 6][1] = xx;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
      double t = 0.0;
      for (int w = 0; w < W; ++w) t += red[w][threadIdx.x];
      norms[2 * size_t(blockIdx.x) + threadIdx.x] = t;
    }
  }
}

// ---- the smallest grids ----------------------------------------------------------
// General vectors in one launch: Y = s2 (K1 + K2) X + (c1 Vr - shift) o X, an entry a
// thread, from the six lines through it.  A vector fits the L2 many times over and a
// call is all latency: one launch and one wait for loads in place of two launches with
// an intermediate between.  Threads of a workgroup run along electron 1, so five of
// the six lines are read in runs along p.  Y must not overlap X: other workgroups read it.
// Every thread of a workgroup reaches its barrier (27 of 64 and 125 of 128 own an entry).
template <int NN>
constexpr int direct_threads() {
  return NN * NN * NN < 256 ? round_up(NN * NN * NN, 64) : 256;
}

template <int NN, typename R, typename XT>
__global__ __launch_bounds__(direct_threads<NN>()) void k_direct(ColPtrs xs, ColPtrsW ys,
                                                                 const double *__restrict__ vn,
                                                                 const double *__restrict__ tinv, MatvecCoef cf) {
  constexpr int N2 = NN * NN, N3 = NN * N2, L = 2 * NN + 1, T = direct_threads<NN>();
  constexpr int TILES = (N3 + T - 1) / T;
  const int q = int(blockIdx.x) / TILES, e1 = int(blockIdx.x) % TILES * T + int(threadIdx.x);
  const int p = e1 < N3 ? e1 : 0;  // threads past the end form entry 0 and do not write it
  const XT *__restrict__ x = static_cast<const XT *>(xs.p[blockIdx.y]);
  const int pi[3] = {p % NN, p / NN % NN, p / N2}, qi[3] = {q % NN, q / NN % NN, q / N2};
  constexpr int stride[3] = {1, NN, N2};
  const XT own = x[p + N3 * q];
  const R vr = R(vn[p] + vn[q] +
                 tinv[(qi[0] - pi[0] + NN) + L * ((qi[1] - pi[1] + NN) + L * (qi[2] - pi[2] + NN))] * cf.inv_d3);
  __shared__ R tau[2 * NN - 1];
  if (threadIdx.x < 2 * NN - 1) tau[threadIdx.x] = R(tau_rt(int(threadIdx.x) - (NN - 1)));
  __syncthreads();
  // each line's sum by itself, then the lines pairwise: fewer roundings on the way than in
  // one running sum
  R kr[3], ki[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    R pr = R(0), pim = R(0), qr = R(0), qim = R(0);
#pragma unroll
    for (int l = 0; l < NN; ++l) {
      const XT u = x[p + stride[a] * (l - pi[a]) + N3 * q], v = x[p + N3 * (q + stride[a] * (l - qi[a]))];
      const R tp = tau[l - pi[a] + NN - 1], tq = tau[l - qi[a] + NN - 1];
      pr += tp * R(u.x);
      pim += tp * R(u.y);
      qr += tq * R(v.x);
      qim += tq * R(v.y);
    }
    kr[a] = pr + qr;
    ki[a] = pim + qim;
  }
  const R sr = (kr[0] + kr[1]) + kr[2], si = (ki[0] + ki[1]) + ki[2];
  const R s2r = R(cf.s2_re), s2i = R(cf.s2_im);
  const R vcr = R(cf.c1_re) * vr - R(cf.sh_re), vci = R(cf.c1_im) * vr - R(cf.sh_im);
  XT o;
  o.x = s2r * sr - s2i * si + vcr * R(own.x) - vci * R(own.y);
  o.y = s2r * si + s2i * sr + vcr * R(own.y) + vci * R(own.x);
  if (e1 < N3) static_cast<XT *>(ys.p[blockIdx.y])[p + N3 * q] = o;
}

// ---- cross-check ---------------------------------------------------------------
// General vectors in FP64 by seven launches that share nothing with the passes above
// (no LDS, no even-odd lines, no fused axes): one launch an axis, a thread a line of
// stride `stride`, and the potential's.  Contexts made under DEX_MATVEC=generic take
// them, so that the two programs can be compared at any grid; no other context does
// (NN = 25: 16.8 ms a vector where the planes take 6.9).
template <int NN>
__global__ __launch_bounds__(256) void k_axis(const double2 *__restrict__ x, double2 *__restrict__ y, int64_t stride,
                                              int64_t nlines, int accumulate) {
  const int64_t line = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (line >= nlines) return;
  const int64_t off = line % stride + line / stride * stride * NN;
  double2 v[NN];
#pragma unroll
  for (int l = 0; l < NN; ++l) v[l] = x[off + stride * l];
#pragma unroll
  for (int i = 0; i < NN; ++i) {
    double2 o = accumulate ? y[off + stride * i] : make_double2(0.0, 0.0);
    double ar = 0.0, ai = 0.0;
#pragma unroll
    for (int l = 0; l < NN; ++l) {
      ar += tau_rt(l - i) * v[l].x;
      ai += tau_rt(l - i) * v[l].y;
    }
    o.x += ar;
    o.y += ai;
    y[off + stride * i] = o;
  }
}

// Y = s2 Y + (c1 Vr - shift) o X
__global__ __launch_bounds__(256) void k_potential(const double2 *__restrict__ x, double2 *__restrict__ y,
                                                   const double *__restrict__ vn, const double *__restrict__ tinv,
                                                   int nn, int64_t m, MatvecCoef cf) {
  const int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= m * m) return;
  const int p = int(idx % m), q = int(idx / m), L = 2 * nn + 1;
  const int ti = (q % nn - p % nn + nn) +
                 L * ((q / nn % nn - p / nn % nn + nn) + L * (q / (nn * nn) - p / (nn * nn) + nn));
  const double vr = vn[p] + vn[q] + tinv[ti] * cf.inv_d3;
  const double fr = vr * cf.c1_re - cf.sh_re, fi = vr * cf.c1_im - cf.sh_im;
  const double2 xv = x[idx], k = y[idx];
  y[idx] = make_double2(cf.s2_re * k.x - cf.s2_im * k.y + (fr * xv.x - fi * xv.y),
                        cf.s2_re * k.y + cf.s2_im * k.x + (fr * xv.y + fi * xv.x));
}

template <int NN>
hipError_t axes_nn(const double2 *x, double2 *y, const PotArgs &pot, hipStream_t s) {
  const int64_t m = int64_t(NN) * NN * NN, lines = m * m / NN;
  int64_t stride = 1;
  for (int axis = 0; axis < 6; ++axis, stride *= NN)
    hipLaunchKernelGGL(k_axis<NN>, dim3(unsigned((lines + 255) / 256)), dim3(256), 0, s, x, y, stride, lines, axis);
  hipLaunchKernelGGL(k_potential, dim3(unsigned((m * m + 255) / 256)), dim3(256), 0, s, x, y, pot.vn, pot.tinv, NN, m,
                     pot.cf);
  return hipGetLastError();
}

// out[e] = sum over nparts of partial[b nelem + e], one workgroup an element.
__global__ __launch_bounds__(1024) void k_reduce_wide(const double *__restrict__ partial, int nparts, int nelem,
                                                      double *__restrict__ out) {
  __shared__ double red[16];
  double s = 0.0;
  for (int b = threadIdx.x; b < nparts; b += 1024) s += partial[size_t(b) * nelem + blockIdx.x];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  // pairwise to the end: the last additions carry most of the rounding error
  if (threadIdx.x < 64) {
    s = threadIdx.x < 16 ? red[threadIdx.x] : 0.0;
    for (int off = 8; off > 0; off >>= 1) s += __shfl_down(s, off);
    if (threadIdx.x == 0) out[blockIdx.x] = s;
  }
}

// Function attributes and occupancy figures are set once per kernel, under
// g_setup_mu: prepare_kernels() does all of them when the first context is
// created, before any launch, so no hipFuncSetAttribute call ever runs while
// another thread launches (the launchers below only read the cached values,
// taking the lock themselves only if prepare_kernels() was never called).
std::mutex g_setup_mu;

// Sets the dynamic LDS limit of one kernel (once: `done` is the kernel's flag).
bool set_lds(const void *kernel, size_t lds, std::atomic<bool> &done) {
  if (done.load(std::memory_order_acquire)) return true;
  std::lock_guard<std::mutex> lk(g_setup_mu);
  if (done.load(std::memory_order_acquire)) return true;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)) != hipSuccess) return false;
  done.store(true, std::memory_order_release);
  return true;
}

// A shift is applied in FP64 only: a complex64 basis takes it in the block kernels
// (a - sig b of the descriptors), which form it in FP64.
bool shifted(const MatvecCoef &cf) { return cf.sh_re != 0.0 || cf.sh_im != 0.0; }

// LDS bytes of the passes' two cubes of reals.
template <int NN, typename R>
constexpr size_t cube_lds() {
  return size_t(2) * NN * NN * NN * sizeof(R);
}

template <int NN, typename R, typename XT, typename ZT>
bool pass1_setup() {
  static std::atomic<bool> plain{false}, shifted{false};
  if constexpr (sizeof(R) == 8) {
    if (!set_lds(reinterpret_cast<const void *>(&k_pass1<NN, R, XT, ZT, true>), cube_lds<NN, R>(), shifted)) return false;
  }
  return set_lds(reinterpret_cast<const void *>(&k_pass1<NN, R, XT, ZT, false>), cube_lds<NN, R>(), plain);
}

template <int NN, typename R, typename XT, typename YT>
bool pass2_setup() {
  static std::atomic<bool> attr{false};
  return set_lds(reinterpret_cast<const void *>(&k_pass2<NN, R, XT, YT>), cube_lds<NN, R>(), attr);
}

template <int NN, typename R, typename XT, typename ZT>
hipError_t pass1_nn(const ColPtrs &xs, const ColPtrsW &zs, int ncols, const PotArgs &pot, double w, hipStream_t s) {
  if (!pass1_setup<NN, R, XT, ZT>()) return hipErrorInvalidDeviceFunction;
  const dim3 g(NN * NN * NN, unsigned(ncols)), b(cube_threads<NN>());
  if (shifted(pot.cf)) {
    if constexpr (sizeof(R) == 8) {
      hipLaunchKernelGGL((k_pass1<NN, R, XT, ZT, true>), g, b, (cube_lds<NN, R>()), s, xs, zs, pot.vn, pot.tinv,
                         pot.cf, w);
      return hipGetLastError();
    }
    return hipErrorInvalidValue;
  }
  hipLaunchKernelGGL((k_pass1<NN, R, XT, ZT, false>), g, b, (cube_lds<NN, R>()), s, xs, zs, pot.vn, pot.tinv, pot.cf,
                     w);
  return hipGetLastError();
}

template <int NN, typename R, typename XT, typename YT>
hipError_t pass2_nn(const void *x, const void *z, void *y, int ncols, const MatvecCoef &cf, hipStream_t s) {
  using C = typename Cplx<R>::type;
  if (!pass2_setup<NN, R, XT, YT>()) return hipErrorInvalidDeviceFunction;
  hipLaunchKernelGGL((k_pass2<NN, R, XT, YT>), dim3(NN * NN * NN, unsigned(ncols)), dim3(cube_threads<NN>()),
                     (cube_lds<NN, R>()), s, static_cast<const XT *>(x), static_cast<const C *>(z),
                     static_cast<YT *>(y), cf);
  return hipGetLastError();
}

template <int NN, typename R>
constexpr size_t plane1_lds() {
  return size_t(2) * kPlane1Planes * NN * NN * sizeof(R);
}
template <int NN, typename R, typename XT>
constexpr size_t plane2_lds() {
  return size_t(2) * plane_run<XT>() * NN * NN * sizeof(R);
}

template <int NN, typename R, typename XT, typename ZT>
bool plane1_setup() {
  static std::atomic<bool> plain{false}, shifted{false};
  if constexpr (sizeof(R) == 8) {
    if (!set_lds(reinterpret_cast<const void *>(&k_plane1<NN, R, XT, ZT, true>), plane1_lds<NN, R>(), shifted)) return false;
  }
  return set_lds(reinterpret_cast<const void *>(&k_plane1<NN, R, XT, ZT, false>), plane1_lds<NN, R>(), plain);
}

template <int NN, typename R, typename XT, typename ZT, typename YT>
bool plane2_setup() {
  static std::atomic<bool> first{false}, second{false}, sums{false};
  if constexpr (sizeof(R) == 8) {
    if (!set_lds(reinterpret_cast<const void *>(&k_plane2<NN, R, XT, ZT, YT, true>), plane2_lds<NN, R, XT>(), sums))
      return false;
  }
  return set_lds(reinterpret_cast<const void *>(&k_plane2<NN, R, XT, ZT, ZT>), plane2_lds<NN, R, XT>(), first) &&
         set_lds(reinterpret_cast<const void *>(&k_plane2<NN, R, XT, ZT, YT>), plane2_lds<NN, R, XT>(), second);
}

template <int NN, typename R, typename XT, typename ZT>
hipError_t plane1_nn(const void *x, void *z, const PotArgs &pot, hipStream_t s) {
  if (!plane1_setup<NN, R, XT, ZT>()) return hipErrorInvalidDeviceFunction;
  constexpr int G = kPlane1Planes;
  const dim3 g(NN * NN * NN, (NN + G - 1) / G), b(round_up(NN * G, 64));
  const XT *xx = static_cast<const XT *>(x);
  ZT *zz = static_cast<ZT *>(z);
  if (shifted(pot.cf)) {
    if constexpr (sizeof(R) == 8) {
      hipLaunchKernelGGL((k_plane1<NN, R, XT, ZT, true>), g, b, (plane1_lds<NN, R>()), s, xx, zz, pot.vn, pot.tinv,
                         pot.cf);
      return hipGetLastError();
    }
    return hipErrorInvalidValue;
  }
  hipLaunchKernelGGL((k_plane1<NN, R, XT, ZT, false>), g, b, (plane1_lds<NN, R>()), s, xx, zz, pot.vn, pot.tinv,
                     pot.cf);
  return hipGetLastError();
}

// k1 and i2, runs along (i1, j1); then j2 and k2, runs along (i1, j1, k1, i2): into Y,
// or (norms, FP64) into the sums of |Y - e X|^2 and |X|^2 in out.
template <int NN, typename R, typename XT, typename ZT, typename YT>
hipError_t plane2_nn(const void *x, void *z, void *y, const MatvecCoef &cf, hipStream_t s, double *norms = nullptr,
                     double e_re = 0.0, double e_im = 0.0, double *out = nullptr) {
  if (!plane2_setup<NN, R, XT, ZT, YT>()) return hipErrorInvalidDeviceFunction;
  constexpr int64_t N2 = NN * NN, N3 = NN * N2, N4 = NN * N3;
  constexpr int P = plane_run<XT>();
  const XT *xx = static_cast<const XT *>(x);
  ZT *zz = static_cast<ZT *>(z);
  auto per_xcd = [](int64_t run) { return ((run + P - 1) / P + 7) / 8; };  // run tiles an XCD takes
  const dim3 block(round_up(NN * P, 64)), last(unsigned(8 * per_xcd(N4)));
  const size_t lds = plane2_lds<NN, R, XT>();
  double *none = nullptr;
  hipLaunchKernelGGL((k_plane2<NN, R, XT, ZT, ZT>), dim3(unsigned(8 * per_xcd(N2)), unsigned(N2)), block, lds, s, xx,
                     static_cast<const ZT *>(zz), zz, N2, N2, N3, N4, per_xcd(N2), cf, 0.0, 0.0, none);
  if constexpr (sizeof(R) == 8) {
    if (norms) {
      YT *noy = nullptr;
      hipLaunchKernelGGL((k_plane2<NN, R, XT, ZT, YT, true>), last, block, lds, s, xx, static_cast<const ZT *>(zz),
                         noy, N4, N4, N4 * NN, int64_t(0), per_xcd(N4), cf, e_re, e_im, norms);
      hipLaunchKernelGGL(k_reduce_wide, dim3(2), dim3(1024), 0, s, norms, int(last.x), 2, out);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((k_plane2<NN, R, XT, ZT, YT>), last, block, lds, s, xx, static_cast<const ZT *>(zz),
                     static_cast<YT *>(y), N4, N4, N4 * NN, int64_t(0), per_xcd(N4), cf, 0.0, 0.0, none);
  return hipGetLastError();
}

// LDS budget per workgroup on gfx950.
constexpr size_t kMaxLds = 160 * 1024;

constexpr bool fast_fits(int nn, size_t rsize) {
  return size_t(2) * nn * nn * nn * rsize <= kMaxLds;
}

}  // namespace

// Largest grid whose general vectors go through the cubes (launch_general_first).
constexpr int kCubeMaxNN = 11;
// Largest grid whose general vectors take one launch (k_direct).  Microseconds of a
// call, two launches and one: one column at NN = 3 23.4 and 20.0, at NN = 5 24.4 and
// 20.3, 16 columns there 33.3 and 24.3; at NN = 7 one column 27.7 and 23.7, but 16
// columns 66.6 and 80.0 (each entry reads its six lines, 42 entries, from L2).
constexpr int kDirectMaxNN = 5;

#define DEX_NN_LIST(X) X(3) X(5) X(7) X(9) X(11) X(13) X(15) X(17) X(19) X(21) X(23) X(25)

bool fast_matvec_supported(int nn, bool single) {
  switch (nn) {
#define CASE(N) \
  case N:       \
    return fast_fits(N, single ? sizeof(float) : sizeof(double));
    DEX_NN_LIST(CASE)
#undef CASE
    default:
      return false;
  }
}

bool generic_matvec_supported(int nn) {
  switch (nn) {
#define CASE(N) \
  case N:       \
    return true;
    DEX_NN_LIST(CASE)
#undef CASE
    default:
      return false;
  }
}

hipError_t launch_pass1(int nn, int io, bool sym, const void *const *x, void *const *z, int ncols,
                        const PotArgs &pot, hipStream_t s) {
  if (ncols < 1 || ncols > kBatchMax) return hipErrorInvalidValue;
  ColPtrs xs{};
  ColPtrsW zs{};
  for (int j = 0; j < ncols; ++j) {
    xs.p[j] = x[j];
    zs.p[j] = z[j];
  }
  const double w = sym ? 0.5 : 1.0;
  switch (nn) {
#define CASE(N)                                                                                         \
  case N:                                                                                               \
    if constexpr (fast_fits(N, sizeof(double))) {                                                       \
      if (io == kIoF64) return pass1_nn<N, double, double2, double2>(xs, zs, ncols, pot, w, s);         \
    }                                                                                                   \
    if constexpr (fast_fits(N, sizeof(float))) {                                                        \
      if (io == kIoF32) return pass1_nn<N, float, float2, float2>(xs, zs, ncols, pot, w, s);            \
      if (io == kIoMixed && sym) return pass1_nn<N, float, double2, double2>(xs, zs, ncols, pot, w, s); \
    }                                                                                                   \
    if constexpr (N <= kCubeMaxNN) {                                                                    \
      if (io == kIoMixed) return pass1_nn<N, float, double2, float2>(xs, zs, ncols, pot, w, s);         \
    }                                                                                                   \
    return hipErrorInvalidValue;
    DEX_NN_LIST(CASE)
#undef CASE
    default:
      return hipErrorInvalidValue;
  }
}

hipError_t launch_symfold(int nn, int io, void *const *y, int ncols, int sign, hipStream_t s) {
  if (ncols < 1 || ncols > kBatchMax) return hipErrorInvalidValue;
  ColPtrsW ys{};
  for (int j = 0; j < ncols; ++j) ys.p[j] = y[j];
  const int m = nn * nn * nn, nblk = sym_blocks(m);
  const dim3 g(unsigned(sym_grid(m)), unsigned(ncols)), b(kSymT, 8);
  if (io == kIoF32)
    hipLaunchKernelGGL((k_symfold<float2>), g, b, 0, s, ys, m, nblk, sign);
  else
    hipLaunchKernelGGL((k_symfold<double2>), g, b, 0, s, ys, m, nblk, sign);
  return hipGetLastError();
}

// General vectors go through the cubes (k_pass1, k_pass2) on the smallest grids and
// through the planes beyond: k_pass2's stride-M reads take 16 (8) bytes of each
// 128-byte line, and the neighbours that share it find it in L2 less and less
// often (3.3 times the bytes from HBM at NN = 13).  Microseconds a vector, cubes
// and planes: NN = 11 FP64 68 and 69; 13: 165 and 135; 17: 997 and 745; 21: 3270 and
// 2850; complex64 at 17: 833 and 455; at 25: 7035 and 4300.
bool general_by_planes(int nn) { return nn > kCubeMaxNN; }

bool general_direct(int nn) { return nn <= kDirectMaxNN; }

hipError_t launch_direct(int nn, int io, const void *x, void *y, int ncols, const PotArgs &pot, hipStream_t s) {
  if (ncols < 1 || ncols > kBatchMax || (io != kIoF64 && shifted(pot.cf))) return hipErrorInvalidValue;
  ColPtrs xs{};
  ColPtrsW ys{};
  const size_t bytes = size_t(nn) * nn * nn * nn * nn * nn * (io == kIoF32 ? 8 : 16);
  for (int j = 0; j < ncols; ++j) {
    xs.p[j] = static_cast<const char *>(x) + size_t(j) * bytes;
    ys.p[j] = static_cast<char *>(y) + size_t(j) * bytes;
  }
  switch (nn) {
#define CASE(N)                                                                                                  \
  case N:                                                                                                        \
    if constexpr (N <= kDirectMaxNN) {                                                                           \
      constexpr int T = direct_threads<N>();                                                                     \
      const dim3 g(N * N * N * ((N * N * N + T - 1) / T), unsigned(ncols)), b(T);                                \
      if (io == kIoF64)                                                                                          \
        hipLaunchKernelGGL((k_direct<N, double, double2>), g, b, 0, s, xs, ys, pot.vn, pot.tinv, pot.cf);        \
      else if (io == kIoF32)                                                                                     \
        hipLaunchKernelGGL((k_direct<N, float, float2>), g, b, 0, s, xs, ys, pot.vn, pot.tinv, pot.cf);          \
      else                                                                                                       \
        hipLaunchKernelGGL((k_direct<N, float, double2>), g, b, 0, s, xs, ys, pot.vn, pot.tinv, pot.cf);         \
      return hipGetLastError();                                                                                  \
    }                                                                                                            \
    return hipErrorInvalidValue;
    DEX_NN_LIST(CASE)
#undef CASE
    default:
      return hipErrorInvalidValue;
  }
}

hipError_t launch_general_first(int nn, int io, const void *x, void *z, int ncols, const PotArgs &pot, hipStream_t s) {
  if (ncols < 1 || ncols > kBatchMax) return hipErrorInvalidValue;
  if (!general_by_planes(nn)) {
    const size_t d = size_t(nn) * nn * nn * nn * nn * nn;
    const void *xs[kBatchMax];
    void *zs[kBatchMax];
    for (int j = 0; j < ncols; ++j) {
      xs[j] = static_cast<const char *>(x) + size_t(j) * d * (io == kIoF32 ? 8 : 16);
      zs[j] = static_cast<char *>(z) + size_t(j) * d * (io == kIoF64 ? 16 : 8);
    }
    return launch_pass1(nn, io, false, xs, zs, ncols, pot, s);
  }
  if (ncols != 1) return hipErrorInvalidValue;
  switch (nn) {
#define CASE(N)                                                                           \
  case N:                                                                                 \
    if constexpr (N > kCubeMaxNN) {                                                       \
      if (io == kIoF64) return plane1_nn<N, double, double2, double2>(x, z, pot, s);      \
      if (io == kIoF32) return plane1_nn<N, float, float2, float2>(x, z, pot, s);         \
      return plane1_nn<N, float, double2, float2>(x, z, pot, s);                          \
    }                                                                                     \
    return hipErrorInvalidValue;
    DEX_NN_LIST(CASE)
#undef CASE
    default:
      return hipErrorInvalidValue;
  }
}

hipError_t launch_general_second(int nn, int io, const void *x, void *z, void *y, int ncols, const MatvecCoef &coef,
                                 hipStream_t s) {
  if (ncols < 1 || ncols > kBatchMax || (ncols != 1 && general_by_planes(nn))) return hipErrorInvalidValue;
  switch (nn) {
#define CASE(N)                                                                                       \
  case N:                                                                                             \
    if constexpr (N > kCubeMaxNN) {                                                                   \
      if (io == kIoF64) return plane2_nn<N, double, double2, double2, double2>(x, z, y, coef, s);     \
      if (io == kIoF32) return plane2_nn<N, float, float2, float2, float2>(x, z, y, coef, s);         \
      return plane2_nn<N, float, double2, float2, double2>(x, z, y, coef, s);                         \
    } else {                                                                                          \
      if (io == kIoF64) return pass2_nn<N, double, double2, double2>(x, z, y, ncols, coef, s);     \
      if (io == kIoF32) return pass2_nn<N, float, float2, float2>(x, z, y, ncols, coef, s);        \
      return pass2_nn<N, float, double2, double2>(x, z, y, ncols, coef, s);                        \
    }
    DEX_NN_LIST(CASE)
#undef CASE
    default:
      return hipErrorInvalidValue;
  }
}

hipError_t launch_axes(int nn, const Dbl2 *x, Dbl2 *y, const PotArgs &pot, hipStream_t s) {
  switch (nn) {
#define CASE(N) \
  case N:       \
    return axes_nn<N>(reinterpret_cast<const double2 *>(x), reinterpret_cast<double2 *>(y), pot, s);
    DEX_NN_LIST(CASE)
#undef CASE
    default:
      return hipErrorInvalidValue;
  }
}

hipError_t launch_general_norms(int nn, const Dbl2 *x, Dbl2 *z, double e_re, double e_im, double *partial,
                                double *out, const MatvecCoef &coef, hipStream_t s) {
  switch (nn) {
#define CASE(N)                                                                                                  \
  case N:                                                                                                        \
    if constexpr (N > kCubeMaxNN)                                                                                \
      return plane2_nn<N, double, double2, double2, double2>(x, z, nullptr, coef, s, partial, e_re, e_im, out);   \
    return hipErrorInvalidValue;
    DEX_NN_LIST(CASE)
#undef CASE
    default:
      return hipErrorInvalidValue;
  }
}

// ---- block kernels ----------------------------------------------------------
namespace {

constexpr int kGramThreads = 256;
constexpr int kGramMaxL = 64;
constexpr int kGramMaxR = 128;
constexpr int kGramBlocks = 1024;

// Element r of a complex128 (fmt 0) or complex64 (fmt 1) column, in FP64.
__device__ __forceinline__ double2 ld_col(const void *p, int fmt, int64_t r) {
  if (fmt != 0) {
    const float2 v = reinterpret_cast<const float2 *>(p)[r];
    return make_double2(double(v.x), double(v.y));
  }
  return reinterpret_cast<const double2 *>(p)[r];
}

__device__ __forceinline__ void st_col(void *p, int fmt, int64_t r, double2 v) {
  if (fmt != 0)
    reinterpret_cast<float2 *>(p)[r] = make_float2(float(v.x), float(v.y));
  else
    reinterpret_cast<double2 *>(p)[r] = v;
}

// Four floats at 8-byte alignment (a row pair that starts at an odd row).
typedef float dex_v4f __attribute__((ext_vector_type(4), aligned(8)));

// Two adjacent rows r, r + 1 of a complex128 (fmt 0) or complex64 (fmt 1)
// column in FP64; `two` false reads only row r (the last row of an odd-length
// column).  A complex64 pair is one 16-byte load, a complex128 pair two.
__device__ __forceinline__ void ld_col2(const void *p, int fmt, int64_t r, bool two, double2 &v0, double2 &v1) {
  if (fmt != 0) {
    const float2 *q = reinterpret_cast<const float2 *>(p) + r;
    if (two) {
      const dex_v4f w = *reinterpret_cast<const dex_v4f *>(q);
      v0 = make_double2(double(w.x), double(w.y));
      v1 = make_double2(double(w.z), double(w.w));
    } else {
      const float2 w = *q;
      v0 = make_double2(double(w.x), double(w.y));
      v1 = make_double2(0.0, 0.0);
    }
    return;
  }
  const double2 *q = reinterpret_cast<const double2 *>(p) + r;
  v0 = q[0];
  v1 = two ? q[1] : make_double2(0.0, 0.0);
}

__device__ __forceinline__ void st_col2(void *p, int fmt, int64_t r, bool two, double2 v0, double2 v1) {
  if (fmt != 0) {
    float2 *q = reinterpret_cast<float2 *>(p) + r;
    if (two)
      *reinterpret_cast<float4 *>(q) = make_float4(float(v0.x), float(v0.y), float(v1.x), float(v1.y));
    else
      *q = make_float2(float(v0.x), float(v0.y));
    return;
  }
  double2 *q = reinterpret_cast<double2 *>(p) + r;
  q[0] = v0;
  if (two) q[1] = v1;
}

__device__ __forceinline__ double2 col_value(const ColDesc &c, int64_t r) {
  const double2 va = ld_col(c.a, c.fmt, r);
  if (c.b == nullptr) return va;
  const double2 vb = ld_col(c.b, c.fmt, r);
  double2 o;
  o.x = va.x - (c.sig_re * vb.x - c.sig_im * vb.y);
  o.y = va.y - (c.sig_re * vb.y + c.sig_im * vb.x);
  return o;
}

// Rows r, r + 1 of a descriptor's column, as ld_col2 reads them.
__device__ __forceinline__ void col_values2(const ColDesc &c, int64_t r, bool two, double2 &v0, double2 &v1) {
  ld_col2(c.a, c.fmt, r, two, v0, v1);
  if (c.b == nullptr) return;
  double2 b0, b1;
  ld_col2(c.b, c.fmt, r, two, b0, b1);
  v0.x -= c.sig_re * b0.x - c.sig_im * b0.y;
  v0.y -= c.sig_re * b0.y + c.sig_im * b0.x;
  v1.x -= c.sig_re * b1.x - c.sig_im * b1.y;
  v1.y -= c.sig_re * b1.y + c.sig_im * b1.x;
}

// The row tiles a workgroup of the Gram kernels takes, in order.
//   !TRI: rows 0 .. d - 1, tiles round robin over the grid.
//   TRI: the columns are exchange-(anti)symmetric M x M matrices, whose products
//     conj(l) r are symmetric: only the 64 x 64 blocks on and above the diagonal
//     are read, those above first (`diag` false: the caller doubles their sum), then
//     the diagonal ones.  A unit is 64 consecutive rows of one matrix column (fewer in
//     the last block); consecutive units go to one XCD, where the lines that two of
//     them share (M is odd) meet in L2.  Tiles cut at whole lines instead: no faster
//     (280 for 290 us at 64 x 10 columns, M = 1331), and 5% slower where 64-row tiles
//     become five a unit.
constexpr int kTriT = 64;

template <int ROWS, bool TRI>
struct RowWalk {
  static_assert(kTriT % ROWS == 0, "whole tiles in a unit");
  int64_t row = 0;  // first row of the tile
  int rows = 0;     // its rows, 0 when none is left
  bool diag = false;

  __device__ RowWalk(int64_t d, int m) : m_(m) {
    if constexpr (!TRI) {
      row = int64_t(blockIdx.x) * ROWS;
      left_ = d - row;
    } else {
      const int b = m / kTriT;
      n_ = kTriT / 2 * b * (b - 1) + (m - kTriT * b) * b;
      i_ = blockIdx.x / 8;
      unit();
    }
    rows = left_ < ROWS ? (left_ > 0 ? int(left_) : 0) : ROWS;
  }
  __device__ void next() {
    const int64_t by = TRI ? int64_t(ROWS) : int64_t(gridDim.x) * ROWS;
    row += by;
    left_ -= by;
    if (TRI && left_ <= 0) {
      i_ += gridDim.x / 8;
      unit();
    }
    rows = left_ < ROWS ? (left_ > 0 ? int(left_) : 0) : ROWS;
  }

 private:

  int64_t left_ = 0;  // rows from `row` to the end (of the unit)
  int m_, i_ = 0, n_ = 0;

  // The first tile of this workgroup's unit i_, or of a later phase.
  __device__ void unit() {
    for (;;) {
      const int per = (n_ + 7) / 8, u = int(blockIdx.x % 8) * per + i_;
      if (i_ < per && u < n_) {
        if (!diag) {
          // block column j from its first unit, 32 j (j - 1)
          int j = int((1.0f + sqrtf(1.0f + float(u) * (8.0f / kTriT))) * 0.5f);
          while (kTriT / 2 * j * (j - 1) > u) --j;
          while (kTriT / 2 * j * (j + 1) <= u) ++j;
          const int v = u - kTriT / 2 * j * (j - 1);
          row = int64_t(kTriT * j + v / j) * m_ + kTriT * (v % j);
          left_ = kTriT;
        } else {
          const int p0 = u / kTriT * kTriT;
          row = int64_t(u) * m_ + p0;
          left_ = m_ - p0 < kTriT ? m_ - p0 : kTriT;
        }
        return;
      }
      if (diag) {
        left_ = 0;
        return;
      }
      diag = true;
      n_ = m_;
      i_ = blockIdx.x / 8;
    }
  }
};

// Partial Gram G = L^H R of each workgroup's row tiles (RowWalk), on the FP64
// matrix cores.  G = L^H R is a GEMM whose
// inner dimension is the vector length: per 4 rows, v_mfma_f64_16x16x4f64
// multiplies a 16 x 4 slice of L^T by a 4 x 16 slice of R into a 16 x 16
// output tile (lane l supplies A[l % 16][l / 16] and B[l / 16][l % 16] and
// holds D[4 v + l / 16][l % 16], v < 4).  A complex tile takes four real
// products: Re += Lr Rr + Li Ri, Im += Lr Ri - Li Rr.  The rows are staged
// through LDS (one coalesced pass over every column); each LDS value then
// feeds 16 MACs of a matrix instruction instead of one vector FMA (a vector-FMA
// version of this kernel was bound by the LDS bandwidth at ~2.5 TB/s).  The 4 waves of a
// workgroup share the output tiles (MT x NT of them) round-robin.
typedef double dex_v4d __attribute__((ext_vector_type(4)));

// Rows per staged tile: 16 (TALL = 32 for the narrowest shapes), halved while
// the tile exceeds 48 KB.  16-row tiles (8-33 KB) leave room for 4+ resident
// workgroups per CU; 32-row tiles measured 10-23% slower at 54-64 x 10 (2
// workgroups per CU, VGPR-bound).  A Gram of one 16 x 16 output tile (the
// inner solve's projections of 4-column groups) keeps few bytes in flight per
// workgroup with 16-row tiles: 32-row tiles measured 5-6% faster there at
// NN=21 (8 x 4, 16 x 4, 12 x 10) and 5-7% slower at 28 x 4 and 32 x 16.
constexpr int gram_mfma_rows(int mt, int nt, int tall = 16) {
  const int cap = tall >= 64 ? 64 * 1024 : 48 * 1024;  // tiles of up to 64 rows may take 64 KB of LDS
  int r = tall;
  while (r > 4 && r * (16 * mt + 16 * nt + 1) * 16 > cap) r /= 2;
  return r;
}

template <int MT, int NT, int TALL, bool TRI>
__global__ __launch_bounds__(kGramThreads) void k_gram_mfma(const ColDesc *__restrict__ descs, int kl,
                                                            int kr, int share, int64_t d, int m,
                                                            double2 *__restrict__ partial) {
  constexpr int LD = 16 * MT + 16 * NT + 1;
  constexpr int ROWS = gram_mfma_rows(MT, NT, TALL);
  constexpr int QMAX = (MT * NT + 3) / 4;
  // With fewer 16 x 16 output tiles than waves, KS waves share each tile and
  // split its rows (k steps) between them, their sums added through LDS at the
  // end: with one wave per tile, a one-tile Gram ran all its MFMAs on one SIMD
  // of four and every workgroup waited on them
  constexpr int KS = MT * NT == 1 ? 4 : (MT * NT == 2 ? 2 : 1);
  static_assert(gram_mfma_rows(MT, NT, TALL) % (4 * KS) == 0, "every wave takes whole row steps");
  // loads per thread per tile, each an adjacent row pair of one column (16-byte
  // accesses for complex64 and complex128 alike): every thread issues all of
  // them before any wait, and the next tile's while the matrix cores work on
  // this one
  constexpr int HALF = ROWS / 2;
  constexpr int PMAX = (HALF * (16 * MT + 16 * NT) + kGramThreads - 1) / kGramThreads;
  // the row tile, reused after the loop for the k-split sums (4 KB per wave)
  constexpr int TILE2 = ROWS * LD > MT * NT * (KS - 1) * 256 ? ROWS * LD : MT * NT * (KS - 1) * 256;
  __shared__ double2 tile[TILE2];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int ks = KS > 1 ? wave % KS : 0;  // this wave's share of the k steps
  const int nload = kl + (kr - share);
  const int mt_valid = (kl + 15) / 16, nt_valid = (kr + 15) / 16;
  int tm[QMAX], tn[QMAX];
  bool tv[QMAX];
#pragma unroll
  for (int q = 0; q < QMAX; ++q) {
    const int t = KS > 1 ? wave / KS : wave + 4 * q;
    tm[q] = t % MT;
    tn[q] = t / MT;
    tv[q] = t < MT * NT && tm[q] < mt_valid && tn[q] < nt_valid &&
            !(tm[q] > tn[q] && 16 * (tm[q] + 1) <= share);
  }
  dex_v4d accr[QMAX], acci[QMAX];
#pragma unroll
  for (int q = 0; q < QMAX; ++q) {
    accr[q] = dex_v4d{0.0, 0.0, 0.0, 0.0};
    acci[q] = dex_v4d{0.0, 0.0, 0.0, 0.0};
  }
  // Element p of this thread is (row pair e % HALF, column e / HALF) of every
  // tile, e = tid + 256 p: its column pointers are fixed for the whole loop.
  const void *pa[PMAX];
  const void *pb[PMAX];
  int pf[PMAX];
#pragma unroll
  for (int p = 0; p < PMAX; ++p) {
    const int e = tid + kGramThreads * p;
    pa[p] = nullptr;
    pb[p] = nullptr;
    pf[p] = 0;
    if (e < HALF * nload) {
      const ColDesc &dc = descs[e / HALF];
      pa[p] = dc.a;
      pb[p] = dc.b;
      pf[p] = dc.fmt;
    }
  }
  // One tile in flight per workgroup while the matrix cores work on the
  // previous one: three register stages (more bytes in flight per workgroup)
  // measured 4-8% slower on the narrow shapes (fewer resident workgroups)
  double2 va[PMAX][2], vb[PMAX][2];
  auto fetch = [&](const RowWalk<ROWS, TRI> &w) {
#pragma unroll
    for (int p = 0; p < PMAX; ++p) {
      const int lr = 2 * ((tid + kGramThreads * p) % HALF);
      const int64_t row = w.row + lr;
      va[p][0] = va[p][1] = vb[p][0] = vb[p][1] = make_double2(0.0, 0.0);
      if (pa[p] != nullptr && lr < w.rows) {
        const bool two = lr + 1 < w.rows;
        ld_col2(pa[p], pf[p], row, two, va[p][0], va[p][1]);
        if (pb[p] != nullptr) ld_col2(pb[p], pf[p], row, two, vb[p][0], vb[p][1]);
      }
    }
  };
  auto store = [&]() {
#pragma unroll
    for (int p = 0; p < PMAX; ++p) {
      if (pa[p] == nullptr) continue;  // beyond the loads, or supplied through a bslot
      const int e = tid + kGramThreads * p;
      const int r = 2 * (e % HALF), c = e / HALF;
      const int slot = c < kl ? c : 16 * MT + (c - kl);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (pb[p] == nullptr) {
          tile[(r + h) * LD + slot] = va[p][h];
        } else {
          const ColDesc &dc = descs[c];
          double2 o;
          o.x = va[p][h].x - (dc.sig_re * vb[p][h].x - dc.sig_im * vb[p][h].y);
          o.y = va[p][h].y - (dc.sig_re * vb[p][h].y + dc.sig_im * vb[p][h].x);
          tile[(r + h) * LD + slot] = o;
          if (dc.bslot >= 0) tile[(r + h) * LD + dc.bslot] = vb[p][h];
        }
      }
    }
  };
  bool halves = TRI;  // the sums so far count half
  auto twice = [&]() {
#pragma unroll
    for (int q = 0; q < QMAX; ++q) {
      accr[q] += accr[q];
      acci[q] += acci[q];
    }
    halves = false;
  };
  RowWalk<ROWS, TRI> walk(d, m);  // one tile ahead: the tile in flight
  if (walk.rows) fetch(walk);
  while (walk.rows) {
    const bool diag = walk.diag;
    walk.next();
    store();
    __syncthreads();
    if (walk.rows) fetch(walk);
    if (halves && diag) twice();
    // this wave's row steps: k0 = 4 (ks + KS s)
#pragma unroll
    for (int st = 0; st < ROWS / (4 * KS); ++st) {
      const int k0 = 4 * (ks + KS * st);
      const double2 *trow = tile + (k0 + lk) * LD;
#pragma unroll
      for (int q = 0; q < QMAX; ++q) {
        if (!tv[q]) continue;
        const double2 av = trow[16 * tm[q] + li];
        const int jj = 16 * tn[q] + li;
        const double2 bv = trow[jj < share ? jj : 16 * MT + (jj - share)];
        accr[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.x, bv.x, accr[q], 0, 0, 0);
        accr[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.y, bv.y, accr[q], 0, 0, 0);
        acci[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.x, bv.y, acci[q], 0, 0, 0);
        acci[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(-av.y, bv.x, acci[q], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  if (halves) twice();
  if constexpr (KS > 1) {
    // the waves with ks > 0 hand their sums to the tile's ks = 0 wave (the last
    // __syncthreads of the loop has freed the row tile)
    double *red = reinterpret_cast<double *>(tile);
    const int t = wave / KS;
    if (ks > 0 && tv[0]) {
      double *slot = red + size_t(t * (KS - 1) + ks - 1) * 512;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        slot[v * 64 + lane] = accr[0][v];
        slot[(4 + v) * 64 + lane] = acci[0][v];
      }
    }
    __syncthreads();
    if (ks == 0 && tv[0]) {
#pragma unroll
      for (int k = 1; k < KS; ++k) {
        const double *slot = red + size_t(t * (KS - 1) + k - 1) * 512;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          accr[0][v] += slot[v * 64 + lane];
          acci[0][v] += slot[(4 + v) * 64 + lane];
        }
      }
    }
  }
  double2 *out = partial + size_t(blockIdx.x) * kl * kr;
#pragma unroll
  for (int q = 0; q < QMAX; ++q) {
    if (!tv[q] || ks != 0) continue;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int i = 16 * tm[q] + 4 * v + lk, j = 16 * tn[q] + li;
      if (i < kl && j < kr) out[i + size_t(kl) * j] = make_double2(accr[q][v], acci[q][v]);
    }
  }
}

// Partial Gram G = L^H R for narrow shapes (kl <= 8 M8 <= 32, kr <= 8: the
// inner solve's projections of 4-column groups) with the real and imaginary
// parts as separate MFMA rows and columns: A = [Re L_c; Im L_c] (16 rows for 8
// left columns), B = [Re R_r, Im R_r] (16 columns for 8 right columns), so one
// v_mfma_f64_16x16x4f64 per 4 rows forms all four real products of an 8 x 8
// complex block, O = [Lr Rr, Lr Ri; Li Rr, Li Ri], and G(c, r) =
// O(c, r) + O(c+8, r+8) + i (O(c, r+8) - O(c+8, r)) at the end.  The 16 x 16
// complex tiles of k_gram_mfma take 4 MFMAs for any kl <= 16, kr <= 16; this
// layout takes ceil(kl / 8).  Rows are staged in LDS as in k_gram_mfma (one
// row tile per workgroup, the next prefetched, tiles round robin over the
// grid); KS waves share each 8 x 8 block and split its row steps.  Right
// columns are unshared (share 0) or all shared with the first left columns
// (share == kr).  Layout of the partials as k_gram_mfma's.
template <int M8, int ROWS, bool TRI>
__global__ __launch_bounds__(kGramThreads) void k_gram_pk(const ColDesc *__restrict__ descs, int kl, int kr,
                                                          int share, int64_t d, int m,
                                                          double2 *__restrict__ partial) {
  constexpr int LD = 8 * M8 + 8 + 1;
  constexpr int KS = M8 == 1 ? 4 : (M8 == 2 ? 2 : 1);
  static_assert(ROWS % (4 * KS) == 0, "every wave takes whole row steps");
  constexpr int HALF = ROWS / 2;
  constexpr int PMAX = (HALF * (8 * M8 + 8) + kGramThreads - 1) / kGramThreads;
  // the row tile, reused after the loop for the waves' 16 x 16 sums (256 doubles each)
  constexpr int TILE2 = ROWS * LD > M8 * KS * 128 ? ROWS * LD : M8 * KS * 128;
  __shared__ double2 tile[TILE2];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int t = KS > 1 ? wave / KS : wave;  // this wave's 8-column block of L
  const int ks = KS > 1 ? wave % KS : 0;    // and its share of the row steps
  const bool tv = t < M8 && 8 * t < kl;
  const int nload = kl + (kr - share);
  dex_v4d acc = dex_v4d{0.0, 0.0, 0.0, 0.0};
  const void *pa[PMAX];
  const void *pb[PMAX];
  int pf[PMAX];
#pragma unroll
  for (int p = 0; p < PMAX; ++p) {
    const int e = tid + kGramThreads * p;
    pa[p] = nullptr;
    pb[p] = nullptr;
    pf[p] = 0;
    if (e < HALF * nload) {
      const ColDesc &dc = descs[e / HALF];
      pa[p] = dc.a;
      pb[p] = dc.b;
      pf[p] = dc.fmt;
    }
  }
  double2 va[PMAX][2], vb[PMAX][2];
  auto fetch = [&](const RowWalk<ROWS, TRI> &w) {
#pragma unroll
    for (int p = 0; p < PMAX; ++p) {
      const int lr = 2 * ((tid + kGramThreads * p) % HALF);
      const int64_t row = w.row + lr;
      va[p][0] = va[p][1] = vb[p][0] = vb[p][1] = make_double2(0.0, 0.0);
      if (pa[p] != nullptr && lr < w.rows) {
        const bool two = lr + 1 < w.rows;
        ld_col2(pa[p], pf[p], row, two, va[p][0], va[p][1]);
        if (pb[p] != nullptr) ld_col2(pb[p], pf[p], row, two, vb[p][0], vb[p][1]);
      }
    }
  };
  auto store = [&]() {
#pragma unroll
    for (int p = 0; p < PMAX; ++p) {
      if (pa[p] == nullptr) continue;
      const int e = tid + kGramThreads * p;
      const int r = 2 * (e % HALF), c = e / HALF;
      const int slot = c < kl ? c : 8 * M8 + (c - kl);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        double2 o = va[p][h];
        if (pb[p] != nullptr) {
          const ColDesc &dc = descs[c];
          o.x -= dc.sig_re * vb[p][h].x - dc.sig_im * vb[p][h].y;
          o.y -= dc.sig_re * vb[p][h].y + dc.sig_im * vb[p][h].x;
        }
        tile[(r + h) * LD + slot] = o;
      }
    }
  };
  // this lane's A row (a part of left column 8 t + (li & 7)) and B column (a
  // part of right column li & 7; shared right columns are the first left ones)
  const int acol = 8 * t + (li & 7);
  const int rj = li & 7;
  const int bcol = rj < share ? rj : 8 * M8 + (rj - share);
  const bool im = li >= 8;
  bool halves = TRI;  // the sums so far count half
  RowWalk<ROWS, TRI> walk(d, m);  // one tile ahead: the tile in flight
  if (walk.rows) fetch(walk);
  while (walk.rows) {
    const bool diag = walk.diag;
    walk.next();
    store();
    __syncthreads();
    if (walk.rows) fetch(walk);
    if (halves && diag) {
      acc += acc;
      halves = false;
    }
    if (tv) {
#pragma unroll
      for (int st = 0; st < ROWS / (4 * KS); ++st) {
        const double2 *trow = tile + (4 * (ks + KS * st) + lk) * LD;
        const double2 av = trow[acol];
        const double2 bv = trow[bcol];
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(im ? av.y : av.x, im ? bv.y : bv.x, acc, 0, 0, 0);
      }
    }
    __syncthreads();
  }
  if (halves) acc += acc;
  // every wave's 16 x 16 sums to LDS (the loop's last __syncthreads freed the
  // tile); element (i, j) of the block, i = 4 v + lk, j = li, sits at
  // [v * 64 + lane] of the wave's 256 doubles
  double *red = reinterpret_cast<double *>(tile);
  if (tv) {
#pragma unroll
    for (int v = 0; v < 4; ++v) red[size_t(t * KS + ks) * 256 + v * 64 + lane] = acc[v];
  }
  __syncthreads();
  double2 *out = partial + size_t(blockIdx.x) * kl * kr;
  for (int e = tid; e < M8 * 64; e += kGramThreads) {
    const int tb = e / 64, c = (e % 64) / 8, r = e % 8;
    const int i = 8 * tb + c;
    if (i >= kl || r >= kr) continue;
    auto O = [&](int k, int ii, int jj) {
      return red[size_t(tb * KS + k) * 256 + (ii / 4) * 64 + (jj + 16 * (ii % 4))];
    };
    double gr = 0.0, gi = 0.0;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      gr += O(k, c, r) + O(k, c + 8, r + 8);
      gi += O(k, c, r + 8) - O(k, c + 8, r);
    }
    out[i + size_t(kl) * r] = make_double2(gr, gi);
  }
}

// Sum of nparts partial results per element: one wavefront per element, each
// lane summing a strided subset, then a shuffle tree (fixed order).
__global__ __launch_bounds__(256) void k_reduce_partials(const double2 *__restrict__ partial,
                                                         int nparts, int nelem,
                                                         double2 *__restrict__ out) {
  const int lane = threadIdx.x & 63;
  const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (e >= nelem) return;
  double sx = 0.0, sy = 0.0;
  for (int b = lane; b < nparts; b += 64) {
    const double2 v = partial[size_t(b) * nelem + e];
    sx += v.x;
    sy += v.y;
  }
  for (int off = 32; off > 0; off >>= 1) {
    sx += __shfl_down(sx, off);
    sy += __shfl_down(sy, off);
  }
  if (lane == 0) out[e] = make_double2(sx, sy);
}

constexpr int kCombRows = 32;
constexpr int kCombThreads = 256;
constexpr int kCombMaxIn = 64;
constexpr int kCombGroups = 8;  // output groups per workgroup (kCombThreads / kCombRows)
constexpr int kCombMaxOut = 48;

// out_j = sum_i in_i C(i, j) (+ beta_j out_j), row by row.  A workgroup stages
// C (nin x nout, padded to kCombGroups * JPT columns) once in LDS, then walks
// tiles of kCombRows rows: the tile of every input column goes to LDS, and
// thread t forms, for row t % kCombRows, the JPT outputs of group
// t / kCombRows.  All loads of a tile finish before any of its outputs is
// written, so an output may alias an input.
template <int JPT>
__global__ __launch_bounds__(kCombThreads) void k_combine(const ColDesc *__restrict__ descs, int nin,
                                                          int nout, const double2 *__restrict__ cm,
                                                          const double2 *__restrict__ beta, int64_t d) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int NP = kCombGroups * JPT;
  // input elements per thread per tile: all issued before any wait, the next
  // tile's while this one is combined; each an adjacent row pair of one
  // column (16-byte accesses for complex64 and complex128 alike)
  constexpr int HALF = kCombRows / 2;
  constexpr int PMAX = HALF * kCombMaxIn / kCombThreads;
  double2 *sc = reinterpret_cast<double2 *>(smem);  // [nin][NP]
  double2 *tin = sc + size_t(nin) * NP;              // [nin][kCombRows]
  const int tid = threadIdx.x;
  const int row = tid % kCombRows;
  const int grp = tid / kCombRows;
  for (int e = tid; e < nin * NP; e += kCombThreads) {
    const int i = e / NP, j = e % NP;
    sc[e] = j < nout ? cm[size_t(nout) * i + j] : make_double2(0.0, 0.0);
  }
  // element p of this thread: row pair e % HALF of input column e / HALF
  const void *pa[PMAX];
  const void *pb[PMAX];
  int pf[PMAX];
#pragma unroll
  for (int p = 0; p < PMAX; ++p) {
    const int e = tid + kCombThreads * p;
    pa[p] = nullptr;
    pb[p] = nullptr;
    pf[p] = 0;
    if (e < HALF * nin) {
      const ColDesc &dc = descs[e / HALF];
      pa[p] = dc.a;
      pb[p] = dc.b;
      pf[p] = dc.fmt;
    }
  }
  double2 va[PMAX][2], vb[PMAX][2];
  auto fetch = [&](int64_t rb) {
#pragma unroll
    for (int p = 0; p < PMAX; ++p) {
      const int64_t r = rb + 2 * ((tid + kCombThreads * p) % HALF);
      if (pa[p] != nullptr && r < d) {
        ld_col2(pa[p], pf[p], r, r + 1 < d, va[p][0], va[p][1]);
        if (pb[p] != nullptr) ld_col2(pb[p], pf[p], r, r + 1 < d, vb[p][0], vb[p][1]);
      }
    }
  };
  const int64_t ntile = (d + kCombRows - 1) / kCombRows;
  if (int64_t(blockIdx.x) < ntile) fetch(int64_t(blockIdx.x) * kCombRows);
  for (int64_t tb = blockIdx.x; tb < ntile; tb += gridDim.x) {
    const int64_t rb = tb * kCombRows;
    const int nr = int(d - rb < kCombRows ? d - rb : kCombRows);
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PMAX; ++p) {
      if (pa[p] == nullptr) continue;
      const int e = tid + kCombThreads * p;
      const int r = 2 * (e % HALF), c = e / HALF;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (r + h >= nr) continue;
        double2 v = va[p][h];
        if (pb[p] != nullptr) {
          const ColDesc &dc = descs[c];
          v.x -= dc.sig_re * vb[p][h].x - dc.sig_im * vb[p][h].y;
          v.y -= dc.sig_re * vb[p][h].y + dc.sig_im * vb[p][h].x;
        }
        tin[c * kCombRows + r + h] = v;
      }
    }
    __syncthreads();
    if (tb + gridDim.x < ntile) fetch((tb + gridDim.x) * kCombRows);
    if (row < nr) {
      double ax[JPT], ay[JPT];
#pragma unroll
      for (int q = 0; q < JPT; ++q) ax[q] = ay[q] = 0.0;
      const double2 *cg = sc + grp * JPT;
#pragma unroll 4
      for (int i = 0; i < nin; ++i) {
        const double2 a = tin[i * kCombRows + row];
#pragma unroll
        for (int q = 0; q < JPT; ++q) {
          const double2 c = cg[i * NP + q];
          ax[q] = fma(a.x, c.x, ax[q]);
          ax[q] = fma(-a.y, c.y, ax[q]);
          ay[q] = fma(a.x, c.y, ay[q]);
          ay[q] = fma(a.y, c.x, ay[q]);
        }
      }
#pragma unroll
      for (int q = 0; q < JPT; ++q) {
        const int j = grp * JPT + q;
        if (j < nout) {
          const ColDesc &od = descs[nin + j];
          void *o = const_cast<Dbl2 *>(od.a);
          const int64_t r = rb + row;
          double ox = ax[q], oy = ay[q];
          if (beta != nullptr) {
            const double2 bj = beta[j];
            const double2 ov = ld_col(o, od.fmt, r);
            ox += bj.x * ov.x - bj.y * ov.y;
            oy += bj.x * ov.y + bj.y * ov.x;
          }
          st_col(o, od.fmt, r, make_double2(ox, oy));
        }
      }
    }
  }
}

// a_k += v_k C(i, .) over the JN outputs (c: C(i, 0), C stored by rows of JN).
template <int JN, int RPL>
__device__ __forceinline__ void add_products(const double2 (&v)[RPL], const double2 *__restrict__ c,
                                             double (&ax)[RPL][JN], double (&ay)[RPL][JN]) {
#pragma unroll
  for (int q = 0; q < JN; ++q) {
    const double2 f = c[q];
#pragma unroll
    for (int k = 0; k < RPL; ++k) {
      ax[k][q] = fma(v[k].x, f.x, ax[k][q]);
      ax[k][q] = fma(-v[k].y, f.y, ax[k][q]);
      ay[k][q] = fma(v[k].x, f.y, ay[k][q]);
      ay[k][q] = fma(v[k].y, f.x, ay[k][q]);
    }
  }
}

// The same over complex128 inputs at the entries `at`: UNR inputs are loaded while the
// UNR before them are used.
template <int JN, int RPL, int UNR>
__device__ __forceinline__ void plain_inputs(const ColDesc *__restrict__ descs, int nin,
                                             const double2 *__restrict__ cm, const int64_t (&at)[2],
                                             double (&ax)[RPL][JN], double (&ay)[RPL][JN]) {
  double2 v[UNR][RPL], next[UNR][RPL];
  auto load = [&](int i, double2(&w)[UNR][RPL]) {
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      const double2 *a = reinterpret_cast<const double2 *>(descs[i + u < nin ? i + u : nin - 1].a);
#pragma unroll
      for (int k = 0; k < RPL; ++k) w[u][k] = a[at[k]];
    }
  };
  load(0, v);
  for (int i = 0; i < nin; i += UNR) {
    load(i + UNR, next);
    __builtin_amdgcn_sched_barrier(0);  // else the loads sink to their uses
#pragma unroll
    for (int u = 0; u < UNR; ++u)
      if (i + u < nin) add_products<JN, RPL>(v[u], cm + size_t(JN) * (i + u), ax, ay);
#pragma unroll
    for (int u = 0; u < UNR; ++u)
#pragma unroll
      for (int k = 0; k < RPL; ++k) v[u][k] = next[u][k];
  }
}

// The combine for narrow outputs (nout <= 16; also 33..48, where the LDS
// kernel's staging would exceed 64 KB per workgroup), without LDS: a wavefront
// owns 64 * RPL consecutive rows and every output column of them, so the
// coefficients C(i, j) are wavefront-uniform (scalar loads, no LDS traffic)
// and each input element is read once, by one lane.  With RPL = 2 a lane owns
// two adjacent rows, so every load and store is 16 bytes wide whatever the
// storage (one complex64 pair, or two complex128 halves of a 32-byte run) and a
// wavefront reads 2 KB (complex128) or 1 KB (complex64) contiguous per column:
// with one complex64 row per lane the loads were 8 bytes wide and the kernel
// moved half the bytes per instruction.  With RPL = 1 a lane owns one row.
// JN, the output width the registers hold, is the smallest of 4, 8, 12, 16, 48
// that covers nout: spare accumulators cost occupancy.  C comes by rows of JN, zeros
// past nout, so an input's coefficients are a few wide scalar loads without a branch
// (by columns they were one load and one branch an output: two iterations of an 8 + 2
// column solve at NN = 9 took 51 ms, now 48).  All inputs of a row are read before any
// output of it is written, so outputs may alias inputs.  Columns start 256-byte
// aligned and row pairs start at even rows, so the 16-byte accesses are aligned.
//
// PLAIN: every column is complex128.  A lane's rows are then 64 apart (each load of a
// wavefront is one 1 KB run) and UNR inputs are loaded while the UNR before them are
// used; with a branch on each column's format the loads of one input waited for the
// products of the one before.  UNR is what measured fastest, loads in flight against
// wavefronts a SIMD: 8, 4 and 1 inputs for 4, 8 and 12 outputs.
template <int JN, int RPL, int UNR, bool PLAIN>
__global__ __launch_bounds__(256) void k_combine_w(const ColDesc *__restrict__ descs, int nin, int nout,
                                                   const double2 *__restrict__ cm,
                                                   const double2 *__restrict__ beta, int64_t d) {
  static_assert(RPL == 1 || RPL == 2, "one row or an adjacent row pair per lane");
  const int lane = threadIdx.x & 63;
  const int64_t wave = int64_t(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t stride = int64_t(gridDim.x) * 4 * 64 * RPL;
  for (int64_t rb = wave * 64 * RPL; rb < d; rb += stride) {
    const int64_t r0 = rb + (PLAIN ? 1 : RPL) * lane;  // this lane's first row
    const bool ok0 = r0 < d, ok1 = RPL == 2 && r0 + (PLAIN ? 64 : 1) < d;
    double ax[RPL][JN], ay[RPL][JN];
#pragma unroll
    for (int k = 0; k < RPL; ++k)
#pragma unroll
      for (int q = 0; q < JN; ++q) ax[k][q] = ay[k][q] = 0.0;
    if constexpr (PLAIN) {
      // rows past the end read row 0 and are not written
      const int64_t at[2] = {ok0 ? r0 : 0, ok1 ? r0 + 64 : 0};
      plain_inputs<JN, RPL, UNR>(descs, nin, cm, at, ax, ay);
    } else {
#pragma unroll UNR
      for (int i = 0; i < nin; ++i) {
        const ColDesc dc = descs[i];
        double2 v[RPL];
#pragma unroll
        for (int k = 0; k < RPL; ++k) v[k] = make_double2(0.0, 0.0);
        if (ok0) {
          if constexpr (RPL == 2) {
            col_values2(dc, r0, ok1, v[0], v[RPL - 1]);
          } else {
            v[0] = col_value(dc, r0);
          }
        }
        add_products<JN, RPL>(v, cm + size_t(JN) * i, ax, ay);
      }
    }
    if (!ok0) continue;
#pragma unroll
    for (int q = 0; q < JN; ++q) {
      if (q < nout) {
        const ColDesc &od = descs[nin + q];
        void *o = const_cast<Dbl2 *>(od.a);
        double2 out[RPL];
#pragma unroll
        for (int k = 0; k < RPL; ++k) out[k] = make_double2(ax[k][q], ay[k][q]);
        if (beta != nullptr) {
          const double2 bq = beta[q];
          double2 ov[RPL];
          if constexpr (PLAIN) {
#pragma unroll
            for (int k = 0; k < RPL; ++k)
              ov[k] = static_cast<const double2 *>(o)[k == 0 || ok1 ? r0 + 64 * k : r0];
          } else if constexpr (RPL == 2) {
            ld_col2(o, od.fmt, r0, ok1, ov[0], ov[RPL - 1]);
          } else {
            ov[0] = ld_col(o, od.fmt, r0);
          }
#pragma unroll
          for (int k = 0; k < RPL; ++k) {
            out[k].x += bq.x * ov[k].x - bq.y * ov[k].y;
            out[k].y += bq.x * ov[k].y + bq.y * ov[k].x;
          }
        }
        if constexpr (PLAIN) {
          double2 *w = static_cast<double2 *>(o) + r0;
          w[0] = out[0];
          if constexpr (RPL == 2) {
            if (ok1) w[64] = out[1];
          }
        } else if constexpr (RPL == 2) {
          st_col2(o, od.fmt, r0, ok1, out[0], out[RPL - 1]);
        } else {
          st_col(o, od.fmt, r0, out[0]);
        }
      }
    }
  }
}

// The combine on exchange-(anti)symmetric columns (M x M matrices, X(q, p) = sign
// X(p, q)): a workgroup reads every input on its 32 x 32 tile (ta <= tb) only, forms
// the outputs there and writes them to the tile and, transposed through LDS, to its
// mirror: half the bytes of the inputs, all of the outputs'.  A thread owns two
// entries of the tile and every output (coefficients wave-uniform, as in
// k_combine_w); it reads all its inputs before it writes, and nobody reads a mirror
// tile, so outputs may alias inputs.  Each output's mirror is the same value: the
// outputs are exactly (anti)symmetric, as the inputs are.  HBM-bound: 5.0 TB/s at 10
// outputs of NN = 11 (two iterations of an 8 + 2 column solve: 34.7 -> 29.9 ms of
// these), 4.5 at 4 outputs of NN = 21 (an order-4 inner solve: 16.8 -> 15.5 ms).
template <int JN, int UNR, bool PLAIN>
__global__ __launch_bounds__(512) void k_combine_sym(const ColDesc *__restrict__ descs, int nin, int nout,
                                                     const double2 *__restrict__ cm,
                                                     const double2 *__restrict__ beta, int m, int nblk, int sign) {
  int ta, tb;
  if (!sym_tile(m, nblk, ta, tb)) return;
  __shared__ double2 tile[2][kSymT][kSymT + 1];
  const int tx = threadIdx.x, ty = threadIdx.y;
  const int p = ta * kSymT + tx, q0 = tb * kSymT + ty;  // entries (p, q0) and (p, q0 + 16)
  const bool ok[2] = {p < m && q0 < m, p < m && q0 + 16 < m};
  const int64_t at[2] = {p + int64_t(m) * q0, p + int64_t(m) * (q0 + 16)};
  double ax[2][JN], ay[2][JN];
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int j = 0; j < JN; ++j) ax[k][j] = ay[k][j] = 0.0;
  if constexpr (PLAIN) {
    // entries past the edge read entry 0 and are not written
    const int64_t from[2] = {ok[0] ? at[0] : 0, ok[1] ? at[1] : 0};
    plain_inputs<JN, 2, UNR>(descs, nin, cm, from, ax, ay);
  } else {
#pragma unroll UNR
    for (int i = 0; i < nin; ++i) {
      const ColDesc dc = descs[i];
      double2 v[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        v[k] = make_double2(0.0, 0.0);
        if (ok[k]) v[k] = col_value(dc, at[k]);
      }
      add_products<JN, 2>(v, cm + size_t(JN) * i, ax, ay);
    }
  }
  const int pm = tb * kSymT + tx, qm = ta * kSymT + ty;  // mirror entries (pm, qm) and (pm, qm + 16)
  const double sg = double(sign);
#pragma unroll
  for (int j = 0; j < JN; ++j) {
    if (j < nout) {
      const ColDesc &od = descs[nin + j];
      void *o = const_cast<Dbl2 *>(od.a);
      double2 (*t)[kSymT + 1] = tile[j & 1];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        double2 r = make_double2(ax[k][j], ay[k][j]);
        if (beta != nullptr && ok[k]) {
          const double2 b = beta[j], ov = ld_col(o, od.fmt, at[k]);
          r.x += b.x * ov.x - b.y * ov.y;
          r.y += b.x * ov.y + b.y * ov.x;
        }
        if (ok[k]) st_col(o, od.fmt, at[k], r);
        t[ty + 16 * k][tx] = r;
      }
      if (ta != tb) {
        __syncthreads();  // the other buffer's readers are past the previous one
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const double2 r = t[tx][ty + 16 * k];
          if (pm < m && qm + 16 * k < m)
            st_col(o, od.fmt, pm + int64_t(m) * (qm + 16 * k), make_double2(sg * r.x, sg * r.y));
        }
      }
    }
  }
}

constexpr int kDotThreads = 256;
constexpr int kDotBlocks = 512;
constexpr int kDotMaxCols = 64;

// Per column: |a|^2, conj(a) b (re, im), |b|^2 -> 4 doubles per column per block.
__global__ __launch_bounds__(kDotThreads) void k_coldots(const ColDesc *__restrict__ descs, int k,
                                                         int64_t d, double *__restrict__ partial) {
  __shared__ double red[kDotThreads / 64][4];
  const int tid = threadIdx.x;
  for (int j = 0; j < k; ++j) {
    const ColDesc ca = descs[j];
    const ColDesc cb = descs[k + j];
    double aa = 0.0, abr = 0.0, abi = 0.0, bb = 0.0;
    for (int64_t r = int64_t(blockIdx.x) * kDotThreads + tid; r < d; r += int64_t(gridDim.x) * kDotThreads) {
      const double2 a = col_value(ca, r);
      const double2 b = cb.a != nullptr ? col_value(cb, r) : make_double2(0.0, 0.0);
      aa += a.x * a.x + a.y * a.y;
      abr += a.x * b.x + a.y * b.y;
      abi += a.x * b.y - a.y * b.x;
      bb += b.x * b.x + b.y * b.y;
    }
    for (int off = 32; off > 0; off >>= 1) {
      aa += __shfl_down(aa, off);
      abr += __shfl_down(abr, off);
      abi += __shfl_down(abi, off);
      bb += __shfl_down(bb, off);
    }
    if ((tid & 63) == 0) {
      red[tid >> 6][0] = aa;
      red[tid >> 6][1] = abr;
      red[tid >> 6][2] = abi;
      red[tid >> 6][3] = bb;
    }
    __syncthreads();
    if (tid < 4) {
      double s = 0.0;
      for (int w = 0; w < kDotThreads / 64; ++w) s += red[w][tid];
      partial[(size_t(blockIdx.x) * k + j) * 4 + tid] = s;
    }
    __syncthreads();
  }
}

// The residual step of GPLMR (gplmr.F90:324-341) for column j = blockIdx.y
// after the scaling s_j = 1 / ||X_j|| and the Rayleigh quotient E_j are known:
// X_j <- s_j X_j, AX_j <- s_j AX_j, W_j = AX_j - E_j X_j (scaled), one pass over
// X and AX (row pairs, 16-byte accesses), with each workgroup's partial sum of
// |W_j|^2 (in FP64, before W is rounded to its storage) in
// partial[blockIdx.x * nev + j].  descs: X (nev), AX (nev), W (nev).
__global__ __launch_bounds__(256) void k_resid(const ColDesc *__restrict__ descs, int nev,
                                               const double *__restrict__ sc, const double2 *__restrict__ ev,
                                               int64_t d, int64_t rows_per_block, double *__restrict__ partial) {
  const int j = blockIdx.y;
  const ColDesc cx = descs[j], cax = descs[nev + j], cw = descs[2 * nev + j];
  const double s = sc[j];
  const double2 f = ev[j];
  const int64_t r0 = int64_t(blockIdx.x) * rows_per_block;
  const int64_t r1 = r0 + rows_per_block < d ? r0 + rows_per_block : d;
  double acc = 0.0;
  for (int64_t r = r0 + 2 * int64_t(threadIdx.x); r < r1; r += 2 * int64_t(blockDim.x)) {
    const bool two = r + 1 < r1;
    double2 x[2], a[2], w[2];
    ld_col2(cx.a, cx.fmt, r, two, x[0], x[1]);
    ld_col2(cax.a, cax.fmt, r, two, a[0], a[1]);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      x[h].x *= s;
      x[h].y *= s;
      a[h].x *= s;
      a[h].y *= s;
      w[h].x = a[h].x - (f.x * x[h].x - f.y * x[h].y);
      w[h].y = a[h].y - (f.x * x[h].y + f.y * x[h].x);
    }
    st_col2(const_cast<Dbl2 *>(cx.a), cx.fmt, r, two, x[0], x[1]);
    st_col2(const_cast<Dbl2 *>(cax.a), cax.fmt, r, two, a[0], a[1]);
    st_col2(const_cast<Dbl2 *>(cw.a), cw.fmt, r, two, w[0], w[1]);
    acc += w[0].x * w[0].x + w[0].y * w[0].y;
    if (two) acc += w[1].x * w[1].x + w[1].y * w[1].y;
  }
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off);
  __shared__ double red[4];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) partial[size_t(blockIdx.x) * nev + j] = red[0] + red[1] + red[2] + red[3];
}

__global__ __launch_bounds__(256) void k_reduce_real(const double *__restrict__ partial, int nparts,
                                                     int nelem, double *__restrict__ out) {
  const int lane = threadIdx.x & 63;
  const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (e >= nelem) return;
  double s = 0.0;
  for (int b = lane; b < nparts; b += 64) s += partial[size_t(b) * nelem + e];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off);
  if (lane == 0) out[e] = s;
}

// Philox4x32-10 (Salmon et al., SC'11) and Box-Muller.
__device__ __forceinline__ void philox10(uint32_t c[4], uint32_t k0, uint32_t k1) {
  const uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u, W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint64_t p0 = uint64_t(M0) * c[0];
    const uint64_t p1 = uint64_t(M1) * c[2];
    const uint32_t hi0 = uint32_t(p0 >> 32), lo0 = uint32_t(p0);
    const uint32_t hi1 = uint32_t(p1 >> 32), lo1 = uint32_t(p1);
    const uint32_t n0 = hi1 ^ c[1] ^ k0;
    const uint32_t n2 = hi0 ^ c[3] ^ k1;
    c[0] = n0;
    c[1] = lo1;
    c[2] = n2;
    c[3] = lo0;
    k0 += W0;
    k1 += W1;
  }
}

__global__ void k_fill_gaussian(double2 *__restrict__ x, int64_t n, uint64_t seed, uint32_t col,
                                uint32_t sid) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t c[4] = {uint32_t(i), uint32_t(uint64_t(i) >> 32), col, sid};
  philox10(c, uint32_t(seed), uint32_t(seed >> 32));
  // 53-bit uniforms in (0, 1]
  const double u1 = (double((uint64_t(c[0]) << 21) ^ (c[1] >> 11)) + 1.0) * (1.0 / 9007199254740992.0);
  const double u2 = double((uint64_t(c[2]) << 21) ^ (c[3] >> 11)) * (1.0 / 9007199254740992.0);
  const double rad = sqrt(-2.0 * log(u1));
  const double ang = 6.283185307179586 * u2;
  double sn, cs;
  sincos(ang, &sn, &cs);
  const double s = 0.7071067811865476;
  x[i] = make_double2(rad * cs * s, rad * sn * s);
}

// Y = (X + sign X^T)/2 on the M x M matrix, tiles of 32 x 32 above the diagonal (Y may be X).
__global__ void k_singlet(const double2 *x, double2 *y, int64_t m, double sign) {
  __shared__ double2 ta[32][33], tb[32][33];
  const int64_t bi = blockIdx.x, bj = blockIdx.y;
  if (bi > bj) return;
  const int tx = threadIdx.x, ty = threadIdx.y;  // 32 x 8
  for (int r = ty; r < 32; r += 8) {
    const int64_t i = bi * 32 + tx, j = bj * 32 + r;  // element (i, j): x[i + m j]
    ta[r][tx] = (i < m && j < m) ? x[i + m * j] : make_double2(0, 0);
    const int64_t i2 = bj * 32 + tx, j2 = bi * 32 + r;
    tb[r][tx] = (i2 < m && j2 < m) ? x[i2 + m * j2] : make_double2(0, 0);
  }
  __syncthreads();
  for (int r = ty; r < 32; r += 8) {
    const int64_t i = bi * 32 + tx, j = bj * 32 + r;
    const double2 a = ta[r][tx], b = tb[tx][r];  // b = x[j + m i]
    const double2 s = make_double2(0.5 * (a.x + sign * b.x), 0.5 * (a.y + sign * b.y));
    if (i < m && j < m) y[i + m * j] = s;
    const int64_t i2 = bj * 32 + tx, j2 = bi * 32 + r;
    const double2 a2 = tb[r][tx], b2 = ta[tx][r];
    const double2 s2 = make_double2(0.5 * (a2.x + sign * b2.x), 0.5 * (a2.y + sign * b2.y));
    if (i2 < m && j2 < m) y[i2 + m * j2] = s2;
  }
}

__global__ void k_to_single(const double2 *__restrict__ x, float2 *__restrict__ y, int64_t n) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) y[i] = make_float2(float(x[i].x), float(x[i].y));
}

__global__ void k_to_double(const float2 *__restrict__ x, double2 *__restrict__ y, int64_t n) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) y[i] = make_double2(double(x[i].x), double(x[i].y));
}

// ---- one-electron (He+) operator and the small block products of its Lanczos --
// H1 x = s2 tau3D x + c1 vn o x on vectors of M = NN^3 entries (i fastest):
// KEMULT1 (hammod.F90:71-134) with the 1/SCALE^2 of the kinetic matrix folded
// into s2 and POTENTIAL1 (hammod.F90:432-498) / SCALE into c1 vn.  One thread
// per entry of one column; the column (at most 315 KB at NN = 27) stays in L2.
__global__ __launch_bounds__(256) void k_h1(const double2 *__restrict__ x, double2 *__restrict__ y, int nn,
                                            int64_t m, int ncols, const double *__restrict__ vn,
                                            MatvecCoef cf) {
  const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= m * ncols) return;
  const int64_t c = e / m, p = e % m;
  const int i = int(p % nn), j = int((p / nn) % nn), k = int(p / (int64_t(nn) * nn));
  const double2 *xc = x + c * m;
  const int64_t base_i = p - i, base_j = p - int64_t(nn) * j, base_k = p - int64_t(nn) * nn * k;
  double sr = 0.0, si = 0.0;
  for (int l = 0; l < nn; ++l) {
    const double ti = tau_rt(l - i), tj = tau_rt(l - j), tk = tau_rt(l - k);
    const double2 a = xc[base_i + l], b = xc[base_j + int64_t(nn) * l], d = xc[base_k + int64_t(nn) * nn * l];
    sr += ti * a.x + tj * b.x + tk * d.x;
    si += ti * a.y + tj * b.y + tk * d.y;
  }
  const double2 xv = xc[p];
  const double v = vn[p];
  double2 o;
  o.x = cf.s2_re * sr - cf.s2_im * si + v * (cf.c1_re * xv.x - cf.c1_im * xv.y);
  o.y = cf.s2_re * si + cf.s2_im * sr + v * (cf.c1_re * xv.y + cf.c1_im * xv.x);
  y[e] = o;
}

// out(i, j) = sum_r op(A_i[r]) B_j[r] over m rows, op = identity (the
// bilinear product of the complex-symmetric Lanczos, MPIDOT) or conj (the
// Hermitian one, MPIHERMDOT); A (m x p) and B (m x q) column-major with
// leading dimension m, out (p x q) column-major.  One workgroup per output
// element, a fixed-order reduction.
__global__ __launch_bounds__(256) void k_small_dots(const double2 *__restrict__ a, int p,
                                                    const double2 *__restrict__ b, int q, int64_t m,
                                                    int herm, double2 *__restrict__ out) {
  const int i = blockIdx.x % p, j = blockIdx.x / p;
  const double2 *ai = a + int64_t(i) * m;
  const double2 *bj = b + int64_t(j) * m;
  const double s = herm ? -1.0 : 1.0;
  double sr = 0.0, si = 0.0;
  for (int64_t r = threadIdx.x; r < m; r += blockDim.x) {
    const double2 u = ai[r], v = bj[r];
    const double uy = s * u.y;
    sr += u.x * v.x - uy * v.y;
    si += u.x * v.y + uy * v.x;
  }
  __shared__ double red[2][256];
  red[0][threadIdx.x] = sr;
  red[1][threadIdx.x] = si;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (int(threadIdx.x) < off) {
      red[0][threadIdx.x] += red[0][threadIdx.x + off];
      red[1][threadIdx.x] += red[1][threadIdx.x + off];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) out[i + int64_t(p) * j] = make_double2(red[0][0], red[1][0]);
}

// Y = beta Y + A C for A (m x p, leading dimension m), C (p x q, leading
// dimension p), Y (m x q, leading dimension m); beta 0 or 1.  One thread per
// element of Y.
__global__ __launch_bounds__(256) void k_small_lincomb(const double2 *__restrict__ a, int p,
                                                       const double2 *__restrict__ cm, int q, int64_t m,
                                                       int beta, double2 *__restrict__ y) {
  const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= m * q) return;
  const int64_t r = e % m;
  const int j = int(e / m);
  double sr = 0.0, si = 0.0;
  for (int i = 0; i < p; ++i) {
    const double2 u = a[r + m * i], c = cm[i + int64_t(p) * j];
    sr += u.x * c.x - u.y * c.y;
    si += u.x * c.y + u.y * c.x;
  }
  if (beta) {
    const double2 o = y[e];
    sr += o.x;
    si += o.y;
  }
  y[e] = make_double2(sr, si);
}

// Two-electron vector of rank <= K over one-electron orbitals:
// out(p, q) = sum_b T(p, b) X(q, b), p electron 1 (fastest), q electron 2;
// T and X are M x K column-major.  One thread per element.
__global__ __launch_bounds__(256) void k_lowrank(const double2 *__restrict__ t, const double2 *__restrict__ x,
                                                 double2 *__restrict__ out, int64_t m, int k) {
  const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= m * m) return;
  const int64_t p = e % m, q = e / m;
  double re = 0.0, im = 0.0;
  for (int b = 0; b < k; ++b) {
    const double2 tv = t[p + m * b];
    const double2 xv = x[q + m * b];
    re += tv.x * xv.x - tv.y * xv.y;
    im += tv.x * xv.y + tv.y * xv.x;
  }
  out[e] = make_double2(re, im);
}

// W = Y X (or Y conj(X)) for the M x M matrix Y (a two-electron vector,
// column q = electron-2 index contiguous) and the M x K orbital block X:
// each thread owns one row p and all K outputs; X(q, .) is the same for the
// whole workgroup (L1-resident), Y is read once, coalesced along p.
template <int KM>
__global__ __launch_bounds__(256) void k_ywx(const double2 *__restrict__ y, const double2 *__restrict__ x,
                                             double2 *__restrict__ w, int64_t m, int k, int conj_x) {
  const int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (p >= m) return;
  double re[KM], im[KM];
#pragma unroll
  for (int b = 0; b < KM; ++b) re[b] = im[b] = 0.0;
  const double sx = conj_x ? -1.0 : 1.0;
  for (int64_t q = 0; q < m; ++q) {
    const double2 yv = y[p + m * q];
#pragma unroll
    for (int b = 0; b < KM; ++b) {
      if (b < k) {
        const double2 xv = x[q + m * b];
        const double xi = sx * xv.y;
        re[b] += yv.x * xv.x - yv.y * xi;
        im[b] += yv.x * xi + yv.y * xv.x;
      }
    }
  }
#pragma unroll
  for (int b = 0; b < KM; ++b)
    if (b < k) w[p + m * b] = make_double2(re[b], im[b]);
}

}  // namespace

hipError_t launch_lowrank(const Dbl2 *t, const Dbl2 *x, Dbl2 *out, int64_t m, int k, hipStream_t s) {
  if (k < 1 || m < 1) return hipErrorInvalidValue;
  const int64_t n = m * m;
  hipLaunchKernelGGL(k_lowrank, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s,
                     reinterpret_cast<const double2 *>(t), reinterpret_cast<const double2 *>(x),
                     reinterpret_cast<double2 *>(out), m, k);
  return hipGetLastError();
}

hipError_t launch_ywx(const Dbl2 *y, const Dbl2 *x, Dbl2 *w, int64_t m, int k, int conj_x, hipStream_t s) {
  if (k < 1 || k > 32 || m < 1) return hipErrorInvalidValue;
  const dim3 grid(unsigned((m + 255) / 256)), block(256);
  const double2 *yy = reinterpret_cast<const double2 *>(y), *xx = reinterpret_cast<const double2 *>(x);
  double2 *ww = reinterpret_cast<double2 *>(w);
  if (k <= 16)
    hipLaunchKernelGGL(k_ywx<16>, grid, block, 0, s, yy, xx, ww, m, k, conj_x);
  else
    hipLaunchKernelGGL(k_ywx<32>, grid, block, 0, s, yy, xx, ww, m, k, conj_x);
  return hipGetLastError();
}

int gram_blocks() { return kGramBlocks; }

size_t gram_partial_elems(int kl, int kr) { return size_t(kGramBlocks) * kl * kr; }

namespace {
// Workgroups of a Gram kernel that fit on the device at once (LDS sets it: 3 or 4
// per CU), capped at kGramBlocks, a multiple of the 8 XCDs.  A grid of exactly that
// many runs in one wave of workgroups; 1024 workgroups at 3 per CU would leave a
// second round on a third of the chip.
int resident_grid(const void *kernel, std::atomic<int> &cached) {
  int grid = cached.load(std::memory_order_acquire);
  if (grid != 0) return grid;
  std::lock_guard<std::mutex> lk(g_setup_mu);
  grid = cached.load(std::memory_order_acquire);
  if (grid != 0) return grid;
  int dev = 0, cus = 0, per_cu = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kGramThreads, 0) != hipSuccess || cus < 1 ||
      per_cu < 1)
    return kGramBlocks;
  grid = cus * per_cu < kGramBlocks ? cus * per_cu : kGramBlocks;
  grid = grid < 8 ? 8 : grid / 8 * 8;
  cached.store(grid, std::memory_order_release);
  return grid;
}

// The packed narrow Gram (on unless DEX_GRAM_PK=0, read once).
bool gram_pk_on() {
  static const bool on = [] {
    const char *v = std::getenv("DEX_GRAM_PK");
    return !(v && std::atoi(v) == 0);
  }();
  return on;
}

// Row-tile heights: 64 in the packed Gram (5-7% less time than 32 on whole NN=21
// block-16 solves, 128 1-3% less); 32 for one-tile Grams, 16 elsewhere (gram_mfma_rows).
constexpr int kPkRows = 64;

template <int M8, bool TRI>
int gram_pk_grid() {
  static std::atomic<int> cached{0};
  return resident_grid(reinterpret_cast<const void *>(&k_gram_pk<M8, kPkRows, TRI>), cached);
}

template <int M8, bool TRI>
int gram_pk_start(const ColDesc *descs, int kl, int kr, int share, int64_t d, int m, double2 *partial,
                  hipStream_t s) {
  const int grid = gram_pk_grid<M8, TRI>();
  hipLaunchKernelGGL((k_gram_pk<M8, kPkRows, TRI>), dim3(grid), dim3(kGramThreads), 0, s, descs, kl, kr, share, d,
                     m, partial);
  return grid;
}

template <int M8>
int gram_pk_launch(const ColDesc *descs, int kl, int kr, int share, int64_t d, int m, double2 *partial,
                   hipStream_t s) {
  return m > 0 ? gram_pk_start<M8, true>(descs, kl, kr, share, d, m, partial, s)
               : gram_pk_start<M8, false>(descs, kl, kr, share, d, m, partial, s);
}

template <int MA, int NB>
constexpr int gram_tall() {
  return MA == 1 && NB == 1 ? 32 : 16;
}

template <int MA, int NB, bool TRI>
int gram_grid() {
  static std::atomic<int> cached{0};
  return resident_grid(reinterpret_cast<const void *>(&k_gram_mfma<MA, NB, gram_tall<MA, NB>(), TRI>), cached);
}

template <int MA, int NB>
void gram_grids() {
  (void)gram_grid<MA, NB, false>();
  (void)gram_grid<MA, NB, true>();
}

template <int MA>
void gram_grids_nb() {
  gram_grids<MA, 1>();
  gram_grids<MA, 2>();
  gram_grids<MA, 3>();
  gram_grids<MA, 4>();
  gram_grids<MA, 5>();
  gram_grids<MA, 6>();
  gram_grids<MA, 7>();
  gram_grids<MA, 8>();
  (void)gram_pk_grid<MA, false>();
  (void)gram_pk_grid<MA, true>();
}

template <int MA, int NB, bool TRI>
int gram_start(const ColDesc *descs, int kl, int kr, int share, int64_t d, int m, double2 *partial,
               hipStream_t s) {
  const int grid = gram_grid<MA, NB, TRI>();
  hipLaunchKernelGGL((k_gram_mfma<MA, NB, gram_tall<MA, NB>(), TRI>), dim3(grid), dim3(kGramThreads), 0, s, descs,
                     kl, kr, share, d, m, partial);
  return grid;
}

template <int MA, int NB>
int gram_launch(const ColDesc *descs, int kl, int kr, int share, int64_t d, int m, double2 *partial,
                hipStream_t s) {
  return m > 0 ? gram_start<MA, NB, true>(descs, kl, kr, share, d, m, partial, s)
               : gram_start<MA, NB, false>(descs, kl, kr, share, d, m, partial, s);
}

template <int MA>
int gram_launch_nb(int nb, const ColDesc *descs, int kl, int kr, int share, int64_t d, int m, double2 *partial,
                   hipStream_t s) {
  switch (nb) {
    case 1: return gram_launch<MA, 1>(descs, kl, kr, share, d, m, partial, s);
    case 2: return gram_launch<MA, 2>(descs, kl, kr, share, d, m, partial, s);
    case 3: return gram_launch<MA, 3>(descs, kl, kr, share, d, m, partial, s);
    case 4: return gram_launch<MA, 4>(descs, kl, kr, share, d, m, partial, s);
    case 5: return gram_launch<MA, 5>(descs, kl, kr, share, d, m, partial, s);
    case 6: return gram_launch<MA, 6>(descs, kl, kr, share, d, m, partial, s);
    case 7: return gram_launch<MA, 7>(descs, kl, kr, share, d, m, partial, s);
    default: return gram_launch<MA, 8>(descs, kl, kr, share, d, m, partial, s);
  }
}
}  // namespace

// Halves from NN = 11 on: there 290 us for a 64 x 10 Gram where all rows take 410, and the
// Grams and combinations of two iterations of an 8 + 2 column solve 53 + 53 -> 32 + 34 ms.
bool half_blocks(int64_t m) { return m >= kHalfMinM; }

hipError_t launch_gram(const ColDesc *descs, int kl, int kr, int share, int64_t d, int m, Dbl2 *partial,
                       Dbl2 *out, hipStream_t s) {
  if (kl < 1 || kr < 1 || kl > kGramMaxL || kr > kGramMaxR) return hipErrorInvalidValue;
  if (share < 0 || share > kl || share > kr) return hipErrorInvalidValue;
  const int ma = (kl + 15) / 16, nb = (kr + 15) / 16;
  double2 *pp = reinterpret_cast<double2 *>(partial);
  int nparts = 0;
  if (kr <= 8 && kl <= 32 && (share == 0 || share == kr) && gram_pk_on()) {
    switch ((kl + 7) / 8) {
      case 1: nparts = gram_pk_launch<1>(descs, kl, kr, share, d, m, pp, s); break;
      case 2: nparts = gram_pk_launch<2>(descs, kl, kr, share, d, m, pp, s); break;
      case 3: nparts = gram_pk_launch<3>(descs, kl, kr, share, d, m, pp, s); break;
      default: nparts = gram_pk_launch<4>(descs, kl, kr, share, d, m, pp, s); break;
    }
    const int nelem = kl * kr;
    hipLaunchKernelGGL(k_reduce_partials, dim3((nelem + 3) / 4), dim3(256), 0, s,
                       reinterpret_cast<const double2 *>(partial), nparts, nelem,
                       reinterpret_cast<double2 *>(out));
    return hipGetLastError();
  }
  switch (ma) {
    case 1: nparts = gram_launch_nb<1>(nb, descs, kl, kr, share, d, m, pp, s); break;
    case 2: nparts = gram_launch_nb<2>(nb, descs, kl, kr, share, d, m, pp, s); break;
    case 3: nparts = gram_launch_nb<3>(nb, descs, kl, kr, share, d, m, pp, s); break;
    default: nparts = gram_launch_nb<4>(nb, descs, kl, kr, share, d, m, pp, s); break;
  }
  const int nelem = kl * kr;
  hipLaunchKernelGGL(k_reduce_partials, dim3((nelem + 3) / 4), dim3(256), 0, s,
                     reinterpret_cast<const double2 *>(partial), nparts, nelem,
                     reinterpret_cast<double2 *>(out));
  return hipGetLastError();
}

namespace {
template <int JPT>
bool combine_setup() {
  static std::atomic<bool> attr{false};
  if (attr.load(std::memory_order_acquire)) return true;
  std::lock_guard<std::mutex> lk(g_setup_mu);
  if (attr.load(std::memory_order_acquire)) return true;
  if (hipFuncSetAttribute(reinterpret_cast<const void *>(&k_combine<JPT>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) != hipSuccess)
    return false;
  attr.store(true, std::memory_order_release);
  return true;
}

template <int JPT>
hipError_t combine_launch(const ColDesc *descs, int nin, int nout, const Dbl2 *c, const Dbl2 *beta,
                          int64_t d, hipStream_t s) {
  const size_t lds = (size_t(nin) * kCombGroups * JPT + size_t(kCombRows) * nin) * sizeof(double2);
  if (!combine_setup<JPT>()) return hipErrorInvalidDeviceFunction;
  const int64_t ntile = (d + kCombRows - 1) / kCombRows;
  const unsigned grid = unsigned(ntile < 2048 ? ntile : 2048);
  hipLaunchKernelGGL((k_combine<JPT>), dim3(grid), dim3(kCombThreads), lds, s, descs, nin, nout,
                     reinterpret_cast<const double2 *>(c), reinterpret_cast<const double2 *>(beta), d);
  return hipGetLastError();
}
}  // namespace

namespace {
template <bool PLAIN>
void combine_w_launch(const ColDesc *descs, int nin, int nout, const double2 *c, const double2 *beta, int64_t d,
                      hipStream_t s) {
  // one wavefront per 64 * RPL rows, at most 2048 workgroups of 4 (grid-stride beyond)
  auto grid = [d](int rpl) {
    const int64_t waves = (d + 64 * rpl - 1) / (64 * rpl);
    return dim3(unsigned((waves + 3) / 4 < 2048 ? (waves + 3) / 4 : 2048));
  };
  const dim3 b(256);
  if (nout <= 4)
    hipLaunchKernelGGL((k_combine_w<4, 2, 8, PLAIN>), grid(2), b, 0, s, descs, nin, nout, c, beta, d);
  else if (nout <= 8)
    hipLaunchKernelGGL((k_combine_w<8, 2, 4, PLAIN>), grid(2), b, 0, s, descs, nin, nout, c, beta, d);
  else if (nout <= 12)
    hipLaunchKernelGGL((k_combine_w<12, 2, PLAIN ? 1 : 2, PLAIN>), grid(2), b, 0, s, descs, nin, nout, c, beta, d);
  else if (nout <= 16)
    hipLaunchKernelGGL((k_combine_w<16, 2, PLAIN ? 1 : 2, PLAIN>), grid(2), b, 0, s, descs, nin, nout, c, beta, d);
  else
    hipLaunchKernelGGL((k_combine_w<kCombMaxOut, 1, 1, PLAIN>), grid(1), b, 0, s, descs, nin, nout, c, beta, d);
}

template <bool PLAIN>
void combine_sym_launch(const ColDesc *descs, int nin, int nout, const double2 *c, const double2 *beta, int m,
                        int sign, hipStream_t s) {
  const dim3 g(unsigned(sym_grid(m))), b(kSymT, 16);
  const int nblk = sym_blocks(m);
  if (nout <= 4)
    hipLaunchKernelGGL((k_combine_sym<4, 8, PLAIN>), g, b, 0, s, descs, nin, nout, c, beta, m, nblk, sign);
  else if (nout <= 8)
    hipLaunchKernelGGL((k_combine_sym<8, 4, PLAIN>), g, b, 0, s, descs, nin, nout, c, beta, m, nblk, sign);
  else if (nout <= 12)
    hipLaunchKernelGGL((k_combine_sym<12, PLAIN ? 1 : 2, PLAIN>), g, b, 0, s, descs, nin, nout, c, beta, m, nblk, sign);
  else
    hipLaunchKernelGGL((k_combine_sym<16, PLAIN ? 1 : 2, PLAIN>), g, b, 0, s, descs, nin, nout, c, beta, m, nblk, sign);
}
}  // namespace

hipError_t launch_combine(const ColDesc *descs, int nin, int nout, const Dbl2 *c, const Dbl2 *beta,
                          int64_t d, bool plain, hipStream_t s) {
  if (nin < 1 || nin > kCombMaxIn || nout < 1 || nout > kCombMaxOut) return hipErrorInvalidValue;
  if (nout <= 16 || nout > kCombGroups * 4) {
    const double2 *cc = reinterpret_cast<const double2 *>(c);
    const double2 *bb = reinterpret_cast<const double2 *>(beta);
    if (plain)
      combine_w_launch<true>(descs, nin, nout, cc, bb, d, s);
    else
      combine_w_launch<false>(descs, nin, nout, cc, bb, d, s);
    return hipGetLastError();
  }
  // 17..32 outputs: C and one row tile in LDS, (64 * 8 * 4 + 32 * 64) * 16 B = 64 KB at most
  switch ((nout + kCombGroups - 1) / kCombGroups) {
    case 3: return combine_launch<3>(descs, nin, nout, c, beta, d, s);
    default: return combine_launch<4>(descs, nin, nout, c, beta, d, s);
  }
}

bool combine_halves(int nout) { return nout <= 16; }

int combine_ld(int nout) {
  if (nout <= 16) return (nout + 3) / 4 * 4;
  return nout > kCombGroups * 4 ? kCombMaxOut : nout;
}

hipError_t launch_combine_sym(const ColDesc *descs, int nin, int nout, const Dbl2 *c, const Dbl2 *beta, int m,
                              int sign, bool plain, hipStream_t s) {
  if (nin < 1 || nin > kCombMaxIn || nout < 1 || !combine_halves(nout)) return hipErrorInvalidValue;
  const double2 *cc = reinterpret_cast<const double2 *>(c);
  const double2 *bb = reinterpret_cast<const double2 *>(beta);
  if (plain)
    combine_sym_launch<true>(descs, nin, nout, cc, bb, m, sign, s);
  else
    combine_sym_launch<false>(descs, nin, nout, cc, bb, m, sign, s);
  return hipGetLastError();
}

size_t coldots_partial_elems(int k) { return size_t(kDotBlocks) * k * 4; }

hipError_t launch_resid(const ColDesc *descs, int nev, const double *sc, const Dbl2 *ev, int64_t d,
                        double *partial, double *out, hipStream_t s) {
  if (nev < 1 || nev > kDotMaxCols) return hipErrorInvalidValue;
  // kDotBlocks * 4 partial sums per column at most: the coldots partial buffer holds them
  const int nb = kDotBlocks;
  int64_t rpb = (d + nb - 1) / nb;
  rpb = (rpb + 1) / 2 * 2;  // row pairs start at even rows
  hipLaunchKernelGGL(k_resid, dim3(unsigned(nb), unsigned(nev)), dim3(256), 0, s, descs, nev, sc,
                     reinterpret_cast<const double2 *>(ev), d, rpb, partial);
  hipLaunchKernelGGL(k_reduce_real, dim3((nev + 3) / 4), dim3(256), 0, s, partial, nb, nev, out);
  return hipGetLastError();
}

hipError_t launch_coldots(const ColDesc *descs, int k, int64_t d, double *partial, double *out,
                          hipStream_t s) {
  if (k < 1 || k > kDotMaxCols) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_coldots, dim3(kDotBlocks), dim3(kDotThreads), 0, s, descs, k, d, partial);
  const int nelem = k * 4;
  hipLaunchKernelGGL(k_reduce_real, dim3((nelem + 3) / 4), dim3(256), 0, s, partial, kDotBlocks,
                     nelem, out);
  return hipGetLastError();
}

hipError_t launch_fill_gaussian(Dbl2 *x, int64_t n, uint64_t seed, uint32_t col, uint32_t stream_id,
                                hipStream_t s) {
  const int bs = 256;
  hipLaunchKernelGGL(k_fill_gaussian, dim3(unsigned((n + bs - 1) / bs)), dim3(bs), 0, s,
                     reinterpret_cast<double2 *>(x), n, seed, col, stream_id);
  return hipGetLastError();
}

hipError_t launch_sym_project(const Dbl2 *x, Dbl2 *y, int64_t m, int sign, hipStream_t s) {
  const unsigned nb = unsigned((m + 31) / 32);
  hipLaunchKernelGGL(k_singlet, dim3(nb, nb), dim3(32, 8), 0, s, reinterpret_cast<const double2 *>(x),
                     reinterpret_cast<double2 *>(y), m, double(sign));
  return hipGetLastError();
}

hipError_t launch_to_single(const Dbl2 *x, void *xs, int64_t n, hipStream_t s) {
  const int bs = 256;
  hipLaunchKernelGGL(k_to_single, dim3(unsigned((n + bs - 1) / bs)), dim3(bs), 0, s,
                     reinterpret_cast<const double2 *>(x), static_cast<float2 *>(xs), n);
  return hipGetLastError();
}

hipError_t launch_h1(const Dbl2 *x, Dbl2 *y, int nn, int ncols, const double *vn, const MatvecCoef &coef,
                     hipStream_t s) {
  const int64_t m = int64_t(nn) * nn * nn;
  const int64_t n = m * ncols;
  if (ncols < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_h1, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, reinterpret_cast<const double2 *>(x),
                     reinterpret_cast<double2 *>(y), nn, m, ncols, vn, coef);
  return hipGetLastError();
}

hipError_t launch_small_dots(const Dbl2 *a, int p, const Dbl2 *b, int q, int64_t m, int herm, Dbl2 *out,
                             hipStream_t s) {
  if (p < 1 || q < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_small_dots, dim3(unsigned(int64_t(p) * q)), dim3(256), 0, s,
                     reinterpret_cast<const double2 *>(a), p, reinterpret_cast<const double2 *>(b), q, m, herm,
                     reinterpret_cast<double2 *>(out));
  return hipGetLastError();
}

hipError_t launch_small_lincomb(const Dbl2 *a, int p, const Dbl2 *c, int q, int64_t m, int beta, Dbl2 *y,
                                hipStream_t s) {
  if (p < 1 || q < 1) return hipErrorInvalidValue;
  const int64_t n = m * q;
  hipLaunchKernelGGL(k_small_lincomb, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s,
                     reinterpret_cast<const double2 *>(a), p, reinterpret_cast<const double2 *>(c), q, m, beta,
                     reinterpret_cast<double2 *>(y));
  return hipGetLastError();
}

hipError_t launch_to_double(const void *xs, Dbl2 *x, int64_t n, hipStream_t s) {
  const int bs = 256;
  hipLaunchKernelGGL(k_to_double, dim3(unsigned((n + bs - 1) / bs)), dim3(bs), 0, s,
                     static_cast<const float2 *>(xs), reinterpret_cast<double2 *>(x), n);
  return hipGetLastError();
}

namespace {
template <int NN>
bool prepare_nn() {
  bool ok = true;
  if constexpr (fast_fits(NN, sizeof(double))) ok = ok && pass1_setup<NN, double, double2, double2>();
  if constexpr (fast_fits(NN, sizeof(float)))
    ok = ok && pass1_setup<NN, float, float2, float2>() && pass1_setup<NN, float, double2, double2>();
  if constexpr (NN > kCubeMaxNN) {
    ok = ok && plane1_setup<NN, double, double2, double2>() && plane1_setup<NN, float, float2, float2>() &&
         plane1_setup<NN, float, double2, float2>();
    ok = ok && plane2_setup<NN, double, double2, double2, double2>() &&
         plane2_setup<NN, float, float2, float2, float2>() && plane2_setup<NN, float, double2, float2, double2>();
  } else {
    ok = ok && pass1_setup<NN, float, double2, float2>();
    ok = ok && pass2_setup<NN, double, double2, double2>() && pass2_setup<NN, float, float2, float2>() &&
         pass2_setup<NN, float, double2, double2>();
  }
  return ok;
}
}  // namespace

hipError_t prepare_kernels() {
  bool ok = true;
#define CASE(N) ok = prepare_nn<N>() && ok;
  DEX_NN_LIST(CASE)
#undef CASE
  ok = combine_setup<3>() && ok;
  ok = combine_setup<4>() && ok;
  gram_grids_nb<1>();
  gram_grids_nb<2>();
  gram_grids_nb<3>();
  gram_grids_nb<4>();
  return ok ? hipSuccess : hipErrorInvalidDeviceFunction;
}

}  // namespace dex
