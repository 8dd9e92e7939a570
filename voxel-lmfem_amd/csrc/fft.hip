// FFT Green preconditioner of an isotropic reference medium, gfx950.
//
// z = IFFT( K0(k)^-1 FFT(r) ) with K0 the exact Fourier symbol of the periodic
// fully integrated HEX8 operator of a uniform isotropic medium (lam, mu):
//   per axis i, theta = 2 pi k_i / n_i:  m = (2+cos)/3, D = (2-2cos)/(h^2 m),
//   v = sin/(h m), d = D - v^2 = 4 sin^4(theta/2)/(3 h^2 m^2);
//   K0 = V m_x m_y m_z [diag(mu sum D + (lam+mu) d_i) + (lam+mu) v v^T]
// (the symbol of repro/bench/solver_comparison/fft_precision.py:65-79 and the
// diagonal + rank-1 form of _core/reference_medium/formula_kernels.cu:104-137).
// The inverse is applied per wavevector with Sherman-Morrison from 1-D tables
// (no Nk-sized coefficient cache); the k = 0 mode is removed and 1/N of the
// inverse transform is folded in.
//
// Transforms are hand-written two-step FFTs on LDS pencils: axes of 2^a and of
// 2^a times 3 or 5 run the four-step kernels below with compile-time factors,
// every other length the general passes of vxl_fftgen.h (twiddles from a host
// table filled with std::cos/std::sin).  Five passes per apply, spectrum
// stored as S[r][z][y][kx][c] with the three components interleaved so the z
// pass sees whole 3-vectors:
//   1. x: real-to-complex (two real rows per complex FFT), half spectrum
//   2. y: forward complex
//   3. z: forward complex, 3x3 Green solve, inverse complex (one pass)
//   4. y: inverse complex
//   5. x: complex-to-real (two rows per complex FFT)
#include <functional>

#include "vxl_fft.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>

namespace vxl {
namespace {

// Green solve at one wavevector (kx, ky, kz), in place:
//   out = 1/(t N) [q/E - gamma (v/E) (v . q/E)],  E_i = mu sum D + (lam+mu) d_i,
//   gamma = (lam+mu)/(1 + (lam+mu) sum v_i^2/E_i),  t N = V N m_x m_y m_z
// (the axis tables hold 1/m, D, v, d);
// k = 0 (sum D = 0) maps to 0.  Returns Re(conj(q) . out) in FP64.
template <typename T, typename C>
__device__ __forceinline__ double green_point(C& q0, C& q1, C& q2, const AxisF<T>& X, const AxisF<T>& Y,
                                              const AxisF<T>& Z, T lam, T mu, T inv_vn) {
  const T sumD = X.b + Y.b + Z.b;
  if (!(sumD > T(0))) {
    q0 = q1 = q2 = C{T(0), T(0)};
    return 0.0;
  }
  const T lm = lam + mu;
  const T i0 = rcp(mu * sumD + lm * X.d);
  const T i1 = rcp(mu * sumD + lm * Y.d);
  const T i2 = rcp(mu * sumD + lm * Z.d);
  const T gamma = lm * rcp(T(1) + lm * (X.c * X.c * i0 + Y.c * Y.c * i1 + Z.c * Z.c * i2));
  const T scale = inv_vn * X.a * Y.a * Z.a;  // tables hold 1/m
  const C a0 = {q0.x * i0, q0.y * i0}, a1 = {q1.x * i1, q1.y * i1}, a2 = {q2.x * i2, q2.y * i2};
  const C sdot = {X.c * a0.x + Y.c * a1.x + Z.c * a2.x, X.c * a0.y + Y.c * a1.y + Z.c * a2.y};
  const T w0 = gamma * X.c * i0, w1 = gamma * Y.c * i1, w2 = gamma * Z.c * i2;
  const C o0 = {scale * (a0.x - w0 * sdot.x), scale * (a0.y - w0 * sdot.y)};
  const C o1 = {scale * (a1.x - w1 * sdot.x), scale * (a1.y - w1 * sdot.y)};
  const C o2 = {scale * (a2.x - w2 * sdot.x), scale * (a2.y - w2 * sdot.y)};
  // Re(conj(q) . out) in FP64 products: a right-hand side at rounding-noise
  // level (a load whose exact fluctuation is zero) has FP32 products below
  // the normal range, which would stop the recurrence.
  const double d = double(q0.x) * o0.x + double(q0.y) * o0.y + double(q1.x) * o1.x + double(q1.y) * o1.y +
                   double(q2.x) * o2.x + double(q2.y) * o2.y;
  q0 = o0;
  q1 = o1;
  q2 = o2;
  return d;
}

// Green solve of the C3D8R-HG element (one-point rule + hourglass penalty,
// femlib/c3d8r.py:62-78) for the isotropic reference medium, derived from its
// plane-wave symbol.  The centroid gradient of a plane wave is i w (times a
// common phase) with w_x = (2/hx) sx cy cz (s = sin(t/2), c = cos(t/2) per
// axis, cyclic for y and z), and the hourglass pattern m has |h_m|^2 =
// 8 prod_{d in m} s_d^2 prod_{d not in m} c_d^2, so per unit volume
//   K(k) = (mu |w|^2 + hg0 H) I + (lam + mu) w w^T,
//   H = 8 (sx^2 sy^2 cz^2 + sy^2 sz^2 cx^2 + sz^2 sx^2 cy^2 + sx^2 sy^2 sz^2),
// inverted by Sherman-Morrison; k = 0 (a = 0) is removed.  Axis factors
// (a, b, c) = (S = (2/h) s, c, s).
template <typename T, typename C>
__device__ __forceinline__ double green_point_hg(C& q0, C& q1, C& q2, const AxisF<T>& X, const AxisF<T>& Y,
                                                 const AxisF<T>& Z, T hg0, T lam, T mu, T inv_vn) {
  const T Sx = X.a, cx = X.b, sx = X.c;
  const T Sy = Y.a, cy = Y.b, sy = Y.c;
  const T Sz = Z.a, cz = Z.b, sz = Z.c;
  const T wx = Sx * cy * cz, wy = cx * Sy * cz, wz = cx * cy * Sz;
  const T ww = wx * wx + wy * wy + wz * wz;
  const T sx2 = sx * sx, sy2 = sy * sy, sz2 = sz * sz, cx2 = cx * cx, cy2 = cy * cy, cz2 = cz * cz;
  const T H = T(8) * (sx2 * sy2 * cz2 + sy2 * sz2 * cx2 + sz2 * sx2 * cy2 + sx2 * sy2 * sz2);
  const T a = mu * ww + hg0 * H;
  if (!(a > T(0))) {
    q0 = q1 = q2 = C{T(0), T(0)};
    return 0.0;
  }
  const T lm = lam + mu;
  const T ia = rcp(a);
  const T g = lm * rcp(a + lm * ww);
  const C wd = {wx * q0.x + wy * q1.x + wz * q2.x, wx * q0.y + wy * q1.y + wz * q2.y};  // w . q
  const T sc = inv_vn * ia;
  const C o0 = {sc * (q0.x - g * wx * wd.x), sc * (q0.y - g * wx * wd.y)};
  const C o1 = {sc * (q1.x - g * wy * wd.x), sc * (q1.y - g * wy * wd.y)};
  const C o2 = {sc * (q2.x - g * wz * wd.x), sc * (q2.y - g * wz * wd.y)};
  // Re(conj(q) . out) in FP64 products: a right-hand side at rounding-noise
  // level (a load whose exact fluctuation is zero) has FP32 products below
  // the normal range, which would stop the recurrence.
  const double d = double(q0.x) * o0.x + double(q0.y) * o0.y + double(q1.x) * o1.x + double(q1.y) * o1.y +
                   double(q2.x) * o2.x + double(q2.y) * o2.y;
  q0 = o0;
  q1 = o1;
  q2 = o2;
  return d;
}

// Green solve of the cell's element at one wavevector.
template <typename T, typename C>
__device__ __forceinline__ double green_solve(C& q0, C& q1, C& q2, const Tables<T>& tb, const AxisF<T>& X,
                                              const AxisF<T>& Y, const AxisF<T>& Z, T lam, T mu, T inv_vn) {
  if (tb.hg0 > T(0)) return green_point_hg<T>(q0, q1, q2, X, Y, Z, tb.hg0, lam, mu, inv_vn);
  return green_point<T>(q0, q1, q2, X, Y, Z, lam, mu, inv_vn);
}

// ---- four-step pencil FFTs for axes of 2^a (times 3 or 5) -----------------------
// n = N1 * N2.  Step 1: thread t < N2 of a column holds x[t + N2 k1] (k1 < N1),
// transforms over k1, multiplies by w_n^(j1 t) and writes to LDS; step 2:
// thread t < N1 reads the N2 values of row t, transforms over k2 and holds
// X[t + N1 j2].  One LDS buffer of n x TJ complex, column-fastest (element e of
// column p at L[e * TJ + p]) so every LDS access is conflict-minimal and every
// global row segment is TJ contiguous complex values.  Twiddles come from the
// axis table w[k] = exp(-2 pi i k / n).

template <int N1, int N2>
struct FourStep {
  static constexpr int n = N1 * N2;
  static constexpr int lanes = N1 > N2 ? N1 : N2;
};

// Step 1 for column p, lane t: v[] = x[t + N2 k1] -> DFT_N1 -> twiddle -> L.
template <bool INV, typename T, int N1, int N2, int TS, typename C, typename Load>
__device__ __forceinline__ void four_step_1(C* L, int p, int t, const C* w, Load load) {
  constexpr int n = N1 * N2;
  C v[N1];
#pragma unroll
  for (int k1 = 0; k1 < N1; ++k1) v[k1] = load(k1);  // element t + N2 k1
  dft_reg<N1, INV, T>(v);
#pragma unroll
  for (int j1 = 0; j1 < N1; ++j1) {
    if (j1 > 0 && t > 0) {
      C tw = w[(j1 * t) % n];
      if (INV) tw = cconj(tw);
      v[j1] = cmul(v[j1], tw);
    }
    L[(j1 * N2 + t) * TS + p] = v[j1];
  }
}

// Step 2 for column p, lane t: u[] = L[t N2 + k2] -> DFT_N2 -> store(t + N1 j2).
template <bool INV, typename T, int N1, int N2, int TS, typename C, typename Store>
__device__ __forceinline__ void four_step_2(const C* L, int p, int t, const C* w, Store store) {
  C u[N2];
#pragma unroll
  for (int k2 = 0; k2 < N2; ++k2) u[k2] = L[(t * N2 + k2) * TS + p];
  dft_reg<N2, INV, T>(u);
#pragma unroll
  for (int j2 = 0; j2 < N2; ++j2) store(t + N1 * j2, u[j2]);
}

// Threads per four-step y / z workgroup, at most.
constexpr int kThreads4 = 512;
constexpr size_t kMaxLds4 = 65536;  // dynamic LDS per y / z workgroup, at most

// Columns per workgroup of the y pass and kx per workgroup of the z pass for
// an axis of N1 x N2: they are also the LDS row strides, fixed at compile time
// so every LDS access of the transforms is an immediate offset from one base
// (the host launches with these or, for short rows, fewer live columns).
// FP32 y: 32 columns (256 B row segments, measured 2.5% faster per apply
// than 16); z: 10 wavenumbers x 3 components (240 B; 0.5% faster per solve
// than 5, while 3 and 4 are slower); FP64 >= 128 B.
template <typename T, int N1, int N2>
constexpr int y4_cols() {
  constexpr int lanes = N1 > N2 ? N1 : N2;
  int c = sizeof(T) == 4 ? 32 : 16;
  if (c > kThreads4 / lanes) c = kThreads4 / lanes;
  while (c > 1 && 2 * sizeof(T) * size_t(N1 * N2) * c > kMaxLds4) --c;
  return c;
}
template <typename T, int N1, int N2>
constexpr int z4_kx() {
  constexpr int lanes = N1 > N2 ? N1 : N2;
  int k = sizeof(T) == 4 ? 10 : 3;
  if (k > kThreads4 / (3 * lanes)) k = kThreads4 / (3 * lanes);
  while (k > 1 && 2 * sizeof(T) * size_t(N1 * N2) * 3 * k + 4 * sizeof(T) * size_t(k) > kMaxLds4) --k;
  return k < 1 ? 1 : k;
}

// src: the spectrum read (S itself: in place; another buffer of the same
// layout: the pass writes S from it).
template <bool INV, typename T, int N1, int N2, typename SC>
__global__ void __launch_bounds__(kThreads4)
fft_y4(SC* S, const SC* src, int W, int TJ, const typename CT<T>::type* __restrict__ w, int64_t spec_stride,
       const int* active) {
  using C = typename CT<T>::type;
  constexpr int n = N1 * N2;
  extern __shared__ double2 smem_raw[];
  const uint3 b = xcd_block3();
  if (active && !active[b.z]) return;
  C* L = reinterpret_cast<C*>(smem_raw);
  constexpr int TS = y4_cols<T, N1, N2>();  // LDS row stride (TJ <= TS)
  const int j0 = b.x * TJ;
  const int tj = min(TJ, W - j0);
  const int64_t off = int64_t(b.z) * spec_stride + int64_t(b.y) * n * W + j0;
  SC* plane = S + off;
  const int p = threadIdx.x % TS, t = threadIdx.x / TS;
  const bool col = p < tj;
  // Offsets inside one (rhs, z) plane of n x W entries stay below 2^31.
  const SC* const base = src + off + (t * W + p);
  const int step = N2 * W;
  if (t < N2)
    four_step_1<INV, T, N1, N2, TS>(L, p, t, w, [&](int k1) -> C {
      return col ? sload<C>(base + k1 * step) : C{T(0), T(0)};
    });
  __syncthreads();
  if (t < N1 && col)
    four_step_2<INV, T, N1, N2, TS>(L, p, t, w, [&](int e, C v) { sstore(plane + (e * W + p), v); });
}

// Launched with a multiple of 64 threads; threads past 3 TK lanes-per-column
// only take part in the Green loop and the reduction.  kDot: r . z by Parseval, sum over the half
// spectrum of w(kx) Re(conj(r^) z^) with w = 1 at kx = 0 and kx = nyq (nx even), 2
// elsewhere; z^ = G r^ already carries the 1/N of the inverse transform, so the sum
// equals the real-space r . z.  One FP64 partial per workgroup at
// partial[(rhs * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x].
template <typename T, int N1, int N2, bool kDot, typename SC>
__global__ void __launch_bounds__(kThreads4)
fft_z4_green(SC* __restrict__ S, int ny, int nxh, int TK, Tables<T> tb, T lam, T mu, T inv_vn,
             int64_t spec_stride, const int* active, int nyq, double* partial, const double* media,
             int group_rhs) {
  using C = typename CT<T>::type;
  constexpr int nz = N1 * N2;
  extern __shared__ double2 smem_raw[];
  __shared__ double red[kThreads4 / 64];
  const uint3 b = xcd_block3();
  if (active && !active[b.z]) return;
  if (media) {  // stacked cells: this right-hand side's reference medium
    lam = T(media[2 * (b.z / group_rhs)]);
    mu = T(media[2 * (b.z / group_rhs) + 1]);
  }
  C* L = reinterpret_cast<C*>(smem_raw);
  constexpr int TKC = z4_kx<T, N1, N2>();  // kx per workgroup (TK <= TKC)
  constexpr int TJ = 3 * TKC;              // columns, also the LDS row stride
  const int k0 = b.x * TK;
  const int y = b.y;
  const int tk = min(TK, nxh - k0);
  const int W = 3 * nxh;
  // Offsets inside one right-hand side's spectrum (nz * ny * W entries, below
  // 2^31: the host checks) in 32-bit arithmetic.
  const int zstride = ny * W;
  SC* col = S + int64_t(b.z) * spec_stride + int64_t(y) * W + 3 * k0;
  const int p = threadIdx.x % TJ, t = threadIdx.x / TJ;
  const bool live = p < 3 * tk;
  const C* w = tb.wz;
  // With the block size a multiple of nz, every thread keeps one kz in the
  // Green pass; its z factors are loaded here, behind the transform's loads.
  const bool hg = tb.hg0 > T(0);
  const bool kz_fixed = blockDim.x % nz == 0;
  AxisF<T> az_own{};
  if (kz_fixed) az_own = axis_factors(tb.gz, nz, int(threadIdx.x % nz), hg);
  // The tile's x factors go to LDS behind the transform data (read after
  // the transform's barriers); the y factors are uniform.
  AxisF<T>* xf = reinterpret_cast<AxisF<T>*>(L + nz * TJ);
  if (int(threadIdx.x) < tk) xf[threadIdx.x] = axis_factors(tb.gx, nxh, k0 + int(threadIdx.x), hg);
  const AxisF<T> ay = axis_factors(tb.gy, ny, y, hg);
  // forward z transform: global -> L (natural kz order)
  if (t < N2)
    four_step_1<false, T, N1, N2, TJ>(L, p, t, w, [&](int k1) -> C {
      return live ? sload<C>(col + ((t + N2 * k1) * zstride + p)) : C{T(0), T(0)};
    });
  __syncthreads();
  C u[N2];
  if (t < N1) {
#pragma unroll
    for (int k2 = 0; k2 < N2; ++k2) u[k2] = L[(t * N2 + k2) * TJ + p];
    dft_reg<N2, false, T>(u);
  }
  __syncthreads();
  if (t < N1) {
#pragma unroll
    for (int j2 = 0; j2 < N2; ++j2) L[(t + N1 * j2) * TJ + p] = u[j2];
  }
  __syncthreads();
  // Green solve per (kz, kx) of this tile, kz fastest over the threads.
  double dot = 0.0;
#pragma unroll 2
  for (int idx = threadIdx.x; idx < nz * tk; idx += blockDim.x) {
    const int kz = idx % nz, kk = idx / nz;
    const int kx = k0 + kk;
    const AxisF<T> az = kz_fixed ? az_own : axis_factors(tb.gz, nz, kz, hg);
    const double d = green_solve<T>(L[kz * TJ + 3 * kk + 0], L[kz * TJ + 3 * kk + 1], L[kz * TJ + 3 * kk + 2],
                                    tb, xf[kk], ay, az, lam, mu, inv_vn);
    if constexpr (kDot) dot += (kx == 0 || kx == nyq) ? d : 2.0 * d;
  }
  if constexpr (kDot) {
    const double total = block_reduce_dyn(dot, red);
    if (threadIdx.x == 0)
      partial[(int64_t(b.z) * gridDim.y + b.y) * gridDim.x + b.x] = total;
  } else {
    __syncthreads();
  }
  // inverse z transform: L -> L (step 1, read before overwrite) -> global
  C v[N1];
  if (t < N2) {
#pragma unroll
    for (int k1 = 0; k1 < N1; ++k1) v[k1] = L[(t + N2 * k1) * TJ + p];
  }
  __syncthreads();
  if (t < N2)
    four_step_1<true, T, N1, N2, TJ>(L, p, t, w, [&](int k1) -> C { return v[k1]; });
  __syncthreads();
  if (t < N1 && live)
    four_step_2<true, T, N1, N2, TJ>(L, p, t, w, [&](int e, C val) { sstore(col + (e * zstride + p), val); });
}

// ---- four-step x passes for nx with a four-step factorisation ----------------
// The x pencils are contiguous in memory, so lanes run along x: pencil p of a
// workgroup is worked by `lanes` consecutive threads (t fastest), every global
// access is a run of consecutive floats, and no integer division by runtime
// values remains.  Pencils 3 pp + {0, 1, 2} of row pair pp are c0 + i c1 of
// row 2pp, of row 2pp + 1, and c2(2pp) + i c2(2pp + 1).
// LDS: the N1 x N2 step-1 tile of pencil p at p * TS + j1 * (N2 + 1) + t
// (row padding: step-2 reads run down a column), and the natural-order
// spectrum at p * (n + 1) + e.
template <int N1, int N2>
struct XTile {
  static constexpr int n = N1 * N2;
  static constexpr int TS = N1 * (N2 + 1) + 1;  // step-1 tile stride per pencil
  static constexpr int NS = n + 1;              // natural-order stride per pencil
  static constexpr int stride = TS > NS ? TS : NS;
};

// kUpd: the CG update r -= alpha q, x += alpha p is applied to every entry as it
// is loaded (r and x written back; upd.x == nullptr leaves x alone), the
// updated r is transformed, and the FP64 ||r||^2 of the workgroup goes to
// upd.partial[rhs * gridDim.x + blockIdx.x].
// kSpec (spectral residual): the input is q and S holds the x spectrum of the
// residual, R^; the transform q^ of each row updates it in place,
// R^ -= alpha q^, and the workgroup's FP64 ||r||^2 = (1/n) sum_k w(k) |R^(k)|^2
// (w = 1 at k = 0 and k = n/2, 2 elsewhere; Parseval over the half spectrum)
// goes to upd.partial as above.  S is then not written otherwise.
template <typename T, int N1, int N2, bool kUpd, typename SC, bool kSpec = false>
__global__ void __launch_bounds__(256)
fft_x4_r2c(const T* __restrict__ r, SC* __restrict__ S, int64_t rows, int PP,
           const typename CT<T>::type* __restrict__ w, int64_t field_stride, int64_t spec_stride,
           const int* active, XUpdate<T> upd) {
  using C = typename CT<T>::type;
  using XT = XTile<N1, N2>;
  constexpr int n = XT::n, nxh = n / 2 + 1, lanes = FourStep<N1, N2>::lanes;
  static_assert(!(kUpd && kSpec), "one update form per launch");
  static_assert(!kSpec || std::is_same<SC, C>::value, "the residual spectrum is stored at full precision");
  extern __shared__ double2 smem_raw[];
  __shared__ double red[4];
  if (active && !active[blockIdx.y]) {
    if constexpr (kUpd || kSpec) update_skipped(upd, blockIdx.y, blockIdx.x == 0);
    return;
  }
  double step = 0.0;
  if constexpr (kUpd || kSpec) step = update_alpha(upd, blockIdx.y, blockIdx.x == 0, red);
  C* L = reinterpret_cast<C*>(smem_raw);
  const int P = 3 * PP;
  const int t = threadIdx.x % lanes, p = threadIdx.x / lanes;
  const int pp = p / 3, q = p - 3 * pp;
  const int64_t plane = rows * n;
  const T* f = r + int64_t(blockIdx.y) * field_stride;
  SC* out = S + int64_t(blockIdx.y) * spec_stride;
  const int64_t rho = 2 * (int64_t(blockIdx.x) * PP + pp);
  const bool live = p < P;
  // component/row of the real and imaginary part of this pencil
  const int64_t re_off = q == 2 ? 2 * plane + rho * n : rho * n + (q == 1 ? n : 0);
  const int64_t im_off = q == 2 ? 2 * plane + (rho + 1) * n : plane + rho * n + (q == 1 ? n : 0);
  const bool re_ok = live && (q == 1 ? rho + 1 < rows : rho < rows);
  const bool im_ok = live && rho + (q == 0 ? 0 : 1) < rows;
  C* T1 = L + p * XT::stride;
  double rr = 0.0;
  const int64_t base = int64_t(blockIdx.y) * field_stride;
  const T alpha = T(step);
  // Distinct fields: restrict lets the loads of later entries run ahead of
  // the stores of earlier ones.
  T* __restrict__ ur = kUpd ? upd.r + base : nullptr;
  T* __restrict__ ux = kUpd && upd.x ? upd.x + base : nullptr;
  const T* __restrict__ up = kUpd && upd.x ? upd.p + base : nullptr;
  const T* __restrict__ uq = kUpd ? upd.q + base : nullptr;
  if (live && t < N2) {
    C v[N1];
    if constexpr (kUpd) {
      // All loads of the pencil first (r into v, q into dq), then the update
      // and the stores, so the loads are in flight together.
      C dq[N1];
#pragma unroll
      for (int k1 = 0; k1 < N1; ++k1) {
        const int e = t + N2 * k1;
        v[k1] = C{re_ok ? ur[re_off + e] : T(0), im_ok ? ur[im_off + e] : T(0)};
        dq[k1] = C{re_ok ? uq[re_off + e] : T(0), im_ok ? uq[im_off + e] : T(0)};
      }
#pragma unroll
      for (int k1 = 0; k1 < N1; ++k1) {
        const int e = t + N2 * k1;
        v[k1].x = fma(-alpha, dq[k1].x, v[k1].x);
        v[k1].y = fma(-alpha, dq[k1].y, v[k1].y);
        if (re_ok) {
          ur[re_off + e] = v[k1].x;
          if (ux) ux[re_off + e] = fma(alpha, up[re_off + e], ux[re_off + e]);
        }
        if (im_ok) {
          ur[im_off + e] = v[k1].y;
          if (ux) ux[im_off + e] = fma(alpha, up[im_off + e], ux[im_off + e]);
        }
        rr += double(v[k1].x) * double(v[k1].x) + double(v[k1].y) * double(v[k1].y);
      }
    } else {
#pragma unroll
      for (int k1 = 0; k1 < N1; ++k1) {
        const int e = t + N2 * k1;
        v[k1] = C{re_ok ? f[re_off + e] : T(0), im_ok ? f[im_off + e] : T(0)};
      }
    }
    dft_reg<N1, false, T>(v);
#pragma unroll
    for (int j1 = 0; j1 < N1; ++j1) {
      if (j1 > 0 && t > 0) v[j1] = cmul(v[j1], w[(j1 * t) % n]);
      T1[j1 * (N2 + 1) + t] = v[j1];
    }
  }
  __syncthreads();
  C u[N2];
  if (live && t < N1) {
#pragma unroll
    for (int k2 = 0; k2 < N2; ++k2) u[k2] = T1[t * (N2 + 1) + k2];
    dft_reg<N2, false, T>(u);
  }
  __syncthreads();
  if (live && t < N1) {
#pragma unroll
    for (int j2 = 0; j2 < N2; ++j2) T1[t + N1 * j2] = u[j2];  // natural order X[e]
  }
  __syncthreads();
  // Two-for-one split.
  double spec_rr = 0.0;  // kSpec: sum of w(k) |R^(k)|^2 over this thread's entries
  const T spec_alpha = T(step);
  for (int idx = threadIdx.x; idx < PP * nxh; idx += blockDim.x) {
    const int a = idx / nxh, k = idx - a * nxh;
    const int64_t rr = 2 * (int64_t(blockIdx.x) * PP + a);
    const int km = k == 0 ? 0 : n - k;
    C sp[3][2];
#pragma unroll
    for (int qq = 0; qq < 3; ++qq) {
      const C* X = L + (3 * a + qq) * XT::stride;
      const C x1 = X[k], x2 = cconj(X[km]);
      const C sm = cadd(x1, x2), df = csub(x1, x2);
      sp[qq][0] = C{T(0.5) * sm.x, T(0.5) * sm.y};
      sp[qq][1] = C{T(0.5) * df.y, T(-0.5) * df.x};
    }
    if constexpr (kSpec) {
      const double wk = (k == 0 || 2 * k == n) ? 1.0 : 2.0;
      auto sub = [&](C* o, C v) {
        C x = *o;
        x.x = fma(-spec_alpha, v.x, x.x);
        x.y = fma(-spec_alpha, v.y, x.y);
        *o = x;
        return double(x.x) * double(x.x) + double(x.y) * double(x.y);
      };
      double e = 0.0;
      if (rr < rows) {
        C* o = reinterpret_cast<C*>(out) + (rr * nxh + k) * 3;
        e += sub(o + 0, sp[0][0]) + sub(o + 1, sp[0][1]) + sub(o + 2, sp[2][0]);
      }
      if (rr + 1 < rows) {
        C* o = reinterpret_cast<C*>(out) + ((rr + 1) * nxh + k) * 3;
        e += sub(o + 0, sp[1][0]) + sub(o + 1, sp[1][1]) + sub(o + 2, sp[2][1]);
      }
      spec_rr += wk * e;
      continue;
    }
    if (rr < rows) {
      SC* o = out + (rr * nxh + k) * 3;
      sstore(o + 0, sp[0][0]);
      sstore(o + 1, sp[0][1]);
      sstore(o + 2, sp[2][0]);
    }
    if (rr + 1 < rows) {
      SC* o = out + ((rr + 1) * nxh + k) * 3;
      sstore(o + 0, sp[1][0]);
      sstore(o + 1, sp[1][1]);
      sstore(o + 2, sp[2][1]);
    }
  }
  if constexpr (kUpd || kSpec) {
    const double total = block_reduce_dyn(kSpec ? spec_rr * (1.0 / n) : rr, red);
    if (threadIdx.x == 0) upd.partial[int64_t(blockIdx.y) * gridDim.x + blockIdx.x] = total;
  }
}

// kDir: the output is the CG search direction p = z + beta[rhs] p_old, p_old from pin
// (pin == z: in place).
template <typename T, int N1, int N2, bool kDir, typename SC>
__global__ void __launch_bounds__(256)
fft_x4_c2r(const SC* __restrict__ S, T* z, int64_t rows, int PP,
           const typename CT<T>::type* __restrict__ w, int64_t field_stride, int64_t spec_stride,
           const int* active, const double* beta, const T* pin, BetaFold fold) {
  using C = typename CT<T>::type;
  using XT = XTile<N1, N2>;
  constexpr int n = XT::n, nxh = n / 2 + 1, lanes = FourStep<N1, N2>::lanes;
  extern __shared__ double2 smem_raw[];
  __shared__ double red[4];
  if (active && !active[blockIdx.y]) return;
  C* L = reinterpret_cast<C*>(smem_raw);
  const int P = 3 * PP;
  const SC* in = S + int64_t(blockIdx.y) * spec_stride;
  // Output position of this thread (pencil p, lane t) and, for the direction
  // update, the previous direction there, loaded first so that its latency
  // overlaps the transform.
  const int t = threadIdx.x % lanes, p = threadIdx.x / lanes;
  const int pp = p / 3, q = p - 3 * pp;
  const bool live = p < P;
  const int64_t plane = rows * n;
  const int64_t rho = 2 * (int64_t(blockIdx.x) * PP + pp);
  const int64_t re_off = q == 2 ? 2 * plane + rho * n : rho * n + (q == 1 ? n : 0);
  const int64_t im_off = q == 2 ? 2 * plane + (rho + 1) * n : plane + rho * n + (q == 1 ? n : 0);
  const bool re_ok = q == 1 ? rho + 1 < rows : rho < rows;
  const bool im_ok = rho + (q == 0 ? 0 : 1) < rows;
  T b = T(0);
  if constexpr (kDir) b = T(fold.partial ? fold_beta(fold, blockIdx.y, blockIdx.x == 0, red) : beta[blockIdx.y]);
  const bool keep = kDir && b != T(0);
  T prev[2][N2];
  if (keep && live && t < N1) {
    const T* g = (pin ? pin : z) + int64_t(blockIdx.y) * field_stride;
#pragma unroll
    for (int j2 = 0; j2 < N2; ++j2) {
      const int e = t + N1 * j2;
      prev[0][j2] = re_ok ? g[re_off + e] : T(0);
      prev[1][j2] = im_ok ? g[im_off + e] : T(0);
    }
  }
  // Hermitian extension and packing of the three pencils per row pair: each
  // stored coefficient kk is read once and fills entry kk and, conjugated,
  // its mirror n - kk.
  for (int idx = threadIdx.x; idx < PP * nxh; idx += blockDim.x) {
    const int a = idx / nxh, kk = idx - a * nxh;
    const int64_t rr = 2 * (int64_t(blockIdx.x) * PP + a);
    const bool realonly = kk == 0 || kk == n / 2;
    C x[2][3];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        C v = {T(0), T(0)};
        if (rr + h < rows) v = sload<C>(in + ((rr + h) * nxh + kk) * 3 + c);
        if (realonly) v.y = T(0);
        x[h][c] = v;
      }
    }
    // pencil value at k from the spectra s0, s1 of its two real rows: s0 + i s1
    C* L0 = L + (3 * a) * XT::stride;
    L0[kk] = C{x[0][0].x - x[0][1].y, x[0][0].y + x[0][1].x};
    L0[XT::stride + kk] = C{x[1][0].x - x[1][1].y, x[1][0].y + x[1][1].x};
    L0[2 * XT::stride + kk] = C{x[0][2].x - x[1][2].y, x[0][2].y + x[1][2].x};
    if (kk > 0 && kk < n - kk) {  // mirror: conj(s0) + i conj(s1)
      const int km = n - kk;
      L0[km] = C{x[0][0].x + x[0][1].y, x[0][1].x - x[0][0].y};
      L0[XT::stride + km] = C{x[1][0].x + x[1][1].y, x[1][1].x - x[1][0].y};
      L0[2 * XT::stride + km] = C{x[0][2].x + x[1][2].y, x[1][2].x - x[0][2].y};
    }
  }
  __syncthreads();
  C* X = L + p * XT::stride;
  C v[N1];
  if (live && t < N2) {
#pragma unroll
    for (int k1 = 0; k1 < N1; ++k1) v[k1] = X[t + N2 * k1];
  }
  __syncthreads();
  if (live && t < N2) {
    dft_reg<N1, true, T>(v);
#pragma unroll
    for (int j1 = 0; j1 < N1; ++j1) {
      if (j1 > 0 && t > 0) v[j1] = cmul(v[j1], cconj(w[(j1 * t) % n]));
      X[j1 * (N2 + 1) + t] = v[j1];
    }
  }
  __syncthreads();
  if (!(live && t < N1)) return;
  C u[N2];
#pragma unroll
  for (int k2 = 0; k2 < N2; ++k2) u[k2] = X[t * (N2 + 1) + k2];
  dft_reg<N2, true, T>(u);
  T* f = z + int64_t(blockIdx.y) * field_stride;
#pragma unroll
  for (int j2 = 0; j2 < N2; ++j2) {
    const int e = t + N1 * j2;
    if (re_ok) f[re_off + e] = keep ? fma(b, prev[0][j2], u[j2].x) : u[j2].x;
    if (im_ok) f[im_off + e] = keep ? fma(b, prev[1][j2], u[j2].y) : u[j2].y;
  }
}

struct PrecondImpl {
  double hg0;  // C3D8R-HG cell: hourglass penalty of the reference medium per unit volume (0: FI)
  int nx, ny, nz, nxh;
  int64_t rows;
  AxisPlan plan[3];  // x, y, z (general passes)
  GenShape shape[3];
  void* tables;      // one allocation; tw, tab and the plans' coefficients point into it
  void* tw[3];
  void* tab[3];
  void* spec;
  int64_t spec_stride;  // complex entries per RHS
  void* rhat;           // x spectrum of the CG residual (spectral-residual form), allocated on demand
  // four-step kernels for y / z axes with a factorisation (0: the general passes)
  int bf16;          // spectrum stored as BF16 pairs (FP32 arithmetic, four-step passes only)
  int x4;            // nx handled by fft_x4_r2c / fft_x4_c2r (0: the general passes)
  int pp4, thr_x4;   // row pairs and threads per x4 workgroup
  size_t lds_x4;
  int y4, z4;        // axis length handled by fft_y4 / fft_z4_green
  int tj4, tk4;      // columns / kx per workgroup
  int thr_y4, thr_z4;
  size_t lds_y4, lds_z4;
};

// Lengths with a four-step kernel (powers of two, and 24, 40, 48, 80, 96, 160,
// 192 = 2^a times 3 or 5); lanes = max(N1, N2).
inline int four_step_lanes(int n) {
  switch (n) {
    case 2: return 2;
    case 4: return 2;
    case 8: return 4;
    case 16: return 4;
    case 32: return 8;
    case 64: return 8;
    case 128: return 16;
    case 256: return 16;
    case 512: return 32;
    // 2^a times 3 or 5 (lanes = the larger factor)
    case 24: return 8;
    case 40: return 8;
    case 48: return 8;
    case 80: return 16;
    case 96: return 16;
    case 160: return 16;
    case 192: return 16;
  }
  return 0;
}

// Compile-time column counts of the y and z kernels for a runtime axis length
// (the factorisations of launch_y4 / launch_z4).
#define VXL_YZ4_FACTORS(M)                                                                                 \
  M(2, 1, 2) M(4, 2, 2) M(8, 2, 4) M(16, 4, 4) M(32, 4, 8) M(64, 8, 8) M(128, 8, 16) M(256, 16, 16) M(512, 16, 32) \
  M(24, 3, 8) M(40, 5, 8) M(48, 6, 8) M(80, 5, 16) M(96, 6, 16) M(160, 10, 16) M(192, 12, 16)
template <typename T>
int y4_cols_of(int n) {
#define VXL_C(N, A, B) \
  case N:              \
    return y4_cols<T, A, B>();
  switch (n) { VXL_YZ4_FACTORS(VXL_C) }
#undef VXL_C
  return 0;
}
template <typename T>
int z4_kx_of(int n) {
#define VXL_C(N, A, B) \
  case N:              \
    return z4_kx<T, A, B>();
  switch (n) { VXL_YZ4_FACTORS(VXL_C) }
#undef VXL_C
  return 0;
}

template <bool INV, typename T, typename SC>
void launch_y4(int n, dim3 grid, int thr, size_t lds, hipStream_t s, SC* S, const SC* src, int W, int TJ,
               const typename CT<T>::type* w, int64_t stride, const int* active) {
#define VXL_Y4(N, A, B)                                                                         \
  case N:                                                                                     \
    hipLaunchKernelGGL((fft_y4<INV, T, A, B, SC>), grid, dim3(thr), lds, s, S, src, W, TJ, w, stride, active); \
    break;
  switch (n) {
    VXL_Y4(2, 1, 2)
    VXL_Y4(4, 2, 2)
    VXL_Y4(8, 2, 4)
    VXL_Y4(16, 4, 4)
    VXL_Y4(32, 4, 8)
    VXL_Y4(64, 8, 8)
    VXL_Y4(128, 8, 16)
    VXL_Y4(256, 16, 16)
    VXL_Y4(512, 16, 32)
    VXL_Y4(24, 3, 8)
    VXL_Y4(40, 5, 8)
    VXL_Y4(48, 6, 8)
    VXL_Y4(80, 5, 16)
    VXL_Y4(96, 6, 16)
    VXL_Y4(160, 10, 16)
    VXL_Y4(192, 12, 16)
  }
#undef VXL_Y4
}

template <typename T, bool kDot, typename SC>
void launch_z4(int n, dim3 grid, int thr, size_t lds, hipStream_t s, SC* S, int ny, int nxh,
               int TK, Tables<T> tb, T lam, T mu, T inv_vn, int64_t stride, const int* active, int nyq,
               double* partial, const double* media, int group_rhs) {
#define VXL_Z4(N, A, B)                                                                              \
  case N:                                                                                          \
    hipLaunchKernelGGL((fft_z4_green<T, A, B, kDot, SC>), grid, dim3(thr), lds, s, S, ny, nxh, TK, tb, lam, mu, \
                       inv_vn, stride, active, nyq, partial, media, group_rhs);                    \
    break;
  switch (n) {
    VXL_Z4(2, 1, 2)
    VXL_Z4(4, 2, 2)
    VXL_Z4(8, 2, 4)
    VXL_Z4(16, 4, 4)
    VXL_Z4(32, 4, 8)
    VXL_Z4(64, 8, 8)
    VXL_Z4(128, 8, 16)
    VXL_Z4(256, 16, 16)
    VXL_Z4(512, 16, 32)
    VXL_Z4(24, 3, 8)
    VXL_Z4(40, 5, 8)
    VXL_Z4(48, 6, 8)
    VXL_Z4(80, 5, 16)
    VXL_Z4(96, 6, 16)
    VXL_Z4(160, 10, 16)
    VXL_Z4(192, 12, 16)
  }
#undef VXL_Z4
}

#define VXL_X4_CASES(M)                                                                                      \
  M(8, 4, 2) M(16, 4, 4) M(32, 8, 4) M(64, 8, 8) M(128, 16, 8) M(256, 16, 16) M(512, 32, 16) M(24, 8, 3) M(40, 8, 5) \
  M(48, 8, 6) M(80, 16, 5) M(96, 16, 6) M(160, 16, 10) M(192, 16, 12)

// The r2c pass loads in step 1, whose threads per pencil are N2, and the c2r
// pass stores in step 2, whose threads are N1: r2c takes the larger factor as
// N2 and c2r as N1, so every lane of a pencil moves data (at 96 = 16 x 6,
// r2c with 16 x 6 had 6 of 16 lanes loading).
#define VXL_X4R_CASES(M)                                                                                     \
  M(8, 2, 4) M(16, 4, 4) M(32, 4, 8) M(64, 8, 8) M(128, 8, 16) M(256, 16, 16) M(512, 16, 32) M(24, 3, 8) M(40, 5, 8) \
  M(48, 6, 8) M(80, 5, 16) M(96, 6, 16) M(160, 10, 16) M(192, 12, 16)

// LDS entries per pencil: the larger of the two passes' tiles.
template <typename T>
size_t x4_stride(int n) {
  size_t sr = 0, sc = 0;
#define VXL_X4S(N, A, B) \
  case N:                \
    sc = XTile<A, B>::stride; \
    break;
  switch (n) { VXL_X4_CASES(VXL_X4S) }
#undef VXL_X4S
#define VXL_X4S(N, A, B) \
  case N:                \
    sr = XTile<A, B>::stride; \
    break;
  switch (n) { VXL_X4R_CASES(VXL_X4S) }
#undef VXL_X4S
  return sr > sc ? sr : sc;
}

template <typename T, bool kUpd, typename SC, bool kSpec = false>
void launch_x4_r2c(int n, dim3 grid, int thr, size_t lds, hipStream_t s, const T* r, SC* S,
                   int64_t rows, int PP, const typename CT<T>::type* w, int64_t fstride, int64_t sstride,
                   const int* active, const XUpdate<T>& upd) {
#define VXL_X4R(N, A, B)                                                                                     \
  case N:                                                                                                  \
    hipLaunchKernelGGL((fft_x4_r2c<T, A, B, kUpd, SC, kSpec>), grid, dim3(thr), lds, s, r, S, rows, PP, w,  \
                       fstride, sstride, active, upd);                                                     \
    break;
  switch (n) { VXL_X4R_CASES(VXL_X4R) }
#undef VXL_X4R
}

template <typename T, bool kDir, typename SC>
void launch_x4_c2r(int n, dim3 grid, int thr, size_t lds, hipStream_t s, const SC* S, T* z,
                   int64_t rows, int PP, const typename CT<T>::type* w, int64_t fstride, int64_t sstride,
                   const int* active, const double* beta, const T* pin, const BetaFold& fold) {
#define VXL_X4C(N, A, B)                                                                                      \
  case N:                                                                                                   \
    hipLaunchKernelGGL((fft_x4_c2r<T, A, B, kDir, SC>), grid, dim3(thr), lds, s, S, z, rows, PP, w, fstride, \
                       sstride, active, beta, pin, fold);                                                         \
    break;
  switch (n) { VXL_X4_CASES(VXL_X4C) }
#undef VXL_X4C
}

// Twiddles, Green factors and dense coefficients of the three axes, in one
// allocation filled by one copy.
template <typename T>
int upload_tables(PrecondImpl* im, const double h[3]) {
  using C = typename CT<T>::type;
  std::vector<T> all;
  size_t at_w[3], at_tab[3], at_coef[3];
  auto put = [&](const T* v, size_t n) {  // each table on a 64-byte boundary
    const size_t at = (all.size() + 15) / 16 * 16;
    all.resize(at);
    all.insert(all.end(), v, v + n);
    return at;
  };
  const int ns[3] = {im->nx, im->ny, im->nz};
  const int counts[3] = {im->nxh, im->ny, im->nz};
  for (int a = 0; a < 3; ++a) {
    const int n = ns[a];
    std::vector<C> w(n);
    for (int k = 0; k < n; ++k) {
      const double ang = 2.0 * M_PI * double(k) / double(n);
      w[k] = C{T(std::cos(ang)), T(-std::sin(ang))};
    }
    at_w[a] = put(reinterpret_cast<const T*>(w.data()), 2 * size_t(n));
    const int cnt = counts[a];
    std::vector<T> tab(7 * size_t(cnt));
    for (int k = 0; k < cnt; ++k) {
      const double th = 2.0 * M_PI * double(k) / double(n);
      const double sh = std::sin(0.5 * th);
      const double m = (2.0 + std::cos(th)) / 3.0;
      const double hh = h[a];
      tab[k] = T(1.0 / m);  // 1/m: the Green scale is a product, no division
      tab[cnt + k] = T(4.0 * sh * sh / (hh * hh * m));
      tab[2 * cnt + k] = T(std::sin(th) / (hh * m));
      tab[3 * cnt + k] = T(4.0 * sh * sh * sh * sh / (3.0 * hh * hh * m * m));
      tab[4 * cnt + k] = T(2.0 * sh / hh);  // C3D8R-HG factors
      tab[5 * cnt + k] = T(std::cos(0.5 * th));
      tab[6 * cnt + k] = T(sh);
    }
    at_tab[a] = put(tab.data(), tab.size());
    const std::vector<T> coef = dense_table<T>(im->plan[a]);
    at_coef[a] = coef.empty() ? SIZE_MAX : put(coef.data(), coef.size());
  }
  VXL_HIP(dev_malloc(&im->tables, sizeof(T) * all.size()));
  VXL_HIP(hipMemcpy(im->tables, all.data(), sizeof(T) * all.size(), hipMemcpyHostToDevice));
  T* base = static_cast<T*>(im->tables);
  for (int a = 0; a < 3; ++a) {
    im->tw[a] = base + at_w[a];
    im->tab[a] = base + at_tab[a];
    im->plan[a].coef = at_coef[a] == SIZE_MAX ? nullptr : base + at_coef[a];
  }
  return VXL_OK;
}

template <typename T>
Tables<T> tables_of(const PrecondImpl* im) {
  using C = typename CT<T>::type;
  Tables<T> t;
  t.wx = static_cast<const C*>(im->tw[0]);
  t.wy = static_cast<const C*>(im->tw[1]);
  t.wz = static_cast<const C*>(im->tw[2]);
  t.gx = static_cast<const T*>(im->tab[0]);
  t.gy = static_cast<const T*>(im->tab[1]);
  t.gz = static_cast<const T*>(im->tab[2]);
  t.hg0 = T(im->hg0);
  return t;
}

constexpr size_t kMaxLds = 65536;
constexpr size_t kMaxLdsGen = 163840 - 1024;  // general passes, longest axes: one workgroup per CU

// Positive integer from the environment (tile-size overrides for sweeps), else 0.
int env_int(const char* name) {
  const char* e = std::getenv(name);
  if (!e) return 0;
  const int v = std::atoi(e);
  return v > 0 ? v : 0;
}

template <typename T>
int create_impl(vxl_precond* pc, PrecondImpl* im) {
  using C = typename CT<T>::type;
  const vxl_cell* cell = pc->cell;
  im->nx = cell->grid.nx;
  im->ny = cell->grid.ny;
  im->nz = cell->grid.nz;
  im->nxh = im->nx / 2 + 1;
  im->rows = int64_t(im->ny) * im->nz;
  const int axis[3] = {im->nx, im->ny, im->nz};
  for (int a = 0; a < 3; ++a) im->plan[a] = make_axis_plan<T>(axis[a], a == 2);
  {
    const int ly = four_step_lanes(im->ny), lz = four_step_lanes(im->nz);
    const char* env = std::getenv("VXL_FFT_FOURSTEP");
    const bool enable = !(env && env[0] == '0');
    im->y4 = (enable && ly) ? im->ny : 0;
    im->z4 = (enable && lz) ? im->nz : 0;
    if (im->y4) {
      // The kernel's compile-time column count sets the LDS stride and the
      // thread layout; rows shorter than it run with fewer live columns.
      const int cols4 = y4_cols_of<T>(im->ny);
      im->tj4 = std::max(1, std::min(cols4, 3 * im->nxh));
      im->thr_y4 = cols4 * ly;
      im->lds_y4 = sizeof(C) * size_t(im->ny) * cols4;
      if (im->lds_y4 > kMaxLds || im->thr_y4 > kThreads4) im->y4 = 0;
    }
    if (im->z4) {
      const int kx4 = z4_kx_of<T>(im->nz);
      if (int64_t(im->nz) * im->ny * 3 * im->nxh >= (int64_t(1) << 31)) im->z4 = 0;  // 32-bit offsets
      im->tk4 = std::max(1, std::min(kx4, im->nxh));
      im->thr_z4 = (3 * kx4 * lz + 63) / 64 * 64;  // whole waves for the block reduction
      im->lds_z4 = sizeof(C) * size_t(im->nz) * 3 * kx4 + 4 * sizeof(T) * size_t(kx4);  // + x factors
      if (im->lds_z4 > kMaxLds || im->thr_z4 > kThreads4 || im->thr_z4 < 1) im->z4 = 0;
    }
  }
  {
    // Four-step x passes for nx >= 8 with a factorisation: 64 / lanes row pairs per
    // workgroup (3 * 64 threads).
    const int lx = four_step_lanes(im->nx);
    const char* env = std::getenv("VXL_FFT_XFOURSTEP");
    im->x4 = (lx && im->nx >= 8 && !(env && env[0] == '0')) ? im->nx : 0;
    if (im->x4) {
      im->pp4 = 64 / lx;  // 3 * 64 = 192 threads, whole waves
      if (const int v = env_int("VXL_FFT_X4PAIRS")) im->pp4 = v;
      im->thr_x4 = 3 * im->pp4 * lx;
      im->lds_x4 = sizeof(C) * x4_stride<T>(im->nx) * 3 * im->pp4;
      if (im->thr_x4 > 256 || im->thr_x4 % 64 != 0 || im->lds_x4 > kMaxLds) im->x4 = 0;
    }
  }
  const int fourstep[3] = {im->x4, im->y4, im->z4};
  for (int a = 0; a < 3; ++a) {
    AxisPlan& p = im->plan[a];
    if (fourstep[a]) {
      p.dense = 0;
      continue;
    }
    im->shape[a] = a == 0 ? gen_shape_x<T>(p, env_int("VXL_FFT_XPAIRS")) : a == 1 ? gen_shape_y<T>(p) : gen_shape_z<T>(p);
    if (im->shape[a].lds > kMaxLdsGen) return fail("grid axis too long for the LDS pencil FFT");
  }
  im->spec_stride = int64_t(im->nz) * im->ny * im->nxh * 3;
  VXL_TRY(upload_tables<T>(im, cell->h));
  // Isotropic reference medium: (I1 + 7 I2) / 60 = (lam + 3 mu) / 2.
  im->hg0 = 0.0;
  if (cell->element == VXL_ELEMENT_C3D8R_HG) {
    const double hbar = (cell->h[0] + cell->h[1] + cell->h[2]) / 3.0;
    im->hg0 = cell->hg_coef * std::max(0.5 * (pc->lam + 3.0 * pc->mu), 1e-12) / (hbar * hbar);
  }
  im->bf16 = pc->precision == VXL_F32_BF16 ? 1 : 0;
  if (im->bf16 && !(im->x4 && im->y4 && im->z4))
    return fail("BF16 spectrum storage needs axes of at least 8 with a four-step factorisation (2^a, or 2^a times 3 or 5 from 24 to 192)");
  const size_t elem = im->bf16 ? sizeof(bf16x2) : sizeof(C);
  VXL_HIP(dev_malloc(&im->spec, elem * size_t(im->spec_stride) * pc->nrhs_max));
  return VXL_OK;
}

// Preconditioner apply z = M r.  CG form (cg != nullptr): the z pass also
// reduces r . z partials (Parseval) into cg->rz_partial, cg->mid() runs
// between the z pass and the inverse y pass (it turns the partials into beta
// on the same stream), and the last pass writes the search direction
// p = z + beta p in place of z.
struct CgHooks {
  double* rz_partial;
  const double* beta;
  std::function<int()> mid;
  const void* pin;  // previous search direction (nullptr: the output buffer, in place)
  BetaFold fold;    // partial != nullptr: the last pass forms beta itself and mid() is not called
};

enum Stages { kForwardX = 1, kRest = 2, kAllStages = 3 };

// Runs the x forward pass (kForwardX, optionally fused with the CG update upd)
// and/or the remaining passes (kRest).
// SC is the spectrum storage type: CT<T>::type, or bf16x2 (four-step passes only).
// sr (spectral residual; full-precision storage): the CG
// residual lives as its x spectrum in im->rhat.  The forward pass writes the
// x spectrum of r there (no upd) or updates it, R^ -= alpha q^, from the
// transform of upd->q (with upd); the y forward pass reads R^ and writes the
// working spectrum, which the later passes use in place.
template <typename T, typename SC>
int apply_stages(vxl_precond* pc, PrecondImpl* im, int nrhs, const T* r, T* z, hipStream_t s, const int* active,
                 const CgHooks* cg, int stages, const XUpdate<T>* upd, bool sr) {
  using C = typename CT<T>::type;
  constexpr bool kFull = std::is_same<SC, C>::value;
  const Tables<T> tb = tables_of<T>(im);
  SC* S = static_cast<SC*>(im->spec);
  const int64_t fstride = 3 * int64_t(im->nx) * im->rows;
  const int64_t pairs = (im->rows + 1) / 2;
  const int W = 3 * im->nxh;
  const unsigned bx4 = im->x4 ? unsigned((pairs + im->pp4 - 1) / im->pp4) : 0u;
  if (sr) {
    if constexpr (!kFull) {
      return fail("the spectral residual needs full-precision spectrum storage");
    } else {
      if (!im->rhat) return fail("the spectral residual has no buffer");
    }
  }
  SC* const Rh = static_cast<SC*>(im->rhat);
  const GenX<T> gx{im->plan[0], im->shape[0], tb.wx, im->rows, fstride, im->spec_stride, active};
  if (stages & kForwardX) {
    if (!im->x4) {
      if constexpr (!kFull)
        return fail("BF16 spectrum storage needs power-of-two axes");
      else
        VXL_TRY(launch_gen_r2c<T>(gx, nrhs, r, sr ? Rh : S, upd, sr, s));
    } else if (sr) {
      if constexpr (kFull) {
        if (upd)
          launch_x4_r2c<T, false, SC, true>(im->x4, dim3(bx4, nrhs), im->thr_x4, im->lds_x4, s, upd->q, Rh, im->rows,
                                            im->pp4, tb.wx, fstride, im->spec_stride, active, *upd);
        else
          launch_x4_r2c<T, false, SC>(im->x4, dim3(bx4, nrhs), im->thr_x4, im->lds_x4, s, r, Rh, im->rows, im->pp4,
                                      tb.wx, fstride, im->spec_stride, active, XUpdate<T>{});
      }
    } else if (upd) {
      launch_x4_r2c<T, true, SC>(im->x4, dim3(bx4, nrhs), im->thr_x4, im->lds_x4, s, r, S, im->rows, im->pp4, tb.wx,
                             fstride, im->spec_stride, active, *upd);
    } else {
      launch_x4_r2c<T, false, SC>(im->x4, dim3(bx4, nrhs), im->thr_x4, im->lds_x4, s, r, S, im->rows, im->pp4, tb.wx,
                              fstride, im->spec_stride, active, XUpdate<T>{});
    }
    VXL_HIP(hipGetLastError());
  }
  if (!(stages & kRest)) return VXL_OK;
  auto y_pass = [&](bool inverse) -> int {
    if (im->y4) {
      const dim3 g((W + im->tj4 - 1) / im->tj4, im->nz, nrhs);
      if (inverse)
        launch_y4<true, T, SC>(im->y4, g, im->thr_y4, im->lds_y4, s, S, S, W, im->tj4, tb.wy, im->spec_stride,
                               active);
      else
        launch_y4<false, T, SC>(im->y4, g, im->thr_y4, im->lds_y4, s, S, sr ? Rh : S, W, im->tj4, tb.wy,
                                im->spec_stride, active);
    } else if constexpr (!kFull) {
      return fail("BF16 spectrum storage needs power-of-two axes");
    } else {
      VXL_TRY(launch_gen_y<T>(im->plan[1], im->shape[1], tb.wy, inverse, nrhs, S, inverse || !sr ? S : Rh, im->nz, W,
                              im->spec_stride, active, s));
    }
    VXL_HIP(hipGetLastError());
    return VXL_OK;
  };
  VXL_TRY(y_pass(false));
  const double V = pc->cell->volume;
  const double N = double(pc->cell->grid.n);
  const T lam = T(pc->lam), mu = T(pc->mu), inv_vn = T(1.0 / (V * N));
  const double* media = pc->groups > 1 ? pc->media : nullptr;
  const int grhs = pc->groups > 1 ? std::max(1, nrhs / pc->groups) : std::max(1, nrhs);
  const int nyq = im->nx % 2 == 0 ? im->nx / 2 : -1;
  double* part = cg ? cg->rz_partial : nullptr;
  if (im->z4) {
    const dim3 g((im->nxh + im->tk4 - 1) / im->tk4, im->ny, nrhs);
    if (cg)
      launch_z4<T, true, SC>(im->z4, g, im->thr_z4, im->lds_z4, s, S, im->ny, im->nxh, im->tk4, tb, lam, mu, inv_vn,
                         im->spec_stride, active, nyq, part, media, grhs);
    else
      launch_z4<T, false, SC>(im->z4, g, im->thr_z4, im->lds_z4, s, S, im->ny, im->nxh, im->tk4, tb, lam, mu, inv_vn,
                          im->spec_stride, active, nyq, part, media, grhs);
  } else if constexpr (kFull) {
    VXL_TRY(launch_gen_z<T>(im->plan[2], im->shape[2], tb, nrhs, S, im->ny, im->nxh, lam, mu, inv_vn, im->spec_stride,
                            active, nyq, part, media, grhs, s));
  }
  VXL_HIP(hipGetLastError());
  const BetaFold fold = cg ? cg->fold : BetaFold{};
  if (cg && !fold.partial) VXL_TRY(cg->mid());
  VXL_TRY(y_pass(true));
  if (im->x4 && cg)
    launch_x4_c2r<T, true, SC>(im->x4, dim3(bx4, nrhs), im->thr_x4, im->lds_x4, s, S, z, im->rows, im->pp4, tb.wx,
                           fstride, im->spec_stride, active, cg->beta, static_cast<const T*>(cg->pin), fold);
  else if (im->x4)
    launch_x4_c2r<T, false, SC>(im->x4, dim3(bx4, nrhs), im->thr_x4, im->lds_x4, s, S, z, im->rows, im->pp4, tb.wx,
                            fstride, im->spec_stride, active, nullptr, static_cast<const T*>(nullptr), fold);
  else if constexpr (!kFull)
    return fail("BF16 spectrum storage needs power-of-two axes");
  else
    VXL_TRY(launch_gen_c2r<T>(gx, nrhs, S, z, cg ? cg->beta : nullptr, cg ? static_cast<const T*>(cg->pin) : nullptr, fold,
                              s));
  VXL_HIP(hipGetLastError());
  return VXL_OK;
}

template <typename T>
int apply_impl(vxl_precond* pc, PrecondImpl* im, int nrhs, const T* r, T* z, hipStream_t s,
               const int* active, const CgHooks* cg, int stages = kAllStages, const XUpdate<T>* upd = nullptr,
               bool sr = false) {
  if constexpr (std::is_same<T, float>::value) {
    if (im->bf16) return apply_stages<T, bf16x2>(pc, im, nrhs, r, z, s, active, cg, stages, upd, sr);
  }
  return apply_stages<T, typename CT<T>::type>(pc, im, nrhs, r, z, s, active, cg, stages, upd, sr);
}

}  // namespace

int precond_create(vxl_precond* pc) {
  auto* im = new PrecondImpl();
  im->tables = nullptr;
  im->tw[0] = im->tw[1] = im->tw[2] = nullptr;
  im->tab[0] = im->tab[1] = im->tab[2] = nullptr;
  for (auto& p : im->plan) p.coef = nullptr;
  im->spec = nullptr;
  im->rhat = nullptr;
  pc->impl = im;
  if (!(pc->lam >= 0.0) || !(pc->mu > 0.0)) return fail("reference medium requires lam >= 0, mu > 0");
  return pc->precision == VXL_F64 ? create_impl<double>(pc, im) : create_impl<float>(pc, im);
}

int precond_apply(vxl_precond* pc, int nrhs, const void* r, void* z, hipStream_t s) {
  return precond_apply_masked(pc, nrhs, r, z, nullptr, s);
}

template <typename T>
int precond_apply_cg(vxl_precond* pc, int nrhs, const T* r, T* p, double* rz_partial, const double* beta,
                     const std::function<int()>& mid, const int* active, hipStream_t s, const BetaFold* fold) {
  auto* im = static_cast<PrecondImpl*>(pc->impl);
  if (nrhs < 1 || nrhs > pc->nrhs_max) return fail("precond nrhs out of range");
  if ((pc->precision == VXL_F64) != std::is_same<T, double>::value) return fail("precond precision mismatch");
  const CgHooks cg{rz_partial, beta, mid, nullptr, fold ? *fold : BetaFold{}};
  return apply_impl<T>(pc, im, nrhs, r, p, s, active, &cg);
}
template int precond_apply_cg<float>(vxl_precond*, int, const float*, float*, double*, const double*,
                                     const std::function<int()>&, const int*, hipStream_t, const BetaFold*);
template int precond_apply_cg<double>(vxl_precond*, int, const double*, double*, double*, const double*,
                                      const std::function<int()>&, const int*, hipStream_t, const BetaFold*);

template <typename T>
int precond_cg_forward(vxl_precond* pc, int nrhs, T* r, T* x, const T* p, const T* q, const double* alpha,
                       double* rr_partial, const int* active, hipStream_t s, bool sr, const AlphaFold* fold) {
  auto* im = static_cast<PrecondImpl*>(pc->impl);
  if (nrhs < 1 || nrhs > pc->nrhs_max) return fail("precond nrhs out of range");
  if ((pc->precision == VXL_F64) != std::is_same<T, double>::value) return fail("precond precision mismatch");
  if (sr && (x || p)) return fail("the spectral residual takes no x update in the forward pass");
  if (!q) return apply_impl<T>(pc, im, nrhs, r, nullptr, s, active, nullptr, kForwardX, nullptr, sr);
  const XUpdate<T> upd{r, x, p, q, alpha, rr_partial, fold ? *fold : AlphaFold{}};
  return apply_impl<T>(pc, im, nrhs, r, nullptr, s, active, nullptr, kForwardX, &upd, sr);
}
template int precond_cg_forward<float>(vxl_precond*, int, float*, float*, const float*, const float*, const double*,
                                       double*, const int*, hipStream_t, bool, const AlphaFold*);
template int precond_cg_forward<double>(vxl_precond*, int, double*, double*, const double*, const double*,
                                        const double*, double*, const int*, hipStream_t, bool, const AlphaFold*);

template <typename T>
int precond_cg_rest(vxl_precond* pc, int nrhs, T* p, double* rz_partial, const double* beta,
                    const std::function<int()>& mid, const int* active, hipStream_t s, const T* p_old, bool sr,
                    const BetaFold* fold) {
  auto* im = static_cast<PrecondImpl*>(pc->impl);
  if (nrhs < 1 || nrhs > pc->nrhs_max) return fail("precond nrhs out of range");
  if ((pc->precision == VXL_F64) != std::is_same<T, double>::value) return fail("precond precision mismatch");
  const CgHooks cg{rz_partial, beta, mid, p_old, fold ? *fold : BetaFold{}};
  return apply_impl<T>(pc, im, nrhs, static_cast<const T*>(nullptr), p, s, active, &cg, kRest, nullptr, sr);
}
template int precond_cg_rest<float>(vxl_precond*, int, float*, double*, const double*, const std::function<int()>&,
                                    const int*, hipStream_t, const float*, bool, const BetaFold*);
template int precond_cg_rest<double>(vxl_precond*, int, double*, double*, const double*,
                                     const std::function<int()>&, const int*, hipStream_t, const double*, bool,
                                     const BetaFold*);

bool precond_spectral_residual_ok(const vxl_precond* pc) {
  const auto* im = static_cast<const PrecondImpl*>(pc->impl);
  const char* env = std::getenv("VXL_SPECTRAL_RESIDUAL");
  return pc->precision == VXL_F32 && !im->bf16 && !(env && env[0] == '0');
}

int precond_residual_spectrum(vxl_precond* pc) {
  auto* im = static_cast<PrecondImpl*>(pc->impl);
  if (im->rhat) return VXL_OK;
  if (!precond_spectral_residual_ok(pc)) return fail("the spectral residual needs FP32 spectrum storage");
  VXL_HIP(dev_malloc(&im->rhat, sizeof(float2) * size_t(im->spec_stride) * pc->nrhs_max));
  return VXL_OK;
}

int precond_fused_update_blocks(const vxl_precond* pc) {
  const auto* im = static_cast<const PrecondImpl*>(pc->impl);
  const int64_t pairs = (im->rows + 1) / 2, per = im->x4 ? im->pp4 : im->shape[0].units;
  return int((pairs + per - 1) / per);
}

bool fused_update_enabled() {
  // On unless VXL_FUSED_UPDATE=0.  At 256^3 x 6 the fused x pass takes
  // 973 us against 616 + 476 us for the separate update and x passes.
  const char* env = std::getenv("VXL_FUSED_UPDATE");
  return !(env && env[0] == '0');
}

int precond_apply_masked(vxl_precond* pc, int nrhs, const void* r, void* z, const int* active,
                         hipStream_t s) {
  auto* im = static_cast<PrecondImpl*>(pc->impl);
  if (nrhs < 1 || nrhs > pc->nrhs_max) return fail("precond nrhs out of range");
  if (pc->precision == VXL_F64)
    return apply_impl<double>(pc, im, nrhs, static_cast<const double*>(r), static_cast<double*>(z), s,
                              active, nullptr);
  return apply_impl<float>(pc, im, nrhs, static_cast<const float*>(r), static_cast<float*>(z), s, active,
                           nullptr);
}

int precond_rz_blocks(const vxl_precond* pc) {
  const auto* im = static_cast<const PrecondImpl*>(pc->impl);
  if (im->z4) return (im->nxh + im->tk4 - 1) / im->tk4 * im->ny;
  const int64_t cols = int64_t(im->ny) * 3 * im->nxh;
  return int((cols + im->shape[2].units - 1) / im->shape[2].units);
}

void precond_release(vxl_precond* pc) {
  auto* im = static_cast<PrecondImpl*>(pc->impl);
  if (!im) return;
  (void)hipStreamSynchronize(pc->cell->stream);
  if (im->tables) dev_free(im->tables);
  if (im->spec) dev_free(im->spec);
  if (im->rhat) dev_free(im->rhat);
  delete im;
  pc->impl = nullptr;
}

}  // namespace vxl
