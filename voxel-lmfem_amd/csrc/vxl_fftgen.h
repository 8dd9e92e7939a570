// FFT passes for axes of any length (instantiated per precision by
// fftgen_f32.hip and fftgen_f64.hip, and fftgen_z32.hip and fftgen_z64.hip).
//
// An axis of n = n1 * n2 runs as two steps over columns ("pencils") whose
// entries sit in LDS as L[entry][column]:
//   step 1, row t < n2: entries t + n2 k1 -> DFT_n1 -> times w_n^(j1 t) -> L[j1 n2 + t]
//           (the very entries it read, so it also runs in place in LDS);
//   step 2, row t < n1: entries t n2 + k2 -> DFT_n2 -> X[t + n1 j2].
// Lanes run along columns and the `rows` of a workgroup take the rows of each
// step in turn.  With 64 columns (SUB = 1) every index, twiddle and dense
// coefficient is uniform over a wave: address arithmetic runs on the scalar
// unit and coefficients arrive by scalar loads, so the vector unit executes
// little beside the transform itself.  With 32 columns (SUB = 2) the two halves
// of a wave take neighbouring rows: dense coefficients stay uniform, and
// twiddles are two scalar loads and a select.  Fewer columns (SUB = 0, the
// longest axes only) index per lane.  DFT_n1 and DFT_n2 are in-register
// transforms (2 to 16; FP32 also 18, 20, 25).  An n2 that is none of these (a prime
// factor above 13, or a product too large) is a dense transform out of LDS:
// the row is folded to a_j = x_j + x_{n2-j}, b_j = x_j - x_{n2-j}, and a thread
// forms kDenseOut output pairs X_k, X_{n2-k} from the cos and sin sums, n2 - 1
// multiply-adds per output.  Where n2 = na * nb has in-register factors, step 2
// is instead two steps of its own (kThree, gen_mid and gen_step3), in place.
//
// Measured, FP32, six loads, against mixed-radix Stockham passes with runtime
// strides (and a direct DFT for prime factors above 13): 111 x 94 x 118 (3 * 37,
// 2 * 47, 2 * 59) z pass 1753 -> 169 us, x 777 / 818 -> 97 / 94 us, y 677 -> 48 us;
// 150 x 100 x 125 z 235 -> 106 us, x 138 / 124 -> 78 / 59 us, y 120 -> 48 us (274 MB
// moved: 5.7 TB/s, the rate of a large copy).
#pragma once

#include <algorithm>
#include <cmath>

#include "vxl_fft.h"
#include "vxl_zlanes.h"

namespace vxl {
namespace {

template <typename T>
constexpr int kGenThreads = sizeof(T) == 4 ? 512 : 256;  // most threads per workgroup
template <typename T>
constexpr int kGenWaves = sizeof(T) == 4 ? 4 : 2;  // least waves per SIMD (128 / 256 registers)
template <typename T>
constexpr bool in_register(int n) {
  return (n >= 1 && n <= 16) || (sizeof(T) == 4 && (n == 18 || n == 20 || n == 25));
}
template <typename T>
constexpr int kDenseOut = sizeof(T) == 4 ? 8 : 4;  // dense output pairs per thread
constexpr int kMidMost = 13;  // largest middle factor of a three-step axis; its other factors:
constexpr bool three_step(int n) { return (n >= 1 && n <= 16) || n == 25; }
constexpr size_t kGenLds = 81408;  // dynamic LDS of a workgroup when two share a CU's 160 KB

// Read-only table in the constant address space: uniform indices become
// scalar loads.
template <typename T>
using CPtr = const __attribute__((address_space(4))) T*;
template <typename T>
__device__ __forceinline__ CPtr<T> cptr(const void* p) {
  return (CPtr<T>)(reinterpret_cast<uintptr_t>(p));
}
template <typename C, typename T>
__device__ __forceinline__ C cload(CPtr<T> p, int i) {
  return C{p[2 * i], p[2 * i + 1]};
}

// Device view of an axis.
template <typename T>
struct GenAxis {
  int n, n1, n2, dense, hpad;
  int na, nb;  // three-step: n2 = na * nb
  int lp;  // log2 of the column count
  const void* w;
  const void* coef;
};

// The rows a thread takes: base + half, base + half + step, ...; base is
// uniform over a wave (SUB = 1, 2).
template <int SUB>
struct RowSet {
  int base, step, half;
  __device__ __forceinline__ explicit RowSet(int lp) : step(int(blockDim.x) >> lp), half(0) {
    if constexpr (SUB == 0) {
      base = int(threadIdx.x) >> lp;
    } else {
      base = SUB * __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
      if constexpr (SUB == 2) half = (int(threadIdx.x) >> 5) & 1;
    }
  }
  // f(base row, row) for every row below n.
  template <typename F>
  __device__ __forceinline__ void each(int n, F&& f) const {
    for (int tb = base; tb < n; tb += step) {
      if constexpr (SUB == 2) {
        if (tb + half < n) f(tb, tb + half);
      } else {
        f(tb, tb);
      }
    }
  }
};
// Entry j * t of the twiddle table for row t = tb + half.  (tb + 1 may be one
// row past the last: j (tb + 1) stays below n.)
template <int SUB, typename C, typename T>
__device__ __forceinline__ C twiddle_at(CPtr<T> w, int j, int tb, int half) {
  C a = cload<C, T>(w, j * tb);
  if constexpr (SUB == 2) {
    const C b = cload<C, T>(w, j * (tb + 1));
    a = C{half ? b.x : a.x, half ? b.y : a.y};
  }
  return a;
}

// Rows of two neighbouring twiddle entries i0 (base row) and i1 (the row after it).
template <int SUB, typename C, typename T>
__device__ __forceinline__ C twiddle_pair(CPtr<T> w, int i0, int i1, int half) {
  C a = cload<C, T>(w, i0);
  if constexpr (SUB == 2) {
    const C b = cload<C, T>(w, i1);
    a = C{half ? b.x : a.x, half ? b.y : a.y};
  }
  return a;
}

template <typename T, bool kThree = false, int MOST = 25, typename F>
__device__ __forceinline__ void with_radix(int r, F&& f) {
  switch (r) {
#define VXL_R(R) \
  case R:        \
    if constexpr (R <= MOST && (kThree ? three_step(R) : in_register<T>(R))) f(std::integral_constant<int, R>()); \
    break;
    VXL_R(1) VXL_R(2) VXL_R(3) VXL_R(4) VXL_R(5) VXL_R(6) VXL_R(7) VXL_R(8) VXL_R(9) VXL_R(10) VXL_R(11) VXL_R(12)
    VXL_R(13) VXL_R(14) VXL_R(15) VXL_R(16) VXL_R(18) VXL_R(20) VXL_R(25)
#undef VXL_R
  }
}

// Step 1 over this thread's rows: load(entry), twiddled outputs to L
// (row stride ps, column p).
template <bool INV, int SUB, bool kThree, typename T, typename C, typename Load>
__device__ __forceinline__ void gen_step1(C* L, int ps, int p, const RowSet<SUB>& rs, const GenAxis<T>& ax, Load load) {
  const CPtr<T> w = cptr<T>(ax.w);
  const int n2 = ax.n2;
  with_radix<T, kThree>(ax.n1, [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    rs.each(n2, [&](int tb, int t) {
      C v[R];
#pragma unroll
      for (int k = 0; k < R; ++k) v[k] = load(t + n2 * k);
      dft_reg<R, INV, T>(v);
#pragma unroll
      for (int j = 0; j < R; ++j) {
        if (j > 0) {
          C tw = twiddle_at<SUB, C, T>(w, j, tb, rs.half);
          if (INV) tw = cconj(tw);
          v[j] = cmul(v[j], tw);
        }
        L[(j * n2 + t) * ps + p] = v[j];
      }
    });
  });
}

// One group of a dense DFT of the n2 entries x[e * ps]: out(k, X_k) for the
// outputs k0 .. k0 + kDenseOut - 1 and their mirrors.
template <bool INV, typename T, typename C, typename Out>
__device__ __forceinline__ void dense_group(const C* x, int ps, int k0, const GenAxis<T>& ax, Out out) {
  constexpr int K = kDenseOut<T>;
  const int n2 = ax.n2, h = (n2 - 1) / 2;
  const CPtr<T> coef = cptr<T>(ax.coef) + 2 * k0;
  C ca[K], sb[K];
#pragma unroll
  for (int q = 0; q < K; ++q) ca[q] = sb[q] = C{T(0), T(0)};
  const C x0 = x[0];
  const C xm = (n2 & 1) ? C{T(0), T(0)} : x[(n2 / 2) * ps];
#pragma unroll 2
  for (int j = 1; j <= h; ++j) {
    const C lo = x[j * ps], hi = x[(n2 - j) * ps];
    const C a = cadd(lo, hi), b = csub(lo, hi);
    const CPtr<T> cj = coef + 2 * (j - 1) * ax.hpad;
#pragma unroll
    for (int q = 0; q < K; ++q) {
      const T c = cj[2 * q], s = cj[2 * q + 1];
      ca[q].x = fma(c, a.x, ca[q].x);
      ca[q].y = fma(c, a.y, ca[q].y);
      sb[q].x = fma(s, b.x, sb[q].x);
      sb[q].y = fma(s, b.y, sb[q].y);
    }
  }
#pragma unroll
  for (int q = 0; q < K; ++q) {
    const int k = k0 + q;
    if (2 * k > n2) break;
    const T sg = (k & 1) ? T(-1) : T(1);
    const C u = {x0.x + sg * xm.x + ca[q].x, x0.y + sg * xm.y + ca[q].y};
    const C is = rot90<INV>(sb[q]);
    out(k, cadd(u, is));
    if (k > 0 && 2 * k != n2) out(n2 - k, csub(u, is));
  }
}

// Dense groups (row, first output) of this thread: f(tb, row, k0).  The
// halves of a wave (SUB = 2) take two rows of the same group, so that the
// coefficients stay uniform.
template <typename T, int SUB, typename F>
__device__ __forceinline__ void each_group(const RowSet<SUB>& rs, const GenAxis<T>& ax, F&& f) {
  constexpr int K = kDenseOut<T>, S = SUB == 2 ? 2 : 1;
  const int groups = ax.hpad / K, sets = (ax.n1 + S - 1) / S;
  for (int i = rs.base / S; i < sets * groups; i += rs.step / S) {
    const int tb = i / groups * S, k0 = (i - i / groups * groups) * K;
    if (S == 1 || tb + rs.half < ax.n1) f(tb, tb + rs.half, k0);
  }
}

// Step 2 over rows: out(t, j2, X[t + n1 j2]); reads L, calls out for every
// output of a row after all reads of that row (in-register form only).
template <bool INV, int SUB, typename T, typename C, typename Out>
__device__ __forceinline__ void gen_step2(const C* L, int ps, int p, const RowSet<SUB>& rs, const GenAxis<T>& ax,
                                          Out out) {
  const int n1 = ax.n1, n2 = ax.n2;
  if (ax.dense) {
    each_group<T>(rs, ax, [&](int, int t, int k0) {
      dense_group<INV, T>(L + t * n2 * ps + p, ps, k0, ax, [&](int k, C v) { out(t, k, v); });
    });
    return;
  }
  with_radix<T>(n2, [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    rs.each(n1, [&](int, int t) {
      C u[R];
#pragma unroll
      for (int k = 0; k < R; ++k) u[k] = L[(t * R + k) * ps + p];
      dft_reg<R, INV, T>(u);
#pragma unroll
      for (int j = 0; j < R; ++j) out(t, j, u[j]);
    });
  });
}

// The two steps of a three-step axis that replace step 2: with n2 = na nb, row
// (t, s) of the middle step takes the entries t n2 + s + nb k (s < nb), row (t, s)
// of the last one t n2 + s nb + k (s < na), whose outputs are X[t + n1 (s + na j)].
// Both write the entries they read.  back: the middle step of the transform run
// backwards (z pass), DFT_na^-1 and then the twiddle that step 1 multiplied by.
template <bool INV, bool BACK, int SUB, typename T, typename C>
__device__ __forceinline__ void gen_mid(C* L, int ps, int p, const RowSet<SUB>& rs, const GenAxis<T>& ax) {
  const CPtr<T> w = cptr<T>(ax.w);
  const int n1 = ax.n1, n2 = ax.n2, nb = ax.nb;
  with_radix<T, true, kMidMost>(ax.na, [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    rs.each(n1 * nb, [&](int rb, int r) {
      const int t0 = rb / nb, s0 = rb - t0 * nb;
      // Twiddle entry of output j: first + j step.
      const int f0 = BACK ? t0 * s0 : 0, d0 = BACK ? t0 * nb : n1 * s0;
      int f1 = f0, d1 = d0, at = t0 * n2 + s0;
      if constexpr (SUB == 2) {
        const bool wrap = s0 + 1 == nb;
        const int t1 = wrap ? t0 + 1 : t0, s1 = wrap ? 0 : s0 + 1;
        f1 = BACK ? t1 * s1 : 0;
        d1 = BACK ? t1 * nb : n1 * s1;
        at = rs.half ? t1 * n2 + s1 : at;
      }
      C* x = L + at * ps + p;
      const int stride = nb * ps;
      C v[R];
#pragma unroll
      for (int k = 0; k < R; ++k) v[k] = x[k * stride];
      dft_reg<R, INV, T>(v);
#pragma unroll
      for (int j = 0; j < R; ++j) {
        if (BACK || j > 0) {
          C tw = twiddle_pair<SUB, C, T>(w, f0 + j * d0, f1 + j * d1, rs.half);
          if (INV) tw = cconj(tw);
          v[j] = cmul(v[j], tw);
        }
        x[j * stride] = v[j];
      }
    });
  });
}
// Row (t, s) of the last step, first entry `at`: f(radix, base t, base s, t, s, at).
template <int SUB, typename T, typename F>
__device__ __forceinline__ void each_last(const RowSet<SUB>& rs, const GenAxis<T>& ax, F&& f) {
  const int na = ax.na, n2 = ax.n2, nb = ax.nb;
  with_radix<T, true>(nb, [&](auto rc) {
    rs.each(ax.n1 * na, [&](int rb, int r) {
      const int t0 = rb / na, s0 = rb - t0 * na;
      int t1 = t0, s1 = s0;
      if constexpr (SUB == 2) {
        const bool wrap = s0 + 1 == na;
        t1 = wrap ? t0 + 1 : t0;
        s1 = wrap ? 0 : s0 + 1;
      }
      f(rc, t0, s0, t1, s1, rs.half ? t1 * n2 + s1 * nb : t0 * n2 + s0 * nb);
    });
  });
}
// out(k, entry, X[k]): output k and the entry of L it was read from.
template <bool INV, int SUB, typename T, typename C, typename Out>
__device__ __forceinline__ void gen_step3(const C* L, int ps, int p, const RowSet<SUB>& rs, const GenAxis<T>& ax,
                                          Out out) {
  const int n1 = ax.n1, na = ax.na;
  each_last<SUB, T>(rs, ax, [&](auto rc, int t0, int s0, int t1, int s1, int at) {
    constexpr int R = decltype(rc)::value;
    const int k0 = rs.half ? t1 + n1 * s1 : t0 + n1 * s0;
    C u[R];
#pragma unroll
    for (int k = 0; k < R; ++k) u[k] = L[(at + k) * ps + p];
    dft_reg<R, INV, T>(u);
#pragma unroll
    for (int j = 0; j < R; ++j) out(k0 + n1 * na * j, at + j, u[j]);
  });
}

// ---- y pass -----------------------------------------------------------------------
// Columns are numbered over all z planes (z W + j), so only the last workgroup
// of a right-hand side has idle columns.
template <bool INV, typename T, int SUB, bool kThree>
__global__ void __launch_bounds__(kGenThreads<T>, kGenWaves<T>)
gen_y(typename CT<T>::type* S, const typename CT<T>::type* src, GenAxis<T> ax, int cols, int W, int64_t spec_stride,
      const int* active) {
  using C = typename CT<T>::type;
  extern __shared__ double2 smem_raw[];
  const uint3 b = xcd_block3();
  if (active && !active[b.y]) return;
  C* L = reinterpret_cast<C*>(smem_raw);
  const int P = SUB ? 64 / SUB : 1 << ax.lp, p = int(threadIdx.x) & (P - 1);
  const RowSet<SUB> rs(ax.lp);
  const int col = int(b.x) * P + p;
  const bool live = col < cols;
  const int c = live ? col : cols - 1;
  const int z = c / W, j = c - z * W;
  const int64_t off = int64_t(b.y) * spec_stride + int64_t(z) * ax.n * W + j;
  const C* in = src + off;
  gen_step1<INV, SUB, kThree, T>(L, P, p, rs, ax, [&](int e) -> C { return in[e * W]; });
  __syncthreads();
  C* o = S + off;
  if constexpr (kThree) {
    gen_mid<INV, false, SUB, T>(L, P, p, rs, ax);
    __syncthreads();
    gen_step3<INV, SUB, T>(L, P, p, rs, ax, [&](int k, int, C v) {
      if (live) o[k * W] = v;
    });
  } else {
    gen_step2<INV, SUB, T>(L, P, p, rs, ax, [&](int t, int k, C v) {
      if (live) o[(t + ax.n1 * k) * W] = v;
    });
  }
}

// ---- z pass with the Green solve -----------------------------------------------------
// Each lane holds one component of one (kx, ky); the three components of a
// wavevector sit in neighbouring lanes of one row of 16 (15 used), so the sums
// over components are DPP moves and the spectrum stays in registers between
// the forward step 2, the Green solve and the first inverse step, which takes
// the factors swapped: row t of the forward step 2 holds X[t + n1 j2] for all
// j2, and the inverse transforms over j2 first.  Two barriers per pass.
template <int CTRL>
__device__ __forceinline__ float dpp_row(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp_row(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
// Sum of v over the three lanes of a wavevector (c: this lane's component).
template <typename T>
__device__ __forceinline__ T sum3(T v, int c) {
  const T t = v + dpp_row<0x101>(v) + dpp_row<0x102>(v);  // valid where c = 0
  const T t1 = dpp_row<0x111>(t), t2 = dpp_row<0x112>(t);
  return c == 0 ? t : c == 1 ? t1 : t2;
}

// Green solve of one component (fft.hip's green_point and green_point_hg
// distributed over the three lanes).
template <typename T>
struct GreenLane {
  int c;
  bool hg;
  T lam, mu, lm, hg0;
  // FI: a = D_x + D_y, b = own (lam + mu) d and v for c < 2, s = 1/(V N m_x m_y).
  // HG: wxy = {S_x c_y, c_x S_y, c_x c_y}, A = s_x^2 s_y^2, B = s_y^2 c_x^2 + s_x^2 c_y^2 + A, s = 1/(V N).
  T a, b, v, s;
  T w0, w1, w2, A, B;
  __device__ __forceinline__ void init(const Tables<T>& tb, int nxh, int ny, int kx, int ky, T inv_vn) {
    const AxisF<T> X = axis_factors(tb.gx, nxh, kx, hg), Y = axis_factors(tb.gy, ny, ky, hg);
    lm = lam + mu;
    if (hg) {
      const T sx2 = X.c * X.c, sy2 = Y.c * Y.c, cx2 = X.b * X.b, cy2 = Y.b * Y.b;
      w0 = X.a * Y.b;
      w1 = X.b * Y.a;
      w2 = X.b * Y.b;
      A = sx2 * sy2;
      B = sy2 * cx2 + sx2 * cy2 + A;
      s = inv_vn;
    } else {
      a = X.b + Y.b;
      b = lm * (c == 0 ? X.d : Y.d);
      v = c == 0 ? X.c : Y.c;
      s = inv_vn * X.a * Y.a;
    }
  }
  // q -> G q (this lane's component); returns Re(conj(q) G q) of it in FP64.
  template <typename C>
  __device__ __forceinline__ double solve(C& q, const AxisF<T>& Z) const {
    C o;
    if (hg) {
      const T wx = w0 * Z.b, wy = w1 * Z.b, wz = w2 * Z.a;
      const T ww = wx * wx + wy * wy + wz * wz;
      const T al = mu * ww + hg0 * (T(8) * (A * (Z.b * Z.b) + B * (Z.c * Z.c)));
      const bool zero = !(al > T(0));
      const T ia = rcp(al), gm = lm * rcp(al + lm * ww);
      const T w = c == 0 ? wx : c == 1 ? wy : wz;
      const C wd = {sum3(w * q.x, c), sum3(w * q.y, c)};
      const T sc = s * ia;
      o = zero ? C{T(0), T(0)} : C{sc * (q.x - gm * w * wd.x), sc * (q.y - gm * w * wd.y)};
    } else {
      const T sum = a + Z.b;
      const bool zero = !(sum > T(0));
      const T vc = c == 2 ? Z.c : v;
      const T i = rcp(fma(mu, sum, c == 2 ? lm * Z.d : b));
      const T vi = vc * i;
      const T gm = lm * rcp(T(1) + lm * sum3(vc * vi, c));
      const C e = {q.x * i, q.y * i};
      const C sd = {sum3(vc * e.x, c), sum3(vc * e.y, c)};
      const T sc = s * Z.a, wv = gm * vi;
      o = zero ? C{T(0), T(0)} : C{sc * (e.x - wv * sd.x), sc * (e.y - wv * sd.y)};
    }
    // FP64 products: a right-hand side at rounding-noise level has FP32
    // products below the normal range, which would stop the recurrence.
    const double d = double(q.x) * o.x + double(q.y) * o.y;
    q = o;
    return d;
  }
};

// partial (optional): FP64 r . z of the workgroup by Parseval, weight 1 at
// kx = 0 and kx = nyq, 2 elsewhere, at partial[rhs * gridDim.x + block].
template <typename T, bool kDot, int SUB, bool kThree>
__global__ void __launch_bounds__(kGenThreads<T>, kGenWaves<T>)
gen_z(typename CT<T>::type* S, GenAxis<T> ax, int ny, int nxh, Tables<T> tb, T lam, T mu, T inv_vn,
      int64_t spec_stride, const int* active, int nyq, double* partial, const double* media, int group_rhs) {
  using C = typename CT<T>::type;
  extern __shared__ double2 smem_raw[];
  __shared__ double red[kGenThreads<T> / 64];
  const uint3 bk = xcd_block3();
  if (active && !active[bk.y]) return;
  if (media) {  // stacked cells: this right-hand side's reference medium
    lam = T(media[2 * (bk.y / group_rhs)]);
    mu = T(media[2 * (bk.y / group_rhs) + 1]);
  }
  const int P = SUB ? 64 / SUB : 1 << ax.lp, p = int(threadIdx.x) & (P - 1);
  const RowSet<SUB> rs(ax.lp);
  const int n1 = ax.n1, n2 = ax.n2, W = 3 * nxh, cols = ny * W;
  C* L = reinterpret_cast<C*>(smem_raw);
  C* L2 = L + ax.n * P;  // dense only
  const ZLane lane = z_lane(P, p, int(bk.x), cols);
  const bool live = lane.live;
  const int cc = lane.col;
  const int ky = cc / W, kx = (cc - ky * W) / 3;
  GreenLane<T> G;
  G.c = lane.comp;
  G.hg = tb.hg0 > T(0);
  G.hg0 = tb.hg0;
  G.lam = lam;
  G.mu = mu;
  G.init(tb, nxh, ny, kx, ky, inv_vn);
  const double wk = (kx == 0 || kx == nyq) ? 1.0 : 2.0;
  C* base = S + int64_t(bk.y) * spec_stride + cc;
  const int64_t zs = int64_t(cols);
  const CPtr<T> gz = cptr<T>(tb.gz);
  const CPtr<T> w = cptr<T>(ax.w);
  auto zload = [&](int kz) -> AxisF<T> {
    const int n = ax.n;
    if (G.hg) return {gz[4 * n + kz], gz[5 * n + kz], gz[6 * n + kz], T(0)};
    return {gz[kz], gz[n + kz], gz[2 * n + kz], gz[3 * n + kz]};
  };
  auto zfactors = [&](int e0, int e1) -> AxisF<T> {  // of entry e0 (base row) or e1 (the row after it)
    AxisF<T> f = zload(e0);
    if constexpr (SUB == 2) {
      const AxisF<T> h = zload(min(e1, ax.n - 1));
      f = {rs.half ? h.a : f.a, rs.half ? h.b : f.b, rs.half ? h.c : f.c, rs.half ? h.d : f.d};
    }
    return f;
  };
  double dot = 0.0;

  gen_step1<false, SUB, kThree, T>(L, P, p, rs, ax, [&](int e) -> C { return base[e * zs]; });
  __syncthreads();
  if constexpr (kThree) {
    gen_mid<false, false, SUB, T>(L, P, p, rs, ax);
    __syncthreads();
    each_last<SUB, T>(rs, ax, [&](auto rc, int t0, int s0, int t1, int s1, int at) {
      constexpr int R = decltype(rc)::value;
      const int e0 = t0 + n1 * s0, e1 = t1 + n1 * s1, step = n1 * ax.na;
      C u[R];
#pragma unroll
      for (int k = 0; k < R; ++k) u[k] = L[(at + k) * P + p];
      dft_reg<R, false, T>(u);
#pragma unroll
      for (int j = 0; j < R; ++j) dot += G.solve(u[j], zfactors(e0 + step * j, e1 + step * j));
      dft_reg<R, true, T>(u);
#pragma unroll
      for (int m = 0; m < R; ++m) {
        if (m > 0) u[m] = cmul(u[m], cconj(twiddle_pair<SUB, C, T>(w, n1 * m * s0, n1 * m * s1, rs.half)));
        L[(at + m) * P + p] = u[m];
      }
    });
    __syncthreads();
    gen_mid<true, true, SUB, T>(L, P, p, rs, ax);
  } else if (ax.dense) {
    each_group<T>(rs, ax, [&](int tb, int t, int k0) {
      dense_group<false, T>(L + t * n2 * P + p, P, k0, ax, [&](int k, C v) {
        dot += G.solve(v, zfactors(tb + n1 * k, tb + 1 + n1 * k));
        L2[(t * n2 + k) * P + p] = v;
      });
    });
    __syncthreads();
    each_group<T>(rs, ax, [&](int tb, int t, int k0) {
      dense_group<true, T>(L2 + t * n2 * P + p, P, k0, ax, [&](int m, C v) {
        L[(t * n2 + m) * P + p] = cmul(v, cconj(twiddle_at<SUB, C, T>(w, m, tb, rs.half)));
      });
    });
  } else {
    with_radix<T>(n2, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      rs.each(n1, [&](int tb, int t) {
        C u[R];
#pragma unroll
        for (int k = 0; k < R; ++k) u[k] = L[(t * R + k) * P + p];
        dft_reg<R, false, T>(u);
#pragma unroll
        for (int k = 0; k < R; ++k) dot += G.solve(u[k], zfactors(tb + n1 * k, tb + 1 + n1 * k));
        dft_reg<R, true, T>(u);
#pragma unroll
        for (int m = 0; m < R; ++m) {
          if (m > 0) u[m] = cmul(u[m], cconj(twiddle_at<SUB, C, T>(w, m, tb, rs.half)));
          L[(t * R + m) * P + p] = u[m];
        }
      });
    });
  }
  __syncthreads();
  with_radix<T, kThree>(n1, [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    rs.each(n2, [&](int, int m) {
      C v[R];
#pragma unroll
      for (int t = 0; t < R; ++t) v[t] = L[(t * n2 + m) * P + p];
      dft_reg<R, true, T>(v);
      if (live) {
#pragma unroll
        for (int k = 0; k < R; ++k) base[(m + n2 * k) * zs] = v[k];
      }
    });
  });
  if constexpr (kDot) {
    const double total = block_reduce_dyn(live ? wk * dot : 0.0, red);
    if (threadIdx.x == 0) partial[int64_t(bk.y) * gridDim.x + bk.x] = total;
  }
}

// ---- x passes ---------------------------------------------------------------------
// Two real rows per complex pencil: row pair a of a workgroup (rows 2a, 2a+1 of
// the flattened (z, y) rows) gives the pencils 3a + {0, 1, 2} = c0 + i c1 of row
// 2a, c0 + i c1 of row 2a + 1, c2(2a) + i c2(2a + 1), as in fft_x4_r2c.  Rows
// are read and written with lanes along x (contiguous), the transform runs
// with lanes along pencils; the odd row stride of L keeps both conflict-free.

// Walks the (row, x) positions of a workgroup with lanes along x and no
// division in the loop.
struct RowWalk {
  int row, x, drow, dx, nx;
  __device__ __forceinline__ RowWalk(int n) : nx(n) {
    row = int(threadIdx.x) / n;
    x = int(threadIdx.x) - row * n;
    drow = int(blockDim.x) / n;
    dx = int(blockDim.x) - drow * n;
  }
  __device__ __forceinline__ void next() {
    row += drow;
    x += dx;
    if (x >= nx) {
      x -= nx;
      ++row;
    }
  }
};

enum GenXMode { kGenPlain = 0, kGenUpd = 1, kGenSpec = 2 };

// The slot of output entry k after step 2: natural order for the dense form
// (second buffer), otherwise in place, (k % n1) n2 + q with q = k / n1, or
// (q % na) nb + q / na in place of q (three-step).
template <bool kThree, typename T>
__device__ __forceinline__ void fill_slots(unsigned short* slot, const GenAxis<T>& ax) {
  for (int k = threadIdx.x; k < ax.n; k += blockDim.x) {
    const int q = k / ax.n1, t = k - q * ax.n1;
    slot[k] = static_cast<unsigned short>(kThree     ? t * ax.n2 + (q % ax.na) * ax.nb + q / ax.na
                                          : ax.dense ? k
                                                     : t * ax.n2 + q);
  }
}
// Both steps of an x pass on the pencils of L; every output at its slot of F.
template <bool INV, bool kThree, int SUB, typename T, typename C>
__device__ __forceinline__ void x_steps(C* L, C* F, int ps, int p, int NP, const RowSet<SUB>& rs,
                                        const GenAxis<T>& ax) {
  if (p < NP)
    gen_step1<INV, SUB, kThree, T>(L, ps, p, rs, ax, [&](int e) -> C { return L[e * ps + p]; });
  __syncthreads();
  if constexpr (kThree) {
    if (p < NP) gen_mid<INV, false, SUB, T>(L, ps, p, rs, ax);
    __syncthreads();
    if (p < NP) gen_step3<INV, SUB, T>(L, ps, p, rs, ax, [&](int, int at, C v) { L[at * ps + p] = v; });
  } else if (p < NP) {
    gen_step2<INV, SUB, T>(L, ps, p, rs, ax, [&](int t, int k, C v) {
      F[(ax.dense ? t + ax.n1 * k : t * ax.n2 + k) * ps + p] = v;
    });
  }
}

template <typename T, int MODE, int SUB, bool kThree>
__global__ void __launch_bounds__(kGenThreads<T>, kGenWaves<T>)
gen_r2c(const T* f, typename CT<T>::type* __restrict__ S, GenAxis<T> ax, int PB, int64_t rows_total,
        int64_t field_stride, int64_t spec_stride, const int* active, XUpdate<T> upd) {
  using C = typename CT<T>::type;
  extern __shared__ double2 smem_raw[];
  __shared__ double red[kGenThreads<T> / 64];
  const int rhs = blockIdx.y;
  if (active && !active[rhs]) {
    if constexpr (MODE != kGenPlain) update_skipped(upd, rhs, blockIdx.x == 0);
    return;
  }
  const int n = ax.n, nxh = n / 2 + 1, NP = 3 * PB, ps = NP | 1;
  C* L = reinterpret_cast<C*>(smem_raw);
  C* F = ax.dense ? L + n * ps : L;  // spectrum after step 2
  unsigned short* slot = reinterpret_cast<unsigned short*>(L + n * ps * (ax.dense ? 2 : 1));
  const int P = SUB ? 64 / SUB : 1 << ax.lp, p = int(threadIdx.x) & (P - 1);
  const RowSet<SUB> rs(ax.lp);
  const int64_t row0 = 2 * int64_t(blockIdx.x) * PB;
  const int have = int(min(int64_t(2 * PB), rows_total - row0));  // rows of this workgroup
  const int64_t plane = rows_total * n;
  const int64_t base = int64_t(rhs) * field_stride + row0 * n;
  T alpha = T(0);
  if constexpr (MODE != kGenPlain) alpha = T(update_alpha(upd, rhs, blockIdx.x == 0, red));
  double acc = 0.0;
  fill_slots<kThree>(slot, ax);
  {
    constexpr int U = MODE == kGenUpd ? 2 : 4;
    RowWalk it(n);
    while (it.row < 2 * PB) {
      int rw[U], xx[U];
      T v[U][3];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        rw[u] = it.row;
        xx[u] = it.x;
        it.next();
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool ok = rw[u] < have;
        const int64_t i = base + rw[u] * n + xx[u];
#pragma unroll
        for (int c = 0; c < 3; ++c) v[u][c] = ok ? f[i + c * plane] : T(0);
      }
      if constexpr (MODE == kGenUpd) {
        T q[U][3];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const bool ok = rw[u] < have;
          const int64_t i = base + rw[u] * n + xx[u];
#pragma unroll
          for (int c = 0; c < 3; ++c) q[u][c] = ok ? upd.q[i + c * plane] : T(0);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int64_t i = base + rw[u] * n + xx[u];
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            v[u][c] = fma(-alpha, q[u][c], v[u][c]);
            acc += double(v[u][c]) * double(v[u][c]);
            if (rw[u] < have) {
              upd.r[i + c * plane] = v[u][c];
              if (upd.x) upd.x[i + c * plane] = fma(alpha, upd.p[i + c * plane], upd.x[i + c * plane]);
            }
          }
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (rw[u] >= 2 * PB) continue;
        const int a = rw[u] >> 1, h = rw[u] & 1;
        C* row = L + xx[u] * ps + 3 * a;
        row[h] = C{v[u][0], v[u][1]};
        reinterpret_cast<T*>(row + 2)[h] = v[u][2];
      }
    }
  }
  __syncthreads();
  x_steps<false, kThree, SUB, T>(L, F, ps, p, NP, rs, ax);
  __syncthreads();
  // Two-for-one split over (pair, k), lanes along k.
  C* out = S + int64_t(rhs) * spec_stride + row0 * nxh * 3;
  for (RowWalk it(nxh); it.row < PB && 2 * it.row < have; it.next()) {
    const int a = it.row, k = it.x;
    const bool second = 2 * a + 1 < have;
    C* o0 = out + (int64_t(2 * a) * nxh + k) * 3;
    C* o1 = o0 + int64_t(nxh) * 3;
    C old[2][3];
    if constexpr (MODE == kGenSpec) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        old[0][c] = o0[c];
        old[1][c] = second ? o1[c] : C{T(0), T(0)};
      }
    }
    const C* x1 = F + int(slot[k]) * ps + 3 * a;
    const C* x2 = F + int(slot[k == 0 ? 0 : n - k]) * ps + 3 * a;
    C sp[3][2];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const C u = x1[q], v = cconj(x2[q]);
      const C s = cadd(u, v), d = csub(u, v);
      sp[q][0] = C{T(0.5) * s.x, T(0.5) * s.y};
      sp[q][1] = C{T(0.5) * d.y, T(-0.5) * d.x};  // d / (2i)
    }
    C nw[2][3] = {{sp[0][0], sp[0][1], sp[2][0]}, {sp[1][0], sp[1][1], sp[2][1]}};
    if constexpr (MODE == kGenSpec) {
      double e = 0.0;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          nw[h][c].x = fma(-alpha, nw[h][c].x, old[h][c].x);
          nw[h][c].y = fma(-alpha, nw[h][c].y, old[h][c].y);
          if (h == 0 || second) e += double(nw[h][c].x) * double(nw[h][c].x) + double(nw[h][c].y) * double(nw[h][c].y);
        }
      acc += ((k == 0 || 2 * k == n) ? 1.0 : 2.0) * e;
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) o0[c] = nw[0][c];
    if (second) {
#pragma unroll
      for (int c = 0; c < 3; ++c) o1[c] = nw[1][c];
    }
  }
  if constexpr (MODE != kGenPlain) {
    const double total = block_reduce_dyn(MODE == kGenSpec ? acc * (1.0 / n) : acc, red);
    if (threadIdx.x == 0) upd.partial[int64_t(rhs) * gridDim.x + blockIdx.x] = total;
  }
}

template <typename T, bool kDir, int SUB, bool kThree>
__global__ void __launch_bounds__(kGenThreads<T>, kGenWaves<T>)
gen_c2r(const typename CT<T>::type* __restrict__ S, T* z, GenAxis<T> ax, int PB, int64_t rows_total,
        int64_t field_stride, int64_t spec_stride, const int* active, const double* beta, const T* pin,
        BetaFold fold) {
  using C = typename CT<T>::type;
  extern __shared__ double2 smem_raw[];
  __shared__ double red[kGenThreads<T> / 64];
  const int rhs = blockIdx.y;
  if (active && !active[rhs]) return;
  const int n = ax.n, nxh = n / 2 + 1, NP = 3 * PB, ps = NP | 1;
  C* L = reinterpret_cast<C*>(smem_raw);
  C* F = ax.dense ? L + n * ps : L;
  unsigned short* slot = reinterpret_cast<unsigned short*>(L + n * ps * (ax.dense ? 2 : 1));
  const int P = SUB ? 64 / SUB : 1 << ax.lp, p = int(threadIdx.x) & (P - 1);
  const RowSet<SUB> rs(ax.lp);
  const int64_t row0 = 2 * int64_t(blockIdx.x) * PB;
  const int have = int(min(int64_t(2 * PB), rows_total - row0));
  const int64_t plane = rows_total * n;
  fill_slots<kThree>(slot, ax);
  // Hermitian extension and packing, lanes along k: each stored coefficient is
  // read once and fills entry k and, conjugated, its mirror n - k.
  const C* in = S + int64_t(rhs) * spec_stride + row0 * nxh * 3;
  {
    constexpr int U = 2;
    RowWalk it(nxh);
    while (it.row < PB) {
      int aa[U], kk[U];
      C v[U][2][3];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        aa[u] = it.row;
        kk[u] = it.x;
        it.next();
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const bool ok = 2 * aa[u] + h < have;
          const C* q = in + (int64_t(2 * aa[u] + h) * nxh + kk[u]) * 3;
#pragma unroll
          for (int c = 0; c < 3; ++c) v[u][h][c] = ok ? q[c] : C{T(0), T(0)};
        }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (aa[u] >= PB) continue;
        const int k = kk[u];
        if (k == 0 || 2 * k == n) {
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int c = 0; c < 3; ++c) v[u][h][c].y = T(0);
        }
        const auto& x = v[u];
        // pencil value at k from the spectra s0, s1 of its two real rows: s0 + i s1
        C* o = L + k * ps + 3 * aa[u];
        o[0] = C{x[0][0].x - x[0][1].y, x[0][0].y + x[0][1].x};
        o[1] = C{x[1][0].x - x[1][1].y, x[1][0].y + x[1][1].x};
        o[2] = C{x[0][2].x - x[1][2].y, x[0][2].y + x[1][2].x};
        if (k > 0 && 2 * k != n) {  // mirror: conj(s0) + i conj(s1)
          C* m = L + (n - k) * ps + 3 * aa[u];
          m[0] = C{x[0][0].x + x[0][1].y, x[0][1].x - x[0][0].y};
          m[1] = C{x[1][0].x + x[1][1].y, x[1][1].x - x[1][0].y};
          m[2] = C{x[0][2].x + x[1][2].y, x[1][2].x - x[0][2].y};
        }
      }
    }
  }
  __syncthreads();
  x_steps<true, kThree, SUB, T>(L, F, ps, p, NP, rs, ax);
  __syncthreads();
  const int64_t base = int64_t(rhs) * field_stride + row0 * n;
  T b = T(0);
  if constexpr (kDir) b = T(fold.partial ? fold_beta(fold, rhs, blockIdx.x == 0, red) : beta[rhs]);
  const bool keep = kDir && b != T(0);
  const T* prev = pin ? pin : z;
  constexpr int U = 4;
  RowWalk it(n);
  while (it.row < have) {
    int rw[U], xx[U];
    T old[U][3];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      rw[u] = it.row;
      xx[u] = it.x;
      it.next();
#pragma unroll
      for (int c = 0; c < 3; ++c)
        old[u][c] = keep && rw[u] < have ? prev[base + rw[u] * n + xx[u] + c * plane] : T(0);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (rw[u] >= have) continue;
      const int a = rw[u] >> 1, h = rw[u] & 1;
      const C* row = F + int(slot[xx[u]]) * ps + 3 * a;
      const C v = row[h];
      const T v2 = reinterpret_cast<const T*>(row + 2)[h];
      T* o = z + base + rw[u] * n + xx[u];
      o[0] = keep ? fma(b, old[u][0], v.x) : v.x;
      o[plane] = keep ? fma(b, old[u][1], v.y) : v.y;
      o[2 * plane] = keep ? fma(b, old[u][2], v2) : v2;
    }
  }
}

// Row form of a shape (see RowSet).
inline int sub_of(const AxisPlan& p, const GenShape& sh) {
  if (sh.P == 64) return 1;
  return sh.P == 32 && !(p.dense && p.n1 == 1) ? 2 : 0;
}
#define VXL_GT(A, K3)     \
  do {                    \
    if (sub == 1)         \
      VXL_G(A, 1, K3);    \
    else if (sub == 2)    \
      VXL_G(A, 2, K3);    \
    else                  \
      VXL_G(A, 0, K3);    \
  } while (0)
#define VXL_GS(A)         \
  do {                    \
    if (ax.nb)            \
      VXL_GT(A, true);    \
    else                  \
      VXL_GT(A, false);   \
  } while (0)

template <typename T>
GenAxis<T> axis_view(const AxisPlan& p, const GenShape& sh, const void* w) {
  GenAxis<T> a;
  a.n = p.n;
  a.n1 = p.n1;
  a.n2 = p.n2;
  a.dense = p.dense;
  a.na = p.na;
  a.nb = p.nb;
  a.hpad = p.hpad;
  a.lp = 31 - __builtin_clz(unsigned(sh.P));
  a.w = w;
  a.coef = p.coef;
  return a;
}

// Columns: the most of 64, 32 and 16 with which two workgroups share a CU's
// LDS, else the most that fit one.  (118-point dense z pass, FP64: 16 columns
// 293 us, 32 in one workgroup per CU 380 us; 150 points, FP32: 64 columns in
// 77 KB 164 us, 32 columns 253 us.)  The row count is the one that finishes the
// two steps in the fewest rounds.
template <typename T>
GenShape pick_shape(const AxisPlan& p, int widest, size_t (*lds)(const AxisPlan&, int P)) {
  GenShape s;
  s.P = 0;
  for (size_t limit : {kGenLds, 2 * kGenLds})
    for (int P = widest; P >= 16 && !s.P; P /= 2)
      if (lds(p, P) <= limit) s.P = P;
  if (!s.P) {
    s.P = std::min(widest, 8);
    while (s.P > 4 && lds(p, s.P) > 2 * kGenLds) s.P /= 2;
  }
  s.lds = lds(p, s.P);
  const int most = kGenThreads<T> / s.P, step = std::max(1, 64 / s.P);
  const int work2 = p.dense ? p.n1 * (p.hpad / kDenseOut<T>) : p.n1;
  const int cost2 = p.dense ? 2 * kDenseOut<T> * p.n2 : 4 * p.n2;
  int64_t best = INT64_MAX;
  s.rows = step;
  for (int r = step; r <= most; r += step) {
    int64_t c = int64_t((p.n2 + r - 1) / r) * 4 * p.n1;
    if (p.nb)
      c += int64_t((p.n1 * p.nb + r - 1) / r) * 4 * p.na + int64_t((p.n1 * p.na + r - 1) / r) * 4 * p.nb;
    else
      c += int64_t((work2 + r - 1) / r) * cost2;
    if (c < best) {
      best = c;
      s.rows = r;
    }
  }
  return s;
}

}  // namespace

// n = n1 * n2 with both factors in-register sizes and the larger one as small
// as possible; else n = n1 * na * nb likewise, na the smallest; otherwise the
// largest in-register n1, which leaves the smallest dense n2 (its cost grows with n2).
// Six loads, one such axis among 64-point ones, apply, us, mixed-radix Stockham passes
// (in use before these) / dense second factor / three steps: FP32 480 points z 526 /
// 538 / 340, x 384 / 460 / 297; FP64 480 z 931 / 1003 / 747, x 798 / 958 / 764, 625 x
// 1239 / 1953 / 1090.
// z: the z pass keeps factors above 16 (FP32) only while 32 columns fit.  With 16 its
// lanes index on their own, and wide factors spill there: 320 points as 16 * 20 take
// 389 us, as 4 * 8 * 10 237 (301 by the Stockham passes).
template <typename T>
AxisPlan make_axis_plan(int n, bool z) {
  AxisPlan p{};
  p.n = n;
  p.n1 = 1;
  p.n2 = n;
  p.dense = 1;
  int best = 0;
  for (int a = 1; a <= 25; ++a) {
    if (n % a || !in_register<T>(a)) continue;
    const int b = n / a;
    if (in_register<T>(b)) {
      const int larger = std::max(a, b);
      if (p.dense || larger < best) {
        best = larger;
        p.n1 = a;
        p.n2 = b;
        p.dense = 0;
      }
    } else if (p.dense) {
      p.n1 = a;
      p.n2 = b;
    }
  }
  if (p.dense || (z && best > 16 && sizeof(typename CT<T>::type) * n * 32 > kGenLds)) {
    int most = 26;
    for (int m = 2; m <= kMidMost; ++m)
      for (int b = m; m * b * b <= n; ++b) {
        const int a = n / (m * b);
        if (a * m * b != n || a >= most || !three_step(a) || !three_step(b)) continue;
        most = a;
        p.n1 = a;
        p.n2 = m * b;
        p.na = m;
        p.nb = b;
        p.dense = 0;
      }
  }
  p.hpad = dense_pad<T>(p);
  return p;
}

template <typename T>
GenShape gen_shape_y(const AxisPlan& plan) {
  GenShape s = pick_shape<T>(plan, 64, [](const AxisPlan& p, int P) {
    return sizeof(typename CT<T>::type) * size_t(p.n) * P;
  });
  s.units = s.P;
  return s;
}

template <typename T>
GenShape gen_shape_z(const AxisPlan& plan) {
  GenShape s = pick_shape<T>(plan, 64, [](const AxisPlan& p, int P) {
    return sizeof(typename CT<T>::type) * size_t(p.n) * P * (p.dense ? 2 : 1);
  });
  s.units = z_units(s.P);
  return s;
}

template <typename T>
GenShape gen_shape_x(const AxisPlan& plan, int pairs_wanted) {
  int widest = 64;
  if (pairs_wanted > 0)
    while (widest > 8 && widest / 2 / 3 >= pairs_wanted) widest /= 2;
  GenShape s = pick_shape<T>(plan, widest, [](const AxisPlan& p, int P) {
    const size_t ps = size_t(P / 3 * 3) | 1;
    return sizeof(typename CT<T>::type) * p.n * ps * (p.dense ? 2 : 1) + (sizeof(unsigned short) * p.n + 15) / 16 * 16;
  });
  s.units = s.P / 3;
  return s;
}

template <typename T>
int dense_pad(const AxisPlan& plan) {
  constexpr int K = kDenseOut<T>;
  return plan.dense ? (plan.n2 / 2 + 1 + K - 1) / K * K : 0;
}

template <typename T>
std::vector<T> dense_table(const AxisPlan& plan) {
  if (!plan.dense) return {};
  const int n2 = plan.n2, h = (n2 - 1) / 2;
  std::vector<double> c(n2), s(n2);
  for (int k = 0; k < n2; ++k) {
    const double ang = 2.0 * M_PI * double(k) / double(n2);
    c[k] = std::cos(ang);
    s[k] = std::sin(ang);
  }
  std::vector<T> tab(size_t(2) * h * plan.hpad, T(0));
  for (int j = 1; j <= h; ++j)
    for (int k = 0; k <= n2 / 2; ++k) {
      const int m = int(int64_t(j) * k % n2);
      T* o = &tab[(size_t(j - 1) * plan.hpad + k) * 2];
      o[0] = T(c[m]);
      o[1] = T(s[m]);
    }
  return tab;
}

template <typename T>
int launch_gen_r2c(const GenX<T>& g, int nrhs, const T* r, typename CT<T>::type* S, const XUpdate<T>* upd, bool spec,
                   hipStream_t s) {
  const int PB = g.shape.units;
  const int64_t pairs = (g.rows + 1) / 2;
  const dim3 grid(unsigned((pairs + PB - 1) / PB), unsigned(nrhs)), block(unsigned(g.shape.P * g.shape.rows));
  const GenAxis<T> ax = axis_view<T>(g.plan, g.shape, g.w);
  const XUpdate<T> u = upd ? *upd : XUpdate<T>{};
  const T* in = upd && spec ? upd->q : r;
  const int sub = sub_of(g.plan, g.shape);
#define VXL_G(MODE, WV, K3)                                                                                              \
  hipLaunchKernelGGL((gen_r2c<T, MODE, WV, K3>), grid, block, g.shape.lds, s, in, S, ax, PB, g.rows, g.field_stride,       \
                     g.spec_stride, g.active, u)
  if (!upd) {
    VXL_GS(kGenPlain);
  } else if (spec) {
    VXL_GS(kGenSpec);
  } else {
    VXL_GS(kGenUpd);
  }
#undef VXL_G
  VXL_HIP(hipGetLastError());
  return VXL_OK;
}

template <typename T>
int launch_gen_c2r(const GenX<T>& g, int nrhs, const typename CT<T>::type* S, T* z, const double* beta, const T* pin,
                   const BetaFold& fold, hipStream_t s) {
  const int PB = g.shape.units;
  const int64_t pairs = (g.rows + 1) / 2;
  const dim3 grid(unsigned((pairs + PB - 1) / PB), unsigned(nrhs)), block(unsigned(g.shape.P * g.shape.rows));
  const GenAxis<T> ax = axis_view<T>(g.plan, g.shape, g.w);
  const int sub = sub_of(g.plan, g.shape);
#define VXL_G(DIR, WV, K3)                                                                                            \
  hipLaunchKernelGGL((gen_c2r<T, DIR, WV, K3>), grid, block, g.shape.lds, s, S, z, ax, PB, g.rows, g.field_stride,     \
                     g.spec_stride, g.active, beta, pin, fold)
  if (beta) {
    VXL_GS(true);
  } else {
    VXL_GS(false);
  }
#undef VXL_G
  VXL_HIP(hipGetLastError());
  return VXL_OK;
}

template <typename T>
int launch_gen_y(const AxisPlan& plan, const GenShape& sh, const typename CT<T>::type* w, bool inverse, int nrhs,
                 typename CT<T>::type* S, const typename CT<T>::type* src, int nz, int W, int64_t stride,
                 const int* active, hipStream_t s) {
  const int64_t cols = int64_t(nz) * W;
  if (cols > INT32_MAX - 64 || int64_t(plan.n) * W > INT32_MAX) return fail("grid too large for the FFT y pass");
  const dim3 grid(unsigned((cols + sh.units - 1) / sh.units), unsigned(nrhs)), block(unsigned(sh.P * sh.rows));
  const GenAxis<T> ax = axis_view<T>(plan, sh, w);
  const int sub = sub_of(plan, sh);
#define VXL_G(INV, WV, K3) \
  hipLaunchKernelGGL((gen_y<INV, T, WV, K3>), grid, block, sh.lds, s, S, src, ax, int(cols), W, stride, active)
  if (inverse) {
    VXL_GS(true);
  } else {
    VXL_GS(false);
  }
#undef VXL_G
  VXL_HIP(hipGetLastError());
  return VXL_OK;
}

template <typename T>
int launch_gen_z(const AxisPlan& plan, const GenShape& sh, const Tables<T>& tb, int nrhs, typename CT<T>::type* S,
                 int ny, int nxh, T lam, T mu, T inv_vn, int64_t stride, const int* active, int nyq,
                 double* partial, const double* media, int group_rhs, hipStream_t s) {
  const int64_t cols = int64_t(ny) * 3 * nxh;
  if (cols > INT32_MAX - 64) return fail("grid too large for the FFT z pass");
  const dim3 grid(unsigned((cols + sh.units - 1) / sh.units), unsigned(nrhs)), block(unsigned(sh.P * sh.rows));
  const GenAxis<T> ax = axis_view<T>(plan, sh, tb.wz);
  const int sub = sub_of(plan, sh);
#define VXL_G(DOT, WV, K3)                                                                                        \
  hipLaunchKernelGGL((gen_z<T, DOT, WV, K3>), grid, block, sh.lds, s, S, ax, ny, nxh, tb, lam, mu, inv_vn, stride, \
                     active, nyq, partial, media, group_rhs)
  if (partial) {
    VXL_GS(true);
  } else {
    VXL_GS(false);
  }
#undef VXL_G
  VXL_HIP(hipGetLastError());
  return VXL_OK;
}

// Explicit instantiation for one precision: the plans with the x and y launchers,
// and the z launcher, whose kernels take as long to compile as all the others.
#define VXL_FFTGEN_INSTANCES(T)                                                                                       \
  template AxisPlan make_axis_plan<T>(int, bool);                                                                     \
  template GenShape gen_shape_y<T>(const AxisPlan&);                                                                  \
  template GenShape gen_shape_z<T>(const AxisPlan&);                                                                  \
  template GenShape gen_shape_x<T>(const AxisPlan&, int);                                                             \
  template int dense_pad<T>(const AxisPlan&);                                                                         \
  template std::vector<T> dense_table<T>(const AxisPlan&);                                                            \
  template int launch_gen_r2c<T>(const GenX<T>&, int, const T*, CT<T>::type*, const XUpdate<T>*, bool, hipStream_t);   \
  template int launch_gen_c2r<T>(const GenX<T>&, int, const CT<T>::type*, T*, const double*, const T*,                   \
                                 const BetaFold&, hipStream_t);                                                     \
  template int launch_gen_y<T>(const AxisPlan&, const GenShape&, const CT<T>::type*, bool, int, CT<T>::type*,         \
                               const CT<T>::type*, int, int, int64_t, const int*, hipStream_t);
#define VXL_FFTGEN_Z_INSTANCES(T)                                                                                     \
  template int launch_gen_z<T>(const AxisPlan&, const GenShape&, const Tables<T>&, int, CT<T>::type*, int, int, T, T,  \
                               T, int64_t, const int*, int, double*, const double*, int, hipStream_t);

}  // namespace vxl
