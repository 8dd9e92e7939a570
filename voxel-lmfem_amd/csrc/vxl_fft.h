// Device helpers shared by the FFT passes (fft.hip: axes with a compile-time
// four-step factorisation; vxl_fftgen.h: every other length) and the host
// interface of the general passes.
#pragma once

#include <type_traits>

#include "vxl_cg.h"

namespace vxl {

template <typename T> struct CT;
template <> struct CT<float> { using type = float2; };
template <> struct CT<double> { using type = double2; };


// Spectrum storage element: the compute complex type itself, or a pair of
// BF16 values (FP32 arithmetic, half the spectrum traffic; round to nearest
// even on store).
struct bf16x2 {
  unsigned short x, y;
};
__device__ __forceinline__ unsigned short to_bf16(float f) {
  const unsigned int b = __float_as_uint(f);
  return static_cast<unsigned short>((b + 0x7FFFu + ((b >> 16) & 1u)) >> 16);
}
__device__ __forceinline__ float from_bf16(unsigned short h) { return __uint_as_float(static_cast<unsigned int>(h) << 16); }
template <typename C, typename SC>
__device__ __forceinline__ C sload(const SC* p) {
  if constexpr (std::is_same<SC, bf16x2>::value) {
    const bf16x2 v = *p;
    return C{from_bf16(v.x), from_bf16(v.y)};
  } else {
    return *p;
  }
}
template <typename C, typename SC>
__device__ __forceinline__ void sstore(SC* p, C v) {
  if constexpr (std::is_same<SC, bf16x2>::value) {
    *p = bf16x2{to_bf16(v.x), to_bf16(v.y)};
  } else {
    *p = v;
  }
}
template <typename C>
__device__ __forceinline__ C cadd(C a, C b) { return {a.x + b.x, a.y + b.y}; }
template <typename C>
__device__ __forceinline__ C csub(C a, C b) { return {a.x - b.x, a.y - b.y}; }
template <typename C>
__device__ __forceinline__ C cmul(C a, C b) { return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
template <typename C>
__device__ __forceinline__ C cconj(C a) { return {a.x, -a.y}; }
// multiply by -i (forward) or +i (inverse)
template <bool INV, typename C>
__device__ __forceinline__ C rot90(C a) { return INV ? C{-a.y, a.x} : C{a.y, -a.x}; }

// In-register DFTs of size R with kernel exp(-+2 pi i / R).
template <bool INV, typename T, typename C>
__device__ __forceinline__ void dft2(C* v) {
  C a = v[0], b = v[1];
  v[0] = cadd(a, b);
  v[1] = csub(a, b);
}
template <bool INV, typename T, typename C>
__device__ __forceinline__ void dft4(C* v) {
  C a0 = cadd(v[0], v[2]), a1 = csub(v[0], v[2]);
  C a2 = cadd(v[1], v[3]), a3 = rot90<INV>(csub(v[1], v[3]));
  v[0] = cadd(a0, a2);
  v[2] = csub(a0, a2);
  v[1] = cadd(a1, a3);
  v[3] = csub(a1, a3);
}
template <bool INV, typename T, typename C>
__device__ __forceinline__ void dft8(C* v) {
  const T s = T(0.70710678118654752440084436210484903928);
  C e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
  dft4<INV, T>(e);
  dft4<INV, T>(o);
  // twiddles w^k, k = 0..3, w = exp(-+ i pi/4)
  C t1 = INV ? C{s * (o[1].x - o[1].y), s * (o[1].x + o[1].y)}
             : C{s * (o[1].x + o[1].y), s * (o[1].y - o[1].x)};
  C t2 = rot90<INV>(o[2]);
  C t3 = INV ? C{-s * (o[3].x + o[3].y), s * (o[3].x - o[3].y)}
             : C{s * (o[3].y - o[3].x), -s * (o[3].x + o[3].y)};
  v[0] = cadd(e[0], o[0]);
  v[4] = csub(e[0], o[0]);
  v[1] = cadd(e[1], t1);
  v[5] = csub(e[1], t1);
  v[2] = cadd(e[2], t2);
  v[6] = csub(e[2], t2);
  v[3] = cadd(e[3], t3);
  v[7] = csub(e[3], t3);
}
template <bool INV, typename T, typename C>
__device__ __forceinline__ void dft3(C* v) {
  const T c = T(-0.5), s = T(INV ? 0.86602540378443864676372317075293618347
                                  : -0.86602540378443864676372317075293618347);
  C a = cadd(v[1], v[2]), b = csub(v[1], v[2]);
  C m = {v[0].x + c * a.x, v[0].y + c * a.y};
  C jb = {-s * b.y, s * b.x};
  v[0] = cadd(v[0], a);
  v[1] = cadd(m, jb);
  v[2] = csub(m, jb);
}
// Radix 5: with a1 = x1 + x4, b1 = x1 - x4, a2 = x2 + x3, b2 = x2 - x3 and
// theta = 2 pi / 5, X1,4 = x0 + a1 cos(theta) + a2 cos(2 theta) -+ i (b1 sin(theta)
// + b2 sin(2 theta)), X2,3 = x0 + a1 cos(2 theta) + a2 cos(theta) -+ i (b1 sin(2 theta)
// - b2 sin(theta)) (signs of i flipped for the inverse).
template <bool INV, typename T, typename C>
__device__ __forceinline__ void dft5(C* v) {
  const T c1 = T(0.30901699437494742410229341718281905886), c2 = T(-0.80901699437494742410229341718281905886);
  const T s1 = T(0.95105651629515357211643933337938214340), s2 = T(0.58778525229247312916870595463907276860);
  const C a1 = cadd(v[1], v[4]), b1 = csub(v[1], v[4]), a2 = cadd(v[2], v[3]), b2 = csub(v[2], v[3]);
  const C t1 = {v[0].x + c1 * a1.x + c2 * a2.x, v[0].y + c1 * a1.y + c2 * a2.y};
  const C t2 = {v[0].x + c2 * a1.x + c1 * a2.x, v[0].y + c2 * a1.y + c1 * a2.y};
  const C u1 = rot90<INV>(C{s1 * b1.x + s2 * b2.x, s1 * b1.y + s2 * b2.y});
  const C u2 = rot90<INV>(C{s2 * b1.x - s1 * b2.x, s2 * b1.y - s1 * b2.y});
  v[0] = cadd(v[0], cadd(a1, a2));
  v[1] = cadd(t1, u1);
  v[4] = csub(t1, u1);
  v[2] = cadd(t2, u2);
  v[3] = csub(t2, u2);
}
// cos and sin of x in [0, pi), evaluated at compile time: reduced to
// [0, pi/4] by the quarter-turn symmetries, then Taylor series (x^2 <= 0.62,
// 14 terms, far below double rounding).
constexpr double kPiD = 3.14159265358979323846264338327950288;
constexpr double taylor_cos(double x) {
  double term = 1.0, sum = 1.0;
  for (int i = 1; i < 15; ++i) {
    term *= -x * x / double((2 * i - 1) * (2 * i));
    sum += term;
  }
  return sum;
}
constexpr double taylor_sin(double x) {
  double term = x, sum = x;
  for (int i = 1; i < 15; ++i) {
    term *= -x * x / double((2 * i) * (2 * i + 1));
    sum += term;
  }
  return sum;
}
constexpr double const_cos(double x) {
  if (x > kPiD / 2) return -const_cos(kPiD - x);
  if (x > kPiD / 4) return taylor_sin(kPiD / 2 - x);
  return taylor_cos(x);
}
constexpr double const_sin(double x) {
  if (x > kPiD / 2) return const_sin(kPiD - x);
  if (x > kPiD / 4) return taylor_cos(kPiD / 2 - x);
  return taylor_sin(x);
}

// a * exp(-+2 pi i K / N) with the root a compile-time constant (0 <= K < N);
// K = 0, N/4 and N/2 take no multiplies.
template <int N, int K, bool INV, typename T, typename C>
__device__ __forceinline__ C twiddle_const(C a) {
  if constexpr (K == 0) {
    return a;
  } else if constexpr (4 * K == N) {
    return rot90<INV>(a);
  } else if constexpr (2 * K == N) {
    return C{-a.x, -a.y};
  } else {
    constexpr bool upper = 2 * K > N;  // exp(-2 pi i K / N) = conj(exp(-2 pi i (N - K) / N))
    constexpr double ang = 2.0 * kPiD * (upper ? N - K : K) / N;
    constexpr double c = const_cos(ang), sn = upper ? -const_sin(ang) : const_sin(ang);
    const C tw = {T(c), T(INV ? sn : -sn)};
    return cmul(a, tw);
  }
}

template <int K, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (K < N) {
    f(std::integral_constant<int, K>());
    static_for<K + 1, N>(f);
  }
}

// Odd prime radix: with a_j = x_j + x_{P-j}, b_j = x_j - x_{P-j},
//   X_k, X_{P-k} = x_0 + sum_j a_j cos(2 pi j k / P) -+ i sum_j b_j sin(2 pi j k / P)
// (signs of i flipped for the inverse), all roots compile-time constants.
template <int P, bool INV, typename T, typename C>
__device__ __forceinline__ void dft_odd(C* v) {
  constexpr int H = (P - 1) / 2;
  C a[H], b[H];
#pragma unroll
  for (int j = 0; j < H; ++j) {
    a[j] = cadd(v[j + 1], v[P - 1 - j]);
    b[j] = csub(v[j + 1], v[P - 1 - j]);
  }
  const C x0 = v[0];
  C dc = x0;
#pragma unroll
  for (int j = 0; j < H; ++j) dc = cadd(dc, a[j]);
  v[0] = dc;
  static_for<0, H>([&](auto kc) {
    constexpr int k = decltype(kc)::value + 1;
    C u = x0, s = {T(0), T(0)};
    static_for<0, H>([&](auto jc) {
      constexpr int j = decltype(jc)::value + 1;
      constexpr int m = (j * k) % P;
      constexpr bool upper = 2 * m > P;
      constexpr double ang = 2.0 * kPiD * (upper ? P - m : m) / P;
      constexpr double c = const_cos(ang), sn = upper ? -const_sin(ang) : const_sin(ang);
      u.x = fma(T(c), a[j - 1].x, u.x);
      u.y = fma(T(c), a[j - 1].y, u.y);
      s.x = fma(T(sn), b[j - 1].x, s.x);
      s.y = fma(T(sn), b[j - 1].y, s.y);
    });
    const C is = rot90<INV>(s);  // -i s forward, +i s inverse
    v[k] = cadd(u, is);
    v[P - k] = csub(u, is);
  });
}

// Smallest factor of an in-register size that is worth splitting off.
constexpr int dft_factor(int n) { return n % 2 == 0 ? 2 : n % 3 == 0 ? 3 : n % 5 == 0 ? 5 : n; }

// In-register DFT of size N (2 to 16, 18, 20, 25): base sizes directly, the
// others as A x B with compile-time roots of unity between the two steps.
template <int N, bool INV, typename T, typename C>
__device__ __forceinline__ void dft_reg(C* v) {
  if constexpr (N == 1) {
    return;
  } else if constexpr (N == 2) {
    dft2<INV, T>(v);
  } else if constexpr (N == 3) {
    dft3<INV, T>(v);
  } else if constexpr (N == 4) {
    dft4<INV, T>(v);
  } else if constexpr (N == 5) {
    dft5<INV, T>(v);
  } else if constexpr (N == 8) {
    dft8<INV, T>(v);
  } else if constexpr (dft_factor(N) == N) {
    dft_odd<N, INV, T>(v);
  } else if constexpr (N % 2 == 0) {
    C e[N / 2], o[N / 2];
#pragma unroll
    for (int k = 0; k < N / 2; ++k) {
      e[k] = v[2 * k];
      o[k] = v[2 * k + 1];
    }
    dft_reg<N / 2, INV, T>(e);
    dft_reg<N / 2, INV, T>(o);
    static_for<0, N / 2>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      const C t = twiddle_const<N, k, INV, T>(o[k]);
      v[k] = cadd(e[k], t);
      v[k + N / 2] = csub(e[k], t);
    });
  } else {
    // x[A m2 + m1]: B-point transforms over m2, w_N^(m1 k2), A-point over m1.
    constexpr int A = dft_factor(N), B = N / A;
    C g[A][B];
#pragma unroll
    for (int m1 = 0; m1 < A; ++m1) {
#pragma unroll
      for (int m2 = 0; m2 < B; ++m2) g[m1][m2] = v[A * m2 + m1];
      dft_reg<B, INV, T>(g[m1]);
    }
    static_for<0, B>([&](auto kc) {
      constexpr int k2 = decltype(kc)::value;
      C u[A];
      static_for<0, A>([&](auto mc) {
        constexpr int m1 = decltype(mc)::value;
        u[m1] = twiddle_const<N, (m1 * k2) % N, INV, T>(g[m1][k2]);
      });
      dft_reg<A, INV, T>(u);
#pragma unroll
      for (int k1 = 0; k1 < A; ++k1) v[k2 + B * k1] = u[k1];
    });
  }
}

template <typename T>
struct Tables {
  const typename CT<T>::type* wx;
  const typename CT<T>::type* wy;
  const typename CT<T>::type* wz;
  const T* gx;  // 7 x (nx/2+1): 1/m, D, v, d (FI symbol); 2 sin(t/2)/h, cos(t/2), sin(t/2) (C3D8R-HG)
  const T* gy;
  const T* gz;
  T hg0;        // > 0: C3D8R-HG symbol with hourglass penalty hg0 = s(C0) / V
};


// Reciprocal for the Green solve: the hardware estimate (<= 1 ulp) in FP32; in
// FP64 the estimate with two Newton steps y += y (1 - x y), a third of the
// instructions of a division.  The steps make NaN of the estimate's 0 or infinity;
// the division's own last instruction puts the quotient of an infinite or zero x back
// (against a test of the estimate's class: 4 instead of 41 more instructions in the z
// pass, whose 40^3 launch the test took from 10.1 to 10.4 us).
__device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double rcp(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = fma(y, fma(-x, y, 1.0), y);
  y = fma(y, fma(-x, y, 1.0), y);
  return __builtin_amdgcn_div_fixup(y, x, 1.0);
}

// Per-axis factors of the Green symbol at one wavenumber: table columns 0-3
// (1/m, D, v, d) for the FI element, columns 4-6 (S, c, s) in a, b, c for
// C3D8R-HG.
template <typename T>
struct AxisF {
  T a, b, c, d;
};
template <typename T>
__device__ __forceinline__ AxisF<T> axis_factors(const T* g, int n, int k, bool hg) {
  if (hg) return {g[4 * n + k], g[5 * n + k], g[6 * n + k], T(0)};
  return {g[k], g[n + k], g[2 * n + k], g[3 * n + k]};
}

template <typename T>
struct XUpdate {
  T* r;
  T* x;
  const T* p;
  const T* q;
  const double* alpha;
  double* partial;
  AlphaFold fold;
};
// alpha of right-hand side k for the update forms.
template <typename T>
__device__ __forceinline__ double update_alpha(const XUpdate<T>& u, int k, bool first, double* red) {
  return u.fold.partial ? fold_alpha(u.fold, k, first, red) : u.alpha[k];
}
// An inactive system takes no step.
template <typename T>
__device__ __forceinline__ void update_skipped(const XUpdate<T>& u, int k, bool first) {
  if (u.fold.partial && u.fold.hist && first && threadIdx.x == 0) u.fold.hist[k] = 0.0;
}


// ---- general passes (vxl_fftgen.h) ------------------------------------------------
// An axis of n = n1 * n2: n1 is transformed in registers; n2 in registers too,
// or in two such steps of na and nb, or, when it has no in-register factors (a
// prime factor above 13), as a dense transform out of LDS.
struct AxisPlan {
  int n, n1, n2;
  int na, nb;   // three-step: n2 = na * nb; otherwise 0
  int dense;    // n2 runs as a dense transform
  int hpad;     // dense: outputs 0 .. n2/2 padded to whole output groups
  void* coef;   // dense: cos and sin of 2 pi j k / n2, device (see dense_table)
};
template <typename T>
AxisPlan make_axis_plan(int n, bool z);  // z: for the z pass
// Padded output count of a dense plan (0 otherwise), and its coefficient table
// (empty otherwise; needs plan.hpad).
template <typename T>
int dense_pad(const AxisPlan& plan);
template <typename T>
std::vector<T> dense_table(const AxisPlan& plan);

// Workgroup shape of a general pass: P columns (pencils) x `rows` threads.
struct GenShape {
  int P, rows;
  size_t lds;
  int units;  // what one workgroup covers: columns (y, z) or row pairs (x)
};
template <typename T>
GenShape gen_shape_y(const AxisPlan& plan);
template <typename T>
GenShape gen_shape_z(const AxisPlan& plan);
template <typename T>
GenShape gen_shape_x(const AxisPlan& plan, int pairs_wanted);

template <typename T>
struct GenX {
  AxisPlan plan;
  GenShape shape;
  const typename CT<T>::type* w;
  int64_t rows;          // ny * nz
  int64_t field_stride, spec_stride;
  const int* active;
};
// Forward x pass of nrhs fields (upd: with the CG update, spec: on the
// residual spectrum; XUpdate and fft_x4_r2c describe both) and the inverse
// one (beta != nullptr: p = z + beta p_old, as fft_x4_c2r).
template <typename T>
int launch_gen_r2c(const GenX<T>& g, int nrhs, const T* r, typename CT<T>::type* S, const XUpdate<T>* upd, bool spec,
                   hipStream_t s);
template <typename T>
int launch_gen_c2r(const GenX<T>& g, int nrhs, const typename CT<T>::type* S, T* z, const double* beta, const T* pin,
                   const BetaFold& fold, hipStream_t s);
template <typename T>
int launch_gen_y(const AxisPlan& plan, const GenShape& sh, const typename CT<T>::type* w, bool inverse, int nrhs,
                 typename CT<T>::type* S, const typename CT<T>::type* src, int nz, int W, int64_t stride,
                 const int* active, hipStream_t s);
template <typename T>
int launch_gen_z(const AxisPlan& plan, const GenShape& sh, const Tables<T>& tb, int nrhs, typename CT<T>::type* S,
                 int ny, int nxh, T lam, T mu, T inv_vn, int64_t stride, const int* active, int nyq,
                 double* partial, const double* media, int group_rhs, hipStream_t s);

}  // namespace vxl
