// Matrix-free periodic HEX8 (fully integrated) stiffness action, RHS and mean
// stress for gfx950.
//
// Element action (exact 2x2x2 Gauss integration of a trilinear element with a
// constant 6x6 stiffness C).  With node a = ax + 2ay + 4az and sign
// s_d(a) = +-1, the Walsh-Hadamard coefficients q[m] = sum_a u_a prod_{d in m}
// s_d(a) give u(xi) = 1/8 sum_m q[m] prod_{d in m} xi_d.  The displacement
// gradient is a polynomial in {1, xi, eta, zeta, eta*zeta, xi*zeta, xi*eta};
// these seven monomials are orthogonal under the Gauss rule with weights
// {1, 1/3, 1/3, 1/3, 1/9, 1/9, 1/9}, so the element energy splits into seven
// independent strain modes and K_e = H^T G^T W C G H with H the 8-point
// Hadamard butterfly network.  This is the same element as the reference's
// modal form (_core/hybrid_operator/fi_modal.cuh:2-255); the code below is
// written from the derivation above, with the weights folded symmetrically
// into the geometric factors.
//
// Stencil schedule: a workgroup owns a TX x TY tile of output nodes and marches
// along z through a chunk of planes.  Each step stages one node plane (with a
// one-node halo) in LDS, computes the (TX+1)(TY+1) elements of one element
// layer (halo elements are recomputed instead of exchanged), writes their 24
// nodal forces to LDS, and every output node gathers its four bottom-layer and
// four top-layer contributions in a fixed order.  No atomics: the result is
// bitwise deterministic.
#pragma once

#include "vxl_internal.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace vxl {
namespace {

template <typename T>
struct G9 {
  T g[3][3];  // [class][axis]
};

// s = C e restricted to the strain components in MASK (bit k = Voigt k).
// kOrtho: C has no entries outside the normal block and the shear diagonal
// (isotropic media, orthotropic media along the axes); those products are
// left out.
template <int MASK, bool kOrtho, typename T>
__device__ __forceinline__ void cmul(const T* c, const T (&e)[6], T (&s)[6]) {
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    if (!((MASK >> i) & 1)) continue;
    T acc = T(0);
#pragma unroll
    for (int j = 0; j < 6; ++j) {
      if (!((MASK >> j) & 1)) continue;
      if (kOrtho && i != j && (i > 2 || j > 2)) continue;
      acc = fma(c[pidx(i, j)], e[j], acc);
    }
    s[i] = acc;
  }
}

// One strain mode.  MX/MY/MZ name the Hadamard mode whose coefficient vector
// forms gradient column x/y/z (-1: column absent); CLS selects the weight
// class.  Accumulates the back-projected modal forces into P.
// kIso (cubic voxels, gx = gy = gz within a class): the gradient scale is
// moved onto the back-projection, P += g^2 C e(q), and g holds g^2.
template <int MX, int MY, int MZ, int CLS, bool kIso, bool kOrtho, typename T>
__device__ __forceinline__ void strain_mode(const T* c, const G9<T>& g, const T (&q)[3][8],
                                            T (&P)[3][8]) {
  constexpr bool HX = MX >= 0, HY = MY >= 0, HZ = MZ >= 0;
  constexpr int MASK = (HX ? 1 : 0) | (HY ? 2 : 0) | (HZ ? 4 : 0) | ((HY || HZ) ? 8 : 0) |
                       ((HX || HZ) ? 16 : 0) | ((HX || HY) ? 32 : 0);
  const T bx = g.g[CLS][0], by = g.g[CLS][1], bz = g.g[CLS][2];
  const T gx = kIso ? T(1) : bx, gy = kIso ? T(1) : by, gz = kIso ? T(1) : bz;
  // Gradient columns col_j[i] = d u_i / d x_j.
  T cx[3], cy[3], cz[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    cx[i] = HX ? (kIso ? q[i][HX ? MX : 0] : gx * q[i][HX ? MX : 0]) : T(0);
    cy[i] = HY ? (kIso ? q[i][HY ? MY : 0] : gy * q[i][HY ? MY : 0]) : T(0);
    cz[i] = HZ ? (kIso ? q[i][HZ ? MZ : 0] : gz * q[i][HZ ? MZ : 0]) : T(0);
  }
  T e[6] = {T(0), T(0), T(0), T(0), T(0), T(0)};
  if constexpr (HX) e[0] = cx[0];
  if constexpr (HY) e[1] = cy[1];
  if constexpr (HZ) e[2] = cz[2];
  if constexpr (HY && HZ) e[3] = cz[1] + cy[2];
  else if constexpr (HY) e[3] = cy[2];
  else if constexpr (HZ) e[3] = cz[1];
  if constexpr (HX && HZ) e[4] = cz[0] + cx[2];
  else if constexpr (HX) e[4] = cx[2];
  else if constexpr (HZ) e[4] = cz[0];
  if constexpr (HX && HY) e[5] = cy[0] + cx[1];
  else if constexpr (HX) e[5] = cx[1];
  else if constexpr (HY) e[5] = cy[0];
  T s[6];
  if constexpr (kIso && CLS == 0) {
    // Constant mode of a cubic voxel: one factor b0 = g^2 on every axis.
    // Scaling the six strains by it (6 products) instead of the nine
    // back-projected stresses makes the back-projection plain assignments;
    // only this mode writes the slots MX = 1, MY = 2, MZ = 4, so P starts at
    // zero there.
    static_assert(MX == 1 && MY == 2 && MZ == 4, "the constant mode");
    const T b0 = bx;
#pragma unroll
    for (int i = 0; i < 6; ++i) e[i] *= b0;
    cmul<MASK, kOrtho>(c, e, s);
    P[0][MX] = s[0];
    P[1][MX] = s[5];
    P[2][MX] = s[4];
    P[0][MY] = s[5];
    P[1][MY] = s[1];
    P[2][MY] = s[3];
    P[0][MZ] = s[4];
    P[1][MZ] = s[3];
    P[2][MZ] = s[2];
    return;
  }
  cmul<MASK, kOrtho>(c, e, s);
  // Back-projection: P[m_j] += g_j * (sigma_0j, sigma_1j, sigma_2j).
  if constexpr (HX) {
    P[0][MX] = fma(bx, s[0], P[0][MX]);
    P[1][MX] = fma(bx, s[5], P[1][MX]);
    P[2][MX] = fma(bx, s[4], P[2][MX]);
  }
  if constexpr (HY) {
    P[0][MY] = fma(by, s[5], P[0][MY]);
    P[1][MY] = fma(by, s[1], P[1][MY]);
    P[2][MY] = fma(by, s[3], P[2][MY]);
  }
  if constexpr (HZ) {
    P[0][MZ] = fma(bz, s[4], P[0][MZ]);
    P[1][MZ] = fma(bz, s[3], P[1][MZ]);
    P[2][MZ] = fma(bz, s[2], P[2][MZ]);
  }
}

template <typename T>
__device__ __forceinline__ void hadamard_forward(T (&v)[8]) {
#pragma unroll
  for (int k = 1; k < 8; k <<= 1) {
#pragma unroll
    for (int a = 0; a < 8; ++a) {
      if (a & k) continue;
      const T lo = v[a], hi = v[a + k];
      v[a] = hi + lo;
      v[a + k] = hi - lo;
    }
  }
}

template <typename T>
__device__ __forceinline__ void hadamard_transpose(T (&v)[8]) {
#pragma unroll
  for (int k = 1; k < 8; k <<= 1) {
#pragma unroll
    for (int a = 0; a < 8; ++a) {
      if (a & k) continue;
      const T s = v[a], d = v[a + k];
      v[a] = s - d;
      v[a + k] = s + d;
    }
  }
}

// Modal element action: Hadamard coefficients q[c][m] in, modal forces P[c][m]
// out (nodal forces f = H^T P).  c: 21 packed stiffness.
template <bool kIso = false, bool kOrtho = false, typename T>
__device__ __forceinline__ void element_modal(const T (&q)[3][8], const T* c, const G9<T>& g,
                                              T (&P)[3][8]) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int m = 0; m < 8; ++m) P[i][m] = T(0);
  // Mode numbering: bit 0 = x, bit 1 = y, bit 2 = z.
  strain_mode<1, 2, 4, 0, kIso, kOrtho>(c, g, q, P);    // constant
  strain_mode<-1, 3, 5, 1, kIso, kOrtho>(c, g, q, P);   // xi
  strain_mode<3, -1, 6, 1, kIso, kOrtho>(c, g, q, P);   // eta
  strain_mode<5, 6, -1, 1, kIso, kOrtho>(c, g, q, P);   // zeta
  strain_mode<7, -1, -1, 2, kIso, kOrtho>(c, g, q, P);  // eta*zeta
  strain_mode<-1, 7, -1, 2, kIso, kOrtho>(c, g, q, P);  // xi*zeta
  strain_mode<-1, -1, 7, 2, kIso, kOrtho>(c, g, q, P);  // xi*eta
}

// C3D8R-HG element (femlib/c3d8r.py:62-78): one-point (centroid) integration,
// V B0^T C B0, which is exactly the constant strain mode above, plus the
// hourglass penalty s(C) H H^T.  H holds, per displacement component, the
// corner patterns xy, yz, zx and xyz over sqrt(8); in Hadamard coefficients
// the penalty is P[c][m] += s / 8 q[c][m] for the modes m = 3, 6, 5, 7.
// hg = coef V / hbar^2 / 8; s / 8 = hg * max((I1 + 7 I2) / 60, 1e-12).
template <bool kIso = false, typename T>
__device__ __forceinline__ void element_hg(const T (&q)[3][8], const T* c, const G9<T>& g, T hg, T (&P)[3][8]) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int m = 0; m < 8; ++m) P[i][m] = T(0);
  strain_mode<1, 2, 4, 0, kIso, false>(c, g, q, P);
  const T normal = c[pidx(0, 0)] + c[pidx(1, 1)] + c[pidx(2, 2)];
  const T i1 = normal + T(2) * (c[pidx(0, 1)] + c[pidx(0, 2)] + c[pidx(1, 2)]);
  const T i2 = normal + T(2) * (c[pidx(3, 3)] + c[pidx(4, 4)] + c[pidx(5, 5)]);
  const T k = hg * fmax((i1 + T(7) * i2) * T(1.0 / 60.0), T(1e-12));
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    P[i][3] = k * q[i][3];
    P[i][5] = k * q[i][5];
    P[i][6] = k * q[i][6];
    P[i][7] = k * q[i][7];
  }
}

// v[c][a]: nodal displacements in, nodal forces out.
template <typename T>
__device__ __forceinline__ void element_action(T (&v)[3][8], const T* c, const G9<T>& g) {
#pragma unroll
  for (int i = 0; i < 3; ++i) hadamard_forward(v[i]);
  T P[3][8];
  element_modal(v, c, g, P);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    hadamard_transpose(P[i]);
#pragma unroll
    for (int a = 0; a < 8; ++a) v[i][a] = P[i][a];
  }
}

// Two-point Hadamard of one face (4 nodes a2 = ax + 2 ay) and its transpose.
template <typename T>
__device__ __forceinline__ void face_forward(T (&v)[4]) {
  T a = v[1] + v[0], b = v[1] - v[0], c = v[3] + v[2], d = v[3] - v[2];
  v[0] = c + a;
  v[2] = c - a;
  v[1] = d + b;
  v[3] = d - b;
}
template <typename T>
__device__ __forceinline__ void face_transpose(T (&v)[4]) {
  T a = v[0] - v[2], c = v[0] + v[2], b = v[1] - v[3], d = v[1] + v[3];
  v[0] = a - b;
  v[1] = a + b;
  v[2] = c - d;
  v[3] = c + d;
}

template <typename T>
struct ApplyArgs {
  const T* u;
  T* out;
  int64_t rhs_stride;  // elements between right-hand sides
  const void* index;
  const T* table;      // rows x 24
  const float* scale;  // optional
  const float4* frames;  // kFrames: unit quaternion (w, x, y, z) of every voxel's material frame
  // Stacked cells: right-hand side r reads index block r / group_rhs, which
  // starts group_stride entries after the previous one (0 for one cell).
  int64_t group_stride;
  int group_rhs;
  int nx, ny, nz;
  int zchunk;
  int tiles_x;
  G9<T> g;
  T hg;  // C3D8R-HG: coef * V / hbar^2 / 8 (hourglass penalty per unit material scale)
  // kResid: r = f - K u written as r32 (if set) or r64, ||r||^2 per workgroup.
  const double* f;
  float* r32;
  double* r64;
  const double* rscale;  // optional power of two per right-hand side applied to r32
  // kFuse: systems with active[r] == 0 are skipped and u . (K u) of each
  // workgroup is written to partial[(r * chunks + chunk) * tiles + tile].
  const int* active;
  double* partial;
};

template <typename T>
void set_groups(ApplyArgs<T>& a, const vxl_cell* cell, int nrhs) {
  const int groups = cell->groups > 1 ? cell->groups : 1;
  a.group_stride = groups > 1 ? cell->grid.n : 0;
  a.group_rhs = groups > 1 ? std::max(1, nrhs / groups) : std::max(1, nrhs);
}

__device__ __forceinline__ int wrapmod(int v, int n) {
  v %= n;
  return v < 0 ? v + n : v;
}

// Workgroups are dealt to the 8 XCDs round-robin by linear id, and each XCD
// has its own L2.  Remap ids so every XCD owns a contiguous run of (tile,
// chunk, rhs) in tile-fastest order: x-neighbouring tiles, whose halo rows
// share cache lines, then run on the same XCD at about the same time.
struct BlockId {
  int tile, chunk, rhs;
};
__device__ __forceinline__ BlockId xcd_block() {
  const unsigned gx = gridDim.x, gy = gridDim.y;
  const unsigned total = gx * gy * gridDim.z;
  unsigned lin = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
  const unsigned full = total & ~7u;
  if (lin < full) lin = (lin & 7u) * (full >> 3) + (lin >> 3);
  BlockId b;
  b.tile = int(lin % gx);
  b.chunk = int((lin / gx) % gy);
  b.rhs = int(lin / (gx * gy));
  return b;
}

// Output-node tile of one workgroup: 32 x TY, TY from a short list per
// precision (the first entry is the default; the autotuner picks per cell).
// FP32 32 x 14 nodes = 33 x 15 elements = 8 waves, so two workgroups (16
// waves, 4 per SIMD) share a CU at up to 128 VGPRs; 32 x 16 (9 waves) fits
// only one at the 96 VGPRs that pairing would need, and ran 1.55x slower.
// Smaller tiles give small cells more workgroups.  FP64's default, 6, is four
// waves (256^3, six loads, schedule 3: 2.68 ms against 3.66 for 32 x 8).
constexpr int kTilesF32[3] = {14, 8, 6};
constexpr int kTilesF64[3] = {6, 8, 4};

// Nodes of a tile option.  All are 32 wide and as high as their name but FP64's
// default, 6, which is 16 x 14 or 32 x 6 by the grid (wide_f64): the 17 x 15 elements
// of the former fill four waves, and it computes 1.14 elements per output node
// against 1.20 (six loads, 64^3 54.9 -> 44.6 us, 100 x 90 x 80 141 -> 121, 118 x 94 x
// 111 243 -> 218, 192 x 160 x 144 815 -> 719, 256^3 2835 -> 2682).
// FP32 gains nothing from 16 x 14 (160^3 347 -> 344 us, 256^3
// 1289 -> 1334).
template <typename T, int OPT>
struct TileOption {
  static constexpr bool kSquare = std::is_same<T, double>::value && OPT == kTilesF64[0];
  static constexpr int tx = kSquare ? 16 : 32, ty = kSquare ? 14 : OPT;
};
using SquareTile = TileOption<double, kTilesF64[0]>;
struct WideTile {  // FP64's option 6 where wide_f64 holds
  static constexpr int tx = 32, ty = 6;
};

template <int TX, int TY>
struct Tile {
  static constexpr int PX = TX + 2, PY = TY + 2, PLANE = PX * PY;
  static constexpr int EX = TX + 1, EY = TY + 1, EL = EX * EY;
  static constexpr int NODES = TX * TY;
  static constexpr int NT0 = EL > NODES ? EL : NODES;
  static constexpr int NT = (NT0 + 63) / 64 * 64;
  static constexpr int ITEMS = (PLANE + NT - 1) / NT;
};

template <typename T, typename Idx, bool kScale, int TX, int TY>
__global__ void __launch_bounds__((Tile<TX, TY>::NT))
apply_kernel(ApplyArgs<T> a) {
  using TL = Tile<TX, TY>;
  __shared__ T su[2][3][TL::PLANE];
  __shared__ T sf[24][TL::EL];

  const int tid = threadIdx.x;
  const BlockId bid = xcd_block();
  const int tile = bid.tile;
  const int x0 = (tile % a.tiles_x) * TX;
  const int y0 = (tile / a.tiles_x) * TY;
  const int z0 = bid.chunk * a.zchunk;
  const int z1 = min(z0 + a.zchunk, a.nz);
  if (z0 >= a.nz) return;
  const int nx = a.nx, ny = a.ny, nz = a.nz;
  const int64_t nxy = int64_t(nx) * ny;
  const int64_t n = nxy * nz;
  const T* u = a.u + int64_t(bid.rhs) * a.rhs_stride;
  T* out = a.out + int64_t(bid.rhs) * a.rhs_stride;

  // Plane staging: each thread copies up to ITEMS halo-tile nodes.
  int ld_lds[TL::ITEMS];
  int ld_off[TL::ITEMS];  // offsets inside one z plane (nx * ny < 2^31)
#pragma unroll
  for (int k = 0; k < TL::ITEMS; ++k) {
    const int idx = tid + k * TL::NT;
    ld_lds[k] = idx < TL::PLANE ? idx : -1;
    const int px = idx % TL::PX, py = idx / TL::PX;
    ld_off[k] = wrapmod(y0 - 1 + py, ny) * nx + wrapmod(x0 - 1 + px, nx);
  }
  auto load_plane = [&](int z, int buf) {
    const int64_t base = int64_t(wrapmod(z, nz)) * nxy;
#pragma unroll
    for (int k = 0; k < TL::ITEMS; ++k) {
      if (ld_lds[k] < 0) continue;
      const int64_t node = base + ld_off[k];
#pragma unroll
      for (int c = 0; c < 3; ++c) su[buf][c][ld_lds[k]] = u[c * n + node];
    }
  };

  // Element ownership.
  const bool is_elem = tid < TL::EL;
  const int exl = tid % TL::EX, eyl = tid / TL::EX;
  const int e_xy = wrapmod(y0 - 1 + eyl, ny) * nx + wrapmod(x0 - 1 + exl, nx);
  auto compute_layer = [&](int z, int bottom, int top) {
    if (!is_elem) return;
    const int64_t voxel = int64_t(wrapmod(z, nz)) * nxy + e_xy;
    const int row = load_row<Idx>(a.index, int64_t(bid.rhs / a.group_rhs) * a.group_stride + voxel);
    const T* crow = a.table + int64_t(row) * kRowWidth;
    T c[21];
#pragma unroll
    for (int k = 0; k < 21; ++k) c[k] = crow[k];
    if constexpr (kScale) {
      const T s = T(a.scale[voxel]);
#pragma unroll
      for (int k = 0; k < 21; ++k) c[k] *= s;
    }
    T v[3][8];
#pragma unroll
    for (int cc = 0; cc < 3; ++cc)
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int ax = q & 1, ay = (q >> 1) & 1, az = q >> 2;
        v[cc][q] = su[az ? top : bottom][cc][(eyl + ay) * TL::PX + exl + ax];
      }
    element_action(v, c, a.g);
#pragma unroll
    for (int q = 0; q < 8; ++q)
#pragma unroll
      for (int cc = 0; cc < 3; ++cc) sf[q * 3 + cc][tid] = v[cc][q];
  };

  // Node ownership.
  const bool is_node = tid < TL::NODES;
  const int xl = tid % TX, yl = tid / TX;
  const bool node_valid = is_node && (x0 + xl) < nx && (y0 + yl) < ny;
  const int n_xy = (y0 + yl) * nx + (x0 + xl);
  // The four elements (ex, ey) in {xl, xl+1} x {yl, yl+1}; corner index
  // (ax, ay) = (xl+1-ex, yl+1-ey).
  auto gather = [&](int zbit, T (&acc)[3]) {
#pragma unroll
    for (int dy = 0; dy < 2; ++dy)
#pragma unroll
      for (int dx = 0; dx < 2; ++dx) {
        const int e = (yl + dy) * TL::EX + xl + dx;
        const int corner = (1 - dx) + 2 * (1 - dy) + 4 * zbit;
#pragma unroll
        for (int cc = 0; cc < 3; ++cc) acc[cc] += sf[corner * 3 + cc][e];
      }
  };

  T acc[3] = {T(0), T(0), T(0)};
  load_plane(z0 - 1, 0);
  load_plane(z0, 1);
  __syncthreads();
  compute_layer(z0 - 1, 0, 1);
  __syncthreads();
  if (is_node) gather(1, acc);
  for (int k = 0; z0 + k < z1; ++k) {
    const int z = z0 + k;
    load_plane(z + 1, k & 1);
    __syncthreads();
    compute_layer(z, (k + 1) & 1, k & 1);
    __syncthreads();
    if (is_node) {
      gather(0, acc);
      if (node_valid) {
        const int64_t node = int64_t(z) * nxy + n_xy;
#pragma unroll
        for (int cc = 0; cc < 3; ++cc) out[cc * n + node] = acc[cc];
      }
      acc[0] = acc[1] = acc[2] = T(0);
      gather(1, acc);
    }
  }
}

// ---- material frames rebuilt in the stencil ---------------------------------
// With per-voxel frames the FP32 stencil reads a phase row (the phase's C21 in
// its local frame; slot 21 holds the kind: 0 global frame, 1 local frame, 2
// local-frame cubic, 3 local-frame orthotropic) and the voxel's unit
// quaternion q = (w, x, y, z), 16 B, and rotates the row in registers: kind 1
// by the Bond stress matrix, C' = T C T^T (the reference's _rotate_packed,
// material_field.py:105-114, in engineering Voigt order 11, 22, 33, 23, 13,
// 12); kind 2 by the cubic closed form C' = C12 d(x)d + C44 (shear part) +
// a sum_m p_m p_m^T, where p_m holds the Voigt pair products of local axis m
// (column m of R) and a = C11 - C12 - 2 C44, which equals T C T^T for a cubic
// C; kind 3 by T C T^T restricted to the nine orthotropic constants: the
// columns of T are p_0, p_1, p_2 (normal) and q_s = (r_a r_b^T + r_b r_a^T)
// in Voigt form for the shear pairs s = (1, 2), (0, 2), (0, 1), so
// C' = sum_{m,n<3} C_mn p_m p_n^T + sum_s G_s q_s q_s^T.
__device__ __forceinline__ void frame_matrix(float4 q, float (&R)[3][3]) {
  const float w = q.x, x = q.y, y = q.z, z = q.w;
  R[0][0] = 1.f - 2.f * (y * y + z * z);
  R[0][1] = 2.f * (x * y - w * z);
  R[0][2] = 2.f * (x * z + w * y);
  R[1][0] = 2.f * (x * y + w * z);
  R[1][1] = 1.f - 2.f * (x * x + z * z);
  R[1][2] = 2.f * (y * z - w * x);
  R[2][0] = 2.f * (x * z - w * y);
  R[2][1] = 2.f * (y * z + w * x);
  R[2][2] = 1.f - 2.f * (x * x + y * y);
}

// Row i of the Bond stress matrix of R; shear rows/columns pair (1, 2),
// (0, 2), (0, 1).
__device__ __forceinline__ void bond_row(const float (&R)[3][3], int i, float (&t)[6]) {
  constexpr int pi[3] = {1, 0, 0}, pj[3] = {2, 2, 1};
  if (i < 3) {
#pragma unroll
    for (int b = 0; b < 3; ++b) t[b] = R[i][b] * R[i][b];
#pragma unroll
    for (int k = 0; k < 3; ++k) t[3 + k] = 2.f * R[i][pi[k]] * R[i][pj[k]];
  } else {
    const int m = i - 3;
#pragma unroll
    for (int b = 0; b < 3; ++b) t[b] = R[pi[m]][b] * R[pj[m]][b];
#pragma unroll
    for (int k = 0; k < 3; ++k) t[3 + k] = R[pi[m]][pi[k]] * R[pj[m]][pj[k]] + R[pi[m]][pj[k]] * R[pj[m]][pi[k]];
  }
}

// kForms: the kinds compiled in, 1 every kind, 2 cubic only, 3 cubic and
// orthotropic (the branches a cell does not need are left out, which keeps
// the register count down).
template <int kForms>
__device__ __forceinline__ void rotate_row(float (&c)[21], float4 q, int kind) {
  float R[3][3];
  frame_matrix(q, R);
  if (kForms == 2 || kind == 2) {
    const float c12 = c[pidx(0, 1)], c44 = c[pidx(3, 3)];
    const float an = c[pidx(0, 0)] - c12 - 2.f * c44;
    float p[3][6];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      p[m][0] = R[0][m] * R[0][m];
      p[m][1] = R[1][m] * R[1][m];
      p[m][2] = R[2][m] * R[2][m];
      p[m][3] = R[1][m] * R[2][m];
      p[m][4] = R[0][m] * R[2][m];
      p[m][5] = R[0][m] * R[1][m];
    }
#pragma unroll
    for (int i = 0; i < 6; ++i)
#pragma unroll
      for (int j = i; j < 6; ++j) {
        float v = (i < 3 && j < 3) ? c12 : 0.f;
        if (i == j) v += i < 3 ? 2.f * c44 : c44;
        const float sum = p[0][i] * p[0][j] + p[1][i] * p[1][j] + p[2][i] * p[2][j];
        c[pidx(i, j)] = fmaf(an, sum, v);
      }
    return;
  }
  if constexpr (kForms == 2) return;
  if (kForms == 3 || kind == 3) {
    constexpr int sa[3] = {1, 0, 0}, sb[3] = {2, 2, 1};  // shear pair s = (sa, sb)
    constexpr int vi[6] = {0, 1, 2, 1, 0, 0}, vj[6] = {0, 1, 2, 2, 2, 1};  // Voigt I = (vi, vj)
    float p[3][6], qs[3][6];
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
      for (int I = 0; I < 6; ++I) p[m][I] = R[vi[I]][m] * R[vj[I]][m];
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
      for (int I = 0; I < 6; ++I)
        qs[s][I] = fmaf(R[vi[I]][sa[s]], R[vj[I]][sb[s]], R[vi[I]][sb[s]] * R[vj[I]][sa[s]]);
    float nrm[3][3], g[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
#pragma unroll
      for (int n = 0; n < 3; ++n) nrm[m][n] = c[pidx(m, n)];
      g[m] = c[pidx(3 + m, 3 + m)];
    }
#pragma unroll
    for (int I = 0; I < 6; ++I) {
      float u[3], v[3];
#pragma unroll
      for (int n = 0; n < 3; ++n) {
        u[n] = fmaf(nrm[2][n], p[2][I], fmaf(nrm[1][n], p[1][I], nrm[0][n] * p[0][I]));
        v[n] = g[n] * qs[n][I];
      }
#pragma unroll
      for (int J = I; J < 6; ++J) {
        float acc = u[0] * p[0][J];
        acc = fmaf(u[1], p[1][J], acc);
        acc = fmaf(u[2], p[2][J], acc);
        acc = fmaf(v[0], qs[0][J], acc);
        acc = fmaf(v[1], qs[1][J], acc);
        c[pidx(I, J)] = fmaf(v[2], qs[2][J], acc);
      }
    }
    return;
  }
  if constexpr (kForms == 3) return;
  float out[21];
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    float ti[6], w[6];
    bond_row(R, i, ti);
#pragma unroll
    for (int l = 0; l < 6; ++l) {
      float acc = 0.f;
#pragma unroll
      for (int k = 0; k < 6; ++k) acc = fmaf(ti[k], c[pidx(k, l)], acc);
      w[l] = acc;
    }
#pragma unroll
    for (int j = i; j < 6; ++j) {
      float tj[6];
      bond_row(R, j, tj);
      float acc = 0.f;
#pragma unroll
      for (int l = 0; l < 6; ++l) acc = fmaf(w[l], tj[l], acc);
      out[pidx(i, j)] = acc;
    }
  }
#pragma unroll
  for (int k = 0; k < 21; ++k) c[k] = out[k];
}

// Stencil v2: element columns persist across the z march.  A column keeps the
// face (xy) Hadamard modes of its bottom node face and the force its previous
// layer put on that face in registers, so each layer transforms one new face
// (4 nodes), runs the modal element action, and exchanges only the 4 corner
// forces of one face through LDS.  kPF (schedule 3): the plane after next is
// prefetched into registers and the staged planes and forces are double
// buffered by layer parity, one barrier per layer; otherwise one staged plane
// and two barriers per layer.  Same arithmetic as the full 8-point
// transform, regrouped.
// kIso: cubic voxels, a.g holds the squared modal factors (strain_mode).
// kHG: the C3D8R-HG element instead of the fully integrated one.
// FP32: the register budget lets two workgroups share a CU (waves per SIMD).
// kResid: the certification form r = f - K u with ||r||^2 (FP64 operator).
// kOrtho: rows without entries outside the normal block and the shear diagonal
// (vxl_cell::ortho): 42 instead of 138 multiply-adds for the strain modes.
template <typename T, typename Idx, bool kScale, int TX, int TY, bool kFuse, bool kPF, bool kIso, bool kHG = false,
          bool kResid = false, int kFrames = 0, bool kOrtho = false>
__global__ void __launch_bounds__((Tile<TX, TY>::NT), (sizeof(T) == 4 ? (2 * Tile<TX, TY>::NT / 64 + 3) / 4 : 0))
apply_kernel_v2(ApplyArgs<T> a) {
  using TL = Tile<TX, TY>;
  // kPF: two staged planes and two force buffers (layer parity), so one
  // barrier per layer separates the writers of one buffer from its readers.
  constexpr int NB = kPF ? 2 : 1;
  __shared__ T su[NB][3][TL::PLANE];
  __shared__ T sc[NB][12][TL::EL];
  __shared__ double red[TL::NT / 64];

  const int tid = threadIdx.x;
  const BlockId bid = xcd_block();
  const int tile = bid.tile;
  const int x0 = (tile % a.tiles_x) * TX;
  const int y0 = (tile / a.tiles_x) * TY;
  const int z0 = bid.chunk * a.zchunk;
  const int z1 = min(z0 + a.zchunk, a.nz);
  if (z0 >= a.nz) return;
  if constexpr (kFuse || kResid) {
    if (a.active && !a.active[bid.rhs]) return;
  }
  const int nx = a.nx, ny = a.ny, nz = a.nz;
  const int64_t nxy = int64_t(nx) * ny;
  const int64_t n = nxy * nz;
  const T* u = a.u + int64_t(bid.rhs) * a.rhs_stride;
  T* out = a.out + int64_t(bid.rhs) * a.rhs_stride;

  int ld_lds[TL::ITEMS];
  int ld_off[TL::ITEMS];  // offsets inside one z plane (nx * ny < 2^31)
#pragma unroll
  for (int k = 0; k < TL::ITEMS; ++k) {
    const int idx = tid + k * TL::NT;
    ld_lds[k] = idx < TL::PLANE ? idx : -1;
    const int px = idx % TL::PX, py = idx / TL::PX;
    ld_off[k] = wrapmod(y0 - 1 + py, ny) * nx + wrapmod(x0 - 1 + px, nx);
  }
  auto load_plane = [&](int z, int buf) {
    const int64_t base = int64_t(wrapmod(z, nz)) * nxy;
#pragma unroll
    for (int k = 0; k < TL::ITEMS; ++k) {
      if (ld_lds[k] < 0) continue;
      const int64_t node = base + ld_off[k];
#pragma unroll
      for (int c = 0; c < 3; ++c) su[buf][c][ld_lds[k]] = u[c * n + node];
    }
  };

  const bool is_elem = tid < TL::EL;
  const int exl = tid % TL::EX, eyl = tid / TL::EX;
  const int e_xy = wrapmod(y0 - 1 + eyl, ny) * nx + wrapmod(x0 - 1 + exl, nx);
  auto face_modes = [&](T (&f)[3][4], int buf) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
#pragma unroll
      for (int a2 = 0; a2 < 4; ++a2) f[c][a2] = su[buf][c][(eyl + (a2 >> 1)) * TL::PX + exl + (a2 & 1)];
      face_forward(f[c]);
    }
  };
  T Bf[3][4], Ftp[3][4];
  // Element of layer z from its bottom (Bb) and top (Tf) face modes; returns the
  // bottom-face force (Fb) and top-face force (Ft) in face-mode form.
  const int64_t gbase = int64_t(bid.rhs / a.group_rhs) * a.group_stride;  // stacked cells
  auto row_of = [&](int z) { return load_row<Idx>(a.index, gbase + int64_t(wrapmod(z, nz)) * nxy + e_xy); };
  static_assert(kFrames == 0 || (std::is_same<T, float>::value && !kScale && !kHG && !kResid),
                "per-voxel frames: FP32 FI operator without a scale field");
  // Coefficients of the element of layer z: its row, times the voxel's scale
  // (kScale), rotated into the voxel's material frame (kFrames: 1 any
  // local-frame phase, 2 cubic local-frame phases only, 3 cubic and
  // orthotropic local-frame phases only).
  auto coeffs = [&](int z, int row, T (&c)[21]) {
    const int64_t voxel = int64_t(wrapmod(z, nz)) * nxy + e_xy;
    const T* crow = a.table + int64_t(row) * kRowWidth;
#pragma unroll
    for (int k = 0; k < 21; ++k)
      if (!kOrtho || ortho_entry(k)) c[k] = crow[k];
    if constexpr (kScale) {
      const T sc_ = T(a.scale[voxel]);
#pragma unroll
      for (int k = 0; k < 21; ++k) c[k] *= sc_;
    }
    if constexpr (kFrames != 0) {
      const int kind = int(crow[21]);
      if (kind != 0) rotate_row<kFrames>(c, a.frames[voxel], kind);
    }
  };
  auto element = [&](const T (&c)[21], const T (&Bb)[3][4], const T (&Tf)[3][4], T (&Fb)[3][4], T (&Ft)[3][4]) {
    T q[3][8], P[3][8];
#pragma unroll
    for (int cc = 0; cc < 3; ++cc)
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        q[cc][m] = Tf[cc][m] + Bb[cc][m];
        q[cc][m + 4] = Tf[cc][m] - Bb[cc][m];
      }
    if constexpr (kHG)
      element_hg<kIso>(q, c, a.g, a.hg, P);
    else
      element_modal<kIso, kOrtho>(q, c, a.g, P);
#pragma unroll
    for (int cc = 0; cc < 3; ++cc) {
      // Mode 0 (a rigid translation) carries no force: P[cc][0] is 0.
      Fb[cc][0] = -P[cc][4];
      Ft[cc][0] = P[cc][4];
#pragma unroll
      for (int m = 1; m < 4; ++m) {
        Fb[cc][m] = P[cc][m] - P[cc][m + 4];
        Ft[cc][m] = P[cc][m] + P[cc][m + 4];
      }
    }
  };

  const bool is_node = tid < TL::NODES;
  const int xl = tid % TX, yl = tid / TX;
  const bool node_valid = is_node && (x0 + xl) < nx && (y0 + yl) < ny;
  const int n_xy = (y0 + yl) * nx + (x0 + xl);
  // kFuse: u . (K u) as the sum over the nodes this thread writes of
  // u_node . (K u)_node; u at the node of plane z is read from LDS while that
  // plane is resident (one layer earlier) and kept in registers.
  double rr = 0.0;  // kResid: sum of r^2 over the nodes this thread writes
  const double rscale = kResid && a.rscale ? a.rscale[bid.rhs] : 1.0;
  // p . q: each node's product in T, summed in FP64, so that the total does not
  // depend on how the nodes are dealt to tiles and chunks.
  double pq = 0.0;
  auto node_value = [&](T (&v)[3], int buf) {
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] = su[buf][c][(yl + 1) * TL::PX + xl + 1];
  };

  // Next-plane prefetch: raw values of the plane after next are loaded into
  // registers before the element computation and stored to LDS after it, so
  // their HBM latency overlaps the arithmetic.
  T pfz[TL::ITEMS][3];
  auto prefetch = [&](int z) {
    const int64_t base = int64_t(wrapmod(z, nz)) * nxy;
#pragma unroll
    for (int k = 0; k < TL::ITEMS; ++k) {
      if (ld_lds[k] < 0) continue;
      const int64_t node = base + ld_off[k];
#pragma unroll
      for (int c = 0; c < 3; ++c) pfz[k][c] = u[c * n + node];
    }
  };
  auto commit = [&](int buf) {
#pragma unroll
    for (int k = 0; k < TL::ITEMS; ++k) {
      if (ld_lds[k] < 0) continue;
#pragma unroll
      for (int c = 0; c < 3; ++c) su[buf][c][ld_lds[k]] = pfz[k][c];
    }
  };

  // Prologue: bottom face of layer z0-1, layer z0-1 itself, then plane z0+1.
  load_plane(z0 - 1, 0);
  __syncthreads();
  if (is_elem) face_modes(Bf, 0);
  __syncthreads();
  load_plane(z0, 0);
  __syncthreads();
  T pnA[3] = {T(0), T(0), T(0)}, pnB[3] = {T(0), T(0), T(0)};  // kFuse: u at this thread's node
  if constexpr (kFuse) {
    if (node_valid) node_value(pnA, 0);
  }
  if (is_elem) {
    T Tf[3][4], Fb[3][4];
    face_modes(Tf, 0);
    T c[21];
    coeffs(z0 - 1, row_of(z0 - 1), c);
    element(c, Bf, Tf, Fb, Ftp);
#pragma unroll
    for (int cc = 0; cc < 3; ++cc)
#pragma unroll
      for (int m = 0; m < 4; ++m) Bf[cc][m] = Tf[cc][m];
  }
  __syncthreads();
  if constexpr (kPF) {
    load_plane(z0 + 1, 0);  // the first layer's buffer
    __syncthreads();
  }
  // The material row of the next layer is fetched one step ahead, so the
  // label -> row -> coefficients chain never stalls a step on two latencies.
  // (The general CG form is at its register limit and fetches it in the step.)
  constexpr bool kRowAhead = !kFuse || kOrtho;
  int row_next = kRowAhead && is_elem ? row_of(z0) : 0;
  // One layer.  Bc/Fp: this layer's bottom face modes and the force the layer
  // below put on that face; Bn/Fn receive the top face modes and top force,
  // which are the next layer's Bc/Fp.  The loop alternates two register sets,
  // so no copies are needed between layers.
  // par: layer parity (kPF: this layer's plane and force buffer; the plane
  // after next goes to the other one).
  auto layer = [&](auto par, int z, const T (&Bc)[3][4], const T (&Fp)[3][4], T (&Bn)[3][4], T (&Fn)[3][4],
                   const T (&pc)[3], T (&pn)[3]) {
    constexpr int P = kPF ? decltype(par)::value : 0;
    int row_cur = row_next;
    if constexpr (!kRowAhead) {
      if (is_elem) row_cur = row_of(z);
    } else {
      if (is_elem && z + 1 < z1) row_next = row_of(z + 1);
    }
    const bool more = kPF && z + 1 < z1;  // another step follows: it needs plane z+2
    // kResid: the right-hand side at this thread's output node, loaded before
    // the element work so that its latency is hidden.
    double fpre[3] = {0.0, 0.0, 0.0};
    if constexpr (kResid) {
      if (node_valid) {
        const int64_t base = int64_t(bid.rhs) * a.rhs_stride + int64_t(z) * nxy + n_xy;
#pragma unroll
        for (int cc = 0; cc < 3; ++cc) fpre[cc] = a.f[base + cc * n];
      }
    }
    // kFrames: the rotation runs before this step's face modes and prefetch
    // are live, which keeps the register count inside the launch bound.
    T c[21];
    if constexpr (kFrames != 0) {
      if (is_elem) coeffs(z, row_cur, c);
    }
    if constexpr (!kPF) {
      load_plane(z + 1, 0);
      __syncthreads();
    }
    // LDS holds plane z+1: read everything this step needs from it first.
    if (is_elem) face_modes(Bn, P);
    if constexpr (kFuse) {
      if (node_valid && z + 1 < z1) node_value(pn, P);
    }
    if (more) prefetch(z + 2);
    if (is_elem) {
      T Fb[3][4];
      if constexpr (kFrames == 0) coeffs(z, row_cur, c);
      element(c, Bc, Bn, Fb, Fn);
#pragma unroll
      for (int cc = 0; cc < 3; ++cc) {
        T F[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) F[m] = Fp[cc][m] + Fb[cc][m];
        face_transpose(F);
#pragma unroll
        for (int a2 = 0; a2 < 4; ++a2) sc[P][a2 * 3 + cc][tid] = F[a2];
      }
    }
    if constexpr (kPF) {
      if (more) commit(1 - P);  // the other plane buffer: last read one layer ago
    }
    __syncthreads();
    if (node_valid) {
      T acc[3] = {T(0), T(0), T(0)};
#pragma unroll
      for (int dy = 0; dy < 2; ++dy)
#pragma unroll
        for (int dx = 0; dx < 2; ++dx) {
          const int e = (yl + dy) * TL::EX + xl + dx;
          const int corner = (1 - dx) + 2 * (1 - dy);
#pragma unroll
          for (int cc = 0; cc < 3; ++cc) acc[cc] += sc[P][corner * 3 + cc][e];
        }
      const int64_t node = int64_t(z) * nxy + n_xy;
      if constexpr (kResid) {
        const int64_t base = int64_t(bid.rhs) * a.rhs_stride;
#pragma unroll
        for (int cc = 0; cc < 3; ++cc) {
          const double v = fpre[cc] - double(acc[cc]);
          if (a.r32)
            a.r32[base + cc * n + node] = float(v * rscale);
          else
            a.r64[base + cc * n + node] = v;
          rr = fma(v, v, rr);
        }
      } else {
#pragma unroll
        for (int cc = 0; cc < 3; ++cc) out[cc * n + node] = acc[cc];
        if constexpr (kFuse) pq += double(fma(pc[2], acc[2], fma(pc[1], acc[1], pc[0] * acc[0])));
      }
    }
    // kPF: no barrier here.  The next layer writes the other force buffer
    // and reads the plane committed above; this layer's buffers are written
    // again two layers on, after the next layer's barrier.
  };
  T Bf2[3][4], Ftp2[3][4];
  for (int z = z0; z < z1; z += 2) {
    layer(std::integral_constant<int, 0>(), z, Bf, Ftp, Bf2, Ftp2, pnA, pnB);
    if (z + 1 < z1) layer(std::integral_constant<int, 1>(), z + 1, Bf2, Ftp2, Bf, Ftp, pnB, pnA);
  }
  if constexpr (kFuse || kResid) {
    const double total = block_reduce_sum<TL::NT>(kResid ? rr : pq, red);
    if (tid == 0)
      a.partial[(int64_t(bid.rhs) * gridDim.y + bid.chunk) * gridDim.x + bid.tile] = total;
  }
}

template <typename T>
G9<T> cast_g(const ModalFactors& f) {
  G9<T> g;
  for (int k = 0; k < 3; ++k)
    for (int a = 0; a < 3; ++a) g.g[k][a] = T(f.g[k][a]);
  return g;
}

// The launch grid: tiles and z chunks.  A chunk of `zchunk` planes marches
// zchunk + 3 steps (the recomputed layer below and two plane loads that nothing
// hides); workgroups run in rounds of two per CU, and a last round with at most
// one per CU is shorter, but not half as long (six loads, default tiles: 2.2 us a
// step with two, 1.7 with one).  The number of chunks with the least total is
// taken, of those with at least `zmin` planes (0: the cell's setting; automatic,
// the default, is two).  Six loads, us, chunks as near eight planes as 4096
// workgroups allow -> this rule: FP32 100 x 90 x 80 74 -> 61, 118 x 94 x 111
// 123 -> 98, 160^3 346 -> 325, 256^3 1273 -> 1275; FP64 118 x 94 x 111 271 -> 243,
// 160^3 700 -> 687.  One load: 160^3 FP32 59.6 -> 50.7, FP64 118 -> 110.
// Planes per chunk of `columns` workgroup columns (at most `limit` chunks), and the
// total in those units.
inline int64_t chunk_rule(int64_t columns, int nz, int zmin, int limit, int& zchunk) {
  constexpr int kCu = 256;
  int64_t best = -1;
  for (int c = 1; c <= limit; ++c) {
    const int depth = (nz + c - 1) / c;
    if (c > 1 && depth < zmin) break;
    const int64_t groups = columns * ((nz + depth - 1) / depth);
    const int64_t rest = groups % (2 * kCu);
    const int64_t cost = (depth + 3) * (4 * (groups / (2 * kCu)) + (rest == 0 ? 0 : rest <= kCu ? 3 : 4));
    if (best < 0 || cost < best) {
      best = cost;
      zchunk = depth;
    }
  }
  return best;
}
inline int chunk_limit(int64_t columns, int nz) {
  return std::max(1, std::min(nz / kMinChunkPlanes, int((4096 + columns - 1) / columns)));
}

// Whether FP64's tile option 6 is 32 x 6 on this grid: where the rule gives it no more
// steps than 16 x 14 (grids that 32 or 6 fit better, and launches of one round), since a
// step of it costs up to a twentieth less (231 elements instead of 255).  General form,
// six loads, us, x last, 16 x 14 -> 32 x 6: 32^3 13.5 -> 12.9, 72 x 16 x 84 30.8 -> 23.5, 64 x 18 x
// 256 68.0 -> 53.3, 20 x 200 x 20 28.6 -> 26.9; with a twentieth more steps 40 x 185 x 149
// 202 -> 205.
inline bool wide_f64(const vxl_cell* cell, int nrhs) {
  const Grid& g = cell->grid;
  int depth;
  auto steps = [&](int tx, int ty) {
    const int64_t columns = int64_t((g.nx + tx - 1) / tx) * ((g.ny + ty - 1) / ty) * nrhs;
    return chunk_rule(columns, g.nz, kMinChunkPlanes, chunk_limit(columns, g.nz), depth);
  };
  return steps(WideTile::tx, WideTile::ty) <= steps(SquareTile::tx, SquareTile::ty);
}

// most: the largest number of chunks any depth setting can give.
template <typename T, int TX, int TY>
void apply_grid(const vxl_cell* cell, int nrhs, int& tiles_x, int& tiles, int& chunks, int& zchunk,
                int zmin = 0, bool most = false) {
  const int nx = cell->grid.nx, ny = cell->grid.ny, nz = cell->grid.nz;
  tiles_x = (nx + TX - 1) / TX;
  const int tiles_y = (ny + TY - 1) / TY;
  tiles = tiles_x * tiles_y;
  if (zmin <= 0) zmin = cell->zmin[std::is_same<T, double>::value ? 1 : 0];
  zmin = std::max(zmin, kMinChunkPlanes);
  const int64_t columns = int64_t(tiles) * nrhs;
  const int limit = chunk_limit(columns, nz);
  if (most) {
    chunks = limit;
    zchunk = (nz + chunks - 1) / chunks;
    return;
  }
  chunk_rule(columns, nz, zmin, limit, zchunk);
  chunks = (nz + zchunk - 1) / zchunk;
}

template <typename T, typename Idx, bool kScale, int TX, int TY, bool kHG, bool kOrtho = false>
int launch_apply_impl(const vxl_cell* cell, int nrhs, const T* u, T* out, hipStream_t s,
                      const int* active = nullptr, double* partial = nullptr, int* blocks = nullptr) {
  using TL = Tile<TX, TY>;
  ApplyArgs<T> a{};
  set_groups(a, cell, nrhs);
  a.u = u;
  a.out = out;
  a.active = active;
  a.partial = partial;
  a.rhs_stride = 3 * cell->grid.n;
  a.index = cell->mat.index;
  a.table = std::is_same<T, double>::value ? reinterpret_cast<const T*>(cell->mat.c64)
                                           : reinterpret_cast<const T*>(cell->mat.c32);
  a.scale = cell->mat.scale;
  a.nx = cell->grid.nx;
  a.ny = cell->grid.ny;
  a.nz = cell->grid.nz;
  int tiles = 0, chunks = 0;
  apply_grid<T, TX, TY>(cell, nrhs, a.tiles_x, tiles, chunks, a.zchunk);
  const ModalFactors mf = modal_factors(cell->h);
  a.g = cast_g<T>(mf);
  dim3 grid(tiles, chunks, nrhs);
  if (blocks) *blocks = tiles * chunks;
  // The C3D8R-HG element runs schedule 3 only.
  const int v = kHG ? 3 : cell->variant[std::is_same<T, double>::value ? 1 : 0];
  a.hg = T(kHG ? hg_factor(cell) / 8.0 : 0.0);
  // Cubic voxels: the squared factors go to the back-projection (one multiply
  // per gradient entry less); schedule 1 keeps the general form.
  const bool iso = cell->h[0] == cell->h[1] && cell->h[1] == cell->h[2] && v != 1;
  if (iso)
    for (int k = 0; k < 3; ++k)
      for (int d = 0; d < 3; ++d) a.g.g[k][d] = T(mf.g[k][d] * mf.g[k][d]);
#define VXL_V2(FUSE, PF)                                                                                   \
  do {                                                                                                     \
    if (iso)                                                                                               \
      hipLaunchKernelGGL((apply_kernel_v2<T, Idx, kScale, TX, TY, FUSE, PF, true, kHG, false, 0, kOrtho>), grid, dim3(TL::NT), 0, s, \
                         a);                                                                               \
    else                                                                                                   \
      hipLaunchKernelGGL((apply_kernel_v2<T, Idx, kScale, TX, TY, FUSE, PF, false, kHG, false, 0, kOrtho>), grid, dim3(TL::NT), 0, \
                         s, a);                                                                            \
  } while (0)
  if constexpr (kHG || kOrtho) {  // schedule 3 only
    if (partial)
      VXL_V2(true, true);
    else
      VXL_V2(false, true);
  } else if (partial) {
    if (v == 3)
      VXL_V2(true, true);
    else
      VXL_V2(true, false);
  } else if (v == 1) {
    hipLaunchKernelGGL((apply_kernel<T, Idx, kScale, TX, TY>), grid, dim3(TL::NT), 0, s, a);
  } else if (v == 3) {
    VXL_V2(false, true);
  } else {
    VXL_V2(false, false);
  }
#undef VXL_V2
  VXL_HIP(hipGetLastError());
  return VXL_OK;
}

// Certification residual r = f - K u (FP64 operator, default FP64 option,
// schedule 3, chunk depth by apply_grid's rule): u FP64, r into r32 or
// r64, ||r||^2 partials per workgroup; systems with active == 0 are skipped.
template <typename Idx, bool kScale, int TX, int TY, bool kOrtho = false>
int launch_resid_impl(const vxl_cell* cell, int nrhs, const double* u, const double* f, float* r32, double* r64,
                      const int* active, double* partial, int* blocks, const double* rscale, hipStream_t s) {
  using TL = Tile<TX, TY>;
  ApplyArgs<double> a{};
  set_groups(a, cell, nrhs);
  a.u = u;
  a.out = nullptr;
  a.f = f;
  a.r32 = r32;
  a.r64 = r64;
  a.rscale = rscale;
  a.active = active;
  a.partial = partial;
  a.rhs_stride = 3 * cell->grid.n;
  a.index = cell->mat.index;
  a.table = cell->mat.c64;
  a.scale = cell->mat.scale;
  a.nx = cell->grid.nx;
  a.ny = cell->grid.ny;
  a.nz = cell->grid.nz;
  int tiles = 0, chunks = 0;
  apply_grid<double, TX, TY>(cell, nrhs, a.tiles_x, tiles, chunks, a.zchunk, kMinChunkPlanes);
  const ModalFactors mf = modal_factors(cell->h);
  a.g = cast_g<double>(mf);
  const bool hg = cell->element == VXL_ELEMENT_C3D8R_HG;
  a.hg = hg ? hg_factor(cell) / 8.0 : 0.0;
  const bool iso = cell->h[0] == cell->h[1] && cell->h[1] == cell->h[2];
  if (iso)
    for (int k = 0; k < 3; ++k)
      for (int d = 0; d < 3; ++d) a.g.g[k][d] = mf.g[k][d] * mf.g[k][d];
  const dim3 grid = dim3(tiles, chunks, nrhs);
  if (blocks) *blocks = tiles * chunks;
#define VXL_R(ISO, HG) \
  hipLaunchKernelGGL((apply_kernel_v2<double, Idx, kScale, TX, TY, false, true, ISO, HG, true, 0, kOrtho>), grid, dim3(TL::NT), 0, s, a)
  if constexpr (kOrtho) {  // FI element only
    if (iso)
      VXL_R(true, false);
    else
      VXL_R(false, false);
  } else if (iso && hg) {
    VXL_R(true, true);
  } else if (iso) {
    VXL_R(true, false);
  } else if (hg) {
    VXL_R(false, true);
  } else {
    VXL_R(false, false);
  }
#undef VXL_R
  VXL_HIP(hipGetLastError());
  return VXL_OK;
}

// The default option's tile (the C3D8R-HG element and the certification have no other).
template <typename T, typename F>
int with_default_tile(const vxl_cell* cell, int nrhs, F&& f) {
  if constexpr (std::is_same<T, double>::value)
    return wide_f64(cell, nrhs) ? f(WideTile()) : f(SquareTile());
  else
    return f(TileOption<float, kTilesF32[0]>());
}

// Runtime tile choice -> template instance.
template <typename T, typename F>
int with_tile_of(const vxl_cell* cell, int nrhs, int ty, F&& f) {
  constexpr bool d = std::is_same<T, double>::value;
  if constexpr (d) {
    if (ty == kTilesF64[0] && wide_f64(cell, nrhs)) return f(WideTile());
  }
  const auto& list = d ? kTilesF64 : kTilesF32;
  if (ty == list[0]) return f(TileOption<T, (d ? kTilesF64[0] : kTilesF32[0])>());
  if (ty == list[1]) return f(TileOption<T, (d ? kTilesF64[1] : kTilesF32[1])>());
  if (ty == list[2]) return f(TileOption<T, (d ? kTilesF64[2] : kTilesF32[2])>());
  return fail("unsupported stencil tile height");
}

}  // namespace

// Orthotropic-form launches (stencil_ortho.hip) of cells with takes_ortho.
template <typename T>
int launch_apply_ortho(const vxl_cell* cell, int nrhs, const T* u, T* out, hipStream_t s, const int* active,
                       double* partial, int* blocks);
int launch_residual_ortho(const vxl_cell* cell, int nrhs, const double* u, const double* f, float* r32, double* r64,
                          const int* active, double* partial, int* blocks, const double* rscale, hipStream_t s);

}  // namespace vxl
