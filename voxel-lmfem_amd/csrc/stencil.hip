// Stencil launchers, RHS, mean stress and centre fields (the stencil itself:
// vxl_stencil.h).
#include "vxl_stencil.h"

#include <cstdlib>

namespace vxl {

ModalFactors modal_factors(const double h[3]) {
  ModalFactors f;
  const double V = h[0] * h[1] * h[2];
  const double w[3] = {1.0, 1.0 / 3.0, 1.0 / 9.0};
  for (int k = 0; k < 3; ++k)
    for (int a = 0; a < 3; ++a) f.g[k][a] = std::sqrt(w[k] * V) / (4.0 * h[a]);
  return f;
}

namespace {

// Stencil schedule: 2 (persistent face columns), 3 (the same with the plane
// after next prefetched into registers) or 1 (per-layer full 8-node
// transform); VXL_STENCIL_VARIANT overrides the per-precision default.
int env_stencil_variant() {
  static const int v = [] {
    const char* e = std::getenv("VXL_STENCIL_VARIANT");
    if (e && e[0] >= '1' && e[0] <= '3') return e[0] - '0';
    return 0;
  }();
  return v;
}

// FP32 stencil with per-voxel material frames (vxl_cell_set_frames): phase
// index (u8), phase rows and quaternions; always the schedule-3 form, on the
// cell's tile.  With the Bond rotation the 32 x 14 tile spills (128 VGPRs,
// 18-27 registers to scratch) and is still faster than the spill-free 32 x 8
// (146 VGPRs, fewer waves per CU and more halo elements): 3.8 against 5.2 ms
// for six right-hand sides at 256^3, random frames.
template <typename F>
int frames_tile(const vxl_cell* cell, F&& f) {
  const int ty = cell->tile_y[0];
  if (ty == kTilesF32[0]) return f(std::integral_constant<int, kTilesF32[0]>());
  if (ty == kTilesF32[2]) return f(std::integral_constant<int, kTilesF32[2]>());
  return f(std::integral_constant<int, kTilesF32[1]>());
}

template <int TX, int TY>
int launch_apply_frames(const vxl_cell* cell, int nrhs, const float* u, float* out, hipStream_t s,
                        const int* active = nullptr, double* partial = nullptr, int* blocks = nullptr) {
  using TL = Tile<TX, TY>;
  ApplyArgs<float> a{};
  set_groups(a, cell, nrhs);
  a.u = u;
  a.out = out;
  a.active = active;
  a.partial = partial;
  a.rhs_stride = 3 * cell->grid.n;
  a.index = cell->frame_index;
  a.table = cell->frame_table;
  a.frames = reinterpret_cast<const float4*>(cell->frame_quat);
  a.nx = cell->grid.nx;
  a.ny = cell->grid.ny;
  a.nz = cell->grid.nz;
  int tiles = 0, chunks = 0;
  apply_grid<float, TX, TY>(cell, nrhs, a.tiles_x, tiles, chunks, a.zchunk);
  const ModalFactors mf = modal_factors(cell->h);
  a.g = cast_g<float>(mf);
  dim3 grid(tiles, chunks, nrhs);
  if (blocks) *blocks = tiles * chunks;
  const bool iso = cell->h[0] == cell->h[1] && cell->h[1] == cell->h[2];
  if (iso)
    for (int k = 0; k < 3; ++k)
      for (int d = 0; d < 3; ++d) a.g.g[k][d] = float(mf.g[k][d] * mf.g[k][d]);
#define VXL_FR(FUSE, ISO, KIND)                                                                              \
  hipLaunchKernelGGL((apply_kernel_v2<float, uint8_t, false, TX, TY, FUSE, true, ISO, false, false, KIND>), grid, \
                     dim3(TL::NT), 0, s, a)
#define VXL_FR2(FUSE, ISO)          \
  do {                              \
    if (cell->frame_forms == 2)     \
      VXL_FR(FUSE, ISO, 2);         \
    else if (cell->frame_forms == 3) \
      VXL_FR(FUSE, ISO, 3);         \
    else                            \
      VXL_FR(FUSE, ISO, 1);         \
  } while (0)
  if (partial) {
    if (iso)
      VXL_FR2(true, true);
    else
      VXL_FR2(true, false);
  } else {
    if (iso)
      VXL_FR2(false, true);
    else
      VXL_FR2(false, false);
  }
#undef VXL_FR2
#undef VXL_FR
  VXL_HIP(hipGetLastError());
  return VXL_OK;
}

template <typename T, int TX, int TY, bool kHG = false, typename... Extra>
int dispatch_apply(const vxl_cell* cell, int nrhs, const T* u, T* out, hipStream_t s, Extra... extra) {
  const bool sc = cell->mat.scale != nullptr;
  switch (cell->mat.index_kind) {
    case VXL_INDEX_U8:
      return sc ? launch_apply_impl<T, uint8_t, true, TX, TY, kHG>(cell, nrhs, u, out, s, extra...)
                : launch_apply_impl<T, uint8_t, false, TX, TY, kHG>(cell, nrhs, u, out, s, extra...);
    case VXL_INDEX_U16:
      return sc ? launch_apply_impl<T, uint16_t, true, TX, TY, kHG>(cell, nrhs, u, out, s, extra...)
                : launch_apply_impl<T, uint16_t, false, TX, TY, kHG>(cell, nrhs, u, out, s, extra...);
    case VXL_INDEX_I32:
      return sc ? launch_apply_impl<T, int32_t, true, TX, TY, kHG>(cell, nrhs, u, out, s, extra...)
                : launch_apply_impl<T, int32_t, false, TX, TY, kHG>(cell, nrhs, u, out, s, extra...);
  }
  return fail("unknown material index kind");
}

// ---- RHS: f = -V sum_e B0^T C_e E, node-owned gather (no atomics) ----------
// sig[(row * nload + r) * 6 + i] = (C_row E_r)_i, once per coefficient row.
__global__ void __launch_bounds__(256)
row_stress_kernel(const double* table, int rows, const double* macro, int nload, double* sig) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= int64_t(rows) * nload) return;
  const int64_t row = t / nload;
  const int r = int(t % nload);
  const double* c = table + row * kRowWidth;
  const double* E = macro + 6 * r;
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    double acc = 0;
#pragma unroll
    for (int j = 0; j < 6; ++j) acc = fma(c[pidx(i, j)], E[j], acc);
    sig[t * 6 + i] = acc;
  }
}

// Direct form for large row tables (one row per voxel): C_e E per element.
template <typename Idx, bool kScale>
__global__ void __launch_bounds__(256)
rhs_direct_kernel(const void* index, const double* table, const float* scale, const double* macro, int nload,
                  double* f, int nx, int ny, int nz, double gx, double gy, double gz, double volume) {
  const int64_t nxy = int64_t(nx) * ny, n = nxy * nz;
  const int64_t node = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (node >= n) return;
  const int x = int(node % nx), y = int((node / nx) % ny), z = int(node / nxy);
  for (int r = 0; r < nload; ++r) {
    const double* E = macro + 6 * r;
    double fx = 0, fy = 0, fz = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int ax = q & 1, ay = (q >> 1) & 1, az = q >> 2;
      const int64_t e = int64_t(wrapmod(z - az, nz)) * nxy + int64_t(wrapmod(y - ay, ny)) * nx +
                        wrapmod(x - ax, nx);
      const double* c = table + int64_t(load_row<Idx>(index, e)) * kRowWidth;
      const double sc = kScale ? double(scale[e]) : 1.0;
      double s[6];
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        double acc = 0;
#pragma unroll
        for (int j = 0; j < 6; ++j) acc = fma(c[pidx(i, j)], E[j], acc);
        s[i] = kScale ? acc * sc : acc;
      }
      const double dx = ax ? gx : -gx, dy = ay ? gy : -gy, dz = az ? gz : -gz;
      fx -= volume * (dx * s[0] + dy * s[5] + dz * s[4]);
      fy -= volume * (dx * s[5] + dy * s[1] + dz * s[3]);
      fz -= volume * (dx * s[4] + dy * s[3] + dz * s[2]);
    }
    double* fr = f + int64_t(r) * 3 * n;
    fr[node] = fx;
    fr[n + node] = fy;
    fr[2 * n + node] = fz;
  }
}

// Node-owned right-hand side from the per-row element stresses.  A thread owns a
// node column and marches up a chunk of `depth` planes for one load: each element
// layer's four stresses around the column give an in-plane part and a z part,
// which serve the node below the layer and the node above it.  Bound by the L1
// gathers of the stresses (16 bytes each, 12 a layer; every element used to be read
// for both of its node planes, 48 single doubles a node).  The parts are sums of
// differences of equal terms, so a uniform neighbourhood gives an exact zero.
// 110 x 96 x 100, six loads: 90 -> 62 us; 256^3: 1283 -> 949 us.
template <typename Idx, bool kScale>
__global__ void __launch_bounds__(256)
rhs_kernel(const void* index, const double* __restrict__ sig, const float* __restrict__ scale, int nload,
           double* __restrict__ f, int nx, int ny, int nz, int depth, double gx, double gy, double gz,
           double volume) {
  const int64_t nxy = int64_t(nx) * ny, n = nxy * nz;
  const int pxy = int(blockIdx.x) * int(blockDim.x) + int(threadIdx.x);
  if (pxy >= int(nxy)) return;
  const int y = pxy / nx, x = pxy - y * nx;
  const int ym = (y == 0 ? ny - 1 : y - 1) * nx, xm = x == 0 ? nx - 1 : x - 1;
  const int at[4] = {y * nx + x, y * nx + xm, ym + x, ym + xm};
  const int z0 = int(blockIdx.y) * depth, z1 = min(z0 + depth, nz);
  for (int r = int(blockIdx.z); r < nload; r += int(gridDim.z)) {
    // a: in-plane part, b: z part of the layer's force on its nodes.
    auto layer = [&](int z, double (&a)[3], double (&b)[3]) {
      const int64_t base = int64_t(z) * nxy;
      double s[4][6];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t row = load_row<Idx>(index, base + at[q]);
        const double2* sp = reinterpret_cast<const double2*>(sig + (row * nload + r) * 6);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const double2 v = sp[i];
          s[q][2 * i] = v.x;
          s[q][2 * i + 1] = v.y;
        }
        if constexpr (kScale) {
          const double sc = double(scale[base + at[q]]);
#pragma unroll
          for (int i = 0; i < 6; ++i) s[q][i] *= sc;
        }
      }
      constexpr int vx[3] = {0, 5, 4}, vy[3] = {5, 1, 3}, vz[3] = {4, 3, 2};
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const int i = vx[c], j = vy[c], k = vz[c];
        a[c] = gx * ((s[1][i] - s[0][i]) + (s[3][i] - s[2][i])) + gy * ((s[2][j] - s[0][j]) + (s[3][j] - s[1][j]));
        b[c] = gz * ((s[0][k] + s[1][k]) + (s[2][k] + s[3][k]));
      }
    };
    double al[3], bl[3];
    layer(z0 == 0 ? nz - 1 : z0 - 1, al, bl);
    double* fr = f + int64_t(r) * 3 * n + pxy;
    for (int z = z0; z < z1; ++z) {
      double au[3], bu[3];
      layer(z, au, bu);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        fr[c * n + int64_t(z) * nxy] = -volume * ((al[c] + bl[c]) + (au[c] - bu[c]));
        al[c] = au[c];
        bl[c] = bu[c];
      }
    }
  }
}

// Planes per block of the kernels that march columns: about 4096 blocks for all
// columns and loads, chunks of 2 to 16 planes (each reads one plane twice); single
// planes where those are at most 1024 blocks, all resident at once, since a second
// plane then only lengthens each thread's chain (32^3, one load, with the launch: centre
// fields 30.2 -> 28.3 us, right-hand side 27.5 -> 26.4; 64^3, six loads, 6144 single
// planes: 62.5 against 64.5, 47.1 against 52.8).
inline dim3 column_grid(int nx, int ny, int nz, int nload, int& depth) {
  const int64_t columns = (int64_t(nx) * ny + 255) / 256;
  const int loads = std::max(1, std::min(nload, 65535));
  const int64_t chunks = std::max<int64_t>(1, 4096 / (columns * loads));
  const int64_t least = columns * loads * nz <= 1024 ? 1 : 2;
  depth = int(std::max<int64_t>({least, std::min<int64_t>(16, nz / chunks), (int64_t(nz) + 65534) / 65535}));
  return dim3(unsigned(columns), unsigned((nz + depth - 1) / depth), unsigned(loads));
}

// ---- mean stress <C (E + B0 u_e)>: per-block partial sums + final reduction --
constexpr int kStressBlock = 256;

template <typename Idx, bool kScale>
__global__ void __launch_bounds__(kStressBlock)
stress_kernel(const void* index, const double* table, const float* scale, const double* u,
              const double* macro, int nload, double* partial, int nx, int ny, int nz, double gx, double gy,
              double gz) {
  __shared__ double red[kStressBlock];
  const int64_t nxy = int64_t(nx) * ny, n = nxy * nz;
  const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const bool valid = e < n;
  int x = 0, y = 0, z = 0;
  const double* c = table;
  double sc = 1.0;
  if (valid) {
    x = int(e % nx);
    y = int((e / nx) % ny);
    z = int(e / nxy);
    c = table + int64_t(load_row<Idx>(index, e)) * kRowWidth;
    if constexpr (kScale) sc = double(scale[e]);
  }
  for (int r = 0; r < nload; ++r) {
    double s[6] = {0, 0, 0, 0, 0, 0};
    if (valid) {
      double eps[6];
#pragma unroll
      for (int j = 0; j < 6; ++j) eps[j] = macro[6 * r + j];
      const double* ur = u + int64_t(r) * 3 * n;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int ax = q & 1, ay = (q >> 1) & 1, az = q >> 2;
        const int64_t node = int64_t(wrapmod(z + az, nz)) * nxy + int64_t(wrapmod(y + ay, ny)) * nx +
                             wrapmod(x + ax, nx);
        const double ux = ur[node], uy = ur[n + node], uz = ur[2 * n + node];
        const double dx = ax ? gx : -gx, dy = ay ? gy : -gy, dz = az ? gz : -gz;
        eps[0] += dx * ux;
        eps[1] += dy * uy;
        eps[2] += dz * uz;
        eps[3] += dz * uy + dy * uz;
        eps[4] += dz * ux + dx * uz;
        eps[5] += dy * ux + dx * uy;
      }
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        double acc = 0;
#pragma unroll
        for (int j = 0; j < 6; ++j) acc = fma(c[pidx(i, j)], eps[j], acc);
        s[i] = acc * sc;
      }
    }
    for (int i = 0; i < 6; ++i) {
      red[threadIdx.x] = s[i];
      __syncthreads();
      for (int w = kStressBlock / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
      }
      if (threadIdx.x == 0) partial[(int64_t(r) * 6 + i) * gridDim.x + blockIdx.x] = red[0];
      __syncthreads();
    }
  }
}

// Element-centre fields as planes [r][i][e] (strain, stress) and [r][e] (energy =
// strain . stress / 2); null outputs are skipped.  A thread owns an element column
// and marches up a chunk of `depth` layers for one load, so every node face is
// gathered once (12 loads an element) and its sums serve the layers below and above
// it.  Bound by the 104 bytes it writes and 24 it reads per element and load;
// gathering all eight nodes of each element for the six loads in turn took 292 us
// at 110 x 96 x 100 (2.8 TB/s), this takes 247 (3.3 TB/s).
template <typename Idx, bool kScale>
__global__ void __launch_bounds__(256)
center_kernel(const void* index, const double* __restrict__ table, const float* __restrict__ scale,
              const double* __restrict__ u, const double* __restrict__ macro, int nload,
              double* __restrict__ strain, double* __restrict__ stress, double* __restrict__ energy, int nx, int ny,
              int nz, int depth, double gx, double gy, double gz) {
  const int64_t nxy = int64_t(nx) * ny, n = nxy * nz;
  const int pxy = int(blockIdx.x) * int(blockDim.x) + int(threadIdx.x);
  if (pxy >= int(nxy)) return;
  const int y = pxy / nx, x = pxy - y * nx;
  const int yp = (y + 1 == ny ? 0 : y + 1) * nx, xp = x + 1 == nx ? 0 : x + 1;
  const int at[4] = {y * nx + x, y * nx + xp, yp + x, yp + xp};
  const int z0 = int(blockIdx.y) * depth, z1 = min(z0 + depth, nz);
  for (int r = int(blockIdx.z); r < nload; r += int(gridDim.z)) {
    const double* ur = u + int64_t(r) * 3 * n;
    // Differences along x and y and the sum over a node face, per component.
    auto face = [&](int z, double (&s)[3][3]) {
      const double* uz = ur + int64_t(z) * nxy;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double v0 = uz[c * n + at[0]], v1 = uz[c * n + at[1]], v2 = uz[c * n + at[2]], v3 = uz[c * n + at[3]];
        s[c][0] = (v1 - v0) + (v3 - v2);
        s[c][1] = (v2 - v0) + (v3 - v1);
        s[c][2] = (v0 + v1) + (v2 + v3);
      }
    };
    double E[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) E[j] = macro[6 * r + j];
    double lo[3][3];
    face(z0, lo);
    for (int z = z0; z < z1; ++z) {
      const int64_t e = int64_t(z) * nxy + pxy;
      double hi[3][3], d[3][3];  // d[c][a]: derivative of component c along a
      face(z + 1 == nz ? 0 : z + 1, hi);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        d[c][0] = gx * (lo[c][0] + hi[c][0]);
        d[c][1] = gy * (lo[c][1] + hi[c][1]);
        d[c][2] = gz * (hi[c][2] - lo[c][2]);
#pragma unroll
        for (int a = 0; a < 3; ++a) lo[c][a] = hi[c][a];
      }
      const double eps[6] = {E[0] + d[0][0],           E[1] + d[1][1],           E[2] + d[2][2],
                             E[3] + (d[1][2] + d[2][1]), E[4] + (d[0][2] + d[2][0]), E[5] + (d[0][1] + d[1][0])};
      if (strain) {
#pragma unroll
        for (int i = 0; i < 6; ++i) strain[(int64_t(r) * 6 + i) * n + e] = eps[i];
      }
      if (!stress && !energy) continue;
      const double* c = table + int64_t(load_row<Idx>(index, e)) * kRowWidth;
      const double sc = kScale ? double(scale[e]) : 1.0;
      double w = 0;
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        double acc = 0;
#pragma unroll
        for (int j = 0; j < 6; ++j) acc = fma(c[pidx(i, j)], eps[j], acc);
        const double v = acc * sc;
        if (stress) stress[(int64_t(r) * 6 + i) * n + e] = v;
        w += v * eps[i];
      }
      if (energy) energy[int64_t(r) * n + e] = 0.5 * w;
    }
  }
}

// Sums partial[row][0..blocks) in a fixed order; one workgroup per row.
__global__ void __launch_bounds__(256)
rows_sum_kernel(const double* partial, int64_t blocks, double scale, double* out) {
  __shared__ double red[256];
  const double* p = partial + int64_t(blockIdx.x) * blocks;
  double acc = 0;
  for (int64_t i = threadIdx.x; i < blocks; i += 256) acc += p[i];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = red[0] * scale;
}

template <typename F>
int by_index(const vxl_cell* cell, F&& f) {
  switch (cell->mat.index_kind) {
    case VXL_INDEX_U8: return f(uint8_t());
    case VXL_INDEX_U16: return f(uint16_t());
    case VXL_INDEX_I32: return f(int32_t());
  }
  return fail("unknown material index kind");
}

}  // namespace

// Measured at 256^3 (six RHS, default tiles): the plane prefetch (3) is the
// fastest schedule in both precisions (FP32 1.37 against 1.42 ms per launch).
int default_stencil_variant(int precision) {
  if (const int v = env_stencil_variant()) return v;
  (void)precision;
  return 3;
}

int launch_residual_apply(const vxl_cell* cell, int nrhs, const double* u, const double* f, float* r32, double* r64,
                          const int* active, double* partial, int* blocks, const double* rscale, hipStream_t s) {
  const bool sc = cell->mat.scale != nullptr;
  if (cell->ortho && !sc && cell->element == VXL_ELEMENT_FI)
    return launch_residual_ortho(cell, nrhs, u, f, r32, r64, active, partial, blocks, rscale, s);
  return with_default_tile<double>(cell, nrhs, [&](auto t) {
    using O = decltype(t);
    return by_index(cell, [&](auto tag) {
      using Idx = decltype(tag);
      return sc ? launch_resid_impl<Idx, true, O::tx, O::ty>(cell, nrhs, u, f, r32, r64, active, partial, blocks, rscale, s)
                : launch_resid_impl<Idx, false, O::tx, O::ty>(cell, nrhs, u, f, r32, r64, active, partial, blocks, rscale,
                                                              s);
    });
  });
}

int residual_apply_blocks(const vxl_cell* cell, int nrhs) {
  return with_default_tile<double>(cell, nrhs, [&](auto t) {
    using O = decltype(t);
    int tx, tiles, chunks, zc;
    apply_grid<double, O::tx, O::ty>(cell, nrhs, tx, tiles, chunks, zc, kMinChunkPlanes);
    return tiles * chunks;
  });
}

// Runtime tile choice -> template instance (the C3D8R-HG element runs the
// default tile only).
template <typename T, typename F>
int with_tile(const vxl_cell* cell, int nrhs, F&& f) {
  constexpr bool d = std::is_same<T, double>::value;
  const int ty = cell->element == VXL_ELEMENT_C3D8R_HG ? (d ? kTilesF64[0] : kTilesF32[0]) : cell->tile_y[d ? 1 : 0];
  return with_tile_of<T>(cell, nrhs, ty, f);
}

// The orthotropic form serves the FI element without a scale field (schedule
// 3, the default; the other schedules keep the general form).  Six loads:
// 160^3 FP32 325 -> 307 us, FP64 676 -> 624 us a launch; the sums are the same bits
// (only products with exact zeros are left out).
template <typename T>
bool takes_ortho(const vxl_cell* cell) {
  return cell->ortho && cell->element == VXL_ELEMENT_FI && !cell->mat.scale &&
         cell->variant[std::is_same<T, double>::value ? 1 : 0] == 3;
}

template <typename T>
int launch_apply_t(const vxl_cell* cell, int nrhs, const T* u, T* out, hipStream_t s) {
  if constexpr (std::is_same<T, float>::value) {
    if (cell->mfma) return launch_mfma_apply(cell, nrhs, u, out, nullptr, nullptr, nullptr, s);
    if (cell->frame_index)
      return frames_tile(cell, [&](auto ty) {
        return launch_apply_frames<32, decltype(ty)::value>(cell, nrhs, u, out, s);
      });
  }
  if (cell->element == VXL_ELEMENT_C3D8R_HG)
    return with_default_tile<T>(cell, nrhs, [&](auto t) {
      using O = decltype(t);
      return dispatch_apply<T, O::tx, O::ty, true>(cell, nrhs, u, out, s);
    });
  if (takes_ortho<T>(cell)) return launch_apply_ortho<T>(cell, nrhs, u, out, s, nullptr, nullptr, nullptr);
  return with_tile<T>(cell, nrhs, [&](auto t) {
    using O = decltype(t);
    return dispatch_apply<T, O::tx, O::ty>(cell, nrhs, u, out, s);
  });
}
template <typename T>
int launch_apply_cg_t(const vxl_cell* cell, int nrhs, const T* p, T* q, const int* active, double* partial,
                      int* blocks, hipStream_t s) {
  if constexpr (std::is_same<T, float>::value) {
    if (cell->mfma) return launch_mfma_apply(cell, nrhs, p, q, active, partial, blocks, s);
    if (cell->frame_index)
      return frames_tile(cell, [&](auto ty) {
        return launch_apply_frames<32, decltype(ty)::value>(cell, nrhs, p, q, s, active, partial, blocks);
      });
  }
  if (cell->element == VXL_ELEMENT_C3D8R_HG)
    return with_default_tile<T>(cell, nrhs, [&](auto t) {
      using O = decltype(t);
      return dispatch_apply<T, O::tx, O::ty, true>(cell, nrhs, p, q, s, active, partial, blocks);
    });
  if (takes_ortho<T>(cell)) return launch_apply_ortho<T>(cell, nrhs, p, q, s, active, partial, blocks);
  return with_tile<T>(cell, nrhs, [&](auto t) {
    using O = decltype(t);
    return dispatch_apply<T, O::tx, O::ty>(cell, nrhs, p, q, s, active, partial, blocks);
  });
}
template <typename T>
int cg_blocks_t(const vxl_cell* cell, int nrhs, bool most) {
  if constexpr (std::is_same<T, float>::value) {
    if (cell->mfma) return mfma_blocks(cell, nrhs);
    if (cell->frame_index)
      return frames_tile(cell, [&](auto ty) {
        int tx, tiles, chunks, zc;
        apply_grid<T, 32, decltype(ty)::value>(cell, nrhs, tx, tiles, chunks, zc, 0, most);
        return tiles * chunks;
      });
  }
  return with_tile<T>(cell, nrhs, [&](auto t) {
    using O = decltype(t);
    int tx, tiles, chunks, zc;
    apply_grid<T, O::tx, O::ty>(cell, nrhs, tx, tiles, chunks, zc, 0, most);
    return tiles * chunks;
  });
}

namespace {
__global__ void zero_flags_kernel(int* flag, int n) {
  if (int(threadIdx.x) < n) flag[threadIdx.x] = 0;
}

__global__ void __launch_bounds__(256)
frames_check_kernel(const uint8_t* __restrict__ index, const float4* __restrict__ quat, int64_t n, int nphase,
                    int* __restrict__ flag) {
  for (int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; e < n; e += int64_t(gridDim.x) * blockDim.x) {
    if (int(index[e]) >= nphase) flag[0] = 1;
    const float4 q = quat[e];
    const float nq = q.x * q.x + q.y * q.y + q.z * q.z + q.w * q.w;
    if (!(fabsf(nq - 1.f) <= 1e-5f)) flag[1] = 1;
  }
}
}  // namespace

void frames_release(vxl_cell* cell) {
  if (cell->frame_index) dev_free(cell->frame_index);
  if (cell->frame_table) dev_free(cell->frame_table);
  if (cell->frame_quat) dev_free(cell->frame_quat);
  cell->frame_index = nullptr;
  cell->frame_table = nullptr;
  cell->frame_quat = nullptr;
}

int launch_frames_check(const uint8_t* index, const float* quat, int64_t n, int nphase, int* flag, hipStream_t s) {
  hipLaunchKernelGGL(zero_flags_kernel, dim3(1), dim3(64), 0, s, flag, 2);
  VXL_HIP(hipGetLastError());
  const int blocks = int(std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 8192)));
  hipLaunchKernelGGL(frames_check_kernel, dim3(blocks), dim3(256), 0, s, index,
                     reinterpret_cast<const float4*>(quat), n, nphase, flag);
  VXL_HIP(hipGetLastError());
  return VXL_OK;
}

template <>
int launch_apply<float>(const vxl_cell* cell, int nrhs, const float* u, float* out, hipStream_t s) {
  return launch_apply_t<float>(cell, nrhs, u, out, s);
}
template <>
int launch_apply<double>(const vxl_cell* cell, int nrhs, const double* u, double* out, hipStream_t s) {
  return launch_apply_t<double>(cell, nrhs, u, out, s);
}

template <>
int launch_apply_cg<float>(const vxl_cell* cell, int nrhs, const float* p, float* q, const int* active,
                           double* partial, int* blocks, hipStream_t s) {
  return launch_apply_cg_t<float>(cell, nrhs, p, q, active, partial, blocks, s);
}
template <>
int launch_apply_cg<double>(const vxl_cell* cell, int nrhs, const double* p, double* q, const int* active,
                            double* partial, int* blocks, hipStream_t s) {
  return launch_apply_cg_t<double>(cell, nrhs, p, q, active, partial, blocks, s);
}
template <>
int apply_cg_blocks<float>(const vxl_cell* cell, int nrhs) {
  return cg_blocks_t<float>(cell, nrhs, false);
}
template <>
int apply_cg_blocks<double>(const vxl_cell* cell, int nrhs) {
  return cg_blocks_t<double>(cell, nrhs, false);
}

// Partial sums the CG form can need for any tile and chunk depth the cell may
// be switched to later (the solver allocates them once).
int apply_cg_blocks_max(const vxl_cell* cell, int nrhs, int precision) {
  vxl_cell probe = *cell;
  int most = 0;
  const bool d = precision == VXL_F64;
  for (int t = 0; t < 3; ++t) {
    probe.tile_y[d ? 1 : 0] = d ? kTilesF64[t] : kTilesF32[t];
    const int b = d ? cg_blocks_t<double>(&probe, nrhs, true) : cg_blocks_t<float>(&probe, nrhs, true);
    most = std::max(most, b);
  }
  if (!d) {  // the matrix-core form, which the cell may be switched to later
    probe.zmin[0] = kMinChunkPlanes;
    most = std::max(most, mfma_blocks(&probe, nrhs));
  }
  return most;
}

bool stencil_tile_supported(int precision, int tile_y) {
  const auto& list = precision == VXL_F64 ? kTilesF64 : kTilesF32;
  return tile_y == list[0] || tile_y == list[1] || tile_y == list[2];
}
int default_stencil_tile(int precision) { return precision == VXL_F64 ? kTilesF64[0] : kTilesF32[0]; }
int stencil_tile_option(int precision, int k) { return precision == VXL_F64 ? kTilesF64[k] : kTilesF32[k]; }

template <typename T>
int launch_info_t(const vxl_cell* cell, int nrhs, int (&out)[3]) {
  int tx, tiles, chunks;
  if constexpr (std::is_same<T, float>::value) {
    if (cell->mfma) {
      mfma_grid(cell, nrhs, tx, tiles, chunks, out[2]);
      out[0] = out[1] = 0;
      return VXL_OK;
    }
    if (cell->frame_index)
      return frames_tile(cell, [&](auto ty) {
        constexpr int TY = decltype(ty)::value;
        apply_grid<T, 32, TY>(cell, nrhs, tx, tiles, chunks, out[2]);
        out[0] = 32;
        out[1] = TY;
        return int(VXL_OK);
      });
  }
  return with_tile<T>(cell, nrhs, [&](auto t) {
    using O = decltype(t);
    apply_grid<T, O::tx, O::ty>(cell, nrhs, tx, tiles, chunks, out[2]);
    out[0] = O::tx;
    out[1] = O::ty;
    return int(VXL_OK);
  });
}

int stencil_launch_info(const vxl_cell* cell, int precision, int nrhs, int* tile_x, int* tile_y, int* depth,
                        int* form) {
  int v[3] = {0, 0, 0};
  VXL_TRY(precision == VXL_F64 ? launch_info_t<double>(cell, nrhs, v) : launch_info_t<float>(cell, nrhs, v));
  if (tile_x) *tile_x = v[0];
  if (tile_y) *tile_y = v[1];
  if (depth) *depth = v[2];
  if (form) {
    const bool hg = cell->element == VXL_ELEMENT_C3D8R_HG, f32 = precision == VXL_F32;
    const bool frames = f32 && cell->frame_index, mfma = f32 && cell->mfma;
    *form = (cell->ortho && !hg && !cell->mat.scale && !frames && !mfma ? VXL_FORM_ORTHO : 0) |
            (cell->h[0] == cell->h[1] && cell->h[1] == cell->h[2] ? VXL_FORM_CUBIC : 0) | (hg ? VXL_FORM_HG : 0) |
            (frames ? VXL_FORM_FRAMES : 0) | (mfma ? VXL_FORM_MFMA : 0);
  }
  return VXL_OK;
}

// One cell of a stacked cell: the same grid and rows, index block g.
vxl_cell group_view(const vxl_cell* cell, int g) {
  vxl_cell v = *cell;
  const size_t es = cell->mat.index_kind == VXL_INDEX_U8 ? 1 : cell->mat.index_kind == VXL_INDEX_U16 ? 2 : 4;
  v.mat.index = static_cast<const char*>(cell->mat.index) + size_t(g) * size_t(cell->grid.n) * es;
  v.groups = 1;
  return v;
}

int launch_rhs(const vxl_cell* cell, int nload, const double* macro_dev, double* f, double* sig, hipStream_t s) {
  if (cell->groups > 1) {  // stacked cells: each group's loads over its own index block
    if (nload % cell->groups) return fail("stacked cells: the load count must be a multiple of the cell count");
    const int per = nload / cell->groups;
    for (int g = 0; g < cell->groups; ++g) {
      const vxl_cell v = group_view(cell, g);
      VXL_TRY(launch_rhs(&v, per, macro_dev + int64_t(6) * per * g, f + int64_t(3) * cell->grid.n * per * g, sig, s));
    }
    return VXL_OK;
  }
  const auto& g = cell->grid;
  const int blocks = int((g.n + 255) / 256);
  const double gx = 0.25 / cell->h[0], gy = 0.25 / cell->h[1], gz = 0.25 / cell->h[2];
  int depth = 0;
  const dim3 gplane = column_grid(g.nx, g.ny, g.nz, nload, depth);
  if (sig) {
    const int64_t work = int64_t(cell->rows) * nload;
    hipLaunchKernelGGL(row_stress_kernel, dim3(unsigned((work + 255) / 256)), dim3(256), 0, s, cell->mat.c64,
                       cell->rows, macro_dev, nload, sig);
    VXL_HIP(hipGetLastError());
  }
  return by_index(cell, [&](auto tag) -> int {
    using Idx = decltype(tag);
    if (!sig) {
      if (cell->mat.scale)
        hipLaunchKernelGGL((rhs_direct_kernel<Idx, true>), dim3(blocks), dim3(256), 0, s, cell->mat.index,
                           cell->mat.c64, cell->mat.scale, macro_dev, nload, f, g.nx, g.ny, g.nz, gx, gy, gz,
                           cell->volume);
      else
        hipLaunchKernelGGL((rhs_direct_kernel<Idx, false>), dim3(blocks), dim3(256), 0, s, cell->mat.index,
                           cell->mat.c64, cell->mat.scale, macro_dev, nload, f, g.nx, g.ny, g.nz, gx, gy, gz,
                           cell->volume);
    } else if (cell->mat.scale)
      hipLaunchKernelGGL((rhs_kernel<Idx, true>), gplane, dim3(256), 0, s, cell->mat.index, sig,
                         cell->mat.scale, nload, f, g.nx, g.ny, g.nz, depth, gx, gy, gz, cell->volume);
    else
      hipLaunchKernelGGL((rhs_kernel<Idx, false>), gplane, dim3(256), 0, s, cell->mat.index, sig,
                         cell->mat.scale, nload, f, g.nx, g.ny, g.nz, depth, gx, gy, gz, cell->volume);
    VXL_HIP(hipGetLastError());
    return VXL_OK;
  });
}

// Per-row stresses pay off while the row table is small next to the grid;
// one-row-per-voxel tables use the direct form (scratch size 0).
int64_t rhs_scratch_size(const vxl_cell* cell, int nload) {
  if (int64_t(cell->rows) * 64 > cell->grid.n && cell->rows > 4096) return 0;
  return int64_t(cell->rows) * nload * 6;
}

// Per-block sums of the 21 coefficients (times the per-voxel scale) over
// the elements: the volume average of C is their total / N.
template <typename Idx, bool kScale>
__global__ void __launch_bounds__(256)
stiffness_sums_kernel(const void* index, const double* table, const float* scale, int64_t n, double* partial) {
  double acc[21];
#pragma unroll
  for (int c = 0; c < 21; ++c) acc[c] = 0.0;
  for (int64_t e = int64_t(blockIdx.x) * 256 + threadIdx.x; e < n; e += int64_t(gridDim.x) * 256) {
    const double* row = table + int64_t(load_row<Idx>(index, e)) * kRowWidth;
    const double sc = kScale ? double(scale[e]) : 1.0;
#pragma unroll
    for (int c = 0; c < 21; ++c) acc[c] = fma(sc, row[c], acc[c]);
  }
  __shared__ double red[4][21];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int c = 0; c < 21; ++c) {
    double v = acc[c];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if (lane == 0) red[wave][c] = v;
  }
  __syncthreads();
  if (threadIdx.x < 21)
    partial[int64_t(threadIdx.x) * gridDim.x + blockIdx.x] =
        red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
}

int64_t stress_partial_size(const vxl_cell* cell, int nload) {
  const int64_t blocks = (cell->grid.n + kStressBlock - 1) / kStressBlock;
  return blocks * 6 * nload;
}

int launch_avg_stress(const vxl_cell* cell, int nload, const double* u, const double* macro_dev,
                      double* partial, double* out_dev, hipStream_t s) {
  if (cell->groups > 1) {  // stacked cells: mean stress per group
    if (nload % cell->groups) return fail("stacked cells: the load count must be a multiple of the cell count");
    const int per = nload / cell->groups;
    for (int g = 0; g < cell->groups; ++g) {
      const vxl_cell v = group_view(cell, g);
      VXL_TRY(launch_avg_stress(&v, per, u + int64_t(3) * cell->grid.n * per * g, macro_dev + int64_t(6) * per * g,
                                partial, out_dev + int64_t(6) * per * g, s));
    }
    return VXL_OK;
  }
  const auto& g = cell->grid;
  const int64_t blocks = (g.n + kStressBlock - 1) / kStressBlock;
  const double gx = 0.25 / cell->h[0], gy = 0.25 / cell->h[1], gz = 0.25 / cell->h[2];
  VXL_TRY(by_index(cell, [&](auto tag) -> int {
    using Idx = decltype(tag);
    if (cell->mat.scale)
      hipLaunchKernelGGL((stress_kernel<Idx, true>), dim3(unsigned(blocks)), dim3(kStressBlock), 0, s,
                         cell->mat.index, cell->mat.c64, cell->mat.scale, u, macro_dev, nload, partial, g.nx, g.ny,
                         g.nz, gx, gy, gz);
    else
      hipLaunchKernelGGL((stress_kernel<Idx, false>), dim3(unsigned(blocks)), dim3(kStressBlock), 0, s,
                         cell->mat.index, cell->mat.c64, cell->mat.scale, u, macro_dev, nload, partial, g.nx, g.ny,
                         g.nz, gx, gy, gz);
    VXL_HIP(hipGetLastError());
    return VXL_OK;
  }));
  hipLaunchKernelGGL(rows_sum_kernel, dim3(6 * nload), dim3(256), 0, s, partial, blocks, 1.0 / double(g.n), out_dev);
  VXL_HIP(hipGetLastError());
  return VXL_OK;
}

int launch_center_fields(const vxl_cell* cell, int nload, const double* u, const double* macro_dev,
                         double* strain, double* stress, double* energy, hipStream_t s) {
  if (!strain && !stress && !energy) return VXL_OK;
  if (cell->groups > 1) return fail("centre fields take one cell, not a stacked cell");
  const auto& g = cell->grid;
  const double gx = 0.25 / cell->h[0], gy = 0.25 / cell->h[1], gz = 0.25 / cell->h[2];
  int depth = 0;
  const dim3 grid = column_grid(g.nx, g.ny, g.nz, nload, depth);
  return by_index(cell, [&](auto tag) -> int {
    using Idx = decltype(tag);
    if (cell->mat.scale)
      hipLaunchKernelGGL((center_kernel<Idx, true>), grid, dim3(256), 0, s, cell->mat.index, cell->mat.c64,
                         cell->mat.scale, u, macro_dev, nload, strain, stress, energy, g.nx, g.ny, g.nz, depth, gx,
                         gy, gz);
    else
      hipLaunchKernelGGL((center_kernel<Idx, false>), grid, dim3(256), 0, s, cell->mat.index, cell->mat.c64,
                         cell->mat.scale, u, macro_dev, nload, strain, stress, energy, g.nx, g.ny, g.nz, depth, gx,
                         gy, gz);
    VXL_HIP(hipGetLastError());
    return VXL_OK;
  });
}

int launch_stiffness_sums(const vxl_cell* cell, double* partial, int blocks, hipStream_t s) {
  return by_index(cell, [&](auto tag) -> int {
    using Idx = decltype(tag);
    if (cell->mat.scale)
      hipLaunchKernelGGL((stiffness_sums_kernel<Idx, true>), dim3(unsigned(blocks)), dim3(256), 0, s, cell->mat.index,
                         cell->mat.c64, cell->mat.scale, cell->grid.n, partial);
    else
      hipLaunchKernelGGL((stiffness_sums_kernel<Idx, false>), dim3(unsigned(blocks)), dim3(256), 0, s, cell->mat.index,
                         cell->mat.c64, cell->mat.scale, cell->grid.n, partial);
    VXL_HIP(hipGetLastError());
    return VXL_OK;
  });
}

}  // namespace vxl
