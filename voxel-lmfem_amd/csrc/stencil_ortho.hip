// Stencil launches for rows without entries outside the normal block and the
// shear diagonal (vxl_stencil.h, kOrtho).
#include "vxl_stencil.h"

namespace vxl {
namespace {

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

template <typename T>
int launch_apply_ortho(const vxl_cell* cell, int nrhs, const T* u, T* out, hipStream_t s, const int* active,
                       double* partial, int* blocks) {
  return with_tile_of<T>(cell, nrhs, cell->tile_y[std::is_same<T, double>::value ? 1 : 0], [&](auto t) {
    using O = decltype(t);
    return by_index(cell, [&](auto tag) {
      return launch_apply_impl<T, decltype(tag), false, O::tx, O::ty, false, true>(cell, nrhs, u, out, s, active,
                                                                                   partial, blocks);
    });
  });
}
template int launch_apply_ortho<float>(const vxl_cell*, int, const float*, float*, hipStream_t, const int*, double*,
                                       int*);
template int launch_apply_ortho<double>(const vxl_cell*, int, const double*, double*, hipStream_t, const int*, double*,
                                        int*);

int launch_residual_ortho(const vxl_cell* cell, int nrhs, const double* u, const double* f, float* r32, double* r64,
                          const int* active, double* partial, int* blocks, const double* rscale, hipStream_t s) {
  return with_default_tile<double>(cell, nrhs, [&](auto t) {
    using O = decltype(t);
    return by_index(cell, [&](auto tag) {
      return launch_resid_impl<decltype(tag), false, O::tx, O::ty, true>(cell, nrhs, u, f, r32, r64, active, partial,
                                                                         blocks, rscale, s);
    });
  });
}

}  // namespace vxl
