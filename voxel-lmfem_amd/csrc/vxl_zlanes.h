// Columns of the general z pass (vxl_fftgen.h, gen_z): which spectrum column
// each of the P columns of a workgroup holds.  Plain integer arithmetic, so that
// the host can check it too.
#pragma once

namespace vxl {

// Lanes of a group that hold a component: whole wavevectors (three components
// each) of one row of 16, of 8 or of 4.
__host__ __device__ constexpr int z_group(int P) { return P >= 16 ? 16 : P; }
__host__ __device__ constexpr int z_used(int P) { return P >= 16 ? 15 : P >= 8 ? 6 : 3; }
// Columns of a workgroup.
__host__ __device__ constexpr int z_units(int P) { return P / z_group(P) * z_used(P); }

struct ZLane {
  int comp;  // component of the wavevector
  int col;   // column that the lane loads
  bool live;
};
// A lane without a column of its own loads its group's last one, and lanes past
// the last column load that: no lane reads outside the columns its workgroup
// owns, since the pass runs in place and another workgroup may be storing there.
__host__ __device__ constexpr ZLane z_lane(int P, int p, int block, int cols) {
  const int r = p % z_group(P), used = z_used(P), first = block * z_units(P) + p / z_group(P) * used;
  const int col = first + (r < used ? r : used - 1);
  return {r % 3, col < cols ? col : cols - 1, r < used && col < cols};
}

}  // namespace vxl
