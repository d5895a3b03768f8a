// Kernels of the row build of the vector VM (vm_vector_row.h): rows of one reduced axis.
#include "vm_vector_row.h"

// Registers a lane: 79, 95, 128, 128 (and 19 more in scratch memory), 167, 200, 255 for 1 to 6 and 8 slabs: 5, 5, 4, 4, 3,
// 2, 2 waves a SIMD (DVM_VEC_ROW_WAVES).
#define DVM_ROW_KERNEL(UR) \
  extern "C" __global__ void __launch_bounds__(DVM_VEC_ROW_LANES(UR##u)) dvm_vm_vec_row##UR(const VmParam p) { vm_vector_row<UR, false>(p); }
DVM_ROW_KERNEL(1)
DVM_ROW_KERNEL(2)
DVM_ROW_KERNEL(3)
DVM_ROW_KERNEL(4)
DVM_ROW_KERNEL(5)
DVM_ROW_KERNEL(6)
DVM_ROW_KERNEL(8)
