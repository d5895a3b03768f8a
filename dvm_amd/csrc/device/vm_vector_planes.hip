// Kernels of the row build of the vector VM (vm_vector_row.h): rows that are the planes of a channel.
#include "vm_vector_row.h"

// Registers a lane: 71, 96, 121, 168, 196, 253 for 1, 2, 3, 5, 6 and 8 slabs, nothing in scratch memory. (Left to itself the
// compiler gives five slabs 171, which is one wave a SIMD less than DVM_VEC_ROW_WAVES counts on.)
#define DVM_PLANES_KERNEL(UR) \
  extern "C" __global__ void __launch_bounds__(DVM_VEC_ROW_LANES(UR##u)) __attribute__((amdgpu_waves_per_eu(DVM_VEC_ROW_WAVES(UR##u)))) dvm_vm_vec_planes##UR(const VmParam p) { vm_vector_row<UR, true>(p); }
DVM_PLANES_KERNEL(1)
DVM_PLANES_KERNEL(2)
DVM_PLANES_KERNEL(3)
DVM_PLANES_KERNEL(5)
DVM_PLANES_KERNEL(6)
DVM_PLANES_KERNEL(8)
