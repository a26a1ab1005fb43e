// gemm_tile_ring_kernel instantiated for OpI8x16
#define PTOAMD_RING_OP OpI8x16
#define PTOAMD_RING_FN launch_gemm_ring_i8
#include "gemm_ring_inst.hpp"
