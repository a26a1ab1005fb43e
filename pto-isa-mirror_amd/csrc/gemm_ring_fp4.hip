// gemm_tile_ring_kernel instantiated for OpFP4x16
#define PTOAMD_RING_OP OpFP4x16
#define PTOAMD_RING_FN launch_gemm_ring_fp4
#include "gemm_ring_inst.hpp"
