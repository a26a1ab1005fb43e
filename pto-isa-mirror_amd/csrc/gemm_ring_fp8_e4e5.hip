// gemm_tile_ring_kernel instantiated for OpFP8x16<0, 1>
#define PTOAMD_RING_OP OpFP8x16<0, 1>
#define PTOAMD_RING_FN launch_gemm_ring_fp8_e4e5
#include "gemm_ring_inst.hpp"
