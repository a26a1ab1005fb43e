// gemm_tile_ring_kernel instantiated for OpBF16x16
#define PTOAMD_RING_OP OpBF16x16
#define PTOAMD_RING_FN launch_gemm_ring_bf16
#define PTOAMD_RING_BND
#include "gemm_ring_inst.hpp"
