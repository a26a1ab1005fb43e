// gemm_tile_ring_kernel instantiated for OpF16x16
#define PTOAMD_RING_OP OpF16x16
#define PTOAMD_RING_FN launch_gemm_ring_f16
#define PTOAMD_RING_BND
#include "gemm_ring_inst.hpp"
