// The kernels of gemm_tiles_bf16.hip with one epilogue and type of result.
#include "gemm_tiles.h"

int tiles_xielu_bf16(const TilesCall& c) { return launch_tiles<EPI_XIELU, bf16_t>(c); }
