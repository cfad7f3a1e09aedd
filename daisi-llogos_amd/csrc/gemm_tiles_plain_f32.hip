// The kernels of gemm_tiles_bf16.hip with one epilogue and type of result.
#include "gemm_tiles.h"

int tiles_plain_f32(const TilesCall& c) { return launch_tiles<EPI_PLAIN, float>(c); }
