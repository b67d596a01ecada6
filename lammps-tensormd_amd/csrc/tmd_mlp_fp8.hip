// The FP8 e4m3 network kernels (tmd_mlp_kernels.h).
#include "tmd_mlp_kernels.h"

namespace tmd {

hipError_t launch_mlp_fp8(int R, const RowLayout &rl, const MlpParams &mp, const float *G, double *E, float *dEdG,
                        size_t lds, hipStream_t s, const BatchDims *dyn, int row_begin, int row_end, bool g_bf16)
{
  return launch_rows<2>(R, rl, mp, G, E, dEdG, lds, s, dyn, row_begin, row_end, g_bf16);
}

}  // namespace tmd
