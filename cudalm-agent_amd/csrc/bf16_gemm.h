// bf16 GEMM of M > 32 activation rows (bf16_gemm.hip), K % 8 == 0, 16 B
// aligned W and X; PACKED: the tile-major copy (N % 16 == 0, K % 256 == 0).
#ifndef CUDALM_BF16_GEMM_H
#define CUDALM_BF16_GEMM_H

#include <hip/hip_runtime_api.h>
#include <stdint.h>

namespace cudalm_hip {

// Whether the tiles fit one launch.
bool bf16_gemm_fits(int N, int M);

template <bool PACKED>
int launch_bf16_gemm(const uint16_t* W, const uint16_t* X, uint16_t* Y, int N, int K, int M,
                     hipStream_t stream);

}  // namespace cudalm_hip

#endif
