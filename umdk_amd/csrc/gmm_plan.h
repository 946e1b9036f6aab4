// Which block of a decode GEMM launch (4 waves, gmm.hip) runs which tiles: plain integer rules, for the kernels and for
// host programs that check them.
#pragma once

#ifdef __HIPCC__
#define CAM_PLAN_FN __host__ __device__ __forceinline__
#else
#define CAM_PLAN_FN inline
#endif

namespace cam {

// 32-row tiles throughout (n32 of them), or 64-row tiles for the experts of more than 32 rows (n64 tiles of both
// heights)?  Blocks run their tiles one after another, so what counts is rounds over the G blocks, and a 64-row tile
// takes 1.25 to 1.35 times a 32-row one (the plain GEMM of 16 fp8 experts of 14 to 66 rows, K = 1024, N = 2304: 306 tiles,
// two rounds, 20.2 us, against 486 tiles, also two rounds, 15.5 us).  64-row tiles from a fifth fewer rounds on (8 experts
// of 47 rows, H = 7168, I = 2048, four rounds to three in GMM2: fp8 88 against 103 us, int8 91 against 94 us at a
// quarter, bf16 152 against 156 us).
CAM_PLAN_FN bool small_rows32(int n32, int n64, int G)
{
    if (n32 <= G)
        return true;
    return n64 == n32 || 5 * ((n64 + G - 1) / G) > 4 * ((n32 + G - 1) / G);
}

}  // namespace cam
