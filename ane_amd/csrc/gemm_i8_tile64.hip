// gemm_i8_tile64.hip -- the contraction loop of gemm_i8_tile256.hip at 64 x 64
// output tiles (4 waves of one 32 x 32 block, a 4-stage ring of 16 KB slices,
// two workgroups per CU), for shapes whose 128-tiles would leave more than
// half of the CUs idle.
#define ANE_TILE 64
#define ANE_TILE_STAGES 4
#define ANE_TILE_KERNEL k_gemm_i8_tile64
#define ANE_TILE_ELIGIBLE tile64_eligible
#define ANE_TILE_LAUNCH launch_gemm_tile64
#include "gemm_i8_tile256.hip"
