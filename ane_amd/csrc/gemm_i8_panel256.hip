// gemm_i8_panel256.hip -- the same at 256 x 256 tiles, one workgroup of eight
// waves per CU, for launches that give every CU a tile.
#define ANE_TILE 256
#define ANE_TILE_PANEL 1
#define ANE_TILE_KERNEL k_gemm_i8_panel256
#define ANE_TILE_ELIGIBLE panel256_eligible
#define ANE_TILE_LAUNCH launch_gemm_panel256
#include "gemm_i8_tile256.hip"
