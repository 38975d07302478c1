// gemm_i8_panel128.hip -- the contraction loop of gemm_i8_tile256.hip at
// 128 x 128 output tiles for dense_i8 / dense_u8s8: B read from the SMOPA
// panels through registers (PanelB), A by copies to LDS, two workgroups of
// four waves per CU.
#define ANE_TILE 128
#define ANE_TILE_PANEL 1
#define ANE_TILE_KERNEL k_gemm_i8_panel128
#define ANE_TILE_ELIGIBLE panel128_eligible
#define ANE_TILE_LAUNCH launch_gemm_panel128
#include "gemm_i8_tile256.hip"
