// gemm_i8.hpp -- parameters shared by the int8 contraction kernels.
#pragma once

#include "common.hpp"

namespace ane {

struct GemmParams {
    const int8_t* A;      // row-major, K contiguous
    uint64_t lda;         // bytes between rows of A
    const int8_t* B;      // Bt (N x K, K contiguous) or SMOPA panels
    uint64_t ldb;         // Bt: bytes between rows; panel: groups per panel (G)
    uint32_t rowsA;       // rows of A that may be read (others read as 0)
    uint32_t colsB;       // columns of B that may be read (others read as 0)
    uint32_t Kp;          // contraction length, multiple of 16
    uint32_t Mout, Nout;  // output rows / columns written
    float s;              // epilogue multiplier (when sdev == nullptr)
    const float* sdev;    // device {sa, sb}: s = (sa*sb)*smul
    float smul;
    const float* bias;    // fp32[Nout] or nullptr (adds +0.0f)
    float lo;             // ReLU floor: +0 or -FLT_MAX
    float* C;             // fp32 output, row stride ldc
    uint64_t ldc;
    int32_t* Craw;        // raw int32 output instead (debug entry)
    // Integer GEMM epilogue (igemm.hip) instead of the one above: C =
    // fl((float)(acc + 128 colsum[j] + 128 rowsum[i] + corr) * s), the sums given
    // as partials of nsum runs of K (colsum[p * Nout + j], rowsum[p * Mout + i];
    // null: none).
    bool ig;
    const int32_t* igc;
    const int32_t* igr;
    uint32_t nsum, corr;
};

// Partials per column or row, at most: each reader adds them up, so they pay
// only while they are few (igemm.hip).
constexpr uint32_t kIgParts = 16;

// 128 * the sum of the partials of column or row x (n columns or rows in all); 0
// without.  U loads are in flight at a time.
template <uint32_t U = 8>
__device__ __forceinline__ uint32_t ig_sum(const int32_t* part, uint32_t nsum, uint32_t n, uint32_t x) {
    if (!part) return 0u;
    const int32_t* c = part + (x < n ? x : n - 1);
    if (nsum == 1) return 128u * (uint32_t)c[0];
    uint32_t t = 0;
    for (uint32_t p = 0; p < nsum; p += U) {
        uint32_t v[U];
#pragma unroll
        for (uint32_t q = 0; q < U; q++) v[q] = (uint32_t)c[(uint64_t)(p + q < nsum ? p + q : p) * n];
#pragma unroll
        for (uint32_t q = 0; q < U; q++) t += p + q < nsum ? v[q] : 0u;
    }
    return 128u * t;
}
__device__ __forceinline__ float ig_out(const GemmParams& p, int32_t acc, uint32_t col, uint32_t row) {
    return __fmul_rn((float)(int32_t)((uint32_t)acc + col + row + p.corr), p.s);
}

// The contraction with any of the epilogues on signed rows of A and Bt
// (gemm_i8.hip chooses the kernel).
int launch_gemm_rows(const GemmParams& p, hipStream_t s);

// dense_fused_i8 operand preparation (quantize_fused.hip): absmax partials
// (kFusedPartials per tensor), qA (M x Kp), qBt (N x Kp), scales {sa, sb},
// and the launch's wait record wstatus: wstatus[0] = the number of
// workgroups that met at the grid-wide wait (0 on the two-pass route, which
// has none), wstatus[1 + w] = what workgroup w saw there (0, or timed-out /
// mixed-arrival bits).  Every launch writes it, so no clearing is needed.
constexpr uint32_t kFusedPartials = 1024;
int launch_fused_quantize(const float* A, const float* B, uint32_t M, uint32_t N, uint32_t K,
                          uint32_t Kp, uint32_t* partials, int8_t* qA, int8_t* qBt, float* scales,
                          uint32_t* wstatus, bool whole_op, hipStream_t s);
// The whole of dense_fused_i8 for small operands (K <= 1024, at most 512
// tiles of 16 x 16): the absmax pass, then one launch that quantizes each tile's rows
// and columns into LDS and contracts them (quantize_fused.hip).  Writes C,
// the scales and the wait record, not qA / qBt.
bool small_fused_eligible(uint32_t M, uint32_t N, uint32_t K);
int launch_fused_small(const float* A, const float* B, uint32_t M, uint32_t N, uint32_t K, float smul, float lo,
                       float* C, uint32_t* partials, float* scales, uint32_t* wstatus, hipStream_t s);
// The whole of dense_fused_i8 for at most 16 rows of A in one launch with a
// grid-wide wait (quantize_fused.hip, k_fused_strip): M <= 16, K % 512 == 0,
// K <= 4096, N % 16 == 0, at most one 16-column strip of B per workgroup,
// 16-byte aligned operands and at least 12 MiB of B.  Writes C, the scales
// and the wait record, not qA / qBt.  Returns false when the route cannot
// run (nothing queued); true when it was queued (*status = ANE_ERR_HIP if the
// launch failed after that).
bool strip_fused_eligible(uint32_t M, uint32_t N, uint32_t K, const float* A, const float* B);
bool launch_fused_strip(const float* A, const float* B, uint32_t M, uint32_t N, uint32_t K, float smul, float lo,
                        float* C, uint32_t* partials, float* scales, uint32_t* wstatus, hipStream_t s,
                        int* status);
// The current device's record of failed grid-wide waits (sticky bits; 0 if
// the resident route never ran): read, and cleared together with the
// counters once the device is idle when nonzero.
int resident_slot_check(uint32_t* bits);
bool resident_mixed_bit(uint32_t bits);

// 256 x 256 tile kernel (gemm_i8_tile256.hip): Bt layout, signed A, K a
// multiple of 64 (run as 128-byte slices, an odd last half read as zeros),
// 16-byte aligned rows, and enough rows/columns to fill 256-wide tiles
// reasonably.
// any_rows: also fewer rows than one tile (rows past Mout read as zeros).
// ksplit > 1 splits K over gridDim.y workgroups per tile, each writing its
// int32 plane y of Craw (Mout x ldc): raw output only.
bool tile256_eligible(const GemmParams& p, bool any_rows = false);
int launch_gemm_tile256(const GemmParams& p, hipStream_t s, uint32_t ksplit = 1);

// The same loop at 128 x 128 tiles (gemm_i8_tile128.hip).
bool tile128_eligible(const GemmParams& p, bool any_rows = false);
int launch_gemm_tile128(const GemmParams& p, hipStream_t s, uint32_t ksplit = 1);
// The same at 128 x 128 tiles on a 3-stage ring with 8 waves, one workgroup
// per CU (gemm_i8_tile128d.hip): for launches of at most one workgroup per CU.
bool tile128d_eligible(const GemmParams& p, bool any_rows = false);
int launch_gemm_tile128d(const GemmParams& p, hipStream_t s, uint32_t ksplit = 1);

// The same at 64 x 64 tiles (gemm_i8_tile64.hip).
bool tile64_eligible(const GemmParams& p, bool any_rows = false);
int launch_gemm_tile64(const GemmParams& p, hipStream_t s, uint32_t ksplit = 1);

// The same loop with B in SMOPA panels (ldb = Kp / 4 groups of 64 bytes per
// panel) and A int8 or uint8, at 256 x 256 (gemm_i8_panel256.hip) and 128 x
// 128 tiles (gemm_i8_panel128.hip).  Rows and columns past the operands'
// ends read as zeros.
bool panel256_eligible(const GemmParams& p);
int launch_gemm_panel256(const GemmParams& p, bool a_unsigned, hipStream_t s);
bool panel128_eligible(const GemmParams& p);
int launch_gemm_panel128(const GemmParams& p, bool a_unsigned, hipStream_t s);

// Few-row kernel (gemm_i8_skinny.hip): Bt layout, signed A, one workgroup per
// 16 columns and up to 128 rows, or per 16 columns and 64 rows while that is
// at most wgs_max workgroups.
bool skinny_eligible(const GemmParams& p, uint64_t wgs_max);
int launch_gemm_skinny(const GemmParams& p, hipStream_t s);
// The same on SMOPA panels, one workgroup per panel, A int8 or uint8.
bool panel_skinny_eligible(const GemmParams& p, uint64_t wgs_max);
int launch_gemm_panel_skinny(const GemmParams& p, bool a_unsigned, hipStream_t s);

}  // namespace ane
