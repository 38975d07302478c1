// q8_0_prompt.hip -- the G-mode Q8_0 product for prompts (many tokens) on
// 32 x 32 MFMA tiles, for rows of any block count and even alignment.
//
// Per output and 32-block: isum = an int8 dot of 32 (exact), s = fl(d_w * d_x),
// p[b % 16] = fmaf((float)isum, s, p[b % 16]); the FADDV tree joins the 16
// partials (the one order of the G mode, q8_0.hip).  An int32 MFMA gives 1024
// isums at once, so what bounds the product is the fp32 work per isum on the
// VALU: convert, multiply, fma.  The multiply leaves the VALU here: s over
// a tile is the outer product of 32 d_x and 32 d_w, one
// v_mfma_f32_32x32x2_f32 whose second k is zero (one rounding per product,
// denormals kept; compared bit for bit with the scalar product), on the matrix
// cores beside the VALU's convert and fma.
//
// Work split: a workgroup of 8 waves takes 64 rows x TT*32 tokens; wave w runs
// the residues b % 16 = 2w and 2w + 1 of all its outputs, so each partial
// is one wave's chain in order, and the eight waves' pair sums meet in LDS for
// the upper levels of the tree.  No wave reads another's blocks, so LDS only
// transposes: the activations are quantized into fragment order ([block][token][32],
// k_q8_act_quantize_bt) and go straight to registers, one block ahead; the
// weights go through registers into two 16-block stages in LDS, whose rows are
// 142 dwords apart (32 rows x 2 halves read dwords from 64 lanes without
// conflicts; 16-byte row strides give four lanes a bank).  (Copies to LDS move
// about 16 bytes per clock and CU here, register loads up to 64: with both
// operands copied, the copies alone took 130 of 165 us.)  Tokens are A and
// rows B of the MFMAs: a lane's results are one row (lane % 32) and 16 tokens,
// so stores of y are 128-byte runs.  The next tile's two MFMAs are issued
// ahead of each tile's VALU work.  The workgroups of one row group run on one
// XCD, whose L2 then reads those weights once for all token groups.
//
// Measured with the quantizer, before (k_q8_0_mmt / k_q8_0_mma, 16 x 16 tiles)
// and now: 14336 x 4096 at 512 tokens 188 -> 143 us (2.4 us per stage of a
// workgroup, of which the VALU's converts and fmas take about 1.2: the two MFMAs
// of a tile issue back to back, so the wave reaches that work only after the
// passes of the first), 4096 x 4096 100 -> 42, 28672 x 4096 310 -> 279, 4096 x 14336
// at 256 tokens 95 -> 63.  The 64-token forms use all 256 VGPRs and spill three or
// four.
#include "common.hpp"
#include "q8_0_prompt.hpp"

namespace ane {
namespace {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr uint32_t kRows = 64, kStageBlocks = 16, kWaves = 8;
constexpr uint32_t kOob = 0x80000000u;
// a row of a stage: 16 blocks and up to 14 bytes of lead-in; 35 chunks of 16
constexpr uint32_t kWRowChunks = (14 + kStageBlocks * 34 + 15) / 16;
constexpr uint32_t kWRow = 568;                 // LDS bytes between rows
constexpr uint32_t kStage = kRows * kWRow + 16;  // and 16 for chunks a row does not have
static_assert(kWRow >= kWRowChunks * 16 && kWRow % 8 == 0 && kWRowChunks <= 40, "eight lanes x five chunks per row");

template <int TT>
struct Lay {
    static constexpr uint32_t kTok = TT * 32;
    static constexpr uint32_t kExch = kWaves * TT * 2 * 16 * 64 * 4;
    static constexpr uint32_t kLds = 2 * kStage > kExch ? 2 * kStage : kExch;
    static_assert(kLds <= 160 * 1024, "LDS");
};

// One workgroup per row group and token group; row groups in eights (XCDs).
template <int TT>
uint64_t grid_of(uint32_t N, uint32_t T) {
    return ceil_to(((uint64_t)N + kRows - 1) / kRows, 8) * (((uint64_t)T + Lay<TT>::kTok - 1) / Lay<TT>::kTok);
}

// AL: every row starts 16-byte aligned (no lead-in bytes).
template <int TT, bool AL>
__global__ void __launch_bounds__(kWaves * 64)
k_q8_0_prompt(uint32_t N, uint32_t nb, uint32_t T, const uint8_t* Wa, uint32_t off, uint32_t wrange,
              const uint8_t* __restrict__ qxb, const float* __restrict__ dxb, uint32_t Tp, uint32_t n_tgroups,
              uint32_t n_rgroups, float* __restrict__ y) {
    using L = Lay<TT>;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t c32 = lane & 31, half = lane >> 5;
    // one row group's token groups are consecutive slots of one XCD
    const uint32_t slot = blockIdx.x >> 3, wg_r = (blockIdx.x & 7) + 8 * (slot / n_tgroups);
    if (wg_r >= n_rgroups) return;
    const uint32_t row_base = wg_r * kRows, tok_base = (slot % n_tgroups) * L::kTok;
    const uint32_t rb = nb * 34, nst = (nb + kStageBlocks - 1) / kStageBlocks;
    const __amdgpu_buffer_rsrc_t wr = make_rsrc(Wa, wrange), xr = make_rsrc(qxb, nb * Tp * 32),
                                 dr = make_rsrc(dxb, nb * Tp * 4);

    // A stage's window of a row is copied by eight lanes, five chunks each
    // (eight lanes: 128 consecutive bytes), in three batches that share registers.
    const uint32_t crow = threadIdx.x >> 3, csub = threadIdx.x & 7;
    const uint32_t wo = row_base + crow < N ? ((off + (row_base + crow) * rb) & ~15u) + 16 * csub : kOob;
    const uint32_t wl = crow * kWRow + 16 * csub;
    v4u wv[2];
    auto load_w = [&](uint32_t s, int batch) {  // past the last stage: in range or zeros, unused
#pragma unroll
        for (int q = 2 * batch; q < 5 && q < 2 * batch + 2; q++)
            wv[q - 2 * batch] =
                __builtin_amdgcn_raw_buffer_load_b128(wr, wo + q * 128, s < nst ? s * (kStageBlocks * 34) : 0, 0);
    };
    auto store_w = [&](uint32_t s, int batch) {
        uint8_t* st = smem + (s & 1) * kStage;
#pragma unroll
        for (int q = 2 * batch; q < 5 && q < 2 * batch + 2; q++) {
            uint8_t* d = st + (q < 4 ? wl + q * 128 : csub + 32 < kWRowChunks ? wl + 512 : kRows * kWRow);
            const v4u v = wv[q - 2 * batch];
            *reinterpret_cast<uint2*>(d) = make_uint2(v.x, v.y);
            *reinterpret_cast<uint2*>(d + 8) = make_uint2(v.z, v.w);
        }
    };

    const uint32_t bb0 = 2 * wave;  // this wave's first block of a stage
    // activations of one block: a lane's 16 bytes of token c32 of each tile
    // and, in the first half (k = 0 of the outer product), its scale.  Loaded
    // one block ahead.  Blocks past nb (the last stage) read block nb - 1 and
    // are taken with weight scale zero and activation scale zero.
    v4i x[TT];
    float dx[TT];
    uint32_t xo[TT];
#pragma unroll
    for (int t = 0; t < TT; t++) {
        const uint32_t tok = tok_base + t * 32 + c32;
        xo[t] = tok < Tp ? tok * 32 + 16 * half : kOob;
    }
    auto load_x = [&](uint32_t b, int t) {  // b: block of the row, wave-uniform
        const uint32_t bc = b < nb ? b : nb - 1;
        x[t] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(xr, xo[t], bc * Tp * 32, 0));
        dx[t] = __uint_as_float(
            __builtin_amdgcn_raw_buffer_load_b32(dr, half == 0 && b < nb ? xo[t] >> 3 : kOob, bc * Tp * 4, 0));
    };

    // this lane's weights: row c32 of each row tile
    auto lead = [&](uint32_t r) { return AL ? 0u : (off + (row_base + r) * rb) & 15u; };
    uint32_t wq[2];
#pragma unroll
    for (uint32_t r = 0; r < 2; r++) wq[r] = (r * 32 + c32) * kWRow + lead(r * 32 + c32) + 34 * bb0;
    v4i w[2];
    float dw[2];
    const uint32_t first = half ? 0u : 0xffffu;  // k = 0 of the outer product is the first half's
    auto read_w = [&](const uint8_t* st, uint32_t left, int j, int r) {
        const uint32_t o = wq[r] + 34 * j + 2 + 16 * half;
        const uint32_t* a = reinterpret_cast<const uint32_t*>(st + (o & ~3u));
        if (AL && j == 1) {  // 34 bb + 2 is a multiple of 4 for odd bb
#pragma unroll
            for (int k = 0; k < 4; k++) w[r][k] = (int)a[k];
        } else {
            const uint32_t sh = AL ? 2u : o & 3u;
            uint32_t d[5];
#pragma unroll
            for (int k = 0; k < 5; k++) d[k] = a[k];
#pragma unroll
            for (int k = 0; k < 4; k++) w[r][k] = (int)__builtin_amdgcn_alignbyte(d[k + 1], d[k], sh);
        }
        // masked, not selected: a select becomes a branch around the read
        const uint32_t db = *reinterpret_cast<const uint16_t*>(st + wq[r] + 34 * j);
        dw[r] = half_bits_to_float(db & (bb0 + j < left ? first : 0u));
    };

    float p[2][TT][2][16];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int t = 0; t < TT; t++)
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int i = 0; i < 16; i++) p[j][t][r][i] = 0.0f;

#pragma unroll
    for (int q = 0; q < 3; q++) {
        load_w(0, q);
        store_w(0, q);
    }
    load_w(1, 0);
#pragma unroll
    for (int t = 0; t < TT; t++) load_x(bb0, t);
    for (uint32_t s = 0; s < nst; s++) {
        wait_lgkmcnt0();  // this wave's chunks of stage s are written
        lds_barrier();    // everyone's are; everyone is done with stage s-1
        const uint8_t* st = smem + (s & 1) * kStage;
        const uint32_t left = nb - s * kStageBlocks;
        v16f sc[2];
        v16i acc[2];
        auto mma = [&](int n) {  // tile n: residue, token tile, row tile
            const int t = (n / 2) % TT, r = n & 1;
            sc[n & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(dx[t], dw[r], v16f{}, 0, 0, 0);
            acc[n & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[t], w[r], v16i{}, 0, 0, 0);
        };
        read_w(st, left, 0, 0);
        read_w(st, left, 0, 1);
        mma(0);
#pragma unroll
        for (int n = 0; n < 4 * TT; n++) {
            const int j = n / (2 * TT), t = (n / 2) % TT, r = n & 1;
            __builtin_amdgcn_sched_barrier(0);
            if (n + 1 < 4 * TT) mma(n + 1);
            __builtin_amdgcn_sched_barrier(0);
            // stage s+1: a batch to LDS, the next on the way
            if (n == TT - 1) {
                store_w(s + 1, 0);
                load_w(s + 1, 1);
            }
            if (n == 2 * TT) {
                store_w(s + 1, 1);
                load_w(s + 1, 2);
            }
            if (n == 4 * TT - 2) {
                store_w(s + 1, 2);
                load_w(s + 2, 0);
            }
            if (n + 2 == 2 * TT) {  // the first residue's tiles are all issued
                read_w(st, left, 1, 0);
                read_w(st, left, 1, 1);
            }
            // the token tile's operands are free once its second row tile is
            // issued (past the last block: nb - 1 again, unused)
            if (n % 2 == 0)
                load_x(s * kStageBlocks + bb0 + (n < 2 * TT ? 1 : kStageBlocks), t);
#pragma unroll
            for (int i = 0; i < 16; i++)
                p[j][t][r][i] = __builtin_fmaf((float)acc[n & 1][i], sc[n & 1][i], p[j][t][r][i]);
        }
    }
    // the pair sums of the eight waves meet in LDS: [tile quad][wave][lane]
    __syncthreads();
    float4* ex = reinterpret_cast<float4*>(smem);
#pragma unroll
    for (int t = 0; t < TT; t++)
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                ex[(((t * 2 + r) * 4 + q) * kWaves + wave) * 64 + lane] =
                    make_float4(p[0][t][r][4 * q] + p[1][t][r][4 * q], p[0][t][r][4 * q + 1] + p[1][t][r][4 * q + 1],
                                p[0][t][r][4 * q + 2] + p[1][t][r][4 * q + 2],
                                p[0][t][r][4 * q + 3] + p[1][t][r][4 * q + 3]);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < TT; k++) {  // 8 TT quads over 8 waves
        const uint32_t u = k * kWaves + wave, t = u >> 3, r = (u >> 2) & 1, q = u & 3;
        float4 v[kWaves];
#pragma unroll
        for (uint32_t w = 0; w < kWaves; w++) v[w] = ex[(u * kWaves + w) * 64 + lane];
        auto tree = [&](float a, float b, float c, float d, float e, float f, float g, float h) {
            return ((a + b) + (c + d)) + ((e + f) + (g + h));
        };
        const float o[4] = {tree(v[0].x, v[1].x, v[2].x, v[3].x, v[4].x, v[5].x, v[6].x, v[7].x),
                            tree(v[0].y, v[1].y, v[2].y, v[3].y, v[4].y, v[5].y, v[6].y, v[7].y),
                            tree(v[0].z, v[1].z, v[2].z, v[3].z, v[4].z, v[5].z, v[6].z, v[7].z),
                            tree(v[0].w, v[1].w, v[2].w, v[3].w, v[4].w, v[5].w, v[6].w, v[7].w)};
        const uint32_t row = row_base + r * 32 + c32, tok = tok_base + t * 32 + 8 * q + 4 * half;
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (row < N && tok + i < T) y[(uint64_t)(tok + i) * N + row] = o[i];
    }
}

template <int TT, bool AL>
int launch(uint32_t N, uint32_t nb, uint32_t T, const uint8_t* Wa, uint32_t off, uint32_t wrange, const uint8_t* qxb,
           const float* dxb, uint32_t Tp, float* y, hipStream_t s) {
    using L = Lay<TT>;
    const uint32_t rg = (N + kRows - 1) / kRows, tg = (T + L::kTok - 1) / L::kTok;
    const auto fn = k_q8_0_prompt<TT, AL>;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)L::kLds) != hipSuccess)
        return ANE_ERR_HIP;
    hipLaunchKernelGGL(fn, dim3((uint32_t)grid_of<TT>(N, T)), dim3(kWaves * 64), L::kLds, s, N, nb, T, Wa, off, wrange, qxb, dxb, Tp,
                       tg, rg, y);
    ANE_HIP_CHECK_LAUNCH();
    return ANE_OK;
}

}  // namespace

bool prompt_eligible(uint32_t N, uint32_t nb, uint32_t T, const void* W) {
    const uint64_t Tp = ((uint64_t)T + 15) & ~15ull;
    // 32-bit buffer offsets, with the windows' and tiles' over-read
    return nb > 0 && (((uintptr_t)W) & 1) == 0 && ((uint64_t)N + kRows) * nb * 34 + 2048 < kOob &&
           (nb + 1ull) * (Tp + 64) * 32 < kOob && launch_fits(T <= 32 ? grid_of<1>(N, T) : grid_of<2>(N, T), kWaves * 64);
}

int prompt_mul_mat(uint32_t N, uint32_t nb, uint32_t T, const void* W, const void* qxb, const float* dxb, uint32_t Tp,
                   float* y, hipStream_t s) {
    if (!prompt_eligible(N, nb, T, W)) return -1;
    const uintptr_t wp = reinterpret_cast<uintptr_t>(W);
    const uint32_t off = (uint32_t)(wp & 15);
    const uint8_t* Wa = reinterpret_cast<const uint8_t*>(wp - off);
    // whole dwords: the range check drops a dword that crosses the end
    const uint32_t wrange = (uint32_t)((off + (uint64_t)N * nb * 34 + 3) & ~(uint64_t)3);
    const uint8_t* q = static_cast<const uint8_t*>(qxb);
    const bool al = off == 0 && nb % 8 == 0;
    if (T <= 32)
        return al ? launch<1, true>(N, nb, T, Wa, off, wrange, q, dxb, Tp, y, s)
                  : launch<1, false>(N, nb, T, Wa, off, wrange, q, dxb, Tp, y, s);
    return al ? launch<2, true>(N, nb, T, Wa, off, wrange, q, dxb, Tp, y, s)
              : launch<2, false>(N, nb, T, Wa, off, wrange, q, dxb, Tp, y, s);
}

}  // namespace ane
