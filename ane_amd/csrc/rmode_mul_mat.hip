// rmode_mul_mat.hip -- the R-mode product (fp32 x, the handlers' 16 fma
// lanes per output) for 2 or more tokens on Q4_0 and Q8_0 weights: what
// q4_0_gemv (0x58, bytecode_interpreter.s:7071-7126) and q8_0_gemv (0x57,
// :7010-7063) compute per token, for all tokens in one launch.
//
// An output y[t][m] is 16 chains: chain l applies acc = fma(w, x, acc) to
// elements l and 16 + l of every 32-block in order; the FADDV tree joins
// them.  One chain step over a 16 x 16 tile of outputs is a rank-1 update,
// and v_mfma_f32_16x16x1_4b_f32 runs four such tiles at once, each output
// one correctly rounded fp32 fma with denormals kept (compared bit for bit
// with fmaf on random, denormal, tiny and special operands).  So the four
// blocks of the instruction are four chains of the same outputs, and the
// chains run on the matrix cores with the handler's own roundings.
//
// What bounds it: the fp32 MFMA rate, 2*N*K*T flops at the 134 TFLOP/s that
// a loop of this instruction reaches, with the weights' decode (about five
// VALU operations per weight, once per 16*TT tokens) on the VALU beside it;
// below that, the barrier and first reads of each stage with two waves per
// SIMD.  Measured at 4096 x 4096 Q4_0 (a call among many), before (one GEMV
// launch per token, decoding every weight again with the fmas on the VALU) and
// now: 2 tokens 17.9 -> 13.0 us, 16 144 -> 13.5, 64 579 -> 32.2, 128 1158 -> 49.7
// (86 TFLOP/s), 512 4614 -> 182 (94 TFLOP/s); one token stays on the GEMV (9.2
// us), and two or three over many rows do (gemvs_faster).  A kernel trace of a
// dozen passes shows longer ones: 14.6, 36.1, 56.5 and 210 us for 16 to 512 tokens.
//
// Work split: a workgroup takes RT*16 rows x WT*TT*16 tokens with 4 x WT
// waves.  Wave j of a token group runs chains 4j .. 4j+3 of all its
// outputs: it reads byte 4j + g of a block's quants (lane group g = lane /
// 16, one weight per lane and half block) and the matching x, so no weight is
// decoded twice in a token group, and the four waves' subtotals are aligned
// quarters of the FADDV tree.  D of the instruction holds block g's tile in
// registers 4g .. 4g+3 (lane: column lane % 16, row 4*(lane/16) + i), so
// a wave's four chains of an output meet in one lane's registers.
//
// Both operands are staged through registers into two LDS buffers of P
// blocks: the loads of stage s+2 are in flight while stage s is multiplied.
// x rows are padded by 16 bytes (lane = token: 16 tokens x 4 lane groups
// read 64 distinct banks).  Weight rows sit at any even byte offset: a
// stage copies the 16-byte-aligned window around its P blocks.
#include "common.hpp"
#include "rmode_mul_mat.hpp"

#include <type_traits>

namespace ane {

// The tile that many tokens take, 512 threads per 64 x 64 outputs.  The others
// run below one such workgroup per CU, or for up to 32 tokens: 16 threads a row
// at most, with N below 2^27 by the weights' 2 GiB.
bool rmode_launch_fits(uint32_t N, uint32_t T) {
    return T <= 32 || launch_fits(((uint64_t)N + 63) / 64 * (((uint64_t)T + 63) / 64), 512);
}

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr uint32_t kMaxP = 16;  // blocks per stage, at most
constexpr uint32_t kOob = 0x80000000u;

// One weight per lane and half block: chains 4j + g, element 4j + g of the
// first half (w0) and of the second (w1).  fetch reads a block's bytes from
// LDS, decode turns them into the two weights.
struct Q40Lane {
    static constexpr uint32_t kBytes = 18;
    uint32_t d, b;
    __device__ void fetch(const uint8_t* s, uint32_t e) {
        d = *reinterpret_cast<const uint16_t*>(s);
        b = s[2 + e];
    }
    __device__ void decode(float& w0, float& w1) const {
        const float df = half_bits_to_float(d);
        // as qf::Q40::acc: q - 8 through the float 2^23 + q, the high nibble
        // in place against d / 16 (exact)
        const float lo = __fsub_rn(__uint_as_float((b & 15u) | 0x4B000000u), 8388616.0f);
        const float hi = __fsub_rn(__uint_as_float((b & 0xF0u) | 0x4B000000u), 8388736.0f);
        w0 = __fmul_rn(lo, df);
        w1 = __fmul_rn(hi, __fmul_rn(df, 0.0625f));
    }
};
struct Q80Lane {
    static constexpr uint32_t kBytes = 34;
    uint32_t d;
    int32_t a, b;
    __device__ void fetch(const uint8_t* s, uint32_t e) {
        d = *reinterpret_cast<const uint16_t*>(s);
        a = (int8_t)s[2 + e];
        b = (int8_t)s[18 + e];
    }
    __device__ void decode(float& w0, float& w1) const {
        const float df = half_bits_to_float(d);
        w0 = __fmul_rn((float)a, df);
        w1 = __fmul_rn((float)b, df);
    }
};

template <class F, int RT, int TT, int WT, int P>
struct RLayout {
    static constexpr int kWaves = 4 * WT, kThreads = kWaves * 64;
    static constexpr uint32_t kRows = RT * 16, kTok = WT * TT * 16;
    static constexpr uint32_t kP = P;                          // 32-blocks per stage
    static constexpr uint32_t kXChunks = P * 8;                // 16-byte chunks of x per token and stage
    static constexpr uint32_t kXStride = (kXChunks + 1) * 16;  // bytes between tokens in LDS
    // a row's window: up to 14 bytes of lead-in before the stage's blocks
    static constexpr uint32_t kWChunks = (14 + kP * F::kBytes + 15) / 16;
    // an odd number of chunks between rows spreads them over the banks
    static constexpr uint32_t kWStride = (kWChunks | 1) * 16;
    static constexpr uint32_t kXBytes = kTok * kXStride, kWBytes = kRows * kWStride;
    static constexpr uint32_t kStage = kXBytes + kWBytes;
    static constexpr uint32_t kXPer = (kTok * kXChunks + kThreads - 1) / kThreads;
    static constexpr uint32_t kWPer = (kRows * kWChunks + kThreads - 1) / kThreads;
    static constexpr uint32_t kExch = WT * RT * TT * 4 * 64 * 16;
    static constexpr uint32_t kLds = 2 * kStage > kExch ? 2 * kStage : kExch;
    static_assert(kLds <= 160 * 1024, "LDS");
};

template <class F, int RT, int TT, int WT, int P>
__global__ void __launch_bounds__(4 * WT * 64)
k_rmode_mul_mat(uint32_t N, uint32_t nb, uint32_t T, const float* __restrict__ x, const uint8_t* Wa, uint32_t off,
                uint32_t wrange, uint32_t n_tgroups, float* __restrict__ y) {
    using L = RLayout<F, RT, TT, WT, P>;
    constexpr uint32_t kP = L::kP, kXChunks = L::kXChunks, kXStride = L::kXStride;
    __shared__ __attribute__((aligned(16))) uint8_t smem[L::kLds];
    const uint32_t tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), j = wave & 3, wt = wave >> 2;
    const uint32_t tok_base = (blockIdx.x % n_tgroups) * L::kTok, row_base = (blockIdx.x / n_tgroups) * L::kRows;
    const uint32_t K = nb * 32, rb = nb * F::kBytes;
    const uint32_t nst = (nb + kP - 1) / kP;
    const __amdgpu_buffer_rsrc_t xr = make_rsrc(x, T * K * 4), wr = make_rsrc(Wa, wrange);

    // this thread's chunks of a stage: x token/chunk, weight row/chunk
    uint32_t xo[L::kXPer], xl[L::kXPer], wo[L::kWPer], wl[L::kWPer];
#pragma unroll
    for (uint32_t i = 0; i < L::kXPer; i++) {
        const uint32_t c = i * L::kThreads + tid, t = c / kXChunks, q = c % kXChunks;
        const bool on = c < L::kTok * kXChunks;
        xo[i] = on && tok_base + t < T ? (tok_base + t) * K * 4 + q * 16 : kOob;
        xl[i] = on ? t * kXStride + q * 16 : kOob;
    }
#pragma unroll
    for (uint32_t i = 0; i < L::kWPer; i++) {
        const uint32_t c = i * L::kThreads + tid, r = c / L::kWChunks, q = c % L::kWChunks;
        const bool on = c < L::kRows * L::kWChunks;
        wo[i] = on && row_base + r < N ? off + (row_base + r) * rb : kOob;  // byte of the row
        wl[i] = on ? L::kXBytes + r * L::kWStride + q * 16 : kOob;
    }
    v4u xv[L::kXPer], wv[L::kWPer];
    auto load = [&](uint32_t s) {
#pragma unroll
        for (uint32_t i = 0; i < L::kXPer; i++) {
            const uint32_t o = xo[i] != kOob && s < nst ? xo[i] + s * (kP * 128) : kOob;
            xv[i] = __builtin_amdgcn_raw_buffer_load_b128(xr, o, 0, 0);
        }
#pragma unroll
        for (uint32_t i = 0; i < L::kWPer; i++) {
            const uint32_t q = (i * L::kThreads + tid) % L::kWChunks;
            const uint32_t o = wo[i] != kOob && s < nst ? ((wo[i] + s * (kP * F::kBytes)) & ~15u) + q * 16 : kOob;
            wv[i] = __builtin_amdgcn_raw_buffer_load_b128(wr, o, 0, 0);
        }
    };
    auto store = [&](uint32_t s) {
        uint8_t* st = smem + (s & 1) * L::kStage;
#pragma unroll
        for (uint32_t i = 0; i < L::kXPer; i++)
            if (xl[i] != kOob) *reinterpret_cast<v4u*>(st + xl[i]) = xv[i];
#pragma unroll
        for (uint32_t i = 0; i < L::kWPer; i++)
            if (wl[i] != kOob) *reinterpret_cast<v4u*>(st + wl[i]) = wv[i];
    };

    v16f acc[RT][TT];
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = 0; t < TT; t++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[r][t][i] = 0.0f;

    const uint32_t e = 4 * j + g;  // this lane's chain
    load(0);
    store(0);
    load(1);
    __syncthreads();
    // one stage of nblk blocks; whole stages pass the constant kP, so their
    // blocks are one straight run of code and the next block's reads and
    // decode sit between this one's MFMAs
    auto stage = [&](uint32_t s, auto whole) {
        constexpr bool kWhole = decltype(whole)::value;
        if (s + 1 < nst) store(s + 1);  // its buffer was last read in stage s-1
        load(s + 2);
        const uint8_t* st = smem + (s & 1) * L::kStage;
        const uint8_t* xs = st + (wt * TT * 16 + c16) * kXStride + e * 4;
        const uint32_t nblk = nb - s * kP;
        const uint8_t* ws[RT];
#pragma unroll
        for (int r = 0; r < RT; r++) {
            const uint32_t lr = r * 16 + c16;
            const uint32_t at = off + (row_base + lr) * rb + s * (kP * F::kBytes);
            ws[r] = st + L::kXBytes + lr * L::kWStride + (at & 15u);
        }
        // block b + 1 is read from LDS ahead of block b's MFMAs and decoded
        // between them
        F raw[RT];
        float w0[2][RT], w1[2][RT], x0[2][TT], x1[2][TT];
        auto fetch = [&](uint32_t b) {
#pragma unroll
            for (int r = 0; r < RT; r++) raw[r].fetch(ws[r] + b * F::kBytes, e);
#pragma unroll
            for (int t = 0; t < TT; t++) {
                x0[b & 1][t] = *reinterpret_cast<const float*>(xs + t * 16 * kXStride + b * 128);
                x1[b & 1][t] = *reinterpret_cast<const float*>(xs + t * 16 * kXStride + b * 128 + 64);
            }
        };
        auto decode = [&](uint32_t b) {
#pragma unroll
            for (int r = 0; r < RT; r++) raw[r].decode(w0[b & 1][r], w1[b & 1][r]);
        };
        fetch(0);
        decode(0);
#pragma unroll
        for (uint32_t b = 0; b < kP; b++) {
            if (!kWhole && b >= nblk) break;
            __builtin_amdgcn_sched_barrier(0);
            if (b + 1 < kP) fetch(b + 1);
#pragma unroll
            for (int r = 0; r < RT; r++)
#pragma unroll
                for (int t = 0; t < TT; t++)
                    acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x1f32(x0[b & 1][t], w0[b & 1][r], acc[r][t], 0, 0, 0);
#pragma unroll
            for (int r = 0; r < RT; r++)
#pragma unroll
                for (int t = 0; t < TT; t++)
                    acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x1f32(x1[b & 1][t], w1[b & 1][r], acc[r][t], 0, 0, 0);
            if (b + 1 < kP) decode(b + 1);
            if (kWhole) {
                // reads first, then the MFMAs with the decode spread over them
                __builtin_amdgcn_sched_group_barrier(0x100, 8 * RT + 2 * TT, 0);
#pragma unroll
                for (int i = 0; i < 2 * RT * TT; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    if (i >= RT * TT / 2) __builtin_amdgcn_sched_group_barrier(0x002, 14 / TT, 0);
                }
            }
        }
        __syncthreads();
    };
    const uint32_t whole = nb / kP;
    for (uint32_t s = 0; s < whole; s++) stage(s, std::true_type{});
    if (whole < nst) stage(whole, std::false_type{});

    // the four chains of each output (one aligned quarter of the FADDV
    // tree), then the four waves' quarters through LDS
    float4* ex = reinterpret_cast<float4*>(smem);
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = 0; t < TT; t++) {
            float4 v;
            float* pv = &v.x;
#pragma unroll
            for (int i = 0; i < 4; i++)
                pv[i] = (acc[r][t][i] + acc[r][t][4 + i]) + (acc[r][t][8 + i] + acc[r][t][12 + i]);
            ex[(((wt * RT + r) * TT + t) * 4 + j) * 64 + lane] = v;
        }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = 0; t < TT; t++) {
            if ((uint32_t)((r * TT + t) & 3) != j) continue;
            const float4* q = ex + ((wt * RT + r) * TT + t) * 4 * 64 + lane;
            const float4 a = q[0], b = q[64], c = q[128], d = q[192];
            const float o[4] = {(a.x + b.x) + (c.x + d.x), (a.y + b.y) + (c.y + d.y), (a.z + b.z) + (c.z + d.z),
                                (a.w + b.w) + (c.w + d.w)};
            const uint32_t row = row_base + r * 16 + c16, tok = tok_base + (wt * TT + t) * 16 + 4 * g;
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (row < N && tok + i < T) y[(uint64_t)(tok + i) * N + row] = o[i];
        }
}

template <class F, int RT, int TT, int WT, int P>
int launch(uint32_t N, uint32_t nb, uint32_t T, const float* x, const uint8_t* Wa, uint32_t off, uint32_t wrange,
           float* y, hipStream_t s) {
    using L = RLayout<F, RT, TT, WT, P>;
    const uint32_t tg = (T + L::kTok - 1) / L::kTok;
    const uint64_t grid = (uint64_t)((N + L::kRows - 1) / L::kRows) * tg;
    hipLaunchKernelGGL((k_rmode_mul_mat<F, RT, TT, WT, P>), dim3((uint32_t)grid), dim3(L::kThreads), 0, s, N, nb, T, x,
                       Wa, off, wrange, tg, y);
    ANE_HIP_CHECK_LAUNCH();
    return ANE_OK;
}

// Two or three tokens on rows the streaming GEMV takes (16-byte aligned): one
// launch here costs the same for 1 to 16 tokens, the GEMVs once per token, and
// from more than one workgroup (16 rows) per CU on they stream the weights two to
// four times as fast.  Where two or three of them are the faster ones, GEMVs /
// this kernel, us:
//  * Q4_0, two tokens, K > 1024 from two workgroups per CU (9216 x 4096 24.3 /
//    28.4, 28672 x 8192 91 / 114; 8192 x 4096 20.3 / 19.0, 14336 x 1024 12.1 /
//    12.0), K > 4096 from one (6144 x 14336 54.6 / 57.8);
//  * Q8_0, two tokens, K <= 4096 (4128 x 4096 18.1 / 24.6, 28672 x 4096 61.6 /
//    88.1), from two workgroups per CU for K <= 1024 (6144 x 1024 9.7 / 9.3, 14336 x
//    1024 14.4 / 18.5); longer rows, whose GEMV keeps fewer waves per CU, up to one
//    and a half workgroups for K <= 8192 (6144 x 8192 32.2 / 45.2) and from three
//    (14336 x 11008 78.7 / 122, 20000 x 11264 138 / 153), not between, where the
//    GEMV's last round of waves is nearly empty (8192 x 8192 54.6 / 45.5, 10000 x
//    11008 99.7 / 92.1);
//  * Q8_0, three tokens, K <= 4096 from eight workgroups per CU (65536 x 2048 87.7 /
//    118; 28672 x 4096 92.2 / 88.3).
bool gemvs_faster(bool q4, uint32_t N, uint32_t nb, uint32_t T, uint64_t cus) {
    const uint64_t wgs = ((uint64_t)N + 15) / 16;
    if (wgs <= cus) return false;
    if (q4) return T == 2 && nb > (wgs > 2 * cus ? 32u : 128u);
    if (T == 3) return nb <= 128 && wgs > 8 * cus;
    if (nb <= 128) return nb > 32 || wgs > 2 * cus;
    return wgs > 3 * cus || (nb <= 256 && 2 * wgs <= 3 * cus);
}

template <class F>
int run(uint32_t N, uint32_t nb, uint32_t T, const float* x, const void* W, float* y, hipStream_t s) {
    const uintptr_t wp = reinterpret_cast<uintptr_t>(W);
    const uint32_t off = (uint32_t)(wp & 15);
    // 32-bit buffer offsets: x, and the weights with the last window's over-read, below 2 GiB
    const uint64_t wbytes = off + (uint64_t)N * nb * F::kBytes;
    if (nb == 0 || (wp & 1) || (((uintptr_t)x) & 3) || wbytes + 2 * kMaxP * F::kBytes + 16 >= kOob ||
        ((uint64_t)T + 64) * nb * 128 + 2 * kMaxP * 128 >= kOob || !rmode_launch_fits(N, T))
        return -1;
    // Token t's y may take the place of an earlier token's x in the one launch
    // per token; here every token is read and written at once.
    const uintptr_t xp = (uintptr_t)x, yp = (uintptr_t)y;
    if (xp < yp + (uint64_t)T * N * 4 && yp < xp + (uint64_t)T * nb * 128) return -1;
    // whole dwords: the range check drops a dword that crosses the end
    const uint32_t wrange = (uint32_t)((wbytes + 3) & ~(uint64_t)3);
    const uint8_t* Wa = reinterpret_cast<const uint8_t*>(wp - off);
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return ANE_ERR_HIP;
    if (T <= 3 && off == 0 && nb % 8 == 0 && gemvs_faster(std::is_same<F, Q40Lane>::value, N, nb, T, (uint64_t)cus))
        return -1;
    auto wgs = [&](uint32_t rows, uint32_t tok) {
        return (uint64_t)((N + rows - 1) / rows) * ((T + tok - 1) / tok);
    };
    // The largest tile that still gives every CU a workgroup; the stages hold
    // more blocks where a stage's MFMAs are few (4 -> 16 blocks for the
    // one-tile workgroups: 16 tokens at 4096 x 4096 19.5 -> 14.9 us, its time
    // being the loads' latency per stage).
    if (T > 32 && wgs(64, 64) >= (uint64_t)cus) return launch<F, 4, 2, 2, 4>(N, nb, T, x, Wa, off, wrange, y, s);
    if (T > 32 && wgs(32, 64) >= (uint64_t)cus) return launch<F, 2, 2, 2, 8>(N, nb, T, x, Wa, off, wrange, y, s);
    if (T > 16 && wgs(32, 32) >= (uint64_t)cus) return launch<F, 2, 2, 1, 8>(N, nb, T, x, Wa, off, wrange, y, s);
    if (T > 16) return launch<F, 1, 2, 1, 8>(N, nb, T, x, Wa, off, wrange, y, s);
    return launch<F, 1, 1, 1, 16>(N, nb, T, x, Wa, off, wrange, y, s);
}

}  // namespace

int rmode_mul_mat(bool q4, uint32_t N, uint32_t K, uint32_t T, const float* x, const void* W, float* y,
                  hipStream_t s) {
    return q4 ? run<Q40Lane>(N, K >> 5, T, x, W, y, s) : run<Q80Lane>(N, K >> 5, T, x, W, y, s);
}

}  // namespace ane
