// quantize.hip -- fp32 <-> int8 element-wise kernels of the ane opcode set:
// quantize_fp32_i8 (0x19), dequantize_i8_fp32 (0x1A),
// quantize_fp32_i8_channelwise (0x1C) and pack_b_i8 (0x1B).
//
// All of them are HBM-bound streaming passes: 16-byte global loads per lane,
// a grid sized to a few waves per CU, no LDS except block reductions.
#include "common.hpp"

namespace ane {

constexpr int kQThreads = 256;
constexpr uint32_t kMaxPartials = 2048;

static uint32_t stream_blocks(uint64_t n_vec4) {
    uint64_t b = (n_vec4 + kQThreads * 4 - 1) / (kQThreads * 4);
    if (b < 1) b = 1;
    if (b > kMaxPartials) b = kMaxPartials;
    return (uint32_t)b;
}

// Pass 1 of 0x19 (bytecode_interpreter.s:1893-1905): per-block max |x| keys.
__global__ void __launch_bounds__(kQThreads)
k_absmax_partial(const float* __restrict__ src, uint64_t n,
                 uint32_t* __restrict__ partials) {
    __shared__ uint32_t red[4];
    uint32_t m = 0;
    const uint64_t tid = (uint64_t)blockIdx.x * kQThreads + threadIdx.x;
    const uint64_t stride = (uint64_t)gridDim.x * kQThreads;
    uint64_t head = 0;
    if ((((uintptr_t)src) & 15) == 0) {
        const uint64_t n4 = n >> 2;
        const float4* s4 = reinterpret_cast<const float4*>(src);
        for (uint64_t i = tid; i < n4; i += stride) {
            float4 v = s4[i];
            uint32_t a = abs_key(v.x), b = abs_key(v.y), c = abs_key(v.z), d = abs_key(v.w);
            a = a > b ? a : b;
            c = c > d ? c : d;
            a = a > c ? a : c;
            m = m > a ? m : a;
        }
        head = n4 << 2;
    }
    for (uint64_t i = head + tid; i < n; i += stride) {
        uint32_t a = abs_key(src[i]);
        m = m > a ? m : a;
    }
    m = block_max_u32_256(m, red);
    if (threadIdx.x == 0) partials[blockIdx.x] = m;
}

// Pass 2 of 0x19 (bytecode_interpreter.s:1906-1950): every block folds the
// partial maxima, derives (scale, inv) and quantizes its grid-stride share.
__global__ void __launch_bounds__(kQThreads)
k_quantize(const float* __restrict__ src, uint64_t n, int8_t* __restrict__ dst,
           const uint32_t* __restrict__ partials, uint32_t np,
           float* __restrict__ scale_out) {
    __shared__ uint32_t red[4];
    uint32_t m = 0;
    for (uint32_t i = threadIdx.x; i < np; i += kQThreads) {
        uint32_t a = partials[i];
        m = m > a ? m : a;
    }
    m = block_max_u32_256(m, red);
    float scale, inv;
    quant_params(__uint_as_float(m), scale, inv);
    if (blockIdx.x == 0 && threadIdx.x == 0 && scale_out) *scale_out = scale;

    const uint64_t tid = (uint64_t)blockIdx.x * kQThreads + threadIdx.x;
    const uint64_t stride = (uint64_t)gridDim.x * kQThreads;
    uint64_t head = 0;
    if ((((uintptr_t)src) & 15) == 0 && (((uintptr_t)dst) & 3) == 0) {
        const uint64_t n4 = n >> 2;
        const float4* s4 = reinterpret_cast<const float4*>(src);
        uint32_t* d4 = reinterpret_cast<uint32_t*>(dst);
        // every value is one whose max |x| was just folded, so pack4_fast
        // (bit-identical, two VALU per value) applies whenever that max and
        // inv are finite
        if (fast_quant_ok(__uint_as_float(m), inv)) {
            for (uint64_t i = tid; i < n4; i += stride) {
                const float4 v = s4[i];
                d4[i] = pack4_fast(v.x, v.y, v.z, v.w, inv);
            }
        } else {
            for (uint64_t i = tid; i < n4; i += stride) {
                const float4 v = s4[i];
                d4[i] = pack4(v.x, v.y, v.z, v.w, inv);
            }
        }
        head = n4 << 2;
    }
    for (uint64_t i = head + tid; i < n; i += stride) dst[i] = (int8_t)quant1(src[i], inv);
}

// 0x1A (bytecode_interpreter.s:1951-1977): scvtf then fmul.
__global__ void __launch_bounds__(kQThreads)
k_dequantize(const int8_t* __restrict__ src, uint64_t n, float scale,
             float* __restrict__ dst) {
    const uint64_t tid = (uint64_t)blockIdx.x * kQThreads + threadIdx.x;
    const uint64_t stride = (uint64_t)gridDim.x * kQThreads;
    uint64_t head = 0;
    if ((((uintptr_t)src) & 3) == 0 && (((uintptr_t)dst) & 15) == 0) {
        const uint64_t n4 = n >> 2;
        const uint32_t* s4 = reinterpret_cast<const uint32_t*>(src);
        float4* d4 = reinterpret_cast<float4*>(dst);
        for (uint64_t i = tid; i < n4; i += stride) {
            uint32_t q = s4[i];
            float4 o;
            o.x = __fmul_rn((float)(int8_t)(q & 0xff), scale);
            o.y = __fmul_rn((float)(int8_t)((q >> 8) & 0xff), scale);
            o.z = __fmul_rn((float)(int8_t)((q >> 16) & 0xff), scale);
            o.w = __fmul_rn((float)(int8_t)(q >> 24), scale);
            d4[i] = o;
        }
        head = n4 << 2;
    }
    for (uint64_t i = head + tid; i < n; i += stride)
        dst[i] = __fmul_rn((float)src[i], scale);
}

// 0x1C (bytecode_interpreter.s:2591-2662): TPR threads per row (64: four
// rows per workgroup; 256: one), cpad a multiple of 16.  Rows of up to
// kCwItems float4 per thread are read once and held in registers between the
// maximum and the quantization; longer rows are read a second time.
// VEC: src 16-byte and dst 4-byte aligned.  HBM-bound: 5 bytes per element;
// 1024 rows of 4096 13.2 -> 4.9 us (scalar loads in two passes before).
constexpr uint32_t kCwItems = 8;

template <int TPR, bool VEC>
__global__ void __launch_bounds__(kQThreads)
k_quantize_channelwise(const float* __restrict__ src, uint32_t rows, uint32_t cpad,
                       int8_t* __restrict__ dst, float* __restrict__ scales) {
    __shared__ uint32_t red[4];
    const uint32_t t = threadIdx.x % TPR;
    const uint64_t row = (uint64_t)blockIdx.x * (kQThreads / TPR) + threadIdx.x / TPR;
    if (TPR == 64 && row >= rows) return;  // whole waves, no barrier on this path
    const float* s = src + row * cpad;
    int8_t* d = dst + row * cpad;
    const uint32_t n4 = cpad / 4;
    auto fold = [](uint32_t m, float4 v) {
        const uint32_t a = max(abs_key(v.x), abs_key(v.y)), b = max(abs_key(v.z), abs_key(v.w));
        return max(m, max(a, b));
    };
    auto row_max = [&](uint32_t m) { return TPR == 64 ? wave_max_u32(m) : block_max_u32_256(m, red); };
    float scale, inv;
    if (VEC && n4 <= kCwItems * TPR) {
        const float4* s4 = reinterpret_cast<const float4*>(s);
        float4 v[kCwItems];
        uint32_t m = 0;
#pragma unroll
        for (uint32_t u = 0; u < kCwItems; u++)
            if (u * TPR < n4) v[u] = u * TPR + t < n4 ? s4[u * TPR + t] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
        for (uint32_t u = 0; u < kCwItems; u++)
            if (u * TPR < n4) m = fold(m, v[u]);
        m = row_max(m);
        quant_params(__uint_as_float(m), scale, inv);
        if (t == 0) scales[row] = scale;
        uint32_t* d4 = reinterpret_cast<uint32_t*>(d);
        const bool fast = fast_quant_ok(__uint_as_float(m), inv);
#pragma unroll
        for (uint32_t u = 0; u < kCwItems; u++)
            if (u * TPR + t < n4)
                d4[u * TPR + t] = fast ? pack4_fast(v[u].x, v[u].y, v[u].z, v[u].w, inv)
                                       : pack4(v[u].x, v[u].y, v[u].z, v[u].w, inv);
        return;
    }
    uint32_t m = 0;
    if (VEC) {
        for (uint32_t i = t; i < n4; i += TPR) m = fold(m, reinterpret_cast<const float4*>(s)[i]);
    } else {
        for (uint32_t i = t; i < cpad; i += TPR) m = max(m, abs_key(s[i]));
    }
    m = row_max(m);
    quant_params(__uint_as_float(m), scale, inv);
    if (t == 0) scales[row] = scale;
    if (VEC) {
        for (uint32_t i = t; i < n4; i += TPR) {
            const float4 v = reinterpret_cast<const float4*>(s)[i];
            reinterpret_cast<uint32_t*>(d)[i] = pack4(v.x, v.y, v.z, v.w, inv);
        }
    } else {
        for (uint32_t i = t; i < cpad; i += TPR) d[i] = (int8_t)quant1(s[i], inv);
    }
}

// 0x1B (bytecode_interpreter.s:2459-2582): the SMOPA panel format,
// dst[(p*G+g)*64 + 4c + d] = B[4g+d][16p+c].  A workgroup takes 16 groups (64
// rows) x 16 panels (256 columns), one 64-byte group per thread: 16 bytes of
// each of its four rows (16 lanes read 256 consecutive bytes), a 4 x 4 byte
// transpose per four columns, and the groups go through LDS so that each
// panel's 1 KB is stored contiguously.  HBM-bound, 2 bytes per element:
// 4096 x 6144 131 -> 8.4 us (6.0 TB/s) (64 single-byte loads per thread before).
constexpr uint32_t kPackT = 16;                     // groups and panels per workgroup
constexpr uint32_t kPackStride = kPackT * 64 + 16;  // LDS bytes between panels

__global__ void __launch_bounds__(kQThreads)
k_pack_b(uint32_t K, uint32_t N, uint32_t G, uint32_t P, uint32_t gbase, uint32_t pbase,
         const int8_t* __restrict__ src, int8_t* __restrict__ dst) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[kPackT * kPackStride];
    const uint32_t g0 = gbase + blockIdx.x * kPackT, p0 = pbase + blockIdx.y * kPackT;
    {
        const uint32_t p = threadIdx.x % kPackT, g = threadIdx.x / kPackT;
        const uint64_t col = 16ull * (p0 + p), k = 4ull * (g0 + g);
        uint32_t r[4][4];
        const int8_t* q = src + k * N + col;
        if (col + 16 <= N && k + 4 <= K) {
#pragma unroll
            for (uint32_t d = 0; d < 4; d++)
                __builtin_memcpy(r[d], q + (uint64_t)d * N, 16);  // any alignment: rows start anywhere when N % 16 != 0
        } else {
#pragma unroll
            for (uint32_t d = 0; d < 4; d++)
#pragma unroll
                for (uint32_t c = 0; c < 16; c++) {
                    if (c % 4 == 0) r[d][c / 4] = 0;
                    if (k + d < K && col + c < N)
                        r[d][c / 4] |= (uint32_t)(uint8_t)q[(uint64_t)d * N + c] << (8 * (c % 4));
                }
        }
        uint4* o = reinterpret_cast<uint4*>(lds + p * kPackStride + g * 64);
#pragma unroll
        for (uint32_t w = 0; w < 4; w++) {
            // columns 4w .. 4w+3: bytes c of the four rows' words
            const uint32_t a = __builtin_amdgcn_perm(r[1][w], r[0][w], 0x05010400u);  // r0.0 r1.0 r0.1 r1.1
            const uint32_t b = __builtin_amdgcn_perm(r[1][w], r[0][w], 0x07030602u);  // r0.2 r1.2 r0.3 r1.3
            const uint32_t c = __builtin_amdgcn_perm(r[3][w], r[2][w], 0x05010400u);
            const uint32_t e = __builtin_amdgcn_perm(r[3][w], r[2][w], 0x07030602u);
            o[w] = make_uint4(__builtin_amdgcn_perm(c, a, 0x05040100u), __builtin_amdgcn_perm(c, a, 0x07060302u),
                              __builtin_amdgcn_perm(e, b, 0x05040100u), __builtin_amdgcn_perm(e, b, 0x07060302u));
        }
    }
    __syncthreads();
    const bool vec = (((uintptr_t)dst) & 15) == 0;
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) {
        const uint32_t p = 4 * i + threadIdx.x / 64, c = threadIdx.x % 64;  // 16-byte chunk c of the panel's 16 groups
        if (p0 + p >= P || g0 + c / 4 >= G) continue;
        const uint8_t* s = lds + p * kPackStride + c * 16;
        int8_t* o = dst + ((uint64_t)(p0 + p) * G + g0) * 64 + c * 16;
        if (vec) {
            *reinterpret_cast<uint4*>(o) = *reinterpret_cast<const uint4*>(s);
        } else {
            for (uint32_t b = 0; b < 16; b++) o[b] = (int8_t)s[b];
        }
    }
}

}  // namespace ane

using namespace ane;

extern "C" size_t ane_hip_quantize_workspace_size(uint64_t n) {
    (void)n;
    return kMaxPartials * sizeof(uint32_t);
}

extern "C" int ane_hip_quantize_fp32_i8(uint64_t count, int pad16, const float* src,
                                        int8_t* dst, float* scale_out, void* workspace,
                                        size_t workspace_bytes, void* stream) {
    uint64_t n = count;
    if (pad16) {
        n = ceil_to(count, 16);
        if (n == 0) n = 16;
    }
    if (!src || !dst) return ANE_ERR_BAD_POINTER;
    if (!workspace || workspace_bytes < ane_hip_quantize_workspace_size(n)) return ANE_ERR_WORKSPACE;
    hipStream_t s = (hipStream_t)stream;
    uint32_t* partials = (uint32_t*)workspace;
    const uint32_t nb = stream_blocks(n / 4 + 1);
    hipLaunchKernelGGL(k_absmax_partial, dim3(nb), dim3(kQThreads), 0, s, src, n, partials);
    hipLaunchKernelGGL(k_quantize, dim3(nb), dim3(kQThreads), 0, s, src, n, dst, partials, nb,
                       scale_out);
    ANE_HIP_CHECK_LAUNCH();
    return ANE_OK;
}

extern "C" int ane_hip_dequantize_i8_fp32(uint64_t count, float scale, const int8_t* src,
                                          float* dst, void* stream) {
    const uint64_t n = ceil_to(count, 16);
    if (n == 0) return ANE_OK;
    if (!src || !dst) return ANE_ERR_BAD_POINTER;
    const uint32_t nb = stream_blocks(n / 4 + 1);
    hipLaunchKernelGGL(k_dequantize, dim3(nb), dim3(kQThreads), 0, (hipStream_t)stream, src, n,
                       scale, dst);
    ANE_HIP_CHECK_LAUNCH();
    return ANE_OK;
}

extern "C" int ane_hip_quantize_channelwise(uint32_t rows, uint32_t cols, const float* src,
                                            int8_t* dst, float* scales, void* stream) {
    if (rows == 0) return ANE_OK;
    if (!src || !dst || !scales) return ANE_ERR_BAD_POINTER;
    uint64_t cpad = ceil_to(cols, 16);
    if (cpad == 0) cpad = 16;
    if (cpad > 0xffffffffull) return ANE_ERR_INVALID_ARG;
    const bool vec = (((uintptr_t)src) & 15) == 0 && (((uintptr_t)dst) & 3) == 0;
    // one wave per row up to the length a wave holds in registers, unless
    // that leaves CUs without a workgroup; 256 threads per row otherwise
    const bool wave_rows = cpad <= kCwItems * 4 * 64 && rows >= 1024;
    const dim3 grid(wave_rows ? (uint32_t)(((uint64_t)rows + 3) / 4) : rows);
    hipStream_t s = (hipStream_t)stream;
    const auto fn = wave_rows ? (vec ? k_quantize_channelwise<64, true> : k_quantize_channelwise<64, false>)
                              : (vec ? k_quantize_channelwise<256, true> : k_quantize_channelwise<256, false>);
    hipLaunchKernelGGL(fn, grid, dim3(kQThreads), 0, s, src, rows, (uint32_t)cpad, dst, scales);
    ANE_HIP_CHECK_LAUNCH();
    return ANE_OK;
}

extern "C" size_t ane_hip_packed_b_size(uint32_t K, uint32_t N) {
    const uint64_t G = ceil_to(K, 4) / 4, P = ceil_to(N, 16) / 16;
    return (size_t)(P * G * 64);
}

extern "C" int ane_hip_pack_b_i8(uint32_t K, uint32_t N, const int8_t* src, int8_t* dst,
                                 void* stream) {
    const uint64_t G = ceil_to(K, 4) / 4, P = ceil_to(N, 16) / 16;
    if (G == 0 || P == 0) return ANE_OK;
    if (!src || !dst) return ANE_ERR_BAD_POINTER;
    const uint64_t gx = (G + kPackT - 1) / kPackT, gy = (P + kPackT - 1) / kPackT;
    if ((G * P + kQThreads - 1) / kQThreads > 0x7fffffffull) return ANE_ERR_INVALID_ARG;
    // a launch holds 65535 workgroups of 16 panels in y and fewer than 2^24 (of 256
    // threads) of 16 groups in x
    constexpr uint64_t kMaxX = (1u << 24) - 1, kMaxY = 65535;
    for (uint64_t y = 0; y < gy; y += kMaxY) {
        for (uint64_t x = 0; x < gx; x += kMaxX) {
            const uint64_t nx = gx - x < kMaxX ? gx - x : kMaxX, ny = gy - y < kMaxY ? gy - y : kMaxY;
            hipLaunchKernelGGL(k_pack_b, dim3((uint32_t)nx, (uint32_t)ny), dim3(kQThreads), 0, (hipStream_t)stream, K,
                               N, (uint32_t)G, (uint32_t)P, (uint32_t)(x * kPackT), (uint32_t)(y * kPackT), src, dst);
        }
    }
    ANE_HIP_CHECK_LAUNCH();
    return ANE_OK;
}
