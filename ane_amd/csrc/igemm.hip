// igemm.hip -- the strided integer GEMMs cblas_igemm / cblas_ugemm /
// cblas_usgemm (opcodes 0x61-0x63) on the int8 MFMA contraction.
//
// Reference: the CBLAS_INTEGER_GEMM macro, src/bytecode_interpreter.s:8328-9135,
// instantiated at :9137-9139 with smopa, umopa and usmopa.  What it computes
// for the outputs it stores (rows < M, columns < N of C, stride ldc):
//   acc  = seed + sum_{k < 64*floor(K/64)} a(i,k) * b(k,j)   (wrapping int32)
//   seed = 0 when the bits of beta are zero, else the BIT PATTERN of
//          fl(beta * C[i][j]) (:8402-8488: the scaled C is moved into the
//          int32 za tiles before the products are accumulated)
//   C    = fl(fl32(acc) * alpha)                              (:8962-8980)
//   a(i,k) = A[i*lda + k]; with transA the handler adds the k offset to
//            A + ti and steps rows by lda (:8513-8514, :8562-8575), so row i
//            reads A[(i%16)*lda + (i - i%16) + k]
//   b(k,j) = B[k*ldb + j], or B[j*ldb + k] with transB (:8768-8872)
// ANE_IGEMM_BLAS instead computes what the handler's header describes:
// op(A) = A^T with transA, and C = fl(fl(fl32(acc)*alpha) + fl(beta*C)),
// C not read when beta == 0.
//
// Design.  The MFMA instruction multiplies signed bytes, so each operand is
// first gathered into K-contiguous signed rows (the layout the contraction
// kernels stream), both operands in one launch of 128-row x 128-k tiles, read
// along whichever direction is contiguous in memory with 16-byte loads.  An
// unsigned byte u is stored as u ^ 0x80 = u - 128, and the contraction's
// epilogue adds back
//   128 * sum_k b'(k,j)   (A unsigned)
//   128 * sum_k a'(i,k)   (B unsigned)
//   16384 * Ke            (both)
// which is exact modulo 2^32, like the handler's own wrapping sums.  Each tile
// writes its rows' partial sums, added up in the epilogue (no atomics, nothing
// to clear), or for long K adds them into one cleared sum per row.  Signed
// operands that are already K-contiguous rows (A without transA, B with transB)
// with 16-byte aligned rows that C does not overlap skip the pre-pass: the
// contraction reads them in place.  With beta = 0 the contraction writes C
// itself; otherwise it leaves int32 sums and k_igemm_epilogue reads C.
// Measured, 1536 x 2048 x 2048 uint8 x int8, both row-major: 27.4 -> 17.3 us
// (byte loads into 64 x 64 tiles with atomic row sums, a fill, two gathers and
// a separate epilogue pass over 12.6 MB of sums before).
#include "gemm_i8.hpp"

namespace ane {
namespace {

constexpr uint32_t kT = 128, kTK = 128;  // rows and k of a pre-pass tile
constexpr uint32_t kTStride = kTK + 16;   // LDS bytes between its rows

// One operand of the pre-pass: dst[r][k] = byte at src + r*rs + (r%16)*r16 +
// k*ks, flipped to signed when `flip`, for r < R, k < Ke (Ke % 64 == 0; ks == 1,
// or rs == 1 and r16 == 0); sums[kt * R + r] = the sum of row r's signed bytes in
// k-tile kt (null: not needed).
struct Gather {
    uint32_t R, tiles_r, tiles;
    const uint8_t* src;
    int64_t rs, r16, ks;
    uint32_t flip;
    int8_t* dst;
    int32_t* sums;
    bool atomic;  // sums[r] += instead of one partial per k-tile
};

__device__ __forceinline__ uint4 load16(const uint8_t* p) {  // any alignment
    uint4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}

__global__ void __launch_bounds__(256) k_igemm_gather(Gather ga, Gather gb, uint32_t Ke) {
    __shared__ __attribute__((aligned(16))) uint8_t tile[kT * kTStride];
    const bool second = blockIdx.x >= ga.tiles;
    const Gather g = second ? gb : ga;
    const uint32_t w = second ? blockIdx.x - ga.tiles : blockIdx.x;
    const uint32_t r0 = (w % g.tiles_r) * kT, kt = w / g.tiles_r, k0 = kt * kTK, t = threadIdx.x;
    const uint32_t flip = g.flip ? 0x80808080u : 0u;
    // 8 lanes per row, 16 bytes each; 32 rows per step
    const uint32_t rr = t >> 3, kk = (t & 7) * 16;
    const bool kin = k0 + kk < Ke;
    if (g.ks != 1) {
        // columns contiguous: 4 k x 16 rows per thread, transposed 4 x 4 bytes
        // at a time into the tile's rows
        const uint32_t rc = (t & 7) * 16, k = (t >> 3) * 4;
        uint32_t v[4][4];
        if (k0 + k < Ke) {
            const uint8_t* p = g.src + (int64_t)(r0 + rc) + (int64_t)(k0 + k) * g.ks;
            if (r0 + rc + 16 <= g.R) {
#pragma unroll
                for (int i = 0; i < 4; i++) *reinterpret_cast<uint4*>(v[i]) = load16(p + i * g.ks);
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (uint32_t e = 0; e < 16; e++) {
                        if (e % 4 == 0) v[i][e / 4] = 0;
                        if (r0 + rc + e < g.R) v[i][e / 4] |= (uint32_t)p[i * g.ks + e] << (8 * (e % 4));
                    }
            }
#pragma unroll
            for (uint32_t q = 0; q < 4; q++) {
                const uint32_t a = __builtin_amdgcn_perm(v[1][q], v[0][q], 0x05010400u);
                const uint32_t b = __builtin_amdgcn_perm(v[1][q], v[0][q], 0x07030602u);
                const uint32_t c = __builtin_amdgcn_perm(v[3][q], v[2][q], 0x05010400u);
                const uint32_t d = __builtin_amdgcn_perm(v[3][q], v[2][q], 0x07030602u);
                const uint32_t o[4] = {__builtin_amdgcn_perm(c, a, 0x05040100u), __builtin_amdgcn_perm(c, a, 0x07060302u),
                                       __builtin_amdgcn_perm(d, b, 0x05040100u), __builtin_amdgcn_perm(d, b, 0x07060302u)};
#pragma unroll
                for (uint32_t e = 0; e < 4; e++)
                    *reinterpret_cast<uint32_t*>(tile + (rc + 4 * q + e) * kTStride + k) = o[e];
            }
        }
        __syncthreads();
    }
    uint4 x[4];
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) {
        const uint32_t r = i * 32 + rr, gr = r0 + r;
        x[i] = make_uint4(0, 0, 0, 0);
        if (!kin || gr >= g.R) continue;
        x[i] = g.ks == 1 ? load16(g.src + (int64_t)gr * g.rs + (int64_t)(gr & 15) * g.r16 + k0 + kk)
                         : *reinterpret_cast<const uint4*>(tile + r * kTStride + kk);
    }
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) {
        const uint32_t gr = r0 + i * 32 + rr;
        const bool on = kin && gr < g.R;
        uint4 v = x[i];
        v.x ^= flip, v.y ^= flip, v.z ^= flip, v.w ^= flip;
        if (on) *reinterpret_cast<uint4*>(g.dst + (uint64_t)gr * Ke + k0 + kk) = v;
        if (g.sums) {  // over the eight lanes of the row
            int s = 0;
            if (on) {
                s = __builtin_amdgcn_sdot4((int)v.x, 0x01010101, s, false);
                s = __builtin_amdgcn_sdot4((int)v.y, 0x01010101, s, false);
                s = __builtin_amdgcn_sdot4((int)v.z, 0x01010101, s, false);
                s = __builtin_amdgcn_sdot4((int)v.w, 0x01010101, s, false);
            }
            s += (int)dpp_u32<kDppQuadXor1>((uint32_t)s);
            s += (int)dpp_u32<kDppQuadXor2>((uint32_t)s);
            s += (int)dpp_u32<kDppHalfMirror>((uint32_t)s);
            if ((t & 7) == 0 && gr < g.R) {
                if (g.atomic)
                    atomicAdd(g.sums + gr, s);
                else
                    g.sums[(uint64_t)kt * g.R + gr] = s;
            }
        }
    }
}

__global__ void __launch_bounds__(256) k_fill_i32(uint32_t n, int32_t* __restrict__ p) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0;
}

// C[i*ldc + j] for i < M, j < N from the signed-operand accumulators and
// the unsigned corrections; SEM 0 = the handler's arithmetic, 1 = BLAS.
template <int SEM>
__global__ void __launch_bounds__(256)
k_igemm_epilogue(uint32_t M, uint32_t N, const int32_t* __restrict__ acc, const int32_t* __restrict__ rowsum,
                 const int32_t* __restrict__ colsum, uint32_t nsum, uint32_t corr, float alpha, float beta,
                 float* __restrict__ C, uint64_t ldc) {
    const uint32_t j = blockIdx.x * 64 + (threadIdx.x & 63);
    const uint32_t i = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (i >= M || j >= N) return;
    uint32_t a = acc ? (uint32_t)acc[(uint64_t)i * N + j] : 0u;
    a += ig_sum(colsum, nsum, N, j) + ig_sum(rowsum, nsum, M, i) + corr;
    float* c = C + (uint64_t)i * ldc + j;
    if (SEM == 0) {
        if (__float_as_uint(beta) != 0u) a += __float_as_uint(__fmul_rn(beta, *c));
        *c = __fmul_rn((float)(int32_t)a, alpha);
    } else {
        float v = __fmul_rn((float)(int32_t)a, alpha);
        if (beta != 0.0f) v = __fadd_rn(v, __fmul_rn(beta, *c));
        *c = v;
    }
}

struct IgemmWs {
    int8_t *a, *bt;
    int32_t *acc, *rowsum, *colsum;
};

size_t igemm_layout(uint32_t M, uint32_t N, uint32_t K, uint8_t* base, IgemmWs* w) {
    const uint64_t Ke = (uint64_t)(K / 64) * 64;
    size_t off = 0;
    auto take = [&](uint64_t bytes) {
        const size_t o = off;
        off += ceil_to(bytes, 256);
        return base ? base + o : nullptr;
    };
    int8_t* a = reinterpret_cast<int8_t*>(take((uint64_t)M * Ke));
    int8_t* bt = reinterpret_cast<int8_t*>(take((uint64_t)N * Ke));
    int32_t* acc = reinterpret_cast<int32_t*>(take(Ke ? (uint64_t)M * N * 4 : 0));
    int32_t* rowsum = reinterpret_cast<int32_t*>(take((uint64_t)M * 4));
    int32_t* colsum = reinterpret_cast<int32_t*>(take((uint64_t)N * 4));
    if (w) *w = IgemmWs{a, bt, acc, rowsum, colsum};
    return off;
}

Gather gather_of(uint32_t R, uint32_t Ke, const void* src, int64_t rs, int64_t r16, int64_t ks, bool flip, int8_t* dst) {
    const uint32_t tr = (R + kT - 1) / kT;
    return Gather{R, tr, tr * ((Ke + kTK - 1) / kTK), static_cast<const uint8_t*>(src), rs, r16, ks, flip ? 1u : 0u,
                  dst, nullptr, false};
}

}  // namespace
}  // namespace ane

using namespace ane;

extern "C" size_t ane_hip_cblas_igemm_workspace_size(uint32_t M, uint32_t N, uint32_t K) {
    return igemm_layout(M, N, K, nullptr, nullptr) + 256;
}

extern "C" int ane_hip_cblas_igemm(int variant, int semantics, uint8_t flags, uint32_t M, uint32_t N, uint32_t K,
                                   uint32_t lda, uint32_t ldb, uint32_t ldc, float alpha, float beta, const void* A,
                                   const void* B, float* C, void* workspace, size_t workspace_bytes, void* stream) {
    if (variant < 0 || variant > 2 || semantics < 0 || semantics > 1) return ANE_ERR_INVALID_ARG;
    if (M == 0 || N == 0) return ANE_OK;
    const uint32_t Ke = K / 64 * 64;
    if (!C || (Ke && (!A || !B))) return ANE_ERR_BAD_POINTER;
    if (ldc < N) return ANE_ERR_INVALID_ARG;
    if (!workspace || (((uintptr_t)workspace) & 255) ||
        workspace_bytes < igemm_layout(M, N, K, nullptr, nullptr))
        return ANE_ERR_WORKSPACE;
    if ((uint64_t)M * N > 0xffffffffull || (N + 63) / 64 > 0x7fffffffu || (M + 3) / 4 > 65535u)
        return ANE_ERR_INVALID_ARG;
    const bool au = variant != 0, bu = variant == 1;
    const bool ta = flags & 1, tb = (flags >> 1) & 1;
    hipStream_t s = (hipStream_t)stream;
    IgemmWs w;
    igemm_layout(M, N, K, static_cast<uint8_t*>(workspace), &w);
    const bool reads_c = semantics == 0 ? __builtin_bit_cast(uint32_t, beta) != 0u : beta != 0.0f;
    const uint32_t corr = (au && bu) ? 16384u * Ke : 0u;
    const int32_t *rows = nullptr, *cols = nullptr;
    uint32_t nsum = 1;
    if (Ke) {
        if ((uint64_t)M * Ke >= (1ull << 31) || (uint64_t)N * Ke >= (1ull << 31) || (M + 63) / 64 > 65535u ||
            (N + 63) / 64 > 65535u)
            return ANE_ERR_INVALID_ARG;
        // Signed operands already in the contraction's layout (A's rows, or
        // B's rows under transB, K contiguous with 16-byte aligned rows) are
        // read in place: no gather pass, no row sums needed (both signed).
        // Not where the contraction would write C over bytes that its other
        // workgroups still read: an operand that overlaps C is gathered.
        const uint64_t c_end = ((uint64_t)(M - 1) * ldc + N) * 4;
        auto under_c = [&](const void* p, uint32_t rows, uint32_t ld) {
            const uintptr_t x = (uintptr_t)p, c = (uintptr_t)C;
            return !reads_c && x < c + c_end && c < x + (uint64_t)(rows - 1) * ld + Ke;
        };
        const bool a_direct = !au && !bu && !ta && (lda & 15) == 0 && lda >= Ke && (((uintptr_t)A) & 15) == 0 &&
                              !under_c(A, M, lda);
        const bool b_direct = !au && !bu && tb && (ldb & 15) == 0 && ldb >= Ke && (((uintptr_t)B) & 15) == 0 &&
                              !under_c(B, N, ldb);
        // A rows: plain, the handler's transA addressing, or A^T (BLAS); Bt
        // rows: B^T of a K x N matrix, or B itself (transB)
        Gather ga = gather_of(M, Ke, A, !ta ? (int64_t)lda : 1, (ta && semantics == 0) ? (int64_t)lda - 1 : 0,
                              (ta && semantics == 1) ? (int64_t)lda : 1, au, w.a);
        Gather gb = gather_of(N, Ke, B, tb ? (int64_t)ldb : 1, 0, tb ? 1 : (int64_t)ldb, bu, w.bt);
        if (a_direct) ga.tiles = 0;
        if (b_direct) gb.tiles = 0;
        if (au || bu) {
            // Partial sums per k-tile in the int32 sums' place when the
            // contraction writes C itself and they fit there (and in the row
            // and column sums after it); else one cleared sum per row.  Not
            // more than kIgParts of them (K <= 2048), which the readers add up:
            // uint8 x uint8, partials without that bound and sums, 128 x 4096 x
            // 8192 63.6 / 52 us, 300 x 300 x 8192 41.0 / 35.1, 1024 x 1024 x 16384
            // 76.2 / 53.4; 128 x 4096 x 1024 13.9 / 15.8, 1536 x 2048 x 2048 21.1 /
            // 22.6.  And not for the narrow products that k_gemm_i8 takes, which
            // adds them up for every element (40000 x 16 x 2048 156 / 74).
            const uint32_t kt = (Ke + kTK - 1) / kTK;
            const uint64_t have = (uint64_t)M * N + M + N, need = (uint64_t)kt * ((au ? N : 0) + (bu ? M : 0));
            const bool parts = !reads_c && need <= have && kt <= kIgParts && (M <= 128 || N >= 128);
            int32_t* const csum = parts ? w.acc : w.colsum;
            int32_t* const rsum = parts ? w.acc + (au ? (uint64_t)kt * N : 0) : w.rowsum;
            if (!parts) {
                const uint32_t n = (uint32_t)(w.colsum + N - w.rowsum);  // rowsum, then colsum
                hipLaunchKernelGGL(k_fill_i32, dim3((n + 255) / 256), dim3(256), 0, s, n, w.rowsum);
            } else {
                nsum = kt;
            }
            if (au) gb.sums = csum, cols = csum;
            if (bu) ga.sums = rsum, rows = rsum;
            ga.atomic = gb.atomic = !parts;
        }
        if (ga.tiles + gb.tiles) {
            hipLaunchKernelGGL(k_igemm_gather, dim3(ga.tiles + gb.tiles), dim3(256), 0, s, ga, gb, Ke);
            ANE_HIP_CHECK_LAUNCH();
        }
        GemmParams p{};
        p.A = a_direct ? static_cast<const int8_t*>(A) : w.a;
        p.lda = a_direct ? lda : Ke;
        p.B = b_direct ? static_cast<const int8_t*>(B) : w.bt;
        p.ldb = b_direct ? ldb : Ke;
        p.rowsA = p.Mout = M;
        p.colsB = p.Nout = N;
        p.Kp = Ke;
        p.s = alpha;
        if (reads_c) {
            p.Craw = w.acc;
            p.ldc = N;
        } else {
            p.C = C;
            p.ldc = ldc;
            p.ig = true;
            p.igc = cols;
            p.igr = rows;
            p.nsum = nsum;
            p.corr = corr;
        }
        const int st = launch_gemm_rows(p, s);
        if (st != ANE_OK || !reads_c) return st;
    }
    const dim3 grid((N + 63) / 64, (M + 3) / 4);
    const auto fn = semantics == 0 ? k_igemm_epilogue<0> : k_igemm_epilogue<1>;
    hipLaunchKernelGGL(fn, grid, dim3(256), 0, s, M, N, Ke ? w.acc : nullptr, rows, cols, nsum, corr, alpha, beta, C,
                       (uint64_t)ldc);
    ANE_HIP_CHECK_LAUNCH();
    return ANE_OK;
}
