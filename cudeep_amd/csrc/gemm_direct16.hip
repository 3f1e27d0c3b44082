// fp16 / bf16 GEMM (fp32 sums and results) without LDS staging, for products too
// small to fill the GPU with the tiled kernels' workgroups: the 16-bit
// companion of gemm_direct.hip.  A wave's step is 32 k, one
// v_mfma_f32_16x16x32_{f16,bf16} per pair of 16-row blocks: lane group lq holds
// k = k0 + 8 lq .. + 7 of its row, one 16-byte load where k is contiguous in
// memory (any 4-byte alignment), eight 2-byte loads of 16 neighbours where the
// other dimension is.  The four waves of a workgroup share one tile of 32 x 32
// or 16 x 16, each with a run of k, summed in wave order through LDS.
#include "cdx_internal.hpp"

namespace cdx {
namespace {

typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4u __attribute__((ext_vector_type(4), aligned(4)));

struct H16Args {
    const unsigned short* A; const unsigned short* B; float* C; const float* bias;
    int64_t M, N, K, lda, ldb, ldc;
    int bias_mode, epilogue;
};

// One operand's 16 F rows (m or n) x 32 k of a wave.  KC: k contiguous.
template <int F, bool KC>
struct Loader16 {
    u32x4 v[F];          // eight 16-bit values: k = k0 + 8 lq + 0 .. 7
    __device__ __forceinline__ void load(const char* base, const uint32_t (&off)[F], int64_t ld_b) {
#pragma unroll
        for (int i = 0; i < F; ++i) {
            if constexpr (KC) {
                v[i] = *(const __attribute__((address_space(1))) u32x4u*)(base + off[i]);
            } else {
                unsigned short e[8];
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    e[q] = *(const __attribute__((address_space(1))) unsigned short*)(base + q * ld_b + off[i]);
#pragma unroll
                for (int q = 0; q < 4; ++q) v[i][q] = e[2 * q] | ((uint32_t)e[2 * q + 1] << 16);
            }
        }
    }
    // the last step: k >= krem reads as 0
    __device__ __forceinline__ void load_tail(const char* base, const uint32_t (&off)[F],
                                              int64_t ld_b, int k, int krem) {
#pragma unroll
        for (int i = 0; i < F; ++i) {
            uint32_t e[8];
#pragma unroll
            for (int q = 0; q < 8; ++q)
                e[q] = k + q < krem ? *(const unsigned short*)(base + (KC ? q * 2 : q * ld_b) + off[i]) : 0u;
#pragma unroll
            for (int q = 0; q < 4; ++q) v[i][q] = e[2 * q] | (e[2 * q + 1] << 16);
        }
    }
};

template <int FM, int FN, int OPA, int OPB, bool BF>
__global__ __launch_bounds__(256)
void gemm_direct16_kernel(H16Args p) {
    constexpr bool KCA = OPA == CDX_OP_N, KCB = OPB == CDX_OP_T;
    constexpr int BM = 16 * FM, BN = 16 * FN, DEPTH = 4, WK = 4;
    const int lane = threadIdx.x & 63;
    const int wk = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, lq = lane >> 4;
    const int tiles_n = (int)ceil_div(p.N, BN);
    const int64_t m0 = (int64_t)(blockIdx.x / tiles_n) * BM, n0 = (int64_t)(blockIdx.x % tiles_n) * BN;
    const int64_t lda_b = p.lda * 2, ldb_b = p.ldb * 2;
    uint32_t offa[FM], offb[FN];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int64_t r = m0 + i * 16 + l16 < p.M ? i * 16 + l16 : p.M - 1 - m0;
        offa[i] = (uint32_t)(KCA ? r * lda_b + 16 * lq : 8 * lq * lda_b + r * 2);
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int64_t r = n0 + j * 16 + l16 < p.N ? j * 16 + l16 : p.N - 1 - n0;
        offb[j] = (uint32_t)(KCB ? r * ldb_b + 16 * lq : 8 * lq * ldb_b + r * 2);
    }
    const char* pa = reinterpret_cast<const char*>(p.A + (KCA ? m0 * p.lda : m0));
    const char* pb = reinterpret_cast<const char*>(p.B + (KCB ? n0 * p.ldb : n0));
    const int64_t sa = KCA ? 64 : 32 * lda_b, sb = KCB ? 64 : 32 * ldb_b;   // bytes per 32 k

    floatx4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    Loader16<FM, KCA> a[DEPTH];
    Loader16<FN, KCB> b[DEPTH];
    auto mul = [&](const Loader16<FM, KCA>& x, const Loader16<FN, KCB>& y) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                if constexpr (BF)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8, x.v[i]), __builtin_bit_cast(bf16x8, y.v[j]), acc[i][j], 0, 0, 0);
                else
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        __builtin_bit_cast(halfx8, x.v[i]), __builtin_bit_cast(halfx8, y.v[j]), acc[i][j], 0, 0, 0);
            }
    };

    // this wave's whole steps [s0, s1); the partial one goes to the last wave
    const int full = (int)(p.K / 32), krem = (int)(p.K % 32);
    const int per = (full + WK - 1) / WK;
    const int s0 = wk * per < full ? wk * per : full, s1 = s0 + per < full ? s0 + per : full;
    if (s0 < s1) {
        // loads past s1 - 1 repeat that step (unused), so that every iteration
        // issues the same loads and a wait counts exactly those it needs
        auto load = [&](int d, int s) {
            const int64_t t = s < s1 ? s : s1 - 1;
            a[d].load(pa + t * sa, offa, lda_b);
            b[d].load(pb + t * sb, offb, ldb_b);
        };
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) load(d, s0 + d);
        int s = s0;
        for (; s + DEPTH <= s1; s += DEPTH) {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
                mul(a[d], b[d]);
                load(d, s + d + DEPTH);
            }
        }
#pragma unroll
        for (int d = 0; d < DEPTH - 1; ++d)
            if (s + d < s1) mul(a[d], b[d]);
    }
    if (krem > 0 && wk == WK - 1) {
        a[0].load_tail(pa + full * sa, offa, lda_b, 8 * lq, krem);
        b[0].load_tail(pb + full * sb, offb, ldb_b, 8 * lq, krem);
        mul(a[0], b[0]);
    }

    const EpiArgs epi{p.C, p.ldc, p.M, p.N, 0, 0, p.bias, p.bias_mode, p.epilogue};
    __shared__ floatx4 red[WK][FM * FN][64];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) red[wk][i * FN + j][lane] = acc[i][j];
    __syncthreads();
    if (wk >= FM * FN) return;
    floatx4 sum[1][1] = {{red[0][wk][lane]}};
#pragma unroll
    for (int w = 1; w < WK; ++w) sum[0][0] += red[w][wk][lane];
    write_acc<1, 1, true, false>(sum, epi, m0 + wk / FN * 16, n0 + wk % FN * 16, lane);
}

template <int F, bool BF>
void launch_ops(const GemmArgs& g, const H16Args& p, hipStream_t stream) {
    const dim3 grid((unsigned)(ceil_div(g.M, 16 * F) * ceil_div(g.N, 16 * F))), block(256);
    if (g.opA == CDX_OP_N && g.opB == CDX_OP_N)
        hipLaunchKernelGGL((gemm_direct16_kernel<F, F, CDX_OP_N, CDX_OP_N, BF>), grid, block, 0, stream, p);
    else if (g.opA == CDX_OP_N)
        hipLaunchKernelGGL((gemm_direct16_kernel<F, F, CDX_OP_N, CDX_OP_T, BF>), grid, block, 0, stream, p);
    else if (g.opB == CDX_OP_N)
        hipLaunchKernelGGL((gemm_direct16_kernel<F, F, CDX_OP_T, CDX_OP_N, BF>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((gemm_direct16_kernel<F, F, CDX_OP_T, CDX_OP_T, BF>), grid, block, 0, stream, p);
}

int64_t tiles_of(const GemmArgs& g, int64_t side) { return ceil_div(g.M, side) * ceil_div(g.N, side); }

}  // namespace

// Up to 256 tiles of 32 x 32 (A transposed, B not: 320), or 768 where the tiled
// kernels would load element by element; tiles of 16 x 16 up to 400 of them.
// Tiled / 16 x 16 / 32 x 32, us:
//   256^3 NT              4.9 /  3.2 /  4.1    100 x 100 x 3000 TN  42.4 /  9.2 / 13.3
//   300^3 NT             11.1 /  3.8 /  4.7    128 x 64 x 1943 TN   41.5 /  7.2 / 10.4
//   1151 x 102 x 2320 NN 70.8 / 15.6 / 11.5    224 x 704 x 2256 NN  34.6 / 14.8 / 14.5
//   512^3 NT              6.5 /  8.7 /  5.6    1000 x 500 x 300 TT  10.6 /  7.3 /  6.0
//   512 x 640 x 1024 NT   9.6 /        11.9    512 x 640 x 1024 TN  17.1 /        10.0
//   640 x 640 x 1280 TN  21.0 / 23.7 / 10.3    768^3 NT              8.2 / 16.6 / 12.1
// A wave sums a quarter of K in one accumulator, the tiled kernels' k-slices
// 1024 k and more each: where those slice, K ends at 4096, beyond which this
// kernel is the less exact one and soon the slower one too.  Tiled / this, us
// and relative error against fp64 (bf16, N(0, 1)):
//   256 x 256 x 4096 NN   19.9 / 12.0   1.9e-7 / 1.9e-7
//   256 x 256 x 8192 NN   20.6 / 37.2   1.9e-7 / 2.7e-7
//   256 x 784 x 8192 NN   32.4 / 44.0   1.9e-7 / 2.7e-7
//   64 x 64 x 65536 NT    20.0 / 112.7  2.4e-7 / 8.5e-7
bool gemm_direct16_ok(const GemmArgs& g) {
    const int64_t lim = int64_t(1) << 22;
    if (g.n_split > 0 || g.batch != 1 || g.M < 1 || g.N < 1 || g.K < 1 || g.K > INT32_MAX / 2 ||
        g.lda >= lim || g.ldb >= lim || tiles_of(g, 16) > INT32_MAX / 2)
        return false;
    // (16-byte loads from 4-byte aligned addresses where k is contiguous)
    if (g.opA == CDX_OP_N && ((uintptr_t)g.A % 4 != 0 || g.lda % 2 != 0)) return false;
    if (g.opB == CDX_OP_T && ((uintptr_t)g.B % 4 != 0 || g.ldb % 2 != 0)) return false;
    const bool whole = g.M % 64 == 0 && g.N % 64 == 0 && g.K % 64 == 0 && g.lda % 8 == 0 &&
                       g.ldb % 8 == 0 && (uintptr_t)g.A % 16 == 0 && (uintptr_t)g.B % 16 == 0;
    if (g.K > 4096 && splitk_applies(tiles_of(g, 64), g.K)) return false;
    const bool tn = g.opA == CDX_OP_T && g.opB == CDX_OP_N;
    return tiles_of(g, 32) <= (!whole ? 768 : tn ? 320 : 256);
}

int launch_gemm_direct16(const GemmArgs& g, bool bf16, hipStream_t stream) {
    const H16Args p{static_cast<const unsigned short*>(g.A), static_cast<const unsigned short*>(g.B),
                    g.C, g.bias, g.M, g.N, g.K, g.lda, g.ldb, g.ldc, g.bias_mode, g.epilogue};
    const bool small = tiles_of(g, 16) <= 400;
    if (small && bf16) launch_ops<1, true>(g, p, stream);
    else if (small) launch_ops<1, false>(g, p, stream);
    else if (bf16) launch_ops<2, true>(g, p, stream);
    else launch_ops<2, false>(g, p, stream);
    return hip_error(hipGetLastError(), "gemm_direct16_kernel launch");
}

}  // namespace cdx
