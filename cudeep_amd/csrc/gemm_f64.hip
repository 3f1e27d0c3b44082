// fp64 GEMM, C = op(A) * op(B), for float64 tensors.
//
// Replaces sgemm_double_kernel (src/kernels/matmul_kernel.cu:691-743), a
// 64x64-tile scalar-FMA kernel.  Here: v_mfma_f64_16x16x4_f64 (64 cycles per
// SIMD: 78.6 TFLOP/s, which is the bound).  Fragment feeding as in the FP32
// kernel: A lane l holds row l%16, k l/16; B lane l holds k l/16, column
// l%16.  The 16x16 fp64 result sits 4 doubles per lane, interleaved unlike
// the fp32 16x16x4 layout: register r of lane l holds row 4*r + l/16, column
// l%16.
//
// Per workgroup (four waves, 2 x 2) one tile and k-tiles of 16, double
// buffered in LDS in the operand's own orientation, so that loads and LDS
// stores both run along it: [m or n][17] where k is contiguous in memory,
// else [k][m or n] (+ 16: the two k a half-wave reads lie 32 banks apart).
// Two register sets keep k-tile t + 2
// in flight while t + 1 is stored and t is multiplied: a 64 x 64 tile has
// 1024 MFMA cycles per k-tile and SIMD to cover one load.  Loads are 8 bytes
// from indices clamped into the operand, so ragged sizes run the same code;
// only the last k-tile zeroes its k past the end.
#include "cdx_internal.hpp"

namespace cdx {
namespace {

constexpr int DBK = 16;

struct DArgs {
    const double* A; const double* B; double* C;
    int64_t M, N, K, lda, ldb, ldc;
};

// One operand's k-tile: BMN (m or n) x 16 k.  KC: k is the contiguous
// dimension.
template <int BMN, bool KC>
struct DLoader {
    static constexpr int NV = BMN * DBK / 256;
    static constexpr int STRIDE = KC ? DBK + 1 : BMN + 16;
    static constexpr int ELEMS = STRIDE * (KC ? BMN : DBK);
    double v[NV];

    __device__ __forceinline__ static int mn_of(int i, int tid) {
        return KC ? (tid + i * 256) / DBK : (tid + i * 256) % BMN;
    }
    __device__ __forceinline__ static int k_of(int i, int tid) {
        return KC ? tid % DBK : (tid + i * 256) / BMN;
    }
    __device__ __forceinline__ static int at(int mn, int k) {
        return KC ? mn * STRIDE + k : k * STRIDE + mn;
    }
    // mnlast, klast: the last valid index of either dimension, from (mn0, k0)
    __device__ __forceinline__ void load(const double* X, int64_t ld, int64_t mn0, int64_t k0,
                                         int64_t mnlast, int64_t klast, int tid) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int64_t mn = mn0 + (mn_of(i, tid) < mnlast ? mn_of(i, tid) : mnlast);
            const int64_t k = k0 + (k_of(i, tid) < klast ? k_of(i, tid) : klast);
            v[i] = X[KC ? mn * ld + k : k * ld + mn];
        }
    }
    __device__ __forceinline__ void store(double* s, int64_t klast, int tid) const {
#pragma unroll
        for (int i = 0; i < NV; ++i)
            s[at(mn_of(i, tid), k_of(i, tid))] = k_of(i, tid) <= klast ? v[i] : 0.0;
    }
};

template <int BM, int BN, int OPA, int OPB>
__global__ __launch_bounds__(256)
void dgemm_kernel(DArgs p) {
    using LA = DLoader<BM, OPA == CDX_OP_N>;
    using LB = DLoader<BN, OPB == CDX_OP_T>;
    constexpr int FM = BM / 32, FN = BN / 32;   // 16 x 16 blocks per wave
    __shared__ double sA[2][LA::ELEMS], sB[2][LB::ELEMS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, lq = lane >> 4;
    const int wm0 = (wave >> 1) * (BM / 2), wn0 = (wave & 1) * (BN / 2);
    const int64_t bm = (int64_t)blockIdx.y * BM, bn = (int64_t)blockIdx.x * BN;

    doublex4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = doublex4{0.0, 0.0, 0.0, 0.0};

    const int64_t nk = ceil_div(p.K, DBK);
    const int64_t mlast = p.M - 1 - bm, nlast = p.N - 1 - bn;
    auto load = [&](LA& a, LB& b, int64_t t) {   // past the last k-tile: that one again, unused
        if (t >= nk) t = nk - 1;
        const int64_t k0 = t * DBK, klast = p.K - 1 - k0;
        a.load(p.A, p.lda, bm, k0, mlast, klast, tid);
        b.load(p.B, p.ldb, bn, k0, nlast, klast, tid);
    };
    auto store = [&](const LA& a, const LB& b, int64_t t) {
        const int64_t klast = p.K - 1 - t * DBK;
        a.store(sA[t & 1], klast, tid);
        b.store(sB[t & 1], klast, tid);
    };
    auto compute = [&](int64_t t) {
        const double* ta = sA[t & 1];
        const double* tb = sB[t & 1];
#pragma unroll
        for (int kk = 0; kk < DBK; kk += 4) {
            double a[FM], b[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i) a[i] = ta[LA::at(wm0 + i * 16 + l16, kk + lq)];
#pragma unroll
            for (int j = 0; j < FN; ++j) b[j] = tb[LB::at(wn0 + j * 16 + l16, kk + lq)];
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    };

    if (nk > 0) {
        LA a0, a1;
        LB b0, b1;
        load(a0, b0, 0);
        load(a1, b1, 1);
        store(a0, b0, 0);
        __syncthreads();
        // top of iteration t (even): stage 0 holds k-tile t, set 1 t + 1
        for (int64_t t = 0; t < nk; t += 2) {
            load(a0, b0, t + 2);
            compute(t);
            if (t + 1 >= nk) break;
            store(a1, b1, t + 1);
            __syncthreads();
            load(a1, b1, t + 3);
            compute(t + 1);
            if (t + 2 >= nk) break;
            store(a0, b0, t + 2);
            __syncthreads();
        }
    }
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t m = bm + wm0 + i * 16 + 4 * r + lq, n = bn + wn0 + j * 16 + l16;
                if (m < p.M && n < p.N) p.C[m * p.ldc + n] = acc[i][j][r];
            }
}

template <int BM, int BN>
int launch_tile(int opA, int opB, const DArgs& p, hipStream_t stream) {
    const int64_t gx = ceil_div(p.N, BN), gy = ceil_div(p.M, BM);
    if (gx > INT32_MAX || gy > 65535) return set_error(CDX_ERR_UNSUPPORTED, "dgemm: grid too large");
    const dim3 grid((unsigned)gx, (unsigned)gy), block(256);
    if (opA == CDX_OP_N && opB == CDX_OP_N)
        hipLaunchKernelGGL((dgemm_kernel<BM, BN, CDX_OP_N, CDX_OP_N>), grid, block, 0, stream, p);
    else if (opA == CDX_OP_N)
        hipLaunchKernelGGL((dgemm_kernel<BM, BN, CDX_OP_N, CDX_OP_T>), grid, block, 0, stream, p);
    else if (opB == CDX_OP_N)
        hipLaunchKernelGGL((dgemm_kernel<BM, BN, CDX_OP_T, CDX_OP_N>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((dgemm_kernel<BM, BN, CDX_OP_T, CDX_OP_T>), grid, block, 0, stream, p);
    return hip_error(hipGetLastError(), "dgemm_kernel launch");
}

}  // namespace

int launch_dgemm(int opA, int opB, int64_t M, int64_t N, int64_t K,
                 const double* A, int64_t lda, const double* B, int64_t ldb,
                 double* C, int64_t ldc, hipStream_t stream) {
    const DArgs p{A, B, C, M, N, K, lda, ldb, ldc};
    // 64 x 64 tiles (half the LDS reads per MFMA) once there are three per CU:
    // 2048^3 389 against 412 us; below that 32 x 32 ones, four times as many
    // (1200^3 108 against 119, 512^3 18 against 35, 256 x 74 x 960 27 against
    // 64).  The one 64 x 64 kernel before this took 507, 259, 65 and 129 us.
    if (ceil_div(M, 64) * ceil_div(N, 64) >= 768) return launch_tile<64, 64>(opA, opB, p, stream);
    return launch_tile<32, 32>(opA, opB, p, stream);
}

}  // namespace cdx
