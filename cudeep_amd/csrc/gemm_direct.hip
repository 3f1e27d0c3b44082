// FP32 GEMM without LDS staging, for products too small to fill the GPU with
// the tiled kernels' workgroups: every wave reads its MFMA operands straight
// from global memory.
//
// A 64 x 64 tile per workgroup leaves 512^3 with 64 workgroups on 256 CUs, one
// wave per SIMD on a quarter of them, each going through load -> LDS ->
// barrier -> MFMA for every 16 k.  Here a wave owns 16 FM x 16 FN outputs and
// keeps four 16-k steps of operands in flight in registers, with no barrier:
// v_mfma_f32_16x16x4_f32 takes 32 cycles, so a 32 x 32 wave tile has 512 MFMA
// cycles per step to cover four 16-byte loads (k-contiguous operands; 4-byte
// loads of 16 neighbours, where the other dimension is contiguous).  The k
// order and grouping per output are the tiled FP32 kernels' (lane group lq
// feeds MFMA q with k = k0 + 4 lq + q), so without a k split the results are
// the same bits.  WK > 1: the waves of a workgroup share its tile, each with
// its own run of k, summed in wave order through LDS.
//
// Any alignment and any size at the same speed: rows and columns past the
// edge read the last one, and only the last, partial step of 16 k is
// bounds-checked.
#include "gemm_f32_tile.hpp"

namespace cdx {
namespace {

using f32::KParams;

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// One operand's 16 F rows (m or n) x 16 k of a wave.  KC: k contiguous.
template <int F, bool KC>
struct DirectLoader {
    f32x4u v[F];         // element q: k = k0 + 4 lq + q
    template <class O>
    __device__ __forceinline__ void load(const char* base, const uint32_t (&off)[F], O ld_b) {
#pragma unroll
        for (int i = 0; i < F; ++i) {
            if constexpr (KC) {
                v[i] = *(const __attribute__((address_space(1))) f32x4u*)(base + off[i]);
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    v[i][q] = *(const __attribute__((address_space(1))) float*)(base + q * ld_b + off[i]);
            }
        }
    }
    // the last step: k >= krem reads as 0
    __device__ __forceinline__ void load_tail(const char* base, const uint32_t (&off)[F],
                                              int64_t ld_b, int k, int krem) {
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                v[i][q] = k + q < krem ? *(const float*)(base + (KC ? q * 4 : q * ld_b) + off[i]) : 0.0f;
    }
};

template <int FM, int FN, int WM, int WN, int WK, int OPA, int OPB, bool SPLITN>
__global__ __launch_bounds__(256)
void gemm_direct_kernel(KParams p) {
    static_assert(WM * WN * WK == 4, "four waves");
    constexpr bool KCA = OPA == CDX_OP_N, KCB = OPB == CDX_OP_T;
    constexpr int BM = 16 * FM * WM, BN = 16 * FN * WN, DEPTH = 4;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, lq = lane >> 4;
    const int wk = wave % WK, wmn = wave / WK;
    int tm, tn;
    f32::tile_of_block((int)ceil_div(p.M, BM), (int)ceil_div(p.N, BN), 8, tm, tn);
    const int64_t m0 = (int64_t)tm * BM + wmn / WN * 16 * FM, n0 = (int64_t)tn * BN + wmn % WN * 16 * FN;
    if (gridDim.z > 1) {
        p.A += (int64_t)blockIdx.z * p.sa;
        p.B += (int64_t)blockIdx.z * p.sb;
        p.C += (int64_t)blockIdx.z * p.sc;
    }
    // (a wave tile wholly past the edge reads the operand's last row / column)
    const int64_t ma = m0 < p.M ? m0 : p.M - 1, nb = n0 < p.nb ? n0 : p.nb - 1;
    uint32_t offa[FM], offb[FN];
    bool one[FN];   // this lane's column is the ones column
    const int64_t lda_b = p.lda * 4, ldb_b = p.ldb * 4;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int64_t r = ma + i * 16 + l16 < p.M ? i * 16 + l16 : p.M - 1 - ma;
        offa[i] = (uint32_t)(KCA ? r * lda_b + 16 * lq : 4 * lq * lda_b + r * 4);
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int64_t r = nb + j * 16 + l16 < p.nb ? j * 16 + l16 : p.nb - 1 - nb;
        offb[j] = (uint32_t)(KCB ? r * ldb_b + 16 * lq : 4 * lq * ldb_b + r * 4);
        one[j] = n0 + j * 16 + l16 == p.ones;
    }
    const char* pa = reinterpret_cast<const char*>(p.A + (KCA ? ma * p.lda : ma));
    const char* pb = reinterpret_cast<const char*>(p.B + (KCB ? nb * p.ldb : nb));
    const int64_t sa = KCA ? 64 : 16 * lda_b, sb = KCB ? 64 : 16 * ldb_b;   // bytes per 16 k

    floatx4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    DirectLoader<FM, KCA> a[DEPTH];
    DirectLoader<FN, KCB> b[DEPTH];
    auto mul = [&](const DirectLoader<FM, KCA>& x, const DirectLoader<FN, KCB>& y) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        x.v[i][q], one[j] ? 1.0f : y.v[j][q], acc[i][j], 0, 0, 0);
    };

    // this wave's whole steps [s0, s1); the partial one goes to the last wave
    const int full = (int)(p.K / 16), krem = (int)(p.K % 16);
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
        a[0].load_tail(pa + full * sa, offa, lda_b, 4 * lq, krem);
        b[0].load_tail(pb + full * sb, offb, ldb_b, 4 * lq, krem);
        mul(a[0], b[0]);
    }

    const EpiArgs epi{p.C, p.ldc, p.M, p.N, p.n_split, p.ldc_split, p.bias, p.bias_mode,
                      p.epilogue, p.aux, p.ldaux, p.colsum, p.nb};
    if constexpr (WK == 1) {
        if (m0 >= p.M || n0 >= p.N) return;
        if (m0 + 16 * FM <= p.M && n0 + 16 * FN <= p.nb)
            write_acc<FM, FN, false, SPLITN>(acc, epi, m0, n0, lane);
        else
            write_acc<FM, FN, true, SPLITN>(acc, epi, m0, n0, lane);
    } else {
        // blocks of the tile dealt to the waves; each summed over k in wave order
        static_assert(WM == 1 && WN == 1, "one tile per workgroup");
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
        write_acc<1, 1, true, SPLITN>(sum, epi, m0 + wk / FN * 16, n0 + wk % FN * 16, lane);
    }
}

template <int FM, int FN, int WM, int WN, int WK>
int launch_cfg(const GemmArgs& g, hipStream_t stream) {
    const KParams kp = f32::kparams_of(g, g.K);
    const int64_t tiles = ceil_div(g.M, 16 * FM * WM) * ceil_div(g.N, 16 * FN * WN);
    const dim3 grid((unsigned)tiles, 1, (unsigned)g.batch), block(256);
    if constexpr (WK == 1) {   // (the NCHW map keeps one k order: launch_gemm_direct)
        if (g.n_split > 0) {
            hipLaunchKernelGGL((gemm_direct_kernel<FM, FN, WM, WN, WK, CDX_OP_N, CDX_OP_N, true>), grid, block, 0, stream, kp);
            return hip_error(hipGetLastError(), "gemm_direct_kernel launch");
        }
    }
    if (g.opA == CDX_OP_N && g.opB == CDX_OP_N)
        hipLaunchKernelGGL((gemm_direct_kernel<FM, FN, WM, WN, WK, CDX_OP_N, CDX_OP_N, false>), grid, block, 0, stream, kp);
    else if (g.opA == CDX_OP_N)
        hipLaunchKernelGGL((gemm_direct_kernel<FM, FN, WM, WN, WK, CDX_OP_N, CDX_OP_T, false>), grid, block, 0, stream, kp);
    else if (g.opB == CDX_OP_N)
        hipLaunchKernelGGL((gemm_direct_kernel<FM, FN, WM, WN, WK, CDX_OP_T, CDX_OP_N, false>), grid, block, 0, stream, kp);
    else
        hipLaunchKernelGGL((gemm_direct_kernel<FM, FN, WM, WN, WK, CDX_OP_T, CDX_OP_T, false>), grid, block, 0, stream, kp);
    return hip_error(hipGetLastError(), "gemm_direct_kernel launch");
}

int64_t tiles_of(const GemmArgs& g, int64_t side) {
    const int64_t nb = g.ones_col >= 0 ? g.ones_col : g.N;
    return ceil_div(g.M, side) * ceil_div(nb, side) * g.batch;
}

}  // namespace

// Configurations: 32 x 32 outputs per workgroup with k in four runs, one per
// wave; 32 x 32 as four 16 x 16 waves; 16 x 16 with k in four runs.  A k split
// costs one pass through LDS and is worth it from a few steps per wave on:
//                      32x32/4   4x 16x16   16x16/4   64x64 tiled kernel (us)
//   512^3 NN             7.4       7.6        9.1       14.0
//   256^3 NN             5.5       5.2        3.9        8.4
//   64 x 256 x 784 NT    9.0       9.6        5.2       19.3
//   200 x 1000 x 70 NN   4.6       4.1        4.6        7.4
//   128 x 1024 x 626 TT  7.6       8.5        6.4       26.6
//   304 x 153 x 1800 NT 15.8      20.4        8.3       63.7
//   877 x 129 x 2046 TT 16.0      26.1       16.8       91.3
//   1021 x 765 x 1533   32.5      51.1       57.5       93.0
//   2000 x 700 x 500    24.4      27.6       34.4       30.4
//   600^3 NT            10.8                            (unaligned rows)
//   768^3 NN / NT       18.8 / 23.2  23.9    22.1       19.9 / 19.9
//   1024^3 NN           28.7      39.9       48.1       25.7
//   8192 x 256 x 784 NT 38.9      60.6       67.2       31.8
// so: all products of up to 400 32 x 32 tiles, and beyond that those whose
// rows or k the tiled kernel would have to check element by element, up to
// where its larger tiles win even so (soonest where k past the last 16 is all
// that it has to check, for a short k, a transposed A, and M or N up to 64,
// which has its own wide tiles there; NT below 128 k by the parity of its 16-k
// steps).  Tiled / this, us (tiles):
//   1200 x 1200 x 300 NT 21.2 / 17.8 (1444)    16896 x 84 x 1564 NT 102 / 68 (1584)
//   1584 x 1552 x 50 NT  11.8 / 9.0 (2450)     4160 x 384 x 680 TN  33.8 / 37.8 (1560)
//   1601^2 x 61 NN       15.9 / 13.5 (2601)
//   1601^2 x 127 NT      19.6 / 23.2           1601^2 x 65 NT       10.5 / 16.0
//   1368 x 1664 x 153 TT 19.2 / 15.0 (2236)    8192 x 300 x 100 TN  13.2 / 16.4 (2560)
//   1999 x 1501 x 701 NT 89.7 / 56.3 (2961)    1999 x 1501 x 701 TN 66.9 / 66.9
//   548 x 4441 x 120 NN  16.7 / 15.5 (2502)    14912 x 196 x 2302 NN 235 / 177 (3262)
//   61 x 100001 x 300 NN 61.9 / 91.0 (6252)
//   NCHW map, with the im2col before it: 96 x 13456 x 585 52.8 / 46.6 (1263),
//   200 x 7688 x 549 49.7 / 52.8 (1687), 256 x 26912 x 459 104.5 / 133.3 (6728);
//   only k ragged, 128 x 6272 x 1044 51.5 / 56.5 (784), 96 x 7688 x 1224 64.5 / 56.5
//   (723: the tiled kernel pads M), 32 x 200704 x 36 40.2 / 34.2 (6272)
// 64-row NN products and the convolutions' output map keep one k order, that
// of the tiled kernels, so that the same column of a wider product (another
// round of images) is the same bits.
bool gemm_direct_ok(const GemmArgs& g) {
    const int64_t nb = g.ones_col >= 0 ? g.ones_col : g.N, lim = int64_t(1) << 22;
    if (g.blocked_sum || g.M < 1 || nb < 1 || g.K < 1 || g.K > INT32_MAX / 2 || g.batch < 1 ||
        g.batch > 65535 || g.lda >= lim || g.ldb >= lim ||
        (g.n_split > 0 && (g.opA != CDX_OP_N || g.opB != CDX_OP_N)))
        return false;
    if (g.batch == 1 && splitk_applies(ceil_div(g.M, 64) * ceil_div(nb, 64), g.K)) return false;
    const int64_t t32 = tiles_of(g, 32);
    if (t32 <= 400) return true;
    const KParams kp = f32::kparams_of(g, g.K);
    if (g.n_split > 0 && g.M <= 32 && t32 <= 8192)   // (64-row tiles at most half used)
        return g.K % 16 != 0 || !kp.vec_a || !kp.vec_b;
    if (t32 > (g.K >= 128 ? 4096 : 3000)) return false;
    const bool nt = g.opA == CDX_OP_N && g.opB == CDX_OP_T;
    if (kp.vec_a && kp.vec_b) {
        if (g.n_split > 0) return g.K % 16 != 0 && g.M % 64 != 0 && t32 <= 1200;
        return g.K % 16 != 0 && t32 <= (nt && g.K >= 384 ? 2200 : 1450);
    }
    if (t32 <= (g.n_split > 0 ? 1500 : 1700)) return true;
    if (g.n_split > 0 || g.M <= 64 || nb <= 64) return false;
    const bool neither = !kp.vec_a && !kp.vec_b;
    if (nt) return g.K >= 128 || (g.K > 48 && ceil_div(g.K, 16) % 2 == 0);
    if (g.opB == CDX_OP_T) return g.K >= 32 && !kp.vec_b;
    if (g.opA == CDX_OP_T) return neither && t32 <= 2500;
    return g.K >= 32 || neither || t32 <= 2500;
}

// In the TF32 modes (exact fp32 products are inside their error bar): while
// the split kernel's tiles leave most CUs idle (512^3 NN 7.5 against 9.5 us, 64
// x 256 x 784 NT 5.2 against 21.0, 304 x 153 x 1800 NT 8.3 against 45.4; 768^3
// 18.9 against 13.3), and where that kernel would have to load element by
// element (1021 x 765 x 1533 NT 32.5 against 63.7, 1336 x 576 x 381 TN 12.7
// against 18.5; with 16-byte rows 2000 x 700 x 500 24.4 against 21.3).
bool gemm_direct_for_tf32(const GemmArgs& g) {
    // (wide 64-row products keep the split kernel's own k-slices)
    if (g.n_split > 0 || (g.M <= 64 && g.N >= 4096) || !gemm_direct_ok(g)) return false;
    const int64_t t32 = tiles_of(g, 32);
    const KParams kp = f32::kparams_of(g, g.K);
    return t32 <= 256 || (t32 <= 1024 && !(kp.vec_a && kp.vec_b));
}

int launch_gemm_direct(const GemmArgs& g, hipStream_t stream) {
    const bool one_order = g.n_split > 0 || (g.M <= 64 && g.opA == CDX_OP_N && g.opB == CDX_OP_N);
    if (one_order || g.K < 128) return launch_cfg<1, 1, 2, 2, 1>(g, stream);
    if (tiles_of(g, 16) <= 512) return launch_cfg<1, 1, 1, 1, 4>(g, stream);
    return launch_cfg<2, 2, 1, 1, 4>(g, stream);
}

}  // namespace cdx
