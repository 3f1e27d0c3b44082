// FP32 GEMM on gfx950 matrix cores: v_mfma_f32_16x16x4_f32.
//
// Replaces the reference's CUDA-core SGEMMs (sgemm_fast_kernel /
// sgemm_general_kernel, src/kernels/matmul_kernel.cu:458-689).  The
// reference computes each output as an fp32 FMA chain over k; here each
// output is an fp32 MFMA accumulation (the same fp32 products, summed by
// the matrix core four k at a time), which is what the relative-Frobenius
// parity gate compares against.
//
// Which products come here is decided in gemm_f32_route.hip: large ones take
// gemm_parts.hip, small and unaligned ones gemm_direct.hip.  The figures below
// compare this kernel's configurations with each other.
//
// Structure (per workgroup, one BM x BN output tile):
//   * A and B k-tiles of depth BK are staged global -> VGPR -> LDS with
//     register double buffering: the loads for tile t+1 are in flight while
//     the waves run the MFMAs of tile t, and one barrier per k-tile
//     separates the two LDS buffers.
//   * LDS keeps each operand in its global orientation (k-contiguous or
//     m/n-contiguous), so the staging copy is a plain 16-byte copy.  Row
//     strides are padded by 4 floats, which makes both the 16-byte stores
//     and the fragment reads bank-conflict free.
//   * Each wave owns a WM x WN sub-tile = (WM/16) x (WN/16) MFMA blocks of
//     16x16, accumulated in 4 fp32 registers per lane each.
//   * k is consumed 16 at a time: a lane feeds MFMA j (j = 0..3) with
//     k = k0 + 4*(lane/16) + j, for A and B alike, so a k-contiguous operand
//     is read with one 16-byte LDS read per fragment and the four MFMAs
//     together cover k0..k0+15 exactly once.
//   * The epilogue adds an optional per-row / per-column bias, applies
//     ReLU / GELU, and writes through the output map (plain row-major, or
//     the conv map that lands the [OC, B*S] result directly in NCHW).
//   * Workgroup -> tile order is XCD-aware: consecutive dispatch slots go
//     round-robin over the 8 XCDs, so the block id is remapped to give each
//     XCD a contiguous run of tiles, walked in GROUP_M-row groups so the
//     A row-panels and B column-panels of a run share that XCD's L2.
#include "gemm_f32_tile.hpp"

namespace cdx {
namespace {

using namespace f32;

// MODE kLoadChecked launches (ragged M / N, unaligned operands, the ones
// column) run their interior tiles -- clear of the edges and of the ones
// column -- through the unchecked 16-byte loads and epilogue when
// p.interior allows (both operands 16-byte loadable, K and the split-K
// chunk whole k-tiles): 8192 x 784 x 256 NN has 12 of every 13 tile
// columns interior (44 -> 40 us).
template <class CF, int OPA, int OPB, int MODE, bool SPLITN, bool BLK>
__global__ __launch_bounds__(CF::NT)
void gemm_f32_mfma_kernel(KParams p) {
    constexpr int BM = CF::BM, BN = CF::BN, BK = CF::BK;
    static_assert(BK % 16 == 0, "BK must be a multiple of 16");
    __shared__ __attribute__((aligned(16))) float lds[Geo<CF, OPA, OPB>::LDS_FLOATS];

    int tiles_m = (int)ceil_div(p.M, BM), tiles_n = (int)ceil_div(p.N, BN);
    int tm, tn;
    tile_of_block(tiles_m, tiles_n, CF::GROUP_M, tm, tn);
    const int64_t bm = (int64_t)tm * BM, bn = (int64_t)tn * BN;

    // Split-K slice: blockIdx.y owns k in [y*k_chunk, min(K, (y+1)*k_chunk))
    // and writes a plain [M, N] partial (the reduction applies the epilogue).
    if (gridDim.y > 1) {
        const int64_t k0 = (int64_t)blockIdx.y * p.k_chunk;
        p.A += OPA == CDX_OP_N ? k0 : k0 * p.lda;
        p.B += OPB == CDX_OP_N ? k0 * p.ldb : k0;
        p.K = p.K - k0 < p.k_chunk ? p.K - k0 : p.k_chunk;
        p.C += (int64_t)blockIdx.y * p.M * p.N;
    }
    if (gridDim.z > 1) {
        p.A += (int64_t)blockIdx.z * p.sa;
        p.B += (int64_t)blockIdx.z * p.sb;
        p.C += (int64_t)blockIdx.z * p.sc;
    }
    if constexpr (MODE == kLoadChecked) {
        // p.nb: op(B)'s own columns, so the ones column stays on the checked path
        if (p.interior && bm + BM <= p.M && bn + BN <= p.nb) {
            gemm_tile<CF, OPA, OPB, kLoadAlignedVec, SPLITN, BLK>(p, bm, bn, lds);
            return;
        }
    }
    gemm_tile<CF, OPA, OPB, MODE, SPLITN, BLK>(p, bm, bn, lds);
}

template <class CF, int OPA, int OPB, int MODE, bool SPLITN, bool BLK>
int launch_cfg(const KParams& kp, int splits, hipStream_t stream) {
    int64_t tiles = ceil_div(kp.M, CF::BM) * ceil_div(kp.N, CF::BN);
    if (tiles > INT32_MAX) return set_error(CDX_ERR_UNSUPPORTED, "gemm: too many tiles");
    if (kp.batch < 1 || kp.batch > 65535) return set_error(CDX_ERR_UNSUPPORTED, "gemm: batch out of range");
    hipLaunchKernelGGL((gemm_f32_mfma_kernel<CF, OPA, OPB, MODE, SPLITN, BLK>),
                       dim3((unsigned)tiles, (unsigned)splits, (unsigned)kp.batch), dim3(CF::NT), 0, stream, kp);
    return hip_error(hipGetLastError(), "gemm_f32_mfma_kernel launch");
}

template <class CF, int OPA, int OPB, bool BLK>
int launch_mode(const GemmArgs& g, int splits, int64_t k_chunk, hipStream_t stream) {
    KParams kp = kparams_of(g, k_chunk);
    bool aligned = g.ones_col < 0 && kp.vec_a && kp.vec_b && g.K > 0 && g.M % CF::BM == 0 &&
                   g.N % CF::BN == 0 &&
                   g.K % CF::BK == 0 && k_chunk % CF::BK == 0;
    bool split = g.n_split > 0;
    kp.interior = kp.vec_a && kp.vec_b && g.K % CF::BK == 0 && k_chunk % CF::BK == 0;
    if (aligned) {
        return split ? launch_cfg<CF, OPA, OPB, kLoadAlignedVec, true, BLK>(kp, splits, stream)
                     : launch_cfg<CF, OPA, OPB, kLoadAlignedVec, false, BLK>(kp, splits, stream);
    }
    return split ? launch_cfg<CF, OPA, OPB, kLoadChecked, true, BLK>(kp, splits, stream)
                 : launch_cfg<CF, OPA, OPB, kLoadChecked, false, BLK>(kp, splits, stream);
}

template <class CF>
int launch_ops(const GemmArgs& g0, hipStream_t stream) {
    const int64_t tiles = ceil_div(g0.M, CF::BM) * ceil_div(g0.N, CF::BN);
    return with_splitk(g0, tiles, CF::BK, stream,
                       [&](const GemmArgs& g, int splits, int64_t k_chunk) {
        if (g.opA == CDX_OP_N && g.opB == CDX_OP_N) return launch_mode<CF, CDX_OP_N, CDX_OP_N, false>(g, splits, k_chunk, stream);
        if (g.opA == CDX_OP_N && g.opB == CDX_OP_T) return launch_mode<CF, CDX_OP_N, CDX_OP_T, false>(g, splits, k_chunk, stream);
        if (g.opA == CDX_OP_T && g.opB == CDX_OP_N) return launch_mode<CF, CDX_OP_T, CDX_OP_N, false>(g, splits, k_chunk, stream);
        return launch_mode<CF, CDX_OP_T, CDX_OP_T, false>(g, splits, k_chunk, stream);
    });
}

// Two-level k sum (GemmArgs::blocked_sum), NN products only, no split-K
// (a split already sums in two levels).
template <class CF>
int launch_blocked(const GemmArgs& g, hipStream_t stream) {
    return launch_mode<CF, CDX_OP_N, CDX_OP_N, true>(g, 1, g.K, stream);
}

// Tile configurations (chosen by measurement on MI355X).  All use the two-set
// register pipeline, which measured 4-12 % faster everywhere (4096^3: 138
// against 133 TFLOP/s; 2048^3: 130 against 114).
//  * Huge: 128x128x16, 4 waves of 64x32 (one per SIMD; several workgroups
//    per CU), for problems with at least two 128x128 tiles per CU: 4096^3
//    in 977-983 us against 997-1000 with Large (64x32 wave tiles read A
//    with four 16-byte fragment reads and B with eight 4-byte reads per 16
//    k for 32 MFMAs).  With one tile per CU (2048^3) one wave per SIMD
//    hides less latency: 133.5 against 131.4 us, so Large stays there.
//    (Measured slower: 256x128 tiles of 16 waves of 64x32 at 2048^3, 64x64
//    wave tiles (spills), 8-byte B reads, one register staging set.)
//  * Large: 128x128x16, 8 waves of 32x64 -> 2 waves per SIMD, 32 fp32
//    accumulators per lane.
//  * Medium: 64x64x16, 4 waves of 16x64, for problems whose 128x128 tiles
//    would spread unevenly over the 256 CUs, for the split-K slices of
//    products with M < 128 and for small problems.  Against 4 waves of 32x32
//    on the same tile: 3072^3 447 against 458 us, 4100^3 1358 against 1385,
//    8192 x 256 x 784 (NT) 31.6 against 32.5; 4 waves of 64x16 about the
//    same, 64x128 / 128x64 tiles of 64x32 / 32x64 waves 1.3-1.8x slower.
//    (8 waves of 16x32 measured slower than 4 of 32x32 earlier: 2048^3 141
//    against 157 us.)
//  * SkinnyM: M <= 64 with a long N (the conv GEMM, M = out channels):
//    64x64x16, 4 waves of 16x64 (16-byte B fragment reads), XCD groups of
//    one tile row: 64 x 100352 x 576 in 70-72 us, against 73-74 with 4
//    waves of 32x32, 81 with 8 waves of 16x32 or 32x16, 81 with 64x128
//    tiles of 8 waves of 16x64, 79-84 with 64x32 / 32x64 tiles, 123-125
//    with 64x128 / 64x256 tiles of 32x64 waves, 218 with BK = 32.  A short
//    last round of tiles runs as 64x32 / 64x16 tiles (gemm_f32_skinny_rem_kernel).
//  * NarrowN: N <= 16 (the MLP's 10-class layer): 32x16 tiles, 2 waves, and
//    a deep k-tile (64): such products read A once and are bound by the
//    latency of their k-loop, so each workgroup takes few, large k-steps and
//    twice as many workgroups share the GPU (64x16x16 tiles: 8192 x 10 x
//    256 in 9.5 us, against 13.4 for mostly-empty 64x64 ones).  A 16-row
//    tile for M <= 16 measured no faster than Medium.
//  * W112: N a multiple of 112 but not of 64 (C4's 784-wide backward-data
//    product): 128x112x16, 8 waves of 16x112, so no tile column is ragged
//    (8192 x 784 x 256 NN: 35.5 us, against 40.0 on 64x64 tiles with a
//    16-wide edge column, 57 with 4 waves of 32x112, 52 with 256x112).
//  * SplitTall: split-K slices of products with M >= 128: 128x64x16, 8
//    waves of 32x32 (C4's weight + bias gradient 256 x 785 x 8192: 48.4 us
//    against 54.5 on 64x64 slices; 128x128: 51.5; any BK = 32 slice: 58-79).
using CfgLarge = Cfg<128, 128, 16, 32, 64, 8, 2>;
using CfgHuge = Cfg<128, 128, 16, 64, 32, 8, 2>;
using CfgMedium = Cfg<64, 64, 16, 16, 64, 8, 2>;
using CfgSkinnyM = Cfg<64, 64, 16, 16, 64, 1, 2>;
using CfgNarrowN = Cfg<32, 16, 64, 16, 16, 8, 2>;
using CfgW112 = Cfg<128, 112, 16, 16, 112, 8, 2>;
using CfgSplitTall = Cfg<128, 64, 16, 32, 32, 8, 2>;
using CfgSkinnyHalf = Cfg<64, 32, 16, 16, 32, 1, 2>;
using CfgSkinnyQuarter = Cfg<64, 16, 16, 16, 16, 1, 2>;

// SkinnyM products whose 64-column tiles leave a last round over the 256 CUs
// well short of full: those last tiles run as f = 2 or 4 times as many
// 64 x (64 / f) tiles (same 256 threads, waves of 16 x 64 / f) after the full
// ones, so the busiest CU's share of the last round drops from one tile to
// ceil(rem * f / 256) / f of one.  C5's im2col rounds, 882 and 686 tiles: 4
// -> 3.5 tiles, 42.1 -> 39.3 us, and 3 -> 2.75 tiles, unchanged at 33.3 us;
// the whole batch, 1568 tiles: 7 -> 6.25, 70.8 -> 64.4 us.  Every output
// keeps its k order: the sums are the same bits as on 64 x 64 tiles.  NN,
// whole tiles only.
template <class CFR, bool SPLITN, bool BLK>
__global__ __launch_bounds__(CfgSkinnyM::NT)
void gemm_f32_skinny_rem_kernel(KParams p, int full_tiles) {
    static_assert(CfgSkinnyM::NT == CFR::NT && CFR::BM == CfgSkinnyM::BM, "same block, same rows");
    constexpr int L1 = Geo<CfgSkinnyM, CDX_OP_N, CDX_OP_N>::LDS_FLOATS;
    constexpr int L2 = Geo<CFR, CDX_OP_N, CDX_OP_N>::LDS_FLOATS;
    __shared__ __attribute__((aligned(16))) float lds[L1 > L2 ? L1 : L2];
    const int b = blockIdx.x;
    if (b < full_tiles)
        gemm_tile<CfgSkinnyM, CDX_OP_N, CDX_OP_N, kLoadAlignedVec, SPLITN, BLK>(
            p, 0, (int64_t)b * CfgSkinnyM::BN, lds);
    else
        gemm_tile<CFR, CDX_OP_N, CDX_OP_N, kLoadAlignedVec, SPLITN, BLK>(
            p, 0, (int64_t)full_tiles * CfgSkinnyM::BN + (int64_t)(b - full_tiles) * CFR::BN, lds);
}

// Full tile count and split factor f of the last round when the split launch
// applies: an unsplit NN product of exactly one 64-row tile, whole 64-column
// tiles, whole k-tiles, 16-byte loadable operands, and a last round of rem
// tiles that f splits to less than one tile per CU: f = 4 for rem <= 64
// (1/4) and 128 < rem <= 192 (3/4), f = 2 for 64 < rem <= 128 (1/2).
bool skinny_rem_plan(const GemmArgs& g, int64_t& full, int& f) {
    const KParams kp = kparams_of(g, g.K);
    if (g.M != CfgSkinnyM::BM || g.N % CfgSkinnyM::BN != 0 || g.K <= 0 ||
        g.K % CfgSkinnyM::BK != 0 || g.batch != 1 || g.ones_col >= 0 || !kp.vec_a ||
        !kp.vec_b || g.opA != CDX_OP_N || g.opB != CDX_OP_N)
        return false;
    const int64_t tiles = g.N / CfgSkinnyM::BN, rem = tiles % 256;
    if (rem == 0 || rem > 192 || tiles + 3 * rem > INT32_MAX) return false;
    full = tiles - rem;
    f = rem > 64 && rem <= 128 ? 2 : 4;
    return true;
}

template <bool BLK>
int launch_skinny_rem(const GemmArgs& g, int64_t full, int f, hipStream_t stream) {
    const KParams kp = kparams_of(g, g.K);
    const int64_t rem = g.N / CfgSkinnyM::BN - full;
    const dim3 grid((unsigned)(full + f * rem)), block(CfgSkinnyM::NT);
    const bool sn = g.n_split > 0;
    if (f == 2 && sn)
        hipLaunchKernelGGL((gemm_f32_skinny_rem_kernel<CfgSkinnyHalf, true, BLK>), grid, block, 0, stream, kp, (int)full);
    else if (f == 2)
        hipLaunchKernelGGL((gemm_f32_skinny_rem_kernel<CfgSkinnyHalf, false, BLK>), grid, block, 0, stream, kp, (int)full);
    else if (sn)
        hipLaunchKernelGGL((gemm_f32_skinny_rem_kernel<CfgSkinnyQuarter, true, BLK>), grid, block, 0, stream, kp, (int)full);
    else
        hipLaunchKernelGGL((gemm_f32_skinny_rem_kernel<CfgSkinnyQuarter, false, BLK>), grid, block, 0, stream, kp, (int)full);
    return hip_error(hipGetLastError(), "gemm_f32_skinny_rem_kernel launch");
}

// Configuration choice, shared by the launcher and the workspace query.
enum class F32Cfg { NarrowN, SkinnyM, Huge, Large, Medium, W112, SplitTall };

// Large tiles are ~8 % faster per tile, but a CU's time is set by its largest
// share of tiles: Large is taken when its busiest-CU share (rounded up to
// whole tiles per CU over the 256 CUs) is within 5 % of Medium's.  (2048^3,
// 256 tiles: 130 against 141 us; 3072^3, 576 tiles: 561 against 459.)
bool large_balanced(int64_t M, int64_t N) {
    const int64_t tl = ceil_div(M, 128) * ceil_div(N, 128);
    const int64_t tm = ceil_div(M, 64) * ceil_div(N, 64);
    const int64_t cus = 256;
    if (tl < cus) return false;
    // ceil(tl/cus)/(tl/cus) <= 1.05 * ceil(tm/cus)/(tm/cus)
    return ceil_div(tl, cus) * tm * 100 <= 105 * ceil_div(tm, cus) * tl;
}

F32Cfg choose_f32(const GemmArgs& g, bool& blocked) {
    const bool split = g.batch == 1 && splitk_applies(ceil_div(g.M, 64) * ceil_div(g.N, 64), g.K);
    blocked = g.blocked_sum && !split && g.opA == CDX_OP_N && g.opB == CDX_OP_N;
    if (g.N <= 16) return F32Cfg::NarrowN;
    if (split && !blocked) return g.M >= 128 ? F32Cfg::SplitTall : F32Cfg::Medium;
    if (!blocked && !split && g.N % 112 == 0 && g.N % 64 != 0 &&
        ceil_div(g.M, 128) * (g.N / 112) >= 256)
        return F32Cfg::W112;
    if (g.M <= 64 && g.N >= 4096) return F32Cfg::SkinnyM;
    if (large_balanced(g.M, g.N))
        return ceil_div(g.M, 128) * ceil_div(g.N, 128) >= 512 ? F32Cfg::Huge : F32Cfg::Large;
    return F32Cfg::Medium;
}

template <class CF>
size_t ws_of(const GemmArgs& g) {
    return splitk_bytes(g, ceil_div(g.M, CF::BM) * ceil_div(g.N, CF::BN), CF::BK);
}

}  // namespace

bool f32_takes_w112(const GemmArgs& g) {
    bool blocked;
    return choose_f32(g, blocked) == F32Cfg::W112;
}

static size_t cfg_workspace(const GemmArgs& g, F32Cfg c) {
    switch (c) {
        case F32Cfg::NarrowN: return ws_of<CfgNarrowN>(g);
        case F32Cfg::SkinnyM: return ws_of<CfgSkinnyM>(g);
        case F32Cfg::Large: return ws_of<CfgLarge>(g);
        case F32Cfg::Huge: return ws_of<CfgHuge>(g);
        case F32Cfg::W112: return ws_of<CfgW112>(g);
        case F32Cfg::SplitTall: return ws_of<CfgSplitTall>(g);
        default: return ws_of<CfgMedium>(g);
    }
}

size_t gemm_f32_tiled_workspace(const GemmArgs& g) {
    bool blocked;
    const F32Cfg c = choose_f32(g, blocked);
    return blocked ? 0 : cfg_workspace(g, c);
}

int launch_gemm_f32_tiled(const GemmArgs& g, hipStream_t stream) {
    bool blocked;
    const F32Cfg c = choose_f32(g, blocked);
    int64_t full = 0;
    int f = 1;
    if (c == F32Cfg::SkinnyM && skinny_rem_plan(g, full, f))
        return blocked ? launch_skinny_rem<true>(g, full, f, stream)
                       : launch_skinny_rem<false>(g, full, f, stream);
    if (blocked) {
        switch (c) {
            case F32Cfg::NarrowN: return launch_blocked<CfgNarrowN>(g, stream);
            case F32Cfg::SkinnyM: return launch_blocked<CfgSkinnyM>(g, stream);
            case F32Cfg::Large: return launch_blocked<CfgLarge>(g, stream);
            case F32Cfg::Huge: return launch_blocked<CfgHuge>(g, stream);
            default: return launch_blocked<CfgMedium>(g, stream);
        }
    }
    switch (c) {
        case F32Cfg::NarrowN: return launch_ops<CfgNarrowN>(g, stream);
        case F32Cfg::SkinnyM: return launch_ops<CfgSkinnyM>(g, stream);
        case F32Cfg::Large: return launch_ops<CfgLarge>(g, stream);
        case F32Cfg::Huge: return launch_ops<CfgHuge>(g, stream);
        case F32Cfg::W112: return launch_ops<CfgW112>(g, stream);
        case F32Cfg::SplitTall: return launch_ops<CfgSplitTall>(g, stream);
        default: return launch_ops<CfgMedium>(g, stream);
    }
}

}  // namespace cdx
