// FP32 GEMM on the bf16 matrix cores: every fp32 operand as the exact sum of
// three bf16 parts.
//
// v_mfma_f32_16x16x4_f32 runs at 157 TFLOP/s, v_mfma_f32_16x16x32_bf16 at 16
// times that rate, so six bf16 products per fp32 product have a ceiling of
// 419 TFLOP/s.  Each element x is split on its way into LDS,
//     h = bf16(x),  m = bf16(x - h),  l = x - h - m   (RNE)
// where both differences are exact and l has at most 8 significant bits, so
// x = h + m + l exactly, and
//     a b = ah bh + (ah bm + am bh) + (am bm + ah bl + al bh)  +  r
// with |r| <= 2^-24 |ab|, 2^-27 in the mean square (am bl + al bm + al bl: |m| <=
// 2^-8 |x|, |l| <= 2^-17 |x|).  The six products of a 32-k step are summed from
// zero, small ones first, and added to the accumulator by an fp32 add: added by
// the matrix instruction itself, whose sums round towards one side, the errors
// of a column of outputs all lean the same way (relative Frobenius error 1.00e-6
// at 4096^3, most of it bias; the column sums off by 1.3e-5).  Relative Frobenius
// error against fp64, N(0, 1) operands (in brackets the fp32-MFMA kernels'):
// 4096^3 1.7e-7 (1.15e-6), 2048^3 1.3e-7 (8.1e-7), 8192 x 784 x 256 6.4e-8
// (2.9e-7), 256 x 785 x 8192 in k-slices 1.6e-7 (3.2e-7).
//
// Sparse rows are where it is the less exact one.  The fp32 matrix instruction
// forms a product whole and rounds to nearest; here r is left out and the
// largest term is added with a one-sided rounding, so an output that is one
// product is off by up to 2^-23 + 2^-24 instead of 2^-24.  2048^3, N(0, 1)
// nonzeros, in brackets the fp32-MFMA kernels': a diagonal A 3.5e-8 (2.5e-8; at
// most 2^-22.6 of an output against 2^-24), 3 per row 5.1e-8 (3.6e-8), 8 6.5e-8
// (5.4e-8), 16 7.8e-8 (7.4e-8), 30 9.3e-8 (9.9e-8); identities, permutations and
// powers of two are exact.  With h h in an accumulator of its own, added to the
// others' sum by fp32 adds, a diagonal A is at 2.6e-8 and three per row at
// 4.3e-8, for 5 % more time (4096^3 731 -> 775 us, 2048^3 94 -> 100).
//
// Range.  The parts are exact for |x| >= 2^-110 (or 0), where l stays above
// bf16's smallest normal magnitude, and finite below bf16's rounding limit.  A
// smaller x loses at most 2^-125, and a product of parts that the matrix core
// flushes 2^-126.  So nothing is lost to speak of while the least magnitudes of
// both operands (0 aside) are at least 2^-110 and their product 2^-98 (2^-28
// of each product); else an output is off by at most K 2^-125 max|x| + K 6
// 2^-126, 2^-25 of one of K 2^-100 max|x| + 2^-80 or more, and it is 0 by mistake only
// if subnormals were staged or the least product is below 2^-125.  A workgroup
// recomputes its tile with the fp32 matrix instruction (f32::gemm_tile, the
// same arithmetic as gemm_f32.hip) when some accumulator is infinite or NaN, or
// in those last two cases; the block-wide extremes they need are formed only
// when an output is below 2^-43 (or an |x| at least 2^40) and an operand below
// 2^-49.  A recomputed product costs both kernels.  us, the fp32 kernel's / this
// one's: 4096^3 with a row of 1e-18, one 2^41 per panel or a mask of -1e30
// 980 / 705-737, 8192 x 784 x 256 35 / 33, as for N(0, 1); recomputed, with a
// mask of -infinity or both operands scaled by 2^-40, 970 / 2250 and 35 / 90.
// Looking costs four VALU operations per two staged elements and two compares
// per output (8192 x 784 x 256 33.3 us against 32.6 without the search for the
// least; a class compare per element instead 36, and a second pass over the
// operands of tiles with a zero output 43 with zero rows).
//
// Structure (per workgroup, one 128 x 128 output tile, k-tiles of 32): eight
// waves in two groups of four, one wave of each per SIMD.  Each group owns the
// whole tile and takes every second k-tile through an LDS stage of its own
// (60 KiB: three k-contiguous bf16 planes per operand, [mn][40], so fragments
// are 16-byte reads), in two barrier-separated slots: split + store the
// k-tile from registers; then read fragments and issue its 96 MFMAs per wave,
// with the global loads of the group's next k-tile between them.  Group 1 is
// one slot behind, so on each SIMD one wave's MFMAs run beside the other's
// split and LDS stores.  At the end the groups exchange halves of their sums
// through LDS and add even + odd k-tiles.
//
// Measured: 4096^3 NN 707-745 us = 185-194 TFLOP/s against 980 = 140 on the fp32
// matrix path, 3072^3 390 against 454, 2048^3 92 against 131.  Bound by the
// MFMA slots: without the split and stores 2048^3 takes 85 us, without the
// global loads 83, without the MFMAs 53 (each measured with the loads issued
// ahead of the MFMAs, 95 in full).  Two independent four-wave workgroups per CU instead of two groups:
// 4096^3 687, but 2048^3 136 (one per CU).  256 x 256 tiles spill.
//
// Ragged sizes run at full speed: loads are always 16 bytes per lane (global
// loads need no more than 4-byte alignment), rows and column groups past the
// edge are loaded from the last whole ones inside, and only the last k-tile
// and the edge tiles run the code that shifts and zeroes them.
#include "gemm_f32_tile.hpp"

namespace cdx {
namespace {

using f32::KParams;

constexpr int PBK = 32;               // k-tile
constexpr int PSTRIDE = PBK + 8;      // LDS row stride (bf16)

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

// 128 x 128 tiles; two groups of four waves, each wave 64 x 64 (an LDS
// fragment feeds four blocks' MFMAs).
struct PTile {
    static constexpr int BM = 128, BN = 128, WM = 64, WN = 64, GROUP_M = 8;
    static constexpr int NTG = 256, NT = 512;   // threads per group, in all
    static constexpr int WAVES_N = BN / WN, FM = WM / 16, FN = WN / 16;
    using Fallback = f32::Cfg<128, 64, 16, 32, 32, 8, 1>;
};

// Three exact bf16 parts of two values, packed (a in the low half).
__device__ __forceinline__ void split3(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
    auto pk = [](float x, float y) {
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{x, y}, bf16x2_t));
    };
    auto lo = [](uint32_t v) { return __builtin_bit_cast(float, v << 16); };
    auto hi = [](uint32_t v) { return __builtin_bit_cast(float, v & 0xffff0000u); };
    h = pk(a, b);
    const float ra = a - lo(h), rb = b - hi(h);
    m = pk(ra, rb);
    l = pk(ra - lo(m), rb - hi(m));
}

// Magnitudes but 0 in order, from a float's bits; that of 2^e; and back.
__device__ __forceinline__ constexpr uint32_t least_code(uint32_t bits) { return (bits << 1) - 1u; }
__device__ __forceinline__ constexpr uint32_t least_code_exp2(int e) {
    return least_code((uint32_t)(e + 127) << 23);
}
__device__ __forceinline__ float least_value(uint32_t code) {   // (none seen: the largest)
    return code == 0xffffffffu ? 3.4028235e38f : __builtin_bit_cast(float, (code >> 1) + 1u);
}

// One operand's k-tile: BMN rows (m or n) x 32 k as 4 x 4 blocks (the walk of
// split::SplitLoader).  KC: k is the contiguous dimension in memory.  Byte
// offsets are from 16 bytes before the tile's first element of the k-tile, so
// that a block moved left at an edge keeps a non-negative 32-bit offset.
template <int BMN, bool KC>
struct PartLoader {
    static constexpr int NT = PTile::NTG, NB = (BMN / 4) * (PBK / 4);
    static constexpr int NV = NB / NT;
    static_assert(NB % NT == 0, "whole blocks per thread");
    f32x4u v[NV][4];       // KC: row q of the block, 4 k; else k row q, 4 mn
    uint32_t off[NV][4];

    __device__ __forceinline__ static void coords(int blk, int& bc, int& br) {
        if (KC) { bc = blk % (PBK / 4); br = blk / (PBK / 4); }
        else    { br = blk % (PBK / 4); bc = blk / (PBK / 4); }
    }
    // columns a block of columns c .. c + 3 moves left to lie within rem (>= 4
    // in all, so it may reach left of the tile by at most 3)
    __device__ __forceinline__ static int left(int c, int rem) {
        return c + 4 > rem ? c + 4 - rem : 0;
    }

    // mnrem: rows (columns) of the operand from the tile's first on, >= 1
    __device__ __forceinline__ void init(int64_t ld, int mnrem, int tid) {
#pragma unroll
        for (int b = 0; b < NV; ++b) {
            int bc, br;
            coords(tid + b * NT, bc, br);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = br * 4 + q;
                if (KC) off[b][q] = (uint32_t)((r < mnrem ? r : mnrem - 1) * ld + bc * 4 + 4) * 4u;
                else    off[b][q] = (uint32_t)(r * ld + (bc * 4 - left(bc * 4, mnrem)) + 4) * 4u;
            }
        }
    }
    __device__ __forceinline__ void load(const char* base) {
#pragma unroll
        for (int b = 0; b < NV; ++b)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                v[b][q] = *(const __attribute__((address_space(1))) f32x4u*)(base + off[b][q]);
    }
    // The last k-tile, of krem < 32 k: from addresses moved back inside.
    __device__ __forceinline__ void load_tail(const char* base, int64_t ld, int krem, int tid) {
#pragma unroll
        for (int b = 0; b < NV; ++b) {
            int bc, br;
            coords(tid + b * NT, bc, br);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = br * 4 + q;
                const uint32_t back = KC ? (uint32_t)left(bc * 4, krem) * 4u
                                         : (r < krem ? 0u : (uint32_t)((r - krem + 1) * ld) * 4u);
                v[b][q] = *(const __attribute__((address_space(1))) f32x4u*)(base + (off[b][q] - back));
            }
        }
    }
    // Element i of a 16-byte run moved s to the left is its element i + s.
    __device__ __forceinline__ static void shift_left(f32x4u& t, int s) {
        const f32x4u u = t;
        t.x = s == 0 ? u.x : s == 1 ? u.y : s == 2 ? u.z : u.w;
        t.y = s == 0 ? u.y : s == 1 ? u.z : u.w;
        t.z = s == 0 ? u.z : u.w;
    }
    // Edge and tail blocks: undoes the moves, sets the ones row / column
    // (`one`, relative to the tile; -1 none) and zeroes k >= krem (32: none).
    __device__ __forceinline__ void fix(int mnrem, int krem, int one, int tid) {
#pragma unroll
        for (int b = 0; b < NV; ++b) {
            int bc, br;
            coords(tid + b * NT, bc, br);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                f32x4u& t = v[b][q];
                shift_left(t, left(bc * 4, KC ? krem : mnrem));
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int mn = KC ? br * 4 + q : bc * 4 + i, k = KC ? bc * 4 + i : br * 4 + q;
                    if (mn == one) t[i] = 1.0f;
                    if (k >= krem) t[i] = 0.0f;
                }
            }
        }
    }
    // Splits into the three planes at s ([mn][PSTRIDE], `plane` apart);
    // amax: the largest magnitude seen; least: the smallest but 0, as
    // least_code() (0's wraps round to the largest).
    __device__ __forceinline__ void store(unsigned short* s, int plane, float& amax,
                                          uint32_t& least, int tid) const {
#pragma unroll
        for (int b = 0; b < NV; ++b) {
            int bc, br;
            coords(tid + b * NT, bc, br);
#pragma unroll
            for (int r = 0; r < 4; ++r) {   // mn within the block
                f32x4u x;                   // 4 consecutive k at this mn
                if (KC) x = v[b][r];
                else x = f32x4u{v[b][0][r], v[b][1][r], v[b][2][r], v[b][3][r]};
                asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(amax) : "v"(x.x), "v"(x.y));
                asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(amax) : "v"(x.z), "v"(x.w));
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t u = least_code(__builtin_bit_cast(uint32_t, x[i]));
                    least = u < least ? u : least;
                }
                uint2 h, m, l;
                split3(x.x, x.y, h.x, m.x, l.x);
                split3(x.z, x.w, h.y, m.y, l.y);
                unsigned short* d = s + ((KC ? br : bc) * 4 + r) * PSTRIDE + (KC ? bc : br) * 4;
                *reinterpret_cast<uint2*>(d) = h;
                *reinterpret_cast<uint2*>(d + plane) = m;
                *reinterpret_cast<uint2*>(d + 2 * plane) = l;
            }
        }
    }
};

template <int OPA, int OPB>
__global__ __launch_bounds__(PTile::NT)
void gemm_parts_kernel(KParams p) {
    using CF = PTile;
    constexpr int BM = CF::BM, BN = CF::BN, FM = CF::FM, FN = CF::FN;
    constexpr bool KCA = OPA == CDX_OP_N, KCB = OPB == CDX_OP_T;
    constexpr int A_PLANE = BM * PSTRIDE, B_PLANE = BN * PSTRIDE;
    constexpr int STAGE = 3 * (A_PLANE + B_PLANE);   // bf16
    using Fallback = CF::Fallback;
    __shared__ __attribute__((aligned(16))) unsigned short lds[2 * STAGE];
    __shared__ int redo, small_out, small_in;
    __shared__ uint32_t ext[3];   // least of A, of B; largest of both (bits)
    static_assert(2 * STAGE * 2 >= 8 * 8 * 64 * 16, "the hand-over needs 64 KiB");
    static_assert(2 * STAGE * 2 >= f32::Geo<Fallback, OPA, OPB>::LDS_FLOATS * 4, "fallback tile");

    const int lane = threadIdx.x & 63, tid = threadIdx.x & (CF::NTG - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = wave >> 2, w = wave & 3;
    const int l16 = lane & 15, lq = lane >> 4;
    const int wm0 = (w / CF::WAVES_N) * CF::WM, wn0 = (w % CF::WAVES_N) * CF::WN;
    unsigned short* sA = lds + grp * STAGE;   // the group's stage
    unsigned short* sB = sA + 3 * A_PLANE;

    int tm, tn;
    f32::tile_of_block((int)ceil_div(p.M, BM), (int)ceil_div(p.N, BN), CF::GROUP_M, tm, tn);
    const int64_t bm = (int64_t)tm * BM, bn = (int64_t)tn * BN;
    if (gridDim.y > 1) {   // split-K slice (plain [M, N] partial)
        const int64_t k0 = (int64_t)blockIdx.y * p.k_chunk;
        p.A += KCA ? k0 : k0 * p.lda;
        p.B += KCB ? k0 : k0 * p.ldb;
        p.K = p.K - k0 < p.k_chunk ? p.K - k0 : p.k_chunk;
        p.C += (int64_t)blockIdx.y * p.M * p.N;
    }
    if (gridDim.z > 1) {
        p.A += (int64_t)blockIdx.z * p.sa;
        p.B += (int64_t)blockIdx.z * p.sb;
        p.C += (int64_t)blockIdx.z * p.sc;
    }

    // op(B)'s own columns end at p.nb; a tile that holds the ones column only
    // loads (and discards) the last four
    const int64_t bo = bn < p.nb ? bn : p.nb - 4;
    const int arem = (int)(p.M - bm < BM ? p.M - bm : BM), brem = (int)(p.nb - bo < BN ? p.nb - bo : BN);
    const int one = p.ones >= bn && p.ones < bn + BN ? (int)(p.ones - bn) : -1;
    const bool edge_a = !KCA && arem < BM, edge_b = (!KCB && brem < BN) || one >= 0;
    PartLoader<BM, KCA> la;
    PartLoader<BN, KCB> lb;
    la.init(p.lda, arem, tid);
    lb.init(p.ldb, brem, tid);
    const char* pa = reinterpret_cast<const char*>(p.A + (KCA ? bm * p.lda : bm)) - 16;
    const char* pb = reinterpret_cast<const char*>(p.B + (KCB ? bo * p.ldb : bo)) - 16;
    const int64_t step_a = (KCA ? (int64_t)PBK : PBK * p.lda) * 4;
    const int64_t step_b = (KCB ? (int64_t)PBK : PBK * p.ldb) * 4;

    const int64_t nk = ceil_div(p.K, PBK);
    const int krem = (int)(p.K - (nk - 1) * PBK);   // 1..32 k in the last k-tile
    auto load_a = [&](int64_t t) {
        if (t + 1 < nk || krem == PBK) la.load(pa + t * step_a);
        else if (t < nk) la.load_tail(pa + t * step_a, p.lda, krem, tid);
    };
    auto load_b = [&](int64_t t) {
        if (t + 1 < nk || krem == PBK) lb.load(pb + t * step_b);
        else if (t < nk) lb.load_tail(pb + t * step_b, p.ldb, krem, tid);
    };
    float amax = 0.0f;
    uint32_t least_a = 0xffffffffu, least_b = 0xffffffffu;
    auto store = [&](int64_t t) {
        const int kr = t + 1 < nk ? PBK : krem;
        if (edge_a || kr < PBK) la.fix(arem, kr, -1, tid);
        la.store(sA, A_PLANE, amax, least_a, tid);
        if (edge_b || kr < PBK) lb.fix(brem, kr, one, tid);
        lb.store(sB, B_PLANE, amax, least_b, tid);
    };

    floatx4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    auto frag = [&](const unsigned short* s, int row) {
        return *reinterpret_cast<const bf16x8*>(s + (row + l16) * PSTRIDE + 8 * lq);
    };
    // The fragments are read in the order of use; the next row's fragments,
    // the additions of the previous row's sums and the global loads of a later
    // k-tile (issue_a, issue_b) go between the MFMAs, pinned there: issued
    // together, either holds up the MFMAs behind it.
    auto pin = []() { __builtin_amdgcn_sched_barrier(0); };
    auto compute = [&](auto&& issue_a, auto&& issue_b) {
        bf16x8 fa[2][3], fb[FN][3];
        auto read_a = [&](int i, int pl) { fa[i & 1][pl] = frag(sA + pl * A_PLANE, wm0 + i * 16); };
        auto read_b = [&](int pl) {
#pragma unroll
            for (int j = 0; j < FN; ++j) fb[j][pl] = frag(sB + pl * B_PLANE, wn0 + j * 16);
        };
        read_a(0, 2);
        read_b(0);
        read_a(0, 0);
        read_b(2);
        read_a(0, 1);
        read_b(1);
        // small terms first: l h, h l, m m, m h, h m, then h h
        constexpr int TA[6] = {2, 0, 1, 1, 0, 0}, TB[6] = {0, 2, 1, 0, 1, 0};
        floatx4 sum[2][FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) {
#pragma unroll
            for (int t = 0; t < 6; ++t) {
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    sum[i & 1][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        fa[i & 1][TA[t]], fb[j][TB[t]],
                        t == 0 ? floatx4{0.f, 0.f, 0.f, 0.f} : sum[i & 1][j], 0, 0, 0);
                pin();
                if (i > 0 && t >= 1 && t <= FN) acc[i - 1][t - 1] += sum[(i - 1) & 1][t - 1];
                if (i + 1 < FM && t == 2) read_a(i + 1, 2);
                if (i + 1 < FM && t == 3) read_a(i + 1, 0);
                if (i + 1 < FM && t == 4) read_a(i + 1, 1);
                if (i == 0 && t == 5) issue_a();
                if (i == 1 && t == 5) issue_b();
                pin();
            }
        }
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[FM - 1][j] += sum[(FM - 1) & 1][j];
    };
    auto slot = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };

    // group g takes the k-tiles g, g + 2, ...; both run the barriers of the
    // longer list, group 1 one slot behind
    if (threadIdx.x == 0) {
        redo = small_out = small_in = 0;
        ext[0] = ext[1] = 0xffffffffu;
        ext[2] = 0u;
    }
    const int64_t slots = (nk + 1) / 2;
    if (grp < nk) {
        load_a(grp);
        load_b(grp);
    }
    if (grp == 1) slot();
    for (int64_t j = 0; j < slots; ++j) {
        const int64_t t = 2 * j + grp;
        if (t < nk) store(t);
        slot();
        if (t < nk) {
            __builtin_amdgcn_s_setprio(1);
            compute([&]() { if (t + 2 < nk) load_a(t + 2); }, [&]() { if (t + 2 < nk) load_b(t + 2); });
            __builtin_amdgcn_s_setprio(0);
        }
        slot();
    }
    if (grp == 0) slot();

    // hand-over: group 0 keeps rows 0-31 of each wave's 64 x 64 and gives rows
    // 32-63, group 1 the opposite; even k-tiles + odd ones, in that order
    floatx4* red = reinterpret_cast<floatx4*>(lds);
    floatx4 res[2][FN];
    if (grp == 0) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) red[((w * 2 + 1) * 8 + i * FN + j) * 64 + lane] = acc[2 + i][j];
    } else {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) red[((w * 2 + 0) * 8 + i * FN + j) * 64 + lane] = acc[i][j];
    }
    __syncthreads();
    if (grp == 0) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
                res[i][j] = acc[i][j] + red[((w * 2 + 0) * 8 + i * FN + j) * 64 + lane];
    } else {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
                res[i][j] = red[((w * 2 + 1) * 8 + i * FN + j) * 64 + lane] + acc[2 + i][j];
    }

    // Recompute? (see Range above.)  Values that are lost need a small operand
    // and show in a small output, or one beside operands that are very large.
    auto any_output = [&](auto&& of) {
        bool any = false;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) any |= of(__builtin_fabsf(res[i][j][e]));
        return any;
    };
    if (any_output([](float c) { return !(c <= 3.4028235e38f); })) redo = 1;   // NaN too
    if (any_output([](float c) { return c < 0x1p-43f; }) || !(amax < 0x1p40f)) small_out = 1;
    if (least_a < least_code_exp2(-49) || least_b < least_code_exp2(-49)) small_in = 1;
    __syncthreads();
    if (!redo && small_out && small_in) {   // (uniform)
        uint32_t top = __builtin_bit_cast(uint32_t, amax);
        for (int d = 32; d > 0; d >>= 1) {
            const uint32_t a = __shfl_xor(least_a, d), b = __shfl_xor(least_b, d), t = __shfl_xor(top, d);
            least_a = a < least_a ? a : least_a;
            least_b = b < least_b ? b : least_b;
            top = t > top ? t : top;
        }
        if (lane == 0) {
            atomicMin(&ext[0], least_a);
            atomicMin(&ext[1], least_b);
            atomicMax(&ext[2], top);
        }
        __syncthreads();
        const uint32_t lo = ext[0] < ext[1] ? ext[0] : ext[1];
        const float least_product = least_value(ext[0]) * least_value(ext[1]);
        if (lo < least_code_exp2(-110) || least_product < 0x1p-98f) {
            const float bound = 0x1p-80f + 0x1p-100f * (float)p.K * __builtin_bit_cast(float, ext[2]);
            const bool zeros = lo < least_code_exp2(-126) || least_product < 0x1p-125f;
            if (any_output([&](float c) { return c == 0.0f ? zeros : c < bound; })) redo = 1;
        }
        __syncthreads();
    }
    if (redo) {   // (uniform) the fp32 matrix path, a smaller tile at a time
        constexpr int TN = BN / Fallback::BN;
#pragma unroll 1
        for (int s = 0; s < BM / Fallback::BM * TN; ++s) {
            const int64_t m = bm + s / TN * Fallback::BM, n = bn + s % TN * Fallback::BN;
            if (m < p.M && n < p.N)
                f32::gemm_tile<Fallback, OPA, OPB, f32::kLoadChecked, false, false>(
                    p, m, n, reinterpret_cast<float*>(lds));
            __syncthreads();
        }
        return;
    }
    const EpiArgs epi{p.C, p.ldc, p.M, p.N, 0, 0, p.bias, p.bias_mode, p.epilogue,
                      p.aux, p.ldaux, p.colsum, p.nb};
    const int rm0 = wm0 + 32 * grp;
    if (bm + BM <= p.M && bn + BN <= p.nb)
        write_acc<2, FN, false, false>(res, epi, bm + rm0, bn + wn0, lane);
    else
        write_acc<2, FN, true, false>(res, epi, bm + rm0, bn + wn0, lane);
}

// Tiles of the product itself, without the ones column: a call that also
// forms the row sums then takes the same tiles and k-slices.
int64_t own_tiles(const GemmArgs& g) {
    const int64_t nb = g.ones_col >= 0 ? g.ones_col : g.N;
    return ceil_div(g.M, PTile::BM) * ceil_div(nb, PTile::BN);
}

// k-slices of a product that does not fill the GPU with its tiles, where K is
// long enough to split (splitk_applies, on these tiles or the tiled kernel's
// slices): the count whose rounds of one workgroup per CU, each its k-tiles
// and about four more for filling the pipeline and the epilogue, plus the pass
// over the partials, are shortest.  256 x 785 x 8192, 14 tiles: 18 slices, one
// round: 38 us with the reduction against 47 in the 29 slices, two rounds, of the
// tiled kernel's policy (made for workgroups of which two or three share a CU).
struct Slices {
    int n;
    int64_t chunk;
};

Slices slices_of(const GemmArgs& g) {
    const int64_t nb = g.ones_col >= 0 ? g.ones_col : g.N, t = own_tiles(g);
    if (g.batch > 1 || !(splitk_applies(t, g.K) ||
                         splitk_applies(ceil_div(g.M, 128) * ceil_div(nb, 64), g.K)))
        return {1, g.K};
    const int64_t nk = ceil_div(g.K, PBK);
    Slices best{1, g.K};
    double least = 0.0;
    for (int64_t s = 1; s <= nk / 8 && s <= 256; ++s) {
        const int64_t per = ceil_div(nk, s), n = ceil_div(nk, per);
        // (a k-tile takes about 0.75 us; partials move at about 4 TB/s)
        const double cost = (double)ceil_div(t * n, 256) * (double)(per + 4) +
                            (n > 1 ? 5.0 + (double)n * (double)(g.M * nb) * 1.3e-6 : 0.0);
        if (s == 1 || cost < least) {
            least = cost;
            best = {(int)n, n > 1 ? per * PBK : g.K};
        }
    }
    return best;
}

}  // namespace

namespace {

// Unsliced products: whether this kernel's rounds of one workgroup per CU beat
// the tiled fp32 kernel's rounds of 64 x 64 tiles.  Both costs are in us, from
// fits to whole tiles with 16-byte rows; A transposed costs this kernel more,
// ragged sizes and rows cost the tiled one more.  Within an eighth this kernel
// is taken, for its smaller error (of which 64 k show little).  Tiled / this, us:
//   4096 x 4096 x 48 NN   37 / 57    2048 x 2304 x 64 NN     11 / 18
//   2048 x 2048 x 64 NN   10 / 11    2048 x 2304 x 512 NN    46 / 52
//   2048 x 2048 x 128 NN  14 / 14    2048 x 2304 x 2048 NN  167 / 179
//   3072 x 3072 x 64 NN   18 / 26    2048 x 2304 x 2048 TN  166 / 210
//   3072 x 3072 x 512 NN  80 / 79    2999 x 1501 x 2048 TN  291 / 200
//   8192 x 784 x 256 NN   35 / 34    2501 x 2503 x 128 NN    33 / 27
// (the slow ones: a pipeline's filling over a k-tile or four, and a second
// round of 32 workgroups)
bool beats_tiled(const GemmArgs& g, int64_t tiles) {
    const KParams kp = f32::kparams_of(g, g.K);
    const int64_t nb = g.ones_col >= 0 ? g.ones_col : g.N;
    const double rounds = (double)ceil_div(tiles * g.batch, 256);
    const double rounds64 = (double)ceil_div(ceil_div(g.M, 64) * ceil_div(nb, 64) * g.batch, 256);
    const bool whole = g.M % 64 == 0 && nb % 64 == 0;
    const double slow = !kp.vec_a && !kp.vec_b ? 1.9 : !kp.vec_a || !kp.vec_b ? 1.45
                        : g.K % 16 != 0 ? 1.25 : whole ? 1.0 : 1.15;
    const double parts = 3.0 + rounds * (5.0 + (g.opA == CDX_OP_T ? 1.5 : 1.25) * (double)ceil_div(g.K, PBK));
    return parts <= (g.K > 64 ? 1.12 : 1.0) * (6.0 + 0.5 * slow * rounds64 * (double)g.K / PBK);
}

}  // namespace

// Which products: those with a 128 x 128 tile for nearly every CU (2048^3 92
// against 131 us on the fp32 matrix path, 5079 x 896 x 920 NT 88 against 93)
// unless beats_tiled() says otherwise, or with enough k-slices of such tiles (256 x
// 785 x 8192 TN 38 against 49; 2539 x 704 x 2624 NT 76 against 124; 512 x 1024
// x 8192 TN 67 against 181; 64 workgroups, 256 x 257 x 4096 TN, 24 against 22).
// With fewer tiles and a short K the smaller fp32 tiles win: 8192 x 256 x 784
// NT (128 tiles) 38 against 32, 1536^3 69 against 67, 1024^3 48 against 26.
// Tiles may be padded by up to 40 %.  Operand panels are addressed with 32-bit
// offsets.
bool gemm_parts_ok(const GemmArgs& g) {
    const int64_t nb = g.ones_col >= 0 ? g.ones_col : g.N, lim = int64_t(1) << 22;
    if (g.n_split > 0 || g.blocked_sum || g.M < 64 || nb < 64 || g.K <= 16 || g.K > 65536 ||
        g.lda >= lim || g.ldb >= lim)
        return false;
    const int64_t tiles = own_tiles(g);
    if (tiles > INT32_MAX / 2 || tiles * (PTile::BM * PTile::BN) > g.M * nb / 5 * 7) return false;
    if (tiles >= 240) return beats_tiled(g, tiles);
    const int n = slices_of(g).n;
    return n > 1 && tiles * n >= 160;
}

size_t gemm_parts_workspace(const GemmArgs& g) {
    const int n = slices_of(g).n;
    return n > 1 ? (size_t)n * (size_t)g.M * (size_t)g.N * sizeof(float) : 0;
}

int launch_gemm_parts(const GemmArgs& g0, hipStream_t stream) {
    const int64_t tiles = ceil_div(g0.M, PTile::BM) * ceil_div(g0.N, PTile::BN);
    if (tiles > INT32_MAX) return set_error(CDX_ERR_UNSUPPORTED, "gemm: too many tiles");
    if (g0.batch < 1 || g0.batch > 65535) return set_error(CDX_ERR_UNSUPPORTED, "gemm: batch out of range");
    const Slices sl = slices_of(g0);
    return with_slices(g0, sl.n, sl.chunk, stream,
                       [&](const GemmArgs& g, int splits, int64_t k_chunk) {
        const KParams kp = f32::kparams_of(g, k_chunk);
        const dim3 grid((unsigned)tiles, (unsigned)splits, (unsigned)g.batch), block(PTile::NT);
        if (g.opA == CDX_OP_N && g.opB == CDX_OP_N)
            hipLaunchKernelGGL((gemm_parts_kernel<CDX_OP_N, CDX_OP_N>), grid, block, 0, stream, kp);
        else if (g.opA == CDX_OP_N)
            hipLaunchKernelGGL((gemm_parts_kernel<CDX_OP_N, CDX_OP_T>), grid, block, 0, stream, kp);
        else if (g.opB == CDX_OP_N)
            hipLaunchKernelGGL((gemm_parts_kernel<CDX_OP_T, CDX_OP_N>), grid, block, 0, stream, kp);
        else
            hipLaunchKernelGGL((gemm_parts_kernel<CDX_OP_T, CDX_OP_T>), grid, block, 0, stream, kp);
        return hip_error(hipGetLastError(), "gemm_parts_kernel launch");
    });
}

}  // namespace cdx
