// One workgroup's tile of the FP32 (v_mfma_f32_16x16x4_f32) GEMM: loaders,
// LDS geometry and the k-loop, shared by the FP32 kernels (gemm_f32.hip, see
// there for the structure) and by the three-part split kernel, which
// recomputes a tile this way when its operands are outside the range in
// which its parts are exact (gemm_parts.hip).
#pragma once

#include "cdx_internal.hpp"

namespace cdx {
namespace f32 {

constexpr int kLoadAlignedVec = 0;  // every tile in bounds, 16-byte loads
constexpr int kLoadChecked = 1;     // bounds-checked; 16-byte loads where whole and the
                                    // operand allows them (per-operand flag), else scalar

struct KParams {
    const float* A; const float* B; float* C; const float* bias;
    int64_t M, N, K, lda, ldb, ldc, n_split, ldc_split;
    int bias_mode, epilogue;
    int64_t k_chunk;    // split-K: k-range per blockIdx.y slice (gridDim.y > 1)
    int64_t sa, sb, sc; // batch strides (elements) for blockIdx.z
    int64_t batch;      // gridDim.z
    int vec_a, vec_b;   // kLoadChecked: operand base, ld and batch stride allow 16-byte loads
    const float* aux;   // activation-backward epilogues: aux [M, N], leading dim ldaux
    int64_t ldaux;
    // op(B)'s own column count and the virtual ones column: with ones >= 0
    // (= nb) op(B)(k, nb) reads as 1 (checked loads only) and the kernel's N
    // is nb + 1; colsum receives that column's results.
    int64_t nb, ones;
    float* colsum;
    int interior;   // kLoadChecked: whole tiles may take the unchecked path
};

// Loads a ROWS x COLS tile (COLS contiguous in memory) starting at (r0, c0)
// of a matrix with leading dimension ld and extent (rmax, cmax) into
// registers; NT threads, each holding NV float4.
template <int ROWS, int COLS, int NT, int MODE>
struct TileLoader {
    static constexpr int C4 = COLS / 4;
    static constexpr int TOTAL = ROWS * C4;           // float4 slots in the tile
    static constexpr int NV = (TOTAL + NT - 1) / NT;
    static constexpr bool PARTIAL = TOTAL % NT != 0;  // last pass: some threads idle
    float4 v[NV];

    // ones_row / ones_col >= 0: that row / column (one past the matrix)
    // reads as 1 within the other dimension's bounds (checked mode only)
    __device__ __forceinline__ void load(const float* __restrict__ X, int64_t ld,
                                         int64_t r0, int64_t c0, int64_t rmax,
                                         int64_t cmax, bool vec, int tid,
                                         int64_t ones_row = -1, int64_t ones_col = -1) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            int idx = tid + i * NT;
            if (PARTIAL && idx >= TOTAL) break;
            int r = idx / C4, c = (idx % C4) * 4;
            int64_t gr = r0 + r, gc = c0 + c;
            const float* p = X + gr * ld + gc;
            if (MODE == kLoadAlignedVec) {
                v[i] = *reinterpret_cast<const float4*>(p);
            } else if (vec && gr < rmax && gc + 3 < cmax) {
                v[i] = *reinterpret_cast<const float4*>(p);
            } else {
                bool rok = gr < rmax;
                v[i].x = (rok && gc + 0 < cmax) ? p[0] : 0.0f;
                v[i].y = (rok && gc + 1 < cmax) ? p[1] : 0.0f;
                v[i].z = (rok && gc + 2 < cmax) ? p[2] : 0.0f;
                v[i].w = (rok && gc + 3 < cmax) ? p[3] : 0.0f;
                if (ones_col >= 0 && rok) {
                    if (gc + 0 == ones_col) v[i].x = 1.0f;
                    if (gc + 1 == ones_col) v[i].y = 1.0f;
                    if (gc + 2 == ones_col) v[i].z = 1.0f;
                    if (gc + 3 == ones_col) v[i].w = 1.0f;
                }
                if (ones_row >= 0 && gr == ones_row) {
                    v[i].x = gc + 0 < cmax ? 1.0f : 0.0f;
                    v[i].y = gc + 1 < cmax ? 1.0f : 0.0f;
                    v[i].z = gc + 2 < cmax ? 1.0f : 0.0f;
                    v[i].w = gc + 3 < cmax ? 1.0f : 0.0f;
                }
            }
        }
    }

    template <int LDS_STRIDE>
    __device__ __forceinline__ void store(float* __restrict__ s, int tid) const {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            int idx = tid + i * NT;
            if (PARTIAL && idx >= TOTAL) break;
            int r = idx / C4, c = (idx % C4) * 4;
            *reinterpret_cast<float4*>(s + r * LDS_STRIDE + c) = v[i];
        }
    }
};

// PIPE: 1 = one register staging set; 2 = two sets (tile k+2 loads while
// tile k+1 is written to LDS).
template <int BM_, int BN_, int BK_, int WM_, int WN_, int GROUP_M_, int PIPE_ = 1>
struct Cfg {
    static constexpr int BM = BM_, BN = BN_, BK = BK_, WM = WM_, WN = WN_;
    static constexpr int GROUP_M = GROUP_M_;
    static constexpr int PIPE = PIPE_;
    static constexpr int WAVES_M = BM / WM, WAVES_N = BN / WN;
    static constexpr int NT = WAVES_M * WAVES_N * 64;
    static constexpr int FM = WM / 16, FN = WN / 16;
};

// Maps the linear workgroup id to an output tile (tm, tn): XCD-contiguous
// runs, then GROUP_M-row groups within the run.
__device__ __forceinline__ void tile_of_block(int tiles_m, int tiles_n, int group_m,
                                              int& tm, int& tn) {
    int nb = gridDim.x;
    int bid = blockIdx.x;
    if ((nb & 7) == 0) bid = (bid & 7) * (nb >> 3) + (bid >> 3);
    int per_group = group_m * tiles_n;
    int g = bid / per_group;
    int first_m = g * group_m;
    int gsize = tiles_m - first_m < group_m ? tiles_m - first_m : group_m;
    int in_g = bid - g * per_group;
    tm = first_m + in_g % gsize;
    tn = in_g / gsize;
}

// Reads V consecutive floats of one LDS row (V = 1, 2 or 4: one 4-, 8- or
// 16-byte read) into fragment slots f[blk0 .. blk0 + V - 1][j].
template <int V, int F>
__device__ __forceinline__ void read_rows(const float* p, float (&f)[F][4], int blk0, int j) {
    if constexpr (V == 4) {
        const float4 t = *reinterpret_cast<const float4*>(p);
        f[blk0][j] = t.x; f[blk0 + 1][j] = t.y; f[blk0 + 2][j] = t.z; f[blk0 + 3][j] = t.w;
    } else if constexpr (V == 2) {
        const float2 t = *reinterpret_cast<const float2*>(p);
        f[blk0][j] = t.x; f[blk0 + 1][j] = t.y;
    } else {
        f[blk0][j] = *p;
    }
}

// LDS geometry and fragment-read widths of one configuration.
//  * m/n-contiguous operands are read V consecutive rows (columns) per lane
//    with one LDS read, feeding V MFMAs whose blocks are interleaved
//    (blk_pos); k-contiguous operands keep the plain layout.  (Measured on
//    MI355X: 16-byte reads gain 1-4 %; 8-byte reads gain only on A when B is
//    read 16 bytes at a time too -- 2048^3 TN 141 -> 132 us -- and lose
//    elsewhere: 2048^3 TT 132 -> 138 us, 8192 x 784 x 256 NN on 64 x 64
//    tiles 44 -> 45 us.)
//  * k-contiguous operands are [mn][BK+4], m/n-contiguous ones [BK][mn+4]:
//    with 4-byte reads, lane groups lq = 0..3 read rows 4 apart, 16 banks
//    apart with the pad; wider reads take one contiguous row segment per
//    16 lanes.
template <class CF, int OPA, int OPB>
struct Geo {
    static constexpr int BM = CF::BM, BN = CF::BN, BK = CF::BK;
    static constexpr int VB = OPB == CDX_OP_T ? 1 : (CF::FN % 4 == 0 ? 4 : 1);
    static constexpr int VA = OPA == CDX_OP_N ? 1 : (CF::FM % 4 == 0 ? 4 : CF::FM % 2 == 0 && VB == 4 ? 2 : 1);
    static constexpr int A_STRIDE = OPA == CDX_OP_N ? BK + 4 : BM + 4;
    static constexpr int A_ELEMS = OPA == CDX_OP_N ? BM * A_STRIDE : BK * A_STRIDE;
    static constexpr int B_STRIDE = OPB == CDX_OP_N ? BN + 4 : BK + 4;
    static constexpr int B_ELEMS = OPB == CDX_OP_N ? BK * B_STRIDE : BN * B_STRIDE;
    static constexpr int LDS_FLOATS = 2 * (A_ELEMS + B_ELEMS);
};

// One workgroup's output tile (top-left (bm, bn)) over the k-range of p.
// BLK: two-level k sum -- each pair of k-tiles (32 k) is summed from zero in
// `part`, then added to `acc` (a rounding chain of ~32 + K/32 additions).
template <class CF, int OPA, int OPB, int MODE, bool SPLITN, bool BLK>
__device__ __forceinline__ void gemm_tile(const KParams& p, int64_t bm, int64_t bn, float* lds) {
    using G = Geo<CF, OPA, OPB>;
    constexpr int BK = CF::BK;
    constexpr int NT = CF::NT, FM = CF::FM, FN = CF::FN;
    constexpr int VA = G::VA, VB = G::VB;
    constexpr int A_STRIDE = G::A_STRIDE, A_ELEMS = G::A_ELEMS;
    constexpr int B_STRIDE = G::B_STRIDE, B_ELEMS = G::B_ELEMS;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm0 = (wave / CF::WAVES_N) * CF::WM;
    const int wn0 = (wave % CF::WAVES_N) * CF::WN;
    const int l16 = lane & 15;
    const int lq = lane >> 4;   // 0..3

    constexpr int BM = CF::BM, BN = CF::BN;
// Global tile loaders in memory orientation.
    using LA = TileLoader<OPA == CDX_OP_N ? BM : BK, OPA == CDX_OP_N ? BK : BM, NT, MODE>;
    using LB = TileLoader<OPB == CDX_OP_N ? BK : BN, OPB == CDX_OP_N ? BN : BK, NT, MODE>;
    LA la;
    LB lb;

    auto load_into = [&](LA& a, LB& b, int64_t k0) {
        if (OPA == CDX_OP_N) a.load(p.A, p.lda, bm, k0, p.M, p.K, p.vec_a, tid);
        else                 a.load(p.A, p.lda, k0, bm, p.K, p.M, p.vec_a, tid);
        // op(B)'s own columns, plus the ones column when p.ones >= 0
        if (OPB == CDX_OP_N) b.load(p.B, p.ldb, k0, bn, p.K, p.nb, p.vec_b, tid, -1, p.ones);
        else                 b.load(p.B, p.ldb, bn, k0, p.nb, p.K, p.vec_b, tid, p.ones, -1);
    };
    auto store_from = [&](const LA& a, const LB& b, int buf) {
        float* sA = lds + buf * (A_ELEMS + B_ELEMS);
        float* sB = sA + A_ELEMS;
        a.template store<A_STRIDE>(sA, tid);
        b.template store<B_STRIDE>(sB, tid);
    };

    floatx4 acc[FM][FN], part[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
            part[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    floatx4 (&tgt)[FM][FN] = BLK ? part : acc;
    // BLK: fold the partial sum into the total and restart it
    auto flush = [&]() {
        if (!BLK) return;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                acc[i][j] += part[i][j];
                part[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
            }
    };

    // MFMAs over the k-tile held in LDS stage `buf`, into `tgt`
    auto compute = [&](int buf) {
        const float* sA = lds + buf * (A_ELEMS + B_ELEMS);
        const float* sB = sA + A_ELEMS;
#pragma unroll
        for (int kk = 0; kk < BK; kk += 16) {
            float a[FM][4], b[FN][4];
            if constexpr (OPA == CDX_OP_N) {
#pragma unroll
                for (int i = 0; i < FM; ++i) {
                    const int m = wm0 + i * 16 + l16;
                    float4 t = *reinterpret_cast<const float4*>(sA + m * A_STRIDE + kk + 4 * lq);
                    a[i][0] = t.x; a[i][1] = t.y; a[i][2] = t.z; a[i][3] = t.w;
                }
            } else {
#pragma unroll
                for (int g = 0; g < FM / VA; ++g)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        read_rows<VA>(sA + (kk + 4 * lq + j) * A_STRIDE + wm0 + 16 * VA * g + VA * l16,
                                      a, g * VA, j);
            }
            if constexpr (OPB == CDX_OP_T) {
#pragma unroll
                for (int jn = 0; jn < FN; ++jn) {
                    const int n = wn0 + jn * 16 + l16;
                    float4 t = *reinterpret_cast<const float4*>(sB + n * B_STRIDE + kk + 4 * lq);
                    b[jn][0] = t.x; b[jn][1] = t.y; b[jn][2] = t.z; b[jn][3] = t.w;
                }
            } else {
#pragma unroll
                for (int g = 0; g < FN / VB; ++g)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        read_rows<VB>(sB + (kk + 4 * lq + j) * B_STRIDE + wn0 + 16 * VB * g + VB * l16,
                                      b, g * VB, j);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int jn = 0; jn < FN; ++jn)
                        tgt[i][jn] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][j], b[jn][j],
                                                                         tgt[i][jn], 0, 0, 0);
        }
    };

    const int64_t nk = ceil_div(p.K, BK);
    if (CF::PIPE == 2 && nk >= 2) {
        // Two register staging sets: tile k+2 is loaded while tile k+1 is
        // written to LDS from the set loaded one iteration earlier, so the
        // LDS stores never wait on global memory.
        LA la1;
        LB lb1;
        load_into(la, lb, 0);
        load_into(la1, lb1, BK);
        store_from(la, lb, 0);
        __syncthreads();
        int64_t kt = 0;
        // loop invariant (kt even): stage 0 holds tile kt, set 1 tile kt+1
        for (; kt + 3 < nk; kt += 2) {
            load_into(la, lb, (kt + 2) * BK);
            compute(0);
            store_from(la1, lb1, 1);
            __syncthreads();
            load_into(la1, lb1, (kt + 3) * BK);
            compute(1);
            store_from(la, lb, 0);
            __syncthreads();
            flush();
        }
        if (kt + 2 < nk) {            // three tiles left
            load_into(la, lb, (kt + 2) * BK);
            compute(0);
            store_from(la1, lb1, 1);
            __syncthreads();
            compute(1);
            store_from(la, lb, 0);
            __syncthreads();
            flush();
            compute(0);
        } else {                      // two tiles left
            compute(0);
            store_from(la1, lb1, 1);
            __syncthreads();
            compute(1);
        }
        flush();
    } else {
        // One staging set: tile k+1 is in flight during the MFMAs of tile k.
        load_into(la, lb, 0);
        store_from(la, lb, 0);
        __syncthreads();
        for (int64_t kt = 0; kt < nk; ++kt) {
            const int buf = (int)(kt & 1);
            const bool has_next = kt + 1 < nk;
            if (has_next) load_into(la, lb, (kt + 1) * BK);
            compute(buf);
            if (has_next) store_from(la, lb, buf ^ 1);
            __syncthreads();
            if (kt & 1) flush();
        }
        flush();
    }

    // epilogue: bias, activation and the output map, straight from the
    // accumulators
    const EpiArgs epi{p.C, p.ldc, p.M, p.N, p.n_split, p.ldc_split,
                      p.bias, p.bias_mode, p.epilogue, p.aux, p.ldaux, p.colsum, p.nb};
    write_acc<FM, FN, MODE != kLoadAlignedVec, SPLITN, VA, VB>(acc, epi, bm + wm0, bn + wn0, lane);
}

inline KParams kparams_of(const GemmArgs& g, int64_t k_chunk) {
    KParams kp{static_cast<const float*>(g.A), static_cast<const float*>(g.B), g.C, g.bias,
               g.M, g.N, g.K, g.lda, g.ldb, g.ldc,
               g.n_split, g.ldc_split, g.bias_mode, g.epilogue, k_chunk,
               g.stride_a, g.stride_b, g.stride_c, g.batch, 0, 0, g.aux, g.ldaux,
               g.ones_col >= 0 ? g.ones_col : g.N, g.ones_col, g.colsum};
    // 16-byte loads need 16-byte aligned bases, leading dimensions and batch
    // strides, decided per operand (a 10-column operand no longer sends the
    // other one down the scalar path: C4's dW2 = dY2^T H, 10 x 256 x 8192,
    // 14 us with both operands scalar)
    kp.vec_a = ((uintptr_t)g.A % 16 == 0) && g.lda % 4 == 0 && g.stride_a % 4 == 0;
    kp.vec_b = ((uintptr_t)g.B % 16 == 0) && g.ldb % 4 == 0 && g.stride_b % 4 == 0;
    return kp;
}

}  // namespace f32
}  // namespace cdx
