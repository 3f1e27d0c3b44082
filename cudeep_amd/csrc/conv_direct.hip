// Convolution (forward, and stride-1 backward data as the forward of dY with
// the flipped filter) without LDS windows, column buffers or barriers in the
// loop over channels: every wave gathers its own MFMA operands from global
// memory.  FP32 MFMA products (v_mfma_f32_16x16x4_f32), k = (ic, kh, kw) in
// the order of the filter, summed in two levels: runs of 32 k from zero, each
// added to the total.
//
// For layers that give the row-window kernel (conv_implicit.hip: 64 channels x
// ~100 pixels per workgroup, all of k in one chain) too few workgroups, and
// for windows it cannot keep in LDS.  A wave owns 16 FM output channels x 32
// pixels; WK = 4: the four waves of a workgroup share one tile, each with a
// quarter of k, summed in wave order at the end, so even one 7 x 7 layer on
// one small image spreads over the chip.
//
// Per 16 k a lane needs four taps of each of its two pixels (k = k0 + 4 lq +
// q, as in the library's GEMMs) and, of every filter row, four consecutive
// elements (one 16-byte load, any 4-byte alignment).  A tap's byte offset from
// the pixel's origin and its (kh, kw) index come from a table in LDS, filled
// once per 1024 k; whether it falls into the padding from a bit mask per pixel
// over the KH KW taps, made once.  The loads of the next two steps are in
// flight during a step's MFMAs (FM = 4: 1024 cycles).
#include "cdx_internal.hpp"

namespace cdx {
namespace {

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int CD_CHUNK = 1024;      // k per table
constexpr int CD_TAPS = 63;         // taps a pixel's mask holds (bit 63: k past the end)

struct CdArgs {
    const float* x; const float* w; const float* bias; float* y;
    int OC, Kc, S, N, OW, IH, IW, plane, KW, KHW, SH, SW, PH, PW;
    int64_t img_x, img_y;           // IC*IH*IW, OC*S (elements)
    DivMagic div_s, div_ow, div_khw, div_kw;
};

template <int FM, int WK>
__global__ __launch_bounds__(256)
void conv_direct_kernel(CdArgs p) {
    constexpr int FN = 2, WN = 4 / WK;
    __shared__ __attribute__((aligned(16))) int offs[CD_CHUNK];
    __shared__ __attribute__((aligned(16))) unsigned char taps[CD_CHUNK];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lq = lane >> 4;
    const int wk = wave % WK;
    const int oc0 = blockIdx.y * 16 * FM;
    const int n0 = (blockIdx.x * WN + wave / WK) * 16 * FN;

    // this lane's pixels (past the end: the last one): byte offset of the
    // window's origin (mod 2^32: it may lie in the padding) and tap mask
    uint32_t org[FN];
    uint64_t mask[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        int n = n0 + j * 16 + l16;
        n = n < p.N ? n : p.N - 1;
        const int b = (int)div_u31((uint32_t)n, p.div_s), s = n - b * p.S;
        const int oh = (int)div_u31((uint32_t)s, p.div_ow), ow = s - oh * p.OW;
        const int ih0 = oh * p.SH - p.PH, iw0 = ow * p.SW - p.PW;
        org[j] = (uint32_t)(b * p.img_x + (int64_t)ih0 * p.IW + iw0) * 4u;
        uint64_t m = 0;
        int kh = 0, kw = 0;
        for (int t = 0; t < p.KHW; ++t) {
            if ((unsigned)(ih0 + kh) < (unsigned)p.IH && (unsigned)(iw0 + kw) < (unsigned)p.IW)
                m |= (uint64_t)1 << t;
            if (++kw == p.KW) { kw = 0; ++kh; }
        }
        mask[j] = m;
    }
    uint32_t offw[FM];   // byte offsets of this lane's filter rows (past the end: the last)
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int oc = oc0 + i * 16 + l16;
        offw[i] = (uint32_t)(oc < p.OC ? oc : p.OC - 1) * (uint32_t)p.Kc * 4u + 16u * lq;
    }
    const char* xb = reinterpret_cast<const char*>(p.x);
    const char* wb = reinterpret_cast<const char*>(p.w);

    floatx4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    struct Step { f32x4u a[FM]; float b[FN][4]; uint32_t ok; };
    Step st[2];

    for (int c0 = 0; c0 < p.Kc; c0 += CD_CHUNK) {
        const int kn = p.Kc - c0 < CD_CHUNK ? p.Kc - c0 : CD_CHUNK;
        const int steps = (kn + 15) / 16;
        if (c0 > 0) __syncthreads();
        for (int i = tid; i < steps * 16; i += 256) {
            const uint32_t k = (uint32_t)(c0 + i);
            const uint32_t ic = div_u31(k, p.div_khw), t = k - ic * (uint32_t)p.KHW;
            const uint32_t kh = div_u31(t, p.div_kw), kw = t - kh * (uint32_t)p.KW;
            const bool in = i < kn;
            offs[i] = in ? (int)((ic * (uint32_t)p.plane + kh * (uint32_t)p.IW + kw) * 4u) : 0;
            taps[i] = in ? (unsigned char)t : (unsigned char)CD_TAPS;
        }
        __syncthreads();
        // this wave's steps [s0, s1), an even number of steps per wave but the last
        const int per = WK == 1 ? steps : ((steps + WK - 1) / WK + 1) / 2 * 2;
        const int s0 = wk * per < steps ? wk * per : steps;
        const int s1 = s0 + per < steps ? s0 + per : steps;
        if (s0 == s1) continue;
        auto load = [&](Step& r, int s) {   // past s1: that step again, unused
            if (s >= s1) s = s1 - 1;
            const int kk = s * 16;
            const char* wk0 = wb + (int64_t)(c0 + kk) * 4;
            if (c0 + kk + 16 <= p.Kc) {
#pragma unroll
                for (int i = 0; i < FM; ++i)
                    r.a[i] = *(const __attribute__((address_space(1))) f32x4u*)(wk0 + offw[i]);
            } else {
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        r.a[i][q] = c0 + kk + 4 * lq + q < p.Kc ? *(const float*)(wk0 + offw[i] + q * 4) : 0.0f;
            }
            const int4 o = *reinterpret_cast<const int4*>(offs + kk + 4 * lq);
            const uint32_t tp = *reinterpret_cast<const uint32_t*>(taps + kk + 4 * lq);
            const int ov[4] = {o.x, o.y, o.z, o.w};
            r.ok = 0;
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t v = (uint32_t)(mask[j] >> ((tp >> (8 * q)) & 63u)) & 1u;
                    const uint32_t at = v ? org[j] + (uint32_t)ov[q] : 0u;
                    r.b[j][q] = *(const __attribute__((address_space(1))) float*)(xb + at);
                    r.ok |= v << (4 * j + q);
                }
        };
        floatx4 sum[FM][FN];
        auto mul = [&](const Step& r, bool first) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    const float b = (r.ok >> (4 * j + q)) & 1u ? r.b[j][q] : 0.0f;
#pragma unroll
                    for (int i = 0; i < FM; ++i)
                        sum[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            r.a[i][q], b, first && q == 0 ? floatx4{0.f, 0.f, 0.f, 0.f} : sum[i][j],
                            0, 0, 0);
                }
        };
        auto fold = [&]() {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[i][j] += sum[i][j];
        };
        load(st[0], s0);
        load(st[1], s0 + 1);
        int s = s0;
        for (; s + 1 < s1; s += 2) {
            mul(st[0], true);
            load(st[0], s + 2);
            mul(st[1], false);
            load(st[1], s + 3);
            fold();
        }
        if (s < s1) {
            mul(st[0], true);
            fold();
        }
    }

    // D: register r of lane l is channel 4 (l / 16) + r, pixel l % 16 of its block
    auto put = [&](const floatx4& v, int i, int j) {
        const int n = n0 + j * 16 + l16;
        if (n >= p.N) return;
        const int b = (int)div_u31((uint32_t)n, p.div_s), s = n - b * p.S;
        float* yb = p.y + (int64_t)b * p.img_y + s;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int oc = oc0 + i * 16 + 4 * lq + r;
            if (oc < p.OC) yb[(int64_t)oc * p.S] = p.bias ? v[r] + p.bias[oc] : v[r];
        }
    };
    if constexpr (WK == 1) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) put(acc[i][j], i, j);
    } else {
        __shared__ floatx4 red[WK][FM * FN][64];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) red[wk][i * FN + j][lane] = acc[i][j];
        __syncthreads();
        for (int e = wk; e < FM * FN; e += WK) {
            floatx4 v = red[0][e][lane];
#pragma unroll
            for (int u = 1; u < WK; ++u) v += red[u][e][lane];
            put(v, e / FN, e % FN);
        }
    }
}

template <int WK>
void launch_fm(int fm, dim3 grid, hipStream_t stream, const CdArgs& p) {
    if (fm == 4) hipLaunchKernelGGL((conv_direct_kernel<4, WK>), grid, dim3(256), 0, stream, p);
    else if (fm == 2) hipLaunchKernelGGL((conv_direct_kernel<2, WK>), grid, dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((conv_direct_kernel<1, WK>), grid, dim3(256), 0, stream, p);
}

// Channels per wave 16 fm and whether the waves of a workgroup split k.  Wider
// waves load less per MFMA (8 x 64 -> 128 channels, 56^2, stride 2: 24 us with
// 64 channels, 29 with 32), unless they pad more (3 x 80 -> 72, 14^2, 7x7: 64
// with 128 padded channels, 49 with 96) or are too few (1 x 148 -> 104, 60^2,
// stride 2, 58 tiles: 25 against 20).  k is split wherever there are at least
// eight steps of 16 of it (20 x 128 -> 168, 28^2, 7x7 stride 2, 1.2 k tiles:
// 165 us against 356) and the unsplit tiles would not fill the SIMDs four times
// over (16 x 3 -> 64, 224^2, 7x7 stride 2, K = 147, 6.3 k tiles: 156 against 92).
struct DirectPlan {
    int fm;
    bool split;
};

DirectPlan plan_of(int64_t N, int64_t OC, int64_t Kc) {
    auto padded = [&](int fm) { return ceil_div(OC, 16 * fm) * 16 * fm; };
    auto tiles = [&](int fm) { return ceil_div(N, 32) * ceil_div(OC, 16 * fm); };
    int fm = OC <= 16 ? 1 : 4;
    if (fm == 4 && (padded(2) * 115 < padded(4) * 100 || tiles(4) < 150)) fm = 2;
    if (fm == 2 && tiles(2) < 64) fm = 1;
    return {fm, Kc >= 128 && tiles(fm) < 4096};
}

}  // namespace

// Where this kernel is taken before the row-window one: that one's tiles (64
// channels x about 112 pixels) leave a third of the CUs or more without work,
// or pad most of their channels.  In us, row-window against this kernel, with
// the row-window tiles:
//   3 x 80 -> 72, 14^2, 7x7 (12)            160 / 39    backward data 185 / 43
//   16 x 107 -> 24, 28^2, 7x7 s2 (28)       327 / 63
//   8 x 128 -> 256, 28^2, 3x3 s2 (56)        55 / 24
//   20 x 128 -> 168, 28^2, 7x7 s2 (105)     338 / 164
//   98 -> 12, 112^2 (112)                              backward data 62 / 18
//   8 x 64 -> 64, 56^2 (224)                 33 / 39                 35 / 40
//   32 x 256 -> 256, 14^2 (224)             112 / 117               116 / 120
//   16 x 64 -> 64, 56^2 (448)                49 / 61
//   16 -> 8 channels, 4 x 112^2, 5x5 (448)                           40 / 29
// With k < 128, unsplit, 64-channel waves have too little to hide their loads
// behind: 2 x 12 -> 512, 28^2 10.6 / 12.4, backward data 256 -> 8, 28^2 10.4 /
// 13.1, 16 x 3 -> 64, 56^2, 5x5 s2 10.2 / 12.8 (with 32 channels 4 x 12 -> 96, 31^2
// s2 10.9 / 8.7); except for 1x1 layers with a stride, of whose window the
// row-window kernel uses one pixel in SH SW (4 x 96 -> 100, 56^2 s2 19 / 10).  Nor
// do up to eight channels of large filters give that kernel's loop over channel
// chunks anything to wait for (16 x 8 -> 51, 28^2, 7x7, 112 tiles 18.6 / 23.1; 14 x
// 8 -> 64, 31^2, 5x5, 121 tiles 12.7 / 14.2), nor four, a chunk without
// padding, at any size (9 x 4 -> 64, 14^2, 5x5 8.7 / 10.8; 1 x 4 -> 81, 56^2, 7x7
// 12.3 / 14.9; but 8 x 3 -> 64, 31^2, 7x7 s2 13.8 / 12.0).
// Where that one's window does not fit LDS, its gathering form (64 channels x
// 128 pixels per workgroup) keeps the layers whose k is not split here (16 x 3
// -> 64, 224^2, 7x7 stride 2: 73 against 92) and those of 2048 tiles of this
// kernel and more (2 x 16 -> 168, 224^2, 7x7 s2, 2352 tiles: 132 against 143; 16 x
// 16 -> 256, 112^2, 7x7 s3, 2888: 144 against 182; 8 x 64 -> 128, 112^2, 7x7 s2,
// 1568: 370 against 317) or eight channels (8 x 8 -> 127, 112^2, 7x7 s2, 1568: 54
// against 75).  Neither line holds where 64-channel tiles pad a third
// more than this kernel's waves (9 x 80 -> 81, 112^2, 7x7 s2, 2646: 460 against
// 329; 16 x 6 -> 24, 31^2, 7x7 21 against 17; a fifth more, 6 x 4 -> 129, 56^2, 7x7 s2
// 12.5 against 18.4).
bool conv_direct_pays(int64_t N, int64_t OC, int64_t Kc, int64_t taps, bool rowwin) {
    if (OC <= 16) return true;
    const DirectPlan pl = plan_of(N, OC, Kc);
    const int64_t rw_tiles = ceil_div(OC, 64) * ceil_div(N, 112), waves = ceil_div(OC, 16 * pl.fm);
    const bool pads_less = ceil_div(OC, 64) * 64 * 3 >= waves * 16 * pl.fm * 4;
    if (rw_tiles < 160) {
        if (taps >= 25 && Kc == 4 * taps) return pads_less;
        return Kc >= 128 ? Kc > 8 * taps || rw_tiles < 100 || pads_less : pl.fm < 4 || taps == 1;
    }
    return !rowwin && pl.split &&
           ((ceil_div(N, 32) * waves < 2048 && Kc > 8 * taps) || pads_less);
}

// 32-bit byte offsets into the input and the filter, taps within the mask.
bool conv_direct_ok(int64_t batch, int64_t IC, int64_t OC, int64_t IH, int64_t IW, int64_t KH,
                    int64_t KW, int64_t SH, int64_t SW, int64_t PH, int64_t PW) {
    const int64_t OH = (IH + 2 * PH - KH) / SH + 1, OW = (IW + 2 * PW - KW) / SW + 1;
    const int64_t lim = INT32_MAX / 4;
    return batch >= 1 && IC >= 1 && OC >= 1 && OH >= 1 && OW >= 1 && KH * KW <= CD_TAPS &&
           batch * IC * IH * IW < lim && OC * IC * KH * KW < lim && batch * OH * OW < lim &&
           OH * SH + PH < lim && OW * SW + PW < lim && (PH + KH) * IW < lim;
}

int launch_conv_direct_f32(const float* x, const float* w, const float* bias, float* y,
                           int64_t batch, int64_t IC, int64_t OC, int64_t IH, int64_t IW,
                           int64_t KH, int64_t KW, int64_t SH, int64_t SW, int64_t PH, int64_t PW,
                           hipStream_t stream) {
    const int64_t OH = (IH + 2 * PH - KH) / SH + 1, OW = (IW + 2 * PW - KW) / SW + 1;
    CdArgs p;
    p.x = x; p.w = w; p.bias = bias; p.y = y;
    p.OC = (int)OC; p.Kc = (int)(IC * KH * KW); p.S = (int)(OH * OW); p.N = (int)(batch * OH * OW);
    p.OW = (int)OW; p.IH = (int)IH; p.IW = (int)IW; p.plane = (int)(IH * IW);
    p.KW = (int)KW; p.KHW = (int)(KH * KW); p.SH = (int)SH; p.SW = (int)SW; p.PH = (int)PH; p.PW = (int)PW;
    p.img_x = IC * IH * IW; p.img_y = OC * OH * OW;
    p.div_s = div_magic(p.S); p.div_ow = div_magic(OW);
    p.div_khw = div_magic(KH * KW); p.div_kw = div_magic(KW);
    const DirectPlan pl = plan_of(p.N, OC, p.Kc);
    const int fm = pl.fm;
    const bool split = pl.split;
    const int wn = split ? 1 : 4;
    const dim3 grid((unsigned)ceil_div(p.N, 32 * wn), (unsigned)ceil_div(OC, 16 * fm));
    if (split) launch_fm<4>(fm, grid, stream, p);
    else launch_fm<1>(fm, grid, stream, p);
    return hip_error(hipGetLastError(), "conv_direct_kernel launch");
}

}  // namespace cdx
