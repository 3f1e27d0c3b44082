// Conv backward weight without LDS staging: every wave gathers its own MFMA
// operands from global memory (the companion of conv_direct.hip).
//
//   dW[oc, n] = sum over images b and pixels s of dY[b, oc, s] x[b, ic, oh SH + kh - PH, ow SW + kw - PW]
//   n = (ic KH + kh) KW + kw,  s = oh OW + ow
//
// The staged kernels (conv_wgrad.hip) own 64 channels x 144 or 192 filter
// elements per workgroup of twelve waves and share each k-tile through LDS and
// a barrier; on small layers that is a handful of workgroups, each waiting for
// its loads at every barrier.  Here a wave owns 16 FM channels x 32 filter
// elements, k = pixels 16 at a time (an image's last step is short); the four
// waves of a workgroup take a quarter each of its slice of the steps and are
// summed in wave order through LDS.  FP32 products (v_mfma_f32_16x16x4_f32; lane
// group lq feeds MFMA q with pixel 4 lq + q), runs of 32 pixels summed from
// zero, then added to the total.
//
// Per step a lane loads four consecutive pixels of each of its dY rows (16
// bytes, any 4-byte alignment) and, for each of its two filter elements, the
// input at those four pixels: the element's byte offset is fixed, the pixels'
// offsets are found once per step by a multiply-high division and shared by
// the lane's elements, and taps in the padding are zeroed.  The next two steps'
// loads are in flight during a step's MFMAs.
#include "cdx_internal.hpp"

namespace cdx {
namespace {

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

struct WdArgs {
    const float* dy; const float* x; float* out;   // out: [slices][OC][Kc] (or dW)
    int OC, Kc, S, OW, IH, IW, plane, KW, KHW, SH, SW, PH, PW;
    int64_t img_x, img_y;        // IC*IH*IW, OC*S (elements)
    int spi, steps, chunk;       // steps per image, in all, per slice
    DivMagic div_ow, div_khw, div_kw;
};

// ONE: 1x1, stride 1, no padding -- a filter element's pixels lie in a row, so
// the input is read like dY (16 x 256 -> 64
// channels at 56^2: 59 -> 43 us).
template <int FM, bool ONE>
__global__ __launch_bounds__(256)
void conv_wgrad_direct_kernel(WdArgs p) {
    constexpr int FN = 2, WK = 4;
    const int lane = threadIdx.x & 63;
    const int wk = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, lq = lane >> 4;
    const int n0 = blockIdx.x * 16 * FN, oc0 = blockIdx.y * 16 * FM;

    uint32_t offy[FM];   // byte offsets in an image of dY (rows past the end: the last)
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int oc = oc0 + i * 16 + l16;
        offy[i] = ((uint32_t)(oc < p.OC ? oc : p.OC - 1) * (uint32_t)p.S + 4u * lq) * 4u;
    }
    uint32_t offx[FN];   // of the element's tap at pixel 0 (mod 2^32: it may lie in the padding)
    int dh[FN], dw[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int n = n0 + j * 16 + l16;
        const uint32_t nn = (uint32_t)(n < p.Kc ? n : p.Kc - 1);
        const uint32_t ic = div_u31(nn, p.div_khw), t = nn - ic * (uint32_t)p.KHW;
        const uint32_t kh = div_u31(t, p.div_kw);
        dh[j] = (int)kh - p.PH;
        dw[j] = (int)(t - kh * (uint32_t)p.KW) - p.PW;
        offx[j] = (uint32_t)((int)ic * p.plane + dh[j] * p.IW + dw[j]) * 4u;
    }

    floatx4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    // this wave's steps [t0, t1): an even number for all waves but the last
    const int c0 = blockIdx.z * p.chunk, c1 = c0 + p.chunk < p.steps ? c0 + p.chunk : p.steps;
    const int per = ((c1 - c0 + WK - 1) / WK + 1) / 2 * 2;
    const int t0 = c0 + wk * per < c1 ? c0 + wk * per : c1, t1 = t0 + per < c1 ? t0 + per : c1;

    struct Step { f32x4u a[FM]; float b[FN][4]; uint32_t ok; };
    Step st[2];
    int ld_b = t0 / p.spi, ld_s = t0 - ld_b * p.spi, ld_t = t0;   // the step the next load() reads
    auto load = [&](Step& r) {   // past t1: the last step again, unused
        const int s0 = ld_s * 16 + 4 * lq;
        const char* yb = reinterpret_cast<const char*>(p.dy + ld_b * p.img_y + ld_s * 16);
        const char* xb = reinterpret_cast<const char*>(p.x + ld_b * p.img_x);
        if (ld_s * 16 + 16 <= p.S) {
#pragma unroll
            for (int i = 0; i < FM; ++i)
                r.a[i] = *(const __attribute__((address_space(1))) f32x4u*)(yb + offy[i]);
        } else {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    r.a[i][q] = s0 + q < p.S ? *(const float*)(yb + offy[i] + q * 4) : 0.0f;
        }
        auto advance = [&]() {
            if (ld_t + 1 < t1) {
                ++ld_t;
                if (++ld_s == p.spi) {
                    ld_s = 0;
                    ++ld_b;
                }
            }
        };
        if constexpr (ONE) {
            r.ok = 0xffu;
            if (ld_s * 16 + 16 <= p.S) {
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    const f32x4u v = *(const __attribute__((address_space(1))) f32x4u*)(xb + offx[j] + 4 * s0);
#pragma unroll
                    for (int q = 0; q < 4; ++q) r.b[j][q] = v[q];
                }
            } else {
#pragma unroll
                for (int j = 0; j < FN; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        r.b[j][q] = s0 + q < p.S ? *(const float*)(xb + offx[j] + 4 * (s0 + q)) : 0.0f;
            }
            advance();
            return;
        }
        int oh = (int)div_u31((uint32_t)s0, p.div_ow), ow = s0 - oh * p.OW;
        r.ok = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int ih = oh * p.SH, iw = ow * p.SW;
            const uint32_t pix = (uint32_t)(ih * p.IW + iw) * 4u;
            const bool in = s0 + q < p.S;
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const bool v = in && (unsigned)(ih + dh[j]) < (unsigned)p.IH &&
                               (unsigned)(iw + dw[j]) < (unsigned)p.IW;
                r.b[j][q] = *(const __attribute__((address_space(1))) float*)(xb + (v ? offx[j] + pix : 0u));
                r.ok |= (uint32_t)v << (4 * j + q);
            }
            const bool wrap = ++ow == p.OW;
            ow = wrap ? 0 : ow;
            oh += wrap ? 1 : 0;
        }
        advance();
    };
    floatx4 sum[FM][FN];
    auto mul = [&](const Step& r, bool first) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const float b = ONE || ((r.ok >> (4 * j + q)) & 1u) ? r.b[j][q] : 0.0f;
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
    if (t0 < t1) {
        load(st[0]);
        load(st[1]);
        int t = t0;
        for (; t + 1 < t1; t += 2) {
            mul(st[0], true);
            load(st[0]);
            mul(st[1], false);
            load(st[1]);
            fold();
        }
        if (t < t1) {
            mul(st[0], true);
            fold();
        }
    }

    __shared__ floatx4 red[WK][FM * FN][64];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) red[wk][i * FN + j][lane] = acc[i][j];
    __syncthreads();
    float* out = p.out + (int64_t)blockIdx.z * p.OC * p.Kc;
    for (int e = wk; e < FM * FN; e += WK) {
        floatx4 v = red[0][e][lane];
#pragma unroll
        for (int u = 1; u < WK; ++u) v += red[u][e][lane];
        const int n = n0 + e % FN * 16 + l16;
        if (n >= p.Kc) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {   // register r: row 4 lq + r of the block
            const int oc = oc0 + e / FN * 16 + 4 * lq + r;
            if (oc < p.OC) out[(int64_t)oc * p.Kc + n] = v[r];
        }
    }
}

template <bool ONE>
void launch_fm(int fm, dim3 grid, hipStream_t stream, const WdArgs& p) {
    if (fm == 4) hipLaunchKernelGGL((conv_wgrad_direct_kernel<4, ONE>), grid, dim3(256), 0, stream, p);
    else if (fm == 2) hipLaunchKernelGGL((conv_wgrad_direct_kernel<2, ONE>), grid, dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((conv_wgrad_direct_kernel<1, ONE>), grid, dim3(256), 0, stream, p);
}

}  // namespace

// Channels per wave, in sixteens: the most, unless that pads more.
int conv_wgrad_direct_fm(int64_t OC) {
    auto padded = [&](int fm) { return ceil_div(OC, 16 * fm) * 16 * fm; };
    return OC <= 16 ? 1 : padded(2) * 115 < padded(4) * 100 ? 2 : 4;
}

// 32-bit byte offsets within an image of either tensor, 32-bit steps.
bool conv_wgrad_direct_ok(int64_t batch, int64_t IC, int64_t OC, int64_t IH, int64_t IW, int64_t KH,
                          int64_t KW, int64_t SH, int64_t SW, int64_t PH, int64_t PW) {
    const int64_t OH = (IH + 2 * PH - KH) / SH + 1, OW = (IW + 2 * PW - KW) / SW + 1;
    const int64_t lim = INT32_MAX / 4;
    return batch >= 1 && IC >= 1 && OC >= 1 && OH >= 1 && OW >= 1 && IC * IH * IW < lim &&
           OC * OH * OW < lim && IC * KH * KW < lim && batch * ceil_div(OH * OW, 16) < lim &&
           (OH + 1) * SH + KH + PH < 32768 && (OW + 1) * SW + KW + PW < 32768 && IW < 32768 &&
           IH < 32768 && ceil_div(OC, 16) <= 65535;
}

// `slices` slices of the pixels: out is [slices][OC][IC KH KW] (dW itself for one).
int launch_conv_wgrad_direct_f32(const float* dy, const float* x, float* out, int slices,
                                 int64_t batch, int64_t IC, int64_t OC, int64_t IH, int64_t IW,
                                 int64_t KH, int64_t KW, int64_t SH, int64_t SW, int64_t PH,
                                 int64_t PW, hipStream_t stream) {
    const int64_t OH = (IH + 2 * PH - KH) / SH + 1, OW = (IW + 2 * PW - KW) / SW + 1;
    WdArgs p;
    p.dy = dy; p.x = x; p.out = out;
    p.OC = (int)OC; p.Kc = (int)(IC * KH * KW); p.S = (int)(OH * OW); p.OW = (int)OW;
    p.IH = (int)IH; p.IW = (int)IW; p.plane = (int)(IH * IW);
    p.KW = (int)KW; p.KHW = (int)(KH * KW); p.SH = (int)SH; p.SW = (int)SW; p.PH = (int)PH; p.PW = (int)PW;
    p.img_x = IC * IH * IW; p.img_y = OC * OH * OW;
    p.spi = (int)ceil_div(p.S, 16);
    p.steps = (int)(batch * p.spi);
    p.chunk = (int)ceil_div(p.steps, slices);
    p.div_ow = div_magic(OW); p.div_khw = div_magic(KH * KW); p.div_kw = div_magic(KW);
    const int fm = conv_wgrad_direct_fm(OC);
    const dim3 grid((unsigned)ceil_div(p.Kc, 32), (unsigned)ceil_div(OC, 16 * fm), (unsigned)slices);
    const bool one = KH == 1 && KW == 1 && SH == 1 && SW == 1 && PH == 0 && PW == 0;
    if (one) launch_fm<true>(fm, grid, stream, p);
    else launch_fm<false>(fm, grid, stream, p);
    return hip_error(hipGetLastError(), "conv_wgrad_direct_kernel launch");
}

}  // namespace cdx
