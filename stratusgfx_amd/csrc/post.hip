// Consumers of the lit buffer.
//
// tonemapKernel — gammaTonemap.fs:125-142 (PerformGammaTonemapPostFx_,
// StratusRendererBackend.cpp:2356-2366): Narkowicz's ACES film fit
// saturate(c (a c + b) / (c (c' c + d) + e)) (:20-29), gamma correction
// pow(c, 1 / gamma) (:112-114), stored to the RGBA8 UNORM target (:674) as
// floor(c * 255 + 0.5), alpha 255.  One thread per pixel: 12 B read and 4 B
// written.  Built with -ffp-contract=off, so the curve's products and sums round
// as the shader writes them; pow is the device library's.  Three pows a pixel
// made it bound by the vector ALU (4K: 100 us); an estimate decides the code
// wherever it is not near a tie, and the kernel is bound by memory (25.6 us, the
// bytes alone 25.8).
#include "launch.h"

namespace {

using namespace sgi_dev;

__device__ __forceinline__ float sat(float x) { return fminf(fmaxf(x, 0.0f), 1.0f); }

__device__ __forceinline__ uint32_t tonemapChannel(float x, float invGamma) {
    const float a = 2.51f, b = 0.03f, c = 2.43f, d = 0.59f, e = 0.14f;
    const float film = sat((x * (a * x + b)) / (x * (c * x + d) + e));
    const float g = powf(film, invGamma);
    return (uint32_t)(sat(g) * 255.0f + 0.5f);
}

// The same code from the hardware's reciprocal, log2 and exp2 where that cannot differ: `margin` (in codes,
// at least 2e-4) bounds the estimate's error and the estimate is at least that far from the next code.
// The reciprocal's and the product's errors move the film value by 3e-7 of it and the power by 1 / gamma
// times that; the exponent's error is 2^-21 of it, and g |log2 g| < 0.54.  Everything else (the
// ranges where an intermediate could overflow or be denormal, NaN) takes the exact form.
__device__ __forceinline__ uint32_t tonemapFast(float x, float invGamma, float margin) {
    const float a = 2.51f, b = 0.03f, c = 2.43f, d = 0.59f, e = 0.14f;
    const float num = x * (a * x + b);
    const float film = sat(num * __builtin_amdgcn_rcpf(x * (c * x + d) + e));
    const float v = __builtin_amdgcn_exp2f(invGamma * __builtin_amdgcn_logf(film)) * 255.0f + 0.5f;
    const float code = floorf(v);
    if (fabsf(x) < 1e9f && (num <= 0.0f || film >= 1e-30f) && v - code > margin && v - code < 1.0f - margin)
        return (uint32_t)code;
    return tonemapChannel(x, invGamma);
}

template <bool EXACT>
__global__ __launch_bounds__(256) void tonemapKernel(const float* __restrict__ lit, long n, float invGamma,
                                                      float margin, uint32_t* __restrict__ out) {
    const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const float r = lit[3 * p], g = lit[3 * p + 1], b = lit[3 * p + 2];
    const auto code = [&](float x) { return EXACT ? tonemapChannel(x, invGamma) : tonemapFast(x, invGamma, margin); };
    out[p] = code(r) | (code(g) << 8) | (code(b) << 16) | 0xFF000000u;
}

// ---- TAA history (PerformTaaPostFx_'s copy, StratusRendererBackend.cpp:2342-2349)
//
// The TAA target is RGBA16F (:708-711): the output rounds to binary16 (RNE);
// the NEAREST blit into the RGB8 UNORM previousFrameBuffer (:449-453) clamps
// to [0, 1] and stores floor(v * 255 + 0.5); the next frame reads k / 255.
// k / 255 correctly rounded for the 256 codes: an estimate and its remainder
__device__ __forceinline__ float codeToFloat(float k) {
    const float q = k * 0x1.010102p-8f;
    return __builtin_fmaf(__builtin_fmaf(-255.0f, q, k), 0x1.010102p-8f, q);
}

// 24 B a pixel and little else: four values per thread and no division, 4K 51 -> 30 us.
__device__ __forceinline__ float historyTexel(float taa) {
    const float k = floorf(sat(__half2float(__float2half_rn(taa))) * 255.0f + 0.5f);
    return codeToFloat(k);
}

// Both images 16-byte aligned: four values per thread, and the last up to three by one more (a launch of
// their own cost a 641x361 image 1.3 us of 4.3).
__global__ __launch_bounds__(256) void taaHistory4Kernel(const float* __restrict__ taa, long n3,
                                                          float* __restrict__ prev) {
    const long q = 4 * ((long)blockIdx.x * blockDim.x + threadIdx.x);
    if (q + 4 <= n3) {
        const float4 v = *reinterpret_cast<const float4*>(taa + q);
        *reinterpret_cast<float4*>(prev + q) =
            make_float4(historyTexel(v.x), historyTexel(v.y), historyTexel(v.z), historyTexel(v.w));
    } else {
        for (long i = q; i < n3; ++i) prev[i] = historyTexel(taa[i]);
    }
}

// Any alignment.
__global__ __launch_bounds__(256) void taaHistoryKernel(const float* __restrict__ taa, long n3,
                                                         float* __restrict__ prev) {
    const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n3) prev[q] = historyTexel(taa[q]);
}

// ---- FXAA (PerformFxaaPostFx_, StratusRendererBackend.cpp:2293-2321)
//
// The reference runs two passes: fxaa_luminance.fs writes the tonemapped
// colour with its luminance in alpha to an RGBA8 target, fxaa_smoothing.fs
// filters that target.  Here one kernel does both: a block computes the stored
// alpha codes of its pixels and of a halo once into LDS, from their tonemapped
// rgb codes (the luminance in the shader's order, then the UNORM8 store), which
// is exactly what the intermediate target would hold, so the intermediate never
// touches HBM (4 B read and 4 B written per pixel).  Pixels below the contrast
// threshold are copied; the others are listed in LDS, so that the edge walks,
// tens of dependent steps each, run on full waves, and a step reads LDS.  With a
// luma per tap and the walks where they fell a 4K frame took 69 us and 640x360
// 16; now 55 and 12, half of it the walks.  Built with -ffp-contract=off, so every product
// and sum rounds as the shaders write them.
struct FxaaImage {
    const uint32_t* px;  // RGBA8 texels [H][W] of the tonemapped target
    int W, H;
};

__device__ __forceinline__ uint32_t fxaaTexel(const FxaaImage& im, int x, int y) {
    return im.px[(size_t)clampi(y, 0, im.H - 1) * im.W + clampi(x, 0, im.W - 1)];
}

__device__ __forceinline__ float unorm8(uint32_t texel, int ch) {
    return codeToFloat((float)((texel >> (8 * ch)) & 0xFFu));
}

__device__ __forceinline__ uint32_t store8(float v) { return (uint32_t)(sat(v) * 255.0f + 0.5f); }

// The alpha of the luminance target at texel (x, y): aa_common.glsl:7-9 on the
// saturated colour (already in [0, 1], so the sum is at most 1 + 1e-7), stored UNORM8, read back as k / 255.
__device__ __forceinline__ float texelLuma(uint32_t t) {
    const float lum = 0.2126f * unorm8(t, 0) + 0.7152f * unorm8(t, 1) + 0.0722f * unorm8(t, 2);
    return codeToFloat(floorf(lum * 255.0f + 0.5f));
}

// A block's TW x TH pixels and HALO more on each side: their luma.  The edge walks reach up to 21
// texels; a step that leaves the halo computes its taps.
template <int TW, int TH, int HALO>
struct FxaaTile {
    static constexpr int kLumaW = TW + 2 * HALO, kLumaH = TH + 2 * HALO;
    FxaaImage im;
    const float* luma;
    int x0, y0;  // the texel of luma[0]
};

// GL LINEAR, CLAMP_TO_EDGE, of the luminance target's alpha at the points of one edge walk: a coordinate
// runs along the edge (u where the edge is horizontal, else v), the other stays.
template <class Tile>
struct FxaaWalk {
    static constexpr int kLumaW = Tile::kLumaW, kLumaH = Tile::kLumaH;
    const Tile& t;
    bool horizontal, acrossIn;
    int size, origin, count, step;  // along: texels, the tile's first texel and number of texels, its stride in luma
    int ja, jb;                     // across: the two texels
    float across;                   // and the weight of the second
    const float* rowA;
    const float* rowB;
    __device__ __forceinline__ FxaaWalk(const Tile& tile, bool isHorizontal, float acrossUv)
        : t(tile), horizontal(isHorizontal) {
        const int acrossSize = horizontal ? t.im.H : t.im.W, acrossOrigin = horizontal ? t.y0 : t.x0;
        const int acrossCount = horizontal ? kLumaH : kLumaW, acrossStep = horizontal ? kLumaW : 1;
        size = horizontal ? t.im.W : t.im.H;
        origin = horizontal ? t.x0 : t.y0;
        count = horizontal ? kLumaW : kLumaH;
        step = horizontal ? 1 : kLumaW;
        const float f = acrossUv * (float)acrossSize - 0.5f, i0f = floorf(f);
        across = f - i0f;
        ja = texelIndex(i0f, acrossSize);
        jb = texelIndex(i0f + 1.0f, acrossSize);
        acrossIn = (uint32_t)(ja - acrossOrigin) < (uint32_t)acrossCount &&
                   (uint32_t)(jb - acrossOrigin) < (uint32_t)acrossCount;
        rowA = t.luma + (ja - acrossOrigin) * acrossStep;
        rowB = t.luma + (jb - acrossOrigin) * acrossStep;
    }
    __device__ __forceinline__ float operator()(float along) const {
        const float f = along * (float)size - 0.5f, i0f = floorf(f);
        const float w = f - i0f, a = horizontal ? w : across, b = horizontal ? across : w;
        const int ia = texelIndex(i0f, size), ib = texelIndex(i0f + 1.0f, size);
        const int la = ia - origin, lb = ib - origin;
        float t00, tAlong, tAcross, t11;
        if (acrossIn && (uint32_t)la < (uint32_t)count && (uint32_t)lb < (uint32_t)count) {
            t00 = rowA[la * step];
            tAlong = rowA[lb * step];
            tAcross = rowB[la * step];
            t11 = rowB[lb * step];
        } else {
            const auto at = [&](int i, int j) {
                return texelLuma(t.im.px[horizontal ? (size_t)j * t.im.W + i : (size_t)i * t.im.W + j]);
            };
            t00 = at(ia, ja);
            tAlong = at(ib, ja);
            tAcross = at(ia, jb);
            t11 = at(ib, jb);
        }
        const float t10 = horizontal ? tAlong : tAcross, t01 = horizontal ? tAcross : tAlong;
        return (1.0f - a) * (1.0f - b) * t00 + a * (1.0f - b) * t10 + (1.0f - a) * b * t01 + a * b * t11;
    }
};

// The contrast test of the smoothing pass.
struct FxaaCross {
    float center, right, left, top, bot, contrast;
    bool edge;
};
// l: the pixel's luma in the tile; the halo holds the clamped texels past the frame's edge, so its neighbours
// are the ones beside it.
template <int kLumaW>
__device__ __forceinline__ FxaaCross fxaaCross(const float* l, float contrastThreshold, float relativeThreshold) {
    const float lumaCenter = l[0], lumaRight = l[1], lumaLeft = l[-1], lumaTop = l[kLumaW], lumaBot = l[-kLumaW];
    const float lumaMax = fmaxf(fmaxf(fmaxf(fmaxf(lumaCenter, lumaRight), lumaLeft), lumaTop), lumaBot);
    const float lumaMin = fminf(fminf(fminf(fminf(lumaCenter, lumaRight), lumaLeft), lumaTop), lumaBot);
    const float contrast = lumaMax - lumaMin;
    const float threshold = fmaxf(contrastThreshold, relativeThreshold * lumaMax);
    return FxaaCross{lumaCenter, lumaRight, lumaLeft, lumaTop, lumaBot, contrast, !(contrast < threshold)};
}

// The smoothing pass of an edge pixel.
template <class Tile>
__device__ __forceinline__ uint32_t fxaaEdge(const Tile& tile, int x, int y, float contrastThreshold,
                                             float relativeThreshold, float subpixelBlending) {
    constexpr int kLumaW = Tile::kLumaW;
    const FxaaImage& im = tile.im;
    const float* const l = tile.luma + (y - tile.y0) * kLumaW + (x - tile.x0);
    const FxaaCross c0 = fxaaCross<kLumaW>(l, contrastThreshold, relativeThreshold);
    const float lumaCenter = c0.center, lumaRight = c0.right, lumaLeft = c0.left, lumaTop = c0.top, lumaBot = c0.bot;
    const float contrast = c0.contrast;
    const float u = texelCentre(x, im.W), v = texelCentre(y, im.H);
    const float lumaTopRight = l[kLumaW + 1], lumaBotRight = l[-kLumaW + 1];
    const float lumaTopLeft = l[kLumaW - 1], lumaBotLeft = l[-kLumaW - 1];
    float average = 2.0f * (lumaRight + lumaLeft + lumaTop + lumaBot) + lumaTopRight + lumaBotRight + lumaTopLeft +
                    lumaBotLeft;
    average = average / 12.0f;
    const float centerAvgContrast = fabsf(average - lumaCenter);
    const float t = sat(sat(centerAvgContrast / contrast));
    float pixelBlendFactor = t * t * (3.0f - 2.0f * t);  // smoothstep(0, 1, .)
    pixelBlendFactor = pixelBlendFactor * pixelBlendFactor * subpixelBlending;
    const float horizontal = fabsf(lumaTop + lumaBot - 2.0f * lumaCenter) * 2.0f +
                             fabsf(lumaTopRight + lumaBotRight - 2.0f * lumaRight) +
                             fabsf(lumaTopLeft + lumaBotLeft - 2.0f * lumaLeft);
    const float vertical = fabsf(lumaRight + lumaLeft - 2.0f * lumaCenter) * 2.0f +
                           fabsf(lumaTopRight + lumaTopLeft - 2.0f * lumaTop) +
                           fabsf(lumaBotRight + lumaBotLeft - 2.0f * lumaBot);
    const bool isHorizontal = horizontal >= vertical;
    const float tsx = 1.0f / (float)im.W, tsy = 1.0f / (float)im.H;  // computeTexelSize
    float pixelStep = isHorizontal ? tsy : tsx;
    const float positiveLuma = isHorizontal ? lumaTop : lumaRight;
    const float negativeLuma = isHorizontal ? lumaBot : lumaLeft;
    const float positiveGradient = fabsf(positiveLuma - lumaCenter);
    const float negativeGradient = fabsf(negativeLuma - lumaCenter);
    float gradient, oppositeLuma;
    if (positiveGradient < negativeGradient) {
        pixelStep = -pixelStep;
        oppositeLuma = negativeLuma;
        gradient = negativeGradient;
    } else {
        oppositeLuma = positiveLuma;
        gradient = positiveGradient;
    }
    // half a texel towards the edge, then along it in steps of es; the other coordinate stays
    const float uvAlong = isHorizontal ? u : v, es = isHorizontal ? tsx : tsy;
    const FxaaWalk<Tile> walk(tile, isHorizontal, (isHorizontal ? v : u) + pixelStep * 0.5f);
    const float edgeLumaAvg = (lumaCenter + oppositeLuma) * 0.5f;
    const float gradientThreshold = gradient * 0.25f;
    // edgeStepOffsets = 1, 1.5, 2 x 7, 4; a guess jump of 8 when no end is found
    // (both directions step together: their taps do not wait for each other)
    float dist[2], deltas[2], at[2];
    bool atEnd[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        at[i] = uvAlong + (i == 0 ? es : -es) * 1.0f;
        deltas[i] = walk(at[i]) - edgeLumaAvg;
        atEnd[i] = fabsf(deltas[i]) >= gradientThreshold;
    }
    for (int j = 0; j < 9 && !(atEnd[0] && atEnd[1]); ++j) {
        const float off = j == 0 ? 1.5f : (j == 8 ? 4.0f : 2.0f);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float next = at[i] + (i == 0 ? es : -es) * off;
            const float delta = walk(next) - edgeLumaAvg;
            if (!atEnd[i]) {
                at[i] = next;
                deltas[i] = delta;
                atEnd[i] = fabsf(delta) >= gradientThreshold;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        if (!atEnd[i]) at[i] += (i == 0 ? es : -es) * 8.0f;
        dist[i] = i == 0 ? at[0] + (-uvAlong) : -at[1] + uvAlong;
    }
    float shortest;
    bool deltaSign;
    if (dist[0] <= dist[1]) {
        shortest = dist[0];
        deltaSign = deltas[0] >= 0.0f;
    } else {
        shortest = dist[1];
        deltaSign = deltas[1] >= 0.0f;
    }
    const float edgeBlendFactor =
        deltaSign == (lumaCenter - edgeLumaAvg >= 0.0f) ? 0.0f : 0.5f - shortest / (dist[0] + dist[1]);
    const float finalBlend = fmaxf(pixelBlendFactor, edgeBlendFactor);
    float fu = u, fv = v;
    if (isHorizontal) fv += pixelStep * finalBlend;
    else fu += pixelStep * finalBlend;
    // the final LINEAR tap of the rgb (the luminance target's rgb = the input's codes)
    const float gu = fu * (float)im.W - 0.5f, gv = fv * (float)im.H - 0.5f;
    const float i0f = floorf(gu), j0f = floorf(gv);
    const float a = gu - i0f, b = gv - j0f;
    const int ia = texelIndex(i0f, im.W), ib = texelIndex(i0f + 1.0f, im.W);
    const int ja = texelIndex(j0f, im.H), jb = texelIndex(j0f + 1.0f, im.H);
    const uint32_t t00 = fxaaTexel(im, ia, ja), t10 = fxaaTexel(im, ib, ja);
    const uint32_t t01 = fxaaTexel(im, ia, jb), t11 = fxaaTexel(im, ib, jb);
    uint32_t o = 0xFF000000u;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const float val = (1.0f - a) * (1.0f - b) * unorm8(t00, c) + a * (1.0f - b) * unorm8(t10, c) +
                          (1.0f - a) * b * unorm8(t01, c) + a * b * unorm8(t11, c);
        o |= store8(val) << (8 * c);
    }
    return o;
}

template <int TW, int TH, int HALO, int THREADS>
__global__ __launch_bounds__(THREADS) void fxaaKernel(FxaaImage im, float contrastThreshold, float relativeThreshold,
                                                   float subpixelBlending, uint32_t* __restrict__ out) {
    using Tile = FxaaTile<TW, TH, HALO>;
    constexpr int kLumaW = Tile::kLumaW, kLumaH = Tile::kLumaH;
    __shared__ float luma[kLumaW * kLumaH];
    __shared__ uint16_t edges[TW * TH];
    __shared__ int numEdges;
    const int tid = (int)threadIdx.x, tilesX = (im.W + TW - 1) / TW;
    const int b = (int)xcdSwizzle(blockIdx.x, gridDim.x), bx = (b % tilesX) * TW, by = (b / tilesX) * TH;
    if (tid == 0) numEdges = 0;
    __syncthreads();
    const Tile tile{im, luma, bx - HALO, by - HALO};
    if (tile.x0 >= 0 && tile.y0 >= 0 && tile.x0 + kLumaW <= im.W && tile.y0 + kLumaH <= im.H) {  // no clamping
        const uint32_t* const px = im.px + (size_t)tile.y0 * im.W + tile.x0;
        for (int i = tid; i < kLumaW * kLumaH; i += THREADS)
            luma[i] = texelLuma(px[(i / kLumaW) * im.W + i % kLumaW]);
    } else {
        for (int i = tid; i < kLumaW * kLumaH; i += THREADS)
            luma[i] = texelLuma(fxaaTexel(im, tile.x0 + i % kLumaW, tile.y0 + i / kLumaW));
    }
    __syncthreads();
    const int lane = tid & 63;
    for (int i = tid; i < TW * TH; i += THREADS) {
        const int x = bx + i % TW, y = by + i / TW;
        const bool in = x < im.W && y < im.H;
        const float* const l = luma + (i / TW + HALO) * kLumaW + i % TW + HALO;
        const bool edge = in && fxaaCross<kLumaW>(l, contrastThreshold, relativeThreshold).edge;
        if (in && !edge)  // the luminance pass re-stores k / 255 as k: the colour is the input's
            out[(size_t)y * im.W + x] = (im.px[(size_t)y * im.W + x] & 0x00FFFFFFu) | 0xFF000000u;
        const uint64_t m = __ballot(edge);
        if (!m) continue;
        int at = 0;
        if (lane == 0) at = atomicAdd(&numEdges, __popcll(m));
        at = __shfl(at, 0);
        if (edge) edges[at + __popcll(m & ((1ull << lane) - 1))] = (uint16_t)i;
    }
    __syncthreads();
    for (int i = tid; i < numEdges; i += THREADS) {
        const int x = bx + edges[i] % TW, y = by + edges[i] / TW;
        out[(size_t)y * im.W + x] = fxaaEdge(tile, x, y, contrastThreshold, relativeThreshold, subpixelBlending);
    }
}

}  // namespace

namespace sgi_launch {

hipError_t taaHistory(const float* taa, long n, float* prev, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    const long n3 = 3 * n;
    if (((uintptr_t)taa | (uintptr_t)prev) % 16 == 0)
        hipLaunchKernelGGL(taaHistory4Kernel, dim3((unsigned)((n3 + 1023) / 1024)), dim3(256), 0, s, taa, n3, prev);
    else
        hipLaunchKernelGGL(taaHistoryKernel, dim3((unsigned)((n3 + 255) / 256)), dim3(256), 0, s, taa, n3, prev);
    return hipGetLastError();
}

hipError_t fxaa(const uint32_t* in, int W, int H, float contrastThreshold, float relativeThreshold,
                float subpixelBlending, uint32_t* out, hipStream_t s) {
    if (W <= 0 || H <= 0) return hipSuccess;
    const auto launch = [&](auto kernel, int tw, int th, int threads) {
        const dim3 grid((unsigned)((W + tw - 1) / tw) * (unsigned)((H + th - 1) / th));
        hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, s, FxaaImage{in, W, H}, contrastThreshold,
                           relativeThreshold, subpixelBlending, out);
    };
    // Large tiles list more edges together and have less halo; small ones with a walk's whole reach in LDS
    // finish sooner where the slowest block decides.  Small / large: 360p 12 / 26 us, 1080p 25 / 31,
    // 1440p (3.7 M pixels) 35.4 / 36.5, 4K 70 / 55.
    if ((long)W * H < (4l << 20))
        launch(fxaaKernel<32, 32, 16, 512>, 32, 32, 512);
    else
        launch(fxaaKernel<64, 64, 8, 512>, 64, 64, 512);
    return hipGetLastError();
}

// Pixels below which every code takes the exact form: with few waves the estimate and, for a lane near a tie,
// the pow behind it are the longer chain.  A city's frame, us with the estimate / without: 64x64 6.03 / 3.20,
// 320x180 4.12 / 3.28, 480x270 4.01 / 3.86, 560x315 4.20 / 4.52, 640x360 4.16 / 5.17, 4K 27.2 / 87.7.
constexpr long kTonemapSmall = 150000;

hipError_t tonemap(const float* lit, long n, float gamma, uint32_t* out, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    const float invGamma = 1.0f / gamma;  // 1.0 / gamma (:113)
    // the estimate's error bound holds for these powers
    const bool bounded = invGamma > 0.0f && invGamma <= 16.0f;
    const dim3 grid((unsigned)((n + 255) / 256));
    if (bounded && n >= kTonemapSmall)
        hipLaunchKernelGGL(tonemapKernel<false>, grid, dim3(256), 0, s, lit, n, invGamma,
                           2e-4f * (invGamma > 1.0f ? invGamma : 1.0f), out);
    else
        hipLaunchKernelGGL(tonemapKernel<true>, grid, dim3(256), 0, s, lit, n, invGamma, 0.0f, out);
    return hipGetLastError();
}

}  // namespace sgi_launch
