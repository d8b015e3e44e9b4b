// VPL culling kernels.
//
// cullVisibilityKernel + cullCompactSplitKernel (cullCompactKernel for a few) — viscull_vpls.cs:47-120: per VPL,
// the sun-visibility test through the cascades, then a stable compaction (wave
// ballot + block prefix) of the visible records in ascending input order.
//
// cullTilesKernel — vpl_tiled_deferred_culling_stage1.cs:50-90 and
// _stage2.cs:61-129 fused: one wave per tile.  Stage 1 reconstructs the
// tile's pixels in parallel into LDS and then sums each of the six components
// serially in row-major local order, which is the reference's summation order
// (thread 0's loop), so the tile mean is bit-identical.  Stage 2 evaluates 64
// VPLs per step across the lanes; the K-th ratio is bounded by a histogram, and
// each candidate below the bound finds its place in the list by counting the
// smaller keys (ratio, slot order), which is the reference's stable strict-<
// insertion sort.
//
// colorVplsKernel — vpl_light_color.cs:41-76: one thread per visible slot
// reads the diffuse and distance texels in direction -sun and writes the
// slot's colour and specular position.
#include <hip/hip_fp16.h>

#include "launch.h"
#include "views.h"

namespace {

using namespace sgi_dev;

constexpr int kCullThreads = 1024;

// Per-VPL sun visibility, one thread per VPL over many blocks (each VPL's two
// 4x4 cascade texel blocks are scattered; spreading them over CUs keeps the
// loads in flight on many L1s).
__device__ __forceinline__ void cullVisibilityBody(const CsmArgs& csm, f3 sun, const sgi_vpl* __restrict__ in, int n,
                                                   uint8_t* __restrict__ flags, int i) {
    if (i >= n) return;
    const f3 p = ld3(in[i].position);
    const f3 blends = cascadeBlends(csm, p);
    // the 4x4-block form of the 36 cascade compares (one read per texel; the same value)
    const float shadowFactor = 1.0f - infiniteShadowValueBlock(csm, sun, p, blends, sun, 0.0f);
    flags[i] = shadowFactor < 1.0f ? 1 : 0;
}

__global__ __launch_bounds__(64) void cullVisibilityKernel(CsmArgs csm, f3 sun, const sgi_vpl* __restrict__ in, int n,
                                                          uint8_t* __restrict__ flags) {
    cullVisibilityBody(csm, sun, in, n, flags, blockIdx.x * 64 + threadIdx.x);
}

// Batched: blocks [v * bpv, (v + 1) * bpv) test the VPLs against view v's cascades.
__global__ __launch_bounds__(64) void cullVisibilityViewsKernel(const sgi_batch::ViewDesc* __restrict__ views,
                                                               const sgi_vpl* __restrict__ in, int n, int bpv) {
    const sgi_batch::ViewDesc& d = views[blockIdx.x / bpv];
    cullVisibilityBody(d.csm, ld3(d.fr.sunDir), in, n, d.visFlags, (blockIdx.x % bpv) * 64 + threadIdx.x);
}

// With `all` given, the visible VPLs' atlas entries are written with their records (a frame's and a
// batch's next launch was that copy: 2 us of a 640x360 frame).  out NULL: the indices alone.  A wave may
// write before another has read, so no output may lie over an input (moveVisibleKernel is for those).
// Stable compaction of the flags: wave ballots and a block prefix, in input
// order. The block takes kCompactRounds chunks of kCullThreads items at a
// time: the chunks' flags are loaded together before the one barrier, then
// positions follow chunk, wave and lane order (each chunk's items after all
// earlier chunks') and the visible records are copied. Few registers, so the
// block is placed beside a large kernel running on another stream.
constexpr int kCompactRounds = 4;
__device__ __forceinline__ void cullCompactBody(const sgi_vpl* __restrict__ in, int n, const uint8_t* __restrict__ flags,
                                                sgi_vpl* __restrict__ out, int32_t* __restrict__ visible,
                                                const sgi_atlas_entry* __restrict__ all,
                                                sgi_atlas_entry* __restrict__ entries,
                                                int (*waveCount)[kCullThreads / 64]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    int running = 0;
    for (int c0 = 0; c0 < n; c0 += kCullThreads * kCompactRounds) {
        uint8_t f[kCompactRounds];
#pragma unroll
        for (int k = 0; k < kCompactRounds; ++k) {
            const int i = c0 + k * kCullThreads + (int)threadIdx.x;
            f[k] = i < n ? flags[i] : 0;
        }
        int lanePrefix[kCompactRounds];
#pragma unroll
        for (int k = 0; k < kCompactRounds; ++k) {
            const uint64_t m = __ballot(f[k] != 0);
            lanePrefix[k] = __popcll(m & below);
            if (lane == 0) waveCount[k][wave] = __popcll(m);
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kCompactRounds; ++k) {
            int wavePrefix = 0, total = 0;
            for (int w = 0; w < kCullThreads / 64; ++w) {
                const int c = waveCount[k][w];
                if (w < wave) wavePrefix += c;
                total += c;
            }
            const int pos = running + wavePrefix + lanePrefix[k];
            if (f[k] != 0 && pos < SGI_MAX_TOTAL_VPLS_PER_FRAME) {
                const int i = c0 + k * kCullThreads + (int)threadIdx.x;
                if (out) out[pos] = in[i];
                visible[1 + pos] = i;
                if (all) entries[pos] = all[i];
            }
            running += total;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) visible[0] = running < SGI_MAX_TOTAL_VPLS_PER_FRAME ? running : SGI_MAX_TOTAL_VPLS_PER_FRAME;
}

__global__ __launch_bounds__(kCullThreads) void cullCompactKernel(const sgi_vpl* __restrict__ in, int n,
                                                                  const uint8_t* __restrict__ flags,
                                                                  sgi_vpl* __restrict__ out,
                                                                  int32_t* __restrict__ visible,
                                                                  const sgi_atlas_entry* __restrict__ all,
                                                                  sgi_atlas_entry* __restrict__ entries) {
    __shared__ int waveCount[kCompactRounds][kCullThreads / 64];
    cullCompactBody(in, n, flags, out, visible, all, entries, waveCount);
}

// The same compaction over many blocks of kSplitThreads items, each counting the flags before its own (a
// few KB from L2) instead of waiting for an earlier block.  The copies of 64 B records are then spread
// over the CUs: 4096 VPLs 16 -> 4.8 us.
constexpr int kSplitThreads = 256, kSplitMin = 256;
__global__ __launch_bounds__(kSplitThreads) void cullCompactSplitKernel(const sgi_vpl* __restrict__ in, int n,
                                                                        const uint8_t* __restrict__ flags,
                                                                        sgi_vpl* __restrict__ out,
                                                                        int32_t* __restrict__ visible,
                                                                        const sgi_atlas_entry* __restrict__ all,
                                                                        sgi_atlas_entry* __restrict__ entries) {
    __shared__ int before[kSplitThreads / 64], within[kSplitThreads / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int first = (int)blockIdx.x * kSplitThreads, i = first + (int)threadIdx.x;
    int earlier = 0;
    for (int j = 4 * (int)threadIdx.x; j < first; j += 4 * kSplitThreads)  // flags are 0 or 1, four to a word
        earlier += __popc(*reinterpret_cast<const uint32_t*>(flags + j));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) earlier += __shfl_xor(earlier, o, 64);
    const bool f = i < n && flags[i] != 0;
    const uint64_t m = __ballot(f);
    if (lane == 0) {
        before[wave] = earlier;
        within[wave] = __popcll(m);
    }
    __syncthreads();
    int pos = __popcll(m & ((1ull << lane) - 1ull)), total = 0;
#pragma unroll
    for (int w = 0; w < kSplitThreads / 64; ++w) {
        pos += before[w] + (w < wave ? within[w] : 0);
        total += before[w] + within[w];
    }
    if (f && pos < SGI_MAX_TOTAL_VPLS_PER_FRAME) {
        if (out) out[pos] = in[i];
        visible[1 + pos] = i;
        if (all) entries[pos] = all[i];
    }
    if (threadIdx.x == 0 && blockIdx.x == gridDim.x - 1) visible[0] = min(total, SGI_MAX_TOTAL_VPLS_PER_FRAME);
}

// Batched: one block per view.
__global__ __launch_bounds__(kCullThreads) void cullCompactViewsKernel(const sgi_batch::ViewDesc* __restrict__ views,
                                                                       const sgi_vpl* __restrict__ in, int n,
                                                                       const sgi_atlas_entry* __restrict__ all) {
    __shared__ int waveCount[kCompactRounds][kCullThreads / 64];
    const sgi_batch::ViewDesc& d = views[blockIdx.x];
    cullCompactBody(in, n, d.visFlags, d.vplUpdated, d.visible, all, d.entries, waveCount);
}

// The visible slots' records (in -> out, unless in is NULL) and atlas entries (all -> entries, likewise)
// where an output lies over an input.  One block holds every slot in registers before it writes the first:
// at most 4480, five a thread, 322 KB of the CU's 512 KB, so any overlap gives what apart buffers do.
constexpr int kMoveSlots = (SGI_MAX_TOTAL_VPLS_PER_FRAME + kCullThreads - 1) / kCullThreads;
__global__ __launch_bounds__(kCullThreads) void moveVisibleKernel(const int32_t* __restrict__ visible, int maxCount,
                                                                  const sgi_vpl* in, sgi_vpl* out,
                                                                  const sgi_atlas_entry* all,
                                                                  sgi_atlas_entry* entries) {
    typedef float Part __attribute__((ext_vector_type(4)));
    typedef int Entry __attribute__((ext_vector_type(2), aligned(4)));
    const int count = min(visible[0], maxCount);
    Part rec[kMoveSlots][4];
    Entry ent[kMoveSlots];
#pragma unroll
    for (int k = 0; k < kMoveSlots; ++k) {
        const int slot = k * kCullThreads + (int)threadIdx.x;
        const int i = slot < count ? visible[1 + slot] : 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) rec[k][q] = in && slot < count ? reinterpret_cast<const Part*>(in + i)[q] : Part{};
        ent[k] = all && slot < count ? *reinterpret_cast<const Entry*>(all + i) : Entry{};
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kMoveSlots; ++k) {
        const int slot = k * kCullThreads + (int)threadIdx.x;
        if (in && slot < count) {
#pragma unroll
            for (int q = 0; q < 4; ++q) reinterpret_cast<Part*>(out + slot)[q] = rec[k][q];
        }
        if (all && slot < count) *reinterpret_cast<Entry*>(entries + slot) = ent[k];
    }
}

__global__ void gatherEntriesKernel(const sgi_atlas_entry* __restrict__ all, const int32_t* __restrict__ visible,
                                    int maxCount, sgi_atlas_entry* __restrict__ out) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    const int count = visible[0];
    if (s < count && s < maxCount) out[s] = all[visible[1 + s]];
}

// vpl_light_color.cs:49-74.  The diffuse and distance atlases have one
// geometry (one framebuffer's two attachments), so both lookups of direction
// -sun share one texel offset.  Built with -ffp-contract=off: every product and
// difference is rounded on its own, in the shader's order.
template <int ZFMT>
__global__ __launch_bounds__(256) void colorVplsKernel(CubeArgs diffuse, CubeArgs dist, f3 sun, f3 sunColor,
                                                        float mult, const int32_t* __restrict__ visible,
                                                        int maxCount, const sgi_atlas_entry* __restrict__ entries,
                                                        sgi_vpl* __restrict__ vpls) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    const int count = visible[0];
    if (s >= count || s >= maxCount) return;
    const sgi_atlas_entry e = entries[s];
    const f3 d{-sun.x, -sun.y, -sun.z};
    const uint32_t off = cubeTexelOffset(d, diffuse.res);
    const uint32_t rgb = ((const uint32_t*)cubeLayerBase(diffuse, e.index, e.layer, 4))[off];
    const void* zb = cubeLayerBase(dist, e.index, e.layer, texelBytes(ZFMT));
    float z;
    if constexpr (ZFMT == SGI_TEXEL_F32) z = ((const float*)zb)[off];
    else z = decode16<ZFMT>(((const unsigned short*)zb)[off]);
    sgi_vpl& v = vpls[s];
    const float intensity = v.intensity;
    const float scaled = 1.1f * (v.radius * z);  // 1.1 * magnitude (:53, :71)
    const float c[3] = {(float)(rgb & 0xFFu) / 255.0f, (float)((rgb >> 8) & 0xFFu) / 255.0f,
                        (float)((rgb >> 16) & 0xFFu) / 255.0f};
    const float sc[3] = {sunColor.x, sunColor.y, sunColor.z}, sd[3] = {sun.x, sun.y, sun.z};
    for (int k = 0; k < 3; ++k) {
        v.color[k] = c[k] * sc[k] * intensity * mult;  // color / totalColors (1) * intensity * colorMultiplier (:73)
        v.specularPosition[k] = v.position[k] - scaled * sd[k];
    }
    v.color[3] = 1.0f;
    v.specularPosition[3] = 1.0f;
}

// A tile-culling block's LDS: the per-pixel components that stage 1 sums (six planes at once, three at a
// time for 32x32 tiles), each plane 4 floats longer than the tile so that the summing lanes read different
// banks; then, in the same words, stage 2's histogram (256 counters), compacted slot list (kListCap) and
// ratio codes (a byte per VPL), and over the codes the candidates' keys.  6.5 KB for 8x8 and 16x16 tiles, with
// room for every VPL that a frame may hold.  (Its last 288 B are for the codes past 4192: 16x16 tiles of a
// 1080p frame take 32.4 us instead of 34.1 without them at 512 VPLs, 101.6 and 102.3 at 4096, and, scanning
// twice, 154 instead of 108 at 4400.)
constexpr int kListCap = 512, kKeyCap = 256;
template <int TS>
struct CullLds {
    static constexpr int kStride = TS * TS + 4;
    static constexpr int kPlanes = TS <= 16 ? 6 : 3;
    static constexpr int kCodesAt = 256 + kListCap / 2;  // in words
    static constexpr int kStage2 = kCodesAt + SGI_MAX_TOTAL_VPLS_PER_FRAME / 4;
    static constexpr int kWords = kPlanes * kStride > kStage2 ? kPlanes * kStride : kStage2;
    static constexpr int kCodeCap = (kWords - kCodesAt) * 4;
    static_assert(kCodesAt % 2 == 0 && kKeyCap * 8 <= kCodeCap, "the keys lie over the codes");
};

// The largest code of a VPL that is kept; 255 marks one that certainly is no candidate.
constexpr uint32_t kMaxCode = 254;
// Code of an estimated ratio: its bucket of the histogram, a bucket lower within 2^-16 above an edge.
__device__ __forceinline__ uint32_t ratioCode(float r) {
    if (r > 1.0f + 0x1p-16f) return 255u;
    const float b = r * (256.0f * (1.0f - 0x1p-16f));
    return b > 0.0f ? (b < (float)kMaxCode ? (uint32_t)b : kMaxCode) : 0u;  // a NaN is kept and fails later
}

template <int TS>
__device__ __forceinline__ void cullTileBody(const GbufArgs& g, const FrameArgs& fr, int t, int tilesX, int K,
                                             const sgi_vpl* __restrict__ vpls, const int32_t* __restrict__ visible,
                                             int remap, sgi_tile_stage1* __restrict__ stage1,
                                             int32_t* __restrict__ tiles, float* comp, float* sums) {
    using Lds = CullLds<TS>;
    constexpr int NPX = TS * TS, S = Lds::kStride;
    const int tx = t % tilesX, ty = t / tilesX;
    const int lane = threadIdx.x;
    const int x0 = tx * TS, y0 = ty * TS;
    const int vw = min(TS, g.W - x0), vh = min(TS, g.H - y0);

    // Stage 1: per-pixel world positions and decoded normals, each summed by the reference's
    // serial loop (one component per lane; a chain of 256 dependent additions for a 16x16 tile, so
    // all six run side by side and a whole tile reads four values at a time).
    constexpr int kPasses = 6 / Lds::kPlanes;
    for (int pass = 0; pass < kPasses; ++pass) {
        for (int l = lane; l < NPX; l += 64) {
            const int lx = l % TS, ly = l / TS;
            if (lx < vw && ly < vh) {
                const int x = x0 + lx, y = y0 + ly;
                const size_t p = (size_t)y * g.W + x;
                float* c = comp + l;
                if (kPasses == 1 || pass == 0) {
                    const f3 v = worldPositionFromDepth(texelCentre(x, g.W), texelCentre(y, g.H), g.depth[p], fr.invPV);
                    c[0] = v.x; c[S] = v.y; c[2 * S] = v.z;
                }
                if (kPasses == 1 || pass == 1) {
                    const f3 v = gNormal(g, p);
                    if (kPasses == 1) c += 3 * S;
                    c[0] = v.x; c[S] = v.y; c[2 * S] = v.z;
                }
            }
        }
        __syncthreads();
        if (lane < Lds::kPlanes) {
            const float* c = comp + lane * S;
            float s = 0.0f;
            if (vw == TS && vh == TS) {
#pragma unroll 8
                for (int i = 0; i < NPX / 4; ++i) {
                    const float4 v = reinterpret_cast<const float4*>(c)[i];
                    s += v.x;
                    s += v.y;
                    s += v.z;
                    s += v.w;
                }
            } else {
                for (int ly = 0; ly < vh; ++ly)
                    for (int lx = 0; lx < vw; ++lx) s += c[ly * TS + lx];
            }
            sums[Lds::kPlanes * pass + lane] = s;
        }
        __syncthreads();
    }
    const float cnt = (float)(vw * vh);
    const f3 P = f3{sums[0], sums[1], sums[2]} / cnt;
    const f3 Nrm = normalize(f3{sums[3], sums[4], sums[5]} / cnt);
    if (stage1 && lane == 0) {
        sgi_tile_stage1 o;
        o.averageLocalPosition[0] = P.x; o.averageLocalPosition[1] = P.y; o.averageLocalPosition[2] = P.z;
        o.averageLocalPosition[3] = 1.0f;
        o.averageLocalNormal[0] = Nrm.x; o.averageLocalNormal[1] = Nrm.y; o.averageLocalNormal[2] = Nrm.z;
        o.averageLocalNormal[3] = 1.0f;
        stage1[t] = o;
    }

    const int numVisible = visible[0];
    // Stage 2a: an upper bound of the K-th smallest candidate ratio, so that stage 2 inserts
    // little beyond the final list. A
    // 256-bucket histogram over [0, 1) of estimated ratios (hardware sqrt and reciprocal: within
    // 2^-21 relative of the correctly rounded ratio) counts only VPLs that are certainly
    // candidates (the exact side test, estimate <= 1 - 2^-18). If K of them fall in buckets up to
    // b, K candidates have ratios below T = (b + 1) / 256 times (1 + 2^-21), so the K-th smallest
    // ratio lies below cap = T (1 + 2^-18): stage 2, started with cap in every slot instead of
    // FLT_MAX, inserts in slot order only the candidates below cap, a subsequence that holds the
    // whole stable top-K, and so ends with the same list. The histogram reuses comp (free once
    // the sums are formed).
    uint32_t* hist = reinterpret_cast<uint32_t*>(comp);
    uint8_t* codes = reinterpret_cast<uint8_t*>(hist + Lds::kCodesAt);
    const bool haveCodes = numVisible <= Lds::kCodeCap;  // unless the caller counts more than a frame holds
    for (int i = lane; i < 256; i += 64) hist[i] = 0u;
    __syncthreads();
    for (int b = 0; b < numVisible; b += 64) {
        const int s = b + lane;
        if (s < numVisible) {
            const f3 lmf = ld3(vpls[s].position) - P;
            uint32_t code = 255u;
            if (!(dot(Nrm, lmf) < 0.0f)) {
                const float r = __builtin_amdgcn_sqrtf(dot(lmf, lmf)) * __builtin_amdgcn_rcpf(vpls[s].radius);
                if (r >= 0.0f && r <= 1.0f - 0x1p-18f) atomicAdd(&hist[(int)(r * 256.0f)], 1u);
                code = ratioCode(r);
            }
            if (haveCodes) codes[s] = (uint8_t)code;
        }
    }
    __syncthreads();
    float cap = kFLOAT_MAX;
    uint32_t keepCode = kMaxCode;
    {
        const uint32_t h0 = hist[4 * lane], h1 = hist[4 * lane + 1], h2 = hist[4 * lane + 2], h3 = hist[4 * lane + 3];
        const uint32_t mine = h0 + h1 + h2 + h3;
        uint32_t incl = mine;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t v = __shfl_up(incl, o, 64);
            if (lane >= o) incl += v;
        }
        const uint64_t reach = __ballot(incl >= (uint32_t)K);
        if (reach) {
            const int L = __builtin_ctzll(reach);
            const uint32_t e0 = incl - mine;
            const int within = e0 + h0 >= (uint32_t)K ? 0 : (e0 + h0 + h1 >= (uint32_t)K ? 1 : (e0 + h0 + h1 + h2 >= (uint32_t)K ? 2 : 3));
            const int bucket = 4 * L + __builtin_amdgcn_readlane(within, L);
            cap = (float)(bucket + 1) * (1.0f / 256.0f) * (1.0f + 0x1p-18f);
            keepCode = min((uint32_t)bucket, kMaxCode);
        }
    }

    // Stage 2b: the slots that may lie below cap, compacted in slot order after the histogram: by
    // their codes, or past kCodeCap VPLs by the side test and the estimate again.  A ratio below cap
    // is at most 2^-17 above its bucket's upper edge, so its code is at most the bucket.  With more
    // slots than the list holds, stage 2 scans every slot.
    uint16_t* list = reinterpret_cast<uint16_t*>(hist + 256);
    int nList = 0;
    for (int b = 0; b < numVisible; b += 64) {
        const int s = b + lane;
        bool keep = false;
        if (s < numVisible) {
            if (haveCodes) {
                keep = codes[s] <= keepCode;
            } else {
                const f3 lmf = ld3(vpls[s].position) - P;
                keep = !(dot(Nrm, lmf) < 0.0f) &&
                       ratioCode(__builtin_amdgcn_sqrtf(dot(lmf, lmf)) * __builtin_amdgcn_rcpf(vpls[s].radius)) <= keepCode;
            }
        }
        const uint64_t m = __ballot(keep);
        const int pos = nList + __popcll(m & ((1ull << lane) - 1ull));
        if (keep && pos < kListCap) list[pos] = (uint16_t)s;
        nList += __popcll(m);
    }
    const bool useList = nList <= kListCap;
    const int n = useList ? nList : numVisible;
    __syncthreads();

    // Stage 2c: the exact candidates below cap, each a key (the ratio's bits, then its place in slot
    // order): the list wanted is the K smallest keys in order, and a candidate's place in it is the
    // number of smaller keys.  Counting them takes two instructions a pair of 64 candidates and key;
    // inserting one by one took some twenty per candidate.  With the sums side by side and the codes: 1080p,
    // 1024 VPLs 64 -> 45 us, 4096 172 -> 109; eight 720p views, 512 VPLs 83 -> 57; 640x360, 64 VPLs 16 -> 10.
    uint64_t* keys = reinterpret_cast<uint64_t*>(codes);
    if (useList) {
        int m = 0;
        bool ordered = true;  // the bits order non-negative ratios
        for (int b = 0; b < n; b += 64) {
            const int i = b + lane;
            bool cand = false;
            float ratio = 0.0f;
            int s = 0;
            if (i < n) {
                s = list[i];
                const f3 lmf = ld3(vpls[s].position) - P;
                if (!(dot(Nrm, lmf) < 0.0f)) {
                    ratio = length(lmf) / vpls[s].radius;
                    cand = !(ratio > 1.0f) && ratio < cap;
                }
            }
            const uint64_t mask = __ballot(cand);
            ordered &= __ballot(cand && (__float_as_uint(ratio) >> 31)) == 0;
            const int pos = m + __popcll(mask & ((1ull << lane) - 1ull));
            if (cand && pos < kKeyCap)
                keys[pos] = (uint64_t)__float_as_uint(ratio) << 32 | (uint32_t)pos << 16 | (uint32_t)s;
            m += __popcll(mask);
        }
        if (ordered && m <= kKeyCap) {
            __syncthreads();
            int32_t* rec = tiles + (size_t)t * (1 + K);
            if (lane == 0) rec[0] = min(m, K);
            for (int q = 0; q < m; q += 64) {
                const uint64_t mine = q + lane < m ? keys[q + lane] : ~0ull;
                int rank = 0;
#pragma unroll 4
                for (int j = 0; j < m; ++j) rank += keys[j] < mine ? 1 : 0;
                if (q + lane < m && rank < K) {
                    const int s = (int)(mine & 0xFFFFu);
                    rec[1 + rank] = remap ? visible[1 + s] : s;
                }
            }
            return;
        }
    }

    // Otherwise (more candidates than keys, or a negative radius): sorted top-K in lane registers, over the
    // compacted slots or every slot.
    float myDist = cap;
    int myIdx = 0;
    int count = 0;
    for (int b = 0; b < n; b += 64) {
        const int i = b + lane;
        const int s = i < n ? (useList ? (int)list[i] : i) : 0;
        bool cand = false;
        float ratio = 0.0f;
        if (i < n) {
            const f3 lmf = ld3(vpls[s].position) - P;
            const float side = dot(Nrm, lmf);
            if (!(side < 0.0f)) {
                const float distance = length(lmf);
                ratio = distance / vpls[s].radius;
                cand = !(ratio > 1.0f) && ratio == ratio;
            }
        }
        // K-1 and c are wave-uniform, so the broadcasts are v_readlane
        const float thr = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(myDist), K - 1));
        uint64_t m = __ballot(cand && ratio < thr);
        while (m) {
            const int c = __builtin_ctzll(m);
            m &= m - 1;
            const float r = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ratio), c));
            const float thrNow = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(myDist), K - 1));
            if (!(r < thrNow)) continue;
            const int p = __popcll(__ballot(lane < K && myDist <= r));
            const int sc = __builtin_amdgcn_readlane(s, c);
            // lane i takes lane i-1's entry: a DPP wave shift, no LDS round trip
            const float upD = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(myDist), __float_as_int(myDist),
                                                                         0x138, 0xF, 0xF, false));
            const int upI = __builtin_amdgcn_update_dpp(myIdx, myIdx, 0x138, 0xF, 0xF, false);
            if (lane < K) {
                if (lane > p) {
                    myDist = upD;
                    myIdx = upI;
                } else if (lane == p) {
                    myDist = r;
                    myIdx = remap ? visible[1 + sc] : sc;
                }
            }
            count = count + 1 < K ? count + 1 : K;
        }
    }
    int32_t* rec = tiles + (size_t)t * (1 + K);
    if (lane == 0) rec[0] = count;
    if (lane < count) rec[1 + lane] = myIdx;
}

template <int TS>
__global__ __launch_bounds__(64) void cullTilesKernel(GbufArgs g, FrameArgs fr, int tilesX, int nTiles, int K,
                                                      const sgi_vpl* __restrict__ vpls,
                                                      const int32_t* __restrict__ visible, int remap,
                                                      sgi_tile_stage1* __restrict__ stage1,
                                                      int32_t* __restrict__ tiles) {
    __shared__ __align__(16) float comp[CullLds<TS>::kWords];
    __shared__ float sums[6];
    const int t = (int)xcdSpread(blockIdx.x);
    if (t < nTiles) cullTileBody<TS>(g, fr, t, tilesX, K, vpls, visible, remap, stage1, tiles, comp, sums);
}

// Batched: the tiles of every view, numbered view after view.
template <int TS>
__global__ __launch_bounds__(64) void cullTilesViewsKernel(const sgi_batch::ViewDesc* __restrict__ views,
                                                           int numViews, int totalTiles, int K) {
    __shared__ __align__(16) float comp[CullLds<TS>::kWords];
    __shared__ float sums[6];
    const int gt = (int)xcdSpread(blockIdx.x);
    if (gt >= totalTiles) return;
    const sgi_batch::ViewDesc& d = views[sgi_batch::findView<sgi_batch::kTiles>(views, numViews, gt)];
    cullTileBody<TS>(d.g, d.fr, gt - d.tileStart, d.tilesX, K, d.vplUpdated, d.visible, 0, nullptr, d.tiles, comp,
                     sums);
}

}  // namespace

namespace sgi_launch {

// Whether na elements at a and nb at b share memory.
template <class A, class B>
static bool overlap(const A* a, int na, const B* b, int nb) {
    return (uintptr_t)a < (uintptr_t)(b + nb) && (uintptr_t)b < (uintptr_t)(a + na);
}

hipError_t cullGlobal(const CsmArgs& csm, const FrameArgs& fr, const sgi_vpl* in, int n, sgi_vpl* out,
                      int32_t* visible, uint8_t* flags, const sgi_atlas_entry* all, sgi_atlas_entry* entries,
                      hipStream_t s) {
    if (n > 0) {
        hipLaunchKernelGGL(cullVisibilityKernel, dim3((n + 63) / 64), dim3(64), 0, s, csm, ld3(fr.sunDir), in, n, flags);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    // an output over an input waits for the indices: it is written by moveVisibleKernel, not as the
    // compaction goes (entries may also take the place of the input records, which are done with by then)
    const int cap = min(n, SGI_MAX_TOTAL_VPLS_PER_FRAME);
    const bool moveRecords = overlap(out, cap, in, n);
    const bool moveEntries = all && (overlap(entries, cap, all, n) || overlap(entries, cap, in, n));
    sgi_vpl* const out0 = moveRecords ? nullptr : out;
    const sgi_atlas_entry* const all0 = moveEntries ? nullptr : all;
    // one block of 1024 threads for a few: 1024 VPLs 5.5 us in one block, 4.7 split
    if (n > kSplitMin)
        hipLaunchKernelGGL(cullCompactSplitKernel, dim3((n + kSplitThreads - 1) / kSplitThreads), dim3(kSplitThreads),
                           0, s, in, n, flags, out0, visible, all0, entries);
    else
        hipLaunchKernelGGL(cullCompactKernel, dim3(1), dim3(kCullThreads), 0, s, in, n, flags, out0, visible, all0,
                           entries);
    if (moveRecords || moveEntries)
        hipLaunchKernelGGL(moveVisibleKernel, dim3(1), dim3(kCullThreads), 0, s, visible, cap,
                           moveRecords ? in : nullptr, out, moveEntries ? all : nullptr, entries);
    return hipGetLastError();
}

hipError_t gatherVisibleEntries(const sgi_atlas_entry* all, const int32_t* visible, int maxCount, sgi_atlas_entry* out,
                                hipStream_t s) {
    if (maxCount <= 0) return hipSuccess;
    // how many entries `all` holds is not given: as many as there may be VPLs, so an output close behind goes
    // the safe way too (64 slots 1.7 -> 2.2 us, 4096 1.7 -> 3.3)
    if (overlap(out, maxCount, all, SGI_MAX_TOTAL_VPLS_BEFORE_CULLING))
        hipLaunchKernelGGL(moveVisibleKernel, dim3(1), dim3(kCullThreads), 0, s, visible, maxCount, nullptr, nullptr,
                           all, out);
    else
        hipLaunchKernelGGL(gatherEntriesKernel, dim3((maxCount + 255) / 256), dim3(256), 0, s, all, visible, maxCount,
                           out);
    return hipGetLastError();
}

hipError_t cullTiles(const GbufArgs& g, const FrameArgs& fr, int tileSize, int tilesX, int tilesY, int K,
                     const sgi_vpl* vpls, const int32_t* visible, int remap, sgi_tile_stage1* stage1, int32_t* tiles,
                     hipStream_t s) {
    const int nTiles = tilesX * tilesY;
    switch (tileSize) {
        case 8:
            hipLaunchKernelGGL(cullTilesKernel<8>, dim3(spreadBlocks(nTiles)), dim3(64), 0, s, g, fr, tilesX, nTiles, K, vpls,
                               visible, remap, stage1, tiles);
            break;
        case 16:
            hipLaunchKernelGGL(cullTilesKernel<16>, dim3(spreadBlocks(nTiles)), dim3(64), 0, s, g, fr, tilesX, nTiles, K, vpls,
                               visible, remap, stage1, tiles);
            break;
        case 32:
            hipLaunchKernelGGL(cullTilesKernel<32>, dim3(spreadBlocks(nTiles)), dim3(64), 0, s, g, fr, tilesX, nTiles, K, vpls,
                               visible, remap, stage1, tiles);
            break;
        default:
            return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t cullGlobalViews(const sgi_batch::ViewDesc* views, int numViews, const sgi_vpl* in, int n,
                           const sgi_atlas_entry* all, hipStream_t s) {
    if (n > 0) {
        const int bpv = (n + 63) / 64;
        hipLaunchKernelGGL(cullVisibilityViewsKernel, dim3(numViews * bpv), dim3(64), 0, s, views, in, n, bpv);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(cullCompactViewsKernel, dim3(numViews), dim3(kCullThreads), 0, s, views, in, n, all);
    return hipGetLastError();
}

hipError_t colorVpls(const sgi_dev::CubeArgs& diffuse, const sgi_dev::CubeArgs& dist, int distFormat,
                     const sgi_dev::FrameArgs& fr, float mult, const int32_t* visible, int maxCount,
                     const sgi_atlas_entry* entries, sgi_vpl* vpls, hipStream_t s) {
    if (maxCount <= 0) return hipSuccess;
    const f3 sun{fr.sunDir[0], fr.sunDir[1], fr.sunDir[2]};
    const f3 col{fr.sunColor[0], fr.sunColor[1], fr.sunColor[2]};
    const dim3 grid((unsigned)((maxCount + 255) / 256));
    if (distFormat == SGI_TEXEL_F16)
        hipLaunchKernelGGL(colorVplsKernel<SGI_TEXEL_F16>, grid, dim3(256), 0, s, diffuse, dist, sun, col, mult,
                           visible, maxCount, entries, vpls);
    else if (distFormat == SGI_TEXEL_UNORM16)
        hipLaunchKernelGGL(colorVplsKernel<SGI_TEXEL_UNORM16>, grid, dim3(256), 0, s, diffuse, dist, sun, col, mult,
                           visible, maxCount, entries, vpls);
    else
        hipLaunchKernelGGL(colorVplsKernel<SGI_TEXEL_F32>, grid, dim3(256), 0, s, diffuse, dist, sun, col, mult,
                           visible, maxCount, entries, vpls);
    return hipGetLastError();
}

hipError_t cullTilesViews(const sgi_batch::ViewDesc* views, int numViews, int totalTiles, int tileSize, int K,
                          hipStream_t s) {
    switch (tileSize) {
        case 8:
            hipLaunchKernelGGL(cullTilesViewsKernel<8>, dim3(spreadBlocks(totalTiles)), dim3(64), 0, s, views, numViews, totalTiles, K);
            break;
        case 16:
            hipLaunchKernelGGL(cullTilesViewsKernel<16>, dim3(spreadBlocks(totalTiles)), dim3(64), 0, s, views, numViews, totalTiles,
                               K);
            break;
        case 32:
            hipLaunchKernelGGL(cullTilesViewsKernel<32>, dim3(spreadBlocks(totalTiles)), dim3(64), 0, s, views, numViews, totalTiles,
                               K);
            break;
        default:
            return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace sgi_launch
