// The shadow-map producers of the pass's inputs: the VPL cube pre-pass and the
// sun cascades' depth render, from world-space triangles.
//
// VPL distance / diffuse cube producer — the reference's shadow pre-pass for
// virtual point lights (StratusRendererBackend.cpp:1426-1575): per updated
// light, the six faces rendered with perspective(90 deg, 1, near, far) x
// lookAt(pos, pos + axis, up) (:873-886, :1450), each face's depth layer
// cleared to 1 and its colour layer to 0 (:1453-1459), then every static
// triangle drawn with gl_FragDepth = saturate(|P - L| / farPlane) and colour =
// its base colour (shadowVpl.fs:17-37 through shadow.vs:22-33), depth test
// LESS, into layer * 6 + face of the light's atlas entry (:1511-1518).
//
// The six lookAt bases are signed permutations of the axes, so the face ray of
// texel (i, j) — the ray through its pixel centre — is exactly the GL
// major-axis table's direction with major component +-1 (window pixel (i, j)
// of face f is cube texel (i, j) of face f).  A fragment at that texel exists
// where the ray meets a triangle: with a, b, c the vertices relative to the
// light, e_k = d . (b x c, c x a, a x b) all of one sign, the view depth
// t = det(a, b, c) / (e0 + e1 + e2) within [near, far] (GL clipping), and the
// fragment's distance t |d|.  The depth test keeps the smallest stored value,
// the first triangle in draw order on ties (LESS), exactly as a per-texel
// minimum over the triangles in their order.
//
// MI355X structure: (1) one thread per (light, triangle) tests the six faces
// and appends the triangle to each face it can overlap (one atomic per block
// and face), with the 32x32-texel regions its projection can touch; (2) each
// 16x16 tile of a face is drawn by one wave (or by four, each a quarter of the
// list, where it is long and the tiles are few): the wave picks
// its triangles from the face list by integer range tests (4 B per triangle),
// sets up 64 at a time (edge vectors in face axes), draws those of a few
// texels one texel per lane into LDS, and tests its texels, 2x2 per lane,
// against the others, near ones first and none that lie behind every texel.
// Lists are in no order: the smaller index wins equal values, which is the
// LESS rule.  Culling is conservative (region margins as the frustum test's
// 2^-12, edge margins from the rounding bound of the edge functions); the
// per-texel test alone decides every value, in the restatement's operation
// order (-ffp-contract=off).  A mesh of a few triangles takes one launch without
// lists (cubeShortKernel).
//
// What bounds it: the latency of a wave's serial triangles, then VALU issue.
// Towards the horizon a region holds more than a thousand triangles of a few
// texels, where scanning the face's triangles with the full frustum test in
// every 32x32 region and testing all its texels against each survivor spent
// most of its time.  24012 triangles, 256^2 cubes: 96 lights 3.51 -> 1.00 ms
// (lists 0.094 -> 0.055, drawing 3.41 -> 0.94), 5 lights with colour 0.98 ->
// 0.15 ms (0.047 -> 0.011, 0.93 -> 0.14).
#include "launch.h"

namespace {

using namespace sgi_dev;

constexpr int kListBlock = 256;
constexpr int kRegion = 32;   // texels per region edge: what the lists sort triangles by
constexpr int kTile = 16;     // texels per tile edge: one wave, 2x2 texels per lane
constexpr int kSmall = 16;    // texels of a bounding box that are drawn texel by texel
constexpr int kScan = 512;    // list entries a wave scans at a time

__global__ void clearIntsKernel(int32_t* p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// First / last region a coordinate range [lo, hi] in [-1, 1] texture units can touch (NaN: all).
__device__ __forceinline__ int firstRegion(float lo, int res, int regions) {
    const float x = floorf((lo + 1.0f) * ((float)res * (0.5f / kRegion)));
    return x > 0.0f ? (x < (float)(regions - 1) ? (int)x : regions - 1) : 0;
}
__device__ __forceinline__ int lastRegion(float hi, int res, int regions) {
    const float x = floorf((hi + 1.0f) * ((float)res * (0.5f / kRegion)));
    return x < (float)(regions - 1) ? (x > 0.0f ? (int)x : 0) : regions - 1;
}

// LDS of one wave, ordered among its own lanes.
__device__ __forceinline__ void waveSync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Maximum over the wave's lanes, in every lane (DPP row shifts and broadcasts).
template <int CTRL>
__device__ __forceinline__ float maxDpp(float v) {
    return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL, 0xF, 0xF, false)));
}
__device__ __forceinline__ float waveMax(float v) {
    v = maxDpp<0x118>(maxDpp<0x114>(maxDpp<0x112>(maxDpp<0x111>(v))));
    v = maxDpp<0x143>(maxDpp<0x142>(v));
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

__device__ __forceinline__ int waveInclusive(int v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int up = __shfl_up(v, o, 64);
        if (lane >= o) v += up;
    }
    return v;
}

// A wave's candidates: positions of list entries whose ranges `touches` accepts, in cand[0 .. have).
// next() scans on, kScan entries at a time (each lane by 16-byte loads, all in flight; `ranges`
// 16-byte aligned and readable up to a multiple of four entries), until 64 are held or the list ends,
// and hands out up to 64 of them.  SLICES waves share a list, each taking every SLICES-th kScan.
constexpr int kCand = 63 + kScan;
template <class R, int SLICES>
struct Candidates {
    const R* ranges;
    int n, pos, have;
    int32_t* cand;
    template <class TOUCH>
    __device__ __forceinline__ int next(TOUCH touches) {
        constexpr int kPer = 16 / sizeof(R), kLoads = kScan / (64 * kPer);
        struct alignas(16) Four {
            R r[kPer];
        };
        const int lane = threadIdx.x & 63;
        while (have < 64 && pos < n) {
            Four v[kLoads];
#pragma unroll
            for (int k = 0; k < kLoads; ++k) {
                const int i = pos + (k * 64 + lane) * kPer;
                if (i < n) v[k] = *reinterpret_cast<const Four*>(ranges + i);
            }
            uint32_t hits = 0;
#pragma unroll
            for (int k = 0; k < kLoads; ++k)
#pragma unroll
                for (int j = 0; j < kPer; ++j) {
                    const int i = pos + (k * 64 + lane) * kPer + j;
                    if (i < n && touches(v[k].r[j])) hits |= 1u << (k * kPer + j);
                }
            if (__ballot(hits != 0)) {
                const int mine = __popc(hits), incl = waveInclusive(mine);
                int slot = have + incl - mine;
                while (hits) {
                    const int b = __builtin_ctz(hits);
                    hits &= hits - 1;
                    cand[slot++] = pos + ((b / kPer) * 64 + lane) * kPer + b % kPer;
                }
                have += __builtin_amdgcn_readlane(incl, 63);
            }
            pos += SLICES * kScan;
        }
        const int out = min(have, 64);
        have -= out;  // the last ones: cand[have .. have + out)
        waveSync();
        return out;
    }
};

// A point relative to the light in face f's coordinates: m along the face's
// axis, (s, t) with s / m, t / m the face's NDC-like coordinates.  Texel (i, j)'s
// ray is the point (m, s, t) = (1, 2 (i + 0.5) / res - 1, 2 (j + 0.5) / res - 1):
// the GL major-axis table inverted.
__device__ __forceinline__ void faceCoords(int f, f3 p, float& m, float& s, float& t) {
    switch (f) {
        case 0: m = p.x; s = -p.z; t = -p.y; break;
        case 1: m = -p.x; s = p.z; t = -p.y; break;
        case 2: m = p.y; s = p.x; t = p.z; break;
        case 3: m = -p.y; s = p.x; t = -p.z; break;
        case 4: m = p.z; s = p.x; t = -p.y; break;
        default: m = -p.z; s = -p.x; t = -p.y; break;
    }
}

__device__ __forceinline__ f3 cross3(f3 a, f3 b) {
    return f3{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

// True when no point of the triangle can lie inside the frustum
// s_lo m <= s <= s_hi m, t_lo m <= t <= t_hi m, near <= m <= far (all three
// vertices strictly beyond one plane, by a relative margin of 2^-12).
__device__ __forceinline__ bool outsideFrustum(const float m[3], const float s[3], const float t[3], float sLo,
                                               float sHi, float tLo, float tHi, float nearP, float farP) {
    bool o0 = true, o1 = true, o2 = true, o3 = true, o4 = true, o5 = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float mar = (fabsf(m[k]) + fabsf(s[k]) + fabsf(t[k])) * 0x1p-12f;
        o0 = o0 && (s[k] - sLo * m[k] < -mar);
        o1 = o1 && (sHi * m[k] - s[k] < -mar);
        o2 = o2 && (t[k] - tLo * m[k] < -mar);
        o3 = o3 && (tHi * m[k] - t[k] < -mar);
        o4 = o4 && (m[k] < nearP - mar);
        o5 = o5 && (m[k] > farP + mar);
    }
    return o0 || o1 || o2 || o3 || o4 || o5;
}

struct CubeJob {
    const float* pos;        // [count][3][3]
    const uint32_t* colors;  // [count] or NULL
    int count;
    const sgi_vpl* vpls;
    const int32_t* updates;  // [numUpdates] VPL indices
    int first;               // first update of this batch
    int batch;               // updates in this batch
    const sgi_atlas_entry* entries;
    float nearPlane;
    int cull;                // SGI_CULLING_* of the meshes
    int stride;              // count rounded up to a multiple of 4
    uint32_t* ranges;        // [batch][6][stride]: the regions an entry touches (x0, x1, y0, y1 bytes)
    int32_t* tris;           // [batch][6][stride]: its triangle
    int32_t* listCounts;     // [batch][6]
};

__device__ __forceinline__ f3 vertexRel(const float* pos, int k, int v, f3 L) {
    const float* q = pos + (size_t)k * 9 + v * 3;
    return f3{q[0] - L.x, q[1] - L.y, q[2] - L.z};
}

// The face culling of SetCullState (StratusRendererBackend.cpp:901-918) for a
// triangle seen from the light: with a, b, c relative to the light,
// V = a . (b x c) = (P - L) . n for n the winding's normal, so the triangle is
// counter-clockwise in window space (its front under glFrontFace(GL_CCW)) when
// V < 0.  The cube faces' views are rotations and their projections keep
// orientation, so window winding is the world winding seen from the light.
__device__ __forceinline__ bool culledFromLight(int cull, float V) {
    if (cull == SGI_CULLING_CCW) return !(V < 0.0f);
    if (cull == SGI_CULLING_CW) return !(V > 0.0f);
    return false;
}

// (1) per (light, triangle): the faces the triangle may overlap, with the regions of each face it
// may touch.  A region is inside the range unless all three vertices lie beyond one of its side
// planes by outsideFrustum's margin (widened by 2^-8 of itself over both forms' rounding); a
// triangle that reaches behind the light along the face's axis is given every region.
__global__ __launch_bounds__(kListBlock) void cubeFaceListKernel(CubeJob job, int res, int regions) {
    const int u = blockIdx.y, k = blockIdx.x * kListBlock + (int)threadIdx.x;
    const sgi_vpl& v = job.vpls[job.updates[job.first + u]];
    const f3 L{v.position[0], v.position[1], v.position[2]};
    const float farP = v.farPlane;
    f3 p[3];
    bool facing = false;
    if (k < job.count) {
        for (int i = 0; i < 3; ++i) p[i] = vertexRel(job.pos, k, i, L);
        const float V = dot(p[0], cross3(p[1], p[2]));
        // V = 0 (the light in the triangle's plane) gives no fragment: its view depth is 0
        facing = (V < 0.0f || V > 0.0f) && !culledFromLight(job.cull, V);
    }
    // the six faces' ballots first, then one atomic per (block, face), all in flight together
    __shared__ int waveCount[6][kListBlock / 64], faceBase[6];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t ranges[6];
    uint64_t bal[6];
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        float m[3], s[3], t[3];
        ranges[f] = 0u;
        bool keep = false;
        if (facing) {
            for (int i = 0; i < 3; ++i) faceCoords(f, p[i], m[i], s[i], t[i]);
            keep = !outsideFrustum(m, s, t, -1.0f, 1.0f, -1.0f, 1.0f, job.nearPlane, farP);
        }
        if (keep) {
            int x0 = 0, x1 = regions - 1, y0 = 0, y1 = regions - 1;
            if (m[0] > 1e-20f && m[1] > 1e-20f && m[2] > 1e-20f) {
                float sLo = kFLOAT_MAX, sHi = -kFLOAT_MAX, tLo = kFLOAT_MAX, tHi = -kFLOAT_MAX;
                for (int i = 0; i < 3; ++i) {
                    const float mar = (fabsf(m[i]) + fabsf(s[i]) + fabsf(t[i])) * (0x1p-12f + 0x1p-20f);
                    sLo = gmin((s[i] - mar) / m[i], sLo);
                    sHi = gmax((s[i] + mar) / m[i], sHi);
                    tLo = gmin((t[i] - mar) / m[i], tLo);
                    tHi = gmax((t[i] + mar) / m[i], tHi);
                }
                x0 = firstRegion(sLo - 0x1p-18f, res, regions);
                x1 = lastRegion(sHi + 0x1p-18f, res, regions);
                y0 = firstRegion(tLo - 0x1p-18f, res, regions);
                y1 = lastRegion(tHi + 0x1p-18f, res, regions);
            }
            ranges[f] = (uint32_t)x0 | (uint32_t)x1 << 8 | (uint32_t)y0 << 16 | (uint32_t)y1 << 24;
        }
        bal[f] = __ballot(keep);
        if (lane == 0) waveCount[f][wave] = __popcll(bal[f]);
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        int total = 0;
        for (int w = 0; w < kListBlock / 64; ++w) total += waveCount[threadIdx.x][w];
        faceBase[threadIdx.x] = total ? atomicAdd(job.listCounts + u * 6 + threadIdx.x, total) : 0;
    }
    __syncthreads();
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        if (!(bal[f] >> lane & 1)) continue;
        int slot = faceBase[f] + __popcll(bal[f] & ((1ull << lane) - 1ull));
        for (int w = 0; w < wave; ++w) slot += waveCount[f][w];
        const size_t e = ((size_t)u * 6 + f) * job.stride + slot;
        job.ranges[e] = ranges[f];
        job.tris[e] = k;
    }
}

// Stored value of a fragment at v = dist / far (>= 0) as an ordered key: the
// depth attachment's own representation, so that key order is LESS's order.
template <int FMT>
__device__ __forceinline__ uint32_t depthKey(float v) {
    v = v < 1.0f ? v : 1.0f;  // saturate (v >= 0)
    if constexpr (FMT == SGI_TEXEL_F32) return __float_as_uint(v);
    else if constexpr (FMT == SGI_TEXEL_F16) return (uint32_t)__half_as_ushort(__float2half_rn(v));
    else return (uint32_t)rintf(v * 65535.0f);
}

// Values v and w further apart than keyCell(max(v, w)) store different keys (or differ by more than
// the estimates' error, 2^-18 relative): the representation's step.
template <int FMT>
__device__ __forceinline__ float keyCell(float v) {
    if constexpr (FMT == SGI_TEXEL_F32) return v * 0x1p-18f;
    else if constexpr (FMT == SGI_TEXEL_F16) return __builtin_fmaf(v, 0x1p-10f + 0x1p-18f, 0x1p-23f);
    else return __builtin_fmaf(v, 0x1p-18f, 1.0f / 65535.0f);
}

// A triangle set up for a face: the edge vectors b x c, c x a, a x b in the face's axes with the
// signs of faceCoords folded in, so that e_k(s, t) = (edge_k . (M, S, T)) at ray coordinates (1, s, t).
struct StagedTri {
    float4 c0;  // M, S, T of b x c; V = det(a, b, c)
    float4 c1;  // of c x a; the triangle's index
    float4 c2;  // of a x b; V, or 0 where V is too small for an estimate of the view depth
};

// dot(d, C) in the order x, y, z for a ray of faces 2 AXIS and 2 AXIS + 1: the axis component's
// product with +-1 is exact, and a sign moved from the ray to the vector changes no rounding.
template <int AXIS>
__device__ __forceinline__ float edgeAt(float M, float S, float T, float s, float t) {
    if constexpr (AXIS == 0) return (M + t * T) + s * S;
    else if constexpr (AXIS == 1) return (s * S + M) + t * T;
    else return (s * S + t * T) + M;
}

// (M, S, T, w) of a vector in the axes of face 2 AXIS + neg: faceCoords' table.
template <int AXIS>
__device__ __forceinline__ float4 faceAxes(bool neg, f3 C, float w) {
    if constexpr (AXIS == 0) return make_float4(neg ? -C.x : C.x, neg ? C.z : -C.z, -C.y, w);
    else if constexpr (AXIS == 1) return make_float4(neg ? -C.y : C.y, C.x, neg ? -C.z : C.z, w);
    else return make_float4(neg ? -C.z : C.z, neg ? -C.x : C.x, -C.y, w);
}

// Bound on a computed edge function's distance from the exact one: two products per cross component and
// three per dot product of vertices at most this far away, |ray| < 2.
__device__ __forceinline__ float edgeError(f3 a, f3 b, f3 c) {
    return 0x1p-20f * gmax(dot(a, a), gmax(dot(b, b), dot(c, c)));
}

// Whether the triangle may have a fragment among the rays within h of (midS, midT) on each axis, and a lower
// bound of their view depth.  A fragment needs e0, e1, e2 all of V's sign (or zero): the view depth
// V / (e0 + e1 + e2) is positive.  So a rectangle over which one edge, after V's sign, stays below -4 err
// has no fragment, and where there are some their view depth is at least |V| over the largest sum of the
// edges.
__device__ __forceinline__ bool mayCover(const float4* e, float V, float err, float midS, float midT, float h,
                                         float farP, float& nearest) {
    const float sg = V < 0.0f ? -1.0f : 1.0f;
    float most = 0.0f;
    bool out = false;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const float top = sg * (e[i].x + midS * e[i].y + midT * e[i].z) + (fabsf(e[i].y) + fabsf(e[i].z)) * h;
        out = out || top < -4.0f * err;
        most += top + 4.0f * err;
    }
    if (out) return false;
    const float t = fabsf(V) * frcp(most) * (1.0f - 0x1p-12f);
    nearest = most > 1e-30f && t < farP ? t : (most > 1e-30f ? farP : 0.0f);
    return true;
}

struct CubeLds {
    int32_t cand[kCand];
    StagedTri stage[64];
    uint16_t items[64 * kSmall];  // (staged lane << 8 | texel) of the wave's small triangles
};

// A tile drawn by SLICES waves: the smallest (key << 32 | index) per texel of its small triangles and,
// with several slices, of every slice.
struct TileDepth {
    unsigned long long drawn[kTile * kTile];
    float s[kTile], t[kTile];  // the tile's texel coordinates
};

// The texels of a tile's axis whose centres may lie in [lo, hi] +- a quarter texel (texel i's centre
// is (2 i + 1) / res - 1), within first .. last.
__device__ __forceinline__ void texelSpan(float lo, float hi, int res, int first, int last, int& i0, int& i1) {
    const float g = 0.5f * (float)res;
    const float a = ceilf((lo + 1.0f) * g - 0.75f), b = floorf((hi + 1.0f) * g - 0.25f);
    i0 = a > (float)first ? (a < (float)(last + 1) ? (int)a : last + 1) : first;
    i1 = b < (float)last ? (b > (float)(first - 1) ? (int)b : first - 1) : last;
}

// |(1, s, t)| of the ray, squares summed in the order x, y, z.
template <int AXIS>
__device__ __forceinline__ float rayLength(float s, float t) {
    if constexpr (AXIS == 0) return __builtin_sqrtf(1.0f + t * t + s * s);
    else if constexpr (AXIS == 1) return __builtin_sqrtf(s * s + 1.0f + t * t);
    else return __builtin_sqrtf(s * s + t * t + 1.0f);
}

// Lists the nt texels of this lane's small triangle (columns i0 .. i1 from row j0, tile offsets) in
// the wave's list as (lane << 8 | texel); returns the number of the wave's texels.
__device__ __forceinline__ int listTexels(int nt, int i0, int i1, int j0, uint16_t* list) {
    const int lane = threadIdx.x & 63;
    if (!__ballot(nt > 0)) return 0;
    const int incl = waveInclusive(nt);
    for (int q = 0, i = i0, j = j0; q < nt; ++q) {
        list[incl - nt + q] = (uint16_t)(lane << 8 | j << 4 | i);
        if (++i > i1) {
            i = i0;
            ++j;
        }
    }
    return __builtin_amdgcn_readlane(incl, 63);
}

// (2) one wave's share of a 16x16 tile of a face: depth-test its texels (at (x0, y0) of face f).
template <int FMT, int AXIS, int SLICES>
__device__ __forceinline__ void cubeTile(const CubeJob& job, int res, int u, int f, int x0, int y0, int slice, void* zb,
                                         uint32_t* cb, CubeLds& lds, TileDepth& tile) {
    const sgi_vpl& v = job.vpls[job.updates[job.first + u]];
    const f3 L{v.position[0], v.position[1], v.position[2]};
    const float farP = v.farPlane;
    const int32_t* tris = job.tris + ((size_t)u * 6 + f) * job.stride;
    const int lane = threadIdx.x & 63;
    const bool neg = (f & 1) != 0;
    const uint32_t clear = depthKey<FMT>(1.0f);  // the depth clear (:1455-1456)
    for (int i = lane; i < kTile * kTile; i += 64) tile.drawn[i] = ~0ull;
    if (lane < kTile) {
        tile.s[lane] = 2.0f * ((float)(x0 + lane) + 0.5f) / (float)res - 1.0f;
        tile.t[lane] = 2.0f * ((float)(y0 + lane) + 0.5f) / (float)res - 1.0f;
    }
    if constexpr (SLICES > 1) __syncthreads();  // (every slice writes the same start)
    else waveSync();
    // This lane's 2x2 texels: the range the nearest triangle's view depth estimate (hardware
    // reciprocal: within 2^-21) and its key's step leave open, and what gives its exact key.  A
    // triangle whose estimate lies outside the range is decided by it; the others are compared by
    // their exact keys.
    const int ox = (lane & 7) * 2, oy = (lane >> 3) * 2;
    float sc[2], tc[2], dlen[4], lo[4], hi[4], bestV[4], bestDen[4];
    int bestTri[4];
    const float invFar = frcp(farP);
    const float nearHi = job.nearPlane * (1.0f + 0x1p-18f), farLo = farP * (1.0f - 0x1p-18f);
    auto setRange = [&](int p, float t) {
        const float step = keyCell<FMT>(t * dlen[p] * invFar) * 1.01f * farP * frcp(dlen[p]);
        lo[p] = t - step;
        hi[p] = t + step;
    };
    auto keyOf = [&](float V, float den, float len) { return depthKey<FMT>(((V / den) * len) / farP); };
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        sc[q] = tile.s[ox + q];
        tc[q] = tile.t[oy + q];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        dlen[q] = rayLength<AXIS>(sc[q & 1], tc[q >> 1]);
        setRange(q, farP * frcp(dlen[q]));  // the view depth stored as 1: the clear
        bestV[q] = bestDen[q] = 0.0f;
        bestTri[q] = -1;  // the colour clear (:1453-1454)
    }
    const float h = (float)(kTile - 1) / (float)res;  // half the tile's span of texel centres
    const float midS = 2.0f * (float)(x0 + kTile / 2) / (float)res - 1.0f;
    const float midT = 2.0f * (float)(y0 + kTile / 2) / (float)res - 1.0f;
    const int rx = x0 / kRegion, ry = y0 / kRegion;
    Candidates<uint32_t, SLICES> list{job.ranges + ((size_t)u * 6 + f) * job.stride, job.listCounts[u * 6 + f],
                                      slice * kScan, 0, lds.cand};
    while (true) {
        const int nc = list.next([&](uint32_t r) {
            return rx >= (int)(r & 255u) && rx <= (int)(r >> 8 & 255u) && ry >= (int)(r >> 16 & 255u) &&
                   ry <= (int)(r >> 24);
        });
        if (nc == 0) break;
        float nearest = kFLOAT_MAX;  // a lower bound of this lane's triangle's view depth in the tile, if it is wide
        int nt = 0, i0 = 0, i1 = 0, j0 = 0, j1 = 0;  // a small triangle's texels
        if (lane < nc) {
            const int k = tris[list.cand[list.have + lane]];
            const f3 a = vertexRel(job.pos, k, 0, L), b = vertexRel(job.pos, k, 1, L), c = vertexRel(job.pos, k, 2, L);
            const f3 C0 = cross3(b, c), C1 = cross3(c, a), C2 = cross3(a, b);
            const float V = dot(a, C0);
            // an estimate V rcp(e0 + e1 + e2) past the far plane is one also where the sum is below the
            // reciprocal's range, unless V is as small itself
            const bool tiny = fabsf(V) < farP * 0x1p-80f;
            const float4 e[3] = {faceAxes<AXIS>(neg, C0, V), faceAxes<AXIS>(neg, C1, __int_as_float(k)),
                                 faceAxes<AXIS>(neg, C2, tiny ? 0.0f : V)};
            lds.stage[lane] = StagedTri{e[0], e[1], e[2]};
            const float err = edgeError(a, b, c);
            if (mayCover(e, V, err, midS, midT, h, farP, nearest)) {
                float m[3], s[3], t3[3];
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    const float4 q = faceAxes<AXIS>(neg, i == 0 ? a : (i == 1 ? b : c), 0.0f);
                    m[i] = q.x;
                    s[i] = q.y;
                    t3[i] = q.z;
                }
                if (m[0] > 1e-20f && m[1] > 1e-20f && m[2] > 1e-20f) {
                    // The exact sum of e_k (m_k, s_k, t_k) is V (1, s, t) for the ray (1, s, t), so at a ray
                    // beyond the projection's bounds by delta some e_k, after V's sign, is below
                    // -|V| delta / (3 max m w), w the projection's width; where that exceeds twice err for
                    // delta = 1/5 texel, no texel outside the bounds +- 1/4 texel has a fragment.
                    float sLo = kFLOAT_MAX, sHi = -kFLOAT_MAX, tLo = kFLOAT_MAX, tHi = -kFLOAT_MAX;
#pragma unroll
                    for (int i = 0; i < 3; ++i) {
                        const float inv = frcp(m[i]);
                        sLo = gmin(s[i] * inv, sLo);
                        sHi = gmax(s[i] * inv, sHi);
                        tLo = gmin(t3[i] * inv, tLo);
                        tHi = gmax(t3[i] * inv, tHi);
                    }
                    const float w = gmax(sHi - sLo, tHi - tLo), mMax = gmax(m[0], gmax(m[1], m[2]));
                    if (fabsf(V) * 0.4f > 6.0f * mMax * w * err * (float)res && w < 2.0f) {
                        texelSpan(sLo, sHi, res, x0, min(x0 + kTile, res) - 1, i0, i1);
                        texelSpan(tLo, tHi, res, y0, min(y0 + kTile, res) - 1, j0, j1);
                        nt = i1 >= i0 && j1 >= j0 ? (i1 - i0 + 1) * (j1 - j0 + 1) : 0;
                        if (nt <= kSmall) nearest = kFLOAT_MAX;
                        else nt = 0;
                    }
                }
            }
        }
        const int items = listTexels(nt, i0 - x0, i1 - x0, j0 - y0, lds.items);
        waveSync();
        for (int q = lane; q < items; q += 64) {
            const uint32_t it = lds.items[q];
            const StagedTri& tri = lds.stage[it >> 8];
            const float4 a = tri.c0, b = tri.c1, c = tri.c2;
            const float s = tile.s[it & 15u], t = tile.t[it >> 4 & 15u];
            const float e0 = edgeAt<AXIS>(a.x, a.y, a.z, s, t), e1 = edgeAt<AXIS>(b.x, b.y, b.z, s, t);
            const float e2 = edgeAt<AXIS>(c.x, c.y, c.z, s, t);
            const float in = fmaxf(fminf(fminf(e0, e1), e2), -fmaxf(fmaxf(e0, e1), e2));
            const float den = e0 + e1 + e2;
            if (!(in < 0.0f) && den != 0.0f) {
                const float tv = a.w / den;
                const uint32_t key = depthKey<FMT>((tv * rayLength<AXIS>(s, t)) / farP);
                if (tv >= job.nearPlane && tv <= farP && key < clear)  // GL clipping to [near, far]
                    atomicMin(&tile.drawn[it & 255u], (unsigned long long)key << 32 | __float_as_uint(b.w));
            }
        }
        // The wide triangles, near ones first: each pass takes those up to four times the nearest one's
        // depth, then what lies behind every texel is dropped.
        while (true) {
            const float first = -waveMax(-nearest);
            const float last = waveMax(fmaxf(fmaxf(hi[0], hi[1]), fmaxf(hi[2], hi[3])));
            // (first NaN: the far plane is, and nothing is nearer.  Otherwise the lane that holds it is taken
            // below, so the passes end.)
            if (first > last || !(first < kFLOAT_MAX)) break;
            const bool now = nearest <= fmaxf(4.0f * first, 4.0f * job.nearPlane) && !(nearest > last);
            uint64_t todo = __ballot(now);
            nearest = now ? kFLOAT_MAX : nearest;
            StagedTri next = lds.stage[__builtin_ctzll(todo)];
            while (todo) {
                const float4 a = next.c0, b = next.c1, c = next.c2;
                todo &= todo - 1;
                if (todo) next = lds.stage[__builtin_ctzll(todo)];
                float den[4], te[4];
                bool want[4];
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const float s = sc[p & 1], t = tc[p >> 1];
                    const float e0 = edgeAt<AXIS>(a.x, a.y, a.z, s, t), e1 = edgeAt<AXIS>(b.x, b.y, b.z, s, t);
                    const float e2 = edgeAt<AXIS>(c.x, c.y, c.z, s, t);
                    // >= 0 where the edges agree in sign; NaN edges give a NaN depth below, never drawn
                    const float in = fmaxf(fminf(fminf(e0, e1), e2), -fmaxf(fmaxf(e0, e1), e2));
                    den[p] = e0 + e1 + e2;
                    te[p] = c.w * frcp(den[p]);
                    want[p] = !(in < 0.0f) && !(te[p] > hi[p]);
                }
                if (!__ballot(want[0] || want[1] || want[2] || want[3])) continue;
                const int k = __float_as_int(b.w);
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    bool take = want[p];
                    if (take && !(te[p] < lo[p] && te[p] > nearHi && te[p] < farLo)) {
                        const float tv = a.w / den[p];
                        const uint32_t key = keyOf(a.w, den[p], dlen[p]);
                        const uint32_t held = bestTri[p] < 0 ? clear : keyOf(bestV[p], bestDen[p], dlen[p]);
                        take = den[p] != 0.0f && tv >= job.nearPlane && tv <= farP &&  // GL clipping to [near, far]
                               (key < held || (key == held && k < bestTri[p]));
                        te[p] = tv;
                    }
                    if (take) {
                        setRange(p, te[p]);
                        bestV[p] = a.w;
                        bestDen[p] = den[p];
                        bestTri[p] = k;
                    }
                }
            }
        }
        waveSync();  // the staged triangles are drawn
    }
    auto store = [&](int q, unsigned long long d) {
        const int i = x0 + q % kTile, j = y0 + q / kTile;
        if (i >= res || j >= res) return;
        const uint32_t key = d == ~0ull ? clear : (uint32_t)(d >> 32);
        const size_t off = ((size_t)f * res + j) * res + i;
        if constexpr (FMT == SGI_TEXEL_F32) ((float*)zb)[off] = __uint_as_float(key);
        else ((uint16_t*)zb)[off] = (uint16_t)key;
        if (cb) cb[off] = (d == ~0ull ? 0u : job.colors[(uint32_t)d]) | 0xFF000000u;
    };
    // the nearest wide triangles meet the small ones (and the other slices') in LDS
#pragma unroll
    for (int p = 0; p < 4; ++p)
        if (bestTri[p] >= 0)
            atomicMin(&tile.drawn[(oy + (p >> 1)) * kTile + ox + (p & 1)],
                      (unsigned long long)keyOf(bestV[p], bestDen[p], dlen[p]) << 32 | (uint32_t)bestTri[p]);
    if constexpr (SLICES > 1) {
        __syncthreads();
        store(threadIdx.x, tile.drawn[threadIdx.x]);
    } else {
        waveSync();
#pragma unroll
        for (int q = 0; q < 4; ++q) store(q * 64 + lane, tile.drawn[q * 64 + lane]);
    }
}

// A block per tile: one wave, or four that share its list.
template <int FMT, int SLICES>
__global__ __launch_bounds__(64 * SLICES, 4) void cubeRasterKernel(CubeJob job, int res, int regionsPerEdge, CubeArgs dist,
                                                           CubeArgs diffuse, int withColor) {
    static_assert(SLICES == 1 || SLICES == 4, "a tile is drawn by one wave or by the block's four");
    __shared__ CubeLds lds[SLICES];
    __shared__ TileDepth tile;
    const int slice = SLICES == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int block = blockIdx.x >> 2, quad = blockIdx.x & 3;
    const int perFace = regionsPerEdge * regionsPerEdge;
    const int r = block % perFace, f = (block / perFace) % 6, u = block / (perFace * 6);
    const int x0 = r % regionsPerEdge * kRegion + (quad & 1) * kTile, y0 = r / regionsPerEdge * kRegion + (quad >> 1) * kTile;
    const sgi_atlas_entry e = job.entries[job.updates[job.first + u]];
    // an entry outside the atlases names no cube: nothing is written for it
    if (e.index < 0 || e.index >= dist.numAtlases || e.layer < 0 || e.layer >= dist.layers) return;
    if (x0 >= res || y0 >= res) return;
    void* zb = const_cast<void*>(cubeLayerBase(dist, e.index, e.layer, texelBytes(FMT)));
    uint32_t* cb = withColor ? (uint32_t*)const_cast<void*>(cubeLayerBase(diffuse, e.index, e.layer, 4)) : nullptr;
    switch (f >> 1) {
        case 0: cubeTile<FMT, 0, SLICES>(job, res, u, f, x0, y0, slice, zb, cb, lds[slice], tile); break;
        case 1: cubeTile<FMT, 1, SLICES>(job, res, u, f, x0, y0, slice, zb, cb, lds[slice], tile); break;
        default: cubeTile<FMT, 2, SLICES>(job, res, u, f, x0, y0, slice, zb, cb, lds[slice], tile); break;
    }
}

// The whole pass for a mesh of at most kShort triangles: a block per 32x32 region tests them all against the
// region's sub-frustum, a triangle per thread, stages those that may touch it in their order, and draws them
// with exact keys at every texel, 2x2 per lane.  More than kDeep are drawn near ones first, until the next
// one lies behind every texel of the wave.
// One launch and no lists: over few triangles the lists' latency and each tile's setup are most of the time.
// GPU us by lists and tiles / this, 84 triangles of a room: 5 lights of 256^2 33 / 19, 64 lights 184 / 106,
// 300 lights of 64^2 83 / 50; 252 of a city, 96 lights of 256^2 237 / 184.  (256 triangles that all cover
// one another are the tiles' case, 1616 / 1930, but few meshes of that size are.)
constexpr int kShort = 256, kDeep = 16;
struct ShortLds {
    StagedTri stage[kShort];
    float nearest[kShort];
    uint8_t order[kShort];
    int waveCount[kShort / 64];
};

template <int FMT, int AXIS>
__device__ __forceinline__ void cubeRegion(const CubeJob& job, int res, int u, int f, int x0, int y0, void* zb,
                                           uint32_t* cb, ShortLds& lds) {
    const sgi_vpl& v = job.vpls[job.updates[job.first + u]];
    const f3 L{v.position[0], v.position[1], v.position[2]};
    const float farP = v.farPlane;
    const bool neg = (f & 1) != 0;
    const int k = (int)threadIdx.x, lane = k & 63, wave = k >> 6;
    bool keep = false;
    float nearest = kFLOAT_MAX;
    StagedTri tri{};
    if (k < job.count) {
        const f3 a = vertexRel(job.pos, k, 0, L), b = vertexRel(job.pos, k, 1, L), c = vertexRel(job.pos, k, 2, L);
        const f3 C0 = cross3(b, c);
        const float V = dot(a, C0);
        if (!culledFromLight(job.cull, V)) {
            const float4 q[3] = {faceAxes<AXIS>(neg, a, 0.0f), faceAxes<AXIS>(neg, b, 0.0f), faceAxes<AXIS>(neg, c, 0.0f)};
            const float m[3] = {q[0].x, q[1].x, q[2].x}, s[3] = {q[0].y, q[1].y, q[2].y}, t[3] = {q[0].z, q[1].z, q[2].z};
            const auto edge = [&](int i) { return 2.0f * (float)i / (float)res - 1.0f; };
            const float4 e[3] = {faceAxes<AXIS>(neg, C0, V), faceAxes<AXIS>(neg, cross3(c, a), __int_as_float(k)),
                                 faceAxes<AXIS>(neg, cross3(a, b), 0.0f)};
            keep = mayCover(e, V, edgeError(a, b, c), edge(x0 + kRegion / 2), edge(y0 + kRegion / 2),
                            (float)(kRegion - 1) / (float)res, farP, nearest) &&
                   !outsideFrustum(m, s, t, edge(x0), edge(min(x0 + kRegion, res)), edge(y0),
                                   edge(min(y0 + kRegion, res)), job.nearPlane, farP);
            tri = StagedTri{e[0], e[1], e[2]};
        }
    }
    const uint64_t bal = __ballot(keep);
    if (lane == 0) lds.waveCount[wave] = __popcll(bal);
    __syncthreads();
    int at = __popcll(bal & ((1ull << lane) - 1ull)), total = 0;
#pragma unroll
    for (int w = 0; w < kShort / 64; ++w) {
        at += w < wave ? lds.waveCount[w] : 0;
        total += lds.waveCount[w];
    }
    if (keep) {
        lds.stage[at] = tri;
        lds.nearest[at] = nearest;
    }
    __syncthreads();
    const int i0 = x0 + (k & 15) * 2, j0 = y0 + (k >> 4) * 2;
    float s[2], t[2], len[4], depth[4];
    uint32_t best[4];
    int drawn[4];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        s[p] = 2.0f * ((float)(i0 + p) + 0.5f) / (float)res - 1.0f;
        t[p] = 2.0f * ((float)(j0 + p) + 0.5f) / (float)res - 1.0f;
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        len[p] = rayLength<AXIS>(s[p & 1], t[p >> 1]);
        depth[p] = farP * frcp(len[p]);  // of the clear
        best[p] = depthKey<FMT>(1.0f);   // the depth clear (:1455-1456)
        drawn[p] = -1;                   // the colour clear (:1453-1454)
    }
    const auto draw = [&](const StagedTri& st) __attribute__((always_inline)) {
        const float4 a = st.c0, b = st.c1, c = st.c2;
        const int index = __float_as_int(b.w);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const float e0 = edgeAt<AXIS>(a.x, a.y, a.z, s[p & 1], t[p >> 1]);
            const float e1 = edgeAt<AXIS>(b.x, b.y, b.z, s[p & 1], t[p >> 1]);
            const float e2 = edgeAt<AXIS>(c.x, c.y, c.z, s[p & 1], t[p >> 1]);
            // >= 0 where the edges agree in sign; NaN edges give a NaN depth, never drawn
            const float in = fmaxf(fminf(fminf(e0, e1), e2), -fmaxf(fmaxf(e0, e1), e2));
            const float den = e0 + e1 + e2;
            if (in < 0.0f || den == 0.0f) continue;
            const float tv = a.w / den;
            if (!(tv >= job.nearPlane && tv <= farP)) continue;  // GL clipping to [near, far]
            const uint32_t key = depthKey<FMT>((tv * len[p]) / farP);
            if (key < best[p] || (key == best[p] && index < drawn[p])) {
                best[p] = key;
                drawn[p] = index;
                depth[p] = tv;
            }
        }
    };
    if (total <= kDeep) {
        for (int q = 0; q < total; ++q) draw(lds.stage[q]);
    } else {
        if (k < total) {  // its place among the depths (their bits: NaN too has one)
            const uint32_t mine = __float_as_uint(lds.nearest[k]);
            int place = 0;
            for (int q = 0; q < total; ++q) {
                const uint32_t other = __float_as_uint(lds.nearest[q]);
                place += other < mine || (other == mine && q < k) ? 1 : 0;
            }
            lds.order[place] = (uint8_t)k;
        }
        __syncthreads();
        const float invFar = frcp(farP);
        for (int q = 0; q < total; ++q) {
            const int n = lds.order[q];
            const float near = lds.nearest[n];
            bool behind = true;  // of what every texel holds, by more than a key's step (NaN: it may not be)
#pragma unroll
            for (int p = 0; p < 4; ++p)
                behind = behind &&
                         near > depth[p] + keyCell<FMT>(depth[p] * len[p] * invFar) * 1.01f * farP * frcp(len[p]);
            if (!__ballot(!behind)) break;
            draw(lds.stage[n]);
        }
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const int i = i0 + (p & 1), j = j0 + (p >> 1);
        if (i >= res || j >= res) continue;
        const size_t o = ((size_t)f * res + j) * res + i;
        if constexpr (FMT == SGI_TEXEL_F32) ((float*)zb)[o] = __uint_as_float(best[p]);
        else ((uint16_t*)zb)[o] = (uint16_t)best[p];
        if (cb) cb[o] = (drawn[p] < 0 ? 0u : job.colors[drawn[p]]) | 0xFF000000u;
    }
}

template <int FMT>
__global__ __launch_bounds__(kShort) void cubeShortKernel(CubeJob job, int res, int regionsPerEdge, CubeArgs dist,
                                                          CubeArgs diffuse, int withColor) {
    __shared__ ShortLds lds;
    const int perFace = regionsPerEdge * regionsPerEdge;
    const int r = blockIdx.x % perFace, f = (blockIdx.x / perFace) % 6, u = blockIdx.x / (perFace * 6);
    const int x0 = r % regionsPerEdge * kRegion, y0 = r / regionsPerEdge * kRegion;
    const sgi_atlas_entry e = job.entries[job.updates[job.first + u]];
    // an entry outside the atlases names no cube: nothing is written for it
    if (e.index < 0 || e.index >= dist.numAtlases || e.layer < 0 || e.layer >= dist.layers) return;
    void* zb = const_cast<void*>(cubeLayerBase(dist, e.index, e.layer, texelBytes(FMT)));
    uint32_t* cb = withColor ? (uint32_t*)const_cast<void*>(cubeLayerBase(diffuse, e.index, e.layer, 4)) : nullptr;
    switch (f >> 1) {
        case 0: cubeRegion<FMT, 0>(job, res, u, f, x0, y0, zb, cb, lds); break;
        case 1: cubeRegion<FMT, 1>(job, res, u, f, x0, y0, zb, cb, lds); break;
        default: cubeRegion<FMT, 2>(job, res, u, f, x0, y0, zb, cb, lds); break;
    }
}

// ---- sun cascades: RenderCSMDepth_ (StratusRendererBackend.cpp:1081-1158) with csm.vs:29-41
//
// Per cascade c, every triangle is transformed by cascadeProjViews[c]
// (projectionViewRender, an orthographic light projection) and rasterised
// into layer c: the window depth z * 0.5 + 0.5 interpolated at the texel
// centre, plus glPolygonOffset(factor, 0)'s slope term factor * m with
// m = max(|dz_w/dx_w|, |dz_w/dy_w|) (the form GL allows in place of the
// gradient's length), clamped to [0, 1] by GL_DEPTH_CLAMP (which also
// disables near / far clipping), depth test LESS against the clear 1.  The
// pass draws with each mesh's culling reversed (RenderImmediate_(..., true),
// :1029-1042): CCW meshes cull their light-facing (counter-clockwise) sides.
// Coverage: the 2-D edge functions of the NDC vertices at the texel centre all
// of one sign (a texel centre on an edge belongs to both triangles, the first
// in order winning LESS ties).
//
// Built as the cubes are: (1) one thread per (cascade, triangle) transforms, culls and appends the
// triangle's record with the regions its bounds touch, (2) one block per (cascade, 32x32 region)
// picks its records by range tests and draws them, the small ones texel by texel, the others by
// quadrants.  The smallest depth does not depend on the order.  24012
// triangles, 4 cascades of 1024^2: 1.32 -> 0.20 ms (list 0.058 -> 0.008, drawing 1.26 -> 0.18).
struct CsmJob {
    const float* pos;
    int count;
    int stride;          // count rounded up to a multiple of 4
    int keepSign;        // +1: keep counter-clockwise (NDC area > 0), -1: clockwise, 0: both
    float slope;         // glPolygonOffset factor
    int res;
    float m[SGI_NUM_CASCADES][16];
    uint2* ranges;       // [4][stride]: the regions an entry touches (x0, x1, y0, y1, 16 bits each)
    float* tris;         // [4][stride][10]: NDC x, y, z of the 3 vertices and the polygon offset
    int32_t* counts;     // [4]
};

// (1) per (cascade, triangle): the triangles that face the kept way and overlap the cascade's window,
// with their NDC vertices, polygon offset and regions (bounds +- 1e-3).
__global__ __launch_bounds__(kListBlock) void csmListKernel(CsmJob job, int regions) {
    const int c = blockIdx.y, k = blockIdx.x * kListBlock + (int)threadIdx.x;
    __shared__ int waveCount[kListBlock / 64];
    __shared__ int base;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    bool keep = false;
    float v[10];
    uint2 ranges = make_uint2(0u, 0u);
    if (k < job.count) {
        const float* q = job.pos + (size_t)k * 9;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            float cl[4];
            mulMat4(job.m[c], q[3 * i], q[3 * i + 1], q[3 * i + 2], 1.0f, cl);
            v[3 * i] = cl[0] / cl[3];
            v[3 * i + 1] = cl[1] / cl[3];
            v[3 * i + 2] = cl[2] / cl[3];
        }
        const float ex1 = v[3] - v[0], ey1 = v[4] - v[1], ez1 = v[5] - v[2];
        const float ex2 = v[6] - v[0], ey2 = v[7] - v[1], ez2 = v[8] - v[2];
        const float det = ex1 * ey2 - ex2 * ey1;  // twice the signed NDC area
        const bool facing = job.keepSign > 0 ? det > 0.0f : (job.keepSign < 0 ? det < 0.0f : det != 0.0f);
        const float mnx = fminf(v[0], fminf(v[3], v[6])), mxx = fmaxf(v[0], fmaxf(v[3], v[6]));
        const float mny = fminf(v[1], fminf(v[4], v[7])), mxy = fmaxf(v[1], fmaxf(v[4], v[7]));
        const bool inWindow = mxx >= -1.001f && mnx <= 1.001f && mxy >= -1.001f && mny <= 1.001f;
        keep = facing && inWindow;
        if (keep) {
            const float A = (ez1 * ey2 - ez2 * ey1) / det;  // dz/dx of the NDC plane
            const float B = (ex1 * ez2 - ex2 * ez1) / det;  // dz/dy
            // window units: z_w = z / 2 + 1/2 and x_w = (x + 1) res / 2, so dz_w/dx_w = A / res
            v[9] = job.slope * (fmaxf(fabsf(A), fabsf(B)) / (float)job.res);
            const float mar = 1.001e-3f;  // 1e-3 and the rounding of the region index
            ranges = make_uint2((uint32_t)firstRegion(mnx - mar, job.res, regions) |
                                    (uint32_t)lastRegion(mxx + mar, job.res, regions) << 16,
                                (uint32_t)firstRegion(mny - mar, job.res, regions) |
                                    (uint32_t)lastRegion(mxy + mar, job.res, regions) << 16);
        }
    }
    const uint64_t bal = __ballot(keep);
    if (lane == 0) waveCount[wave] = __popcll(bal);
    __syncthreads();
    int off = 0, total = 0;
    for (int w = 0; w < kListBlock / 64; ++w) {
        off += w < wave ? waveCount[w] : 0;
        total += waveCount[w];
    }
    if (threadIdx.x == 0) {
        if (gridDim.x == 1) job.counts[c] = total;  // the only block: nothing to add to, or to clear before
        base = gridDim.x > 1 && total ? atomicAdd(job.counts + c, total) : 0;
    }
    __syncthreads();
    if (keep) {
        const size_t e = (size_t)c * job.stride + base + off + __popcll(bal & ((1ull << lane) - 1ull));
        job.ranges[e] = ranges;
#pragma unroll
        for (int i = 0; i < 10; ++i) job.tris[e * 10 + i] = v[i];
    }
}

// A record set up for drawing: edge k runs from vertex k + 1 by (ex, ey)_k, so that its function at
// (sx, sy) is ex (sy - y_(k+1)) - ey (sx - x_(k+1)), edgeFn's products and differences.
struct StagedCsm {
    float4 x;  // x of vertices 1, 2, 0; z of vertex 0
    float4 y;  // y of vertices 1, 2, 0; z of vertex 1
    float4 ex; // and z of vertex 2
    float4 ey; // and the polygon offset
};

struct CsmLds {
    int32_t cand[kCand];
    StagedCsm stage[64];
    uint16_t items[64 * kSmall];  // (staged lane << 8 | texel) of the wave's small triangles
};

struct CsmTile {
    uint32_t drawn[kTile * kTile];  // the smallest depth drawn (a depth in [0, 1] orders as its bits)
    float s[kTile], t[kTile];
};

// The window depth of edge functions w0, w1, w2 (their sum not 0), clamped (GL_DEPTH_CLAMP).
__device__ __forceinline__ float csmDepth(const StagedCsm& q, float w0, float w1, float w2, float sum) {
    const float z = (w0 * q.x.w + w1 * q.y.w + w2 * q.ex.w) / sum;
    const float dw = z * 0.5f + 0.5f + q.ey.w;
    return dw < 0.0f ? 0.0f : (dw > 1.0f ? 1.0f : dw);
}

// (2) per (cascade, 16x16 tile): rasterise the records that touch the tile at every texel centre.
template <int SLICES>
__global__ __launch_bounds__(64 * SLICES, 4) void csmRasterKernel(CsmJob job, int regionsPerEdge, float* __restrict__ depth) {
    __shared__ CsmLds ldsAll[SLICES];
    __shared__ CsmTile tile;
    const int lane = threadIdx.x & 63, slice = SLICES == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int block = blockIdx.x >> 2, quad = blockIdx.x & 3;
    const int perLayer = regionsPerEdge * regionsPerEdge;
    const int c = block / perLayer, r = block % perLayer, rx = r % regionsPerEdge, ry = r / regionsPerEdge;
    const int x0 = rx * kRegion + (quad & 1) * kTile, y0 = ry * kRegion + (quad >> 1) * kTile, res = job.res;
    if (x0 >= res || y0 >= res) return;
    CsmLds& lds = ldsAll[slice];
    const float* records = job.tris + (size_t)c * job.stride * 10;
    for (int i = lane; i < kTile * kTile; i += 64) tile.drawn[i] = __float_as_uint(1.0f);  // the clear
    if (lane < kTile) {
        tile.s[lane] = 2.0f * ((float)(x0 + lane) + 0.5f) / (float)res - 1.0f;
        tile.t[lane] = 2.0f * ((float)(y0 + lane) + 0.5f) / (float)res - 1.0f;
    }
    if constexpr (SLICES > 1) __syncthreads();  // (every slice writes the same start)
    else waveSync();
    const int ox = (lane & 7) * 2, oy = (lane >> 3) * 2;
    float sx[2], sy[2], best[4];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        sx[p] = tile.s[ox + p];
        sy[p] = tile.t[oy + p];
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) best[p] = 1.0f;
    const float h = (float)(kTile - 1) / (float)res;  // half the tile's span of texel centres
    const float midX = 2.0f * (float)(x0 + kTile / 2) / (float)res - 1.0f;
    const float midY = 2.0f * (float)(y0 + kTile / 2) / (float)res - 1.0f;
    Candidates<uint2, SLICES> list{job.ranges + (size_t)c * job.stride, job.counts[c],
                                   slice * kScan, 0, lds.cand};
    while (true) {
        const int nc = list.next([&](uint2 q) {
            return rx >= (int)(q.x & 0xFFFFu) && rx <= (int)(q.x >> 16) && ry >= (int)(q.y & 0xFFFFu) &&
                   ry <= (int)(q.y >> 16);
        });
        if (nc == 0) break;
        float lowest = kFLOAT_MAX;  // a lower bound of this lane's triangle's depth, if it is wide
        int nt = 0, i0 = 0, i1 = 0, j0 = 0, j1 = 0;  // a small triangle's texels
        if (lane < nc) {
            const float* v = records + (size_t)list.cand[list.have + lane] * 10;
            const float ax = v[0], ay = v[1], az = v[2], bx = v[3], by = v[4], bz = v[5], cx = v[6], cy = v[7];
            const float cz = v[8];
            StagedCsm q;
            q.x = make_float4(bx, cx, ax, az);
            q.y = make_float4(by, cy, ay, bz);
            q.ex = make_float4(cx - bx, ax - cx, bx - ax, cz);
            q.ey = make_float4(cy - by, ay - cy, by - ay, v[9]);
            lds.stage[lane] = q;
            const float mnx = fminf(ax, fminf(bx, cx)), mxx = fmaxf(ax, fmaxf(bx, cx));
            const float mny = fminf(ay, fminf(by, cy)), mxy = fmaxf(ay, fmaxf(by, cy));
            const float w = fmaxf(mxx - mnx, mxy - mny), texel = 2.0f / (float)res;
            const float det = (bx - ax) * (cy - ay) - (cx - ax) * (by - ay);
            // A tile over which one edge, after det's sign, stays below -edgeErr has no texel whose three
            // functions agree in sign (the other two sum to more than edgeErr there).
            const float sg = det < 0.0f ? -1.0f : 1.0f;
            const float ex[3] = {q.ex.x, q.ex.y, q.ex.z}, ey[3] = {q.ey.x, q.ey.y, q.ey.z};
            const float vx[3] = {bx, cx, ax}, vy[3] = {by, cy, ay};
            float reach = 0.0f;
#pragma unroll
            for (int i = 0; i < 3; ++i) reach = fmaxf(reach, fmaxf(fabsf(midX - vx[i]), fabsf(midY - vy[i])));
            const float edgeErr = 0x1p-18f * w * (reach + h);
            bool out = false;
#pragma unroll
            for (int i = 0; i < 3; ++i)
                out = out || sg * (ex[i] * (midY - vy[i]) - ey[i] * (midX - vx[i])) + (fabsf(ex[i]) + fabsf(ey[i])) * h < -edgeErr;
            if (!out) {
                // a covered texel's depth is a mean of the vertices' (weights of one sign) to 2^-20 of the largest
                const float mag = fmaxf(fabsf(az), fmaxf(fabsf(bz), fabsf(cz))) + fabsf(v[9]) + 1.0f;
                lowest = fminf(az, fminf(bz, cz)) * 0.5f + 0.5f + v[9] - mag * 0x1p-18f;
                lowest = lowest > 0.0f ? lowest : 0.0f;  // the clamp; NaN: tested
                // At a point beyond the bounds by delta the barycentric coordinates sum x_k - x_max to delta,
                // so some edge function is below -|det| delta / (3 w) after det's sign; the computed ones lie
                // within 2^-21 w (w + delta).  Where the first exceeds four times the second for delta = 1/5
                // texel (and so for every larger one: that edge is then surely negative, and the two others,
                // which with it sum to |det|, are not both negative), no texel outside the bounds +- 1/4 texel
                // is covered.
                if (fabsf(det) * 0.2f * texel > 12.0f * 0x1p-21f * w * w * (w + texel)) {
                    texelSpan(mnx, mxx, res, x0, min(x0 + kTile, res) - 1, i0, i1);
                    texelSpan(mny, mxy, res, y0, min(y0 + kTile, res) - 1, j0, j1);
                    nt = i1 >= i0 && j1 >= j0 ? (i1 - i0 + 1) * (j1 - j0 + 1) : 0;
                    if (nt <= kSmall) lowest = kFLOAT_MAX;
                    else nt = 0;
                }
            }
        }
        const int items = listTexels(nt, i0 - x0, i1 - x0, j0 - y0, lds.items);
        waveSync();
        for (int q = lane; q < items; q += 64) {
            const uint32_t it = lds.items[q];
            const StagedCsm t = lds.stage[it >> 8];
            const float px = tile.s[it & 15u], py = tile.t[it >> 4 & 15u];
            const float w0 = t.ex.x * (py - t.y.x) - t.ey.x * (px - t.x.x);
            const float w1 = t.ex.y * (py - t.y.y) - t.ey.y * (px - t.x.y);
            const float w2 = t.ex.z * (py - t.y.z) - t.ey.z * (px - t.x.z);
            const float in = fmaxf(fminf(fminf(w0, w1), w2), -fmaxf(fmaxf(w0, w1), w2));
            const float sum = w0 + w1 + w2;
            if (!(in < 0.0f) && sum != 0.0f) {
                const float dw = csmDepth(t, w0, w1, w2, sum);
                if (dw < 1.0f) atomicMin(&tile.drawn[it & 255u], __float_as_uint(dw));
            }
        }
        // the wide triangles that are not behind every texel
        const float deepest = waveMax(fmaxf(fmaxf(best[0], best[1]), fmaxf(best[2], best[3])));
        uint64_t todo = __ballot(lowest <= deepest);
        StagedCsm next;
        if (todo) next = lds.stage[__builtin_ctzll(todo)];
        while (todo) {
            const StagedCsm t = next;
            todo &= todo - 1;
            if (todo) next = lds.stage[__builtin_ctzll(todo)];
            float w0[4], w1[4], w2[4], sum[4];
            bool open[4];  // covered texels whose estimate may be below the best
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const float px = sx[p & 1], py = sy[p >> 1];
                w0[p] = t.ex.x * (py - t.y.x) - t.ey.x * (px - t.x.x);
                w1[p] = t.ex.y * (py - t.y.y) - t.ey.y * (px - t.x.y);
                w2[p] = t.ex.z * (py - t.y.z) - t.ey.z * (px - t.x.z);
                // >= 0 where the functions agree in sign; NaN ones give a NaN depth, which is below nothing
                const float in = fmaxf(fminf(fminf(w0[p], w1[p]), w2[p]), -fmaxf(fmaxf(w0[p], w1[p]), w2[p]));
                sum[p] = w0[p] + w1[p] + w2[p];
                const float z = (w0[p] * t.x.w + w1[p] * t.y.w + w2[p] * t.ex.w) * frcp(sum[p]);
                const float mag = fabsf(z) + fabsf(t.ey.w) + 1.0f;
                const bool above = z * 0.5f + 0.5f + t.ey.w > __builtin_fmaf(mag, 0x1p-18f, best[p]);
                open[p] = !(in < 0.0f) && !(above && fabsf(sum[p]) > 1e-30f);
            }
            if (!__ballot(open[0] || open[1] || open[2] || open[3])) continue;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const float dw = csmDepth(t, w0[p], w1[p], w2[p], sum[p]);
                best[p] = open[p] && sum[p] != 0.0f && dw < best[p] ? dw : best[p];
            }
        }
        waveSync();  // the staged triangles are drawn
    }
    // the depths meet the small triangles' (and the other slices') in LDS
#pragma unroll
    for (int p = 0; p < 4; ++p)
        if (best[p] < 1.0f) atomicMin(&tile.drawn[(oy + (p >> 1)) * kTile + ox + (p & 1)], __float_as_uint(best[p]));
    float* layer = depth + (size_t)c * res * res;
    auto store = [&](int q) {
        const int i = x0 + q % kTile, j = y0 + q / kTile;
        if (i < res && j < res) layer[(size_t)j * res + i] = __uint_as_float(tile.drawn[q]);
    };
    if constexpr (SLICES > 1) {
        __syncthreads();
        store(threadIdx.x);
    } else {
        waveSync();
#pragma unroll
        for (int q = 0; q < 4; ++q) store(q * 64 + lane);
    }
}

// Whether a tile is drawn by a whole block that shares its list, or by one wave.  A block shortens a long
// list's chain, which the launch waits for, and repeats the tile's setup; both grow, the first with the
// triangles and the second with the tiles, and they are equal about where there are 3 triangles to 4 tiles
// (us by waves / by blocks).  Cubes: 1212 triangles, 7680 tiles 70 / 95; 4812, 1536 91 / 71, 7680 112 / 115,
// 18432 126 / 177; 12012, 7680 132 / 115, 18432 150 / 186; 24012, 7680 208 / 137, 30720 360 / 337, 49152
// 373 / 495, 147456 850 / 1343; 96012, 46080 1683 / 1287, 147456 3898 / 3592.  Cascades: 12012, 4096 91 / 57,
// 16384 105 / 107, 30976 143 / 177; 96012, 33856 992 / 932, 141376 3163 / 3346.  Up to `spare` tiles, one
// wave each would leave SIMDs idle: cascades of 4096, 516 triangles 32 / 32, 2412 65 / 41 (cubes' lists,
// of six faces, are shorter: 0).  A list within one scan is the first wave's alone: 516, the cubes of 15
// lights 83 / 155.  (A launch holds fewer than 2^32 threads.)
static bool drawnByBlocks(long tiles, int count, long spare) {
    return count > kScan && tiles < 1L << 23 && (tiles <= spare || tiles * 3 < (long)count * 4);
}

}  // namespace

namespace sgi_launch {

static int listStride(int count) { return (count + 3) & ~3; }  // 16-byte aligned range arrays

size_t csmScratchFloats(int count) { return (size_t)SGI_NUM_CASCADES * listStride(count) * 12 + SGI_NUM_CASCADES; }

hipError_t renderCsm(const float* pos, int count, int keepSign, float slope, int res,
                     const float (*projViews)[16], float* scratch, float* depth, hipStream_t s) {
    CsmJob job{};
    job.pos = pos;
    job.count = count;
    job.stride = listStride(count);
    job.keepSign = keepSign;
    job.slope = slope;
    job.res = res;
    for (int c = 0; c < SGI_NUM_CASCADES; ++c)
        for (int k = 0; k < 16; ++k) job.m[c][k] = projViews[c][k];
    const size_t entries = (size_t)SGI_NUM_CASCADES * job.stride;
    job.ranges = (uint2*)scratch;
    job.tris = scratch + 2 * entries;
    job.counts = (int32_t*)(scratch + 12 * entries);
    const int rpe = (res + kRegion - 1) / kRegion;
    const int listBlocks = max(1, (count + kListBlock - 1) / kListBlock);
    if (listBlocks > 1)
        hipLaunchKernelGGL(clearIntsKernel, dim3(1), dim3(64), 0, s, job.counts, SGI_NUM_CASCADES);
    hipLaunchKernelGGL(csmListKernel, dim3((unsigned)listBlocks, SGI_NUM_CASCADES), dim3(kListBlock), 0, s, job, rpe);
    const long tiles = 4L * SGI_NUM_CASCADES * rpe * rpe;
    if (drawnByBlocks(tiles, count, 4096))
        hipLaunchKernelGGL(csmRasterKernel<4>, dim3((unsigned)tiles), dim3(256), 0, s, job, rpe, depth);
    else
        hipLaunchKernelGGL(csmRasterKernel<1>, dim3((unsigned)tiles), dim3(64), 0, s, job, rpe, depth);
    return hipGetLastError();
}

size_t cubeListInts(int batch, int count) {
    return (size_t)batch * 12 * (size_t)listStride(count) + (size_t)batch * 6;
}

hipError_t renderVplCubes(const float* pos, const uint32_t* colors, int count, int cull, const sgi_vpl* vpls,
                          const int32_t* updates, int numUpdates, const sgi_atlas_entry* entries, float nearPlane,
                          const sgi_dev::CubeArgs& dist, int format, const sgi_dev::CubeArgs& diffuse,
                          bool withDiffuse, int batchMax, int32_t* scratch, hipStream_t s) {
    const int res = dist.res;
    const int rpe = (res + kRegion - 1) / kRegion;
    for (int first = 0; first < numUpdates; first += batchMax) {
        const int batch = min(batchMax, numUpdates - first);
        const int stride = listStride(count);
        const size_t entriesMax = (size_t)batch * 6 * (size_t)stride;
        CubeJob job{pos, colors, count, vpls, updates, first, batch, entries, nearPlane, cull, stride,
                    reinterpret_cast<uint32_t*>(scratch), scratch + entriesMax, scratch + 2 * entriesMax};
        const int wc = withDiffuse ? 1 : 0;
        const bool brief = count <= kShort;
        if (!brief) {
            hipLaunchKernelGGL(clearIntsKernel, dim3((unsigned)((batch * 6 + 255) / 256)), dim3(256), 0, s,
                               job.listCounts, batch * 6);
            hipLaunchKernelGGL(cubeFaceListKernel,
                               dim3((unsigned)((count + kListBlock - 1) / kListBlock), (unsigned)batch),
                               dim3(kListBlock), 0, s, job, res, rpe);
        }
        const long tiles = 4L * batch * 6 * rpe * rpe;
#define SGI_CUBE_RASTER(F)                                                                                            \
    if (brief)                                                                                                        \
        hipLaunchKernelGGL(cubeShortKernel<F>, dim3((unsigned)(tiles / 4)), dim3(kShort), 0, s, job, res, rpe, dist, diffuse, wc); \
    else if (drawnByBlocks(tiles, count, 0))                                                                          \
        hipLaunchKernelGGL((cubeRasterKernel<F, 4>), dim3((unsigned)tiles), dim3(256), 0, s, job, res, rpe, dist, diffuse, wc); \
    else                                                                                                              \
        hipLaunchKernelGGL((cubeRasterKernel<F, 1>), dim3((unsigned)tiles), dim3(64), 0, s, job, res, rpe, dist, diffuse, wc)
        if (format == SGI_TEXEL_F32) {
            SGI_CUBE_RASTER(SGI_TEXEL_F32);
        } else if (format == SGI_TEXEL_F16) {
            SGI_CUBE_RASTER(SGI_TEXEL_F16);
        } else {
            SGI_CUBE_RASTER(SGI_TEXEL_UNORM16);
        }
#undef SGI_CUBE_RASTER
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace sgi_launch
