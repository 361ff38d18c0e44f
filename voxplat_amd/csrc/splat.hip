// splat.hip -- per-pixel ray/AABB splat resolve and its colour backward, gfx950.
//
// Replaces the splat draw of gfx_svl_draw (src/gfx/vsplat.c:104-193): the
// vertex stage of resources/splat.vert.glsl:34-54 (view translation, clip
// position, point-sprite size) and the fragment stage of
// resources/splat.frag.glsl:60-156 (view ray, slab ray/AABB test, depth
// t0/far, GL_LESS), with GL's point clipping and sprite coverage made
// explicit:
//  * a point survives iff its clip-space vertex is inside the clip volume;
//  * its sprite covers pixel p iff wx - s/2 <= p.x + 0.5 < wx + s/2 (same in y),
//    s = the point size clamped to [1, 2048];
//  * the nearest hit wins, ties to the lower splat index (GL submission
//    order): one 64-bit atomicMin per fragment on (depth bits << 32 | index).
// All float arithmetic is written one IEEE operation at a time, contraction
// off, correctly rounded division and square root, GLSL min/max as selects,
// so the results are those of the stated operation order.
#pragma clang fp contract(off)

#include <type_traits>

#include "vp_internal.h"

namespace vp {

struct SplatCam {
    float T[16], PR[16], IPR[16];
    uint32_t W, H;
    float far_plane;
    float inv_far;     // 1 / far_plane where that is exact (a power of two), else 0
};

// t / far_plane: where the reciprocal is a power of two, the product rounds
// the same quotient.
__device__ __forceinline__ float over_far(const SplatCam &c, float t)
{
    return c.inv_far != 0.0f ? t * c.inv_far : t / c.far_plane;
}

__device__ __forceinline__ void mv4(const float *m, const float v[4], float o[4])
{
#pragma unroll
    for (int r = 0; r < 4; r++) {
        float s = m[0 * 4 + r] * v[0];
        s = s + m[1 * 4 + r] * v[1];
        s = s + m[2 * 4 + r] * v[2];
        s = s + m[3 * 4 + r] * v[3];
        o[r] = s;
    }
}

__device__ __forceinline__ float gmin(float x, float y) { return (y < x) ? y : x; }
__device__ __forceinline__ float gmax(float x, float y) { return (x < y) ? y : x; }
__device__ __forceinline__ float gsign(float x)
{
    return x > 0.0f ? 1.0f : (x < 0.0f ? -1.0f : 0.0f);
}

struct VS {
    float vx, vy, vz, half;
    int x0, x1, y0, y1;   // the covered pixels (empty where x0 > x1 or y0 > y1)
    uint64_t lb;   // (lower bound of the splat's depth t0/far) << 32 | 1: no fragment key
                   // is below the bound, and one equal to it in the high word cannot win
};

// Position of a splat record (its first three int16).
__device__ __forceinline__ float rec_x(uint2 r) { return (float)(int16_t)(r.x & 0xFFFFu); }
__device__ __forceinline__ float rec_y(uint2 r) { return (float)(int16_t)(r.x >> 16); }
__device__ __forceinline__ float rec_z(uint2 r) { return (float)(int16_t)(r.y & 0xFFFFu); }

// A record of a list that need only be aligned as int16.
__device__ __forceinline__ uint2 ld_rec(const int16_t *splats, uint64_t i)
{
    const int16_t *r = splats + 4 * i;
    return make_uint2((uint32_t)(uint16_t)r[0] | (uint32_t)(uint16_t)r[1] << 16,
                      (uint32_t)(uint16_t)r[2]);
}

__device__ __forceinline__ bool vertex_stage(uint2 rec, float lodf, const SplatCam &c, VS &o)
{
    const float half = 0.5f * lodf;
    const float a[4] = {rec_x(rec) + half, rec_y(rec) + half, rec_z(rec) + half, 1.0f};
    float v[4], clip[4];
    mv4(c.T, a, v);
    mv4(c.PR, v, clip);
    const float W = (float)c.W, H = (float)c.H, cw = clip[3];
    if (!(clip[0] >= -cw && clip[0] <= cw && clip[1] >= -cw && clip[1] <= cw &&
          clip[2] >= -cw && clip[2] <= cw))
        return false;
    const float ratio = W / H;
    const float rx = fabsf((clip[0] * ratio) / cw);
    const float ry = fabsf(clip[1] / cw);
    float reduce = gmax(rx, ry);
    reduce = reduce + 0.03f;
    float size = (H * 1.1f) / clip[2];
    size = size * gmax(reduce, 1.0f);
    float ps = size * lodf;
    ps = (ps > 1.0f) ? ps : 1.0f;
    ps = (ps < 2048.0f) ? ps : 2048.0f;
    const float ndx = clip[0] / cw, ndy = clip[1] / cw;
    const float wx = (ndx + 1.0f) * (0.5f * W);
    const float wy = (ndy + 1.0f) * (0.5f * H);
    const float hs = 0.5f * ps;
    const float lox = wx - hs, hix = wx + hs, loy = wy - hs, hiy = wy + hs;
    // pixel p is covered iff lo <= p + 0.5 < hi: every such p lies in
    // [floor(lo), ceil(hi) - 1], and only the two ends of that range can fail
    int x0 = (int)floorf(lox), x1 = (int)ceilf(hix) - 1;
    int y0 = (int)floorf(loy), y1 = (int)ceilf(hiy) - 1;
    if (!(lox <= (float)x0 + 0.5f)) x0++;
    if (!((float)x1 + 0.5f < hix)) x1--;
    if (!(loy <= (float)y0 + 0.5f)) y0++;
    if (!((float)y1 + 0.5f < hiy)) y1--;
    o.x0 = x0 < 0 ? 0 : x0;
    o.y0 = y0 < 0 ? 0 : y0;
    o.x1 = x1 > (int)c.W - 1 ? (int)c.W - 1 : x1;
    o.y1 = y1 > (int)c.H - 1 ? (int)c.H - 1 : y1;
    o.vx = v[0]; o.vy = v[1]; o.vz = v[2];
    o.half = half;
    // Distance from the eye (the origin of the translated frame) to the box
    // v +- half bounds every ray's entry time t0 from below; shrunk by 2^-10,
    // far more than the rounding of the slab test, it stays below the computed
    // t0, and t0/far keeps the order after rounding.
    const float ex = gmax(fabsf(v[0]) - half, 0.0f), ey = gmax(fabsf(v[1]) - half, 0.0f);
    const float ez = gmax(fabsf(v[2]) - half, 0.0f);
    float dd = ex * ex;
    dd = dd + ey * ey;
    dd = dd + ez * ez;
    const float lbd = over_far(c, sqrtf(dd) * 0.9990234375f);
    // + 1: above a key of 0, which nothing can lower and which stands for
    // "no pixel" in a batch
    o.lb = (uint64_t)__float_as_uint(lbd) << 32 | 1u;
    return true;
}

__device__ __forceinline__ void pixel_dir(const SplatCam &c, int px, int py, float d[3])
{
    const float fx = ((float)px + 0.5f) / (float)c.W;
    const float fy = ((float)py + 0.5f) / (float)c.H;
    const float cl[4] = {fx * 2.0f - 1.0f, fy * 2.0f - 1.0f, -1.0f, 1.0f};
    float r[4];
    mv4(c.IPR, cl, r);
    const float x = r[0] / r[3], y = r[1] / r[3], z = r[2] / r[3];
    float dd = x * x;
    dd = dd + y * y;
    dd = dd + z * z;
    const float len = sqrtf(dd);
    d[0] = x / len; d[1] = y / len; d[2] = z / len;
}

__device__ __forceinline__ void aabb(float lx, float hx, float ly, float hy, float lz, float hz,
                                     float ix, float iy, float iz, float &t0, float &t1)
{
    const float tbx = lx * ix, ttx = hx * ix;
    const float tby = ly * iy, tty = hy * iy;
    const float tbz = lz * iz, ttz = hz * iz;
    const float mnx = gmin(ttx, tbx), mny = gmin(tty, tby), mnz = gmin(ttz, tbz);
    const float mxx = gmax(ttx, tbx), mxy = gmax(tty, tby), mxz = gmax(ttz, tbz);
    t0 = gmax(gmax(mnx, mny), gmax(mnx, mnz));
    t1 = gmin(gmin(mxx, mxy), gmin(mxx, mxz));
}

// A frame's start, one thread per pixel: its ray, its key, and (by the first
// threads) the tile bounds nt of them and the block counters nc.
__global__ void k_frame_start(SplatCam c, float4 *rays, uint64_t *frame, uint32_t *hiz, uint32_t nt,
                              uint32_t *cnt, uint32_t nc)
{
    const uint32_t px = blockIdx.x * blockDim.x + threadIdx.x, py = blockIdx.y;
    if (px >= c.W) return;
    const size_t p = (size_t)py * c.W + px;
    frame[p] = ~0ull;
    if (p < nt) hiz[p] = ~0u;              // at most one tile per pixel
    for (size_t k = p; k < nc; k += (size_t)c.W * c.H) cnt[k] = 0u;
    float d[3];
    pixel_dir(c, (int)px, (int)py, d);
    // w marks a ray along a coordinate plane: an infinite (or no) reciprocal
    const float ix = 1.0f / d[0], iy = 1.0f / d[1], iz = 1.0f / d[2];
    const bool fin = fabsf(ix) < INFINITY && fabsf(iy) < INFINITY && fabsf(iz) < INFINITY;
    rays[p] = make_float4(ix, iy, iz, fin ? 0.0f : 1.0f);
}

// The slab planes of a splat's cube, v -+ half.
struct Slabs {
    float lx, hx, ly, hy, lz, hz;
};
__device__ __forceinline__ Slabs slabs_of(float vx, float vy, float vz, float half)
{
    return {vx - half, vx + half, vy - half, vy + half, vz - half, vz + half};
}

// aabb() of the cube for a ray of finite reciprocals: no product is a NaN, and
// then the GLSL selects are plain minima and maxima (a zero's sign is lost,
// which neither the hit test nor the clamped depth sees).
__device__ __forceinline__ void aabb_finite(const Slabs &s, float4 inv, float &t0, float &t1)
{
    const float tbx = s.lx * inv.x, ttx = s.hx * inv.x;
    const float tby = s.ly * inv.y, tty = s.hy * inv.y;
    const float tbz = s.lz * inv.z, ttz = s.hz * inv.z;
    t0 = fmaxf(fmaxf(fminf(ttx, tbx), fminf(tty, tby)), fminf(ttz, tbz));
    t1 = fminf(fminf(fmaxf(ttx, tbx), fmaxf(tty, tby)), fmaxf(ttz, tbz));
}

// The fragment of pixel p whose frame key was read as cur: GL_LESS on
// (depth bits << 32 | id) by one atomicMin.  cur may be older than the
// frame (the loads of a batch go out before any of its tests): a key at or
// above an older value is at or above the current one too, so the tests
// only ever skip fragments that could not win.
__device__ __forceinline__ void fragment_test(const SplatCam &c, float4 inv, uint64_t *frame,
                                              const Slabs &s, uint32_t id, uint32_t p, uint64_t cur)
{
    float t0, t1;
    if (inv.w == 0.0f) {
        aabb_finite(s, inv, t0, t1);
    } else {
        aabb(s.lx, s.hx, s.ly, s.hy, s.lz, s.hz, inv.x, inv.y, inv.z, t0, t1);
    }
    if (!(t0 <= t1)) return;
    float d = over_far(c, t0);
    if (!(d < 1.0f)) return;
    if (d <= 0.0f) d = 0.0f;
    const uint64_t key = ((uint64_t)__float_as_uint(d) << 32) | id;
    if (key < cur) atomicMin(reinterpret_cast<unsigned long long *>(frame + p), key);
}

// Sprites of up to kSmallArea pixels are rasterised by their own lane,
// larger ones by the whole wave, a few at a time.  Most fragments end at
// the depth lower bound after one frame load, so the loads are issued in
// batches (kLoads per lane) before any test: the lane waits once per batch
// instead of once per pixel.  A lane's own sprite takes batches of 4: a slot
// costs its instructions whether a lane has a pixel for it or not, and a splat
// covers 6 pixels on average (8: 913 against 881 us per 1080p frame, 4776
// against 4426 us for 16 views of 512x512; 2: 975 us; 12 leaves three waves per
// SIMD: 1367 us).  Wave-shared sprites fill their slots, and take 8 (two close
// views of a 7.7 M list at 1697x1495: 8030 us with 4, 5810 with 8; of a 31 M
// list at 1920x1080: 5760, 4440).
constexpr int kSmallArea = 64;
constexpr int kLoads = 4;
constexpr int kGroup = 4;                 // wave-shared sprites per round
constexpr int kSteps = 2;                 // pixels of each per lane per round
constexpr int kShared = kGroup * kSteps;

// Lane src's value (src wave-uniform) through a scalar register: no LDS
// traffic, unlike a general shuffle.
__device__ __forceinline__ int lane_i(int v, int src) { return __builtin_amdgcn_readlane(v, src); }
__device__ __forceinline__ float lane_f(float v, int src)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
}

// A wave-shared sprite: the owning lane's vertex stage, broadcast.
struct WaveSprite {
    Slabs s;
    int x0, y0, w, a, dq, dr;
    uint32_t id;
    uint64_t lb;
};

__device__ __forceinline__ WaveSprite wave_sprite(const VS &vs, int area, uint32_t id, int src)
{
    WaveSprite s;
    s.s = slabs_of(lane_f(vs.vx, src), lane_f(vs.vy, src), lane_f(vs.vz, src), lane_f(vs.half, src));
    s.x0 = lane_i(vs.x0, src);
    s.y0 = lane_i(vs.y0, src);
    s.w = lane_i(vs.x1, src) - s.x0 + 1;
    s.a = lane_i(area, src);
    s.id = (uint32_t)lane_i((int)id, src);
    s.lb = (uint64_t)(uint32_t)lane_i((int)(uint32_t)(vs.lb >> 32), src) << 32;
    return s;
}

// One splat per lane (ok: the lane has one), record rec of edge lodf; every
// lane of the wave calls it.  AHEAD: a batch's rays are loaded together before
// its tests.  Near to far, few fragments pass the bound and their rays' waits
// add up; in list order many pass, and the loads beside those that do not cost
// more than the waits (a 7.7 M list at 1920x1080 without blocks, four far views:
// 5220 us ahead, 4900 on demand).
template <bool AHEAD>
__device__ __forceinline__ void raster_splat(bool ok, uint2 rec, float lodf, uint32_t id,
                                             const SplatCam &c, const float4 *rays,
                                             uint64_t *frame)
{
    VS vs;
    ok = ok && vertex_stage(rec, lodf, c, vs);
    int area = 0;
    if (ok && vs.x0 <= vs.x1 && vs.y0 <= vs.y1) area = (vs.x1 - vs.x0 + 1) * (vs.y1 - vs.y0 + 1);
    if (area > 0 && area <= kSmallArea) {
        // the box's pixels row by row, kLoads at a time
        const Slabs sl = slabs_of(vs.vx, vs.vy, vs.vz, vs.half);
        const uint32_t turn = c.W - (uint32_t)(vs.x1 - vs.x0);   // from a row's end to the next row
        uint32_t p = (uint32_t)vs.y0 * c.W + (uint32_t)vs.x0, end = p + (uint32_t)(vs.x1 - vs.x0);
        for (int k0 = 0; k0 < area; k0 += kLoads) {
            uint32_t pp[kLoads];
            uint64_t cur[kLoads];
            float4 inv[kLoads];
#pragma unroll
            for (int u = 0; u < kLoads; u++) {
                pp[u] = p;
                cur[u] = 0;
                if (k0 + u < area) cur[u] = frame[p];
                const bool last = p == end;
                p += last ? turn : 1u;
                end += last ? c.W : 0u;
            }
            // AHEAD: the rays of the pixels that pass the bound, together
#pragma unroll
            for (int u = 0; u < kLoads; u++) {
                inv[u] = make_float4(1.0f, 1.0f, 1.0f, 0.0f);
                if (AHEAD && vs.lb <= cur[u]) inv[u] = rays[pp[u]];
            }
#pragma unroll
            for (int u = 0; u < kLoads; u++)
                if (vs.lb <= cur[u])
                    fragment_test(c, AHEAD ? inv[u] : rays[pp[u]], frame, sl, id, pp[u], cur[u]);
        }
    }
    uint64_t big = __ballot(area > kSmallArea);
    const int lane = (int)(threadIdx.x & 63u);
    while (big) {
        // up to kGroup sprites; lane k takes their pixels k, k + 64, ... row
        // by row, the column and row advancing by 64 % w and 64 / w per step.
        // The quotients come from an approximate reciprocal: for a < 2^7 the
        // fraction of (a + 1/2)/w is at least 1/(2w) >= 2^-12 away from an
        // integer, far above the reciprocal's error, so the floor is exact.
        WaveSprite sp[kGroup];
        int row[kGroup], col[kGroup];
        int amax = 0;
#pragma unroll
        for (int g = 0; g < kGroup; g++) {
            sp[g] = WaveSprite{};
            sp[g].w = 1;
            row[g] = col[g] = 0;
            if (big) {
                const int src = __builtin_ctzll(big);
                big &= big - 1ull;
                sp[g] = wave_sprite(vs, area, id, src);
                const float rw = __builtin_amdgcn_rcpf((float)sp[g].w);
                sp[g].dq = (int)(64.5f * rw);
                sp[g].dr = 64 - sp[g].dq * sp[g].w;
                row[g] = (int)(((float)lane + 0.5f) * rw);
                col[g] = lane - row[g] * sp[g].w;
                amax = sp[g].a > amax ? sp[g].a : amax;
            }
        }
        for (int k0 = 0; k0 < amax; k0 += 64 * kSteps) {
            uint32_t pp[kShared];
            uint64_t cur[kShared];
            uint32_t live = 0;
#pragma unroll
            for (int g = 0; g < kGroup; g++)
#pragma unroll
                for (int j = 0; j < kSteps; j++) {
                    const int u = g * kSteps + j;
                    const int px = sp[g].x0 + col[g], py = sp[g].y0 + row[g];
                    col[g] += sp[g].dr;
                    row[g] += sp[g].dq;
                    if (col[g] >= sp[g].w) { col[g] -= sp[g].w; row[g] += 1; }
                    pp[u] = (uint32_t)py * c.W + (uint32_t)px;
                    cur[u] = 0;
                    if (k0 + 64 * j + lane < sp[g].a) {
                        cur[u] = frame[pp[u]];
                        live |= 1u << u;
                    }
                }
#pragma unroll
            for (int g = 0; g < kGroup; g++)
#pragma unroll
                for (int j = 0; j < kSteps; j++) {
                    const int u = g * kSteps + j;
                    if (((live >> u) & 1u) && sp[g].lb <= cur[u])
                        fragment_test(c, rays[pp[u]], frame, sp[g].s, sp[g].id, pp[u], cur[u]);
                }
        }
    }
}

// Splat i (i >= n: none) of the list.
__device__ __forceinline__ void raster_list(const int16_t *splats, const uint8_t *lod,
                                            uint32_t lod_log2, uint64_t n, uint64_t i,
                                            const SplatCam &c, const float4 *rays, uint64_t *frame)
{
    uint2 rec = make_uint2(0u, 0u);
    float lodf = 1.0f;
    if (i < n) {
        rec = ld_rec(splats, i);
        lodf = (float)(1u << (lod ? lod[i] : lod_log2));
    }
    raster_splat<false>(i < n, rec, lodf, (uint32_t)i, c, rays, frame);
}

// One thread per splat, in list order.
__global__ void __launch_bounds__(256) k_raster(const int16_t *splats, const uint8_t *lod,
                                                uint32_t lod_log2, uint64_t n, SplatCam c,
                                                const float4 *rays, uint64_t *frame)
{
    const uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    raster_list(splats, lod, lod_log2, n, i, c, rays, frame);
}

// ---- block culling and near-to-far order -------------------------------------
// Block b is splats [256b, 256b+256); its bounds are the box of the splat
// centres and their largest half-size.  Blocks wholly outside the view volume
// are dropped; the rest are bucketed by distance and rasterised nearest bucket
// first, so the early depth rejection in the raster sees the occluders first.
constexpr int kBlock = VP_SPLAT_BLOCK;
constexpr int kBins = 256;
// counters: [0, kBins) bin counts, [kBins, 2 kBins) blocks placed per bin, then
// the total and the number of near blocks
constexpr int kTotal = 2 * kBins, kNear = kTotal + 1;
constexpr int kCounters = kNear + 1;

// One wave per block of kBlock splats (lane l takes splats l, l + 64, ...),
// blocks strided over the grid's waves; a wave-wide min reduction, no LDS.
__global__ void __launch_bounds__(256) k_bounds(const int16_t *splats, const uint8_t *lod,
                                                uint32_t lod_log2, uint64_t n, uint64_t nb,
                                                float *bounds, const uint64_t *d_n)
{
    constexpr int PER = kBlock / 64;
    if (d_n) {          // the list length lives in device memory (n is its bound)
        n = min(*d_n, n);
        nb = (n + kBlock - 1) / kBlock;
    }
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t nwaves = (uint64_t)gridDim.x * (blockDim.x >> 6);
    for (uint64_t b = (uint64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); b < nb;
         b += nwaves) {
        float v[7];   // min x y z, max half, -max x y z (all reduced with min)
        for (int k = 0; k < 7; k++) v[k] = INFINITY;
        uint2 r[PER];
        uint32_t lv[PER];
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const uint64_t i = b * kBlock + (uint64_t)q * 64 + lane;
            const bool in = i < n;
            r[q] = in ? *reinterpret_cast<const uint2 *>(splats + 4 * i) : make_uint2(0u, 0u);
            lv[q] = (in && lod) ? (uint32_t)lod[i] : lod_log2;
        }
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const uint64_t i = b * kBlock + (uint64_t)q * 64 + lane;
            if (i < n) {
                const float half = 0.5f * (float)(1u << lv[q]);
                const float cx = (float)(int16_t)(r[q].x & 0xFFFFu) + half;
                const float cy = (float)(int16_t)(r[q].x >> 16) + half;
                const float cz = (float)(int16_t)(r[q].y & 0xFFFFu) + half;
                v[0] = fminf(v[0], cx); v[1] = fminf(v[1], cy); v[2] = fminf(v[2], cz);
                v[3] = fminf(v[3], -half);
                v[4] = fminf(v[4], -cx); v[5] = fminf(v[5], -cy); v[6] = fminf(v[6], -cz);
            }
        }
        for (int k = 0; k < 7; k++)
            for (int d = 32; d >= 1; d >>= 1) v[k] = fminf(v[k], __shfl_xor(v[k], d, 64));
        if (lane == 0) {
            float4 *o = reinterpret_cast<float4 *>(bounds + 8 * b);
            o[0] = make_float4(v[0], v[1], v[2], -v[3]);
            o[1] = make_float4(-v[4], -v[5], -v[6], 0.0f);
        }
    }
}

struct CullPlanes {
    float p[6][4];   // inside: p.x*cx + p.y*cy + p.z*cz + p.w >= 0 for a splat centre
    float eye[3];
    float far_plane;
};

// ---- block occlusion -----------------------------------------------------------
// Most splats of a terrain list lie under its surface (cave walls): behind
// nearer splats on every pixel they cover.  hiz holds, per kHzTile x kHzTile
// pixels, a depth no stored key of the tile is above.  Frame keys only ever
// go down, so a tile's largest key of any earlier moment is such a bound:
// the raster's own waves refresh it from the frame as they go, with no
// ordering against the fragments, and a stale entry only keeps a block that
// could have been dropped.  A block is dropped unread when its depth lower
// bound is above the bound of every tile its sprites can touch.
constexpr int kHzLog = 3, kHzTile = 1 << kHzLog;
__host__ __device__ __forceinline__ uint32_t hz_tiles(uint32_t px)
{
    return (px + kHzTile - 1) >> kHzLog;
}

// A block's screen box in tiles (x0 | x1 << 16, y0 | y1 << 16) and its depth
// lower bound as float bits; bound 0 never drops it.
__device__ __forceinline__ uint4 block_box(const float *o, const SplatCam &c)
{
    const uint4 keep = make_uint4(0u, 0u, 0u, 0u);
    const float half = o[3], W = (float)c.W, H = (float)c.H;
    // view-space corners of the centres' box, their clip coordinates, and the
    // nearest point of the box (grown by half) to the eye
    float vlo[3] = {INFINITY, INFINITY, INFINITY}, vhi[3] = {-INFINITY, -INFINITY, -INFINITY};
    float nx0 = INFINITY, nx1 = -INFINITY, ny0 = INFINITY, ny1 = -INFINITY;
    float wmin = INFINITY, zmin = INFINITY, vmax = 0.0f;
    for (int k = 0; k < 8; k++) {
        const float a[4] = {o[k & 1 ? 4 : 0], o[k & 2 ? 5 : 1], o[k & 4 ? 6 : 2], 1.0f};
        float v[4], q[4];
        mv4(c.T, a, v);
        mv4(c.PR, v, q);
        for (int d = 0; d < 3; d++) {
            vlo[d] = fminf(vlo[d], v[d]);
            vhi[d] = fmaxf(vhi[d], v[d]);
            vmax = fmaxf(vmax, fabsf(v[d]));
        }
        wmin = fminf(wmin, q[3]);
        zmin = fminf(zmin, q[2]);
        const float nx = q[0] / q[3], ny = q[1] / q[3];
        nx0 = fminf(nx0, nx); nx1 = fmaxf(nx1, nx);
        ny0 = fminf(ny0, ny); ny1 = fmaxf(ny1, ny);
    }
    // near the eye the projection's bounds are loose and its rounding grows
    if (!(wmin > 1.0f && zmin > 1.0f && vmax < 1e6f && half <= 128.0f)) return keep;
    // a splat in the view volume projects into the corners' hull and into the
    // screen; its sprite reaches at most hs further.  The margin covers the
    // rounding of both computations (some 1e-6 of vmax / wmin of the screen).
    const float ratio = W / H;
    float red = fmaxf(fmaxf(fabsf(nx0), fabsf(nx1)) * ratio, fmaxf(fabsf(ny0), fabsf(ny1)));
    red = fmaxf(fminf(red, fmaxf(ratio, 1.0f)) + 0.04f, 1.0f);
    float ps = H * 1.1f / zmin * red * (2.0f * half) * 1.01f;
    ps = fminf(fmaxf(ps, 1.0f), 2048.0f);
    const float m = 0.5f * ps + 2.0f + 1e-5f * (vmax / wmin) * fmaxf(W, H);
    const float x0 = fmaxf((fmaxf(nx0, -1.0f) + 1.0f) * (0.5f * W) - m, 0.0f);
    const float x1 = fminf((fminf(nx1, 1.0f) + 1.0f) * (0.5f * W) + m, W - 1.0f);
    const float y0 = fmaxf((fmaxf(ny0, -1.0f) + 1.0f) * (0.5f * H) - m, 0.0f);
    const float y1 = fminf((fminf(ny1, 1.0f) + 1.0f) * (0.5f * H) + m, H - 1.0f);
    if (!(x0 <= x1 && y0 <= y1)) return keep;
    // as the splats' own lower bound (vertex_stage), below each of theirs
    float dd = 0.0f;
    for (int d = 0; d < 3; d++) {
        const float e = fmaxf(fmaxf(vlo[d] - half, -vhi[d] - half), 0.0f);
        dd += e * e;
    }
    const float lb = sqrtf(dd) * 0.998f / c.far_plane;
    if (!(lb > 0.0f)) return keep;
    return make_uint4(((uint32_t)x0 >> kHzLog) | ((uint32_t)x1 >> kHzLog) << 16,
                      ((uint32_t)y0 >> kHzLog) | ((uint32_t)y1 >> kHzLog) << 16,
                      __float_as_uint(lb), 0u);
}

// The queue of a wave is written and read by different lanes of that wave.
__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The tile bounds of a block's box, row by row over the lanes of a wave, all
// of whose lanes call with the same box.  The first 64 or fewer are loaded
// ahead (box_first); more of them are read when the block is tested.
struct BoxWalk {
    uint32_t x0, y0, w, h, rows, r, x;
};

__device__ __forceinline__ BoxWalk box_walk(const uint4 box)
{
    BoxWalk k;
    const uint32_t lane = threadIdx.x & 63u;
    k.x0 = box.x & 0xFFFFu;
    k.y0 = box.y & 0xFFFFu;
    k.w = (box.x >> 16) - k.x0 + 1u;
    k.h = (box.y >> 16) - k.y0 + 1u;
    k.rows = k.w > 64u ? 0u : 64u / k.w;     // wide boxes belong to near blocks: never hidden
    k.r = lane / k.w;
    k.x = lane - k.r * k.w;
    return k;
}

__device__ __forceinline__ uint32_t box_at(const BoxWalk &k, uint32_t y, const uint32_t *hiz,
                                           uint32_t tx)
{
    return k.r < k.rows && y + k.r < k.h ? hiz[(size_t)(k.y0 + y + k.r) * tx + k.x0 + k.x] : 0u;
}

// Whether every tile of the box is bounded below the block's depth lb;
// first: box_at of its first rows, read at any earlier moment of the frame.
__device__ __forceinline__ bool box_hidden(const BoxWalk &k, uint32_t lb, uint32_t first,
                                           const uint32_t *hiz, uint32_t tx)
{
    if (k.rows == 0u || lb == 0u || __ballot(first >= lb)) return false;
    for (uint32_t y = k.rows; y < k.h; y += k.rows)
        if (__ballot(box_at(k, y, hiz, tx) >= lb)) return false;
    return true;
}

// Largest value over each group of 8 consecutive lanes.
__device__ __forceinline__ uint32_t max8(uint32_t v)
{
    // quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, true));
    return v;
}

// Groups of eight tiles side by side.
__host__ __device__ __forceinline__ uint32_t hz_groups(uint32_t W, uint32_t H)
{
    return ((hz_tiles(W) + 7u) >> 3) * hz_tiles(H);
}

// Refresh the tile groups [g0, g1) from the frame: lane l reads column l of
// the group's 64 x 8 pixels, row by row (whole lines), and the tile's bound is
// the largest depth of its eight lanes.
__device__ __forceinline__ void hiz_refresh(const uint64_t *frame, uint32_t *hiz, uint32_t W,
                                            uint32_t H, uint32_t g0, uint32_t g1)
{
    const uint32_t tx = hz_tiles(W), gx = (tx + 7u) >> 3, lane = threadIdx.x & 63u;
    for (uint32_t g = g0; g < g1; g++) {
        const uint32_t ty = g / gx, px = (g - ty * gx) * 64u + lane;
        uint32_t k[kHzTile], d = 0u;
#pragma unroll
        for (int j = 0; j < kHzTile; j++) {
            const uint32_t py = ty * kHzTile + j;
            k[j] = 0u;
            if (px < W && py < H) k[j] = (uint32_t)(frame[(size_t)py * W + px] >> 32);
        }
#pragma unroll
        for (int j = 0; j < kHzTile; j++) d = max(d, k[j]);
        d = max8(d);
        if ((lane & 7u) == 0 && px < W)
            __hip_atomic_store(hiz + (size_t)ty * tx + (px >> kHzLog), d, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }
}

__device__ __forceinline__ uint32_t block_bin(const float *bounds, uint64_t b,
                                              const CullPlanes &cp)
{
    const float *o = bounds + 8 * b;
    const float lo[3] = {o[0], o[1], o[2]}, hi[3] = {o[4], o[5], o[6]};
    if (!(lo[0] <= hi[0])) return 0xFFFFFFFFu;   // empty block
    for (int k = 0; k < 6; k++) {
        // the largest value of the plane function over the box of centres
        float f = cp.p[k][3], mag = fabsf(cp.p[k][3]);
        for (int a = 0; a < 3; a++) {
            const float c = cp.p[k][a];
            f += c * (c > 0.0f ? hi[a] : lo[a]);
            mag += fabsf(c) * fmaxf(fabsf(lo[a]), fabsf(hi[a]));
        }
        // the rounding of the vertex stage's clip test is far below 1e-3 of mag
        if (f < -1e-3f * mag) return 0xFFFFFFFFu;
    }
    float dd = 0.0f;
    for (int a = 0; a < 3; a++) {
        const float e = fmaxf(fmaxf(lo[a] - o[3] - cp.eye[a], cp.eye[a] - hi[a] - o[3]), 0.0f);
        dd += e * e;
    }
    const float t = sqrtf(sqrtf(dd) / cp.far_plane);
    return (uint32_t)fminf(t * (float)kBins, (float)(kBins - 1));
}

// Bins of the blocks, counted per workgroup in LDS and added to the global
// counts once per workgroup and bin.
__global__ void __launch_bounds__(256) k_blk_cull(const float *bounds, uint64_t nb, CullPlanes cp,
                                                  SplatCam c, uint32_t *bin, uint4 *box,
                                                  uint32_t *cnt, const uint64_t *d_n)
{
    __shared__ uint32_t hist[kBins];
    if (d_n) nb = min((*d_n + kBlock - 1) / kBlock, nb);
    for (int k = threadIdx.x; k < kBins; k += blockDim.x) hist[k] = 0u;
    __syncthreads();
    for (uint64_t b = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; b < nb;
         b += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t k = block_bin(bounds, b, cp);
        bin[b] = k;
        if (k != 0xFFFFFFFFu) {
            atomicAdd(hist + k, 1u);
            if (box) box[b] = block_box(bounds + 8 * b, c);
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < kBins; k += blockDim.x)
        if (hist[k]) atomicAdd(cnt + k, hist[k]);
}

// Blocks into their bins' ranges of the order: per 256 blocks, a workgroup
// counts its blocks per bin in LDS, reserves each bin's share with one global
// add, then places every block inside its share.  Every workgroup scans the bin
// counts for itself; the first one notes their total, and the blocks of the
// first near_bin bins.
__global__ void __launch_bounds__(kBins) k_blk_scatter(const uint32_t *bin, uint64_t nb,
                                                       uint32_t *cnt, uint32_t *order,
                                                       const uint64_t *d_n, uint32_t near_bin)
{
    __shared__ uint32_t num[kBins], base[kBins], wsum[kBins / 64];
    if (d_n) nb = min((*d_n + kBlock - 1) / kBlock, nb);
    uint32_t wt;
    uint32_t first = wave_excl_scan(cnt[threadIdx.x], wt);
    if ((threadIdx.x & 63u) == 0) wsum[threadIdx.x >> 6] = wt;
    __syncthreads();
    for (uint32_t w = 0; w < threadIdx.x >> 6; w++) first += wsum[w];
    if (blockIdx.x == 0) {
        if (threadIdx.x == kBins - 1) cnt[kTotal] = first + cnt[kBins - 1];
        if (threadIdx.x + 1 == near_bin) cnt[kNear] = first + cnt[threadIdx.x];
    }
    for (uint64_t b0 = blockIdx.x * (uint64_t)blockDim.x; b0 < nb;
         b0 += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t b = b0 + threadIdx.x;
        num[threadIdx.x] = 0u;
        __syncthreads();
        const uint32_t k = b < nb ? bin[b] : 0xFFFFFFFFu;
        if (k != 0xFFFFFFFFu) atomicAdd(num + k, 1u);
        __syncthreads();
        const uint32_t mine = num[threadIdx.x];
        base[threadIdx.x] = first + (mine ? atomicAdd(cnt + kBins + threadIdx.x, mine) : 0u);
        num[threadIdx.x] = 0u;
        __syncthreads();
        if (k != 0xFFFFFFFFu) order[base[k] + atomicAdd(num + k, 1u)] = (uint32_t)b;
        __syncthreads();
    }
}

// Whether splat (rec, lodf) can still win a pixel of its sprite, as far as the
// tile bounds tell: approximate arithmetic, every bound on the safe side, and
// true wherever the approximation is loose (near the eye, large sprites).
__device__ __forceinline__ bool splat_open(const uint2 rec, float lodf, const SplatCam &c,
                                           const uint32_t *hiz, uint32_t tx)
{
    const float half = 0.5f * lodf, W = (float)c.W, H = (float)c.H;
    const float a[3] = {(float)(int16_t)(rec.x & 0xFFFFu) + half, (float)(int16_t)(rec.x >> 16) + half,
                        (float)(int16_t)(rec.y & 0xFFFFu) + half};
    float v[4], q[4];
#pragma unroll
    for (int r = 0; r < 4; r++)
        v[r] = fmaf(c.T[r], a[0], fmaf(c.T[4 + r], a[1], fmaf(c.T[8 + r], a[2], c.T[12 + r])));
#pragma unroll
    for (int r = 0; r < 4; r++)
        q[r] = fmaf(c.PR[r], v[0], fmaf(c.PR[4 + r], v[1], fmaf(c.PR[8 + r], v[2], c.PR[12 + r] * v[3])));
    // outside the view volume by more than rounding: no fragment
    const float cw = q[3] + 1e-4f * fabsf(q[3]) + 1e-3f;
    if (!(fabsf(q[0]) <= cw && fabsf(q[1]) <= cw && fabsf(q[2]) <= cw)) return false;
    if (!(q[3] > 2.0f && q[2] > 2.0f)) return true;
    const float rw = __builtin_amdgcn_rcpf(q[3]);
    const float nx = q[0] * rw, ny = q[1] * rw;
    const float red = fmaxf(fmaxf(fabsf(nx) * (W / H), fabsf(ny)) + 0.04f, 1.0f);
    const float ps = H * 1.12f * lodf * red * __builtin_amdgcn_rcpf(q[2]);
    const float m = 0.5f * fmaxf(ps, 1.0f) + 0.25f;
    if (!(m < 0.5f * kHzTile)) return true;       // wider than two tiles
    const float wx = (nx + 1.0f) * (0.5f * W), wy = (ny + 1.0f) * (0.5f * H);
    const uint32_t x0 = (uint32_t)fmaxf(wx - m, 0.0f) >> kHzLog;
    const uint32_t x1 = (uint32_t)fminf(fmaxf(wx + m, 0.0f), W - 1.0f) >> kHzLog;
    const uint32_t y0 = (uint32_t)fmaxf(wy - m, 0.0f) >> kHzLog;
    const uint32_t y1 = (uint32_t)fminf(fmaxf(wy + m, 0.0f), H - 1.0f) >> kHzLog;
    if (x0 > x1 || y0 > y1) return true;          // rounding at the screen's edge
    float dd = 0.0f;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const float e = fmaxf(fabsf(v[d]) - half, 0.0f);
        dd = fmaf(e, e, dd);
    }
    const uint32_t lb = __float_as_uint(sqrtf(dd) * 0.998f * __builtin_amdgcn_rcpf(c.far_plane));
    uint32_t far = max(hiz[(size_t)y0 * tx + x0], hiz[(size_t)y0 * tx + x1]);
    far = max(far, max(hiz[(size_t)y1 * tx + x0], hiz[(size_t)y1 * tx + x1]));
    return far >= lb;
}

// Blocks whose splats are at least this many pixels wide are handed out in
// quarters: their sprites cost so much that a wave with a whole block of them
// outlasts the others (two views close to a 7.7 M list: 5870 against 9860 us at
// 1697x1495, 13310 against 20970 at 2422x2321; to a 31 M list at 1920x1080: 4370
// against 7620).  Farther blocks are cheaper whole, one look at their bounds each
// (all of them in quarters: 1.2x the time).
constexpr float kNearPixels = 5.0f;
// Frames of up to this many pixels are rasterised without the tile bounds: the
// whole frame stays in the L2s, and rejecting a fragment by its own load is
// then cheaper than a pass over bounds (183x151 of a 65 M list: 340 against
// 421 us, 489x499 of 114 M: 524 against 552 us; 757x591: 489 against 498 us, and
// 928x743 of 3.3 M: 152 against 131 us).
constexpr uint64_t kFewPixels = 1u << 18;
// Tile groups (4 KiB of keys each) a wave refreshes at a time.  Its whole share
// is up to 4 groups on 256 CUs at 3840x2160 and 128 at 16384x16384, where reading
// all of it every second block cost more than the bounds saved (four far views of
// a 31 M list 207.6 ms; 4 at a time 165.2; without the bounds 175; one at a time
// 2422x2321 takes 5430 against 5060 us).
constexpr uint32_t kRefresh = 4;
constexpr uint32_t kHeld = kBlock + 64;   // a wave's queue: less than a wave, and a block
// Wave w takes the ordered blocks w, w + G, w + 2G, ... (G waves): every wave
// starts at the near end of the order, no counter is shared, and the waves
// never wait for each other.  A block that is hidden is skipped; of the others
// the splats that may still win a pixel go to the wave's queue in LDS, and
// full waves of them are rasterised.  Every second block a wave refreshes up to
// kRefresh groups of its share of the tile bounds, in turn (every block or every
// fourth: within 3%).
// Bound by latency and instructions together (vector instructions fill a third of
// the SIMDs' cycles, 1.3e8 of them a frame): a 1920x1080 frame of a 133.5 M list
// has 297 K blocks, 76 M splats in view, of which 60% and 27% are not dropped here
// (four worlds: 55-60%, 21-27%); each splat rasterised costs some hundred
// instructions per 4 pixels.  1573 -> 846 us per frame (kernel) against rasterising
// every splat in view.  The order's counter is not shared on purpose: an atomic
// ticket per block (13 ns each on one address) took 1242-3786 us.
__global__ void __launch_bounds__(kBlock) k_raster_blocks(const int16_t *splats,
                                                           const uint8_t *lod, uint32_t lod_log2,
                                                           uint64_t n, SplatCam c,
                                                           const float4 *rays, uint64_t *frame,
                                                           const uint32_t *order,
                                                           const uint4 *box, uint32_t *hiz,
                                                           const uint32_t *cnt,
                                                           const uint64_t *d_n,
                                                           const uint32_t *tiles_ok)
{
    // splats that may still win a pixel: record, index and level
    struct Held {
        uint32_t x[kHeld], y[kHeld], id[kHeld];
        uint8_t lv[kHeld];
    };
    __shared__ Held queue[kBlock / 64];
    if (tiles_ok && *tiles_ok) return;    // the screen-tile path resolved this frame
    const uint32_t total = cnt[kTotal];
    if (d_n) n = min(*d_n, n);
    const uint32_t tx = hz_tiles(c.W), nt = hz_groups(c.W, c.H);
    const uint32_t nw = gridDim.x * (blockDim.x >> 6), lane = threadIdx.x & 63u;
    // consecutive blocks of the order go to different workgroups
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane(
        (int)(blockIdx.x + gridDim.x * (threadIdx.x >> 6)));
    Held &q = queue[threadIdx.x >> 6];
    const uint32_t share = (nt + nw - 1) / nw;
    const uint32_t h0 = min(w * share, nt), h1 = min(h0 + share, nt);
    constexpr int PER = kBlock / 64;
    uint32_t held = 0, turn = 0, hg = h0;
    auto flush = [&](uint32_t at, bool ok) {
        const uint32_t e = at + lane;
        const uint2 rec = ok ? make_uint2(q.x[e], q.y[e]) : make_uint2(0u, 0u);
        raster_splat<true>(ok, rec, ok ? (float)(1u << q.lv[e]) : 1.0f, ok ? q.id[e] : 0u, c, rays, frame);
    };
    // units of work: the quarters of the near blocks, then whole blocks
    const uint32_t near = cnt[kNear], units = total + 3u * near;
    // one block ahead: its box and its first tile bounds, so that their loads
    // are in flight while the block before it is worked on
    uint32_t b = 0, lb = 0, first = 0, part = 0;
    BoxWalk walk = {};
    uint2 rec[PER];
    uint32_t lv[PER];
    auto fetch = [&](uint32_t t) {
        const bool quarter = t < 4u * near;
        b = (uint32_t)__builtin_amdgcn_readfirstlane((int)order[quarter ? t >> 2 : t - 3u * near]);
        part = quarter ? 1u << (t & 3u) : (1u << PER) - 1u;
        const uint4 bx = box[b];
        lb = bx.z;
        walk = box_walk(bx);
        first = box_at(walk, 0u, hiz, tx);
    };
    auto records = [&]() {
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const uint64_t i = (uint64_t)b * kBlock + (uint64_t)(k * 64) + lane;
            rec[k] = make_uint2(0u, 0u);
            lv[k] = lod_log2;
            if (!((part >> k) & 1u)) continue;
            if (i < n) {
                rec[k] = *reinterpret_cast<const uint2 *>(splats + 4 * i);
                if (lod) lv[k] = lod[i];
            }
        }
    };
    if (w < units) fetch(w);
    for (uint32_t t = w; t < units; t += nw) {
        const bool hidden = box_hidden(walk, lb, first, hiz, tx);
        if (!hidden) {
            records();
            bool open[PER];
#pragma unroll
            for (int k = 0; k < PER; k++) {
                const uint64_t i = (uint64_t)b * kBlock + (uint64_t)(k * 64) + lane;
                open[k] = ((part >> k) & 1u) && i < n &&
                          splat_open(rec[k], (float)(1u << lv[k]), c, hiz, tx);
            }
#pragma unroll
            for (int k = 0; k < PER; k++) {
                if (!((part >> k) & 1u)) continue;
                const uint64_t m = __ballot(open[k]);
                const uint32_t e = held + __builtin_amdgcn_mbcnt_hi(
                    (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                if (open[k]) {
                    q.x[e] = rec[k].x;
                    q.y[e] = rec[k].y;
                    q.id[e] = b * kBlock + k * 64 + lane;
                    q.lv[e] = (uint8_t)lv[k];
                }
                held += (uint32_t)__popcll(m);
            }
        }
        if (t + nw < units) fetch(t + nw);
        wave_fence();
        while (held >= 64) {
            held -= 64;
            flush(held, true);
        }
        wave_fence();
        if (++turn & 1u) {
            const uint32_t he = min(hg + kRefresh, h1);
            hiz_refresh(frame, hiz, c.W, c.H, hg, he);
            hg = he < h1 ? he : h0;
        }
    }
    flush(0u, lane < held);
}

// The visible blocks without the tile bounds (frames of up to kFewPixels, and
// cameras that bounds_hold rules out): a workgroup per block, a splat per thread.
__global__ void __launch_bounds__(kBlock) k_raster_few(const int16_t *splats, const uint8_t *lod,
                                                        uint32_t lod_log2, uint64_t n, SplatCam c,
                                                        const float4 *rays, uint64_t *frame,
                                                        const uint32_t *order,
                                                        const uint32_t *cnt, const uint64_t *d_n,
                                                        const uint32_t *tiles_ok)
{
    if (tiles_ok && *tiles_ok) return;    // the screen-tile path resolved this frame
    const uint32_t total = cnt[kTotal];
    if (d_n) n = min(*d_n, n);
    for (uint32_t t = blockIdx.x; t < total; t += gridDim.x) {
        const uint64_t i = (uint64_t)order[t] * kBlock + threadIdx.x;
        uint2 rec = make_uint2(0u, 0u);
        uint32_t lv = lod_log2;
        if (i < n) {
            rec = *reinterpret_cast<const uint2 *>(splats + 4 * i);
            if (lod) lv = lod[i];
        }
        raster_splat<true>(i < n, rec, (float)(1u << lv), (uint32_t)i, c, rays, frame);
    }
}

// ---- screen-tile resolve ------------------------------------------------------
// The visible blocks' splats are binned into kTile x kTile pixel tiles; each
// tile is then resolved by one workgroup with its rays and frame keys in LDS,
// so a fragment costs LDS reads and one LDS atomicMin instead of global
// gathers and an L2 atomic.  A splat whose pixel box is at most kTileSide
// pixels on a side goes into each tile it touches (at most four entries); a
// larger one -- a near splat, few of them, many pixels each -- goes to the big
// list, which is drawn first against the frame in device memory, spread over
// the whole grid.  The tiles then start from those keys, so the near
// occluders reject the small splats behind them from the first entry on.
// The keys are the same (depth bits << 32 | id) and min is order-free, so the
// frame is identical to the global path's.  If a frame needs more entries
// than the buffers hold, the scan leaves the flag clear and the global path
// (k_raster_blocks) draws the whole frame instead.
constexpr int kTileLog = 5, kTile = 1 << kTileLog, kTilePx = kTile * kTile;
constexpr int kTileSide = 8;                  // larger pixel boxes go to the big list
static_assert(kTilePx % kBlock == 0, "k_tile_raster: whole pixels per thread");
constexpr uint32_t kMaxTiles = 8192;          // LDS bins of the binning kernels: 32 KiB
constexpr uint32_t kItem = 8192;              // tile entries per raster work item
constexpr uint32_t kSingle = 1u << 31;        // item flag: the tile's only item
// tile counters (u32): [0] raster items, [1] entries, [2] big splats counted,
// [3] flag: the tile path draws this frame, [4] big-list cursor
constexpr int kTcItems = 0, kTcPairs = 1, kTcBig = 2, kTcOk = 3, kTcBigCur = 4, kTcWords = 8;

struct TileBufs {
    uint32_t tx, ty, nt;      // tiles across, down, total
    uint32_t *hist;           // [G][nt] per-workgroup entry counts
    uint32_t *cnt;            // [nt] entries per tile
    uint32_t *cur;            // [nt] placement cursors
    uint32_t *tc;             // kTcWords counters
    uint4    *items;          // (tile | kSingle, begin, end, 0)
    uint32_t  item_cap;
    uint32_t *pairs;          // splat index per entry, tile-major
    uint32_t  pair_cap;
    uint32_t *big;            // splat indices of the big list
    uint32_t  big_cap;
};

// Vertex stage of splat i (i < n), and the tiles its pixel box touches:
// 0 none, 1 tile entries (t0 = first tile, span bits: +1 tile in x, +1 in y),
// 2 big.
__device__ __forceinline__ int splat_tiles(const int16_t *splats, const uint8_t *lod,
                                           uint32_t lod_log2, uint64_t i, const SplatCam &c,
                                           uint32_t tx, VS &vs, uint32_t &t0, uint32_t &span)
{
    const float lodf = (float)(1u << (lod ? lod[i] : lod_log2));
    if (!vertex_stage(ld_rec(splats, i), lodf, c, vs)) return 0;
    if (vs.x0 > vs.x1 || vs.y0 > vs.y1) return 0;
    if (vs.x1 - vs.x0 >= kTileSide || vs.y1 - vs.y0 >= kTileSide) return 2;
    // a box of at most kTileSide <= kTile pixels touches at most 2 x 2 tiles
    const uint32_t a = (uint32_t)vs.x0 >> kTileLog, b = (uint32_t)vs.x1 >> kTileLog;
    const uint32_t d = (uint32_t)vs.y0 >> kTileLog, e = (uint32_t)vs.y1 >> kTileLog;
    t0 = d * tx + a;
    span = (b - a) | ((e - d) << 1);
    return 1;
}

__global__ void k_tile_reset(uint32_t *cnt, uint32_t nt, uint32_t *tc)
{
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < nt; t += gridDim.x * blockDim.x)
        cnt[t] = 0u;
    if (blockIdx.x == 0 && threadIdx.x < kTcWords) tc[threadIdx.x] = 0u;
}

// Workgroup g takes the ordered visible blocks g, g + G, ... (the same
// assignment as k_tile_scatter) and counts its entries per tile in LDS; the
// counts go to its row of the histogram and are added to the tile totals.
__global__ void __launch_bounds__(kBlock) k_tile_count(const int16_t *splats, const uint8_t *lod,
                                                       uint32_t lod_log2, uint64_t n, SplatCam c,
                                                       const uint32_t *order, const uint32_t *cnt,
                                                       const uint64_t *d_n, TileBufs tb)
{
    extern __shared__ uint32_t hist[];
    for (uint32_t t = threadIdx.x; t < tb.nt; t += blockDim.x) hist[t] = 0u;
    __syncthreads();
    const uint32_t total = cnt[kTotal];
    if (d_n) n = min(*d_n, n);
    uint32_t nbig = 0;
    for (uint32_t b = blockIdx.x; b < total; b += gridDim.x) {
        const uint64_t i = (uint64_t)order[b] * kBlock + threadIdx.x;
        if (i >= n) continue;
        VS vs;
        uint32_t t0 = 0, span = 0;
        const int k = splat_tiles(splats, lod, lod_log2, i, c, tb.tx, vs, t0, span);
        if (k == 2) nbig++;
        if (k != 1) continue;
        atomicAdd(hist + t0, 1u);
        if (span & 1u) atomicAdd(hist + t0 + 1, 1u);
        if (span & 2u) atomicAdd(hist + t0 + tb.tx, 1u);
        if (span == 3u) atomicAdd(hist + t0 + tb.tx + 1, 1u);
    }
    __syncthreads();
    uint32_t *row = tb.hist + (size_t)blockIdx.x * tb.nt;
    for (uint32_t t = threadIdx.x; t < tb.nt; t += blockDim.x) {
        const uint32_t v = hist[t];
        row[t] = v;
        if (v) atomicAdd(tb.cnt + t, v);
    }
    for (int d = 32; d >= 1; d >>= 1) nbig += (uint32_t)__shfl_xor((int)nbig, d, 64);
    if ((threadIdx.x & 63u) == 0 && nbig) atomicAdd(tb.tc + kTcBig, nbig);
}

// One workgroup: tile offsets (exclusive scan of the counts), placement
// cursors, the raster items (runs of at most kItem entries of one tile) and
// the flag that hands the frame to the tile path when everything fits.
constexpr int kScanThreads = 1024;
__device__ __forceinline__ uint64_t shfl_up64(uint64_t v, int d)
{
    const uint32_t lo = (uint32_t)__shfl_up((int)(uint32_t)v, d, 64);
    const uint32_t hi = (uint32_t)__shfl_up((int)(uint32_t)(v >> 32), d, 64);
    return ((uint64_t)hi << 32) | lo;
}
__global__ void __launch_bounds__(kScanThreads) k_tile_scan(TileBufs tb)
{
    __shared__ uint64_t wsum[2][kScanThreads / 64];
    __shared__ uint32_t s_ok;
    const uint32_t per = (tb.nt + kScanThreads - 1) / kScanThreads;
    const uint32_t t0 = min(threadIdx.x * per, tb.nt), t1 = min(t0 + per, tb.nt);
    // entry totals in 64 bits: four entries per splat can pass 2^32
    uint64_t sc = 0, si = 0;
    for (uint32_t t = t0; t < t1; t++) {
        const uint32_t v = tb.cnt[t];
        sc += v;
        si += (v + kItem - 1) / kItem;
    }
    // block-wide exclusive scans of (entries, items)
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    uint64_t ic = sc, ii = si;
    for (int d = 1; d < 64; d <<= 1) {
        const uint64_t a = shfl_up64(ic, d), b = shfl_up64(ii, d);
        if ((int)lane >= d) { ic += a; ii += b; }
    }
    if (lane == 63) { wsum[0][w] = ic; wsum[1][w] = ii; }
    __syncthreads();
    uint64_t bc = 0, bi = 0, tc = 0, ti = 0;
    for (uint32_t k = 0; k < kScanThreads / 64; k++) {
        if (k < w) { bc += wsum[0][k]; bi += wsum[1][k]; }
        tc += wsum[0][k];
        ti += wsum[1][k];
    }
    if (threadIdx.x == 0) {
        const uint32_t big = tb.tc[kTcBig];
        const bool ok = tc <= tb.pair_cap && ti <= tb.item_cap && big <= tb.big_cap;
        s_ok = ok ? 1u : 0u;
        tb.tc[kTcPairs] = (uint32_t)min(tc, (uint64_t)0xFFFFFFFFu);
        tb.tc[kTcItems] = ok ? (uint32_t)ti : 0u;
        tb.tc[kTcOk] = s_ok;
    }
    __syncthreads();
    if (!s_ok) return;
    // every total now fits in 32 bits
    uint32_t off = (uint32_t)(bc + ic - sc), io = (uint32_t)(bi + ii - si);
    for (uint32_t t = t0; t < t1; t++) {
        const uint32_t v = tb.cnt[t];
        tb.cur[t] = off;
        const uint32_t k = (v + kItem - 1) / kItem;
        for (uint32_t q = 0; q < k; q++) {
            const uint32_t b = off + q * kItem, e = min(b + kItem, off + v);
            tb.items[io + q] = make_uint4(t | (k == 1 ? kSingle : 0u), b, e, 0u);
        }
        off += v;
        io += k;
    }
}

// The same blocks as k_tile_count: reserve the workgroup's range of every
// tile it touches, then place each entry (LDS cursors); big splats are
// appended to the big list.
__global__ void __launch_bounds__(kBlock) k_tile_scatter(const int16_t *splats, const uint8_t *lod,
                                                         uint32_t lod_log2, uint64_t n, SplatCam c,
                                                         const uint32_t *order, const uint32_t *cnt,
                                                         const uint64_t *d_n, TileBufs tb)
{
    extern __shared__ uint32_t lcur[];
    if (!tb.tc[kTcOk]) return;
    const uint32_t *row = tb.hist + (size_t)blockIdx.x * tb.nt;
    for (uint32_t t = threadIdx.x; t < tb.nt; t += blockDim.x) {
        const uint32_t v = row[t];
        lcur[t] = v ? atomicAdd(tb.cur + t, v) : 0u;
    }
    __syncthreads();
    const uint32_t total = cnt[kTotal];
    if (d_n) n = min(*d_n, n);
    const uint32_t lane = threadIdx.x & 63u;
    for (uint32_t b = blockIdx.x; b < total; b += gridDim.x) {
        const uint64_t i = (uint64_t)order[b] * kBlock + threadIdx.x;
        VS vs;
        uint32_t t0 = 0, span = 0;
        const int k = i < n ? splat_tiles(splats, lod, lod_log2, i, c, tb.tx, vs, t0, span) : 0;
        if (k == 1) {
            uint32_t q = atomicAdd(lcur + t0, 1u);
            if (q < tb.pair_cap) tb.pairs[q] = (uint32_t)i;
            if (span & 1u) {
                q = atomicAdd(lcur + t0 + 1, 1u);
                if (q < tb.pair_cap) tb.pairs[q] = (uint32_t)i;
            }
            if (span & 2u) {
                q = atomicAdd(lcur + t0 + tb.tx, 1u);
                if (q < tb.pair_cap) tb.pairs[q] = (uint32_t)i;
            }
            if (span == 3u) {
                q = atomicAdd(lcur + t0 + tb.tx + 1, 1u);
                if (q < tb.pair_cap) tb.pairs[q] = (uint32_t)i;
            }
        }
        const uint64_t m = __ballot(k == 2);
        if (m) {
            uint32_t base = 0;
            if (lane == (uint32_t)__builtin_ctzll(m))
                base = atomicAdd(tb.tc + kTcBigCur, (uint32_t)__popcll(m));
            base = (uint32_t)lane_i((int)base, __builtin_ctzll(m));
            if (k == 2) {
                const uint32_t q = base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
                if (q < tb.big_cap) tb.big[q] = (uint32_t)i;
            }
        }
    }
}

// One tile's fragment in LDS: lp indexes the tile's pixel.
__device__ __forceinline__ void fragment_lds(const float4 *lray, uint64_t *lkey, float far_plane,
                                             float vx, float vy, float vz, float half, uint32_t id,
                                             uint64_t lb, int lp)
{
    const uint64_t cur = lkey[lp];
    if (lb > cur) return;
    const float4 inv = lray[lp];
    float t0, t1;
    aabb(vx - half, vx + half, vy - half, vy + half, vz - half, vz + half, inv.x, inv.y, inv.z, t0,
         t1);
    if (!(t0 <= t1)) return;
    float d = t0 / far_plane;
    if (!(d < 1.0f)) return;
    if (d <= 0.0f) d = 0.0f;
    const uint64_t key = ((uint64_t)__float_as_uint(d) << 32) | id;
    if (key < cur) atomicMin(reinterpret_cast<unsigned long long *>(lkey + lp), key);
}

// Entry i (i >= n: none) of one lane, clipped to the tile at (px0, py0);
// every lane of the wave calls it.  As raster_splat: boxes of up to
// kSmallArea pixels by their own lane, larger ones by the whole wave.
__device__ __forceinline__ void tile_splat(const int16_t *splats, const uint8_t *lod,
                                           uint32_t lod_log2, uint64_t n, uint64_t i,
                                           const SplatCam &c, int px0, int py0,
                                           const float4 *lray, uint64_t *lkey)
{
    VS vs;
    bool ok = false;
    if (i < n) {
        const float lodf = (float)(1u << (lod ? lod[i] : lod_log2));
        ok = vertex_stage(ld_rec(splats, i), lodf, c, vs);
    }
    int x0 = 0, x1 = -1, y0 = 0, y1 = -1;
    if (ok) {
        x0 = vs.x0 > px0 ? vs.x0 : px0;
        x1 = vs.x1 < px0 + kTile - 1 ? vs.x1 : px0 + kTile - 1;
        y0 = vs.y0 > py0 ? vs.y0 : py0;
        y1 = vs.y1 < py0 + kTile - 1 ? vs.y1 : py0 + kTile - 1;
    }
    int area = 0;
    if (x0 <= x1 && y0 <= y1) area = (x1 - x0 + 1) * (y1 - y0 + 1);
    const uint32_t id = (uint32_t)i;
    if (area > 0 && area <= kSmallArea) {
        for (int py = y0; py <= y1; py++) {
            for (int px = x0; px <= x1; px++) {
                fragment_lds(lray, lkey, c.far_plane, vs.vx, vs.vy, vs.vz, vs.half, id, vs.lb,
                             ((py - py0) << kTileLog) + (px - px0));
            }
        }
    }
    uint64_t big = __ballot(area > kSmallArea);
    const int lane = (int)(threadIdx.x & 63u);
    while (big) {
        const int src = __builtin_ctzll(big);
        big &= big - 1ull;
        const float vx = lane_f(vs.vx, src), vy = lane_f(vs.vy, src);
        const float vz = lane_f(vs.vz, src), half = lane_f(vs.half, src);
        const int bx0 = lane_i(x0, src), bx1 = lane_i(x1, src);
        const int by0 = lane_i(y0, src);
        const int a = lane_i(area, src);
        const uint32_t sid = (uint32_t)lane_i((int)id, src);
        const uint64_t lb = (uint64_t)(uint32_t)lane_i((int)(uint32_t)(vs.lb >> 32), src) << 32;
        // lane k takes pixels k, k + 64, ... of the clipped box, row by row
        // (w <= kTile, so 64 / w and the row of k come exactly from the
        // approximate reciprocal, as in raster_splat)
        const int w = bx1 - bx0 + 1;
        const float rw = __builtin_amdgcn_rcpf((float)w);
        const int dq = (int)(64.5f * rw), dr = 64 - dq * w;
        int row = (int)(((float)lane + 0.5f) * rw), col = lane - row * w;
        for (int k = lane; k < a; k += 64) {
            const int px = bx0 + col, py = by0 + row;
            col += dr;
            row += dq;
            if (col >= w) { col -= w; row += 1; }
            fragment_lds(lray, lkey, c.far_plane, vx, vy, vz, half, sid, lb,
                         ((py - py0) << kTileLog) + (px - px0));
        }
    }
}

// Raster items, strided over the grid: a tile's rays in LDS and its keys as
// the big list left them, its entries in kBlock-wide steps, then its keys out
// -- stored when the item is the tile's only one, else merged with a global
// atomicMin where the item lowered a key.
__global__ void __launch_bounds__(kBlock) k_tile_raster(const int16_t *splats, const uint8_t *lod,
                                                        uint32_t lod_log2, uint64_t n, SplatCam c,
                                                        const float4 *rays, uint64_t *frame,
                                                        const uint64_t *d_n, TileBufs tb)
{
    __shared__ float4 lray[kTilePx];
    __shared__ uint64_t lkey[kTilePx];
    if (!tb.tc[kTcOk]) return;
    const uint32_t nitems = tb.tc[kTcItems];
    if (d_n) n = min(*d_n, n);
    for (uint32_t it = blockIdx.x; it < nitems; it += gridDim.x) {
        const uint4 item = tb.items[it];
        const uint32_t t = item.x & ~kSingle;
        const int px0 = (int)(t % tb.tx) << kTileLog, py0 = (int)(t / tb.tx) << kTileLog;
        uint64_t start[kTilePx / kBlock];
#pragma unroll
        for (int k = 0; k < kTilePx / kBlock; k++) {
            const int q = (int)threadIdx.x + k * kBlock;
            const int px = px0 + (q & (kTile - 1)), py = py0 + (q >> kTileLog);
            start[k] = ~0ull;
            if (px < (int)c.W && py < (int)c.H) {
                lray[q] = rays[(size_t)py * c.W + px];
                start[k] = frame[(size_t)py * c.W + px];
            }
            lkey[q] = start[k];
        }
        __syncthreads();
        for (uint32_t j0 = item.y; j0 < item.z; j0 += blockDim.x) {
            const uint32_t j = j0 + threadIdx.x;
            const uint64_t i = j < item.z ? (uint64_t)tb.pairs[j] : n;
            tile_splat(splats, lod, lod_log2, n, i, c, px0, py0, lray, lkey);
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kTilePx / kBlock; k++) {
            const int q = (int)threadIdx.x + k * kBlock;
            const int px = px0 + (q & (kTile - 1)), py = py0 + (q >> kTileLog);
            if (px >= (int)c.W || py >= (int)c.H) continue;
            const uint64_t key = lkey[q];
            if (key >= start[k]) continue;
            uint64_t *f = frame + (size_t)py * c.W + px;
            if (item.x & kSingle)
                *f = key;
            else
                atomicMin(reinterpret_cast<unsigned long long *>(f), key);
        }
        __syncthreads();
    }
}

// The big list against the global frame, before the tiles.
__global__ void __launch_bounds__(kBlock) k_tile_big(const int16_t *splats, const uint8_t *lod,
                                                     uint32_t lod_log2, uint64_t n, SplatCam c,
                                                     const float4 *rays, uint64_t *frame,
                                                     const uint64_t *d_n, TileBufs tb)
{
    if (!tb.tc[kTcOk]) return;
    const uint32_t nbig = min(tb.tc[kTcBigCur], tb.big_cap);
    if (d_n) n = min(*d_n, n);
    for (uint32_t j0 = blockIdx.x * blockDim.x; j0 < nbig; j0 += gridDim.x * blockDim.x) {
        const uint32_t j = j0 + threadIdx.x;
        const uint64_t i = j < nbig ? (uint64_t)tb.big[j] : n;
        raster_list(splats, lod, lod_log2, n, i, c, rays, frame);
    }
}

__global__ void k_resolve(const int16_t *splats, const uint8_t *lod, uint32_t lod_log2,
                          uint64_t n, SplatCam c, const float *voxel_rgb, const uint64_t *frame,
                          const float4 *rays, float *depth, uint32_t *idbuf, float *rgb,
                          float *weight)
{
    const uint32_t px = blockIdx.x * blockDim.x + threadIdx.x, py = blockIdx.y;
    if (px >= c.W) return;
    const size_t p = (size_t)py * c.W + px;
    const uint64_t key = frame[p];
    if (key == ~0ull) {
        depth[p] = 1.0f;
        idbuf[p] = 0xFFFFFFFFu;
        if (rgb) { rgb[3 * p] = 0.5f; rgb[3 * p + 1] = 0.5f; rgb[3 * p + 2] = 0.7f; }
        if (weight) weight[p] = 0.0f;
        return;
    }
    const uint32_t i = (uint32_t)key;
    const float d = __uint_as_float((uint32_t)(key >> 32));
    depth[p] = d;
    idbuf[p] = i;
    if (!rgb && !weight) return;
    // shading, splat.vert.glsl:24-32 and splat.frag.glsl:93-154
    const float lodf = (float)(1u << (lod ? lod[i] : lod_log2));
    const float half = 0.5f * lodf;
    const int16_t *rec = splats + 4 * (size_t)i;
    const float a[4] = {(float)rec[0] + half, (float)rec[1] + half, (float)rec[2] + half, 1.0f};
    float v[4];
    mv4(c.T, a, v);
    float dir[3];
    pixel_dir(c, (int)px, (int)py, dir);
    const float4 inv = rays[p];
    float t0, t1;
    aabb(v[0] - half, v[0] + half, v[1] - half, v[1] + half, v[2] - half, v[2] + half, inv.x, inv.y,
         inv.z, t0, t1);
    float hit[3], ha[3];
    for (int k = 0; k < 3; k++) {
        hit[k] = v[k] - dir[k] * t0;
        ha[k] = fabsf(hit[k]);
    }
    const float md = gmax(gmax(ha[0], ha[1]), ha[2]);
    float nrm[3];
    for (int k = 0; k < 3; k++) nrm[k] = (ha[k] == md ? 1.0f : 0.0f) * gsign(hit[k]);
    const float lx = -0.70710677f, ly = 0.70710677f, lz = 0.0f;
    float nd = (-nrm[0]) * lx;
    nd = nd + (-nrm[1]) * ly;
    nd = nd + (-nrm[2]) * lz;
    const int attr = rec[3];
    const float sh = (float)((attr >> 6) & 1);
    const float s1 = gmax(0.7f, 1.0f - sh);
    const float s2 = gmax(gmax(0.7f, sh), gsign(nd));
    float base[3];
    if (voxel_rgb) {
        for (int k = 0; k < 3; k++) base[k] = voxel_rgb[3 * (size_t)i + k];
    } else {
        base[0] = (float)((attr >> 4) & 3) / 3.0f;
        base[1] = (float)((attr >> 2) & 3) / 3.0f;
        base[2] = (float)(attr & 3) / 3.0f;
    }
    const float fs = 256.0f / c.far_plane;
    const float fog = sqrtf(gmax(d - fs, 0.0001f));
    const float keep = 1.0f - fog;
    const float fogc[3] = {0.5f, 0.5f, 0.7f};
    if (rgb)
        for (int k = 0; k < 3; k++) {
            const float vcol = base[k] * s1;
            const float col = vcol * s2;
            rgb[3 * p + k] = col * keep + fogc[k] * fog;
        }
    if (weight) weight[p] = (s1 * s2) * keep;
}

// v of the lane d (1, 2 or 4) further in the row of 16, 0 past its end.
template <int D>
__device__ __forceinline__ uint32_t lane_up(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x100 + D, 0xF, 0xF, true);
}

// Gradient of the splat colours.  Neighbouring pixels of a row mostly show the
// same splat, so runs of one splat inside groups of 8 lanes are added up first
// (three DPP steps) and their first lane adds the sum: the kernel is bound by
// its atomics (a 512x512 frame: 29.9 -> 22.7 us).
__global__ void k_backward(uint64_t np, uint64_t n, const uint32_t *idbuf, const float *weight,
                           const float *dL, float *grad)
{
    const uint32_t lane = threadIdx.x & 63u;
    for (uint64_t p0 = blockIdx.x * (uint64_t)blockDim.x; p0 < np;
         p0 += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t p = p0 + threadIdx.x;
        uint32_t i = 0xFFFFFFFFu;
        float w = 0.0f, v[3] = {0.0f, 0.0f, 0.0f};
        if (p < np) {
            i = idbuf[p];
            if (i != 0xFFFFFFFFu && i < n) w = weight[p];
        }
        if (w != 0.0f)
            for (int k = 0; k < 3; k++) v[k] = w * dL[3 * p + k];
        else
            i = 0xFFFFFFFFu;
        // a run starts where the splat changes and at every 8th lane
        const uint32_t before = (uint32_t)__builtin_amdgcn_update_dpp((int)~i, (int)i, 0x111, 0xF, 0xF, false);
        const bool head = (lane & 7u) == 0u || before != i;
        const uint64_t heads = __ballot(head);
        const uint32_t run = __builtin_amdgcn_mbcnt_hi(
            (uint32_t)(heads >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)heads, 0u)) + (head ? 1u : 0u);
        auto step = [&](auto dc) {
            constexpr int D = decltype(dc)::value;
            const bool same = lane_up<D>(run) == run;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const float o = __uint_as_float(lane_up<D>(__float_as_uint(v[k])));
                v[k] += same ? o : 0.0f;
            }
        };
        step(std::integral_constant<int, 1>{});
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 4>{});
        if (head && i != 0xFFFFFFFFu)
            for (int k = 0; k < 3; k++) atomicAdd(grad + 3 * (size_t)i + k, v[k]);
    }
}

static SplatCam to_cam(const vp_camera *cam)
{
    SplatCam c;
    for (int i = 0; i < 16; i++) {
        c.T[i] = cam->view_translation[i];
        c.PR[i] = cam->proj_view_rot[i];
        c.IPR[i] = cam->inv_proj_view_rot[i];
    }
    c.W = cam->width;
    c.H = cam->height;
    c.far_plane = cam->far_plane;
    int e = 0;
    const float f = cam->far_plane;
    c.inv_far = f > 1e-30f && f < 1e30f && frexpf(f, &e) == 0.5f ? 1.0f / f : 0.0f;
    return c;
}

}  // namespace vp

using namespace vp;

static CullPlanes cull_planes(const vp_camera *cam)
{
    // M = proj_view_rot * view_translation (column-major), in double: clip = M (c, 1)
    double M[4][4];
    for (int r = 0; r < 4; r++)
        for (int k = 0; k < 4; k++) {
            double acc = 0.0;
            for (int j = 0; j < 4; j++)
                acc += (double)cam->proj_view_rot[j * 4 + r] * (double)cam->view_translation[k * 4 + j];
            M[r][k] = acc;
        }
    CullPlanes cp;
    // -w <= x, x <= w, -w <= y, y <= w, -w <= z, z <= w
    for (int a = 0; a < 3; a++)
        for (int sgn = 0; sgn < 2; sgn++)
            for (int k = 0; k < 4; k++)
                cp.p[2 * a + sgn][k] = (float)(M[3][k] + (sgn ? -M[a][k] : M[a][k]));
    for (int a = 0; a < 3; a++) cp.eye[a] = -cam->view_translation[12 + a];
    cp.far_plane = cam->far_plane;
    return cp;
}

// Whether the tile bounds' approximate arithmetic (splat_open, block_box) stays
// within its margins for this camera.  It does for a view translation followed
// by a perspective projection of a rotated view, the camera vp_camera names:
//  * a translation gives the view position one rounding, fl(a + t), however it
//    is summed, so both sides start from the same position v; any other matrix
//    rounds at the size of the world's coordinates, not of v, and splats near
//    the eye would be judged by an error of their own size;
//  * clip coordinates are sums of four products, at most 8 half-ulps apart on
//    the two sides: g = 8 2^-24 times a row's absolute sum, times |v|.  A splat
//    in the volume has |clip x|, |clip y| <= w, so |v| <= L w (+ a constant),
//    L from the inverse of the rows x, y and w;
//  * the third row follows the fourth, so clip z, which sizes the sprites, is
//    no smaller than half of w beside its own constant.
// 2 g L must stay below splat_open's 1e-4 of w, and its share of a pixel, g L
// times the wider side, below 0.2 of its margin of 0.25.
static bool bounds_hold(const vp_camera *cam)
{
    const float *T = cam->view_translation, *P = cam->proj_view_rot;
    for (int k = 0; k < 3; k++)
        for (int r = 0; r < 4; r++)
            if (T[4 * k + r] != (r == k ? 1.0f : 0.0f)) return false;
    if (T[15] != 1.0f || !(cam->far_plane > 1e-30f && cam->far_plane < 1e30f)) return false;
    const double ulps = 8.0 / 16777216.0;
    double sum = 0.0, con = 0.0, A[3][3];          // A: rows x, y, w
    for (int r = 0; r < 4; r++) {
        double s = 0.0;
        for (int k = 0; k < 3; k++) s += fabs((double)P[4 * k + r]);
        sum = fmax(sum, s);
        con = fmax(con, fabs((double)P[12 + r]));
        for (int k = 0; k < 3 && r != 2; k++) A[r == 3 ? 2 : r][k] = P[4 * k + r];
    }
    auto cof = [&](int r, int k) {
        const int r1 = (r + 1) % 3, r2 = (r + 2) % 3, k1 = (k + 1) % 3, k2 = (k + 2) % 3;
        return A[r1][k1] * A[r2][k2] - A[r1][k2] * A[r2][k1];
    };
    const double det = A[0][0] * cof(0, 0) + A[0][1] * cof(0, 1) + A[0][2] * cof(0, 2);
    double L = 0.0, zz = 0.0, zw = 0.0;
    for (int k = 0; k < 3; k++) {
        double s = 0.0;
        for (int r = 0; r < 3; r++) s += fabs(cof(r, k));
        L = fmax(L, s / fabs(det));
        zw += (double)P[4 * k + 2] * A[2][k];
        zz += A[2][k] * A[2][k];
    }
    const double scale = zw / zz;                  // the third row in the fourth's
    for (int k = 0; k < 3; k++)
        if (!(fabs(P[4 * k + 2] - scale * A[2][k]) <= 1e-5 * sqrt(zz))) return false;
    // |v| <= L (w + |constant|): the constants of x, y and w count as w's
    for (int r = 0; r < 4; r++)
        if (r != 2 && !(fabs(P[12 + r]) <= 1.0f)) return false;
    const double e = ulps * sum * L, e0 = e + ulps * con, side = fmax(cam->width, cam->height);
    return scale >= 0.5 && con <= 100.0 && 2.0 * e <= 1e-4 && 2.0 * e0 <= 1e-3 &&
           (e + 0.5 * e0) * side <= 0.2 && sum < 1e6;
}

// The splat frame.  d_n (nullable): the list length in device memory, n its
// bound; with d_n the block bounds are computed into d_bounds here first (the
// list is assembled on the device each frame).
static int splat_frame(vp_ctx *ctx, const int16_t *d_splats, const uint8_t *d_lod,
                       uint32_t lod_log2, uint64_t n, const float *d_bounds,
                       const vp_camera *cam, const float *d_voxel_rgb, const vp_frame *out,
                       void *stream, const uint64_t *d_n = nullptr)
{
    if (!ctx || !cam || !out || !out->d_depth || !out->d_id) return VP_ERR_ARG;
    if (n && !d_splats) return VP_ERR_ARG;
    if (cam->width == 0 || cam->height == 0 || cam->width > 16384 || cam->height > 16384)
        return VP_ERR_ARG;
    if (lod_log2 > 8) return VP_ERR_ARG;
    if (n > 0xFFFFFFFFull) return VP_ERR_UNSUPPORTED;   // ids are 32-bit
    const uint64_t np = (uint64_t)cam->width * cam->height;
    const uint64_t nb = (n + kBlock - 1) / kBlock;
    hipStream_t st = as_stream(stream);
    uint64_t *frame;
    float4 *rays;
    uint32_t *blk = nullptr, *hiz;
    int ncu;
    // screen tiles (block-culled frames of at most kMaxTiles tiles)
    TileBufs tb = {};
    tb.tx = (cam->width + kTile - 1) / kTile;
    tb.ty = (cam->height + kTile - 1) / kTile;
    tb.nt = tb.tx * tb.ty;
    uint32_t tgrid = 0;
    bool tiles = false;
    {
        std::lock_guard<std::mutex> g(ctx->mu);
        tiles = ctx->splat_tiles && d_bounds && nb && tb.nt <= kMaxTiles;
        int rc = ensure_frame(ctx, np);
        if (rc) return rc;
        if (d_bounds && nb) {
            rc = ensure_blocks(ctx, nb);
            if (rc) return rc;
            blk = ctx->d_blk;
        }
        frame = ctx->d_frame;
        hiz = reinterpret_cast<uint32_t *>(frame + ctx->frame_cap);
        rays = ctx->d_rays;
        ncu = ctx->num_cus;
        if (tiles) {
            // entries: at most four per splat; beyond 2^26 in one frame the
            // global path draws it
            tgrid = (uint32_t)ncu * 4u;
            const uint64_t lim = ctx->splat_tile_entries ? ctx->splat_tile_entries : (1ull << 26);
            tb.pair_cap = (uint32_t)(4 * n < lim ? 4 * n : lim);
            tb.big_cap = (uint32_t)(n < (1ull << 22) ? n : (1ull << 22));
            tb.item_cap = tb.nt + tb.pair_cap / kItem + 1;
            const uint64_t words = (uint64_t)tgrid * tb.nt + 2ull * tb.nt + kTcWords +
                                   4ull * tb.item_cap + tb.pair_cap + tb.big_cap;
            rc = ensure_tiles(ctx, words);
            if (rc) return rc;
            uint32_t *w = ctx->d_tiles;
            tb.items = reinterpret_cast<uint4 *>(w);            // 16-byte aligned
            w += 4ull * tb.item_cap;
            tb.hist = w;
            w += (uint64_t)tgrid * tb.nt;
            tb.cnt = w;
            w += tb.nt;
            tb.cur = w;
            w += tb.nt;
            tb.tc = w;
            w += kTcWords;
            tb.pairs = w;
            w += tb.pair_cap;
            tb.big = w;
        }
    }
    const SplatCam c = to_cam(cam);
    const dim3 pg((cam->width + 255) / 256, cam->height);
    // blk: [screen box per block | bin per block | order | counters]
    uint4 *box = reinterpret_cast<uint4 *>(blk);
    uint32_t *bin = blk + 4 * nb, *order = bin + nb, *cnt = order + nb;
    hipLaunchKernelGGL(k_frame_start, pg, dim3(256), 0, st, c, rays, frame, hiz,
                       hz_tiles(c.W) * hz_tiles(c.H), cnt, n && blk ? (uint32_t)kCounters : 0u);
    if (n && blk && d_n) {
        const uint64_t wgs = (nb + 3) / 4, cap = (uint64_t)ncu * 32u;
        hipLaunchKernelGGL(k_bounds, dim3((uint32_t)(wgs < cap ? wgs : cap)), dim3(256), 0, st,
                           d_splats, d_lod, lod_log2, n, nb, const_cast<float *>(d_bounds), d_n);
    }
    if (n && blk) {
        // the distance at which a splat is kNearPixels wide, as block_bin's bin
        const float reach = (float)c.H * 1.1f * (float)(1u << lod_log2) / kNearPixels;
        const uint32_t near_bin =
            (uint32_t)fminf(fmaxf(sqrtf(reach / c.far_plane) * (float)kBins, 0.0f), (float)kBins);
        const bool few = np <= kFewPixels || !bounds_hold(cam);
        const uint32_t g = (uint32_t)((nb + 255) / 256 < 4096 ? (nb + 255) / 256 : 4096);
        hipLaunchKernelGGL(k_blk_cull, dim3(g), dim3(256), 0, st, d_bounds, nb, cull_planes(cam),
                           c, bin, few ? nullptr : box, cnt, d_n);
        hipLaunchKernelGGL(k_blk_scatter, dim3(g), dim3(kBins), 0, st, bin, nb, cnt, order, d_n,
                           near_bin);
        if (tiles) {
            const size_t lds = (size_t)tb.nt * sizeof(uint32_t);
            hipLaunchKernelGGL(k_tile_reset, dim3((tb.nt + 255) / 256), dim3(256), 0, st, tb.cnt,
                               tb.nt, tb.tc);
            hipLaunchKernelGGL(k_tile_count, dim3(tgrid), dim3(kBlock), lds, st, d_splats, d_lod,
                               lod_log2, n, c, order, cnt, d_n, tb);
            hipLaunchKernelGGL(k_tile_scan, dim3(1), dim3(kScanThreads), 0, st, tb);
            hipLaunchKernelGGL(k_tile_scatter, dim3(tgrid), dim3(kBlock), lds, st, d_splats, d_lod,
                               lod_log2, n, c, order, cnt, d_n, tb);
            hipLaunchKernelGGL(k_tile_big, dim3((uint32_t)ncu * 4u), dim3(kBlock), 0, st, d_splats,
                               d_lod, lod_log2, n, c, rays, frame, d_n, tb);
            hipLaunchKernelGGL(k_tile_raster, dim3((uint32_t)ncu * 6u), dim3(kBlock), 0, st,
                               d_splats, d_lod, lod_log2, n, c, rays, frame, d_n, tb);
        }
        // 4 workgroups per CU: fewer hide less latency (3: 1248 us against
        // 1090 for the 1080p frame), more start further from the near end
        // before anything is hidden (6 resident: 911 against 879 us)
        const dim3 grid((uint32_t)ncu * 4u);
        const uint32_t *ok = tiles ? tb.tc + kTcOk : nullptr;
        if (few) {
            hipLaunchKernelGGL(k_raster_few, grid, dim3(kBlock), 0, st, d_splats, d_lod, lod_log2,
                               n, c, rays, frame, order, cnt, d_n, ok);
        } else {
            hipLaunchKernelGGL(k_raster_blocks, grid, dim3(kBlock), 0, st, d_splats, d_lod,
                               lod_log2, n, c, rays, frame, order, box, hiz, cnt, d_n, ok);
        }
    } else if (n) {
        hipLaunchKernelGGL(k_raster, dim3((uint32_t)nb), dim3(256), 0, st, d_splats, d_lod,
                           lod_log2, n, c, rays, frame);
    }
    hipLaunchKernelGGL(k_resolve, pg, dim3(256), 0, st, d_splats, d_lod, lod_log2, n, c,
                       d_voxel_rgb, frame, rays, out->d_depth, out->d_id, out->d_rgb,
                       out->d_weight);
    VP_HIP_TRY(hipGetLastError());
    return VP_OK;
}

extern "C" int vp_gpu_splat(vp_ctx *ctx, const int16_t *d_splats, const uint8_t *d_lod,
                            uint32_t lod_log2, uint64_t n, const vp_camera *cam,
                            const float *d_voxel_rgb, const vp_frame *out, void *stream)
{
    return splat_frame(ctx, d_splats, d_lod, lod_log2, n, nullptr, cam, d_voxel_rgb, out, stream);
}

extern "C" int vp_gpu_splat_bounds(vp_ctx *ctx, const int16_t *d_splats, const uint8_t *d_lod,
                                   uint32_t lod_log2, uint64_t n, float *d_bounds, void *stream)
{
    if (!ctx || (n && (!d_splats || !d_bounds))) return VP_ERR_ARG;
    if (lod_log2 > 8) return VP_ERR_ARG;
    if (n > 0xFFFFFFFFull) return VP_ERR_UNSUPPORTED;
    if (n == 0) return VP_OK;
    const uint64_t nb = (n + kBlock - 1) / kBlock;
    // four blocks per workgroup (a wave each), at most 32 workgroups per CU
    const uint64_t wgs = (nb + 3) / 4, cap = (uint64_t)ctx->num_cus * 32u;
    hipLaunchKernelGGL(k_bounds, dim3((uint32_t)(wgs < cap ? wgs : cap)), dim3(256), 0,
                       as_stream(stream), d_splats, d_lod, lod_log2, n, nb, d_bounds, nullptr);
    VP_HIP_TRY(hipGetLastError());
    return VP_OK;
}

extern "C" int vp_gpu_splat_blocks(vp_ctx *ctx, const int16_t *d_splats, const uint8_t *d_lod,
                                   uint32_t lod_log2, uint64_t n, const float *d_bounds,
                                   const vp_camera *cam, const float *d_voxel_rgb,
                                   const vp_frame *out, void *stream)
{
    return splat_frame(ctx, d_splats, d_lod, lod_log2, n, d_bounds, cam, d_voxel_rgb, out, stream);
}

extern "C" int vp_ctx_set_splat_tiles(vp_ctx *ctx, int enable, uint64_t max_entries)
{
    if (!ctx || max_entries > 0xFFFFFFFFull) return VP_ERR_ARG;
    std::lock_guard<std::mutex> g(ctx->mu);
    ctx->splat_tiles = enable ? 1 : 0;
    ctx->splat_tile_entries = max_entries;
    return VP_OK;
}

extern "C" int vp_gpu_splat_backward(vp_ctx *ctx, uint64_t n, const vp_camera *cam,
                                     const uint32_t *d_id, const float *d_weight,
                                     const float *d_dL_drgb, float *d_grad, void *stream)
{
    if (!ctx || !cam || !d_id || !d_weight || !d_dL_drgb || !d_grad) return VP_ERR_ARG;
    const uint64_t np = (uint64_t)cam->width * cam->height;
    if (np == 0) return VP_OK;
    uint64_t blocks = (np + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_backward, dim3((uint32_t)blocks), dim3(256), 0, as_stream(stream), np, n,
                       d_id, d_weight, d_dL_drgb, d_grad);
    VP_HIP_TRY(hipGetLastError());
    return VP_OK;
}

extern "C" int vp_gpu_splat_counted(vp_ctx *ctx, const int16_t *d_splats, const uint8_t *d_lod,
                                    uint32_t lod_log2, uint64_t capacity, const uint64_t *d_count,
                                    float *d_bounds, const vp_camera *cam,
                                    const float *d_voxel_rgb, const vp_frame *out, void *stream)
{
    if (!d_count || (capacity && !d_bounds)) return VP_ERR_ARG;
    return splat_frame(ctx, d_splats, d_lod, lod_log2, capacity, d_bounds, cam, d_voxel_rgb, out,
                       stream, d_count);
}
