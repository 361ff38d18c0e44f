// mesh.hip -- near-field quad mesh with ambient occlusion for gfx950.
//
// Replaces chunk_make_mesh (src/chunkset/mesher.c:184-357) with its ambient
// samples (sample_ao / sample_ao_border, mesher.c:72-171) and the shadow
// samples it takes (shadow_sample / shadow_sample_normal,
// src/chunkset/shadow.h:52-75), batched over a chunk list.
//
// One workgroup per chunk (persistent, ticket order = list order):
//  1. the chunk's occupancy and a one-voxel shell around it, (R+2)^3 bits,
//     go to LDS as one row of R+2 bits per (z, y) in [-1, R]^2, in 32-bit
//     words (three at R = 64).  Rows of uniform chunks (and of chunks beyond
//     the world: air) are synthesised without a read.
//  2. face bits of a row are XORs of rows: +x = row ^ row >> 1, +y / +z =
//     row ^ the next row.  Their popcounts give per-row counts,
//     per-group (8 rows at R = 64) offsets by a workgroup scan, and the
//     chunk's face count, which is published and turned into an output
//     offset by a decoupled look-back before any face is written.
//  3. faces are written in passes of whole row groups that fit an LDS list
//     of (row, x, axis) entries, in (z, y, x, axis) order -- the reference's
//     emission order.  Each (row, 8-voxel segment) item finds its slots from
//     its row's offset and the popcounts of the row's earlier bits.
//  4. per pass, each thread first does everything but the stores for its
//     faces (ambient terms from the LDS bits, the solid voxel's colour and
//     the shadow-map entries from memory), packed into one word per face,
//     and then only the stores, shared out by address: half a vertex quad
//     (16 of 32 B) or a third of an index row (8 of 24 B) per lane, whole
//     lines per instruction.  A load issued after a store completes after it
//     (the vector memory counter retires in order), so keeping the loads
//     ahead of the stores keeps the stores from stalling the next face's
//     loads.
// 2048x256x2048 world, 150.3 M faces: 2985 -> 2645 us, 3.7 TB/s (the kernel).
#include "vp_internal.h"

#include <algorithm>
#include <type_traits>

namespace vp {

constexpr uint64_t kMFlagAgg = 1ull << 62;
constexpr uint64_t kMFlagPre = 2ull << 62;
constexpr uint64_t kMValMask = (1ull << 62) - 1;
constexpr int kMeshBS = 512;

struct MeshArgs {
    const uint8_t  *voxels;
    const int16_t  *uniform;
    const uint16_t *map;
    uint32_t        map_sx;
    const uint32_t *ids;
    uint32_t        n;
    uint32_t        nchunks;
    uint32_t        mb0, mb1, mb2;
    uint32_t        single;
    uint32_t        parts;         // workgroups that share a chunk's faces
    int16_t        *geom;
    uint32_t       *index;
    uint64_t        cap;
    uint64_t       *offsets;
    uint32_t       *ticket;
    uint64_t       *state;
    uint32_t       *status;
};

// corners of the unit cube's +x, +y, +z faces in vertex order, packed as
// 3 bits (x | y << 1 | z << 2) per vertex (mesher.c:19-31)
__device__ __forceinline__ uint32_t m_corner(uint32_t axis, uint32_t v)
{
    // axis 0: (1,0,0) (1,0,1) (1,1,1) (1,1,0) -> 1 5 7 3
    // axis 1: (0,1,0) (1,1,0) (1,1,1) (0,1,1) -> 2 3 7 6
    // axis 2: (1,0,1) (0,0,1) (0,1,1) (1,1,1) -> 5 4 6 7
    constexpr uint32_t lut = (1u | 5u << 3 | 7u << 6 | 3u << 9) |
                             (2u | 3u << 3 | 7u << 6 | 6u << 9) << 12;
    constexpr uint32_t lut2 = 5u | 4u << 3 | 6u << 6 | 7u << 9;
    const uint32_t w = axis == 2 ? lut2 : (lut >> (12 * axis));
    return (w >> (3 * v)) & 7u;
}

// triangle index rows by normal | rotated << 1 (mesher.c:54-66), 2 bits each
__device__ __forceinline__ uint32_t m_tri_row(uint32_t normal, uint32_t rot)
{
    constexpr uint32_t r00 = 0u | 3u << 2 | 1u << 4 | 2u << 6 | 1u << 8 | 3u << 10;
    constexpr uint32_t r01 = 3u | 2u << 2 | 0u << 4 | 1u << 6 | 0u << 8 | 2u << 10;
    constexpr uint32_t r10 = 1u | 3u << 2 | 0u << 4 | 3u << 6 | 1u << 8 | 2u << 10;
    constexpr uint32_t r11 = 0u | 2u << 2 | 3u << 4 | 2u << 6 | 0u << 8 | 1u << 10;
    return normal ? (rot ? r11 : r10) : (rot ? r01 : r00);
}

// Vertex ambient terms, 2 bits each in vertex order, and the rotated flag at
// bit 8, of a face whose air cell has the in-plane neighbours nb: bit
// 3 (1 + d1) + 1 + d0 for the step d0 along the lower and d1 along the higher
// of the face's two axes (sample_ao, mesher.c:72-171, vertex order of
// mesher.c:254-272).
constexpr uint32_t m_ambient(uint32_t axis, uint32_t nb)
{
    auto at = [&](int d0, int d1) -> uint32_t { return (nb >> (3 * (1 + d1) + 1 + d0)) & 1u; };
    const uint32_t n0 = at(-1, 0), n1 = at(0, -1), n2 = at(1, 0), n3 = at(0, 1);
    const uint32_t c0 = (n0 + n1) | at(-1, -1), c1 = (n1 + n2) | at(1, -1);
    const uint32_t c2 = (n2 + n3) | at(1, 1), c3 = (n3 + n0) | at(-1, 1);
    const uint32_t v0 = axis == 2 ? c1 : c0, v2 = axis == 2 ? c3 : c2;
    const uint32_t v1 = axis == 0 ? c3 : (axis == 1 ? c1 : c0);
    const uint32_t v3 = axis == 0 ? c1 : (axis == 1 ? c3 : c2);
    return v0 | v1 << 2 | v2 << 4 | v3 << 6 | (v0 + v2 < v1 + v3 ? 1u : 0u) << 8;
}

// m_ambient of all axes and neighbours, two 16-bit entries to a word
struct AmbientTable {
    uint32_t w[3 * 256];
};
constexpr AmbientTable ambient_table()
{
    AmbientTable t = {};
    for (uint32_t i = 0; i < 3 * 256; i++)
        t.w[i] = m_ambient(i >> 8, 2 * i & 511u) | m_ambient(i >> 8, (2 * i + 1) & 511u) << 16;
    return t;
}
__constant__ const AmbientTable kAmbient = ambient_table();

// 16 bytes -> 16 occupancy bits
__device__ __forceinline__ uint32_t nz4(uint32_t w)
{
    const uint32_t m = (((w & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | w) & 0x80808080u;
    return (((m >> 7) * 0x00204081u) >> 21) & 0xFu;
}

// sums of the two 16-bit halves
__device__ __forceinline__ uint32_t add_u16x2(uint32_t a, uint32_t b)
{
    typedef unsigned short v2 __attribute__((ext_vector_type(2)));
    const v2 s = __builtin_bit_cast(v2, a) + __builtin_bit_cast(v2, b);
    return __builtin_bit_cast(uint32_t, s);
}

template <int B>
struct MeshShape {
    static constexpr int R = 1 << B;
    static constexpr int P = R + 2;                        // rows per axis with the shell
    static constexpr int ROWS = R * R;                     // (z, y) rows of the chunk
    static constexpr int GR = ROWS >= kMeshBS ? ROWS / kMeshBS : 1;   // rows per group
    static constexpr int NG = ROWS / GR;                   // groups (one per thread)
    static constexpr int LIST = 3 * R * R * R < 2048 ? 3 * R * R * R : 2048;   // faces per pass
    static constexpr int W = (R + 2 + 31) / 32;            // words of a row with its shell
    static constexpr int QW = R >= 16 ? 16 : R;            // bytes per row load
    static constexpr int Q = R / QW;                       // loads per row
    static constexpr uint64_t FULL = R == 64 ? ~0ull : ((1ull << R) - 1ull);
    static_assert(GR * 3 * R <= LIST, "a group's faces must fit one pass");
};

template <int QW> struct RowLoad;
template <> struct RowLoad<16> {
    using T = uint4;
    static __device__ __forceinline__ uint32_t bits(T v)
    {
        return nz4(v.x) | nz4(v.y) << 4 | nz4(v.z) << 8 | nz4(v.w) << 12;
    }
};
template <> struct RowLoad<8> {
    using T = uint2;
    static __device__ __forceinline__ uint32_t bits(T v) { return nz4(v.x) | nz4(v.y) << 4; }
};
template <> struct RowLoad<4> {
    using T = uint32_t;
    static __device__ __forceinline__ uint32_t bits(T v) { return nz4(v); }
};

template <int BS>
__device__ __forceinline__ uint32_t m_scan_excl(uint32_t v, uint32_t *wsum, uint32_t &total)
{
    constexpr int NW = BS / 64;
    const uint32_t w = threadIdx.x >> 6;
    uint32_t wt, before = 0;
    const uint32_t ex = wave_excl_scan(v, wt);
    if ((threadIdx.x & 63u) == 0) wsum[w] = wt;
    __syncthreads();
    total = 0;
#pragma unroll
    for (uint32_t i = 0; i < NW; i++) {
        before += i < w ? wsum[i] : 0u;
        total += wsum[i];
    }
    return before + ex;
}

// An occupancy row: bit x + 1 is voxel x, bits 0 and R + 1 the shell.
template <int B>
__device__ __forceinline__ uint64_t row_from(const uint32_t *w, int sh)
{
    using S = MeshShape<B>;
    if constexpr (S::W == 3)
        return (uint64_t)__builtin_amdgcn_alignbit(w[2], w[1], sh) << 32 |
               __builtin_amdgcn_alignbit(w[1], w[0], sh);
    else if constexpr (S::W == 2)
        return __builtin_amdgcn_alignbit(w[1], w[0], sh);
    else
        return (w[0] >> sh) & (uint32_t)S::FULL;
}
// voxels x = 0..R-1 as bits, and the same of their +x neighbours
template <int B>
__device__ __forceinline__ uint64_t row_own(const uint32_t *w) { return row_from<B>(w, 1); }
template <int B>
__device__ __forceinline__ uint64_t row_next(const uint32_t *w) { return row_from<B>(w, 2); }

// The nine occupancy bits around the air cell (px, py, pz) in the face's plane,
// as m_ambient takes them: three bits of three rows for y and z faces, one bit
// of nine rows for x faces.
template <int B>
__device__ __forceinline__ uint32_t plane_bits(const uint32_t *occ, uint32_t axis, int px, int py, int pz)
{
    constexpr int P = MeshShape<B>::P, W = MeshShape<B>::W;
    const int row = (pz + 1) * P + (py + 1);
    uint32_t nb = 0;
    if (axis == 0) {
        const uint32_t ix = (uint32_t)px + 1u;
        const uint32_t *w = occ + (row - P - 1) * W + (ix >> 5);
#pragma unroll
        for (int d1 = 0; d1 < 3; d1++)
#pragma unroll
            for (int d0 = 0; d0 < 3; d0++)
                nb |= ((w[(d1 * P + d0) * W] >> (ix & 31u)) & 1u) << (3 * d1 + d0);
    } else {
        const uint32_t ix = (uint32_t)px;              // bits px - 1 .. px + 1
        const int step = (axis == 1 ? P : 1) * W;
        const uint32_t *w = occ + row * W - step + (ix >> 5);
#pragma unroll
        for (int d1 = 0; d1 < 3; d1++)
            nb |= (__builtin_amdgcn_alignbit(w[d1 * step + 1], w[d1 * step], ix & 31u) & 7u) << (3 * d1);
    }
    return nb;
}

template <int B>
__global__ void __launch_bounds__(kMeshBS, 4) k_mesh(MeshArgs a)
{
    using S = MeshShape<B>;
    constexpr int R = S::R, P = S::P, W = S::W, BS = kMeshBS;
    using RL = RowLoad<S::QW>;
    __shared__ uint32_t occ[P * P * W + 2];  // row (z, y) in shell coordinates + 1, bits as row_own
    __shared__ uint8_t  rowcnt[S::ROWS];     // faces of each chunk row
    __shared__ uint32_t goff[S::NG + 1];     // face offset of each row group
    __shared__ uint32_t list[S::LIST];       // solid << 20 | row << 8 | x << 2 | axis of a pass's faces
    __shared__ uint32_t packed[S::LIST];     // and all else their vertices and indices take
    __shared__ uint32_t wsum[BS / 64];
    __shared__ AmbientTable s_amb;           // u16 by axis << 9 | plane bits
    __shared__ uint4    s_corner[6];         // per axis and half: two vertices' (xy, z | number << 27)
    __shared__ int16_t  s_uni[27];           // 3x3x3 neighbourhood: value if uniform (0 = air/outside), -1 mixed
    __shared__ uint32_t s_nid[27];
    __shared__ uint32_t s_ticket;
    __shared__ uint64_t s_base;

    const uint32_t mx = 1u << a.mb0, my = 1u << a.mb1, mz = 1u << a.mb2;
    // the ambient table on its way to LDS, stored there by the first visit
    constexpr int TW = (3 * 256 + BS - 1) / BS;
    uint32_t tab[TW] = {};
    if (a.geom) {
        for (int i = 0; i < TW; i++)
            if (i * BS + threadIdx.x < 3u * 256u) tab[i] = kAmbient.w[i * BS + threadIdx.x];
        if (threadIdx.x < 6) {
            uint32_t w[4];
            for (uint32_t h = 0; h < 2; h++) {
                const uint32_t v = 2u * (threadIdx.x & 1u) + h, c = m_corner(threadIdx.x >> 1, v);
                w[2 * h] = (c & 1u) | ((c >> 1) & 1u) << 16;
                w[2 * h + 1] = (c >> 2) | v << 27;
            }
            s_corner[threadIdx.x] = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
    for (uint32_t visit = 0;; visit++) {
        // a single chunk takes no ticket: workgroup p does part p of list entry 0
        if (threadIdx.x == 0)
            s_ticket = a.single ? (visit == 0 ? blockIdx.x : a.parts) : atomicAdd(a.ticket, 1u);
        __syncthreads();
        const uint32_t tk = s_ticket;
        const uint32_t k = a.parts > 1u ? tk / a.parts : tk, part = tk - k * a.parts;
        if (k >= a.n) return;
        const uint32_t id = a.ids[k];
        const bool bad = id >= a.nchunks;
        const uint32_t cx = id & (mx - 1u), cy = (id >> a.mb0) & (my - 1u), cz = id >> (a.mb0 + a.mb1);
        if (threadIdx.x < 27 && !bad) {
            const int dx = (int)(threadIdx.x % 3) - 1, dy = (int)(threadIdx.x / 3 % 3) - 1,
                      dz = (int)(threadIdx.x / 9) - 1;
            const int64_t nx = (int64_t)cx + dx, ny = (int64_t)cy + dy, nz = (int64_t)cz + dz;
            int16_t u = 0;
            uint32_t nid = 0;
            if (nx >= 0 && nx < mx && ny >= 0 && ny < my && nz >= 0 && nz < mz) {
                nid = (((uint32_t)nz << a.mb1 | (uint32_t)ny) << a.mb0) | (uint32_t)nx;
                u = a.uniform ? a.uniform[nid] : (int16_t)-1;
            }
            s_uni[threadIdx.x] = u;
            s_nid[threadIdx.x] = nid;
        }
        __syncthreads();

        // ---- 1. occupancy with the one-voxel shell, 4 loads in flight ----
        if (!bad) {
            constexpr int NI = P * P * S::Q, U = 4;
            for (int t0 = threadIdx.x; t0 < NI; t0 += U * BS) {
                typename RL::T v[U];
                int mode[U];                     // 0 air, 1 solid, 2 loaded
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int t = t0 + u * BS;
                    mode[u] = 0;
                    v[u] = typename RL::T{};
                    if (t < NI) {
                        const int row = t / S::Q, q = t % S::Q;
                        const int yy = row % P, zz = row / P;
                        const int nb = 13 + 3 * (yy == 0 ? -1 : (yy == P - 1 ? 1 : 0)) +
                                       9 * (zz == 0 ? -1 : (zz == P - 1 ? 1 : 0));
                        const int16_t un = s_uni[nb];
                        if (un >= 0) {
                            mode[u] = un ? 1 : 0;
                        } else {
                            const uint32_t ly = (uint32_t)(yy - 1) & (R - 1), lz = (uint32_t)(zz - 1) & (R - 1);
                            const uint8_t *p = a.voxels + ((uint64_t)s_nid[nb] << (3 * B)) +
                                               ((((uint64_t)lz << B) | ly) << B) + q * S::QW;
                            v[u] = *reinterpret_cast<const typename RL::T *>(p);
                            mode[u] = 2;
                        }
                    }
                }
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int t = t0 + u * BS;
                    const uint32_t bits = mode[u] == 2 ? RL::bits(v[u])
                                                       : (mode[u] == 1 ? (1u << S::QW) - 1u : 0u);
                    uint64_t r = (uint64_t)bits << ((t % S::Q) * S::QW);
                    if constexpr (S::Q > 1) {
#pragma unroll
                        for (int d = 1; d < S::Q; d <<= 1) r |= __shfl_xor(r, d, 64);
                    }
                    if (t < NI && t % S::Q == 0) {
                        uint32_t *w = occ + t / S::Q * W;
                        w[0] = (uint32_t)r << 1;
                        if constexpr (W > 1) w[1] = (uint32_t)(r >> 31);
                        if constexpr (W > 2) w[2] = (uint32_t)(r >> 63);
                    }
                }
            }
            __syncthreads();
            // the shell's x = -1 and x = R
            constexpr int NE = P * P, UE = 3;
            for (int t0 = threadIdx.x; t0 < NE; t0 += UE * BS) {
                uint8_t lo[UE], hi[UE];
#pragma unroll
                for (int u = 0; u < UE; u++) {
                    const int row = t0 + u * BS;
                    lo[u] = hi[u] = 0;
                    if (row < NE) {
                        const int yy = row % P, zz = row / P;
                        const int nb = 13 + 3 * (yy == 0 ? -1 : (yy == P - 1 ? 1 : 0)) +
                                       9 * (zz == 0 ? -1 : (zz == P - 1 ? 1 : 0));
                        const uint64_t ro = ((((uint64_t)((uint32_t)(zz - 1) & (R - 1))) << B) |
                                             ((uint32_t)(yy - 1) & (R - 1))) << B;
                        const int16_t ul = s_uni[nb - 1], uh = s_uni[nb + 1];
                        lo[u] = ul >= 0 ? (uint8_t)(ul != 0)
                                        : a.voxels[((uint64_t)s_nid[nb - 1] << (3 * B)) + ro + (R - 1)];
                        hi[u] = uh >= 0 ? (uint8_t)(uh != 0)
                                        : a.voxels[((uint64_t)s_nid[nb + 1] << (3 * B)) + ro];
                    }
                }
#pragma unroll
                for (int u = 0; u < UE; u++) {
                    const int row = t0 + u * BS;
                    if (row < NE) {
                        if (lo[u]) occ[row * W] |= 1u;
                        if (hi[u]) occ[row * W + (R + 1) / 32] |= 1u << ((R + 1) % 32);
                    }
                }
            }
        }
        __syncthreads();

        // ---- 2. per-row face counts, group offsets, output offset ----
        uint32_t gcnt = 0;
        if (!bad && threadIdx.x < S::NG) {
#pragma unroll
            for (int i = 0; i < S::GR; i++) {
                const int r = threadIdx.x * S::GR + i;
                const int z = r / R, y = r % R;
                const uint32_t *w = occ + ((z + 1) * P + (y + 1)) * W;
                const uint64_t o = row_own<B>(w);
                const uint32_t c = __popcll(o ^ row_next<B>(w)) + __popcll(o ^ row_own<B>(w + W)) +
                                   __popcll(o ^ row_own<B>(w + P * W));
                rowcnt[r] = (uint8_t)c;
                gcnt += c;
            }
        }
        uint32_t faces;
        const uint32_t gex = m_scan_excl<BS>(gcnt, wsum, faces);
        if (a.geom && visit == 0)
            for (int i = 0; i < TW; i++)
                if (i * BS + threadIdx.x < 3u * 256u) s_amb.w[i * BS + threadIdx.x] = tab[i];
        if (threadIdx.x < S::NG) goff[threadIdx.x] = gex;
        if (threadIdx.x == 0) goff[S::NG] = faces;
        if (threadIdx.x < 64) {
            uint64_t excl = 0;
            if (!a.single) {
                if (k == 0) {
                    if (threadIdx.x == 0 && part == 0) st_relaxed(a.state, kMFlagPre | faces);
                } else {
                    if (threadIdx.x == 0 && part == 0) st_relaxed(a.state + k, kMFlagAgg | faces);
                    int64_t top = (int64_t)k - 1;
                    const uint32_t ln = threadIdx.x & 63u;
                    for (;;) {
                        const int64_t j = top - (int64_t)ln;
                        const uint64_t s = (j >= 0) ? ld_relaxed(a.state + j) : kMFlagPre;
                        const uint64_t f = s >> 62;
                        const uint64_t pre = __ballot(f == 2);
                        const uint64_t zero = __ballot(f == 0);
                        const uint64_t need = pre ? (pre & (~pre + 1ull)) * 2ull - 1ull : ~0ull;
                        if (zero & need) {
                            __builtin_amdgcn_s_sleep(1);
                            continue;
                        }
                        uint64_t v = ((need >> ln) & 1ull) ? (s & kMValMask) : 0ull;
#pragma unroll
                        for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
                        excl += v;
                        if (pre) break;
                        top -= 64;
                    }
                    if (threadIdx.x == 0 && part == 0)
                        st_relaxed(a.state + k, kMFlagPre | (excl + faces));
                }
            }
            if (threadIdx.x == 0) s_base = excl;
            if (threadIdx.x == 0 && part == 0) {
                a.offsets[k] = excl;
                if (k + 1 == a.n) a.offsets[a.n] = excl + faces;
                if (bad) atomicOr(a.status, (uint32_t)VP_STATUS_BAD_ID);
                if (a.geom && excl + faces > a.cap) atomicOr(a.status, (uint32_t)VP_STATUS_OVERFLOW);
            }
        }
        __syncthreads();
        const uint64_t base = s_base;
        if (bad || !a.geom || faces == 0 || base + faces > a.cap) continue;

        // ---- 3./4. faces, in passes of whole row groups that fit the list ----
        const uint32_t ox = cx << B, oy = cy << B, oz = cz << B;
        const int16_t own_u = s_uni[13];
        const uint8_t *own = a.voxels + ((uint64_t)id << (3 * B));
        // this part's row groups: those whose first face lies in its share
        uint32_t g0 = 0, gend = (uint32_t)S::NG;
        if (a.parts > 1u) {
            const uint32_t f0 = (uint32_t)((uint64_t)faces * part / a.parts),
                           f1 = (uint32_t)((uint64_t)faces * (part + 1u) / a.parts);
            const bool g = threadIdx.x < (uint32_t)S::NG;
            const uint32_t first = goff[g ? threadIdx.x : 0u];
            g0 = (uint32_t)__syncthreads_count(g && first < f0);
            gend = (uint32_t)__syncthreads_count(g && first < f1);
        }
        while (g0 < gend) {
            const uint32_t lo = goff[g0];
            const bool in = threadIdx.x >= g0 && threadIdx.x < gend &&
                            goff[threadIdx.x + 1] - lo <= (uint32_t)S::LIST;
            const uint32_t g1 = g0 + (uint32_t)__syncthreads_count(in);
            const uint32_t pf = goff[g1] - lo;
            // list entries, one (row, 8-voxel segment) item per thread at a
            // time: a segment's first slot is its row's offset plus the faces
            // of the row's earlier segments, so no scan is needed
            {
                constexpr int SEG = R >= 8 ? R / 8 : 1, SW = R >= 8 ? 8 : R;
                const uint32_t rfirst = g0 * S::GR, nitems = (g1 - g0) * S::GR * SEG;
                for (uint32_t it = threadIdx.x; it < nitems; it += BS) {
                    const uint32_t r = rfirst + it / SEG, sg = it % SEG;
                    if (!rowcnt[r]) continue;
                    const uint32_t g = r / S::GR;
                    uint32_t pos = goff[g] - lo;
                    for (uint32_t q = g * S::GR; q < r; q++) pos += rowcnt[q];
                    const int z = (int)(r / R), y = (int)(r % R);
                    const uint32_t *w = occ + ((z + 1) * P + (y + 1)) * W;
                    const uint64_t o = row_own<B>(w);
                    const uint64_t fx = o ^ row_next<B>(w), fy = o ^ row_own<B>(w + W),
                                   fz = o ^ row_own<B>(w + P * W);
                    const uint32_t sh = sg * SW;
                    const uint64_t below = (1ull << sh) - 1ull;
                    pos += __popcll(fx & below) + __popcll(fy & below) + __popcll(fz & below);
                    constexpr uint32_t SM = (1u << SW) - 1u;
                    const uint32_t mxb = (uint32_t)(fx >> sh) & SM, myb = (uint32_t)(fy >> sh) & SM,
                                   mzb = (uint32_t)(fz >> sh) & SM, ob = (uint32_t)(o >> sh) & SM;
                    uint32_t any = mxb | myb | mzb;
                    while (any) {
                        const uint32_t j = (uint32_t)__builtin_ctz(any);
                        any &= any - 1u;
                        const uint32_t e = ((ob >> j) & 1u) << 20 | r << 8 | (sh + j) << 2;
                        if ((mxb >> j) & 1u) list[pos++] = e | 0u;
                        if ((myb >> j) & 1u) list[pos++] = e | 1u;
                        if ((mzb >> j) & 1u) list[pos++] = e | 2u;
                    }
                }
            }
            __syncthreads();
            // E1: everything but the stores -- ambient terms from LDS, the
            // colour byte and the shadow samples from memory -- packed into
            // one word per face: the vertices' common attribute bits below,
            // then the ambient terms and the rotated flag
            auto prepare = [&](auto uc, uint32_t j0) {
                constexpr int U = decltype(uc)::value;      // faces of a thread in flight
                uint32_t amb[U], col[U], cval[U], pair[U], pair2[U], e[U], wy[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    e[u] = list[min(j0 + (uint32_t)u * BS, pf - 1u)];
                    const uint32_t axis = e[u] & 3u, x = (e[u] >> 2) & 63u, r = (e[u] >> 8) & 4095u;
                    const uint32_t solid = e[u] >> 20, air = solid ^ 1u;
                    const uint32_t z = r >> B, yl = r & (R - 1);
                    const uint32_t ax = axis == 0, ay = axis == 1, az = axis == 2;
                    // the air cell of the pair is A, or B when A is solid
                    const uint32_t nb = plane_bits<B>(occ, axis, (int)(x + (ax & solid)),
                                                      (int)(yl + (ay & solid)), (int)(z + (az & solid)));
                    amb[u] = reinterpret_cast<const uint16_t *>(s_amb.w)[axis << 9 | nb];
                    // the solid voxel: A, or B at +axis (maybe in the next chunk)
                    const uint32_t sx = x + (ax & air), sy = yl + (ay & air), sz = z + (az & air);
                    const uint32_t at = ((sz & (R - 1)) << B | (sy & (R - 1))) << B | (sx & (R - 1));
                    int16_t un = own_u;
                    const uint8_t *p = own + at;
                    if ((sx | sy | sz) & (uint32_t)R) {
                        const int nbr = 13 + (sx >> B) + 3 * (sy >> B) + 9 * (sz >> B);
                        un = s_uni[nbr];
                        p = a.voxels + ((uint64_t)s_nid[nbr] << (3 * B)) + at;
                    }
                    cval[u] = un >= 0 ? (uint32_t)un : 0u;
                    col[u] = 0u;
                    if (un < 0) col[u] = *p;
                    // Shadow samples (mesher.c:282-320, shadow.h:52-75), pairs of
                    // neighbouring map entries: (i - 1, i) of the solid +x cell for
                    // x faces of air; (i, i + 1) of the voxel for y faces of solid
                    // voxels; for z faces (i, i + 1) of the cell in front and
                    // (i - 1, i) one below it
                    const uint32_t wx = ox + x;
                    wy[u] = oy + yl;
                    const uint32_t i = wx + wy[u] + ax + a.map_sx * (oz + z + (az & solid));
                    const bool first = ax ? air != 0u : (ay ? solid != 0u : wy[u] != 0u);
                    pair[u] = pair2[u] = 0u;
                    if (first) __builtin_memcpy(&pair[u], a.map + (i - (ay ^ 1u)), 4);
                    if (az) __builtin_memcpy(&pair2[u], a.map + i, 4);
                }
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const uint32_t axis = e[u] & 3u, solid = e[u] >> 20, top = wy[u] + 1u;
                    const uint32_t m1 = max(pair[u] & 0xFFFFu, pair[u] >> 16);
                    const uint32_t m2 = max(pair2[u] & 0xFFFFu, pair2[u] >> 16);
                    uint32_t shadow = 0, diamond = 3;
                    if (axis == 2) {
                        diamond = (m2 < top ? 2u : 0u) | (wy[u] != 0u && m1 < wy[u] ? 1u : 0u);
                    } else if (axis == solid) {          // x faces of air, y faces of solid voxels
                        shadow = m1 < top ? 0u : 1u;
                    }
                    const uint32_t code = axis + (solid ? 0u : 3u);
                    const uint32_t j = j0 + (uint32_t)u * BS;
                    if (j < pf)
                        packed[j] = (col[u] | cval[u]) | code << 8 | shadow << 13 | diamond << 14 | amb[u] << 16;
                }
            };
            for (uint32_t j0 = 0; j0 < pf;) {
                const uint32_t left = (pf - j0 + BS - 1u) / BS;
                if (left >= 3u) {
                    prepare(std::integral_constant<int, 4>{}, j0 + threadIdx.x);
                    j0 += 4u * BS;
                } else {
                    prepare(std::integral_constant<int, 1>{}, j0 + threadIdx.x);
                    j0 += BS;
                }
            }
            __syncthreads();
            // E2: the stores, whole lines per instruction: half a face's vertices
            // per lane, then a third of its indices
            {
                uint4 *gp = reinterpret_cast<uint4 *>(a.geom + 16 * (base + lo));
                const uint32_t oxy = (ox & 0xFFFFu) | oy << 16;
                for (uint32_t i = threadIdx.x; i < 2u * pf; i += BS) {
                    const uint32_t e = list[i >> 1], pk = packed[i >> 1];
                    const uint32_t x = (e >> 2) & 63u, r = (e >> 8) & 4095u;
                    const uint4 c = s_corner[(e & 3u) << 1 | (i & 1u)];
                    const uint32_t xy = oxy + (x | (r & (R - 1)) << 16);
                    const uint32_t za = ((oz + (r >> B)) & 0xFFFFu) | pk << 16;
                    const uint32_t amb = pk >> (16 + 4 * (i & 1u));
                    nt_store16(gp + i, make_uint4(add_u16x2(xy, c.x),
                                                  add_u16x2(za, c.y) | (amb & 3u) << 22,
                                                  add_u16x2(xy, c.z),
                                                  add_u16x2(za, c.w) | (amb & 12u) << 20));
                }
                uint2 *ip = reinterpret_cast<uint2 *>(a.index + 6 * (base + lo));
                for (uint32_t i = threadIdx.x; i < 3u * pf; i += BS) {
                    const uint32_t f = (i * 0xAAABu) >> 17, k = i - 3u * f;     // f = i / 3
                    const uint32_t pk = packed[f];
                    const uint32_t t = m_tri_row(((pk >> 8) & 7u) >= 3u, (pk >> 24) & 1u) >> (4u * k);
                    const uint32_t vb = 4u * (lo + f);
                    nt_store8(ip + i, make_uint2(vb + (t & 3u), vb + ((t >> 2) & 3u)));
                }
            }
            __syncthreads();
            g0 = g1;
        }
    }
}

__global__ void k_mesh_reset(uint32_t *ticket, uint64_t *state, uint32_t n, uint64_t *offsets)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) {
        ticket[0] = 0u;
        offsets[0] = 0ull;
    }
    for (uint32_t j = i; j < n; j += gridDim.x * blockDim.x) state[j] = 0ull;
}

template <int B>
static hipError_t mesh_launch(const MeshArgs &a, int grid, hipStream_t st)
{
    hipLaunchKernelGGL((k_mesh<B>), dim3(grid), dim3(kMeshBS), 0, st, a);
    return hipGetLastError();
}

}  // namespace vp

using namespace vp;

extern "C" int vp_gpu_mesh(vp_ctx *ctx, const vp_world_desc *world, const uint8_t *d_voxels,
                           const int16_t *d_uniform, const vp_shadow_desc *shadow,
                           const uint32_t *d_chunk_ids, uint32_t n, const vp_mesh_out *out,
                           void *stream)
{
    if (!ctx || !world || !d_voxels || !shadow || !shadow->d_map || (!d_chunk_ids && n) || !out ||
        !out->d_face_offsets)
        return VP_ERR_ARG;
    const bool count_only = !out->d_geometry && !out->d_index && out->capacity_faces == 0;
    if (!count_only && (!out->d_geometry || !out->d_index)) return VP_ERR_ARG;
    const uint32_t root_bitw = world->root_bitw;
    if (root_bitw < 2 || root_bitw > 6) return VP_ERR_UNSUPPORTED;
    const uint32_t mbs = (uint32_t)world->max_bitw[0] + world->max_bitw[1] + world->max_bitw[2];
    if (mbs > 31u || mbs + 3u * root_bitw > 40u) return VP_ERR_ARG;
    const uint64_t sx = ((uint64_t)1 << (world->max_bitw[0] + root_bitw)) +
                        ((uint64_t)1 << (world->max_bitw[1] + root_bitw));
    if (shadow->size_x != sx) return VP_ERR_ARG;
    hipStream_t st = as_stream(stream);
    MeshArgs a = {};
    a.voxels = d_voxels;
    a.uniform = d_uniform;
    a.map = shadow->d_map;
    a.map_sx = shadow->size_x;
    a.ids = d_chunk_ids;
    a.n = n;
    a.nchunks = (uint32_t)(1ull << mbs);
    a.mb0 = world->max_bitw[0];
    a.mb1 = world->max_bitw[1];
    a.mb2 = world->max_bitw[2];
    a.single = (n == 1) ? 1u : 0u;
    // Short lists: a chunk's face count takes a small part of its time, so
    // several workgroups repeat it and share out the faces, as many as the
    // grid holds at once and at most R / 4 (100 chunks around a camera:
    // 358 -> 136 us).
    const uint32_t resident = (uint32_t)ctx->num_cus * 2u;
    a.parts = 1u;
    if (!count_only && root_bitw >= 5 && n && n <= resident / 2u)
        a.parts = std::min(1u << (root_bitw - 2u), resident / n);
    a.geom = count_only ? nullptr : out->d_geometry;
    a.index = count_only ? nullptr : out->d_index;
    a.cap = out->capacity_faces;
    a.offsets = out->d_face_offsets;
    a.status = ctx->d_status;
    std::lock_guard<std::mutex> g(ctx->mu);
    int grid = (int)a.parts;
    if (!a.single) {
        int rc = ensure_state(ctx, n ? n : 1);
        if (rc) return rc;
        a.ticket = ctx->d_ticket;
        a.state = ctx->d_state;
        grid = (int)(a.parts > 1u ? n * a.parts : std::min(n, resident));
        const int rgrid = (int)((n + 255u) / 256u);
        hipLaunchKernelGGL(k_mesh_reset, dim3(rgrid < 1 ? 1 : (rgrid < 1024 ? rgrid : 1024)),
                           dim3(256), 0, st, a.ticket, a.state, n, a.offsets);
        VP_HIP_TRY(hipGetLastError());
        if (n == 0) return VP_OK;
    }
    hipError_t e;
    switch (root_bitw) {
    case 2: e = mesh_launch<2>(a, grid, st); break;
    case 3: e = mesh_launch<3>(a, grid, st); break;
    case 4: e = mesh_launch<4>(a, grid, st); break;
    case 5: e = mesh_launch<5>(a, grid, st); break;
    default: e = mesh_launch<6>(a, grid, st); break;
    }
    return e == hipSuccess ? VP_OK : VP_ERR_HIP;
}
