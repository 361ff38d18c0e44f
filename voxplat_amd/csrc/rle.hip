// rle.hip -- chunk RLE encode/decode for gfx950.
//
// Replaces rle_compress / rle_decompress (src/chunkset/rle.c:44-116) and the
// per-chunk (de)compression done by chunk_compress / chunk_open_*
// (src/chunkset.c:133-230).  Word format: (value << 24) | run, runs maximal
// in voxel order, one 0 word after each chunk's runs.
//
// Encode, one workgroup per chunk (persistent, ticket order = list order):
//  1. 16-byte loads; a run starts where a byte differs from the byte before it
//     -> one start bit per voxel in an LDS bitmap (R^3 bits = 32 KiB at R=64).
//  2. starts and first start of each 64 bitmap words; a scan over these groups
//     gives a group's first run index, and the first start after it.
//  3. the chunk's word count is published and its output offset taken by a
//     decoupled look-back (same scheme as the remesh kernel).
//  4. each wave lists the starts of a group in LDS and writes their words.
// Decode, one workgroup per chunk (or, of few chunks, several): a stream of one
// full-chunk run is a fill; otherwise the words are read eight per thread at a
// time, their values kept in LDS and their lengths scanned into start
// positions, set as bits of an LDS bitmap; an output byte's run is the rank of
// the last start at or before it, so every 16-byte store is independent.
// Bound by its stores and by the scan's latency: a 2048x256x2048 world (1.07 GB
// of voxels from 0.2 GB of words) 554 -> 270 us, 4.7 TB/s (the kernel; reopening
// the world with it, the uniform table included, 600 -> 333 us).
#include "vp_internal.h"

namespace vp {

constexpr uint64_t kRFlagAgg = 1ull << 62;
constexpr uint64_t kRFlagPre = 2ull << 62;
constexpr uint64_t kRValMask = (1ull << 62) - 1;

struct RleArgs {
    uint8_t        *voxels;
    const uint32_t *ids;
    uint32_t        n;
    const uint32_t *d_n;           // nullable: device-resident count <= n (encode)
    uint32_t       *words;
    uint64_t        cap;
    uint64_t       *offsets;
    int16_t        *uniform_out;
    const int16_t  *uniform_in;    // nullable: a chunk marked uniform here is not read (encode)
    uint32_t       *ticket;
    uint64_t       *state;
    uint32_t       *status;
    uint8_t         single;
    uint32_t        nchunks;
    uint32_t        parts;         // workgroups that share a chunk's bytes (decode)
};

__device__ __forceinline__ uint32_t r_lane() { return threadIdx.x & 63u; }

// start bits of the 4 bytes of w given the byte before it
__device__ __forceinline__ uint32_t diff4(uint32_t w, uint32_t prev)
{
    const uint32_t shifted = (w << 8) | (prev & 0xFFu);
    const uint32_t d = w ^ shifted;
    const uint32_t m = (((d & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | d) & 0x80808080u;
    return (((m >> 7) * 0x00204081u) >> 21) & 0xFu;
}

// LDS of the encoder: two workgroups per CU at R = 64.
template <int B, int BS>
struct EncodeLds {
    static constexpr int VOX = 1 << (3 * B), WORDS = VOX / 64, NG = (WORDS + 63) / 64;
    static constexpr int CAP = VOX < 960 ? VOX : 960;       // starts a wave lists at a time
    static constexpr int GB = VOX < 4096 ? VOX : 4096;      // bytes of a group of 64 words
    uint64_t bm[WORDS];             // bit per voxel: a run starts here
    uint32_t gtot[NG], gfirst[NG];  // per 64 bitmap words: starts, and the first of them
    uint64_t base;
    uint32_t ticket;
    uint4    vox[BS / 64][(GB + 15) / 16];
    uint16_t list[BS / 64][CAP];
};

// Accesses of a wave's LDS list by its different lanes stay in program order.
__device__ __forceinline__ void wave_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int B, int BS>
__device__ void rle_encode_chunk(const RleArgs &a, uint32_t k, uint32_t n, EncodeLds<B, BS> &L)
{
    constexpr int R = 1 << B, VOX = R * R * R, WORDS = VOX / 64;
    uint32_t chunk = a.ids[k];
    if (chunk >= a.nchunks) {       // encode the all-air null chunk instead
        if (threadIdx.x == 0) atomicOr(a.status, (uint32_t)VP_STATUS_BAD_ID);
        chunk = 0xFFFFFFFFu;
    }
    const uint8_t *src = chunk == 0xFFFFFFFFu ? nullptr : a.voxels + ((size_t)chunk << (3 * B));
    // A chunk the caller's uniform table marks uniform (every voxel holds that
    // value; edits mark their chunks mixed) is one run and the terminator:
    // none of its voxels is read.
    int uval = (src && a.uniform_in) ? (int)a.uniform_in[chunk] : -1;
    bool fast = uval >= 0;
    uint32_t runs = 1, gbeg = 0, gnext = 0;
    constexpr int NW = BS / 64, NG = EncodeLds<B, BS>::NG;
    const uint32_t ln = r_lane();
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (!fast) {

    // ---- 1. start bits ----
    // DEPTH 16-byte loads per thread in flight; the byte before a piece is
    // the previous lane's last byte, except at lane 0, which loads it.
    if constexpr (VOX >= 16) {
        constexpr int PIECES = VOX / 16;
        constexpr int PER = PIECES / BS;
        constexpr int DEPTH = PER >= 8 ? 8 : (PER >= 1 ? PER : 1);
        uint16_t *b16 = reinterpret_cast<uint16_t *>(L.bm);
        if (!src) {
            for (int s = threadIdx.x; s < PIECES; s += BS) b16[s] = s ? 0 : 1;
        } else {
#pragma unroll 1
            for (int s0 = 0; s0 < PIECES; s0 += BS * DEPTH) {
                uint4 v[DEPTH];
                uint32_t pb[DEPTH];
#pragma unroll
                for (int d = 0; d < DEPTH; d++) {
                    const int sp = s0 + d * BS + (int)threadIdx.x;
                    const int sc = sp < PIECES ? sp : 0;
                    v[d] = *reinterpret_cast<const uint4 *>(src + (size_t)sc * 16);
                    pb[d] = (ln == 0u && sp > 0 && sp < PIECES) ? src[(size_t)sp * 16 - 1] : 0u;
                }
#pragma unroll
                for (int d = 0; d < DEPTH; d++) {
                    const int sp = s0 + d * BS + (int)threadIdx.x;
                    uint32_t prev = (uint32_t)__shfl_up((int)(v[d].w >> 24), 1, 64);
                    if (ln == 0u) prev = sp ? pb[d] : (~v[d].x & 0xFFu);
                    uint32_t m = diff4(v[d].x, prev);
                    m |= diff4(v[d].y, v[d].x >> 24) << 4;
                    m |= diff4(v[d].z, v[d].y >> 24) << 8;
                    m |= diff4(v[d].w, v[d].z >> 24) << 12;
                    if (sp < PIECES) b16[sp] = (uint16_t)m;
                }
            }
        }
    }
    __syncthreads();

    // ---- 2. runs and first start of each group of 64 bitmap words ----
    // lane g then holds group g's first run index and the first start after it
    for (int g = wv; g < NG; g += NW) {
        const int w = g * 64 + (int)ln;
        const uint64_t b = w < WORDS ? L.bm[w] : 0ull;
        uint32_t tot;
        (void)wave_excl_scan((uint32_t)__popcll(b), tot);
        const uint64_t nz = __ballot(b != 0ull);
        const uint32_t at = nz ? (uint32_t)__builtin_ctzll(nz) : 0u;
        const uint32_t bit = b ? (uint32_t)__builtin_ctzll(b) : 0u;
        const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)bit, (int)at);
        if (ln == 0) {
            L.gtot[g] = tot;
            L.gfirst[g] = nz ? (uint32_t)(g * 64 + (int)at) * 64u + first : (uint32_t)VOX;
        }
    }
    __syncthreads();
    const bool has = (int)ln < NG;
    gbeg = wave_excl_scan(has ? L.gtot[ln] : 0u, runs);
    gnext = (uint32_t)__shfl_down((int)(has ? L.gfirst[ln] : (uint32_t)VOX), 1, 64);
    if (ln == 63u) gnext = (uint32_t)VOX;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = (uint32_t)__shfl_down((int)gnext, d, 64);
        if (ln + d < 64u) gnext = min(gnext, y);
    }
    }   // !fast

    if (runs == 1u && !fast) {          // one value after all
        uval = src ? (int)src[0] : 0;
        fast = true;
    }
    // the voxels of a wave's first group are on their way during the look-back
    constexpr int GQ = (EncodeLds<B, BS>::GB / 16 + 63) / 64;
    uint4 ahead[GQ];
    auto fetch = [&](int g) {
#pragma unroll
        for (int q = 0; q < GQ; q++) {
            const int i = (int)ln + 64 * q;
            ahead[q] = make_uint4(0u, 0u, 0u, 0u);
            if (src && g < NG && i * 16 < EncodeLds<B, BS>::GB)
                ahead[q] = *reinterpret_cast<const uint4 *>(src + (size_t)g * 4096 + (size_t)i * 16);
        }
    };
    if (!fast && a.words) fetch(wv);

    // ---- 3. publish the word count (runs + terminator), look back ----
    const uint64_t nwords = (uint64_t)runs + 1u;
    if (threadIdx.x < 64) {
        uint64_t excl = 0;
        if (!a.single) {
            if (k == 0) {
                if (threadIdx.x == 0) st_relaxed(a.state, kRFlagPre | nwords);
            } else {
                if (threadIdx.x == 0) st_relaxed(a.state + k, kRFlagAgg | nwords);
                int64_t top = (int64_t)k - 1;
                const uint32_t ln = r_lane();
                for (;;) {
                    const int64_t j = top - (int64_t)ln;
                    const uint64_t s = (j >= 0) ? ld_relaxed(a.state + j) : kRFlagPre;
                    const uint64_t f = s >> 62;
                    const uint64_t pre = __ballot(f == 2);
                    const uint64_t zero = __ballot(f == 0);
                    const uint64_t need = pre ? (pre & (~pre + 1ull)) * 2ull - 1ull : ~0ull;
                    if (zero & need) {
                        __builtin_amdgcn_s_sleep(1);
                        continue;
                    }
                    uint64_t v = ((need >> ln) & 1ull) ? (s & kRValMask) : 0ull;
#pragma unroll
                    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
                    excl += v;
                    if (pre) break;
                    top -= 64;
                }
                if (threadIdx.x == 0) st_relaxed(a.state + k, kRFlagPre | (excl + nwords));
            }
        }
        if (threadIdx.x == 0) {
            L.base = excl;
            a.offsets[k] = excl;
            if (k + 1 == n) a.offsets[n] = excl + nwords;
            if (a.uniform_out)
                a.uniform_out[k] = fast ? (int16_t)uval : (int16_t)-1;
            if (a.words && excl + nwords > a.cap) atomicOr(a.status, (uint32_t)VP_STATUS_OVERFLOW);
        }
    }
    __syncthreads();
    const uint64_t base = L.base;
    if (!a.words || base + nwords > a.cap) return;

    // ---- 4. words ----
    // A wave takes a group of 64 bitmap words at a time: each lane lists its
    // word's starts in LDS, then consecutive lanes take consecutive runs, so
    // that the words' stores are whole lines.  The group's voxels come through
    // LDS, loaded a group ahead.
    // A group with more starts than the list holds goes in batches of words.
    uint32_t *out = a.words + base;
    if (fast) {
        if (threadIdx.x == 0) out[0] = ((uint32_t)uval << 24) | (uint32_t)VOX;
    } else {
        constexpr uint32_t CAP = EncodeLds<B, BS>::CAP;
        uint16_t *list = L.list[wv];
        for (int g = wv; g < NG; g += NW) {
            const int w = g * 64 + (int)ln;
            const uint64_t b = w < WORDS ? L.bm[w] : 0ull;
            const uint32_t cnt = (uint32_t)__popcll(b);
            uint32_t tot;
            const uint32_t off = wave_excl_scan(cnt, tot);
            uint32_t *og = out + (uint32_t)__builtin_amdgcn_readlane((int)gbeg, g);
            const uint8_t *sg = reinterpret_cast<const uint8_t *>(L.vox[wv]);
            wave_order();                      // the previous group's reads are done
#pragma unroll
            for (int q = 0; q < GQ; q++)
                if (((int)ln + 64 * q) * 16 < EncodeLds<B, BS>::GB) L.vox[wv][(int)ln + 64 * q] = ahead[q];
            fetch(g + NW);
            const uint32_t gend = (uint32_t)__builtin_amdgcn_readlane((int)gnext, g) - (uint32_t)g * 4096u;
#pragma unroll 1
            for (uint32_t b0 = 0; b0 < tot;) {
                // the words [b0, b1) of the group, and the start after them
                uint32_t b1 = tot, after = gend;
                if (tot - b0 > CAP) {
                    const uint64_t over = __ballot(cnt && off >= b0 && off + cnt > b0 + CAP);
                    const int f = __builtin_ctzll(over);
                    b1 = (uint32_t)__builtin_amdgcn_readlane((int)off, f);
                    after = (uint32_t)f * 64u +
                            (uint32_t)__builtin_amdgcn_readlane((int)(b ? __builtin_ctzll(b) : 0), f);
                }
                wave_order();                  // the previous batch's reads are done
                if (cnt && off >= b0 && off < b1) {
                    uint16_t *q = list + (off - b0);
                    auto half = [&](uint32_t m, uint32_t x0) {
                        while (m) {
                            *q++ = (uint16_t)(x0 + (uint32_t)__builtin_ctz(m));
                            m &= m - 1u;
                        }
                    };
                    half((uint32_t)b, ln * 64u);
                    half((uint32_t)(b >> 32), ln * 64u + 32u);
                }
                wave_order();
                const uint32_t nb = b1 - b0;
                constexpr int U = 4;           // runs per lane in flight
#pragma unroll 1
                for (uint32_t j0 = 0; j0 < nb; j0 += 64 * U) {
                    uint32_t pos[U], end[U], val[U];
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const uint32_t j = min(j0 + (uint32_t)u * 64u + ln, nb - 1u);
                        pos[u] = list[j];
                        end[u] = j + 1u < nb ? (uint32_t)list[j + 1u] : after;
                        val[u] = (uint32_t)sg[pos[u]];
                    }
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const uint32_t j = j0 + (uint32_t)u * 64u + ln;
                        if (j < nb) og[b0 + j] = val[u] << 24 | (end[u] - pos[u]);
                    }
                }
                b0 = b1;
            }
        }
    }
    if (threadIdx.x == 0) out[runs] = 0u;
}

template <int B, int BS>
__global__ void __launch_bounds__(BS, 4) k_rle_encode(RleArgs a)
{
    __shared__ EncodeLds<B, BS> L;
    if (a.single) {
        rle_encode_chunk<B, BS>(a, 0u, 1u, L);
        return;
    }
    const uint32_t n = a.d_n ? min(*a.d_n, a.n) : a.n;
    for (;;) {
        if (threadIdx.x == 0) L.ticket = atomicAdd(a.ticket, 1u);
        __syncthreads();
        const uint32_t k = L.ticket;
        if (k >= n) break;
        rle_encode_chunk<B, BS>(a, k, n, L);
        __syncthreads();
    }
}

// 16 bytes of stream words at any word address
struct __attribute__((packed, aligned(4))) Words4 {
    uint32_t w[4];
};

template <int B, int BS>
__global__ void __launch_bounds__(BS) k_rle_decode(RleArgs a)
{
    constexpr int R = 1 << B, VOX = R * R * R, WORDS = VOX / 64, WPT = (WORDS + BS - 1) / BS;
    constexpr int NW = BS / 64;
    constexpr int K = 8;             // stream words per thread per batch, loads in flight
    // run values kept in LDS for streams of up to VCAP runs: at R = 64 what
    // leaves two workgroups per CU (2 x 81.9 KB); a chunk with 5% of its
    // voxels as single-voxel holes has about 26,000 runs
    constexpr int VCAP = VOX < 32448 ? VOX : 32448;
    constexpr uint32_t LMAX = (uint32_t)VOX + 1u;   // longer runs are malformed; clamped
    __shared__ uint64_t bm[WORDS];
    __shared__ uint32_t rank[WORDS];
    __shared__ uint32_t val32[VCAP / 4 + 4];        // the value of run i is byte i + 1
    __shared__ uint32_t wtot[WPT * NW > 2 * NW ? WPT * NW : 2 * NW];   // totals of the waves
    __shared__ uint32_t s_bad, s_nz;
    static_assert(WPT * NW <= 64, "one wave scans the wave totals");
    uint8_t *val8 = reinterpret_cast<uint8_t *>(val32);
    uint32_t *bm32 = reinterpret_cast<uint32_t *>(bm);
    const uint32_t ln = r_lane();
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    bool fresh = true;               // bm was never cleared; later each chunk leaves it clear
    // Round r hands entries r G .. r G + G - 1 to the G workgroups, rotated by a
    // golden-section step per round: with the plain stride a workgroup of a
    // whole world meets the same height every time, all air or all caves.
    // (2048x256x2048 world: 324 -> 265 us, the kernel.)
    const uint32_t G = gridDim.x / a.parts, turn = (uint32_t)(0.618f * (float)G) | 1u;
    uint32_t slot = blockIdx.x / a.parts;
    // a part's share of the chunk's 16-byte pieces, in multiples of the workgroup
    const uint32_t part = blockIdx.x - slot * a.parts;
    const int p_lo = (int)((uint32_t)(VOX / 16) / a.parts * part),
              p_hi = p_lo + (int)((uint32_t)(VOX / 16) / a.parts);
    for (uint64_t k0 = 0; k0 < a.n; k0 += G, slot = (slot + turn) % G) {
        if (k0 + slot >= a.n) break;
        const uint32_t k = (uint32_t)k0 + slot;
        const uint32_t chunk = a.ids[k];
        const uint64_t o0 = a.offsets[k], o1 = a.offsets[k + 1];
        if (chunk >= a.nchunks || o0 > o1 || o1 > a.cap) {
            if (threadIdx.x == 0) atomicOr(a.status, (uint32_t)VP_STATUS_BAD_ID);
            continue;   // uniform across the workgroup
        }
        uint8_t *dst = a.voxels + ((size_t)chunk << (3 * B));
        const uint32_t *wd = a.words + o0;
        const uint64_t avail = o1 - o0;
        // one run over the whole chunk, then the terminator: a fill
        if (avail >= 2) {
            const uint32_t w0 = wd[0], w1 = wd[1];   // the same address in every lane
            if ((w0 & 0xFFFFFFu) == (uint32_t)VOX && w1 == 0u) {
                const uint32_t b = w0 >> 24;
                const uint32_t v4 = b * 0x01010101u;
                const uint4 q = make_uint4(v4, v4, v4, v4);
                for (int s = p_lo + (int)threadIdx.x; s < p_hi; s += BS)
                    nt_store16(dst + (size_t)s * 16, q);
                continue;   // uniform across the workgroup
            }
        }
        if (fresh)
            for (int w = threadIdx.x; w < WORDS; w += BS) bm[w] = 0ull;
        fresh = false;
        // The runs end at the first 0 word after word 0 (rle.c:100-108: the
        // first word is always expanded): the last word of a well-formed
        // stream.  One found earlier takes its batch again.
        uint64_t nz = avail;
        if (avail >= 2 && wd[avail - 1] == 0u) nz = avail - 1;
        if (threadIdx.x == 0) {
            s_bad = 0u;
            s_nz = (uint32_t)(nz < 0xFFFFFFFFull ? nz : 0xFFFFFFFFull);
        }
        __syncthreads();
        // run starts: batches of K words per thread; the terminator search,
        // the run values (into LDS) and a scan of the lengths into start bits.
        // The next batch's words are loaded while a batch is worked on.
        auto fetch = [&](uint64_t i0, uint32_t (&wv8)[K]) {
            if (i0 + K <= avail) {
#pragma unroll
                for (int q = 0; q < K / 4; q++) {
                    const Words4 v = *reinterpret_cast<const Words4 *>(wd + i0 + 4 * q);
#pragma unroll
                    for (int j = 0; j < 4; j++) wv8[4 * q + j] = v.w[j];
                }
            } else {
#pragma unroll
                for (int j = 0; j < K; j++) wv8[j] = (i0 + j < avail) ? wd[i0 + j] : 1u;
            }
        };
        uint64_t pos = 0;
        uint32_t cur[K], par = 0;
        if (nz) fetch((uint64_t)threadIdx.x * K, cur);
        for (uint64_t b0 = 0; b0 < nz; b0 += (uint64_t)BS * K) {
            const uint64_t i0 = b0 + (uint64_t)threadIdx.x * K;
            uint32_t nxt[K] = {};
            if (b0 + (uint64_t)BS * K < nz) fetch(i0 + (uint64_t)BS * K, nxt);
            uint32_t len[K];
            uint64_t st = 0;
            uint32_t tot = 0;
            for (;;) {
                uint32_t lsum = 0;
                bool bad = false;
#pragma unroll
                for (int j = 0; j < K; j++) {
                    const uint64_t i = i0 + j;
                    uint32_t l = (i < nz) ? (cur[j] & 0xFFFFFFu) : 0u;
                    // a 0 word before the known end is the end
                    if (cur[j] == 0u && i >= 1 && i < nz && i <= 0xFFFFFFFFull)
                        atomicMin(&s_nz, (uint32_t)i);
                    bad |= (i < nz) && (l == 0u || l > LMAX);   // zero-length or oversized runs
                    l = l < LMAX ? l : LMAX;
                    len[j] = l;
                    lsum += l;
                }
                uint32_t wt;
                const uint32_t ex = wave_excl_scan(lsum, wt);
                if (ln == 0) wtot[par * NW + wv] = wt;
                __syncthreads();
                // a wave ahead of this one may have met an end in the next batch
                const uint64_t end = s_nz, stop = min(nz, b0 + (uint64_t)BS * K);
                uint32_t before = 0;
                tot = 0;
#pragma unroll
                for (int q = 0; q < NW; q++) {
                    const uint32_t t = wtot[par * NW + q];
                    before += q < wv ? t : 0u;
                    tot += t;
                }
                par ^= 1u;
                st = pos + before + ex;
                if (end < stop && end < 0xFFFFFFFFull) {   // uniform: an early end
                    nz = end;
                    continue;
                }
                if (bad) s_bad = 1u;
                break;
            }
#pragma unroll
            for (int j = 0; j < K; j++) {
                const uint64_t i = i0 + j;
                if (i < nz && i < (uint64_t)VCAP) val8[i + 1] = (uint8_t)(cur[j] >> 24);
            }
            // the starts of a 32-bit word of the map go there together
            uint32_t at = 0, bits = 0;
#pragma unroll
            for (int j = 0; j < K; j++) {
                if (len[j] && st < (uint64_t)VOX) {
                    const uint32_t w = (uint32_t)st >> 5;
                    if (w != at) {
                        if (bits) atomicOr(&bm32[at], bits);
                        at = w;
                        bits = 0;
                    }
                    bits |= 1u << ((uint32_t)st & 31u);
                }
                st += len[j];
            }
            if (bits) atomicOr(&bm32[at], bits);
            pos += tot;
#pragma unroll
            for (int j = 0; j < K; j++) cur[j] = nxt[j];
        }
        if (threadIdx.x == 0 && pos != (uint64_t)VOX) s_bad = 1u;
        __syncthreads();
        const uint64_t nw = nz;
        // rank of each bitmap word = starts before it: words strided over the
        // threads, a scan per wave and row of words, then one of the totals
        uint32_t rk[WPT];
#pragma unroll
        for (int j = 0; j < WPT; j++) {
            const int w = j * BS + (int)threadIdx.x;
            const uint32_t c = w < WORDS ? (uint32_t)__popcll(bm[w]) : 0u;
            uint32_t wt;
            rk[j] = wave_excl_scan(c, wt);
            if (ln == 0) wtot[j * NW + wv] = wt;
        }
        __syncthreads();
        {
            uint32_t all;
            const uint32_t t = wave_excl_scan((int)ln < WPT * NW ? wtot[ln] : 0u, all);
#pragma unroll
            for (int j = 0; j < WPT; j++) {
                const int w = j * BS + (int)threadIdx.x;
                const uint32_t base = (uint32_t)__builtin_amdgcn_readlane((int)t, j * NW + wv);
                if (w < WORDS) rank[w] = base + rk[j];
            }
        }
        __syncthreads();
        // bytes: run index of byte p = starts at or before p, minus one; each
        // start belongs to a run index below nw.  A piece of 16 bytes with up
        // to 7 starts takes its values from 8 consecutive bytes, picked by the
        // running count of its starts: four counts at a time from a multiply
        // and two adds, one byte permute per four bytes.
        const bool in_lds = nw <= (uint64_t)VCAP;
        for (int s = p_lo + (int)threadIdx.x; s < p_hi; s += BS) {
            const int w = s >> 2;
            const uint64_t b = bm[w];
            if ((s & 3) == 3) bm[w] = 0ull;     // cleared for the next chunk: its four readers are this wave's
            const int sh = (s & 3) * 16;
            const uint64_t below = b & ((1ull << sh) - 1ull);
            const uint32_t idx = rank[w] + (uint32_t)__popcll(below);   // run index + 1 of byte -1
            const uint32_t bits16 = (uint32_t)(b >> sh) & 0xFFFFu;
            uint32_t out[4] = {0, 0, 0, 0};
            const uint64_t p0 = (uint64_t)s * 16;
            if (in_lds && p0 + 16 <= pos && __popc(bits16) <= 7) {
                const uint32_t *v = val32 + (idx >> 2);
                const uint32_t v0 = v[0], v1 = v[1], v2 = v[2];
                const uint32_t lo = __builtin_amdgcn_alignbyte(v1, v0, idx & 3u);
                const uint32_t hi = __builtin_amdgcn_alignbyte(v2, v1, idx & 3u);
                uint32_t base = 0;              // starts so far, in each byte
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    uint32_t t = __umul24((bits16 >> (4 * d)) & 15u, 0x204081u) & 0x01010101u;
                    t += t << 8;
                    t += t << 16;               // byte j: starts in bytes 0..j
                    t += base;
                    out[d] = __builtin_amdgcn_perm(hi, lo, t);
                    base = __builtin_amdgcn_perm(t, t, 0x03030303u);
                }
            } else {
#pragma unroll
                for (int j = 0; j < 16; j++) {
                    const int ri = (int)idx - 1 + __popc(bits16 & ((2u << j) - 1u));
                    uint32_t v = 0;
                    if (ri >= 0 && p0 + j < pos)
                        v = in_lds ? (uint32_t)val8[ri + 1] : (wd[ri] >> 24);
                    out[j >> 2] |= v << ((j & 3) * 8);
                }
            }
            nt_store16(dst + p0, make_uint4(out[0], out[1], out[2], out[3]));
        }
        if (threadIdx.x == 0 && s_bad) atomicOr(a.status, (uint32_t)VP_STATUS_BAD_RLE);
        __syncthreads();
    }
}

__global__ void k_rle_reset(uint32_t *ticket, uint64_t *state, uint32_t n, uint64_t *offsets)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) {
        ticket[0] = 0u;
        offsets[0] = 0ull;
    }
    for (uint32_t j = i; j < n; j += gridDim.x * blockDim.x) state[j] = 0ull;
}

template <int B>
static hipError_t rle_launch(int dir, const RleArgs &a, int grid, hipStream_t st)
{
    if (dir == VP_RLE_ENCODE)
        hipLaunchKernelGGL((k_rle_encode<B, 512>), dim3(grid), dim3(512), 0, st, a);
    else
        hipLaunchKernelGGL((k_rle_decode<B, 512>), dim3(grid), dim3(512), 0, st, a);
    return hipGetLastError();
}

static int rle_check(const vp_world_desc *world)
{
    if (!world) return VP_ERR_ARG;
    if (world->root_bitw < 2 || world->root_bitw > 6) return VP_ERR_UNSUPPORTED;
    if ((int)world->max_bitw[0] + world->max_bitw[1] + world->max_bitw[2] > 32) return VP_ERR_ARG;
    return VP_OK;
}

static hipError_t rle_dispatch(uint32_t root_bitw, int dir, const RleArgs &a, int grid,
                               hipStream_t st)
{
    switch (root_bitw) {
    case 2: return rle_launch<2>(dir, a, grid, st);
    case 3: return rle_launch<3>(dir, a, grid, st);
    case 4: return rle_launch<4>(dir, a, grid, st);
    case 5: return rle_launch<5>(dir, a, grid, st);
    default: return rle_launch<6>(dir, a, grid, st);
    }
}

int rle_encode_launch(vp_ctx *ctx, const vp_world_desc *world, const uint8_t *d_voxels,
                      const uint32_t *d_chunk_ids, uint32_t n, const uint32_t *d_n,
                      uint32_t *d_words, uint64_t capacity_words, uint64_t *d_word_offsets,
                      int16_t *d_uniform_out, const int16_t *d_uniform_in, uint32_t *ticket,
                      uint64_t *state, hipStream_t st)
{
    int rc = rle_check(world);
    if (rc) return rc;
    if (!d_voxels || !d_chunk_ids || !d_word_offsets || !ticket || !state) return VP_ERR_ARG;
    if (!d_words && capacity_words != 0) return VP_ERR_ARG;
    if (n == 0) return VP_OK;
    RleArgs a = {};
    a.voxels = const_cast<uint8_t *>(d_voxels);
    a.ids = d_chunk_ids;
    a.n = n;
    a.d_n = d_n;
    a.words = d_words;
    a.cap = capacity_words;
    a.offsets = d_word_offsets;
    a.uniform_out = d_uniform_out;
    a.uniform_in = d_uniform_in;
    a.status = ctx->d_status;
    a.single = 0;
    a.nchunks = (uint32_t)(1ull << (world->max_bitw[0] + world->max_bitw[1] + world->max_bitw[2]));
    a.ticket = ticket;
    a.state = state;
    const int resident = ctx->num_cus * 2;
    const int grid = (int)(n < (uint32_t)resident ? n : (uint32_t)resident);
    const int rgrid = (int)((n + 255u) / 256u);
    hipLaunchKernelGGL(k_rle_reset, dim3(rgrid < 1024 ? rgrid : 1024), dim3(256), 0, st, a.ticket,
                       a.state, n, a.offsets);
    VP_HIP_TRY(hipGetLastError());
    VP_HIP_TRY(rle_dispatch(world->root_bitw, VP_RLE_ENCODE, a, grid, st));
    return VP_OK;
}

}  // namespace vp

using namespace vp;

extern "C" int vp_gpu_rle(vp_ctx *ctx, int dir, const vp_world_desc *world,
                          uint8_t *d_voxels, const uint32_t *d_chunk_ids, uint32_t n,
                          uint32_t *d_words, uint64_t capacity_words,
                          uint64_t *d_word_offsets, int16_t *d_uniform_out, void *stream)
{
    if (!ctx || !world || !d_voxels || !d_chunk_ids || !d_word_offsets) return VP_ERR_ARG;
    if (dir != VP_RLE_ENCODE && dir != VP_RLE_DECODE) return VP_ERR_ARG;
    // d_words == NULL with capacity 0: an encode that only sizes the streams
    if (!d_words && (dir != VP_RLE_ENCODE || capacity_words != 0)) return VP_ERR_ARG;
    const uint32_t root_bitw = world->root_bitw;
    if (root_bitw < 2 || root_bitw > 6) return VP_ERR_UNSUPPORTED;
    if ((int)world->max_bitw[0] + world->max_bitw[1] + world->max_bitw[2] > 32) return VP_ERR_ARG;
    if (n == 0) return VP_OK;
    hipStream_t st = as_stream(stream);
    RleArgs a = {};
    a.voxels = d_voxels;
    a.ids = d_chunk_ids;
    a.n = n;
    a.words = d_words;
    a.cap = capacity_words;
    a.offsets = d_word_offsets;
    a.uniform_out = d_uniform_out;
    a.status = ctx->d_status;
    a.single = (n == 1) ? 1 : 0;
    a.parts = 1u;
    a.nchunks = (uint32_t)(1ull << (world->max_bitw[0] + world->max_bitw[1] + world->max_bitw[2]));
    int grid = 1;
    if (dir == VP_RLE_ENCODE) {
        std::lock_guard<std::mutex> g(ctx->mu);
        if (!a.single) {
            int rc = ensure_state(ctx, n);
            if (rc) return rc;
            a.ticket = ctx->d_ticket;
            a.state = ctx->d_state;
            const int resident = ctx->num_cus * 2;
            grid = (int)(n < (uint32_t)resident ? n : (uint32_t)resident);
            const int rgrid = (int)((n + 255u) / 256u);
            hipLaunchKernelGGL(k_rle_reset, dim3(rgrid < 1024 ? rgrid : 1024), dim3(256), 0, st,
                               a.ticket, a.state, n, a.offsets);
            VP_HIP_TRY(hipGetLastError());
        }
    } else {
        const uint32_t resident = (uint32_t)ctx->num_cus * 2u;
        // Few 64^3 chunks: up to eight workgroups repeat a chunk's scan and
        // share out its bytes, as many as fit at once (two chunks: 50 -> 26 us
        // by one workgroup each, 18 us by eight; smaller edges are done
        // within a launch's latency).
        while (root_bitw == 6 && a.parts < 8u && (uint64_t)n * a.parts * 2u <= resident) a.parts *= 2u;
        grid = (int)(n < resident ? n * a.parts : resident);
    }
    return rle_dispatch(root_bitw, dir, a, grid, st) == hipSuccess ? VP_OK : VP_ERR_HIP;
}
