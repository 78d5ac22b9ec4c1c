// lmhist.hip -- list-mode histogramming (lmhistogram_mp) on gfx950, and its C ABI
// (include/hrrt_lmhist.h).
//
// The reference walks each packet of PACKET_SIZE 64-bit words sequentially: a word pair is an
// event or a tag and advances the walk by two words, an out-of-sync word advances it by one
// (rebin_packet histogram_mp.cpp:1053-1060).  The walk is split here into 2048-word chunks,
// one wave each:
//   lm_summary_kernel  bitmasks of the out-of-sync words of each parity in the chunk, and from
//                      them the parity the walk leaves the chunk with, for either entry parity
//   lm_resolve_kernel  per packet, the entry parity of every chunk (the walk restarts at word 0
//                      of each packet)
//   lm_window_kernel   the frame's start and end time tags (first in walk order)
//   lm_hist_kernel     every word pair the walk visits inside the frame: tags into the
//                      statistics, events decoded and rebinned through the module-pair LUT with
//                      the reference's float operations; each binned event written as a key
//                      2*bin + delayed into its chunk's CHUNK/2 key slots, and each event's two
//                      crystals as 16-bit entries into the chunk's per-head segments
//   lm_count_kernel, lm_part_sums_kernel, lm_scatter_kernel  the keys into buckets of 2^20 bins
//   lm_tile_count_kernel, lm_tile_scatter_kernel  the buckets' keys into their tiles of 8192 bins,
//                      and the first key of every tile
//   lm_tile_kernel     per tile: its keys counted in LDS, then the tile's int16 bins (wrapping)
//                      and saturating uint8 delayed bins written in order
//   lm_coin_kernel     per head and range of chunks: the head's crystal entries counted in LDS
//   lm_coin_sum_kernel the ranges' counts summed into the coincidence maps
// No global atomics touch a sinogram bin or a crystal counter: scattered device-scope atomics
// into a 1.9 GB int32 count array and the 0.5 MB maps took 5.6 ms of a 6.8 ms call for 40 M
// events at span 3, against 1.9 ms for the whole call this way.
// Integer counts do not depend on the order of the events, so the result equals the
// reference's sequential histogram exactly.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "../../include/hrrt_lmhist.h"
#include "delays.h"
#include "kernels.h"

using namespace hrrt_dl;

namespace {

constexpr long long PACKET = HRRT_LM_PACKET_WORDS;
constexpr int CHUNK = 2048;                          // words per chunk, one wave
constexpr int TILE_BITS = 13, TILE = 1 << TILE_BITS;  // sinogram bins per histogram tile
constexpr int BUCKET_BITS = 20;                      // sinogram bins per bucket of the first partition
constexpr int BUCKET_TILES = 1 << (BUCKET_BITS - TILE_BITS);
constexpr int MAX_BUCKETS = 1 << (30 - BUCKET_BITS);  // the sinogram has at most 2^30 bins
constexpr int MAX_PARTS = 512;                       // workgroups of the first partition
constexpr int COIN_HEAD = 2 * NDOIS * NY * NX;        // coincidence counters of one head: [map][layer][ring][x]
constexpr int COIN_RANGES = 32;                       // chunk ranges of the coincidence-map pass
constexpr int CHUNKS_PER_PACKET = (int)(PACKET / CHUNK);
constexpr int WAVES = 4;                             // chunks per workgroup
constexpr int NBLOCKS = HRRT_LM_NBLOCKS;
constexpr unsigned long long NONE = ~0ull;

// statistics scratch (u64 words); each counter on its own 128-byte line, since every wave adds
// into all of them
constexpr int ST_LINE = 16;
enum { ST_PROMPTS = 0, ST_RANDOMS = ST_LINE, ST_EVENTS = 2 * ST_LINE, ST_TAGS = 3 * ST_LINE,
       ST_TIME_TAGS = 4 * ST_LINE, ST_REJECTED = 5 * ST_LINE, ST_TX = 6 * ST_LINE, ST_LAST_TIME = 7 * ST_LINE,
       ST_START = 8 * ST_LINE, ST_END = 9 * ST_LINE, ST_BLOCKS = 10 * ST_LINE };
constexpr int ST_WORDS = ST_BLOCKS + 3 * NBLOCKS;    // then block totals, sample counts, last (packed)

// EWTYPES geometry_info.h:75 packed 2 bits per entry: 0 prompt, 1 delayed, 2 tag, 3 out of sync
constexpr unsigned ewtypes_packed() {
    constexpr int t[16] = {3, 3, 1, 0, 3, 3, 2, 2, 3, 3, 3, 3, 3, 3, 3, 3};
    unsigned v = 0;
    for (int i = 0; i < 16; i++) v |= (unsigned)t[i] << (2 * i);
    return v;
}
constexpr unsigned EWT = ewtypes_packed();

// HRRT_MPAIRS geometry_info.h:68-73, packed 3 bits per module pair (A heads, B heads)
constexpr int MPAIRS[NMP + 1][2] = {{-1, -1}, {0, 2}, {0, 3}, {0, 4}, {0, 5}, {0, 6}, {1, 3}, {1, 4},
                                    {1, 5},   {1, 6}, {1, 7}, {2, 4}, {2, 5}, {2, 6}, {2, 7}, {3, 5},
                                    {3, 6},   {3, 7}, {4, 6}, {4, 7}, {5, 7}};
constexpr unsigned long long mp_pack(int side) {
    unsigned long long v = 0;
    for (int m = 0; m <= NMP; m++) v |= (unsigned long long)(MPAIRS[m][side] & 7) << (3 * m);
    return v;
}
constexpr unsigned long long MP_A = mp_pack(0), MP_B = mp_pack(1);

__device__ inline int word_type(unsigned ew1, unsigned ew2) {
    const unsigned idx = ((ew2 & 0xc0000000u) >> 30) | ((ew1 & 0xc0000000u) >> 28);
    return (int)((EWT >> (2 * idx)) & 3u);
}

struct LmArgs {
    const unsigned *w;
    long long nwords;
    int mode, start_ms, end_ms, ignore_border, doi;
    const int3 *sol;        // [21][144][144] {nsino, bits(d), bits(z)}
    const float2 *z;        // [104] {ring z, ring z in planes + 0.5}
    const int2 *seg;        // [128] by 2*(int)seg + (seg < 0) + 64: {first | last << 16, offset}
    int nsino;
    long long S;            // nplanes * nsino
    unsigned *keys;         // [nchunks][CHUNK/2] binned events 2*bin + (delayed)
    unsigned *kcnt;         // [nchunks] keys of each chunk
    unsigned *coin_p, *coin_d;
    unsigned short *cseg;   // [nchunks][NHEADS][CHUNK/2] crystal entries (index in COIN_HEAD) by head
    unsigned *ccnt;         // [nchunks][NHEADS] entries per chunk and head
    unsigned *chunks;       // per chunk: exit parity for entry 0 (bit 0) and 1 (bit 1), entry parity (bit 2)
    unsigned *cmask;        // [nchunks][64] out-of-sync masks of each chunk (chunk_mask_word)
    bool w16;               // the stream is 16-byte aligned
    unsigned long long *st;
};

__device__ inline long long packet_end(long long q, long long nwords) {
    const long long pe = (q / PACKET + 1) * PACKET;
    return pe < nwords ? pe : nwords;
}

// bits 0..15 of x -> bits 0, 2, 4, ..., 30
__device__ inline unsigned spread16(unsigned x) {
    x &= 0xffffu;
    x = (x | (x << 8)) & 0x00ff00ffu;
    x = (x | (x << 4)) & 0x0f0f0f0fu;
    x = (x | (x << 2)) & 0x33333333u;
    x = (x | (x << 1)) & 0x55555555u;
    return x;
}

// Mask word `lane` of chunk cs (a multiple of CHUNK): mask[parity * 32 + i] bit j says word
// cs + 2*(32 i + j) + parity is out of sync and inside its packet's walk (it has a successor
// in the packet).  One wave; each lane reads four consecutive words per 256-word block (one
// 16-byte load when the stream is 16-byte aligned), the fifth from its neighbour.
__device__ unsigned chunk_mask_word(const unsigned *__restrict__ w, long long cs, long long nwords, bool w16, int lane) {
    const long long pend = packet_end(cs, nwords);
    const int par = lane >> 5, mi = lane & 3, kk = (lane & 31) >> 2;
    constexpr int BLOCKS = CHUNK / 256;
    uint4 v[BLOCKS];
    if (w16 && cs + CHUNK <= nwords) {     // every load in flight before the first is used
#pragma unroll
        for (int k = 0; k < BLOCKS; k++) v[k] = *reinterpret_cast<const uint4 *>(w + cs + 256 * k + 4 * lane);
    } else {
#pragma unroll
        for (int k = 0; k < BLOCKS; k++) {
            const long long q = cs + 256 * k + 4 * lane;
            v[k].x = q < nwords ? w[q] : 0u;
            v[k].y = q + 1 < nwords ? w[q + 1] : 0u;
            v[k].z = q + 2 < nwords ? w[q + 2] : 0u;
            v[k].w = q + 3 < nwords ? w[q + 3] : 0u;
        }
    }
    const unsigned tail = cs + CHUNK < pend ? w[cs + CHUNK] : 0u;
    const int last = (int)min(pend - cs, (long long)CHUNK + 1) - 1;    // positions below it have a successor
    unsigned long long lo = 0, hi = 0;
#pragma unroll
    for (int k = 0; k < BLOCKS; k++) {
        const unsigned block_next = k + 1 < BLOCKS ? (unsigned)__builtin_amdgcn_readfirstlane((int)v[(k + 1) % BLOCKS].x) : tail;
        unsigned next = __shfl_down(v[k].x, 1);
        if (lane == 63) next = block_next;
        const unsigned u[5] = {v[k].x, v[k].y, v[k].z, v[k].w, next};
        unsigned long long b[4];
#pragma unroll
        for (int j = 0; j < 4; j++) b[j] = __ballot(256 * k + 4 * lane + j < last && word_type(u[j], u[j + 1]) == 3);
        // relative position 256 k + 4 l + j: parity j & 1, bit 2 (l mod 16) + (j >> 1) of mask word 4 k + l / 16
        if (kk == k) lo = par ? b[1] : b[0], hi = par ? b[3] : b[2];
    }
    const unsigned mine = spread16((unsigned)(lo >> (16 * mi))) | (spread16((unsigned)(hi >> (16 * mi))) << 1);
    return mine;
}

// The walk through one chunk from relative position `entry` (0 or 1), by one wave: lane l holds mask
// word l (chunk_mask_word).  The relative positions of the out-of-sync words it steps on go to sw
// (may be null), their number to nsw; returns the parity it leaves with.  All of it is scalar: a
// ballot says which mask words hold any, so a chunk without them costs a few instructions (one
// lane searching the 32 words of its parity in LDS took 40 us of a 40 M word stream's 80).
// RUNS: the chunk has 64 out-of-sync words in a row from a multiple of 64 (a stream's zero tail), which are
// taken at once (8 M zero words: 0.38 ms, 1.51 one by one).
template <bool RUNS>
__device__ __forceinline__ int chunk_steps(unsigned mask, unsigned runs, int entry, unsigned short *sw, int &nsw, int lane) {
    const unsigned long long some = __ballot(mask != 0);
    int p = entry;
    nsw = 0;
    while (p < CHUNK) {
        if (RUNS && (p & 63) == 0 && (runs >> (p >> 6)) & 1) {
            if (sw) sw[nsw + lane] = (unsigned short)(p + lane);
            nsw += 64;
            p += 64;
            continue;
        }
        const int par = p & 1, k = p >> 1;
        int wi = k >> 5;
        unsigned m = (unsigned)__builtin_amdgcn_readlane((int)mask, par * 32 + wi) & (~0u << (k & 31));
        if (!m) {
            const unsigned later = (unsigned)(some >> (32 * par)) & (unsigned)(~1ull << wi);
            if (!later) break;
            wi = __builtin_ctz(later);
            m = (unsigned)__builtin_amdgcn_readlane((int)mask, par * 32 + wi);
        }
        const int pos = 2 * ((wi << 5) + __builtin_ctz(m)) + par;
        if (sw && lane == 0) sw[nsw] = (unsigned short)pos;
        nsw++;
        p = pos + 1;
    }
    return p & 1;
}
__device__ int chunk_walk(unsigned mask, int entry, unsigned short *sw, int &nsw, int lane) {
    const unsigned long long full = __ballot(mask == ~0u);
    const unsigned runs = (unsigned)full & (unsigned)(full >> 32);      // bit w: words 64 w .. 64 w + 63
    return runs ? chunk_steps<true>(mask, runs, entry, sw, nsw, lane) : chunk_steps<false>(mask, 0u, entry, sw, nsw, lane);
}

// Also clears the statistics (workgroup 0), which only later kernels of the call add to.
__global__ __launch_bounds__(WAVES * 64) void lm_summary_kernel(LmArgs a, long long nchunks) {
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < ST_WORDS; i += WAVES * 64) a.st[i] = (i == ST_START || i == ST_END) ? NONE : 0ull;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long c = (long long)blockIdx.x * WAVES + wv;
    if (c >= nchunks) return;
    const unsigned m = chunk_mask_word(a.w, c * CHUNK, a.nwords, a.w16, lane);
    a.cmask[c * 64 + lane] = m;
    int n;
    const int e0 = chunk_walk(m, 0, nullptr, n, lane), e1 = chunk_walk(m, 1, nullptr, n, lane);
    if (lane == 0) a.chunks[c] = (unsigned)(e0 | (e1 << 1));
}

// One workgroup per packet (the walk enters the packet's first chunk at word 0).  A chunk maps its
// entry parity to its exit parity: to a constant, to itself or to the other.  The entry of a chunk
// follows from the last constant before it and the number of exchanges since, so ballots give it
// for a wave of chunks at once, and the waves' own maps chain the 16 of them (a single thread
// walking the 1024 summaries took 27 us).
__global__ __launch_bounds__(CHUNKS_PER_PACKET) void lm_resolve_kernel(unsigned *chunks, long long nchunks) {
    __shared__ unsigned wave_map[CHUNKS_PER_PACKET / 64];   // exit parity for entry 0 (bit 0) and 1 (bit 1)
    const long long c = (long long)blockIdx.x * CHUNKS_PER_PACKET + threadIdx.x;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const unsigned v = c < nchunks ? chunks[c] & 3u : 2u;   // past the end: the identity
    const unsigned long long constant = __ballot(v == 0u || v == 3u), value = __ballot(v & 1u), flip = __ballot(v == 1u);
    // the parity entering position n of the wave for an entry parity of `in`
    auto entering = [&](int n, unsigned in) {
        const unsigned long long below = n < 64 ? (1ull << n) - 1 : ~0ull, cb = constant & below;
        if (!cb) return (in ^ (unsigned)__popcll(flip & below)) & 1u;
        const int j = 63 - __clzll((long long)cb);
        return ((unsigned)(value >> j) ^ (unsigned)__popcll(flip & below & (~1ull << j))) & 1u;
    };
    if (lane == 0) wave_map[wv] = entering(64, 0) | (entering(64, 1) << 1);
    __syncthreads();
    unsigned in = 0;
    for (int w = 0; w < wv; w++) in = (wave_map[w] >> in) & 1u;
    if (c < nchunks) chunks[c] = v | (entering(lane, in) << 2);
}

// Per wave: the switch list of the walk through chunk c; returns the entry parity.
__device__ int chunk_visit_setup(const LmArgs &a, long long c, unsigned short *sw, int &nsw, int lane) {
    const int entry = __builtin_amdgcn_readfirstlane((int)((a.chunks[c] >> 2) & 1u));
    chunk_walk(a.cmask[c * 64 + lane], entry, sw, nsw, lane);
    __builtin_amdgcn_wave_barrier();
    return entry;
}

// Does the walk start a word pair at relative position r?
__device__ inline bool visited(int r, int entry, const unsigned short *sw, int nsw) {
    int lo = 0, hi = nsw;                  // switches before r
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (sw[mid] < r) lo = mid + 1;
        else hi = mid;
    }
    const int start = lo == 0 ? entry : sw[lo - 1] + 1;
    if (lo < nsw && sw[lo] == r) return false;   // an out-of-sync word the walk steps on
    return r >= start && ((r - start) & 1) == 0;
}

template <int PASS>
__global__ __launch_bounds__(WAVES * 64) void lm_window_kernel(LmArgs a, long long nchunks) {
    __shared__ unsigned short sws[WAVES][CHUNK];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long c = (long long)blockIdx.x * WAVES + wv;
    if (c >= nchunks) return;
    // pass 1 looks for the end tag from the start tag on (the start tag itself may end the frame)
    long long from = 0;
    if (PASS == 1 && a.start_ms > 0) {
        if (a.st[ST_START] == NONE) return;
        from = (long long)a.st[ST_START];
    }
    int nsw;
    const int entry = chunk_visit_setup(a, c, sws[wv], nsw, lane);
    const long long cs = c * CHUNK, pend = packet_end(cs, a.nwords);
    const int bound = PASS == 0 ? a.start_ms : a.end_ms;
    for (int i = 0; i < CHUNK / 64; i++) {
        const int r = i * 64 + lane;
        const long long q = cs + r;
        if (q + 1 >= pend || q < from) continue;
        if (!visited(r, entry, sws[wv], nsw)) continue;
        const unsigned ew1 = a.w[q], ew2 = a.w[q + 1];
        if (word_type(ew1, ew2) != 2) continue;
        const unsigned tag = (ew1 & 0xffffu) | ((ew2 & 0xffffu) << 16);
        if ((tag & 0xE0000000u) != 0x80000000u) continue;
        if ((int)(tag & 0x3fffffffu) >= bound) atomicMin(&a.st[PASS == 0 ? ST_START : ST_END], (unsigned long long)q);
    }
}

// Event fields (rebin_packet histogram_mp.cpp:1111-1227) of a word pair; a pair of zeros is out of
// sync, neither event nor tag.
struct Event {
    int type, mpe, ax, ay, bx, by, doia, doib;
    bool is_event, bad, tx, em, binnable;
};
__device__ inline Event decode(const LmArgs &a, unsigned ew1, unsigned ew2) {
    Event v;
    v.type = word_type(ew1, ew2);
    v.is_event = v.type < 2;
    v.mpe = (int)(((ew1 & 0x00070000u) >> 16) | ((ew2 & 0x00070000u) >> 13));
    v.ax = (int)(ew1 & 0xff), v.ay = (int)((ew1 & 0xff00) >> 8);
    v.bx = (int)(ew2 & 0xff), v.by = (int)((ew2 & 0xff00) >> 8);
    v.doia = a.doi ? (int)((ew1 & 0x01C00000u) >> 22) : 1;
    v.doib = a.doi ? (int)((ew2 & 0x01C00000u) >> 22) : 1;
    const int outside = (int)((unsigned)(v.mpe - 1) >= (unsigned)NMP) | (int)(max(v.ax, v.bx) >= NX) | (int)(max(v.ay, v.by) >= NY);
    v.bad = v.is_event & (outside != 0);
    const bool ok = v.is_event & !v.bad;
    v.tx = ok & ((v.doia == 7) | (v.doib == 7));
    v.em = ok & !v.tx & (max(v.doia, v.doib) <= 1);
    const int xhigh = NX - 1;
    v.binnable = v.em & !(a.ignore_border & ((v.ax * v.bx == 0) | (v.ax == xhigh) | (v.bx == xhigh))) &
                 !((a.mode == 2) & (v.type != 0));
    return v;
}

__device__ inline unsigned lanes_below(unsigned long long mask, unsigned base) {
    return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, base));
}

// p by a 32-bit byte offset: a uniform base and an offset register, no 64-bit address per lane
template <typename T>
__device__ inline T *at_byte(T *p, unsigned off) {
    return (T *)((char *)p + off);
}

// two words at any word address
struct __attribute__((packed, aligned(4))) WordPair {
    unsigned x, y;
};

// One wave per chunk.  The walk visits one position of each aligned word pair (2k, 2k + 1): the
// one of its parity, entry parity flipped by every out-of-sync word before 2k; an out-of-sync word
// is visited but not decoded, and when it is the pair's even word the walk goes on to the odd one.
// Each lane takes a pair per row of 64; rows go in groups of G.  What bounds the kernel is vector
// instructions and the latency of its gathers, so every load is unconditional: the words of the next
// group and the LUT records of this one are in flight together (a record of an undecoded pair is
// record 0, module pair 0, which has no bin), a chunk that the walk passes in step inside the frame
// needs no position tests, and what is counted is counted in scalar registers from ballots.
template <bool COIN>
__global__ __launch_bounds__(WAVES * 64, 6) void lm_hist_kernel(LmArgs a, long long nchunks) {
    __shared__ unsigned short sws[WAVES][CHUNK];
    __shared__ float2 zs[256];                  // by the ring byte
    __shared__ int2 segs[128];
    __shared__ unsigned heads[64];              // by module pair: A head's bit, B head's bit << 8
    __shared__ unsigned counts[7];
    const int tid = threadIdx.x;
    for (int j = tid; j < 256; j += WAVES * 64) zs[j] = j < NY ? a.z[j] : make_float2(0.0f, 0.0f);
    for (int j = tid; j < 128; j += WAVES * 64) segs[j] = a.seg[j];
    if (tid < 64) heads[tid] = tid >= 1 && tid <= NMP ? (1u << ((MP_A >> (3 * tid)) & 7)) | (256u << ((MP_B >> (3 * tid)) & 7)) : 0u;
    if (tid < 7) counts[tid] = 0;
    __syncthreads();
    const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const long long c = (long long)blockIdx.x * WAVES + wv;
    // the frame: from its start tag (or word 0) through its end tag (or the last word)
    const unsigned long long s0 = a.st[ST_START], s1 = a.st[ST_END];
    const long long lo = a.start_ms > 0 ? (long long)s0 : 0;
    const long long hi = (a.end_ms > 0 && s1 != NONE) ? (long long)s1 + 1 : a.nwords;
    const long long cs = c * CHUNK, pend = packet_end(cs, a.nwords);
    // a chunk holds at most CHUNK/2 events (the walk steps two words past an event)
    unsigned *keys = a.keys + c * (CHUNK / 2);
    unsigned n_tags = 0, n_time = 0, n_events = 0, n_rej = 0, n_tx = 0, n_prompts = 0, n_randoms = 0;
    unsigned nk = 0;   // keys of the chunk so far
    unsigned cc[NHEADS];   // crystal entries per head so far
#pragma unroll
    for (int h = 0; h < NHEADS; h++) cc[h] = 0;
    unsigned long long last_time = 0;
    if (c < nchunks && cs + 1 < a.nwords && !(a.start_ms > 0 && s0 == NONE) && cs + CHUNK > lo && cs < hi) {
        unsigned short *cseg = COIN ? a.cseg + c * (NHEADS * (CHUNK / 2)) : nullptr;
        const unsigned short *sw = sws[wv];
        int nsw;
        const int entry = chunk_visit_setup(a, c, sws[wv], nsw, lane);
        const bool in_step = entry == 0 && nsw == 0 && cs + CHUNK <= a.nwords && cs >= lo && cs + CHUNK <= hi;
        constexpr int G = 4, ROWS = CHUNK / 128;
        static_assert(ROWS % G == 0, "whole groups");
        unsigned x[G], y[G], xn[G], yn[G];
        const int last = (int)min(a.nwords - 2 - cs, (long long)CHUNK - 2);   // the chunk's last word pair in the stream
        auto load_words = [&](int r0) __attribute__((always_inline)) {
#pragma unroll
            for (int g = 0; g < G; g++) {
                const WordPair v = *reinterpret_cast<const WordPair *>(a.w + cs + min(128 * (r0 + g) + 2 * lane, last));
                xn[g] = v.x, yn[g] = v.y;
            }
        };
        load_words(0);
        for (int r0 = 0; r0 < ROWS; r0 += G) {
            int odd[G];      // the position taken is 2k + odd
            int3 e[G];
#pragma unroll
            for (int g = 0; g < G; g++) x[g] = xn[g], y[g] = yn[g], odd[g] = 0;
            // x, y become the pair of words at the position visited, zeros where there is none
            if (!in_step) {
                const long long qa = cs + 128 * (r0 + G);
                const unsigned after = qa < a.nwords ? a.w[qa] : 0u;    // the word after the group
#pragma unroll
                for (int g = 0; g < G; g++) {       // words past the stream's end are zeros
                    const int r = 128 * (r0 + g) + 2 * lane;
                    x[g] = r <= last ? x[g] : (r == last + 1 ? y[g] : 0u);
                    y[g] = r <= last ? y[g] : 0u;
                }
#pragma unroll
                for (int g = 0; g < G; g++) {
                    const int p0 = 2 * ((r0 + g) * 64 + lane);
                    int n = 0, m = nsw;   // out-of-sync words visited before p0
                    while (n < m) {
                        const int mid = (n + m) >> 1;
                        if (sw[mid] < p0) n = mid + 1;
                        else m = mid;
                    }
                    const int par = (entry + n) & 1;
                    int p = p0 + par;
                    if (n < nsw && sw[n] == p) p = (par == 0 && !(n + 1 < nsw && sw[n + 1] == p0 + 1)) ? p0 + 1 : -1;
                    const long long q = cs + p;
                    const bool live = p >= 0 && q + 1 < pend && q >= lo && q < hi;
                    unsigned next = __shfl_down(x[g], 1);
                    const unsigned row_next = g + 1 < G ? (unsigned)__builtin_amdgcn_readfirstlane((int)x[(g + 1) % G]) : after;
                    if (lane == 63) next = row_next;
                    odd[g] = p & 1;
                    const unsigned w1 = odd[g] ? y[g] : x[g], w2 = odd[g] ? next : y[g];
                    x[g] = live ? w1 : 0u, y[g] = live ? w2 : 0u;
                }
            }
#pragma unroll
            for (int g = 0; g < G; g++) {
                const Event v = decode(a, x[g], y[g]);
                const unsigned i = (unsigned)(((v.mpe * NXD) + v.ax + NX * v.doia) * NXD + v.bx + NX * v.doib);
                e[g] = *at_byte(a.sol, v.binnable ? i * 12u : 0u);
            }
            // the fields are decoded again below: held across the gathers they would cost the occupancy
#pragma unroll
            for (int g = 0; g < G; g++) asm volatile("" : "+v"(x[g]), "+v"(y[g]));
            load_words(min(r0 + G, ROWS - G));      // always a group, or the gathers would wait for it
#pragma unroll
            for (int g = 0; g < G; g++) {
                const Event v = decode(a, x[g], y[g]);
                // tags (process_tagword histogram_mp.cpp:225-295)
                const bool is_tag = v.type == 2;
                const unsigned long long tags = __ballot(is_tag);
                if (tags) {
                    const long long q = cs + 2 * ((r0 + g) * 64 + lane) + odd[g];
                    const unsigned tag = (x[g] & 0xffffu) | ((y[g] & 0xffffu) << 16);
                    const bool time_tag = is_tag && (tag & 0xE0000000u) == 0x80000000u;
                    n_tags += (unsigned)__popcll(tags);
                    n_time += (unsigned)__popcll(__ballot(time_tag));
                    if (time_tag) last_time = ((unsigned long long)q << 30) | (tag & 0x3fffffffu);   // q grows along the lane
                    if (is_tag && (tag & 0xE0000000u) == 0xA0000000u) {
                        const int block = (int)((tag & 0x1ff80000u) >> 19);
                        const unsigned val = tag & 0x0007ffffu;
                        if (block < NBLOCKS) {
                            atomicAdd(&a.st[ST_BLOCKS + block], (unsigned long long)val);
                            atomicAdd(&a.st[ST_BLOCKS + NBLOCKS + block], 1ull);
                            atomicMax(&a.st[ST_BLOCKS + 2 * NBLOCKS + block], ((unsigned long long)q << 19) | val);
                        }
                    }
                }
                n_events += (unsigned)__popcll(__ballot(v.is_event));
                n_rej += (unsigned)__popcll(__ballot(v.bad));
                n_tx += (unsigned)__popcll(__ballot(v.tx));
                // rebin_event LM_Rebinner_mp.cpp:188-219
                const float sd = __int_as_float(e[g].y), sz = __int_as_float(e[g].z);
                const float2 za = zs[v.ay];
                const float dz = zs[v.by].x - za.x;
                const int plane = (int)(za.y + sz * dz);
                const float sg = 0.5f + dz * sd;
                const int si = (int)sg;
                const int2 ent = segs[64 + min(max(2 * si + (sg < 0.0f ? 1 : 0), -64), 63)];
                const bool has = v.binnable & (e[g].x >= 0) & (plane >= (ent.x & 0xffff)) & (plane <= (ent.x >> 16));
                // trues mode counts prompt - delayed, mode 1 the two apart, mode 2 prompts only (the
                // delayed events have no bin there): every mode keeps the delayed flag in bit 0
                const unsigned key = 2u * ((unsigned)(plane + ent.y) * (unsigned)a.nsino + (unsigned)e[g].x) + (unsigned)v.type;
                const unsigned long long bal = __ballot(has), del = __ballot(has & (v.type != 0));
                n_randoms += (unsigned)__popcll(del);
                n_prompts += (unsigned)__popcll(bal & ~del);
                if (has) *at_byte(keys, 4u * lanes_below(bal, nk)) = key;
                nk += (unsigned)__popcll(bal);
                // coincidence maps (histogram_mp.cpp:1218-1222, ring stride of histogram_mp_fromarchive.cpp:1092):
                // the event's two crystals, each an entry [map][layer][ring][x] in its head's segment of the
                // chunk (the two heads of a module pair differ)
                if (COIN) {
                    const bool counted = v.em & (v.type == 0 ? a.coin_p != nullptr : a.coin_d != nullptr);
                    const unsigned hb = counted ? heads[v.mpe] : 0u;
                    const int mo = v.type == 0 ? 0 : NDOIS * NY * NX;
                    const unsigned ka = (unsigned)(mo + (v.doia * NY + v.ay) * NX + v.ax);
                    const unsigned kb = (unsigned)(mo + (v.doib * NY + v.by) * NX + v.bx);
#pragma unroll
                    for (int h = 0; h < NHEADS; h++) {
                        const bool on = (hb & (0x101u << h)) != 0;
                        const unsigned long long bh = __ballot(on);
                        if (on) *at_byte(cseg, 2u * lanes_below(bh, h * (CHUNK / 2) + cc[h])) = (unsigned short)((hb >> h) & 1 ? ka : kb);
                        cc[h] += (unsigned)__popcll(bh);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);   // rows interleaved would hold their masks in spilled scalars
            }
        }
    }
    if (c < nchunks) {
        if (lane == 0) a.kcnt[c] = nk;
        if (COIN) {
            unsigned n = 0;
#pragma unroll
            for (int h = 0; h < NHEADS; h++) n = lane == h ? cc[h] : n;
            if (lane < NHEADS) a.ccnt[c * NHEADS + lane] = n;
        }
        // the counters of the workgroup's waves, then one add per counter to the statistics
        const unsigned mine = lane == 0 ? n_prompts : lane == 1 ? n_randoms : lane == 2 ? n_events : lane == 3 ? n_tags :
                              lane == 4 ? n_time : lane == 5 ? n_rej : n_tx;
        if (lane < 7 && mine) atomicAdd(&counts[lane], mine);
        if (__ballot(last_time != 0)) {
            for (int o = 32; o > 0; o >>= 1) {
                const unsigned long long other = __shfl_xor(last_time, o);
                last_time = other > last_time ? other : last_time;
            }
            if (lane == 0) atomicMax(&a.st[ST_LAST_TIME], last_time);
        }
    }
    __syncthreads();
    if (tid < 7 && counts[tid]) atomicAdd(&a.st[ST_LINE * tid], (unsigned long long)counts[tid]);
}
static_assert(ST_PROMPTS == 0 && ST_RANDOMS == ST_LINE && ST_EVENTS == 2 * ST_LINE && ST_TAGS == 3 * ST_LINE &&
              ST_TIME_TAGS == 4 * ST_LINE && ST_REJECTED == 5 * ST_LINE && ST_TX == 6 * ST_LINE, "order of the counters");

// ---- the keys by tile.  The order within a tile does not matter (a tile counts its keys), so two
// counting partitions do it: first into buckets of 2^BUCKET_BITS bins, by up to 512 workgroups with a
// range of chunks each, then slices of the buckets into tiles.  Stores of single keys to their places
// would bound both (each is a request of its own: 67 us for the first at 20 M keys, 44 this way), so a
// batch of keys is put in order in LDS first and its runs are stored whole.
// 20 M keys, span 3: 136 us in five launches (a library radix sort of the tile bits: 280 us in nine).
constexpr int PART_THREADS = 1024;
constexpr int CHUNK_KEYS = CHUNK / 2 / 64;   // key slots of a chunk per lane

// the chunk's key slots, 16 bytes a lane: v[u] is slot chunk_slot(u)
__device__ inline void load_chunk(const unsigned *__restrict__ keys, long long c, unsigned (&v)[CHUNK_KEYS]) {
    const uint4 *src = reinterpret_cast<const uint4 *>(keys + c * (CHUNK / 2)) + (threadIdx.x & 63);
#pragma unroll
    for (int i = 0; i < CHUNK_KEYS / 4; i++) {
        const uint4 x = src[64 * i];
        v[4 * i] = x.x, v[4 * i + 1] = x.y, v[4 * i + 2] = x.z, v[4 * i + 3] = x.w;
    }
}
__device__ inline unsigned chunk_slot(int u) { return 256 * (u >> 2) + 4 * (threadIdx.x & 63) + (u & 3); }

// Exclusive sums of v[0 .. PART_THREADS) over the workgroup, one element per thread; total gets the sum.
__device__ inline unsigned block_exclusive(unsigned v, unsigned *wave_sum, unsigned &total) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    unsigned inc = v;
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned up = __shfl_up(inc, o);
        if (lane >= o) inc += up;
    }
    if (lane == 63) wave_sum[wv] = inc;
    __syncthreads();
    unsigned before = 0;
    total = 0;
    for (int w = 0; w < PART_THREADS / 64; w++) {
        before += w < wv ? wave_sum[w] : 0u;
        total += wave_sum[w];
    }
    return before + inc - v;
}

// Up to U keys per thread (those with ok) into their digits' places in out: next[d] is the index of the
// next key of digit d, advanced by the workgroup's keys of it; reserve(n), called once by the thread of
// each digit with the number of its keys, gives how many others have put there.  The keys go
// through buf in the order of their digits.  Ends with a barrier.
template <int U, typename Digit, typename Reserve>
__device__ inline void partition_batch(const unsigned (&v)[U], const bool (&ok)[U], Digit digit, unsigned *next,
                                       unsigned *cnt, unsigned *buf, unsigned *wave_sum, unsigned *__restrict__ out,
                                       Reserve reserve) {
    const int tid = threadIdx.x;
    cnt[tid] = 0;
    __syncthreads();
    unsigned rank[U];
#pragma unroll
    for (int u = 0; u < U; u++)
        if (ok[u]) rank[u] = atomicAdd(&cnt[digit(v[u])], 1u);
    __syncthreads();
    unsigned total;
    const unsigned n = cnt[tid], before = block_exclusive(n, wave_sum, total), others = reserve(n);
    cnt[tid] = before;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; u++)
        if (ok[u]) buf[cnt[digit(v[u])] + rank[u]] = v[u];
    __syncthreads();
    const unsigned place = next[tid];
    next[tid] = place + n;
    cnt[tid] = place + others - before;
    __syncthreads();
    for (unsigned i = tid; i < total; i += PART_THREADS) {
        const unsigned k = buf[i];
        out[cnt[digit(k)] + i] = k;
    }
    __syncthreads();
}

// counts[b * parts + part]: keys of bucket b in the part's chunks
__global__ __launch_bounds__(PART_THREADS) void lm_count_kernel(const unsigned *__restrict__ keys,
                                                                const unsigned *__restrict__ kcnt, long long nchunks,
                                                                int nbuckets, unsigned *__restrict__ counts) {
    __shared__ unsigned cnt[PART_THREADS];
    cnt[threadIdx.x] = 0;
    __syncthreads();
    const long long per = (nchunks + gridDim.x - 1) / gridDim.x, c0 = blockIdx.x * per, c1 = min(nchunks, c0 + per);
    for (long long c = c0 + (threadIdx.x >> 6); c < c1; c += PART_THREADS / 64) {
        unsigned v[CHUNK_KEYS];
        load_chunk(keys, c, v);
        const unsigned n = kcnt[c];
#pragma unroll
        for (int u = 0; u < CHUNK_KEYS; u++)
            if (chunk_slot(u) < n) atomicAdd(&cnt[v[u] >> (BUCKET_BITS + 1)], 1u);
    }
    __syncthreads();
    if ((int)threadIdx.x < nbuckets) counts[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = cnt[threadIdx.x];
}
static_assert(MAX_BUCKETS <= PART_THREADS && BUCKET_TILES <= PART_THREADS, "a thread per digit");

// one wave per bucket: the parts' counts into their exclusive sums, the bucket's total, and its tiles'
// counters cleared
__global__ __launch_bounds__(64) void lm_part_sums_kernel(unsigned *__restrict__ counts, int parts,
                                                          unsigned *__restrict__ totals, unsigned *__restrict__ tcount,
                                                          unsigned *__restrict__ used) {
    unsigned *row = counts + (size_t)blockIdx.x * parts;
    const int lane = threadIdx.x;
    for (int t = lane; t < BUCKET_TILES; t += 64) tcount[blockIdx.x * BUCKET_TILES + t] = used[blockIdx.x * BUCKET_TILES + t] = 0;
    unsigned sum = 0;
    for (int p0 = 0; p0 < parts; p0 += 64) {
        const unsigned v = p0 + lane < parts ? row[p0 + lane] : 0u;
        unsigned inc = v;
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned up = __shfl_up(inc, o);
            if (lane >= o) inc += up;
        }
        if (p0 + lane < parts) row[p0 + lane] = sum + inc - v;
        sum += __shfl(inc, 63);
    }
    if (lane == 0) totals[blockIdx.x] = sum;
}

__global__ __launch_bounds__(PART_THREADS) void lm_scatter_kernel(const unsigned *__restrict__ keys,
                                                                  const unsigned *__restrict__ kcnt, long long nchunks,
                                                                  int nbuckets, const unsigned *__restrict__ counts,
                                                                  const unsigned *__restrict__ totals,
                                                                  unsigned *__restrict__ out) {
    __shared__ unsigned next[PART_THREADS], cnt[PART_THREADS], wave_sum[PART_THREADS / 64], buf[CHUNK_KEYS * PART_THREADS];
    const int b = threadIdx.x;
    unsigned total;
    const unsigned base = block_exclusive(b < nbuckets ? totals[b] : 0u, wave_sum, total);
    next[b] = base + (b < nbuckets ? counts[(size_t)b * gridDim.x + blockIdx.x] : 0u);
    const long long per = (nchunks + gridDim.x - 1) / gridDim.x, c0 = blockIdx.x * per, c1 = min(nchunks, c0 + per);
    for (long long cb = c0; cb < c1; cb += PART_THREADS / 64) {      // a chunk per wave
        const long long c = cb + (threadIdx.x >> 6);
        unsigned v[CHUNK_KEYS];
        bool ok[CHUNK_KEYS];
        load_chunk(keys, min(c, c1 - 1), v);
        const unsigned n = c < c1 ? kcnt[c] : 0u;
#pragma unroll
        for (int u = 0; u < CHUNK_KEYS; u++) ok[u] = chunk_slot(u) < n;
        partition_batch(v, ok, [](unsigned k) { return k >> (BUCKET_BITS + 1); }, next, cnt, buf, wave_sum, out,
                        [](unsigned) { return 0u; });
    }
}

// A workgroup of the second partition takes a slice of up to SLICE keys of one bucket: a bucket has as
// many slices as its keys need and at least one (planes at a segment's ends can hold ten times the mean:
// with a workgroup per bucket the fullest one took 190 of 190 us).
constexpr int SLICE_KEYS = 8, SLICE = SLICE_KEYS * PART_THREADS;
struct Slice {
    unsigned bucket, start, k0, k1;     // the bucket, its first key, the slice's keys
    int first;                          // the bucket's first slice
};
__device__ inline bool find_slice(const unsigned *__restrict__ totals, int nbuckets, unsigned item, unsigned (*wave_sum)[PART_THREADS / 64],
                                  Slice *found) {
    const unsigned tid = threadIdx.x, n = (int)tid < nbuckets ? totals[tid] : 0u;
    const unsigned slices = (int)tid < nbuckets ? max(1u, (n + SLICE - 1) / SLICE) : 0u;
    unsigned keys, all;
    const unsigned start = block_exclusive(n, wave_sum[0], keys), s0 = block_exclusive(slices, wave_sum[1], all);
    if (item >= s0 && item < s0 + slices) {
        const unsigned k0 = start + (item - s0) * SLICE;
        *found = Slice{tid, start, k0, min(start + n, k0 + SLICE), item == s0};
    }
    __syncthreads();
    return item < all;
}
__device__ inline unsigned tile_of(unsigned k) { return (k >> (TILE_BITS + 1)) & (BUCKET_TILES - 1); }
__device__ inline void load_slice(const unsigned *__restrict__ keys, const Slice &sl, unsigned (&v)[SLICE_KEYS], bool (&ok)[SLICE_KEYS]) {
#pragma unroll
    for (int u = 0; u < SLICE_KEYS; u++) {
        const unsigned i = sl.k0 + u * PART_THREADS + threadIdx.x;
        ok[u] = i < sl.k1;
        v[u] = ok[u] ? keys[i] : 0u;
    }
}

// tcount[t]: keys of tile t, added up over the slices
__global__ __launch_bounds__(PART_THREADS) void lm_tile_count_kernel(const unsigned *__restrict__ in,
                                                                     const unsigned *__restrict__ totals, int nbuckets,
                                                                     unsigned *__restrict__ tcount) {
    __shared__ unsigned cnt[BUCKET_TILES], wave_sum[2][PART_THREADS / 64];
    __shared__ Slice sl;
    const int tid = threadIdx.x;
    if (tid < BUCKET_TILES) cnt[tid] = 0;
    if (!find_slice(totals, nbuckets, blockIdx.x, wave_sum, &sl)) return;
    unsigned v[SLICE_KEYS];
    bool ok[SLICE_KEYS];
    load_slice(in, sl, v, ok);
#pragma unroll
    for (int u = 0; u < SLICE_KEYS; u++)
        if (ok[u]) atomicAdd(&cnt[tile_of(v[u])], 1u);
    __syncthreads();
    if (tid < BUCKET_TILES && cnt[tid]) atomicAdd(&tcount[sl.bucket * BUCKET_TILES + tid], cnt[tid]);
}

// The slices' keys into their tiles, each slice behind what others have reserved of a tile (used[t]), and
// tiles[t] = index of the first key of tile t (tiles[ntiles] = number of keys).
__global__ __launch_bounds__(PART_THREADS) void lm_tile_scatter_kernel(const unsigned *__restrict__ in,
                                                                       const unsigned *__restrict__ totals, int nbuckets,
                                                                       const unsigned *__restrict__ tcount,
                                                                       unsigned *__restrict__ used, long long ntiles,
                                                                       unsigned *__restrict__ out,
                                                                       unsigned *__restrict__ tiles) {
    __shared__ unsigned next[PART_THREADS], cnt[PART_THREADS], wave_sum[2][PART_THREADS / 64], buf[SLICE];
    __shared__ Slice sl;
    const int tid = threadIdx.x;
    if (!find_slice(totals, nbuckets, blockIdx.x, wave_sum, &sl)) return;
    unsigned v[SLICE_KEYS], total;
    bool ok[SLICE_KEYS];
    load_slice(in, sl, v, ok);
    const long long t = (long long)sl.bucket * BUCKET_TILES + tid;
    const unsigned start = sl.start + block_exclusive(tid < BUCKET_TILES ? tcount[t] : 0u, wave_sum[0], total);
    if (sl.first) {
        if (tid < BUCKET_TILES && t < ntiles) tiles[t] = start;
        if (tid == 0 && (int)sl.bucket == nbuckets - 1) tiles[ntiles] = sl.start + total;
    }
    next[tid] = start;
    partition_batch(v, ok, tile_of, next, cnt, buf, wave_sum[1], out,
                    [&](unsigned n) { return tid < BUCKET_TILES && n ? atomicAdd(&used[t], n) : 0u; });
}

constexpr int TILE_THREADS = 512, TILE_ROUNDS = TILE / (8 * TILE_THREADS);   // 8 bins per thread and round

__device__ inline unsigned pack16(int lo, int hi) { return ((unsigned)lo & 0xffffu) | ((unsigned)hi << 16); }
__device__ inline uint4 pack16x8(const int4 &u, const int4 &v) {
    return make_uint4(pack16(u.x, u.y), pack16(u.z, u.w), pack16(v.x, v.y), pack16(v.z, v.w));
}
__device__ inline unsigned pack8(const int4 &v) {
    return (unsigned)min(v.x, 255) | (unsigned)min(v.y, 255) << 8 | (unsigned)min(v.z, 255) << 16 |
           (unsigned)min(v.w, 255) << 24;
}

// Tiles of TILE bins, grid-strided: a tile's keys counted per bin in LDS, then its bins written in
// order, 8 per thread and round, whole lines a wave: mode 0 int16(prompts - delayed), mode 2
// int16(prompts), mode 1 (BOTH: the two counted apart) int16(prompts) and min(delayed, 255) as bytes, or
// int16 delayed at sino[S + bin] without a byte output.  int16 values wrap as the reference's short
// counters do.  The kernel is bound by its writes: the next tile's first keys are loaded while a tile is
// written, and a thread clears the counters that it has read.  vec: the outputs take 16-byte stores (sino, and
// delayed or sino + S, 16-byte aligned).
template <bool BOTH>
__global__ __launch_bounds__(TILE_THREADS) void lm_tile_kernel(const unsigned *__restrict__ keys,
                                                               const unsigned *__restrict__ tiles, long long ntiles,
                                                               long long S, int mode, int16_t *__restrict__ sino,
                                                               uint8_t *__restrict__ delayed, int vec) {
    constexpr int NC = BOTH ? 2 : 1;
    __shared__ int4 cnt4[NC * TILE / 4];
    int *cnt = reinterpret_cast<int *>(cnt4);
    const int tid = threadIdx.x;
    for (int j = tid; j < NC * TILE / 4; j += TILE_THREADS) cnt4[j] = make_int4(0, 0, 0, 0);
    auto count = [&](unsigned k) {
        const int bin = (int)((k >> 1) & (TILE - 1));
        if (BOTH) atomicAdd(&cnt[(int)(k & 1) * TILE + bin], 1);
        else atomicAdd(&cnt[bin], (mode == 0 && (k & 1)) ? -1 : 1);
    };
    // the ranges of this tile and the next, and this thread's first key of this tile
    auto range = [&](long long t) { return t < ntiles ? make_uint2(tiles[t], tiles[t + 1]) : make_uint2(0, 0); };
    auto first = [&](uint2 r) { return r.x + tid < r.y ? keys[r.x + tid] : 0u; };
    long long t = blockIdx.x;
    uint2 r = range(t), rn = range(t + gridDim.x);
    unsigned k = first(r);
    __syncthreads();
    for (; t < ntiles; t += gridDim.x) {
        if (r.x + tid < r.y) count(k);
        for (unsigned i = r.x + TILE_THREADS + tid; i < r.y; i += TILE_THREADS) count(keys[i]);
        r = rn;
        k = first(r);
        rn = range(t + 2 * gridDim.x);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < TILE_ROUNDS; q++) {
            const int j = 2 * (q * TILE_THREADS + tid);      // in fours of bins
            const long long b0 = t * TILE + 4 * j;
            const int4 p0 = cnt4[j], p1 = cnt4[j + 1];
            int4 d0 = make_int4(0, 0, 0, 0), d1 = d0;
            cnt4[j] = cnt4[j + 1] = make_int4(0, 0, 0, 0);
            if (BOTH) {
                d0 = cnt4[TILE / 4 + j], d1 = cnt4[TILE / 4 + j + 1];
                cnt4[TILE / 4 + j] = cnt4[TILE / 4 + j + 1] = make_int4(0, 0, 0, 0);
            }
            if (vec && b0 + 8 <= S) {
                *reinterpret_cast<uint4 *>(sino + b0) = pack16x8(p0, p1);
                if (BOTH) {
                    if (delayed) *reinterpret_cast<uint2 *>(delayed + b0) = make_uint2(pack8(d0), pack8(d1));
                    else *reinterpret_cast<uint4 *>(sino + S + b0) = pack16x8(d0, d1);
                }
            } else {
                const int p[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
                const int d[8] = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y, d1.z, d1.w};
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    if (b0 + i < S) {
                        sino[b0 + i] = (int16_t)(uint16_t)(unsigned)p[i];
                        if (BOTH) {
                            if (delayed) delayed[b0 + i] = (uint8_t)min(d[i], 255);
                            else sino[S + b0 + i] = (int16_t)(uint16_t)(unsigned)d[i];
                        }
                    }
                }
            }
        }
        __syncthreads();   // the counters are clear for the next tile
    }
}

// Coincidence maps, pass 1: per (chunk range, head) the head's entries of the range's chunks
// counted in LDS, written as the range's partial counts.  Each wave takes one chunk at a time.
__global__ __launch_bounds__(1024) void lm_coin_kernel(const unsigned short *__restrict__ cseg,
                                                       const unsigned *__restrict__ ccnt, long long nchunks,
                                                       unsigned *__restrict__ part) {
    __shared__ unsigned cnt[COIN_HEAD];
    const int r = blockIdx.x, h = blockIdx.y;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
    for (int j = threadIdx.x; j < COIN_HEAD; j += blockDim.x) cnt[j] = 0;
    __syncthreads();
    const long long per = (nchunks + COIN_RANGES - 1) / COIN_RANGES;
    const long long c0 = r * per, c1 = min(nchunks, c0 + per);
    // a chunk's first COIN_FIRST * 64 entries (a head has 256 of a full chunk on average) are loaded
    // with its count, one chunk ahead: the loads of one chunk at a time left the wave waiting
    constexpr int COIN_FIRST = 6;
    unsigned n = 0, nn = 0;
    unsigned short v[COIN_FIRST], vn[COIN_FIRST];
    auto load = [&](long long c) __attribute__((always_inline)) {
        const unsigned short *e = cseg + (c * NHEADS + h) * (CHUNK / 2);
        nn = ccnt[c * NHEADS + h];
#pragma unroll
        for (int k = 0; k < COIN_FIRST; k++) vn[k] = e[k * 64 + lane];   // inside the chunk's 1024 slots
    };
    if (c0 + wv < c1) load(c0 + wv);
    for (long long c = c0 + wv; c < c1; c += nw) {
        n = nn;
#pragma unroll
        for (int k = 0; k < COIN_FIRST; k++) v[k] = vn[k];
        if (c + nw < c1) load(c + nw);
#pragma unroll
        for (int k = 0; k < COIN_FIRST; k++)
            if ((unsigned)(k * 64 + lane) < n) atomicAdd(&cnt[v[k]], 1u);
        const unsigned short *e = cseg + (c * NHEADS + h) * (CHUNK / 2);
        for (unsigned j = COIN_FIRST * 64 + lane; j < n; j += 64) atomicAdd(&cnt[e[j]], 1u);
    }
    __syncthreads();
    unsigned *o = part + ((long long)r * NHEADS + h) * COIN_HEAD;
    for (int j = threadIdx.x; j < COIN_HEAD; j += blockDim.x) o[j] = cnt[j];
}

// Coincidence maps, pass 2: the ranges' partial counts summed into the .ch halves
// [layer][ring][head][x] (a NULL map is skipped).
__global__ void lm_coin_sum_kernel(const unsigned *__restrict__ part, unsigned *__restrict__ coin_p,
                                   unsigned *__restrict__ coin_d) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 2 * NCRYS) return;
    const int map = i / NCRYS, k = i % NCRYS;
    unsigned *out = map ? coin_d : coin_p;
    if (!out) return;
    const int x = k % NX, head = (k / NX) % NHEADS, ring = (k / HX) % NY, layer = k / XYH;
    const int local = ((map * NDOIS + layer) * NY + ring) * NX + x;
    unsigned sum = 0;
    for (int r = 0; r < COIN_RANGES; r++) sum += part[((long long)r * NHEADS + head) * COIN_HEAD + local];
    out[k] = sum;
}

// The module-pair LUT by (module pair, A crystal, B crystal) on the device, and the counts.
int ensure_lm(hrrt_delays &c, long long nchunks, bool coin) {
    int r = upload(c);
    if (r != HRRT_OK) return r;
    int dev = -1;
    DTRY(hipGetDevice(&dev));
    if (dev != c.device) return hrrt_dl::fail(HRRT_ERR_ARG, "context tables live on another device");
    if (!c.d_sol) {
        // 12-byte records as the host holds them: 5.2 MB gather better from a 4 MB L2 than padded ones
        static_assert(sizeof(int3) == sizeof(Sol), "LUT record is three words");
        DTRY(hipMalloc(&c.d_sol, sizeof(int3) * c.lut.size()));
        DTRY(hipMemcpy(c.d_sol, c.lut.data(), sizeof(int3) * c.lut.size(), hipMemcpyHostToDevice));
    }
    if (!c.d_lm_stats) DTRY(hipMalloc(&c.d_lm_stats, sizeof(unsigned long long) * ST_WORDS));
    if (!c.h_lm_stats) DTRY(hipHostMalloc((void **)&c.h_lm_stats, sizeof(unsigned long long) * ST_WORDS));
    if (!c.d_lm_tiles) {    // first keys of the tiles, then two counters per tile of whole buckets
        const long long S = (long long)c.nplanes * c.nsino, nb = (S + (1ll << BUCKET_BITS) - 1) >> BUCKET_BITS;
        DTRY(hipMalloc(&c.d_lm_tiles, sizeof(unsigned) * (size_t)((S + TILE - 1) / TILE + 1 + 2 * nb * BUCKET_TILES)));
    }
    const long long keys = nchunks * (CHUNK / 2);
    if (keys > c.lm_key_cap) {
        if (c.d_lm_keys) DTRY(hipFree(c.d_lm_keys));
        c.d_lm_keys = nullptr;
        c.lm_key_cap = 0;
        DTRY(hipMalloc(&c.d_lm_keys, sizeof(unsigned) * 2 * (size_t)keys));
        c.lm_key_cap = keys;
    }
    if (!c.d_lm_part) DTRY(hipMalloc(&c.d_lm_part, sizeof(unsigned) * (size_t)(MAX_BUCKETS * MAX_PARTS + MAX_BUCKETS)));
    if (coin && !c.d_lm_coin_part)
        DTRY(hipMalloc(&c.d_lm_coin_part, sizeof(unsigned) * (size_t)COIN_RANGES * NHEADS * COIN_HEAD));
    if (coin && nchunks > c.lm_coin_cap) {
        if (c.d_lm_coin_seg) DTRY(hipFree(c.d_lm_coin_seg));
        if (c.d_lm_coin_cnt) DTRY(hipFree(c.d_lm_coin_cnt));
        c.d_lm_coin_seg = nullptr;
        c.d_lm_coin_cnt = nullptr;
        c.lm_coin_cap = 0;
        DTRY(hipMalloc(&c.d_lm_coin_seg, sizeof(unsigned short) * (size_t)nchunks * NHEADS * (CHUNK / 2)));
        DTRY(hipMalloc(&c.d_lm_coin_cnt, sizeof(unsigned) * (size_t)nchunks * NHEADS));
        c.lm_coin_cap = nchunks;
    }
    if (nchunks > c.lm_chunk_cap) {
        if (c.d_lm_chunks) DTRY(hipFree(c.d_lm_chunks));
        c.d_lm_chunks = nullptr;
        c.lm_chunk_cap = 0;
        DTRY(hipMalloc(&c.d_lm_chunks, sizeof(unsigned) * 66 * (size_t)nchunks));   // summaries, masks, key counts
        c.lm_chunk_cap = nchunks;
    }
    return HRRT_OK;
}

}  // namespace

extern "C" int hrrt_lm_histogram(hrrt_delays *c, const uint32_t *d_words, long long nwords, const hrrt_lm_options *opt,
                                 int16_t *d_sino, uint8_t *d_delayed, uint32_t *d_coin_p, uint32_t *d_coin_d,
                                 hrrt_lm_stats *stats, void *stream) {
    if (!c || !opt || !d_sino || (nwords > 0 && !d_words) || nwords < 0) return hrrt_dl::fail(HRRT_ERR_ARG, "null argument");
    if (opt->mode == 7) return hrrt_dl::fail(HRRT_ERR_UNSUPPORTED, "transmission histogramming is not supported");
    if (opt->mode < 0 || opt->mode > 2) return hrrt_dl::fail(HRRT_ERR_ARG, "mode must be 0, 1 or 2");
    if (nwords >= (1ll << 34)) return hrrt_dl::fail(HRRT_ERR_ARG, "stream longer than 2^34 words");
    if ((long long)c->nplanes * c->nsino > (1ll << 30)) return hrrt_dl::fail(HRRT_ERR_ARG, "sinogram larger than 2^30 bins");
    // key slots (one per two words) are indexed in 32 bits
    if (nwords > (1ll << 33) - (1ll << 22)) return hrrt_dl::fail(HRRT_ERR_ARG, "stream longer than 2^33 - 2^22 words");
    hipStream_t s = (hipStream_t)stream;
    const long long nchunks = (nwords + CHUNK - 1) / CHUNK;
    const bool coin = d_coin_p || d_coin_d;
    int r = ensure_lm(*c, std::max(nchunks, 1ll), coin);
    if (r != HRRT_OK) return r;
    const long long S = (long long)c->nplanes * c->nsino;
    LmArgs a;
    a.w = d_words;
    a.nwords = nwords;
    a.mode = opt->mode;
    a.start_ms = opt->start_ms;
    a.end_ms = opt->end_ms;
    a.ignore_border = opt->ignore_border != 0;
    a.doi = opt->no_doi == 0;
    a.sol = c->d_sol;
    a.z = c->d_z;
    a.seg = c->d_seg;
    a.nsino = c->nsino;
    a.S = S;
    a.keys = c->d_lm_keys;
    a.coin_p = d_coin_p;
    a.coin_d = d_coin_d;
    a.cseg = coin ? c->d_lm_coin_seg : nullptr;
    a.ccnt = coin ? c->d_lm_coin_cnt : nullptr;
    a.chunks = c->d_lm_chunks;
    a.cmask = c->d_lm_chunks + c->lm_chunk_cap;
    a.kcnt = c->d_lm_chunks + 65 * c->lm_chunk_cap;
    a.w16 = (uintptr_t)d_words % 16 == 0;
    a.st = c->d_lm_stats;
    const unsigned grid = (unsigned)std::max((nchunks + WAVES - 1) / WAVES, 1ll);
    lm_summary_kernel<<<grid, WAVES * 64, 0, s>>>(a, nchunks);
    if (nchunks > 0) {
        const long long npackets = (nchunks + CHUNKS_PER_PACKET - 1) / CHUNKS_PER_PACKET;
        lm_resolve_kernel<<<(unsigned)npackets, CHUNKS_PER_PACKET, 0, s>>>(a.chunks, nchunks);
        if (opt->start_ms > 0) lm_window_kernel<0><<<grid, WAVES * 64, 0, s>>>(a, nchunks);
        if (opt->end_ms > 0) lm_window_kernel<1><<<grid, WAVES * 64, 0, s>>>(a, nchunks);
        if (coin) lm_hist_kernel<true><<<grid, WAVES * 64, 0, s>>>(a, nchunks);
        else lm_hist_kernel<false><<<grid, WAVES * 64, 0, s>>>(a, nchunks);
    }
    DTRY(hipGetLastError());
    const long long ntiles = (S + TILE - 1) / TILE;
    const int nbuckets = (int)((S + (1ll << BUCKET_BITS) - 1) >> BUCKET_BITS);
    // a wave per chunk of a short stream, at most two workgroups per CU of a long one
    const int parts = (int)std::min<long long>(std::max<long long>((nchunks + PART_THREADS / 64 - 1) / (PART_THREADS / 64), 1), MAX_PARTS);
    unsigned *by_bucket = c->d_lm_keys + c->lm_key_cap, *by_tile = c->d_lm_keys, *totals = c->d_lm_part + MAX_BUCKETS * MAX_PARTS;
    unsigned *tcount = c->d_lm_tiles + ntiles + 1, *used = tcount + (size_t)nbuckets * BUCKET_TILES;
    const unsigned slices = (unsigned)(nbuckets + nchunks * (CHUNK / 2) / SLICE);    // at least as many as there are
    lm_count_kernel<<<parts, PART_THREADS, 0, s>>>(a.keys, a.kcnt, nchunks, nbuckets, c->d_lm_part);
    lm_part_sums_kernel<<<nbuckets, 64, 0, s>>>(c->d_lm_part, parts, totals, tcount, used);
    lm_scatter_kernel<<<parts, PART_THREADS, 0, s>>>(a.keys, a.kcnt, nchunks, nbuckets, c->d_lm_part, totals, by_bucket);
    lm_tile_count_kernel<<<slices, PART_THREADS, 0, s>>>(by_bucket, totals, nbuckets, tcount);
    lm_tile_scatter_kernel<<<slices, PART_THREADS, 0, s>>>(by_bucket, totals, nbuckets, tcount, used, ntiles, by_tile, c->d_lm_tiles);
    DTRY(hipGetLastError());
    // four workgroups per CU, all resident (two are in mode 1, whose counters take twice the LDS; the others follow)
    const unsigned tgrid = (unsigned)std::min(ntiles, 1024ll);
    const bool both = opt->mode == 1;
    const int vec = (uintptr_t)d_sino % 16 == 0 &&
                    (!both || (d_delayed ? (uintptr_t)d_delayed % 16 == 0 : S % 8 == 0));
    if (both)
        lm_tile_kernel<true><<<tgrid, TILE_THREADS, 0, s>>>(by_tile, c->d_lm_tiles, ntiles, S, opt->mode, d_sino, d_delayed, vec);
    else
        lm_tile_kernel<false><<<tgrid, TILE_THREADS, 0, s>>>(by_tile, c->d_lm_tiles, ntiles, S, opt->mode, d_sino, d_delayed, vec);
    if (coin) {
        lm_coin_kernel<<<dim3(COIN_RANGES, NHEADS), 1024, 0, s>>>(a.cseg, a.ccnt, nchunks, c->d_lm_coin_part);
        lm_coin_sum_kernel<<<(2 * NCRYS + 255) / 256, 256, 0, s>>>(c->d_lm_coin_part, d_coin_p, d_coin_d);
    }
    DTRY(hipGetLastError());
    if (stats) {
        const unsigned long long *h = c->h_lm_stats;
        DTRY(hipMemcpyAsync(c->h_lm_stats, a.st, sizeof(unsigned long long) * ST_WORDS, hipMemcpyDeviceToHost, s));
        DTRY(hipStreamSynchronize(s));
        memset(stats, 0, sizeof(*stats));
        stats->prompts = (long long)h[ST_PROMPTS];
        stats->randoms = (long long)h[ST_RANDOMS];
        stats->events = (long long)h[ST_EVENTS];
        stats->tags = (long long)h[ST_TAGS];
        stats->time_tags = (long long)h[ST_TIME_TAGS];
        stats->rejected = (long long)h[ST_REJECTED];
        stats->transmission = (long long)h[ST_TX];
        const bool never = opt->start_ms > 0 && h[ST_START] == NONE;
        stats->first_word = never ? -1 : (opt->start_ms > 0 ? (long long)h[ST_START] : 0);
        stats->end_word = never ? -1 : ((opt->end_ms > 0 && h[ST_END] != NONE) ? (long long)h[ST_END] + 2 : nwords);
        stats->last_time_ms = h[ST_TIME_TAGS] ? (int)(h[ST_LAST_TIME] & 0x3fffffffu) : -1;
        for (int b = 0; b < NBLOCKS; b++) {
            stats->block_total[b] = (long long)h[ST_BLOCKS + b];
            stats->block_nsamples[b] = (int)h[ST_BLOCKS + NBLOCKS + b];
            stats->block_last[b] = (int)(h[ST_BLOCKS + 2 * NBLOCKS + b] & 0x7ffffu);
        }
    }
    return HRRT_OK;
}
