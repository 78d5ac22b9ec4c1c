// kernels.hip -- CDNA4 (gfx950) kernels of the OSEM hot path.
//
// Every kernel issues its float operations in the order the reference does
// (no fused multiply-add: this file is compiled with -ffp-contract=off and
// the pragma below), so results are bit-identical to the reference
// arithmetic for the same inputs.  Citations: PJ = hrrt_osem3d/
// hrrt_osem3dv_sbrt_span3.cpp, S3 = hrrt_osem3d/hrrt_osem3d_span3.cpp,
// FIO = hrrt_osem3d/file_io_processor.cpp.
#include "kernels.h"

#include <algorithm>
#include <type_traits>

#pragma clang fp contract(off)

namespace hrrt {

namespace {

__device__ __forceinline__ float4 f4(float a) { return make_float4(a, a, a, a); }
__device__ __forceinline__ float4 add4(float4 a, float4 b) {
    return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}
__device__ __forceinline__ float4 mul4(float4 a, float s) {
    return make_float4(a.x * s, a.y * s, a.z * s, a.w * s);
}
__device__ __forceinline__ float half_at(const uint16_t *p, size_t i) { return __half2float(__ushort_as_half(p[i])); }

// Compensated (Kahan) summation: s accumulates, c carries the low-order bits lost so far.
__device__ __forceinline__ void kahan_add(float &s, float &c, float x) {
    const float y = x - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
}

__device__ __forceinline__ void ll_add(LlSum &s, double t) {
    constexpr double M = 0x1.8p52;                          // v + M holds v, rounded to a whole number, in its low bits
    constexpr long long MB = 0x4338000000000000ll;
    if (fabs(t) < 0x1p32) {
        const double w = t + M;
        s.whole += __double_as_longlong(w) - MB;
        s.frac += __double_as_longlong((t - (w - M)) * 0x1p46 + M) - MB;
    } else {
        s.large += t;
    }
}

// The workgroup's sum, in thread 0 (red: one element per wave)
__device__ __forceinline__ LlSum ll_block_sum(LlSum s, LlSum *red) {
    auto add = [&](const LlSum &o) {
        s.whole += o.whole;
        s.frac += o.frac;
        s.large += o.large;
    };
    auto carry = [&] {
        s.whole += s.frac >> 46;
        s.frac &= (1ll << 46) - 1;
    };
    carry();
    for (int o = 32; o > 0; o >>= 1) add(LlSum{__shfl_xor(s.whole, o), __shfl_xor(s.frac, o), __shfl_xor(s.large, o)});
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)(blockDim.x >> 6); w++) add(red[w]);
        carry();
    }
    return s;
}

// f(0), f(1), ..., f(N - 1) with the index as a constant
template <int N, int I = 0, typename F>
__device__ __forceinline__ void unroll(F &&f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        unroll<N, I + 1>(f);
    }
}

__device__ __forceinline__ float lane(const float4 &v, int l) {
    return l == 0 ? v.x : (l == 1 ? v.y : (l == 2 ? v.z : v.w));
}

// The eight symmetric sample positions of (x, y) (PJ:1856-1864).  Samples 0..3
// feed "pam" (near half of the ray), 4..7 feed "pam2" (mirrored half).
// i: (x, y), (N-x, y), (N-y, x), (N-y, N-x), (x, N-y), (N-x, N-y), (y, x), (y, N-x).  Bit 0
// mirrors x, bit 1 swaps the two coordinates, bit 2 mirrors y.
//
// Transposed staging of a row.  A wave owns 16 chunks (4 planes
// each) of one half of the row's samples: lane l samples chunk 16 b + (l & 15) of sample
// 4 h + (l >> 4), so each row of 16 lanes loads 256 contiguous bytes of one image column.
// A 4x4 transpose across the four 16-lane rows (two permlane32 swaps, then two permlane16
// swaps) leaves lane l with plane 4 q + (l >> 4) of all four samples, stored with one
// 16-byte LDS write instead of four scattered 4-byte ones.
// Staged planes per column: at most 256 image planes and the zero plane behind them, as a
// constant so that every LDS read of a row takes its buffer and neighbour as immediate offsets.
constexpr int FP_PL = 264;

__device__ __forceinline__ void swap_pl32(float &a, float &b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}

__device__ __forceinline__ void swap_pl16(float &a, float &b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}

// v: planes 4q..4q+3 of sample (l >> 4) -> plane 4q + (l >> 4) of samples 0..3.
__device__ __forceinline__ float4 xpose4(float4 v) {
    swap_pl32(v.x, v.z);   // rows 0-1 receive plane 0 of samples 2-3, rows 2-3 plane 2 of samples 0-1
    swap_pl32(v.y, v.w);
    swap_pl16(v.x, v.y);   // odd rows' x <-> even rows' y
    swap_pl16(v.z, v.w);
    return v;
}

// One bilinear sample of a z chunk (PJ:1865-1892), its four neighbours in flight.
struct Sample {
    float4 r1, r2, r3, r4;
    float x1, y1;
    bool ok;
};

__device__ __forceinline__ void sample_load(const DevGeom &g, const float4 *__restrict__ image, float cosv, float sinv,
                                            float dx, float dy, int q, Sample &s) {
    const int NQ = g.NQ, N = g.N, c = g.c;
    const float xx0 = dx * cosv - dy * sinv + c;
    const float yy0 = dx * sinv + dy * cosv + c;
    s.ok = q < NQ && !(xx0 < 0 || xx0 > N - 2 || yy0 < 0 || xx0 > N - 2);
    if (!s.ok) return;
    const int xi = (int)xx0, yi = (int)yy0;
    s.x1 = xx0 - xi;
    s.y1 = yy0 - yi;
    // 32-bit chunk offsets from the uniform image base (an image holds < 2^32 chunks)
    const unsigned o = ((unsigned)xi * (unsigned)N + (unsigned)yi) * (unsigned)NQ + (unsigned)q;
    const unsigned nx = (unsigned)N * (unsigned)NQ;
    s.r1 = image[o];
    s.r2 = image[o + nx];
    s.r3 = image[o + (unsigned)NQ];
    s.r4 = image[o + nx + (unsigned)NQ];
}

// Combined and transposed: plane 4 q + (l >> 4) of the wave's four samples (every lane must call).
__device__ __forceinline__ float4 sample_combine(const Sample &s) {
    const float x1 = s.x1, y1 = s.y1;
    const float w1 = (1 - x1) * (1 - y1), w2 = x1 * (1 - y1), w3 = y1 * (1 - x1), w4 = y1 * x1;
    const float4 v = s.ok ? add4(add4(mul4(s.r1, w1), mul4(s.r2, w2)), add4(mul4(s.r3, w3), mul4(s.r4, w4))) : f4(0.f);
    return xpose4(v);
}

// What a lane samples of every row: its item's position relative to the centre is linear in
// fy = y - c (small integers, so these float operations are exact), its chunk and its LDS slot.
struct SampleLane {
    float kx, sx, ky, sy;
    int q;      // chunk, NQ or more: nothing to load
    int slot;   // float4 index in the row's two halves, negative: nothing to store
};

__device__ __forceinline__ SampleLane sample_lane(const DevGeom &g, int it, int x) {
    SampleLane s;
    const int nq16 = (g.NQ + 15) >> 4, chunk = it >> 6, l = it & 63;
    const int h = chunk >= nq16 ? 1 : 0;
    s.q = 16 * (chunk - h * nq16) + (l & 15);
    const int i = 4 * h + (l >> 4), z = 4 * s.q + (i & 3);
    if (chunk >= 2 * nq16) s.q = g.NQ;
    s.slot = s.q < g.NQ && z < g.Z ? h * FP_PL + z : -1;
    const float X = (float)((i & 1) ? g.c - x : x - g.c);       // x - c or its mirror
    const float Yd = (i & 4) ? -1.f : 1.f, Ys = -Yd;             // coefficients of y - c
    s.kx = (i & 2) ? 0.f : X;
    s.sx = (i & 2) ? Ys : 0.f;
    s.ky = (i & 2) ? X : 0.f;
    s.sy = (i & 2) ? 0.f : Yd;
    return s;
}

// Forward grid.  Workgroups are dispatched round-robin over the 8 XCDs (blockIdx k runs on XCD
// k mod 8), each with its own L2.  A strip is FP_STRIP neighbouring rays of one (view pair,
// frame), whose rotated rows share image columns; the strips of every pair and frame are ordered
// from the centre (the longest rays) outwards and dealt to the XCDs in turn, so that an XCD
// holds neighbouring rays at a time, all XCDs get the same work and the short rays come last (9 view
// pairs at 256 x 256: 0.825 -> 0.783 ms against a contiguous range of rays per XCD, whose
// longest took 520 rows of a CU's time where the mean is 434).
constexpr int FP_STRIP = 16;
static inline long long fp_blocks(int c, int npf, int nsplit) {
    const long long items = (long long)((c + FP_STRIP - 1) / FP_STRIP) * npf;
    return (items + 7) / 8 * 8 * FP_STRIP * nsplit;
}
__device__ __forceinline__ bool fp_block(const DevGeom &g, const PairBatch &b, int nsplit, int bid, int &frame, int &lp,
                                         int &ray, int &split) {
    const int npf = b.npairs * b.nframes, per = FP_STRIP * nsplit;
    const int r = bid >> 3, k = r / per, j = r - k * per;
    const int item = 8 * k + (bid & 7);
    const int strip = item / npf, pf = item - strip * npf;
    ray = strip * FP_STRIP + j / nsplit;
    split = j % nsplit;
    frame = pf / b.npairs;
    lp = pf - frame * b.npairs;
    return ray < g.c;
}

// Rotation grid: voxel column x and group of 4 rows yg.  Each XCD owns a band of row
// groups and walks it in blocks of 16 columns, so the bilinear neighbourhoods that
// concurrent workgroups gather stay in that XCD's L2.
__device__ __forceinline__ void rot_block(int bid, int N, int NYG, int &x, int &yg) {
    if ((NYG & 7) == 0 && (N & 15) == 0) {
        const int xcd = bid & 7, r = bid >> 3;
        const int band = NYG >> 3, blk = 16 * band;
        x = (r / blk) * 16 + (r & 15);
        yg = xcd * band + (r % blk) / 16;
    } else {
        x = bid % N;
        yg = bid / N;
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// Forward projector (forward_proj3d_view1_thread PJ:1728-1978 + scatter
// PJ:1397-1436), optionally fused with the OP ratio (pt_update_est_w3
// S3:2493-2505) and the back-projection rescale (PJ:1638-1649).
//
// One workgroup per (view pair, x in [1, N/2], share of the planes).  The
// eight rotated z-columns of each row y are staged in LDS (double buffered);
// a thread accumulates its planes over y in the reference's order.  A plane's
// axial positions for row y are recomputed from per-plane constants with the
// float operations that build the reference's flookup table and middle-plane
// positions (PJ:544-562, 1929-1944).
//
// The middle planes of a segment group share their positions up to the plane
// shift, so a thread takes a run of RL of them: one position per row, and
// 4 (RL + 1) LDS reads of 16 bytes in place of 8 RL.  End planes and axial
// planes go one per thread (single).
//
// What bounds it: LDS reads and FP32 VALU, about equally (span 3, 9 view pairs at 256 x 256: 16 runs and 5 singles
// of 64 lanes per row; LDS busy for 52 % of the time, VALU for 54 % at 2.2 cycles an instruction).  With one plane per thread slot and 8 reads per plane the LDS alone
// took 2 of the 2.9 thousand cycles of a row.  RL = 3 is odd, so the 16 lanes of a quarter-wave read
// 16 different bank groups, and its sums fit 128 registers with 16 waves in a CU: 0.69 -> 0.586 ms for
// such a subset.  The samples of a step are loaded a whole step ahead and stored at its beginning,
// so that no wave waits for memory before the barrier, and a step of 16 waves holds two
// rows (0.70 -> 0.68 ms).
// ---------------------------------------------------------------------------
// Axial sample positions of a plane in a row: LDS byte offsets of the two lower planes (the plane
// shift included) and their fractions.
struct FpPos {
    int o1, o2;
    float f1, f2;
};

template <bool FAST>
__device__ __forceinline__ FpPos fp_pos(float base, float tan, float fy2, int dbyte) {
    FpPos q;
    const float pt = fy2 * tan;
    const float zz1 = base - pt, zz2 = base + pt;
    const int i1 = (int)zz1, i2 = (int)zz2;
    if (FAST) {        // zz >= 0: zz - trunc(zz) = zz - floor(zz)
        q.f1 = __builtin_amdgcn_fractf(zz1);
        q.f2 = __builtin_amdgcn_fractf(zz2);
    } else {
        q.f1 = zz1 - i1;
        q.f2 = zz2 - i2;
    }
    q.o1 = i1 * (int)sizeof(float4) + dbyte;
    q.o2 = i2 * (int)sizeof(float4) + dbyte;
    return q;
}

// PJ:1934-1944 for R consecutive planes: acc[j] += (pb[z2+1] + pa[z])*f2 + (pa[z+1] + pb[z2])*f1
template <int RL>
__device__ __forceinline__ void fp_add(float4 (&acc)[RL], const float4 *pa, const float4 *pb, const FpPos &q) {
    const float4 *qa = reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(pa) + q.o1);
    const float4 *qb = reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(pb) + q.o2);
    float4 a[RL + 1], d[RL + 1];
#pragma unroll
    for (int j = 0; j <= RL; j++) a[j] = qa[j], d[j] = qb[j];
#pragma unroll
    for (int j = 0; j < RL; j++)
        acc[j] = add4(acc[j], add4(mul4(add4(d[j + 1], a[j]), q.f2), mul4(add4(a[j + 1], d[j]), q.f1)));
}

// What a plane's bins need at the write-out, RL consecutive planes of one segment: the inputs of the
// bins of the four lanes (v, x), (v, N-x), (v+90, x), (v+90, N-x).
template <int MODE, int RL>
struct FpBins {
    float a[4][RL];
    int16_t pr[4][RL];
    uint16_t wn[4][RL];
};

template <int MODE, int RL>
__device__ __forceinline__ void fp_bins_load(const DevGeom &g, int pidx, int cnt, int x, int view, const FpIO &io,
                                             FpBins<MODE, RL> &b) {
    if (MODE == FP_PLAIN) return;
#pragma unroll
    for (int l = 0; l < 4; l++) {
        const int col = ((l & 1) && x != g.c) ? g.N - x : x, h = l >> 1;
        const size_t gi = ((size_t)(view * 2 + h) * g.N + col) * g.spp + pidx;
#pragma unroll
        for (int j = 0; j < RL; j++) {
            const int jj = j < cnt ? j : 0;
            if (MODE == FP_RATIO16) b.a[l][j] = half_at(static_cast<const uint16_t *>(io.add), gi + jj);
            else b.a[l][j] = static_cast<const float *>(io.add)[gi + jj];
            if (MODE != FP_RATIO_W012) b.pr[l][j] = io.prompt[gi + jj];
            if (MODE == FP_RATIO16 && io.ll_part) b.wn[l][j] = io.invnorm[gi + jj];
        }
    }
}

// Write-out of RL planes of one segment for the four lanes (PJ:1397-1436), optionally through the OP
// ratio (S3:2493-2505) and the back-projection rescale (PJ:1638-1649).
template <int MODE, int RL>
__device__ __forceinline__ void fp_bins_write(const DevGeom &g, const float4 (&acc)[RL], float sc, float resc, int pidx,
                                              int cnt, int x, int lp, float *__restrict__ out, const FpIO &io,
                                              const FpBins<MODE, RL> &b, LlSum &ll) {
#pragma unroll
    for (int l = 0; l < 4; l++) {
        if ((l & 1) && x == g.c) continue;   // at x == N/2 lanes 1/3 duplicate lanes 0/2
        const int col = (l & 1) ? g.N - x : x, h = l >> 1;
        float r[RL];
#pragma unroll
        for (int j = 0; j < RL; j++) {
            float v = lane(acc[j], l) * sc;
            if (MODE == FP_RATIO_W012) {   // pt_update_est_w012 S3:2436-2447
                const float q = v > g.eps3 ? b.a[l][j] / v : 0.0f;
                v = q * resc;
            } else if (MODE != FP_PLAIN) {
                const float den = v + b.a[l][j];
                const int16_t pr = b.pr[l][j];
                float q;
                if (pr == 0) q = 0.0f;
                else if (den > g.eps3) q = (float)pr / den;
                else q = 1.0f;
                if (MODE == FP_RATIO16 && io.ll_part && j < cnt) {
                    // Poisson log-likelihood of the bin (without log y!) at the mean (est + add) / (N*A)
                    const float w = __half2float(__ushort_as_half(b.wn[l][j]));
                    if (w > 0.0f && den > g.eps3) {
                        const double mu = (double)den * (double)w;
                        ll_add(ll, (pr > 0 ? (double)pr * log(mu) : 0.0) - mu);
                    }
                }
                v = q * resc;
            }
            r[j] = v;
        }
        float *o = out + ((size_t)(lp * 2 + h) * g.N + col) * g.spp + pidx;
        if (RL == 3 && cnt == 3) {
            typedef float f3 __attribute__((ext_vector_type(3), aligned(4)));
            f3 v3;
            v3.x = r[0], v3.y = r[RL > 1 ? 1 : 0], v3.z = r[RL > 2 ? 2 : 0];
            *reinterpret_cast<f3 *>(o) = v3;
        } else {
#pragma unroll
            for (int j = 0; j < RL; j++)
                if (j < cnt) o[j] = r[j];
        }
    }
}

// FAST: no row is skipped and no axial position is negative (checked on the host), so the axial
// fraction is one v_fract and the planes need no row test.
template <int RL, int R, int MODE, bool FAST>
__global__ void __launch_bounds__(1024) fp_kernel(const DevGeom g, const PairBatch b, const float4 *__restrict__ image,
                                                  float *__restrict__ out, FpIO io, int nsplit) {
    __shared__ float4 lds[(1 + 4 * R) * FP_PL];
    float4 *rimc = lds;
    float4 *stage = lds + FP_PL;  // [2][R][2][FP_PL]
    int frame, lp, ray, split;
    if (!fp_block(g, b, nsplit, blockIdx.x, frame, lp, ray, split)) return;
    const int L0 = ((frame * b.npairs + lp) * g.c + ray) * nsplit + split;
    image += frame * b.img_stride / 4;
    out += frame * b.ratio_stride;
    if (MODE == FP_RATIO || MODE == FP_RATIO16) io.prompt += frame * b.sino_stride;
    if (MODE == FP_RATIO || MODE == FP_RATIO_W012) io.add = static_cast<const float *>(io.add) + frame * b.sino_stride;
    else if (MODE == FP_RATIO16) io.add = static_cast<const uint16_t *>(io.add) + frame * b.sino_stride;
    LlSum ll{};
    const int x = g.c - ray;
    const int view = b.view0 + b.view_stride * lp;
    const int N = g.N, c = g.c;
    if (g.cyl_lo[x] == g.cyl_hi[x] || g.nzmask[view * (c + 1) + x] == 0) {
        if (MODE == FP_RATIO16 && io.ll_part && threadIdx.x == 0) io.ll_part[L0] = LlSum{};
        return;
    }
    const float cosv = g.cos_psi[view], sinv = g.sin_psi[view];
    const int ystart = g.cyl_lo[x];

    // This thread's run {k | first plane << 8 | planes << 16, bits(base), bits(tan), delta | ymin << 16}
    // and single (the same with one plane; k = 0: axial).  Singles go to the waves behind the runs, then
    // over again from the first wave.
    int4 er = make_int4(0, 0, 0, 0), es = er;
    {
        const int r_lo = (int)((long long)g.fp_nr[RL == 3] * split / nsplit), r_hi = (int)((long long)g.fp_nr[RL == 3] * (split + 1) / nsplit);
        const int s_lo = (int)((long long)g.fp_ns * split / nsplit), s_hi = (int)((long long)g.fp_ns * (split + 1) / nsplit);
        const int nr = r_hi - r_lo, ns = s_hi - s_lo, tid = threadIdx.x;
        int ts = tid - ((nr + 63) & ~63);
        if (ts < 0) ts += blockDim.x;
        if (tid < nr) er = g.fp_runs[RL == 3][r_lo + tid];
        if (ts < ns) es = g.fp_single[s_lo + ts];
    }

    // The centre row's samples (x,c),(N-x,c),(c,x),(c,N-x) (PJ:1815-1829) and the first rows.  A wave
    // samples one item of a step: wave w the (w mod n)-th of the n of row w / n.
    Sample s0, nxt;
    const int per_row = 128 * ((g.NQ + 15) >> 4);
    const int srow = __builtin_amdgcn_readfirstlane((int)threadIdx.x / per_row);
    SampleLane sl = sample_lane(g, (int)threadIdx.x - srow * per_row, x);
    if (srow >= R) sl.q = g.NQ, sl.slot = -1;
    const bool wave_samples = __any(sl.slot >= 0);
    const int cq = 16 * (threadIdx.x >> 6) + (threadIdx.x & 15), ci = (threadIdx.x & 63) >> 4;
    {
        const int xx = ci == 0 ? x : (ci == 1 ? N - x : c), yy = ci < 2 ? c : (ci == 2 ? x : N - x);
        sample_load(g, image, cosv, sinv, (float)(xx - c), (float)(yy - c), cq, s0);
    }
    // loads of rows y .. y + R - 1 (rows from c on are not staged), and their combination into LDS
    auto load_rows = [&](int y) __attribute__((always_inline)) {
        nxt.ok = false;
        if (y + srow >= c) return;
        const float fy = (float)(y + srow - c);
        sample_load(g, image, cosv, sinv, __builtin_fmaf(sl.sx, fy, sl.kx), __builtin_fmaf(sl.sy, fy, sl.ky), sl.q, nxt);
    };
    auto store_rows = [&](float4 *buf) __attribute__((always_inline)) {
        if (!wave_samples) return;
        const float4 v = sample_combine(nxt);
        if (sl.slot >= 0) buf[srow * 2 * FP_PL + sl.slot] = v;
    };
    load_rows(ystart);
    for (int i = threadIdx.x; i < 4 * R * FP_PL; i += blockDim.x) stage[i] = f4(0.f);   // the planes behind the image stay zero
    __syncthreads();
    {
        const float4 v = sample_combine(s0);
        if (cq < g.NQ) rimc[4 * cq + ci] = v;
    }
    store_rows(stage);
    load_rows(ystart + R);
    __syncthreads();

    const bool run = er.x != 0, single = (es.x & 0xff) != 0, axial = !single && (es.x >> 16) != 0;
    const int ryr = (er.x >> 8) & 0xff, syr = (es.x >> 8) & 0xff;
    const float rbase = __int_as_float(er.y), rtan = __int_as_float(er.z);
    const float sbase = __int_as_float(es.y), stan = __int_as_float(es.z);
    const int rbyte = (er.w & 0xffff) * (int)sizeof(float4);                      // plane shift, in LDS bytes
    const int sbyte = (axial ? syr : es.w & 0xffff) * (int)sizeof(float4);        // (an axial plane: its row)
    const int rmin = FAST ? 0 : er.w >> 16, smin = FAST ? 0 : es.w >> 16;
    // centre row samples (PJ:1830-1838)
    float4 r1[RL], r2[RL], s1[1], s2[1];
#pragma unroll
    for (int j = 0; j < RL; j++) r1[j] = r2[j] = rimc[ryr + j];
    s1[0] = s2[0] = rimc[syr];

    // project the staged row y (halves pa, pb) into this thread's planes
    auto project = [&](const float4 *pa, const float4 *pb, int y) __attribute__((always_inline)) {
        const float fy2 = (float)(c - y);   // (y - c) * tan = -((c - y) * tan) exactly
        if (run && (FAST || y >= rmin)) {   // PJ:1920-1921
            const FpPos q = fp_pos<FAST>(rbase, rtan, fy2, rbyte);
            fp_add<RL>(r1, pa, pb, q);
            fp_add<RL>(r2, pb, pa, q);
        }
        if (single && (FAST || y >= smin)) {
            const FpPos q = fp_pos<FAST>(sbase, stan, fy2, sbyte);
            fp_add<1>(s1, pa, pb, q);
            fp_add<1>(s2, pb, pa, q);
        }
        if (axial) {   // theta = 0 PJ:1907-1910
            const float4 *qa = reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(pa) + sbyte);
            const float4 *qb = reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(pb) + sbyte);
            s1[0] = add4(s1[0], add4(qa[0], qb[0]));
        }
    };
    // R rows per barrier: the samples of the next R rows, loaded during the step before, go into the
    // other buffer, the loads of the R rows behind them are issued, then this step's rows are projected
    auto step = [&](auto stc, int y) __attribute__((always_inline)) {
        constexpr int st = decltype(stc)::value;
        if (y + R < c) {
            store_rows(stage + (st ^ 1) * 2 * R * FP_PL);
            load_rows(y + 2 * R);
        }
        unroll<R>([&](auto rc) __attribute__((always_inline)) {
            constexpr int r = decltype(rc)::value;
            const float4 *pa = stage + (st * R + r) * 2 * FP_PL;
            if (r == 0 || y + r < c) project(pa, pa + FP_PL, y + r);
        });
        __syncthreads();
    };
    for (int y = ystart; y < c; y += 2 * R) {   // steps alternate between the two buffers
        step(std::integral_constant<int, 0>{}, y);
        if (y + R < c) step(std::integral_constant<int, 1>{}, y + R);
    }

    // scaling PJ:1953-1975 and write-out; every plane of a run has the run's scale, and the planes of a
    // segment are consecutive
    if (run) {
        const int k = er.x & 0xff, cnt = er.x >> 16;
        const float sc = g.rescalearray[(k - 1) * g.Z + ryr];
        const int p1 = g.seg_data[2 * k] + (ryr - g.yb[2 * k]), p2 = g.seg_data[2 * k - 1] + (ryr - g.yb[2 * k - 1]);
        const float c1 = g.bp_rescale[2 * k], c2 = g.bp_rescale[2 * k - 1];
        FpBins<MODE, RL> b1, b2;
        fp_bins_load(g, p1, cnt, x, view, io, b1);
        if (MODE != FP_RATIO16) fp_bins_load(g, p2, cnt, x, view, io, b2);
        fp_bins_write(g, r1, sc, c1, p1, cnt, x, lp, out, io, b1, ll);
        if (MODE == FP_RATIO16) fp_bins_load(g, p2, cnt, x, view, io, b2);   // the registers of its sums hold one set
        fp_bins_write(g, r2, sc, c2, p2, cnt, x, lp, out, io, b2, ll);
    }
    if (single || axial) {
        const int k = es.x & 0xff, seg = 2 * k;
        const float sc = k == 0 ? g.y_size : g.rescalearray[(k - 1) * g.Z + syr];
        const int p1 = g.seg_data[seg] + (syr - g.yb[seg]);
        FpBins<MODE, 1> b1;
        fp_bins_load(g, p1, 1, x, view, io, b1);
        fp_bins_write(g, s1, sc, g.bp_rescale[seg], p1, 1, x, lp, out, io, b1, ll);
        if (single) {
            const int p2 = g.seg_data[seg - 1] + (syr - g.yb[seg - 1]);
            fp_bins_load(g, p2, 1, x, view, io, b1);
            fp_bins_write(g, s2, sc, g.bp_rescale[seg - 1], p2, 1, x, lp, out, io, b1, ll);
        }
    }
    if (MODE == FP_RATIO16 && io.ll_part) {
        const LlSum t = ll_block_sum(ll, reinterpret_cast<LlSum *>(lds));
        if (threadIdx.x == 0) io.ll_part[L0] = t;
    }
}

// ---------------------------------------------------------------------------
// Back projector, direct variant (back_proj3d2 PJ:1457-1620 with
// back_proj3d_view_n1 PJ:2927-3086), as a gather.  For a rotated-frame voxel
// (X, Y) the reference's pass over view v gives A(X,Y) from sinogram column X
// and its pass over view v+90 gives B(X,Y) from column Y; R = A + B.  One
// workgroup per (column, role, view pair) stages the column in LDS and
// evaluates every voxel of the disk row/column that reads it; a wave owns one
// voxel and its lanes the planes z = lane + 64 j.
//
// LDS holds (p[i], p[i+1] - p[i]) per plane, the difference rounded as the
// reference rounds it, and every oblique segment sits inside a window of zero
// planes sized on the host from its rows' shifts.  Slots 0-2 (z < 192) are
// therefore evaluated without any range test: lanes outside the reference's
// range [zsa, zea] (PJ:2986-2995) interpolate between zeros and add exactly +0;
// slot 3 runs only when the range reaches it (a wave-uniform test).  The wave
// keeps its voxel row's lookup entries in VGPRs (lane k-1: row sl, lane 32+k-1:
// row N-sl) and takes entry k with readlane, so the loop over segment groups
// waits on nothing but its own LDS reads.
// ---------------------------------------------------------------------------
template <typename SRC_T, bool KAHAN>
__global__ void __launch_bounds__(1024) bp_kernel(const DevGeom g, const PairBatch b, const SRC_T *__restrict__ src,
                                                  int src_global, int apply_rescale, const int16_t *__restrict__ pseg,
                                                  float *__restrict__ bufA, float *__restrict__ bufB) {
    extern __shared__ float2 colpq[];
    const int col = blockIdx.x + 1, role = blockIdx.y, lp = blockIdx.z % b.npairs, frame = blockIdx.z / b.npairs;
    const int view = b.view0 + b.view_stride * lp;
    const int N = g.N, c = g.c, Z = g.Z, GM = g.GM, K = g.K;
    src += frame * b.ratio_stride;
    bufA += frame * b.buf_stride;
    bufB += frame * b.buf_stride;
    const int lo = g.cyl_lo[col], hi = g.cyl_hi[col];
    if (lo == hi) return;
    const int gp = src_global ? view : lp;
    const SRC_T *cp = src + ((size_t)(gp * 2 + role) * N + col) * g.spp;
    auto value = [&](int i) -> float {
        float v;
        if constexpr (sizeof(SRC_T) == 2) v = half_at(reinterpret_cast<const uint16_t *>(cp), i);
        else v = cp[i];
        return apply_rescale ? v * g.bp_rescale[pseg[i]] : v;
    };
    for (int i = threadIdx.x; i < g.bp_lds; i += blockDim.x) {
        const int s0 = g.bp_src[i], s1 = g.bp_src[i + 1];
        const float v0 = s0 >= 0 ? value(s0) : 0.0f, v1 = s1 >= 0 ? value(s1) : 0.0f;
        colpq[i] = make_float2(v0, v1 - v0);
    }
    __syncthreads();
    const int mcol = col <= c ? col : N - col;
    const bool masked = g.nzmask[view * (c + 1) + mcol] == 0;
    float *dst = role == 0 ? bufA : bufB;
    dst += (size_t)lp * N * N * g.Z4;
    const int lanei = threadIdx.x & 63, nw = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (lo == c && hi == c + 1) {
        // a one-pixel column: the incremental variant also writes rows c-1 and c+1, zero here
        for (int t = threadIdx.x; t < 2 * 64; t += blockDim.x) {
            const int V = (t >> 6) ? c + 1 : c - 1;
            const int X = role == 0 ? col : V, Y = role == 0 ? V : col;
            for (int z = t & 63; z < Z; z += 64) dst[((size_t)X * N + Y) * g.Z4 + z] = 0.0f;
        }
    }
    for (int Vv = lo + wave; Vv < hi; Vv += nw) {
        const int V = __builtin_amdgcn_readfirstlane(Vv);
        const int X = role == 0 ? col : V, Y = role == 0 ? V : col;
        float *o = dst + ((size_t)X * N + Y) * g.Z4;
        if (masked && V != c) {
            for (int z = lanei; z < Z; z += 64) o[z] = 0.0f;
            continue;
        }
        const int sl = V <= c ? V : N - V, ll = N - sl;
        const bool first_even = role == 0 ? (V <= c) : (V >= c);
        // lookup entries of rows sl (lanes 0..GM-1) and ll (lanes 32..32+GM-1), with the LDS base
        // of the segment each row reads already chosen
        int range = 0, base = 0, frac = 0;   // frac: float bits (readlane moves 32-bit integers)
        {
            const bool own = lanei < GM, other = lanei >= 32 && lanei - 32 < GM;
            if (own || other) {
                const int4 e = g.bp_lut2[(own ? sl : ll) * GM + (lanei & 31)];
                range = e.x;
                base = (own == first_even) ? e.y : e.z;
                frac = e.w;
            }
        }
        float i1[4], i2[4], c1[4], c2[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int z = lanei + 64 * j;
            const float t0 = z < Z ? colpq[z].x : 0.0f;
            i1[j] = first_even ? t0 : 0.0f;
            i2[j] = first_even ? 0.0f : t0;
            c1[j] = c2[j] = 0.0f;
        }
        for (int k = 1; k <= K; k++) {
            const int b1 = __builtin_amdgcn_readlane(base, k - 1), b2 = __builtin_amdgcn_readlane(base, 31 + k);
            const float f1 = __int_as_float(__builtin_amdgcn_readlane(frac, k - 1));
            const float f2 = __int_as_float(__builtin_amdgcn_readlane(frac, 31 + k));
            const float2 *q1 = colpq + b1 + lanei, *q2 = colpq + b2 + lanei;
            float2 a[3], bq[3];
#pragma unroll
            for (int j = 0; j < 3; j++) {
                a[j] = q1[64 * j];
                bq[j] = q2[64 * j];
            }
#pragma unroll
            for (int j = 0; j < 3; j++) {
                if (KAHAN) {
                    kahan_add(i1[j], c1[j], a[j].x + f1 * a[j].y);
                    kahan_add(i2[j], c2[j], bq[j].x + f2 * bq[j].y);
                } else {
                    i1[j] = i1[j] + (a[j].x + f1 * a[j].y);
                    i2[j] = i2[j] + (bq[j].x + f2 * bq[j].y);
                }
            }
            const int r1 = __builtin_amdgcn_readlane(range, k - 1), r2 = __builtin_amdgcn_readlane(range, 31 + k);
            const int zs1 = r1 & 0xffff, ze1 = r1 >> 16, zs2 = r2 & 0xffff;
            if (ze1 >= 192) {
                const float2 t = q1[192];
                if (KAHAN) kahan_add(i1[3], c1[3], t.x + f1 * t.y);
                else i1[3] = i1[3] + (t.x + f1 * t.y);
            }
            if (zs2 + (ze1 - zs1) >= 192) {
                const float2 t = q2[192];
                if (KAHAN) kahan_add(i2[3], c2[3], t.x + f2 * t.y);
                else i2[3] = i2[3] + (t.x + f2 * t.y);
            }
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int z = lanei + 64 * j;
            if (z < Z) o[z] = i1[j] + i2[j];
        }
    }
}

// ---------------------------------------------------------------------------
// Back projector, incremental variant (back_proj3d_thread1 PJ:1622-1699 with
// back_proj3d_view_n1thread PJ:4162-4668), the reference's default.  Walking a
// column's rows away from the centre, each plane keeps running sums s1 (row y)
// and s2 (row N-y) and their per-row increments d1, d2; at the rows where a
// group's integer shift changes (the breakpoints of blutacc, PJ:718-784) the
// increments are corrected.  One workgroup per (column x <= N/2, view v or
// v+90, view pair), for NB = 2 bins x and N-x, or for one of them (NB = 1); a thread
// owns one plane of its bins and applies, to its own accumulators, exactly the terms the
// reference's loops apply to that plane, in the reference's order.  View v
// writes the rotated-frame half A, view v+90 the half B, so each voxel of A and
// of B has one writer and R = A + B as for the direct variant.
//
// LDS: segment 0, then per group a window of cells by row (layout described with the host tables).  The
// centre and the first row read the raw column and form the reference's differences from it; the window
// is then converted once, in place, to the values the breakpoint terms read.  A breakpoint
// is then, for every plane, two clamped reads and eight fixed operations per bin (b-term first, then
// a-term, each one s += m*coef, d -= m for both sums); the reads that fall outside the breakpoint's rows
// hit the window's zero cells and add +0.
//
// What bounds it (9 pairs at 256 x 256, span 3, 0.346 ms; 0.435 with one bin per workgroup, scalar loads of the
// records and table-driven staging): the chains of sums of the three waves a SIMD holds (149 M vector instructions, one
// per 5.7 cycles and SIMD where independent additions go one per 2.2; LDS busy for 18 % of the time), then the 0.7 GB
// of halves written, which alone take 0.11 ms. Two bins per thread share a breakpoint's record, addresses and
// reads; its cells are read while the one before is applied, across the rows; the longest columns start first.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// A cell of the window: {segment 2k, segment 2k-1} of each of the NB bins.
template <int NB>
struct __attribute__((aligned(8 * NB))) IncCell {
    float2 b[NB];
};
__device__ __forceinline__ float2 sub2(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 mul2(float2 a, float s) { return make_float2(a.x * s, a.y * s); }

template <int NB>
__global__ void __launch_bounds__(256, NB == 2 ? 3 : 6) bp_inc_kernel(const DevGeom g, const PairBatch b,
                                                                    const float *__restrict__ src, int src_global,
                                                                    int apply_rescale, float *__restrict__ bufA,
                                                                    float *__restrict__ bufB) {
    constexpr int ITEMS = 4;    // chunks a thread has in flight while the column loads
    constexpr int CELLS = 13;        // cells a thread converts between two barriers
    extern __shared__ float4 inc_lds[];
    typedef IncCell<NB> Cell;
    Cell *W = reinterpret_cast<Cell *>(inc_lds);
    float *S0 = reinterpret_cast<float *>(inc_lds);   // [Z][NB]
    const int N = g.N, c = g.c, Z = g.Z, K = g.K, NT = blockDim.x;
    const int x = c - blockIdx.x, h = NB == 2 ? blockIdx.y : blockIdx.y >> 1, second = NB == 2 ? 0 : blockIdx.y & 1;
    const int lp = blockIdx.z % b.npairs, frame = blockIdx.z / b.npairs;
    const int lo = g.cyl_lo[x], hi = g.cyl_hi[x];
    if (lo == hi || (second && x == c)) return;    // at x == N/2 the second bin duplicates the first
    const int view = b.view0 + b.view_stride * lp;
    const int tid = threadIdx.x;
    const int z = tid < Z ? tid : Z - 1;    // the threads behind the last plane repeat it: no store is masked
    const int col = second ? N - x : x;     // the first bin
    const bool two = NB == 2 && x != c;
    // s1 of row y goes to A(col, y) / B(N-y, col), s2 to A(col, N-y) / B(y, col)
    float *dst = (h == 0 ? bufA : bufB) + frame * b.buf_stride + (size_t)lp * N * N * g.Z4;
    const long long step = h == 0 ? -g.Z4 : (long long)N * g.Z4;             // of s1 per row towards the edge
    const long long other = (h == 0 ? (long long)(N - 2 * x) * N : N - 2 * x) * g.Z4;   // from bin x to bin N-x
    float *o1 = dst + (h == 0 ? (size_t)col * N + c : (size_t)c * N + col) * g.Z4, *o2 = o1;   // row c
    auto put = [&](float *o, const float (&v)[NB]) __attribute__((always_inline)) {
        o[z] = v[0];
        if (two) o[other + z] = v[NB - 1];
    };
    const int ylast = lo < c - 1 ? lo : c - 1;                       // rows c-1 .. ylast are written
    if (g.nzmask[view * (c + 1) + x] == 0) {                          // masked column PJ:4236-4262
        const float zero[NB] = {};
        put(o1, zero);
        for (int y = c - 1; y >= ylast; y--) {
            o1 += step;
            o2 -= step;
            put(o1, zero);
            put(o2, zero);
        }
        return;
    }
    src += frame * b.ratio_stride;
    const int gp = src_global ? view : lp;
    const float *cp[NB];
    cp[0] = src + ((size_t)(gp * 2 + h) * N + col) * g.spp;
    if (NB == 2) cp[NB - 1] = cp[0] + (long long)(N - 2 * x) * g.spp;
    // column -> LDS (transpose PJ:1654-1693): chunks of four planes of the segments 2k and 2k-1
    const bool wide = (reinterpret_cast<uintptr_t>(src) & 15) == 0;   // columns are whole 16-byte words apart
    auto load4 = [&](const float *p) __attribute__((always_inline)) {
        if (wide) return *reinterpret_cast<const float4 *>(p);
        return make_float4(p[0], p[1], p[2], p[3]);
    };
    for (int base = tid; base < g.inc_nchunk; base += ITEMS * NT) {
        int4 it[ITEMS];
        float4 va[ITEMS][NB], vb[ITEMS][NB];
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            it[j] = make_int4(0, 0, 0, 0);
            if (base + j * NT < g.inc_nchunk) it[j] = g.inc_chunk[base + j * NT];
        }
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            if (it[j].w == 0) continue;
#pragma unroll
            for (int n = 0; n < NB; n++) {
                va[j][n] = load4(cp[n] + it[j].x);
                vb[j][n] = load4(cp[n] + it[j].y);
            }
        }
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            const int cnt = it[j].w & 0xff, k = it[j].w >> 8;
            if (cnt == 0) continue;
            if (apply_rescale) {
                const float ra = g.bp_rescale[2 * k], rb = g.bp_rescale[2 * k - 1];
#pragma unroll
                for (int n = 0; n < NB; n++) {
                    va[j][n] = mul4(va[j][n], ra);
                    vb[j][n] = mul4(vb[j][n], rb);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                Cell w;
#pragma unroll
                for (int n = 0; n < NB; n++) w.b[n] = make_float2(lane(va[j][n], i), lane(vb[j][n], i));
                if (i < cnt) W[it[j].z + i] = w;
            }
        }
    }
#pragma unroll
    for (int n = 0; n < NB; n++) {
        const float v = cp[n][g.seg_data[0] + z];
        S0[NB * z + n] = apply_rescale ? v * g.bp_rescale[0] : v;
    }
    for (int i = tid; i < 4 * K + 1; i += NT) W[g.inc_zero[i]] = Cell{};
    __syncthreads();
    // Every group's terms on the raw column: the centre voxel (PJ:4265-4285), the first row y = c-1 by direct
    // interpolation (PJ:4287-4312), and the increments from the scaled differences
    // P'(yr) = (p(yr+1) - p(yr)) * tan (PJ:4313-4335).  Reads clamped to the zero cells around the segment
    // give exactly +0 where the reference's plane ranges end.
    float sv[NB], s1[NB], s2[NB], d1[NB], d2[NB];
#pragma unroll
    for (int n = 0; n < NB; n++) sv[n] = s1[n] = s2[n] = S0[NB * z + n], d1[n] = d2[n] = 0.0f;
    for (int k = 0; k < K; k++) {
        const int4 e0 = g.inc_group[3 * k], e1 = g.inc_group[3 * k + 1], e2 = g.inc_group[3 * k + 2];
        const int gb = e0.x, yb = e0.y, yt = e0.z;
        const float tn = __int_as_float(e0.w);
        const Cell *G = W + gb;
        const int ra = clampi(z + e1.x, yb - 2, yt + 1), rb = clampi(z + e1.z, yb - 2, yt + 1);
        const int rd = clampi(z, yb - 2, yt + 1);
        const Cell w0 = G[rd], w1 = G[rd + 1], pa = G[ra], qa = G[ra + 1], pb = G[rb], qb = G[rb + 1];
        const float f1 = __int_as_float(e1.y), f2 = __int_as_float(e1.w);
        const int zs = e2.x, ze = e2.y, j = z - zs;
        const bool vj = j >= 0 && j <= ze - zs;
        const int row = e2.z + clampi(j, 0, ze > zs ? ze - zs : 0);
        const Cell q0 = G[row], q1 = G[row + 1];
#pragma unroll
        for (int n = 0; n < NB; n++) {
            sv[n] = sv[n] + (w0.b[n].x + w0.b[n].y);
            const float a1 = pa.b[n].x + f1 * (qa.b[n].x - pa.b[n].x), a2 = pa.b[n].y + f1 * (qa.b[n].y - pa.b[n].y);
            const float b1 = pb.b[n].y + f2 * (qb.b[n].y - pb.b[n].y), b2 = pb.b[n].x + f2 * (qb.b[n].x - pb.b[n].x);
            if (e2.w) {              // the row-y term first
                s1[n] = (s1[n] + a1) + b1;
                s2[n] = (s2[n] + a2) + b2;
            } else {
                s1[n] = (s1[n] + b1) + a1;
                s2[n] = (s2[n] + b2) + a2;
            }
            const float2 w = mul2(sub2(w1.b[n], w0.b[n]), tn);
            d1[n] = d1[n] + w.x;
            d2[n] = d2[n] + w.y;
            const float2 u = row <= yt ? mul2(sub2(q1.b[n], q0.b[n]), tn) : q0.b[n];   // row yt+1 is a zero cell
            d1[n] = vj ? d1[n] - u.y : d1[n];
            d2[n] = vj ? d2[n] - u.x : d2[n];
        }
    }
    put(o1, sv);
    o1 += step;
    o2 -= step;
    put(o1, s1);
    put(o2, s2);
    // The window, in place and upwards (a cell needs only itself and the two above): M(yr) = P'(yr) - P'(yr+1), M(yb-2) =
    // -P'(yb-1), M(yt) = P'(yt)
    for (int base = 0; base < g.inc_ncell; base += CELLS * NT) {
        Cell m[CELLS];
        int cell[CELLS];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < CELLS; j++) {
            const int i = base + j * NT + tid;
            cell[j] = -1;
            if (i < g.inc_ncell) {
                const int2 e = g.inc_cell[i];   // {cell | kind << 16, bits(tan)}
                const float tn = __int_as_float(e.y);
                const int kind = e.x >> 16;
                cell[j] = e.x & 0xffff;
                const Cell *r = W + cell[j];
                const Cell p0 = r[0], p1 = r[1], p2 = r[2];
#pragma unroll
                for (int n = 0; n < NB; n++) {
                    const float2 lower = mul2(sub2(p1.b[n], p0.b[n]), tn), upper = mul2(sub2(p2.b[n], p1.b[n]), tn);
                    m[j].b[n] = kind == 1 ? make_float2(-upper.x, -upper.y) : (kind == 2 ? lower : sub2(lower, upper));
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < CELLS; j++)
            if (cell[j] >= 0) W[cell[j]] = m[j];
    }
    __syncthreads();
    // rows c-2 .. lo PJ:4337-4562: breakpoints, then the running sums advance by their increments.  Stores
    // take 32-bit byte offsets from two scalar bases (a pair's half holds < 2^32 bytes); LDS addresses are
    // absolute, so the clamped offset is the address.
    char *const h0 = reinterpret_cast<char *>(dst), *const h1 = h0 + 4 * other;
    unsigned off1 = (unsigned)((o1 - dst + z) * 4), off2 = (unsigned)((o2 - dst + z) * 4);
    const unsigned step4 = (unsigned)(int)(4 * step);
    constexpr int CB = 8 * NB;   // bytes of a cell
    const int lds0 = (int)(unsigned)(uintptr_t)(__attribute__((address_space(3))) const float4 *)inc_lds;
    const int zoff = lds0 + CB * z, lane64 = tid & 63;
    const int4 *__restrict__ T = g.inc_sched;
    struct Record {
        int cf, oa, ob, lo, hi, row;
    };
    struct Cells {
        Cell a, b;
    };
    auto read = [&](const Record &r) __attribute__((always_inline)) {
        typedef float vn __attribute__((ext_vector_type(2 * NB)));
        typedef __attribute__((address_space(3))) const vn *LdsCell;
        // lo < hi always, so the clamp is max(lo, min(v, hi))
        const int ra = max(r.lo, min(zoff + r.oa, r.hi)), rb = max(r.lo, min(zoff + r.ob, r.hi));
        const vn va = *(LdsCell)(uintptr_t)(unsigned)ra, vb = *(LdsCell)(uintptr_t)(unsigned)rb;
        Cells m;
#pragma unroll
        for (int n = 0; n < NB; n++) m.a.b[n] = make_float2(va[2 * n], va[2 * n + 1]), m.b.b[n] = make_float2(vb[2 * n], vb[2 * n + 1]);
        return m;
    };
    int y = c - 2;
    auto rows_to = [&](int row) __attribute__((always_inline)) {   // rows y .. row + 1
        for (; y > row; y--) {
#pragma unroll
            for (int n = 0; n < NB; n++) s1[n] = s1[n] + d1[n], s2[n] = s2[n] + d2[n];
            off1 += step4;
            off2 -= step4;
            *reinterpret_cast<float *>(h0 + off1) = s1[0];
            *reinterpret_cast<float *>(h0 + off2) = s2[0];
            if (two) {
                *reinterpret_cast<float *>(h1 + off1) = s1[NB - 1];
                *reinterpret_cast<float *>(h1 + off2) = s2[NB - 1];
            }
        }
    };
    auto apply = [&](const Record &r, const Cells &m) __attribute__((always_inline)) {
        rows_to(r.row);
        const float cf = __int_as_float(r.cf);
#pragma unroll
        for (int n = 0; n < NB; n++) {
            // b-term (PJ:4386-4391 for rows N-y): s1 += m2*coef, s2 += m1*coef, d1 -= m2, d2 -= m1
            s1[n] = s1[n] + m.b.b[n].y * cf; d1[n] = d1[n] - m.b.b[n].y;
            s2[n] = s2[n] + m.b.b[n].x * cf; d2[n] = d2[n] - m.b.b[n].x;
            // a-term (PJ:4382-4385): s1 += m1*coef, s2 += m2*coef, d1 -= m1, d2 -= m2
            s1[n] = s1[n] + m.a.b[n].x * cf; d1[n] = d1[n] - m.a.b[n].x;
            s2[n] = s2[n] + m.a.b[n].y * cf; d2[n] = d2[n] - m.a.b[n].y;
        }
    };
    const int E = lo < c - 1 ? g.inc_count[lo] : 0;   // breakpoints of rows c-2 .. lo
    // A wave holds 64 records, one per lane, unpacked once, and takes them with readlane (scalar loads
    // would make every wait for a cell one for the records behind it too: 0.371 ms against 0.351).  The last
    // two of a batch are the first two of the next, so that a record's successors are always at hand.
    auto unpack = [&](const int4 &t) __attribute__((always_inline)) {
        return Record{t.x, (t.y >> 4) * CB, (t.z >> 4) * CB, lds0 + (t.w & 0xffff) * CB, lds0 + (int)((unsigned)t.w >> 16) * CB,
                      (t.y & 15) | ((t.z & 15) << 4)};
    };
    int4 ahead = T[lane64];
    for (int e0 = 0; e0 < E; e0 += 62) {
        const Record rec = unpack(ahead);
        ahead = T[e0 + 62 + lane64];
        auto get = [&](int i) __attribute__((always_inline)) {
            auto rl = [&](int v) __attribute__((always_inline)) { return __builtin_amdgcn_readlane(v, i); };
            return Record{rl(rec.cf), rl(rec.oa), rl(rec.ob), rl(rec.lo), rl(rec.hi), rl(rec.row)};
        };
        const int n = E - e0 < 62 ? E - e0 : 62;
        Record r0 = get(0);
        Cells m0 = read(r0);
        int i = 0;
        for (; i + 2 <= n; i += 2) {
            const Record r1 = get(i + 1);
            const Cells m1 = read(r1);
            apply(r0, m0);
            r0 = get(i + 2);
            m0 = read(r0);
            apply(r1, m1);
        }
        if (i < n) apply(r0, m0);
    }
    rows_to(lo - 1);
}

// ---------------------------------------------------------------------------
// Rotation (rotateimage2 PJ:1137-1186) of R = A + B of every pair of a
// batch, accumulated in pair order, fused with the image update
// (pt_cal_updateimage S3:2033-2056); a single pair added to an image further down.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float update1(float img, float corr, float nf, float image_max) {
    const float amin = 0.01f, amax = 100.00f;
    float cl = amin > corr ? amin : corr;   // _mm_max_ps(amin, corr)
    cl = amax < cl ? amax : cl;             // _mm_min_ps(amax, .)
    const float t = img * (cl * nf);
    return image_max < t ? image_max : t;   // _mm_min_ps(image_max, .)
}

__device__ __forceinline__ float invert1(float s, float eps1) { return fabsf(s) > eps1 ? (1.0f / s) : 0.0f; }

// The rotation of a batch by tiles: a workgroup takes ROT_TILE x ROT_TILE voxel columns and ROT_Q chunks
// of four planes of them.  Read from memory by each voxel, the eight neighbours (four of A, four of B) moved
// 308 MB a view pair of a 256 x 256 x 207 image from L2 into the L1s (33 us a pair, the same
// when both buffers lie in the last-level cache).  Here a tile's columns in the rotated frame are read
// once per pair, summed as A + B, and kept in LDS, double buffered: the next pair's columns are
// loaded while a pair is accumulated.  They lie in a box of 12 x 12 for a tile of 8 x 8; a mask says which
// of the box a voxel touches (at most 91 of the 144, 79 on average).  The tiles come from the host (rot_tiles: those
// with a FOV voxel first, strip by strip so that an XCD's share of them is compact), the boxes from rot_box_kernel.
// Nine pairs, 256 x 256 x 207: 300 -> 235 us for 0.81 GB (the FOV of A, B, image and factors once each); eight
// frames of four pairs, 128 x 128: 310 -> 259 us for 0.78 GB.
//   ROT_UPDATE  the image update with the sum;  ROT_SUM  the sum itself (rotate_image_buf into a zeroed
//   correction, PJ:1701-1725);  ROT_SENS  its inverse, and zeros outside the FOV (all tiles)
enum RotMode { ROT_UPDATE, ROT_SUM, ROT_SENS };
constexpr int ROT_Q = 8, ROT_THREADS = ROT_TILE * ROT_TILE * ROT_Q, ROT_COLS = ROT_BOX * ROT_BOX;
constexpr int ROT_LOADS = (ROT_COLS * ROT_Q + ROT_THREADS - 1) / ROT_THREADS;

template <bool KAHAN, int MODE>
__global__ void __launch_bounds__(ROT_THREADS) rot_tile_kernel(const DevGeom g, const PairBatch b,
                                                               const float4 *__restrict__ A,
                                                               const float4 *__restrict__ B, float4 *__restrict__ out,
                                                               const float4 *__restrict__ nf, int nchunks) {
    __shared__ float4 box[2][ROT_COLS * ROT_Q];
    const int N = g.N, NQ = g.NQ, tid = threadIdx.x;
    const int frame = blockIdx.y;
    A += frame * b.buf_stride / 4;
    B += frame * b.buf_stride / 4;
    out += frame * b.img_stride / 4;
    // workgroups are dealt to the XCDs in turn: each takes a run of the FOV tiles, all chunks of a tile
    const int per = (g.rot_ntiles + 7) >> 3;
    int ti, chunk;
    if ((int)blockIdx.x < 8 * per * nchunks) {
        const int i = blockIdx.x >> 3;
        ti = (blockIdx.x & 7) * per + i / nchunks;
        chunk = i % nchunks;
        if (i / nchunks >= per || ti >= g.rot_ntiles) return;
    } else {
        const int i = blockIdx.x - 8 * per * nchunks;
        ti = g.rot_ntiles + i / nchunks;
        chunk = i % nchunks;
    }
    const int tile = g.rot_tiles[ti];
    const int col = tid / ROT_Q, ql = tid % ROT_Q, q = chunk * ROT_Q + ql;
    const int x = (tile & 0xffff) * ROT_TILE + col / ROT_TILE, y = (tile >> 16) * ROT_TILE + col % ROT_TILE;
    const bool inside = x < N && y < N && q < NQ, live = inside && y >= g.cyl_lo[x] && y < g.cyl_hi[x];
    const size_t o = ((size_t)x * N + y) * NQ + q;
    if (ti >= g.rot_ntiles) {       // ROT_SENS: no FOV voxel
        if (inside) out[o] = f4(0.f);
        return;
    }
    // this thread's columns of a box (col + 64 k): their byte offsets from the box's first column
    unsigned off[ROT_LOADS];
#pragma unroll
    for (int k = 0; k < ROT_LOADS; k++) {
        const int c = col + k * (ROT_TILE * ROT_TILE);
        off[k] = (unsigned)(((c / ROT_BOX) * N + c % ROT_BOX) * NQ + q) * 16u;
    }
    const int half = __builtin_amdgcn_readfirstlane(tid >> 8);      // a wave's columns lie in one word of the mask
    const unsigned bit = q < NQ ? 1u << (col & 31) : 0u;
    const RotBox *boxes = g.rot_box + (size_t)b.view0 * g.rot_ntiles + ti;
    const float2 *rt = g.rot + ((size_t)b.view0 * N + min(x, N - 1)) * N + min(y, N - 1);
    const size_t vstride = (size_t)N * N * b.view_stride, bstride = (size_t)g.rot_ntiles * b.view_stride;
    float4 va[ROT_LOADS], vb[ROT_LOADS];
    auto load = [&](int lp, const RotBox &r) __attribute__((always_inline)) {
        const size_t base = (size_t)lp * N * N * NQ + ((size_t)r.x * N + r.y) * NQ;
        const char *pa = reinterpret_cast<const char *>(A + base), *pb = reinterpret_cast<const char *>(B + base);
#pragma unroll
        for (int k = 0; k < ROT_LOADS; k++) {
            if ((half ? r.mask[2 * k + 1] : r.mask[2 * k]) & bit) {
                va[k] = *reinterpret_cast<const float4 *>(pa + off[k]);
                vb[k] = *reinterpret_cast<const float4 *>(pb + off[k]);
            }
        }
    };
    auto store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < ROT_LOADS; k++)
            if (tid + k * ROT_THREADS < ROT_COLS * ROT_Q) box[buf][tid + k * ROT_THREADS] = add4(va[k], vb[k]);
    };
#pragma unroll
    for (int k = 0; k < ROT_LOADS; k++) va[k] = vb[k] = f4(0.f);
    float4 corr = f4(0.f), comp = f4(0.f);
    RotBox r = boxes[0];
    float2 p = rt[0];
    load(0, r);
    store(0);
    __syncthreads();
    for (int lp = 0; lp < b.npairs; lp++) {
        const bool more = lp + 1 < b.npairs;
        const RotBox rn = boxes[more ? bstride * (lp + 1) : 0];
        const float2 pn = rt[more ? vstride * (lp + 1) : 0];
        if (more) load(lp + 1, rn);
        const int xi = (int)p.x, yi = (int)p.y;
        if (live && !(xi < 0 || xi > N - 2 || yi < 0 || yi > N - 2)) {
            const float x1 = p.x - xi, y1 = p.y - yi;
            const float w1 = (1 - x1) * (1 - y1), w2 = x1 * (1 - y1), w3 = y1 * (1 - x1), w4 = y1 * x1;
            const float4 *m = &box[lp & 1][((xi - r.x) * ROT_BOX + yi - r.y) * ROT_Q + ql];
            const float4 m1 = m[0], m2 = m[ROT_BOX * ROT_Q], m3 = m[ROT_Q], m4 = m[(ROT_BOX + 1) * ROT_Q];
            const float4 v = add4(add4(mul4(m1, w1), mul4(m2, w2)), add4(mul4(m3, w3), mul4(m4, w4)));
            if (KAHAN) {
                kahan_add(corr.x, comp.x, v.x);
                kahan_add(corr.y, comp.y, v.y);
                kahan_add(corr.z, comp.z, v.z);
                kahan_add(corr.w, comp.w, v.w);
            } else {
                corr = add4(corr, v);
            }
        }
        if (more) store((lp + 1) & 1);
        r = rn;
        p = pn;
        __syncthreads();
    }
    if (MODE == ROT_UPDATE) {
        if (!live) return;
        const float4 im = out[o], n = nf[o];
        out[o] = make_float4(update1(im.x, corr.x, n.x, g.image_max), update1(im.y, corr.y, n.y, g.image_max),
                             update1(im.z, corr.z, n.z, g.image_max), update1(im.w, corr.w, n.w, g.image_max));
    } else if (MODE == ROT_SUM) {
        if (live) out[o] = corr;
    } else if (inside) {
        const int z = 4 * q;
        out[o] = make_float4(live && z + 0 < g.Z ? invert1(corr.x, g.eps1) : 0.0f, live && z + 1 < g.Z ? invert1(corr.y, g.eps1) : 0.0f,
                             live && z + 2 < g.Z ? invert1(corr.z, g.eps1) : 0.0f, live && z + 3 < g.Z ? invert1(corr.w, g.eps1) : 0.0f);
    }
}

// The boxes of the FOV tiles, a wave per (view, tile) and a lane per voxel column: the smallest box around the positions
// whose neighbours rot_tile_kernel reads, and the columns of it that it reads.  Once per context: on the host this
// took 39 of the 57 ms of creating a 256 x 256, 288-view one.
__global__ void __launch_bounds__(256) rot_box_kernel(const DevGeom g, RotBox *__restrict__ boxes, int *__restrict__ wide) {
    constexpr int WORDS = sizeof(RotBox::mask) / sizeof(unsigned);
    static_assert(ROT_TILE * ROT_TILE == 64 && ROT_BOX * ROT_BOX <= 32 * WORDS, "a lane per column, a bit per column of the box");
    __shared__ unsigned mask[4][WORDS];
    const int wv = threadIdx.x >> 6, l = threadIdx.x & 63, N = g.N, t = blockIdx.x * 4 + wv, v = blockIdx.y;
    if (l < WORDS) mask[wv][l] = 0;
    __syncthreads();
    int xi = 0, yi = 0;
    bool ok = false;
    if (t < g.rot_ntiles) {
        const int tile = g.rot_tiles[t], x = (tile & 0xffff) * ROT_TILE + l / ROT_TILE, y = (tile >> 16) * ROT_TILE + l % ROT_TILE;
        if (x < N && y >= g.cyl_lo[x] && y < g.cyl_hi[x]) {
            const float2 p = g.rot[((size_t)v * N + x) * N + y];
            xi = (int)p.x, yi = (int)p.y;
            ok = xi >= 0 && xi <= N - 2 && yi >= 0 && yi <= N - 2;
        }
    }
    int x0 = ok ? xi : N, y0 = ok ? yi : N, x1 = ok ? xi + 1 : 0, y1 = ok ? yi + 1 : 0;
    for (int o = 32; o > 0; o >>= 1) {
        x0 = min(x0, __shfl_xor(x0, o)), y0 = min(y0, __shfl_xor(y0, o));
        x1 = max(x1, __shfl_xor(x1, o)), y1 = max(y1, __shfl_xor(y1, o));
    }
    const bool fits = x1 - x0 < ROT_BOX && y1 - y0 < ROT_BOX;
    if (!fits && l == 0) atomicMax(wide, 1 + v);
    if (ok && fits) {
        const int c = (xi - x0) * ROT_BOX + yi - y0, near[4] = {c, c + 1, c + ROT_BOX, c + ROT_BOX + 1};
#pragma unroll
        for (int i = 0; i < 4; i++) atomicOr(&mask[wv][near[i] >> 5], 1u << (near[i] & 31));
    }
    __syncthreads();
    if (t >= g.rot_ntiles) return;
    RotBox &r = boxes[(size_t)v * g.rot_ntiles + t];
    if (l == 0) r.x = x0, r.y = y0;
    if (l < WORDS) r.mask[l] = mask[wv][l];
}

// ---------------------------------------------------------------------------
// PSF resolution model (convolve3d psf.cpp:441-476).  The x pass (convolvex
// psf.cpp:168-219) sums, for a FOV voxel, the taps mask = -h .. h-1 whose column
// lies inside the row's FOV and divides by their sum unless it is 0 or 1.  The
// y/z pass (convolveyz psf.cpp:324-439) sums the y taps the same way into a
// z column kept in LDS, then every plane z < z_pixels takes, with the y kernel,
// the planes z + mask inside [z_min, z_max), and is scaled by normz(z) * (1/sum
// of the y taps).  Only FOV voxels are written, as in the reference.
// ---------------------------------------------------------------------------
// Both passes were bound by their loads (a float4 per tap and output) and the z pass by its LDS reads and
// tests (a float per tap and plane).  A wave now makes PSF_R outputs that follow each other along the axis of its
// taps from one walk over their inputs, and a lane makes four planes from whole float4s of the column.
// 256 x 256 x 207, 13 taps: x pass 45 -> 30 us, y/z pass 88 -> 48 us (60 with the update).
constexpr int PSF_R = 4;

// acc[j] += in * tap and norm[j] += tap for every output first + j and input m in [m0, m1) with a tap m - (first + j)
// in [-h, h), taps ascending; at(m) is the input of position m (wave-uniform).  Four inputs at a time, the next
// four in flight; inputs and outputs the same distance apart share their tap, so it is tested and read once
// for them (an output still meets its inputs in order).
__device__ __forceinline__ void psf_tap(float f, const float4 &v, float4 &acc, float &norm) {
    norm = norm + f;
    acc = add4(acc, mul4(v, f));
}
template <typename At>
__device__ __forceinline__ void psf_walk(int first, int m0, int m1, const float *__restrict__ taps, int h, At at,
                                         float4 (&acc)[PSF_R], float (&norm)[PSF_R]) {
    float4 v[PSF_R], vn[PSF_R];
#pragma unroll
    for (int j = 0; j < PSF_R; j++) acc[j] = f4(0.f), norm[j] = 0.0f;
    if (m0 >= m1) return;
    auto load = [&](int m) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PSF_R; i++) vn[i] = at(min(m + i, m1 - 1));
    };
    load(m0);
    for (int m = m0; m < m1; m += PSF_R) {
#pragma unroll
        for (int i = 0; i < PSF_R; i++) v[i] = vn[i];
        if (m + PSF_R < m1) load(m + PSF_R);
        if (m + PSF_R <= m1) {
#pragma unroll
            for (int d = 1 - PSF_R; d < PSF_R; d++) {
                const int t = m + d - first + h;
                if (t < 0 || t >= 2 * h) continue;
                const float f = taps[t];
#pragma unroll
                for (int j = 0; j < PSF_R; j++)
                    if (j + d >= 0 && j + d < PSF_R) psf_tap(f, v[(j + d) & (PSF_R - 1)], acc[j], norm[j]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < PSF_R; i++) {
                if (m + i >= m1) break;
#pragma unroll
                for (int j = 0; j < PSF_R; j++) {
                    const int t = m + i - (first + j) + h;
                    if (t >= 0 && t < 2 * h) psf_tap(taps[t], v[i], acc[j], norm[j]);
                }
            }
        }
    }
}

// workgroup -> (line, run of PSF_R outputs along it): an XCD gets a band of lines, run after run
__device__ __forceinline__ bool psf_block(int bid, int nlines, int nruns, int &line, int &run) {
    const int per = (nlines + 7) >> 3, r = bid >> 3;
    line = (bid & 7) * per + r / nruns;
    run = r % nruns;
    return r / nruns < per && line < nlines;
}

// a workgroup's four waves take four rows y
__global__ void __launch_bounds__(256) psf_x_kernel(const DevGeom g, const float4 *__restrict__ in,
                                                    float4 *__restrict__ out, const float *__restrict__ taps, int h) {
    int yg, run;
    if (!psf_block(blockIdx.x, (g.N + 3) / 4, (g.N + PSF_R - 1) / PSF_R, yg, run)) return;
    const int q = threadIdx.x, y = yg * 4 + __builtin_amdgcn_readfirstlane(threadIdx.y), x0 = run * PSF_R;
    if (q >= g.NQ || y >= g.N) return;
    float4 acc[PSF_R];
    float norm[PSF_R];
    psf_walk(x0, max(x0 - h, g.cyl_lo[y]), min(x0 + PSF_R - 1 + h, g.cyl_hi[y]), taps, h,
             [&](int m) { return in[((size_t)m * g.N + y) * g.NQ + q]; }, acc, norm);
#pragma unroll
    for (int j = 0; j < PSF_R; j++) {
        const int x = x0 + j;
        if (x >= g.N || y < g.cyl_lo[x] || y >= g.cyl_hi[x]) continue;
        if (norm[j] != 1.0f && norm[j] != 0.0f) acc[j] = mul4(acc[j], 1.0f / norm[j]);
        out[((size_t)x * g.N + y) * g.NQ + q] = acc[j];
    }
}

// UPDATE: the blurred column is the correction of the image update of `out` (pt_cal_updateimage
// S3:2033-2056) instead of the result.  Dynamic LDS: PSF_R columns a wave with pad zero quads at each end.
template <bool UPDATE>
__global__ void __launch_bounds__(256) psf_yz_kernel(const DevGeom g, const float4 *__restrict__ in,
                                                     float4 *__restrict__ out, const float4 *__restrict__ nf,
                                                     const float *__restrict__ taps, int h, int pad,
                                                     const float *__restrict__ normz, int z_min, int z_max) {
    extern __shared__ float4 cols[];
    int x, run;
    if (!psf_block(blockIdx.x, g.N, (g.N + 4 * PSF_R - 1) / (4 * PSF_R), x, run)) return;
    const int q = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int y0 = (run * 4 + wv) * PSF_R, lo = g.cyl_lo[x], hi = g.cyl_hi[x], len = g.NQ + 2 * pad;
    float4 *col = cols + wv * PSF_R * len;
    float norm[PSF_R];
    if (q < g.NQ) {
        float4 acc[PSF_R];
        psf_walk(y0, max(y0 - h, lo), min(y0 + PSF_R - 1 + h, hi), taps, h,
                 [&](int m) { return in[((size_t)x * g.N + m) * g.NQ + q]; }, acc, norm);
        // planes outside [z_min, z_max) take no part in the z sums: zeros there (adding a zero leaves a sum
        // that began at +0 as it is)
        const int z = 4 * q;
#pragma unroll
        for (int j = 0; j < PSF_R; j++)
            col[j * len + pad + q] = make_float4(z + 0 >= z_min && z + 0 < z_max ? acc[j].x : 0.0f, z + 1 >= z_min && z + 1 < z_max ? acc[j].y : 0.0f,
                                                 z + 2 >= z_min && z + 2 < z_max ? acc[j].z : 0.0f, z + 3 >= z_min && z + 3 < z_max ? acc[j].w : 0.0f);
    }
    for (int i = q; i < 2 * pad * PSF_R; i += 64) {
        const int j = i / (2 * pad), k = i % (2 * pad);
        col[j * len + (k < pad ? k : g.NQ + k)] = f4(0.f);
    }
    __syncthreads();
    if (q >= g.NQ) return;
    // the z sums of all columns, a tap (the same for planes the same distance apart) tested and read once
    float v[PSF_R][4];
#pragma unroll
    for (int j = 0; j < PSF_R; j++) v[j][0] = v[j][1] = v[j][2] = v[j][3] = 0.0f;
    for (int i = -pad; i <= pad; i++) {
        float w[PSF_R][4];
#pragma unroll
        for (int j = 0; j < PSF_R; j++) {
            const float4 c = col[j * len + pad + q + i];
            w[j][0] = c.x, w[j][1] = c.y, w[j][2] = c.z, w[j][3] = c.w;
        }
#pragma unroll
        for (int d = -3; d < 4; d++) {
            const int t = 4 * i + d + h;
            if (t < 0 || t >= 2 * h) continue;
            const float f = taps[t];
#pragma unroll
            for (int j = 0; j < PSF_R; j++)
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (k + d >= 0 && k + d < 4) v[j][k] = v[j][k] + w[j][(k + d) & 3] * f;
        }
    }
    const float4 nz = reinterpret_cast<const float4 *>(normz)[q];
    const int z = 4 * q;
#pragma unroll
    for (int j = 0; j < PSF_R; j++) {
        const int y = y0 + j;
        if (y < lo || y >= hi) continue;
        float4 r = f4(0.f);
        if (norm[j] != 0.0f) {
            const float in1 = 1.0f / norm[j];
            r = make_float4((z + 0 < g.Z ? v[j][0] : 0.0f) * (nz.x * in1), (z + 1 < g.Z ? v[j][1] : 0.0f) * (nz.y * in1),
                            (z + 2 < g.Z ? v[j][2] : 0.0f) * (nz.z * in1), (z + 3 < g.Z ? v[j][3] : 0.0f) * (nz.w * in1));
        }
        const size_t o = ((size_t)x * g.N + y) * g.NQ + q;
        if (UPDATE) {
            const float4 im = out[o], n = nf[o];
            r = make_float4(update1(im.x, r.x, n.x, g.image_max), update1(im.y, r.y, n.y, g.image_max),
                            update1(im.z, r.z, n.z, g.image_max), update1(im.w, r.w, n.w, g.image_max));
        }
        out[o] = r;
    }
}

// ---------------------------------------------------------------------------
// Flat image files, planes [z][v][u] (SaveImage S3:4023-4035 with write_flat_image
// FIO:300-333; the -I read of Init_Image S3:3970-3993).  Image voxel (a, b) holds flat
// (v, u) = (b, a), or (a, b) when flipped; only FOV voxels are copied, the rest is 0.
// A workgroup transposes a 64 (u) x 64 (z) tile of one v through LDS, so both sides
// move whole 256-byte rows.
// ---------------------------------------------------------------------------
template <bool TO_FLAT>
__global__ void __launch_bounds__(256) flat_image_kernel(const DevGeom g, const float *__restrict__ src,
                                                         float *__restrict__ dst, int flip) {
    __shared__ float tile[64][65];
    const int v = blockIdx.y, u0 = blockIdx.x * 64, z0 = blockIdx.z * 64, N = g.N;
    const int t = threadIdx.x & 63, w = threadIdx.x >> 6;
    auto voxel = [&](int u, int &a, int &b) {
        a = flip ? v : u;
        b = flip ? u : v;
        return u < N && b >= g.cyl_lo[a] && b < g.cyl_hi[a];
    };
    if (TO_FLAT) {
        for (int i = w; i < 64; i += 4) {            // image rows: u0 + i, planes z0 + t
            int a, b;
            const int z = z0 + t;
            float val = 0.0f;
            if (voxel(u0 + i, a, b) && z < g.Z) val = src[((size_t)a * N + b) * g.Z4 + z];
            tile[i][t] = val;
        }
        __syncthreads();
        for (int i = w; i < 64; i += 4) {            // flat rows: plane z0 + i, columns u0 + t
            const int z = z0 + i, u = u0 + t;
            if (z < g.Z && u < N) dst[((size_t)z * N + v) * N + u] = tile[t][i];
        }
    } else {
        for (int i = w; i < 64; i += 4) {            // flat rows: plane z0 + i, columns u0 + t
            const int z = z0 + i, u = u0 + t;
            tile[t][i] = (z < g.Z && u < N) ? src[((size_t)z * N + v) * N + u] : 0.0f;
        }
        __syncthreads();
        for (int i = w; i < 64; i += 4) {            // image rows: u0 + i, planes z0 + t
            int a, b;
            const int z = z0 + t;
            if (u0 + i >= N || z >= g.Z4) continue;
            const bool in = voxel(u0 + i, a, b);       // (a, b) set either way; every voxel is written
            dst[((size_t)a * N + b) * g.Z4 + z] = (in && z < g.Z) ? tile[i][t] : 0.0f;
        }
    }
}

// ima += the rotation of one view pair's R = A + B: the bilinear interpolation at the position that the reference's
// rotation table gives (x, y) for the view.  Block (64, 4): x lanes over z chunks of 4.
__global__ void __launch_bounds__(256) rot_add_kernel(const DevGeom g, int view, const float4 *__restrict__ A,
                                                      const float4 *__restrict__ B, float4 *__restrict__ ima) {
    int x, yg;
    const int N = g.N, NQ = g.NQ;
    rot_block(blockIdx.x, N, (N + 3) / 4, x, yg);
    const int q = threadIdx.x, y = yg * blockDim.y + threadIdx.y;
    if (q >= NQ || y < g.cyl_lo[x] || y >= g.cyl_hi[x]) return;
    const float2 p = g.rot[((size_t)view * N + x) * N + y];
    const int xi = (int)p.x, yi = (int)p.y;
    float4 r = f4(0.f);
    if (!(xi < 0 || xi > N - 2 || yi < 0 || yi > N - 2)) {
        const float x1 = p.x - xi, y1 = p.y - yi;
        const float w1 = (1 - x1) * (1 - y1), w2 = x1 * (1 - y1), w3 = y1 * (1 - x1), w4 = y1 * x1;
        const size_t i1 = ((size_t)xi * N + yi) * NQ + q, i2 = i1 + (size_t)N * NQ;
        const float4 m1 = add4(A[i1], B[i1]), m2 = add4(A[i2], B[i2]);
        const float4 m3 = add4(A[i1 + NQ], B[i1 + NQ]), m4 = add4(A[i2 + NQ], B[i2 + NQ]);
        r = add4(r, add4(add4(mul4(m1, w1), mul4(m2, w2)), add4(mul4(m3, w3), mul4(m4, w4))));
    }
    const size_t i = ((size_t)x * N + y) * NQ + q;
    ima[i] = add4(ima[i], r);
}

// The rotated-frame buffer of one view pair, R = A + B on the FOV columns: the reference's
// imagebuf after back_proj3d_thread1 (back_proj3d_view_n1thread PJ:4162-4668), whose two
// halves it writes with = and += (the sum is the same single addition).  Like the reference,
// it leaves the pad planes z >= z_pixels as they were.
__global__ void __launch_bounds__(256) halves_sum_kernel(const DevGeom g, const float4 *__restrict__ A,
                                                         const float4 *__restrict__ B, float4 *__restrict__ out) {
    int x, yg;
    rot_block(blockIdx.x, g.N, (g.N + 3) / 4, x, yg);
    const int q = threadIdx.x, y = yg * blockDim.y + threadIdx.y;
    if (q >= g.NQ || y < g.cyl_lo[x] || y >= g.cyl_hi[x]) return;
    const size_t i = ((size_t)x * g.N + y) * g.NQ + q;
    float4 r = add4(A[i], B[i]);
    if (4 * q + 3 >= g.Z) {
        const float4 o = out[i];
        const int z = 4 * q;
        r = make_float4(z + 0 < g.Z ? r.x : o.x, z + 1 < g.Z ? r.y : o.y, z + 2 < g.Z ? r.z : o.z,
                        z + 3 < g.Z ? r.w : o.w);
    }
    out[i] = r;
}

// ---------------------------------------------------------------------------
// Layout conversions for the per-view-pair API.
// ---------------------------------------------------------------------------
// Both turn 64 x 64 tiles of (bin, padded plane) in LDS, so that either side moves whole 256-byte
// rows; one side at stride N or spp took 52 and 33 us for a view pair of 6367 x 256, now 13 and 16.
// Guard planes have no estimate and stay as they are.
constexpr int LT = 64;
// estimate plane of padded plane q, or -1 on a guard
__device__ __forceinline__ int estimate_plane(const DevGeom &g, int q, int &s) {
    s = q < g.spp ? g.pseg[q] : -1;
    return s < 0 ? -1 : g.segment_offset[s] + q - g.seg_data[s];
}

// pair-column -> estimate [2S][N], covered bins only (PJ:1397-1436).
__global__ void __launch_bounds__(256) paircol_to_estimate_kernel(const DevGeom g, int view, const float *__restrict__ pc,
                                                                  float *__restrict__ prj) {
    __shared__ float tile[LT][LT + 1];
    const int q0 = blockIdx.x * LT, c0 = blockIdx.y * LT, h = blockIdx.z, N = g.N, c = g.c;
    const int t = threadIdx.x & 63, w = threadIdx.x >> 6;
    float v[LT / 4];
#pragma unroll
    for (int i = 0; i < LT / 4; i++) {
        const int col = c0 + w + 4 * i;
        v[i] = col < N && q0 + t < g.spp ? pc[((size_t)h * N + col) * g.spp + q0 + t] : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < LT / 4; i++) tile[w + 4 * i][t] = v[i];
    __syncthreads();
    const int col = c0 + t, m = col <= c ? col : N - col;
    if (col == 0 || col >= N || g.cyl_lo[m] == 0 || g.nzmask[view * (c + 1) + m] == 0) return;
#pragma unroll
    for (int i = 0; i < LT / 4; i++) {
        int s;
        const int p = estimate_plane(g, q0 + w + 4 * i, s);
        if (p >= 0) prj[((size_t)h * g.S + p) * N + col] = tile[t][w + 4 * i];
    }
}

// estimate [2S][N] -> pair-column with the back-projection rescale; the
// estimate itself is rescaled in place as back_proj3d2 does (PJ:1496-1507).  A small scanner has few tiles and
// then the latency of a thread's loads is what counts: a thread takes four elements, and no load waits for the test of
// another (the tables are read for guards and planes past the end too, at an index inside).  Direct back
// projection of a view pair, 48 rings at 92 x 92: 33.8 -> 28.2 us (sixteen elements, each behind its tests); 104 rings
// at 256 x 256: 205 -> 200.
constexpr int EP = 4;
__global__ void __launch_bounds__(64 * LT / EP) estimate_to_paircol_kernel(const DevGeom g, float *__restrict__ prj,
                                                                         float *__restrict__ pc) {
    __shared__ float tile[LT][LT + 1];
    const int q0 = blockIdx.x * LT, c0 = blockIdx.y * LT, h = blockIdx.z, N = g.N;
    const int t = threadIdx.x & 63, w = threadIdx.x >> 6, col = c0 + t;
    constexpr int ROWS = LT / EP;     // planes (then bins) of a pass
    float v[EP], r[EP];
    int s[EP], p[EP];
#pragma unroll
    for (int i = 0; i < EP; i++) s[i] = g.pseg[min(q0 + w + ROWS * i, g.spp - 1)];
#pragma unroll
    for (int i = 0; i < EP; i++) {
        const int sg = max(s[i], 0);
        p[i] = g.segment_offset[sg] + min(q0 + w + ROWS * i, g.spp - 1) - g.seg_data[sg];
        r[i] = g.bp_rescale[sg];
    }
#pragma unroll
    for (int i = 0; i < EP; i++) {
        if (col >= N || q0 + w + ROWS * i >= g.spp) s[i] = -1;
        v[i] = 0.0f;
        if (s[i] >= 0) v[i] = prj[((size_t)h * g.S + p[i]) * N + col];
    }
#pragma unroll
    for (int i = 0; i < EP; i++) {
        const float e = v[i] * r[i];
        if (s[i] >= 0) prj[((size_t)h * g.S + p[i]) * N + col] = e;
        tile[w + ROWS * i][t] = e;
    }
    __syncthreads();
    if (q0 + t >= g.spp || g.pseg[q0 + t] < 0) return;
#pragma unroll
    for (int i = 0; i < EP; i++)
        if (c0 + w + ROWS * i < N) pc[((size_t)h * N + c0 + w + ROWS * i) * g.spp + q0 + t] = tile[t][w + ROWS * i];
}

// ---------------------------------------------------------------------------
// Elementwise kernels.
// ---------------------------------------------------------------------------
__global__ void ratio_w3_kernel(const DevGeom g, float *__restrict__ est, const float *__restrict__ add,
                                const int16_t *__restrict__ prompt, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float den = est[i] + add[i];
        const int16_t pr = prompt[i];
        if (pr == 0) est[i] = 0.0f;
        else if (den > g.eps3) est[i] = (float)pr / den;
        else est[i] = 1.0f;
    }
}

__global__ void ratio_w012_kernel(const DevGeom g, float *__restrict__ est, const float *__restrict__ data, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float e = est[i];
        est[i] = e > g.eps3 ? data[i] / e : 0.0f;
    }
}

// The voxelwise image kernels take four columns a workgroup, a wave each; a lane takes the 16 bytes of a quad at a
// time in the update, a plane at a time in the others (a workgroup per x left 3/4 of the chip's wavefronts empty: 121 us for the update of a 256 x 256 x 207 image,
// 35 us for the end of an iteration at 128 x 128).
__device__ __forceinline__ bool image_voxels(const DevGeom &g, int &x, int &y, size_t &i) {
    int yg;
    rot_block(blockIdx.x, g.N, (g.N + 3) / 4, x, yg);
    y = yg * 4 + threadIdx.y;
    i = ((size_t)x * g.N + y) * g.NQ + threadIdx.x;
    return y < g.N;
}

__global__ void __launch_bounds__(256) update_image_kernel(const DevGeom g, float4 *__restrict__ image,
                                                           float4 *__restrict__ corr, const float4 *__restrict__ nf) {
    int x, y;
    size_t i;
    if (!image_voxels(g, x, y, i) || y < g.cyl_lo[x] || y >= g.cyl_hi[x]) return;
    for (int q = threadIdx.x; q < g.NQ; q += 64, i += 64) {
        const float4 im = image[i], c = corr[i], n = nf[i];
        image[i] = make_float4(update1(im.x, c.x, n.x, g.image_max), update1(im.y, c.y, n.y, g.image_max),
                               update1(im.z, c.z, n.z, g.image_max), update1(im.w, c.w, n.w, g.image_max));
        corr[i] = f4(0.f);
    }
}

__global__ void __launch_bounds__(256) normfac_invert_kernel(const DevGeom g, const float *__restrict__ sens,
                                                             float *__restrict__ out) {
    int x, y;
    size_t i;
    if (!image_voxels(g, x, y, i) || y < g.cyl_lo[x] || y >= g.cyl_hi[x]) return;
    const size_t o = ((size_t)x * g.N + y) * g.Z4;
    for (int z = threadIdx.x; z < g.Z; z += 64) out[o + z] = invert1(sens[o + z], g.eps1);
}

__global__ void __launch_bounds__(256) init_image_kernel(const DevGeom g, float *__restrict__ image, int z_min,
                                                         int z_max) {
    int x, y;
    size_t i;
    if (!image_voxels(g, x, y, i)) return;
    const bool fov = y >= g.cyl_lo[x] && y < g.cyl_hi[x];
    for (int z = threadIdx.x; z < g.Z4; z += 64)
        image[((size_t)x * g.N + y) * g.Z4 + z] = fov && z >= z_min && z < z_max ? 1.0f : 0.0f;
}

__global__ void __launch_bounds__(256) end_iteration_kernel(const DevGeom g, float *__restrict__ image, int z_min,
                                                            int z_max) {
    int x, y;
    size_t i;
    if (!image_voxels(g, x, y, i) || y < g.cyl_lo[x] || y >= g.cyl_hi[x]) return;
    for (int z = z_min + (int)threadIdx.x; z < z_max; z += 64) {
        float *v = image + ((size_t)x * g.N + y) * g.Z4 + z;
        if ((double)*v < 1e-16) *v = 0.0f;
    }
}

__global__ void fill_u64_kernel(unsigned long long *__restrict__ p, int n) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0;
}

// ---------------------------------------------------------------------------
// Staging (prepare_osem3dw3 S3:1666-1770, prepare_norm S3:841-1003 with
// norm_ANW S3:796-821, read_flat_* FIO:110-259, sino_rebin FIO:29-74).
// ---------------------------------------------------------------------------
struct StageArgs {
    const int16_t *prompt_f;
    const float *delayed_f, *norm_f, *scatter_f, *atten_f;
    int16_t *prompt;
    float *add, *invnorm;
    const uint8_t *gapmask;   // [th][def_angles][def_elements] when rebinning the norm
    int *colmask;             // [views][N]
    // UW/AW/ANW staging (weighting 0, 1, 2; 3 = OP above): prompt_f holds short prompts or
    // trues, dataf_f a float sinogram (fully precorrected when precor); data is the output
    int weighting = 3, precor = 0;
    const float *dataf_f = nullptr;
    float *data = nullptr;
    int q_lo = 0, q_hi = 0;   // padded planes [q_lo, q_hi) of a column written by this launch
    bool wide = false;        // the outputs are 16-byte aligned
};

__device__ __forceinline__ float rebin_sum(const DevGeom &g, const float *f, size_t fplane, int v, int col) {
    const int DE = g.def_elements;
    if (g.x_rebin * g.v_rebin == 1) return f[fplane * (size_t)g.def_angles * DE + (size_t)v * DE + col];
    // sino_rebin FIO:38-66: views summed first (in place), then radial bins
    const float *p = f + fplane * (size_t)g.def_angles * DE;
    float out = 0.0f;
    for (int xr = 0; xr < g.x_rebin; xr++) {
        float s = p[(size_t)(v * g.v_rebin) * DE + col * g.x_rebin + xr];
        for (int vr = 1; vr < g.v_rebin; vr++) s += p[(size_t)(v * g.v_rebin + vr) * DE + col * g.x_rebin + xr];
        out = xr == 0 ? s : out + s;
    }
    return out;
}

__device__ __forceinline__ float rebin_norm(const DevGeom &g, const float *f, size_t fplane, int v, int col) {
    const int DE = g.def_elements;
    const float *p = f + fplane * (size_t)g.def_angles * DE;
    float out = 0.0f;
    for (int xr = 0; xr < g.x_rebin; xr++) {
        float s = p[(size_t)(v * g.v_rebin) * DE + col * g.x_rebin + xr];
        if (s > 0.0f) s = 1.0f / s;
        for (int vr = 1; vr < g.v_rebin; vr++) {
            const float a = p[(size_t)(v * g.v_rebin + vr) * DE + col * g.x_rebin + xr];
            if (a > 0.0f) s += 1.0f / a;
        }
        out = xr == 0 ? s : out + s;
    }
    if (out > 0.0f) out = 1.0f / out;
    return out;
}

// read_flat_short_proj_ori_to_float_array_theta FIO:185-224 with sino_rebin_float FIO:77-104:
// views summed as shorts (wrapping), then the bins added in float from 0
__device__ __forceinline__ float rebin_short_f(const DevGeom &g, const int16_t *f, size_t fplane, int v, int col) {
    const int DE = g.def_elements;
    const int16_t *p = f + fplane * (size_t)g.def_angles * DE;
    if (g.x_rebin * g.v_rebin == 1) return (float)p[(size_t)v * DE + col];
    float out = 0.0f;
    for (int xr = 0; xr < g.x_rebin; xr++) {
        int16_t s = p[(size_t)(v * g.v_rebin) * DE + col * g.x_rebin + xr];
        for (int vr = 1; vr < g.v_rebin; vr++)
            s = (int16_t)(s + p[(size_t)(v * g.v_rebin + vr) * DE + col * g.x_rebin + xr]);
        out = out + (float)s;
    }
    return out;
}

__device__ __forceinline__ int16_t rebin_short(const DevGeom &g, const int16_t *f, size_t fplane, int v, int col) {
    const int DE = g.def_elements;
    const int16_t *p = f + fplane * (size_t)g.def_angles * DE;
    int16_t out = 0;
    for (int xr = 0; xr < g.x_rebin; xr++) {
        int16_t s = p[(size_t)(v * g.v_rebin) * DE + col * g.x_rebin + xr];
        for (int vr = 1; vr < g.v_rebin; vr++)
            s = (int16_t)(s + p[(size_t)(v * g.v_rebin + vr) * DE + col * g.x_rebin + xr]);
        out = xr == 0 ? s : (int16_t)(out + s);
    }
    return out;
}

// Four consecutive file values.  The files may begin at any element: a load of 16 (8) bytes needs no more than the
// alignment of its values (one file 4 bytes off, 2 x 2 file bins per bin, span 9 to 128 x 128: 1.82 ms staged bin by
// bin, 0.83 this way, 0.82 with every file aligned; 256 x 256, 104 rings: 1.82, 1.41, 1.41).
typedef float file4 __attribute__((ext_vector_type(4), aligned(4)));
typedef short file4s __attribute__((ext_vector_type(4), aligned(2)));

// mask of file (view, bin) with a positive norm in some non-killed plane of segment th (FIO:158-160).  A
// thread takes four file bins (VEC: a row is a multiple of four) and eight planes at a time.
template <bool VEC>
__global__ void __launch_bounds__(256) gapmask_kernel(const DevGeom g, const float *__restrict__ norm_f,
                                                      uint8_t *__restrict__ gm, int th0) {
    constexpr int NB = VEC ? 4 : 1;
    const int th = th0 + blockIdx.y;
    const size_t fp = (size_t)g.def_angles * g.def_elements;
    const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * NB;
    if (i >= fp) return;
    const int np = g.yt[th] - g.yb[th] + 1, p1 = np - g.npskip;
    const float *f = norm_f + (size_t)g.file_seg[th] * fp + i;
    bool m[NB] = {};
    int pl = g.npskip;
    auto take = [&](int p) __attribute__((always_inline)) {
        if constexpr (VEC) {
            const file4 x = *reinterpret_cast<const file4 *>(f + (size_t)p * fp);
#pragma unroll
            for (int n = 0; n < NB; n++) m[n] |= x[n] > 0.0f;
        } else {
            m[0] |= f[(size_t)p * fp] > 0.0f;
        }
    };
    for (; pl + 8 <= p1; pl += 8) {
#pragma unroll
        for (int k = 0; k < 8; k++) take(pl + k);
    }
    for (; pl < p1; pl++) take(pl);
#pragma unroll
    for (int n = 0; n < NB; n++) gm[th * fp + i + n] = m[n];
}

// What the files hold for one bin of the staging, rebinned: the norm (0 where the plane is killed or the gap mask
// says so, 1 without a norm file), the delayed and scatter (0 without), the attenuation (1 without), and
// the prompts (OP) or the data (UW, AW, ANW).
struct StageBin {
    float nrm, d, sc, at, data;
    int16_t pr;
};

// One element of the staging: the corrected data or the additive term (o1), the sensitivity weight
// (o_inv) and, for OP, the prompt (pr).
template <bool OP>
__device__ __forceinline__ void stage_one(const DevGeom &g, const StageArgs &a, StageBin &in, float &o1, float &o_inv) {
    const float nrm = in.nrm, at = in.at;
    const float am = at < 1.0f ? 1.0f : at;
    if constexpr (!OP) {
        // prepare_osem3dw0 S3:1198-1256, w1 S3:1346-1407 and w2 S3:1505-1546; precorrected data
        // S3:1309-1323, 1410-1482, 1548-1636; then setnegative2zero simd_operation.cpp:78-96
        float t = in.data;
        if (!a.precor) {
            if (a.delayed_f) t = t - in.d;                            // readsinogram S3:1124-1131
            if (a.weighting == 0) {
                if (a.norm_f) {
                    t = t * nrm;                                      // S3:1224, 1244
                    if (a.scatter_f) t = t - nrm;                     // S3:1233: subtracts the norm buffer
                }
                if (a.atten_f) t = t * at;                            // S3:1253
            } else if (a.weighting == 1) {
                if (a.scatter_f) {
                    if (a.norm_f) t = nrm > 0.0f ? t - in.sc / nrm : 0.0f;   // S3:1380-1382
                    else t = t - in.sc;                                      // S3:1389
                }
                if (a.norm_f) t = t * nrm;                                // S3:1405
            } else if (a.scatter_f) {
                t = nrm > 0.0f ? t - in.sc / nrm : 0.0f;                  // S3:1535-1537
            }
        } else {
            if (a.weighting == 2) t = nrm > 0.0f ? t / nrm : 0.0f;        // S3:1564-1566
            if (a.weighting >= 1 && a.atten_f && at > 0.0f) t = t / at;  // divideprojection simd_operation.cpp:34
        }
        o1 = t > 0.0f ? t : 0.0f;
        if (a.weighting == 0) {                                           // norm_UW S3:756-771
            o_inv = nrm > 0.0f ? 1.0f : nrm;
            return;
        }
        if (a.weighting == 1) {                                           // norm_AW S3:774-791
            o_inv = nrm > 0.0f ? 1.0f / am : 0.0f;
            return;
        }
    } else {
        float ad = in.d * nrm;                                  // mulprojection S3:1715
        if (nrm == 0.0f) in.pr = 0;                             // S3:1720-1724
        if (a.scatter_f) ad = ad + in.sc;                       // addprojection S3:1753
        o1 = ad * at;                                           // mulprojection S3:1769
    }
    if (nrm > 0.0f) {                                           // norm_ANW S3:796-821
        const float den = nrm * am;
        o_inv = den > g.eps2 ? 1.0f / den : 0.0f;
    } else {
        o_inv = nrm;
    }
}

// The bins of one staging item from the files: NB output bins from `col` of file plane fplane, view v, by
// loads of four values (RB = 1: four bins; RB = 2: two bins of 2 x 2 file bins) or one by one (RB = 0).
template <bool OP, int RB, int NB>
__device__ __forceinline__ void stage_load(const DevGeom &g, const StageArgs &a, int th, size_t fplane, int v, int col,
                                           bool killed, StageBin (&in)[NB]) {
    const bool norm = a.norm_f && !killed;
    const int DE = g.def_elements;
#pragma unroll
    for (int n = 0; n < NB; n++) {
        in[n].nrm = a.norm_f ? 0.0f : 1.0f;
        in[n].d = in[n].sc = in[n].data = 0.0f;
        in[n].at = 1.0f;
        in[n].pr = 0;
    }
    if constexpr (RB == 0) {
        const size_t fp = (size_t)g.def_angles * DE;
        if (norm) {
            if (g.x_rebin * g.v_rebin == 1) {
                in[0].nrm = rebin_sum(g, a.norm_f, fplane, v, col);
            } else {
                in[0].nrm = rebin_norm(g, a.norm_f, fplane, v, col);
                int cnt = 0;
                for (int vr = 0; vr < g.v_rebin; vr++)
                    for (int xr = 0; xr < g.x_rebin; xr++)
                        cnt += a.gapmask[th * fp + (size_t)(v * g.v_rebin + vr) * DE + col * g.x_rebin + xr];
                if (cnt < g.x_rebin * g.v_rebin) in[0].nrm = 0.0f;
            }
        }
        if (a.delayed_f) in[0].d = rebin_sum(g, a.delayed_f, fplane, v, col);
        if (a.scatter_f) in[0].sc = rebin_sum(g, a.scatter_f, fplane, v, col);
        if (a.atten_f) in[0].at = rebin_sum(g, a.atten_f, fplane, v, col);
        if (OP) {
            if (a.prompt_f) in[0].pr = rebin_short(g, a.prompt_f, fplane, v, col);
        } else {
            in[0].data = a.prompt_f && !a.precor ? rebin_short_f(g, a.prompt_f, fplane, v, col) : rebin_sum(g, a.dataf_f, fplane, v, col);
        }
    } else {
        // rows of the item: RB file rows of four file bins each
        const size_t row = fplane * (size_t)g.def_angles * DE + (size_t)(v * RB) * DE + col * RB;
        struct F {
            file4 r[RB];
        };
        struct S {
            file4s r[RB];
        };
        auto rows = [&](const float *f) __attribute__((always_inline)) {
            F x;
#pragma unroll
            for (int k = 0; k < RB; k++) x.r[k] = *reinterpret_cast<const file4 *>(f + row + (size_t)k * DE);
            return x;
        };
        auto srows = [&](const int16_t *f) __attribute__((always_inline)) {
            S x;
#pragma unroll
            for (int k = 0; k < RB; k++) x.r[k] = *reinterpret_cast<const file4s *>(f + row + (size_t)k * DE);
            return x;
        };
        F fn{}, fd{}, fs{}, fa{}, ff{};
        S sp{};
        uchar4 gm[RB];
        if (norm) {
            fn = rows(a.norm_f);
            if (RB > 1) {
                const size_t fp = (size_t)g.def_angles * DE;
#pragma unroll
                for (int k = 0; k < RB; k++)
                    gm[k] = *reinterpret_cast<const uchar4 *>(a.gapmask + th * fp + (size_t)(v * RB + k) * DE + col * RB);
            }
        }
        if (a.delayed_f) fd = rows(a.delayed_f);
        if (a.scatter_f) fs = rows(a.scatter_f);
        if (a.atten_f) fa = rows(a.atten_f);
        const bool shorts = a.prompt_f && (OP || !a.precor);
        if (shorts) sp = srows(a.prompt_f);
        else if (!OP) ff = rows(a.dataf_f);
        // sino_rebin FIO:38-66: views summed first, then radial bins
        auto sum = [&](const F &x, int n) __attribute__((always_inline)) {
            if constexpr (RB == 1) return x.r[0][n];
            else return (x.r[0][2 * n] + x.r[1][2 * n]) + (x.r[0][2 * n + 1] + x.r[1][2 * n + 1]);
        };
        auto glane = [](const uchar4 &x, int l) { return l == 0 ? x.x : (l == 1 ? x.y : (l == 2 ? x.z : x.w)); };
#pragma unroll
        for (int n = 0; n < NB; n++) {
            if (norm) {
                if constexpr (RB == 1) {
                    in[n].nrm = fn.r[0][n];
                } else {   // rebin_norm
                    float c[2];
                    int cnt = 0;
#pragma unroll
                    for (int xr = 0; xr < 2; xr++) {
                        float t = fn.r[0][2 * n + xr];
                        const float u = fn.r[1][2 * n + xr];
                        if (t > 0.0f) t = 1.0f / t;
                        if (u > 0.0f) t += 1.0f / u;
                        c[xr] = t;
                        cnt += glane(gm[0], 2 * n + xr) + glane(gm[1], 2 * n + xr);
                    }
                    float t = c[0] + c[1];
                    if (t > 0.0f) t = 1.0f / t;
                    in[n].nrm = cnt < 4 ? 0.0f : t;
                }
            }
            if (a.delayed_f) in[n].d = sum(fd, n);
            if (a.scatter_f) in[n].sc = sum(fs, n);
            if (a.atten_f) in[n].at = sum(fa, n);
            if constexpr (OP) {
                if (shorts) {
                    if constexpr (RB == 1) in[n].pr = sp.r[0][n];
                    else in[n].pr = (int16_t)((int16_t)(sp.r[0][2 * n] + sp.r[1][2 * n]) +
                                              (int16_t)(sp.r[0][2 * n + 1] + sp.r[1][2 * n + 1]));
                }
            } else if (shorts) {   // rebin_short_f
                if constexpr (RB == 1) in[n].data = (float)sp.r[0][n];
                else in[n].data = (0.0f + (float)(int16_t)(sp.r[0][2 * n] + sp.r[1][2 * n])) +
                                  (float)(int16_t)(sp.r[0][2 * n + 1] + sp.r[1][2 * n + 1]);
            } else {
                in[n].data = sum(ff, n);
            }
        }
    }
}

// Staging of the padded planes [q_lo, q_hi) of every column (the zero guard planes among them): a workgroup
// computes a tile of 64 planes x 64 bins of one view in the files' layout (bins contiguous, 16-byte loads),
// turns it in LDS, and writes it in the pair-column layout (planes contiguous, 16-byte stores of whole 256-byte lines).
// A column's flag is set once per tile, by a look before the atomic.
//
// What bounds it: HBM (a span-3 study: 8.5 GB read, 4.8 GB written).  With 32 x 64 tiles, one element per lane, a
// flag atomic per element and the guards cleared beforehand it took 7.8 ms + 0.75 ms of clearing; now 3.7 ms, 3.6
// TB/s, where a copy of that size reaches 4.35.  Tiles of 32 bins or planes take 3.95-4.04 ms.
constexpr int STAGE_TILE = 64;

template <bool OP, int RB>
__global__ void __launch_bounds__(256) stage_kernel(const DevGeom g, StageArgs a) {
    constexpr int NB = RB == 1 ? 4 : (RB == 2 ? 2 : 1);   // bins of an item
    constexpr int LANES = STAGE_TILE / NB, ROWS = 256 / LANES;    // items across the tile's bins, planes per pass
    __shared__ float t_o1[STAGE_TILE][STAGE_TILE + 1], t_inv[STAGE_TILE][STAGE_TILE + 1];
    __shared__ int16_t t_pr[OP ? STAGE_TILE : 1][STAGE_TILE + 2];
    __shared__ int t_live[STAGE_TILE];
    const int N = g.N, V = g.views;
    const int q0 = (a.q_lo & ~63) + STAGE_TILE * (int)blockIdx.z, v = blockIdx.y, c0 = STAGE_TILE * (int)blockIdx.x;
    const int cl = NB * (threadIdx.x % LANES), r = threadIdx.x / LANES, col = c0 + cl;
    if (threadIdx.x < STAGE_TILE) t_live[threadIdx.x] = 0;
    bool live[NB] = {};
    if (col < N) {
#pragma unroll 4
        for (int pl = r; pl < STAGE_TILE; pl += ROWS) {
            const int q = q0 + pl;
            int2 e = make_int2(-1, 0);   // {file plane, segment | killed << 8}; -1: a guard plane
            if (q >= a.q_lo && q < a.q_hi) e = g.stage_plane[q];
            float o1[NB] = {}, inv[NB] = {};
            StageBin in[NB];
            if (e.x >= 0) {
                stage_load<OP, RB>(g, a, e.y & 0xff, (size_t)e.x, v, col, (e.y >> 8) != 0, in);
#pragma unroll
                for (int n = 0; n < NB; n++) {
                    live[n] |= in[n].nrm != 0.0f;
                    stage_one<OP>(g, a, in[n], o1[n], inv[n]);
                }
            } else {
#pragma unroll
                for (int n = 0; n < NB; n++) in[n].pr = 0;
            }
#pragma unroll
            for (int n = 0; n < NB; n++) {
                t_o1[cl + n][pl] = o1[n];
                t_inv[cl + n][pl] = inv[n];
                if (OP) t_pr[cl + n][pl] = in[n].pr;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NB; n++)
        if (live[n]) atomicOr(&t_live[cl + n], 1);
    const int pair = v % (V / 2), h = v / (V / 2);
    constexpr int QL = STAGE_TILE / 4, BR = 256 / QL;     // the write-out's groups of four planes, bins per pass
    const int pq = 4 * (threadIdx.x % QL), q = q0 + pq;
#pragma unroll
    for (int j = 0; j < STAGE_TILE / BR; j++) {
        const int b = threadIdx.x / QL + BR * j;
        if (c0 + b >= N) continue;
        const size_t o = ((size_t)(pair * 2 + h) * N + c0 + b) * g.spp + q;
        float x[4], w[4];
        int16_t p[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            x[k] = t_o1[b][pq + k];
            w[k] = t_inv[b][pq + k];
            p[k] = OP ? t_pr[b][pq + k] : (int16_t)0;
        }
        float *const o1 = OP ? a.add : a.data;
        if (a.wide && q >= a.q_lo && q + 4 <= a.q_hi) {
            *reinterpret_cast<float4 *>(o1 + o) = make_float4(x[0], x[1], x[2], x[3]);
            *reinterpret_cast<float4 *>(a.invnorm + o) = make_float4(w[0], w[1], w[2], w[3]);
            if (OP) *reinterpret_cast<short4 *>(a.prompt + o) = make_short4(p[0], p[1], p[2], p[3]);
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                if (q + k < a.q_lo || q + k >= a.q_hi) continue;
                o1[o + k] = x[k];
                a.invnorm[o + k] = w[k];
                if (OP) a.prompt[o + k] = p[k];
            }
        }
    }
    __syncthreads();
    if (threadIdx.x < STAGE_TILE && t_live[threadIdx.x]) {
        int *m = &a.colmask[v * N + c0 + threadIdx.x];
        if (*m == 0) atomicOr(m, 1);
    }
}

// norm_zero_mask S3:899-909
__global__ void nzmask_kernel(const DevGeom g, const int *__restrict__ colmask, int8_t *__restrict__ nz) {
    const int v = blockIdx.x, N = g.N, V = g.views;
    for (int xr = threadIdx.x; xr <= N / 2; xr += blockDim.x) {
        int8_t m = 1;
        if (xr >= 1) {
            const bool z = colmask[v * N + xr] == 0 && colmask[(v + V / 2) * N + xr] == 0 &&
                           colmask[v * N + N - xr] == 0 && colmask[(v + V / 2) * N + N - xr] == 0;
            m = z ? 0 : 1;
        }
        nz[v * (N / 2 + 1) + xr] = m;
    }
}

// ---------------------------------------------------------------------------
// FP64 reductions (log-likelihood, count normalisation) and FP16 conversion.
// Every sum runs in a fixed order or is the same in any, so results are reproducible run to run.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double block_sum_fixed(double v, double *red) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x == 0)
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) t += red[w];
    return t;   // valid in thread 0
}

__global__ void __launch_bounds__(256) ll_reduce_kernel(const LlSum *__restrict__ part, int per, double *__restrict__ out) {
    __shared__ LlSum red[4];
    const LlSum *p = part + (size_t)blockIdx.x * per;
    LlSum v{};
    for (int i = threadIdx.x; i < per; i += blockDim.x) {
        v.whole += p[i].whole;
        v.frac += p[i].frac;
        v.large += p[i].large;
    }
    const LlSum t = ll_block_sum(v, red);
    if (threadIdx.x == 0) out[blockIdx.x] = t.large + ((double)t.whole + (double)t.frac * 0x1p-46);
}

__global__ void to_half_kernel(const float *__restrict__ in, uint16_t *__restrict__ out, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        out[i] = __half_as_ushort(__float2half_rn(in[i]));
}

// The same conversion, counting the finite inputs that become +-inf ([0]) and the non-zero
// inputs that become FP16 subnormals or zero ([1]); one atomic per wave and counter.
__global__ void to_half_range_kernel(const float *__restrict__ in, uint16_t *__restrict__ out, size_t n,
                                     unsigned long long *__restrict__ counts) {
    unsigned long long over = 0, small = 0;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float x = in[i];
        const __half h = __float2half_rn(x);
        const uint16_t b = __half_as_ushort(h);
        out[i] = b;
        const bool finite_in = isfinite(x);
        over += (finite_in && (b & 0x7fffu) == 0x7c00u) ? 1 : 0;   // exponent all ones, mantissa 0
        small += (x != 0.0f && finite_in && (b & 0x7c00u) == 0) ? 1 : 0;   // exponent 0: subnormal or zero
    }
    for (int o = 32; o > 0; o >>= 1) {
        over += __shfl_xor(over, o);
        small += __shfl_xor(small, o);
    }
    if ((threadIdx.x & 63) == 0) {
        if (over) atomicAdd(&counts[0], over);
        if (small) atomicAdd(&counts[1], small);
    }
}

// moments of one pair-column block (pair p, half h, column col): sum prompt, sum w*add, sum w*est
__global__ void __launch_bounds__(256) count_moments_kernel(const DevGeom g, const int16_t *__restrict__ prompt,
                                                            const float *__restrict__ add,
                                                            const float *__restrict__ invnorm,
                                                            const float *__restrict__ est, int view0,
                                                            int view_stride, double *__restrict__ part) {
    __shared__ double red[4];
    const int col = blockIdx.x, h = blockIdx.y, lp = blockIdx.z;
    const int view = view0 + view_stride * lp;
    const size_t gbase = ((size_t)(view * 2 + h) * g.N + col) * g.spp;
    const size_t ebase = ((size_t)(lp * 2 + h) * g.N + col) * g.spp;
    double sy = 0.0, sa = 0.0, se = 0.0;
    for (int i = threadIdx.x; i < g.spp; i += blockDim.x) {
        const double w = invnorm[gbase + i];
        sy += prompt[gbase + i];
        sa += w * add[gbase + i];
        se += w * est[ebase + i];
    }
    const size_t bi = ((size_t)lp * 2 + h) * g.N + col;
    const size_t nb = (size_t)gridDim.x * gridDim.y * gridDim.z;
    double t = block_sum_fixed(sy, red);
    if (threadIdx.x == 0) part[bi] = t;
    t = block_sum_fixed(sa, red);
    if (threadIdx.x == 0) part[nb + bi] = t;
    t = block_sum_fixed(se, red);
    if (threadIdx.x == 0) part[2 * nb + bi] = t;
}

__global__ void __launch_bounds__(256) moments_reduce_kernel(const double *__restrict__ part, int nb,
                                                             double *__restrict__ out) {
    __shared__ double red[4];
    const double *p = part + (size_t)blockIdx.x * nb;
    double v = 0.0;
    for (int i = threadIdx.x; i < nb; i += blockDim.x) v += p[i];
    const double t = block_sum_fixed(v, red);
    if (threadIdx.x == 0) out[blockIdx.x] = out[blockIdx.x] + t;   // accumulates over calls
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
// Launch shape: runs of `run` middle planes per thread (1 or 3); the planes of one ray column are
// split over nsplit workgroups of 4 to 16 waves (a multiple of 4, one per SIMD each, and enough for
// a row's sampling).  The caller's shape (fp_maxt, fp_nsplit) is kept where it is given; otherwise:
// * Two rays or more per CU: runs of 3, and no more waves than the runs or the singles need, so that
//   two workgroups share a CU where the planes allow it (span 9, 8 frames of 128 x 128: 0.277 ms with
//   8 waves, 0.40 with 12; runs of 1 0.32), unless 4 waves hold the planes one by one (3 frames of a
//   30-ring scanner at 132 x 132: 0.424 ms a subset against 0.466).
// * Fewer rays: a CU holds one workgroup, and what counts is the time of a row: 16 waves, and one plane
//   per thread if that holds them (one span-9 subset at 128 x 128: 51 us, 66 with runs of 3 in 12 waves; a
//   16-ring subset: 30 against 44); below one ray per two CUs the planes are split once
//   (one view pair at span 3: 0.344 ms against 0.390).
void forward_shape(const DevGeom &g, int npf, int &run, int &nsplit, int &threads) {
    constexpr int CUS = 256;
    const long long rays = (long long)g.c * npf;
    const bool few = rays < 2 * CUS;
    nsplit = g.fp_nsplit;
    if (nsplit < 1) nsplit = 2 * rays <= CUS ? 2 : 1;
    auto waves_of = [&](int n) { return ((n + nsplit - 1) / nsplit + 63) / 64; };
    const int least = g.NQ > 32 ? 8 : 4;   // waves that sample a row
    if (g.fp_maxt > 0) run = g.fp_maxt < 3 ? 1 : 3;
    else run = waves_of(g.fp_nr[0]) <= (few ? 16 : 4) ? 1 : 3;
    const int nr = g.fp_nr[run == 3], need = (std::max(nr, g.fp_ns) + 1023) / 1024;
    if (nsplit < need) nsplit = need;
    const int waves = std::max(waves_of(nr), waves_of(g.fp_ns));
    threads = few ? 1024 : 64 * std::min(std::max((waves + 3) / 4 * 4, least), 16);
}

template <int MODE>
static hipError_t fp_launch(const DevGeom &g, const PairBatch &b, const float *image, float *out, const FpIO &io,
                            hipStream_t s) {
    int run, nsplit, threads;
    const int npf = b.npairs * b.nframes;
    forward_shape(g, npf, run, nsplit, threads);
    const long long blocks = fp_blocks(g.c, npf, nsplit);
    if (blocks > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    const float4 *im = reinterpret_cast<const float4 *>(image);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(threads), 0, s, g, b, im, out, io, nsplit);
        return hipGetLastError();
    };
    auto pick = [&](auto fast) {
        constexpr bool F = decltype(fast)::value;
        if (run == 3) return threads == 1024 ? go(fp_kernel<3, 2, MODE, F>) : go(fp_kernel<3, 1, MODE, F>);
        return threads == 1024 ? go(fp_kernel<1, 2, MODE, F>) : go(fp_kernel<1, 1, MODE, F>);
    };
    return g.fp_fast ? pick(std::true_type{}) : pick(std::false_type{});
}

hipError_t launch_forward(const DevGeom &g, const PairBatch &b, const float *image, float *out, const FpIO &io,
                          int mode, hipStream_t s) {
    switch (mode) {
        case FP_RATIO: return fp_launch<FP_RATIO>(g, b, image, out, io, s);
        case FP_RATIO16: return fp_launch<FP_RATIO16>(g, b, image, out, io, s);
        case FP_RATIO_W012: return fp_launch<FP_RATIO_W012>(g, b, image, out, io, s);
        default: return fp_launch<FP_PLAIN>(g, b, image, out, io, s);
    }
}

hipError_t launch_backproject(const DevGeom &g, const PairBatch &b, const void *src, int src_half, int src_global,
                              int apply_rescale, int kahan, float *bufA, float *bufB, hipStream_t s) {
    dim3 grid(g.N - 1, 2, b.npairs * b.nframes), block(64 * g.bp_waves);
    size_t shm = sizeof(float2) * g.bp_lds;
    const float *sf = static_cast<const float *>(src);
    const uint16_t *sh = static_cast<const uint16_t *>(src);
    if (src_half) {
        if (kahan) hipLaunchKernelGGL((bp_kernel<uint16_t, true>), grid, block, shm, s, g, b, sh, src_global, apply_rescale, g.pseg, bufA, bufB);
        else hipLaunchKernelGGL((bp_kernel<uint16_t, false>), grid, block, shm, s, g, b, sh, src_global, apply_rescale, g.pseg, bufA, bufB);
    } else {
        if (kahan) hipLaunchKernelGGL((bp_kernel<float, true>), grid, block, shm, s, g, b, sf, src_global, apply_rescale, g.pseg, bufA, bufB);
        else hipLaunchKernelGGL((bp_kernel<float, false>), grid, block, shm, s, g, b, sf, src_global, apply_rescale, g.pseg, bufA, bufB);
    }
    return hipGetLastError();
}

static dim3 rot_grid(const DevGeom &g, int nframes = 1) { return dim3(g.N * ((g.N + 3) / 4), nframes); }

hipError_t launch_backproject_incremental(const DevGeom &g, const PairBatch &b, const float *src, int src_global,
                                          int apply_rescale, float *bufA, float *bufB, hipStream_t s) {
    if (!g.inc_ok) return hipErrorInvalidValue;   // tables failed the host's window checks
    const dim3 block((g.Z + 63) / 64 * 64);
    const int npf = b.npairs * b.nframes;
    // Both bins of a ray in one workgroup share the breakpoints' work (9 pairs at 256 x 256, span 3: 0.346 ms
    // against 0.408 with a bin each); below two such workgroups per CU a bin each fills the chip better (one
    // view pair of that size, forward to image: 0.318 ms against 0.324; a 16-ring subset: 50.6 us against 51.9).
    // Two bins also take twice the LDS: where a CU's 160 KB hold a single such workgroup, its four waves are too few
    // (128 rings, 97 ring differences, 83 KB, nine pairs at 256 x 256: 1.20 ms against 0.88 with a bin each).
    if ((long long)g.c * 2 * npf >= 512 && 2 * g.inc_shm <= 160 * 1024)
        hipLaunchKernelGGL(bp_inc_kernel<2>, dim3(g.c, 2, npf), block, g.inc_shm, s, g, b, src, src_global, apply_rescale,
                           bufA, bufB);
    else
        hipLaunchKernelGGL(bp_inc_kernel<1>, dim3(g.c, 4, npf), block, g.inc_shm / 2, s, g, b, src, src_global,
                           apply_rescale, bufA, bufB);
    return hipGetLastError();
}

template <bool KAHAN, int MODE>
static void launch_rot_tile(const DevGeom &g, const PairBatch &b, const float4 *A, const float4 *B, float4 *out,
                            const float4 *nf, hipStream_t s) {
    const int nchunks = (g.NQ + ROT_Q - 1) / ROT_Q, side = (g.N + ROT_TILE - 1) / ROT_TILE;
    const int ntiles = 8 * ((g.rot_ntiles + 7) / 8) + (MODE == ROT_SENS ? side * side - g.rot_ntiles : 0);
    hipLaunchKernelGGL((rot_tile_kernel<KAHAN, MODE>), dim3(ntiles * nchunks, b.nframes), dim3(ROT_THREADS), 0, s, g, b, A, B,
                       out, nf, nchunks);
}

hipError_t launch_rot_boxes(const DevGeom &g, RotBox *boxes, int *wide, hipStream_t s) {
    if (g.rot_ntiles == 0) return hipSuccess;
    hipLaunchKernelGGL(rot_box_kernel, dim3((g.rot_ntiles + 3) / 4, g.views / 2), dim3(256), 0, s, g, boxes, wide);
    return hipGetLastError();
}

hipError_t launch_rotate_update(const DevGeom &g, const PairBatch &b, const float *bufA, const float *bufB,
                                float *image, const float *normfac, int kahan, hipStream_t s) {
    const float4 *A = reinterpret_cast<const float4 *>(bufA), *B = reinterpret_cast<const float4 *>(bufB);
    float4 *im = reinterpret_cast<float4 *>(image);
    const float4 *nf = reinterpret_cast<const float4 *>(normfac);
    if (kahan) launch_rot_tile<true, ROT_UPDATE>(g, b, A, B, im, nf, s);
    else launch_rot_tile<false, ROT_UPDATE>(g, b, A, B, im, nf, s);
    return hipGetLastError();
}

hipError_t launch_rotate_sens(const DevGeom &g, const PairBatch &b, const float *bufA, const float *bufB,
                              float *normfac_out, int kahan, hipStream_t s) {
    const float4 *A = reinterpret_cast<const float4 *>(bufA), *B = reinterpret_cast<const float4 *>(bufB);
    float4 *o = reinterpret_cast<float4 *>(normfac_out);
    if (kahan) launch_rot_tile<true, ROT_SENS>(g, b, A, B, o, nullptr, s);
    else launch_rot_tile<false, ROT_SENS>(g, b, A, B, o, nullptr, s);
    return hipGetLastError();
}

hipError_t launch_ll_reduce(const LlSum *part, int per_frame, int nframes, double *out, hipStream_t s) {
    hipLaunchKernelGGL(ll_reduce_kernel, dim3(nframes), dim3(256), 0, s, part, per_frame, out);
    return hipGetLastError();
}

hipError_t launch_to_half(const float *in, uint16_t *out, size_t n, hipStream_t s) {
    hipLaunchKernelGGL(to_half_kernel, dim3(2048), dim3(256), 0, s, in, out, n);
    return hipGetLastError();
}

hipError_t launch_to_half_range(const float *in, uint16_t *out, size_t n, unsigned long long *counts, hipStream_t s) {
    hipLaunchKernelGGL(fill_u64_kernel, dim3(1), dim3(64), 0, s, counts, 2);
    hipLaunchKernelGGL(to_half_range_kernel, dim3(2048), dim3(256), 0, s, in, out, n, counts);
    return hipGetLastError();
}

hipError_t launch_count_moments(const DevGeom &g, const int16_t *prompt, const float *add, const float *invnorm,
                                const float *est, int view0, int view_stride, int npairs, double *part,
                                double *out, hipStream_t s) {
    dim3 grid(g.N, 2, npairs);
    hipLaunchKernelGGL(count_moments_kernel, grid, dim3(256), 0, s, g, prompt, add, invnorm, est, view0, view_stride,
                       part);
    hipLaunchKernelGGL(moments_reduce_kernel, dim3(3), dim3(256), 0, s, part, (int)(grid.x * grid.y * grid.z), out);
    return hipGetLastError();
}

hipError_t launch_halves_sum(const DevGeom &g, const float *bufA, const float *bufB, float *out, hipStream_t s) {
    hipLaunchKernelGGL(halves_sum_kernel, rot_grid(g), dim3(64, 4), 0, s, g, reinterpret_cast<const float4 *>(bufA),
                       reinterpret_cast<const float4 *>(bufB), reinterpret_cast<float4 *>(out));
    return hipGetLastError();
}

hipError_t launch_rotate_add(const DevGeom &g, int view, const float *bufA, const float *bufB, float *ima,
                             hipStream_t s) {
    hipLaunchKernelGGL(rot_add_kernel, rot_grid(g), dim3(64, 4), 0, s, g, view,
                       reinterpret_cast<const float4 *>(bufA), reinterpret_cast<const float4 *>(bufB),
                       reinterpret_cast<float4 *>(ima));
    return hipGetLastError();
}

hipError_t launch_paircol_to_estimate(const DevGeom &g, int view, const float *paircol, float *prj, hipStream_t s) {
    hipLaunchKernelGGL(paircol_to_estimate_kernel, dim3((g.spp + LT - 1) / LT, (g.N + LT - 1) / LT, 2), dim3(256), 0, s, g, view, paircol, prj);
    return hipGetLastError();
}

hipError_t launch_estimate_to_paircol(const DevGeom &g, float *prj, float *paircol, hipStream_t s) {
    hipLaunchKernelGGL(estimate_to_paircol_kernel, dim3((g.spp + LT - 1) / LT, (g.N + LT - 1) / LT, 2), dim3(64 * LT / EP), 0, s, g, prj, paircol);
    return hipGetLastError();
}

hipError_t launch_ratio_w3(const DevGeom &g, float *est, const float *add, const int16_t *prompt, hipStream_t s) {
    size_t n = (size_t)2 * g.S * g.N;
    hipLaunchKernelGGL(ratio_w3_kernel, dim3(1024), dim3(256), 0, s, g, est, add, prompt, n);
    return hipGetLastError();
}

hipError_t launch_ratio_w012(const DevGeom &g, float *est, const float *data, hipStream_t s) {
    const size_t n = (size_t)2 * g.S * g.N;
    hipLaunchKernelGGL(ratio_w012_kernel, dim3(1024), dim3(256), 0, s, g, est, data, n);
    return hipGetLastError();
}

hipError_t launch_update_image(const DevGeom &g, float *image, float *corr, const float *nf, hipStream_t s) {
    hipLaunchKernelGGL(update_image_kernel, rot_grid(g), dim3(64, 4), 0, s, g, reinterpret_cast<float4 *>(image),
                       reinterpret_cast<float4 *>(corr), reinterpret_cast<const float4 *>(nf));
    return hipGetLastError();
}

hipError_t launch_rotate_sum(const DevGeom &g, const PairBatch &b, const float *bufA, const float *bufB, float *corr,
                             hipStream_t s) {
    launch_rot_tile<false, ROT_SUM>(g, b, reinterpret_cast<const float4 *>(bufA), reinterpret_cast<const float4 *>(bufB),
                                    reinterpret_cast<float4 *>(corr), nullptr, s);
    return hipGetLastError();
}

hipError_t launch_convolve3d(const DevGeom &g, const float *in, float *out, float *buf, const float *taps_x, int hx,
                             const float *taps_y, int hy, const float *normz, int z_min, int z_max,
                             const float *normfac, hipStream_t s) {
    if (g.Z4 > 256 || g.NQ > 64 || z_min < 0 || z_max > g.Z) return hipErrorInvalidValue;   // one z column per wave
    const int runs = (g.N + PSF_R - 1) / PSF_R, runs4 = (g.N + 4 * PSF_R - 1) / (4 * PSF_R);
    hipLaunchKernelGGL(psf_x_kernel, dim3(8 * (((g.N + 3) / 4 + 7) / 8) * runs), dim3(64, 4), 0, s, g,
                       reinterpret_cast<const float4 *>(in), reinterpret_cast<float4 *>(buf), taps_x, hx);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int pad = std::min((hy + 3) / 4, g.NQ);      // quads further off lie outside the column
    const size_t lds = sizeof(float4) * 4 * PSF_R * (g.NQ + 2 * pad);
    const dim3 grid(8 * ((g.N + 7) / 8) * runs4), block(64, 4);
    const float4 *b4 = reinterpret_cast<const float4 *>(buf), *nf = reinterpret_cast<const float4 *>(normfac);
    float4 *o4 = reinterpret_cast<float4 *>(out);
    if (normfac) hipLaunchKernelGGL(psf_yz_kernel<true>, grid, block, lds, s, g, b4, o4, nf, taps_y, hy, pad, normz, z_min, z_max);
    else hipLaunchKernelGGL(psf_yz_kernel<false>, grid, block, lds, s, g, b4, o4, nf, taps_y, hy, pad, normz, z_min, z_max);
    return hipGetLastError();
}

hipError_t launch_flat_image(const DevGeom &g, const float *src, float *dst, int to_flat, int flip, hipStream_t s) {
    dim3 grid((g.N + 63) / 64, g.N, (g.Z4 + 63) / 64), block(256);
    if (to_flat) hipLaunchKernelGGL(flat_image_kernel<true>, grid, block, 0, s, g, src, dst, flip);
    else hipLaunchKernelGGL(flat_image_kernel<false>, grid, block, 0, s, g, src, dst, flip);
    return hipGetLastError();
}

hipError_t launch_normfac_invert(const DevGeom &g, const float *sens, float *out, hipStream_t s) {
    hipLaunchKernelGGL(normfac_invert_kernel, rot_grid(g), dim3(64, 4), 0, s, g, sens, out);
    return hipGetLastError();
}

hipError_t launch_init_image(const DevGeom &g, float *image, int z_min, int z_max, hipStream_t s) {
    hipLaunchKernelGGL(init_image_kernel, rot_grid(g), dim3(64, 4), 0, s, g, image, z_min, z_max);
    return hipGetLastError();
}

hipError_t launch_end_iteration(const DevGeom &g, float *image, int z_min, int z_max, hipStream_t s) {
    hipLaunchKernelGGL(end_iteration_kernel, rot_grid(g), dim3(64, 4), 0, s, g, image, z_min, z_max);
    return hipGetLastError();
}

// Segments [th0, th0 + nth), which write the padded planes [q_lo, q_hi): their gap masks first when the
// norm is rebinned, then their planes; finish derives the zero-column mask from the column
// flags of every segment staged so far.
template <bool OP>
static void stage_launch(const DevGeom &g, StageArgs a, int th0, int nth, int q_lo, int q_hi, bool finish,
                         hipStream_t s) {
    a.q_lo = q_lo;
    a.q_hi = q_hi;
    auto off = [](const void *p, uintptr_t n) { return reinterpret_cast<uintptr_t>(p) % n; };
    // loads of four values: the rows of the files are whole groups of them (rebinned files may have bins to spare)
    const bool files = g.def_elements % 4 == 0;
    // 16-byte stores: columns and tiles are whole groups of four values, so what remains is where the buffers begin
    a.wide = !off(a.prompt, 8) && !off(a.add, 16) && !off(a.invnorm, 16) && !off(a.data, 16);
    const bool one = g.x_rebin == 1 && g.v_rebin == 1, two = g.x_rebin == 2 && g.v_rebin == 2;
    if (a.norm_f && !one && nth > 0) {
        const size_t fp = (size_t)g.def_angles * g.def_elements;
        const size_t n = files ? fp / 4 : fp;
        const dim3 grid((unsigned)((n + 255) / 256), nth);
        uint8_t *gm = const_cast<uint8_t *>(a.gapmask);
        if (files) hipLaunchKernelGGL(gapmask_kernel<true>, grid, dim3(256), 0, s, g, a.norm_f, gm, th0);
        else hipLaunchKernelGGL(gapmask_kernel<false>, grid, dim3(256), 0, s, g, a.norm_f, gm, th0);
    }
    if (q_hi > q_lo) {
        // the tiles of a view's rows next to each other: 3.7 ms against 4.0 with its planes next to each other
        const dim3 grid((g.N + STAGE_TILE - 1) / STAGE_TILE, g.views, (q_hi - (q_lo & ~63) + STAGE_TILE - 1) / STAGE_TILE);
        if (files && one) hipLaunchKernelGGL((stage_kernel<OP, 1>), grid, dim3(256), 0, s, g, a);
        else if (files && two) hipLaunchKernelGGL((stage_kernel<OP, 2>), grid, dim3(256), 0, s, g, a);
        else hipLaunchKernelGGL((stage_kernel<OP, 0>), grid, dim3(256), 0, s, g, a);
    }
    if (finish) hipLaunchKernelGGL(nzmask_kernel, dim3(g.views / 2), dim3(256), 0, s, g, a.colmask, g.nzmask);
}

hipError_t launch_stage(const DevGeom &g, const int16_t *prompt_f, const float *delayed_f, const float *norm_f,
                        const float *scatter_f, const float *atten_f, int16_t *prompt, float *add, float *invnorm,
                        uint8_t *gapmask, int *colmask, int th0, int nth, int q_lo, int q_hi, bool finish,
                        hipStream_t s) {
    StageArgs a{prompt_f, delayed_f, norm_f, scatter_f, atten_f, prompt, add, invnorm, gapmask, colmask};
    stage_launch<true>(g, a, th0, nth, q_lo, q_hi, finish, s);
    return hipGetLastError();
}

hipError_t launch_stage_w012(const DevGeom &g, int weighting, int precor, const int16_t *data_f16,
                             const float *data_ff, const float *delayed_f, const float *norm_f, const float *scatter_f,
                             const float *atten_f, float *data, float *invnorm, uint8_t *gapmask, int *colmask,
                             int th0, int nth, int q_lo, int q_hi, bool finish, hipStream_t s) {
    StageArgs a{data_f16, delayed_f, norm_f, scatter_f, atten_f, nullptr, nullptr, invnorm, gapmask, colmask};
    a.weighting = weighting;
    a.precor = precor;
    a.dataf_f = data_ff;
    a.data = data;
    stage_launch<false>(g, a, th0, nth, q_lo, q_hi, finish, s);
    return hipGetLastError();
}

}  // namespace hrrt
