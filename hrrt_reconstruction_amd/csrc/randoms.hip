// randoms.hip -- smoothed randoms from crystal singles (gen_delays_lib) on gfx950, and its
// C ABI (include/hrrt_randoms.h).
//
// Host side (once per context): HRRT crystal geometry, segment tables, the module-pair LUT
// (each transaxial crystal pair of 20 head pairs -> sinogram bin, 1/(d tan), closest-approach
// z), the LUT grouped by sinogram bin, and the singles iteration.
// Device side (per smoothing):
//   sings_prepare_kernel    singles [layer][ring][head][x] -> [layer][head][x][ring], so that a
//                           crystal's 104 rings are contiguous, and each column's largest magnitude
//   bin_scale_kernel        per sinogram bin, its fixed-point unit from the largest possible term
//   delays_column_kernel    per sinogram bin: every crystal pair of every LOR that
//                           lands in the bin, accumulated into the bin's column of planes in
//                           LDS (64-bit fixed point, ds_add_u64), then stored as a
//                           contiguous column
//   column_transpose_kernel [bin][plane] columns -> [plane][view][bin], 64 x 64 tiles
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/hrrt_randoms.h"
#include "delays.h"
#include "kernels.h"

using namespace hrrt_dl;

namespace {

struct Tables {    // device tables of one context
    const int4 *lor;      // [nlor] {A ring-column offset, B ring-column offset, bits(d), bits(z)}
    const int *lor_off;   // [nsino + 1] LORs of bin b: lor[lor_off[b] .. lor_off[b+1])
    const int2 *seg;      // [128] {planes from 103 to the segment's end, 8 * file offset} by segment code
    const float2 *z;      // [104] {ring z (cm), ring z in planes + 0.5}
    int nsino, nplanes, window;
};

// ---------------------------------------------------------------- kernels

// Singles [layer][ring][head][x] -> [layer][head][x][ring] (a crystal's 104 rings contiguous),
// then the largest |singles| of each such crystal column into out[NCRYS + column], which sets the
// fixed-point scale of every sinogram bin.  A workgroup turns 8 columns in LDS (one workgroup for
// all of them took 67 us, 144 take 3).  A NaN contributes nothing, as a term of value zero.
constexpr int PREP_COLS = 8;
constexpr int NCOLS = NCRYS / NY;   // 1152 crystal columns
static_assert(NX % PREP_COLS == 0, "whole column groups per head");

__global__ __launch_bounds__(256) void sings_prepare_kernel(const float *__restrict__ in, float *__restrict__ out) {
    __shared__ float v[PREP_COLS][NY];
    const int j0 = blockIdx.x * PREP_COLS;      // first column
    const int x = j0 % NX, head = (j0 / NX) % NHEADS, layer = j0 / (NX * NHEADS);
    const float *src = in + layer * XYH + head * NX + x;
    for (int i = threadIdx.x; i < PREP_COLS * NY; i += 256) {
        const float f = src[(i / PREP_COLS) * HX + i % PREP_COLS];
        v[i % PREP_COLS][i / PREP_COLS] = f == f ? f : 0.0f;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < PREP_COLS * NY; i += 256) out[j0 * NY + i] = (&v[0][0])[i];
    const int c = threadIdx.x >> 5, l = threadIdx.x & 31;
    float m = 0.0f;
    for (int ring = l; ring < NY; ring += 32) m = fmaxf(m, fabsf(v[c][ring]));
    for (int o = 16; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 32));
    if (l == 0) out[NCRYS + j0 + c] = m;
}

// Exponent k of a bin's fixed-point unit 2^-k.  A term s_A*tau*T*s_B of the bin is at most
// about m = max over its LORs of colmax(A)*colmax(B)*tau*T < 2^E, and an element of the bin
// sums at most nlor*1664 terms (104 A rings, each with at most 16 B rings on one segment and
// plane), so terms below 2^(62-bits) with 2^bits >= nlor*1664 keep every sum inside int64.
// bits is at least 11; where it is 11 and m lies just below 2^E, a term that rounds up to 2^E
// would reach 2^51, which to_fixed does not take: the unit doubles there.
__device__ inline int fixed_point_exponent(float m, int nlor) {
    int e = 0;
    float f = 0.5f;
    if (m > 0.0f && m <= 3.0e38f) f = frexpf(m, &e);
    const int bits = 32 - __clz(nlor * 1664);
    return max(min(62 - bits - e - (bits < 12 && f > 0.9999f ? 1 : 0), 127), -126);
}

// Per bin its fixed-point exponent, and 256 more where a factor or a term may not be finite.
__global__ __launch_bounds__(256) void bin_scale_kernel(Tables t, const float *__restrict__ sings, float tauftime,
                                                        int *__restrict__ scale) {
    const int bin = blockIdx.x * 256 + threadIdx.x;
    if (bin >= t.nsino) return;
    const int k0 = t.lor_off[bin], k1 = t.lor_off[bin + 1];
    float m = 0.0f, mb = 0.0f;
    bool finite = true;
    for (int k = k0; k < k1; k++) {
        const int2 L = *reinterpret_cast<const int2 *>(t.lor + k);
        const float a = sings[NCRYS + L.x / NY], b = sings[NCRYS + L.y / NY];
        m = fmaxf(m, a * b);
        mb = fmaxf(mb, b);
        finite &= a * tauftime <= 3.0e38f;      // the factor itself, and no infinite a (a NaN product counts as not finite)
    }
    m *= tauftime;
    const int k = fixed_point_exponent(m, max(k1 - k0, 1));
    finite &= m <= 3.0e38f && mb * ldexpf(1.0f, k) <= 3.0e38f;
    scale[bin] = k + (finite ? 0 : 256);
}

// Term -> int64 in units of 2^-k, rounded to nearest.  FINITE (|x| < 2^51): x + 1.5*2^52 in
// double rounds at the last bit of its mantissa, whose low bits are then the integer (3
// instructions; splitting x into two 32-bit halves takes 6 and gives the same integer).  Otherwise
// the halves, which saturate: x = hi*2^32 + lo (hi integral), x - hi*2^32 exact by one fused
// multiply-add.
template <bool FINITE>
__device__ inline unsigned long long to_fixed(float x) {
    if (FINITE) return (unsigned long long)__double_as_longlong((double)x + 0x1.8p52) - 0x4338000000000000ull;
    const float hi = floorf(x * 0x1p-32f);
    const float lo = __builtin_fmaf(hi, -0x1p32f, x);
    return ((unsigned long long)(long long)(int)hi << 32) + (unsigned long long)(unsigned)rintf(lo);
}

// |a - b| of unsigned numbers, in one instruction
__device__ inline unsigned abs_diff(unsigned a, unsigned b) {
    unsigned d;
    asm("v_sad_u32 %0, %1, %2, 0" : "=v"(d) : "v"(a), "s"(b));
    return d;
}

// COL_BINS consecutive sinogram bins per workgroup of 832 threads (13 full waves), one after the
// other.  Each crystal pair (A ring ay, B ring by) of each LOR of the bin adds s_A*tau*T*s_B to
// plane segplane(code, plane) of the bin's column, with the reference's float operations
// (compute_delays gen_delays_fromarchive.cpp:205-222):
//   plane = (int)(cay + z*dz),  seg = 0.5 + dz*d,  code = seg < 0 ? 1 - 2(int)seg : 2(int)seg
// The kernel is bound by vector instructions, then by LDS, so the pairs are laid out for few of
// both: a thread keeps A ring ay = tid mod 104 and takes the 13 B rings by = (ay + tid / 104 +
// 8 i) mod 104.  Every lane has a pair (64 + 40 B rings over two waves left 19 % idle), dz of its
// pairs stays in registers for all LORs and bins, s_A and cay too, and pairs outside the ring
// window carry a dz whose segment does not exist instead of a test.  s_B comes from LDS at a
// constant offset (each LOR's B column twice in a row, so the index needs no wrap).  Lanes of a
// wave share by - ay, so their segment entries are broadcast and their adds go to every second
// plane of a segment or two.
// An entry is {103 - first plane + 1, 8 * file offset}: a segment's planes lie symmetrically
// about 103, so |plane - 103| < that count says whether the pair has a plane.
// The column accumulates in 64-bit fixed point (ds_add_u64; LDS float atomics run about
// four times slower on gfx950), in units of 2^-k with k from the largest possible term:
// the sum is order-independent, hence reproducible, and each element differs from the
// exact sum of its float terms by at most n*2^-(k+1) for n terms before the final rounding
// to float.
// The next bin's LORs and singles are loaded while a bin is summed, and a cell is cleared by the
// thread that stores it.  Columns go bin-major into scratch and through column_transpose_kernel:
// stores straight into the plane-major output, one 4-byte request each, took 0.35 ms longer at
// span 9 (2209 planes) and 1 ms at span 3 with maxrd 25.
// 73728 bins of 6367 planes, 0.29 M LORs: 2.36 ms (2.42 with a group's segment reads behind the adds of the
// group before, 2.78 with the layout by B ring and two-halves conversion); a pair takes 17 vector
// instructions (31 before).  72 registers, for the 7 waves a SIMD of two workgroups per CU.
constexpr int COL_ROWS = 8, COL_STEPS = NY / COL_ROWS, COL_THREADS = NY * COL_ROWS;
static_assert(COL_STEPS * COL_ROWS == NY && COL_THREADS % 64 == 0, "rings split evenly");
constexpr int COL_BINS = 8;     // bins per workgroup (the bin count is a multiple of 8)
// steps 4..8 (B - A ring differences of 32 to 72, modulo 104) lie outside ring windows below 32
constexpr int MID_LO = 4, MID_HI = 9, MID_WINDOW = 32;
constexpr float NO_PAIR = 1e38f;
constexpr int MID_PLANE = NY - 1;   // 103
// Planes of the LDS column (span 3 at maxrd up to 68 has 6367).
constexpr int COLUMN_PLANES = 6400;

template <int NI>
struct Group {      // pairs between their two stages
    static constexpr int N = NI;
    unsigned plane[NI];
    int2 ent[NI];
    float b[NI];
};

__global__ __launch_bounds__(COL_THREADS, 7) void delays_column_kernel(Tables t, const float *__restrict__ sings,
                                                                    const int *__restrict__ scale, float tauftime,
                                                                    float *__restrict__ cols, int cstride) {
    __shared__ int2 seg[128];
    // the bin's column of planes (a static array: its adds take their LDS base as an immediate)
    __shared__ unsigned long long col[COLUMN_PLANES];
    __shared__ float sB[COL_ROWS][2 * NY], sA[COL_ROWS][NY];
    __shared__ float2 sL[COL_ROWS];
    // workgroups are dealt to the 8 XCDs in turn: XCD x gets bins [x*nsino/8, (x+1)*nsino/8)
    const int per = t.nsino >> 3, wg = blockIdx.x >> 3, tid = threadIdx.x;
    const int end = (blockIdx.x & 7) * per + min(per, (wg + 1) * COL_BINS);
    const int first = (blockIdx.x & 7) * per + wg * COL_BINS;
    for (int i = tid; i < t.nplanes; i += COL_THREADS) col[i] = 0ull;
    if (tid < 128) seg[tid] = t.seg[tid];
    const int row = tid / NY, ay = tid % NY;
    const float2 za = t.z[ay];
    float dz[COL_STEPS];
#pragma unroll
    for (int i = 0; i < COL_STEPS; i++) {
        int by = ay + row + COL_ROWS * i;
        by -= by >= NY ? NY : 0;
        dz[i] = abs(by - ay) <= t.window ? t.z[by].x - za.x : NO_PAIR;
    }
    const bool mid = t.window >= MID_WINDOW;
    // this thread's LOR of the first eight of a bin, and its singles
    int k0 = t.lor_off[first], k1 = t.lor_off[first + 1], n1 = t.lor_off[min(first + 2, end)], sc = scale[first];
    int4 L = make_int4(0, 0, 0, 0);
    float a = 0.0f, b = 0.0f;
    auto load_lor = [&](int k, int kend) { if (k < kend) L = t.lor[k]; };
    auto load_sings = [&](int k, int kend) { if (k < kend) a = sings[L.x + ay], b = sings[L.y + ay]; };
    load_lor(k0 + row, k1);
    load_sings(k0 + row, k1);
    for (int bin = first; bin < end; bin++) {
        const int kexp = sc >= 128 ? sc - 256 : sc;
        const float up = ldexpf(1.0f, kexp);
        // the next bin's LORs are [k1, n1); what the bin after it needs is on its way (beyond the last bin: none)
        const int n0 = k1, n2 = t.lor_off[min(bin + 3, end)], sc_next = scale[min(bin + 1, end - 1)];
        auto sum = [&](auto finite) __attribute__((always_inline)) {
            for (int kb = k0; kb < k1; kb += COL_ROWS) {
                if (kb > k0) {
                    load_lor(kb + row, k1);
                    load_sings(kb + row, k1);
                    __syncthreads();
                }
                // the term s_B*(s_A*tau*T) scaled by 2^k: scaling s_B first is exact and rounds the
                // same product (a power of two commutes with rounding)
                sB[row][ay] = sB[row][NY + ay] = b * up;
                sA[row][ay] = a * tauftime;
                if (ay == 0) sL[row] = make_float2(__int_as_float(L.z), __int_as_float(L.w));
                __syncthreads();
                if (kb + COL_ROWS >= k1) load_lor(n0 + row, n1);
                const int n = min(COL_ROWS, k1 - kb);
                for (int k = 0; k < n; k++) {
                    const float sd = sL[k].x, sz = sL[k].y, awt = sA[k][ay];
                    const float *bk = &sB[k][ay + row];
                    // A pair in two stages: its plane, segment entry and B single, then its add.  A group's reads are
                    // issued before the adds of the group before it, since LDS answers in order.
                    auto first_stage = [&](auto i0, auto &g) __attribute__((always_inline)) {
                        constexpr int I0 = decltype(i0)::value;
#pragma unroll
                        for (int i = 0; i < g.N; i++) {
                            const float dzi = dz[I0 + i];
                            g.plane[i] = (unsigned)(int)(za.y + sz * dzi);
                            const float s = 0.5f + dzi * sd;
                            const unsigned j = (unsigned)fminf(fabsf(s), 63.5f);
                            // byte offset of entry 2 |(int)s| + (s < 0)
                            const unsigned e8 = __builtin_amdgcn_alignbit(j, __float_as_uint(s), 28) & ~7u;
                            g.ent[i] = *reinterpret_cast<const int2 *>(reinterpret_cast<const char *>(seg) + e8);
                            g.b[i] = bk[COL_ROWS * (I0 + i)];
                        }
                        asm volatile("" ::: "memory");
                    };
                    auto second_stage = [&](auto &g) __attribute__((always_inline)) {
                        constexpr int NI = std::remove_reference_t<decltype(g)>::N;
                        bool ok[NI];
                        int idx8[NI];
                        unsigned long long q[NI];
#pragma unroll
                        for (int i = 0; i < NI; i++) {
                            ok[i] = abs_diff(g.plane[i], MID_PLANE) < (unsigned)g.ent[i].x;
                            idx8[i] = (int)(g.plane[i] << 3) + g.ent[i].y;
                            q[i] = to_fixed<decltype(finite)::value>(g.b[i] * awt);
                        }
                        // whole groups before their adds, or each add would wait for its own chain
#pragma unroll
                        for (int i = 0; i < NI; i++) asm volatile("" : "+v"(idx8[i]), "+v"(q[i]));
#pragma unroll
                        for (int i = 0; i < NI; i++)
                            if (ok[i]) atomicAdd(reinterpret_cast<unsigned long long *>(reinterpret_cast<char *>(col) + idx8[i]), q[i]);
                        asm volatile("" ::: "memory");
                    };
                    Group<2> ga, gb, gd, ge, gf;
                    Group<3> gc;
                    first_stage(std::integral_constant<int, 0>(), ga);
                    first_stage(std::integral_constant<int, 2>(), gb);
                    second_stage(ga);
                    if (mid) {
                        first_stage(std::integral_constant<int, MID_LO>(), gc);
                        second_stage(gb);
                        first_stage(std::integral_constant<int, MID_LO + 3>(), gd);
                        second_stage(gc);
                        first_stage(std::integral_constant<int, MID_HI>(), ge);
                        second_stage(gd);
                    } else {
                        first_stage(std::integral_constant<int, MID_HI>(), ge);
                        second_stage(gb);
                    }
                    first_stage(std::integral_constant<int, MID_HI + 2>(), gf);
                    second_stage(ge);
                    second_stage(gf);
                }
            }
        };
        if (k0 == k1) load_lor(n0 + row, n1);
        else if (sc < 128) sum(std::true_type());
        else sum(std::false_type());
        load_sings(n0 + row, n1);       // the LOR has arrived; these arrive while the column is stored
        __syncthreads();
        const double down = ldexp(1.0, -kexp);
        for (int i = tid; i < t.nplanes; i += COL_THREADS) {
            cols[(size_t)bin * cstride + i] = (float)((double)(long long)col[i] * down);
            col[i] = 0ull;
        }
        k0 = n0, k1 = n1, n1 = n2, sc = sc_next;
    }
}

// [nsino][cstride] columns -> [nplanes][nsino]; 64 x 64 tiles through LDS, 256 threads (16
// elements each), TT tiles along the planes per workgroup with the next tile's loads in flight
// while the current one is stored.  A column stride of whole 256-byte lines keeps every tile
// row's read on line boundaries.
constexpr int TT = 4;

__global__ __launch_bounds__(256) void column_transpose_kernel(const float *__restrict__ cols, float *__restrict__ out,
                                                               int nsino, int nplanes, int cstride) {
    __shared__ float tile[2][64][65];
    const int b0 = blockIdx.y * 64, pt0 = blockIdx.x * TT * 64;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    float v[16];
    auto load = [&](int p0) {
#pragma unroll
        for (int k = 0; k < 16; k++) {
            const int b = b0 + ty + 4 * k, p = p0 + tx;
            v[k] = (b < nsino && p < nplanes) ? cols[(size_t)b * cstride + p] : 0.0f;
        }
    };
    load(pt0);
    for (int i = 0; i < TT; i++) {
        const int p0 = pt0 + 64 * i;
        if (p0 >= nplanes) break;
        float(*T)[65] = tile[i & 1];
#pragma unroll
        for (int k = 0; k < 16; k++) T[ty + 4 * k][tx] = v[k];
        __syncthreads();
        if (i + 1 < TT && p0 + 64 < nplanes) load(p0 + 64);
#pragma unroll
        for (int k = 0; k < 16; k++) {
            const int p = p0 + ty + 4 * k, b = b0 + tx;
            if (p < nplanes && b < nsino) out[(size_t)p * nsino + b] = T[tx][ty + 4 * k];
        }
    }
}

}  // namespace

namespace {

int make_tables(hrrt_delays &c, const hrrt_delays_params &p, std::string &err) {
    if (p.span != 3 && p.span != 9) return err = "span must be 3 or 9", HRRT_ERR_ARG;
    if (p.maxrd < 0 || p.maxrd > NY - 1) return err = "maxrd out of range", HRRT_ERR_ARG;
    if (p.lr_type < 0 || p.lr_type > 2) return err = "lr_type must be 0, 1 or 2", HRRT_ERR_ARG;
    c.span = p.span;
    c.maxrd = p.maxrd;
    c.lr_type = p.lr_type;
    c.tau = p.tau > 0.0f ? p.tau : 6.0e-9f;
    // init_geometry_hrrt geometry_info.cpp:169-221
    const float pitch = p.pitch > 0.0f ? p.pitch : 0.24375f;
    const float diam = p.diam > 0.0f ? p.diam : 46.9f;
    c.depth = p.thick > 0.0f ? p.thick : 1.0f;
    for (int i = 0; i < NHEADS; i++) {
        c.sin_head[i] = std::sin(i * 2.0 * M_PI / NHEADS);
        c.cos_head[i] = std::cos(i * 2.0 * M_PI / NHEADS);
    }
    c.crystal_radius = diam / 2.0;
    if (c.lr_type == 0) {
        c.nprojs = 256, c.nviews = 288, c.binsize = pitch / 2.0, c.plane_sep = pitch / 2.0;
    } else if (c.lr_type == 1) {
        c.nprojs = 160, c.nviews = 144, c.binsize = 0.2f, c.plane_sep = pitch;
    } else {
        c.nprojs = 128, c.nviews = 144, c.binsize = pitch, c.plane_sep = pitch;
    }
    c.nsino = c.nprojs * c.nviews;
    // init_segment_info segment_info_fromarchive.cpp:118-141: planes of the span; the plane
    // map is span 3, with span-9 file offsets through the conversion table
    int z0[SEGMAP], zmax[SEGMAP], off[SEGMAP];
    c.nsegs = 2 * (c.maxrd / 3) + 1;
    if (c.nsegs > 45) return err = "maxrd above 68 leaves the segment tables", HRRT_ERR_ARG;
    c.nplanes = c.segments(c.span, z0, zmax, off);
    c.segments(3, c.segz0, c.segzmax, c.segoff);
    if (c.span == 9) {
        const int n9 = 2 * (c.maxrd / 9) + 1;
        for (int i = 0; i < c.nsegs; i++) {
            if (kS3toS9[i] >= n9) return err = "span-9 segment table too short for maxrd", HRRT_ERR_ARG;
            c.segoff[i] = off[kS3toS9[i]];
        }
    }
    c.d_tan_theta = 3 * c.plane_sep / c.crystal_radius;
    return HRRT_OK;
}

// init_sol lor_sinogram_map.cpp:141-209: the LUT and the ring z tables from the geometry
void compute_lut(hrrt_delays &c) {
    c.lut.assign((size_t)(NMP + 1) * NXD * NXD, Sol{-1, 0.0f, 0.0f});
    for (int mp = 1; mp <= NMP; mp++) {
        for (int al = 0; al < NDOIS; al++)
            for (int ax = 0; ax < NX; ax++) {
                float pa[3];
                c.crystal(kMpairs[mp][0], al, ax, 0, pa);
                Sol *row = &c.lut[((size_t)mp * NXD + ax + NX * al) * NXD];
                for (int bl = 0; bl < NDOIS; bl++)
                    for (int bx = 0; bx < NX; bx++) {
                        float pb[3];
                        c.crystal(kMpairs[mp][1], bl, bx, 0, pb);
                        row[bx + NX * bl] = c.lor(pa, pb);
                    }
            }
    }
    for (int i = 0; i < NY; i++) {
        float pos[3];
        c.crystal(0, 0, 0, i, pos);
        c.zpos[i] = pos[2];
        c.zpos2[i] = (float)((double)pos[2] / c.plane_sep + 0.5);
    }
}

// init_lut_sol lor_sinogram_map.cpp:224-303
int read_lut(hrrt_delays &c, const char *path, std::string &err) {
    FILE *f = fopen(path, "rb");
    if (!f) return err = std::string("cannot open LUT file ") + path, HRRT_ERR_ARG;
    c.lut.assign((size_t)(NMP + 1) * NXD * NXD, Sol{-1, 0.0f, 0.0f});
    const size_t n = (size_t)NMP * NXD * NXD;
    bool ok = fread(&c.lut[(size_t)NXD * NXD], sizeof(Sol), n, f) == n;
    ok = ok && fread(c.zpos, sizeof(float), NY, f) == (size_t)NY && fread(c.zpos2, sizeof(float), NY, f) == (size_t)NY;
    fclose(f);
    if (!ok) return err = std::string("short LUT file ") + path, HRRT_ERR_ARG;
    return HRRT_OK;
}



// Group the valid LORs by sinogram bin (host tables; uploaded by the first smoothing).
int group_lors(hrrt_delays &c) {
    std::vector<int> &count = c.h_lor_off;
    count.assign(c.nsino + 1, 0);
    for (int mp = 1; mp <= NMP; mp++)
        for (int i = 0; i < NXD * NXD; i++) {
            const Sol &s = c.lut[(size_t)mp * NXD * NXD + i];
            if (s.nsino < -1 || s.nsino >= c.nsino)
                return hrrt_dl::fail(HRRT_ERR_ARG, "LUT bin outside the sinogram (LUT built for another LR type?)");
            if (s.nsino >= 0) count[s.nsino + 1]++;
        }
    for (int b = 0; b < c.nsino; b++) count[b + 1] += count[b];
    c.nlor = count[c.nsino];
    std::vector<int4> &lor = c.h_lor;
    lor.assign(std::max(c.nlor, 1), make_int4(0, 0, 0, 0));
    std::vector<int> fill(count.begin(), count.end() - 1);
    // per A ring, the B rings inside |ay - by| < maxrd + 6 (gen_delays_fromarchive.cpp:175-184)
    const int window = c.maxrd + 5;
    long long ring_pairs = 0;
    for (int ay = 0; ay < NY; ay++) ring_pairs += std::min(NY - 1, ay + window) - std::max(0, ay - window) + 1;
    c.pairs_full = 0;
    for (int mp = 1; mp <= NMP; mp++) {
        const int ahead = kMpairs[mp][0], bhead = kMpairs[mp][1];
        for (int axx = 0; axx < NXD; axx++)
            for (int bxx = 0; bxx < NXD; bxx++) {
                const Sol &s = c.lut[((size_t)mp * NXD + axx) * NXD + bxx];
                if (s.nsino < 0) continue;
                const int al = axx / NX, ax = axx % NX, bl = bxx / NX, bx = bxx % NX;
                int4 e;
                e.x = ((al * NHEADS + ahead) * NX + ax) * NY;
                e.y = ((bl * NHEADS + bhead) * NX + bx) * NY;
                // a slope of zero (a record of zeros in a LUT file) becomes one that leaves 0.5 + dz*d at
                // 0.5 for every ring difference but not for a pair outside the window; so does one that is no
                // number, which names segment 0 too
                const float d = std::fabs(s.d) >= 1e-30f ? s.d : std::copysign(1e-30f, s.d);
                memcpy(&e.z, &d, 4);
                memcpy(&e.w, &s.z, 4);
                lor[fill[s.nsino]++] = e;
                c.pairs_full += ring_pairs;
            }
    }
    if (c.nplanes > COLUMN_PLANES) return hrrt_dl::fail(HRRT_ERR_UNSUPPORTED, "more sinogram planes than the LDS column holds");
    if (c.nsino % 8) return hrrt_dl::fail(HRRT_ERR_UNSUPPORTED, "sinogram bins not a multiple of 8");
    return HRRT_OK;
}

// Head totals of the singles (compute_drate gen_delays_lib.cpp:168-176): layer, x, ring order.
void head_sums(const float *srate, float *hsum) {
    for (int head = 0; head < NHEADS; head++) {
        float s = 0.0f;
        for (int layer = 0; layer < NDOIS; layer++)
            for (int cx = 0; cx < NX; cx++)
                for (int cy = 0; cy < NY; cy++) s += srate[NX * head + cx + HX * cy + XYH * layer];
        hsum[head] = s;
    }
}

// Sum over the five heads in coincidence with `head` (gen_delays_lib.cpp:180-186).
float fan_sum(const float *hsum, int head) {
    float s = 0.0f;
    for (int j = 0; j < 5; j++) s += hsum[(head + j + 2) % NHEADS];
    return s;
}

}  // namespace

int hrrt_dl::fail(int code, const std::string &msg) { return hrrt::set_last_error(code, msg.c_str()); }

// Device copies of the tables, on the current device, at the first smoothing.
int hrrt_dl::upload(hrrt_delays &c) {
    if (c.uploaded) return HRRT_OK;
    const std::vector<int4> &lor = c.h_lor;
    const std::vector<int> &count = c.h_lor_off;
    // segment entries by e = 2*(int)seg + (seg < 0) + 64 (the kernel's index): e - 64 even and
    // >= 0 is code e - 64, odd and <= 1 is code 2 - (e - 64); {first plane, last plane, offset}
    std::vector<int2> seg(128, make_int2(0x7fff, 0));            // first 32767 > last 0: no plane
    for (int e = 0; e < 128; e++) {
        const int ee = e - 64;
        const int code = (ee >= 0 && ee % 2 == 0) ? ee : ((ee <= 1 && (ee & 1)) ? 2 - ee : -1);
        if (code >= 0 && code < c.nsegs) seg[e] = make_int2(c.segz0[code] | (c.segzmax[code] << 16), c.segoff[code]);
    }
    std::vector<int2> seg_col(128, make_int2(0, 0));   // no plane
    for (int code = 0; code < c.nsegs; code++) seg_col[code] = make_int2(MID_PLANE + 1 - c.segz0[code], 8 * c.segoff[code]);
    std::vector<float2> z(NY);
    for (int i = 0; i < NY; i++) z[i] = make_float2(c.zpos[i], c.zpos2[i]);
    int dev = -1;
    DTRY(hipGetDevice(&dev));
    if (c.d_lor && dev != c.device) return hrrt_dl::fail(HRRT_ERR_ARG, "context tables live on another device");
    c.device = dev;
    auto table = [](auto *&dst, size_t bytes, const void *src) {     // a table that an earlier, failed upload left is kept
        const hipError_t e = dst ? hipSuccess : hipMalloc(&dst, bytes);
        return e == hipSuccess && src ? hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice) : e;
    };
    DTRY(table(c.d_lor, sizeof(int4) * lor.size(), lor.data()));
    DTRY(table(c.d_lor_off, sizeof(int) * count.size(), count.data()));
    DTRY(table(c.d_seg, sizeof(int2) * 128, seg.data()));
    DTRY(table(c.d_seg_col, sizeof(int2) * 128, seg_col.data()));
    DTRY(table(c.d_scale, sizeof(int) * c.nsino, nullptr));
    DTRY(table(c.d_z, sizeof(float2) * NY, z.data()));
    DTRY(table(c.d_sings, sizeof(float) * (NCRYS + NCOLS), nullptr));
    c.uploaded = true;
    return HRRT_OK;
}

// ---------------------------------------------------------------- C ABI

extern "C" int hrrt_delays_create(const hrrt_delays_params *params, hrrt_delays **out) {
    if (!params || !out) return hrrt_dl::fail(HRRT_ERR_ARG, "null argument");
    *out = nullptr;
    hrrt_delays *c = new (std::nothrow) hrrt_delays();
    if (!c) return hrrt_dl::fail(HRRT_ERR_NOMEM, "host allocation failed");
    std::string err;
    int r = make_tables(*c, *params, err);
    if (r == HRRT_OK) {
        if (params->lut_file) r = read_lut(*c, params->lut_file, err);
        else compute_lut(*c);
    }
    if (r != HRRT_OK) {
        delete c;
        return hrrt_dl::fail(r, err);
    }
    if ((r = group_lors(*c)) != HRRT_OK) {
        delete c;
        return r;
    }
    *out = c;
    return HRRT_OK;
}

extern "C" void hrrt_delays_destroy(hrrt_delays *c) {
    if (!c) return;
    for (void *p : {(void *)c->d_lor, (void *)c->d_lor_off, (void *)c->d_seg, (void *)c->d_seg_col, (void *)c->d_scale, (void *)c->d_z, (void *)c->d_sings,
                    (void *)c->d_cols, (void *)c->d_sol, (void *)c->d_lm_keys, (void *)c->d_lm_part, (void *)c->d_lm_tiles,
                    (void *)c->d_lm_coin_seg, (void *)c->d_lm_coin_cnt, (void *)c->d_lm_coin_part, (void *)c->d_lm_chunks,
                    (void *)c->d_lm_stats})
        if (p) (void)hipFree(p);
    if (c->h_lm_stats) (void)hipHostFree(c->h_lm_stats);
    delete c;
}

extern "C" int hrrt_delays_get_dims(const hrrt_delays *c, int *nprojs, int *nviews, int *nplanes, int *nsegs,
                                    long long *pairs_full) {
    if (!c) return hrrt_dl::fail(HRRT_ERR_ARG, "null context");
    if (nprojs) *nprojs = c->nprojs;
    if (nviews) *nviews = c->nviews;
    if (nplanes) *nplanes = c->nplanes;
    if (nsegs) *nsegs = c->nsegs;
    if (pairs_full) *pairs_full = c->pairs_full;
    return HRRT_OK;
}

extern "C" int hrrt_delays_get_lut(const hrrt_delays *c, int mp, int32_t *nsino, float *d, float *z) {
    if (!c) return hrrt_dl::fail(HRRT_ERR_ARG, "null context");
    if (mp < 1 || mp > NMP) return hrrt_dl::fail(HRRT_ERR_ARG, "module pair must be 1..20");
    const Sol *s = &c->lut[(size_t)mp * NXD * NXD];
    for (int i = 0; i < NXD * NXD; i++) {
        if (nsino) nsino[i] = s[i].nsino;
        if (d) d[i] = s[i].d;
        if (z) z[i] = s[i].z;
    }
    return HRRT_OK;
}

// save_lut_sol lor_sinogram_map.cpp:305-340
extern "C" int hrrt_delays_save_lut(const hrrt_delays *c, const char *path) {
    if (!c || !path) return hrrt_dl::fail(HRRT_ERR_ARG, "null argument");
    FILE *f = fopen(path, "wb");
    if (!f) return hrrt_dl::fail(HRRT_ERR_ARG, std::string("cannot create ") + path);
    const size_t n = (size_t)NMP * NXD * NXD;
    bool ok = fwrite(&c->lut[(size_t)NXD * NXD], sizeof(Sol), n, f) == n;
    ok = ok && fwrite(c->zpos, sizeof(float), NY, f) == (size_t)NY && fwrite(c->zpos2, sizeof(float), NY, f) == (size_t)NY;
    ok = (fclose(f) == 0) && ok;
    return ok ? HRRT_OK : hrrt_dl::fail(HRRT_ERR_ARG, std::string("write failed: ") + path);
}

// compute_csings_from_drates gen_delays_lib.cpp:254-271 with compute_initial_srate (:233-241),
// compute_drate (:162-196), errtotal (:244-252) and estimate_srate (:198-230).  The error
// sum is 64-bit (the reference's int overflows on large errors; only its zero test matters).
extern "C" int hrrt_delays_singles(const hrrt_delays *c, const int32_t *coins, float scan_duration, float *singles,
                                   int *niter) {
    if (!c || !coins || !singles) return hrrt_dl::fail(HRRT_ERR_ARG, "null argument");
    const float dt = scan_duration > 0.0f ? scan_duration : 1.0f, tau = c->tau;
    const int32_t *dcoins = coins + NCRYS;
    std::vector<float> drates(NCRYS), xrates(NCRYS);
    float dtotal = 0.0f;
    for (int i = 0; i < NCRYS; i++) drates[i] = (float)dcoins[i] / dt;
    for (int i = 0; i < NCRYS; i++) dtotal += drates[i];
    const float stotal = (float)(8.0 * std::sqrt((double)dtotal / (40. * (double)tau)));
    for (int i = 0; i < NCRYS; i++) singles[i] = drates[i] * stotal / dtotal;
    float hsum[NHEADS];
    int iter;
    for (iter = 0; iter < 100; iter++) {
        head_sums(singles, hsum);
        long long err = 0;
        for (int head = 0; head < NHEADS; head++) {
            const float fan = fan_sum(hsum, head);
            for (int layer = 0; layer < NDOIS; layer++)
                for (int cx = 0; cx < NX; cx++)
                    for (int cy = 0; cy < NY; cy++) {
                        const int i = NX * head + cx + HX * cy + XYH * layer;
                        xrates[i] = singles[i] * tau * fan;
                    }
        }
        for (int i = 0; i < NCRYS; i++) {
            const long long e = (int)((double)dcoins[i] - (0.5 + (double)(xrates[i] * dt)));
            err += e * e;
        }
        if (iter && err == 0) break;
        head_sums(singles, hsum);
        for (int head = 0; head < NHEADS; head++) {
            const float fan = fan_sum(hsum, head);
            for (int layer = 0; layer < NDOIS; layer++)
                for (int cx = 0; cx < NX; cx++)
                    for (int cy = 0; cy < NY; cy++) {
                        const int i = NX * head + cx + HX * cy + XYH * layer;
                        singles[i] = (singles[i] + drates[i] / (tau * fan)) / 2.0f;
                    }
        }
    }
    if (niter) *niter = iter;
    return HRRT_OK;
}

extern "C" int hrrt_delays_smooth(hrrt_delays *c, const float *d_singles, float scan_duration, float *d_delays,
                                  void *stream) {
    if (!c || !d_singles || !d_delays) return hrrt_dl::fail(HRRT_ERR_ARG, "null argument");
    hipStream_t s = (hipStream_t)stream;
    int r = upload(*c), dev = -1;
    if (r != HRRT_OK) return r;
    DTRY(hipGetDevice(&dev));
    if (dev != c->device) return hrrt_dl::fail(HRRT_ERR_ARG, "context tables live on another device");
    const int cstride = (c->nplanes + 63) & ~63;
    if (!c->d_cols) {
        // The first smoothing may be recorded into a graph (a histogram has uploaded the tables): the allocation
        // belongs to the context, not to the graph, so it is made whatever the thread's capture mode.
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        DTRY(hipThreadExchangeStreamCaptureMode(&mode));
        const hipError_t e = hipMalloc(&c->d_cols, sizeof(float) * (size_t)c->nsino * cstride);
        (void)hipThreadExchangeStreamCaptureMode(&mode);
        DTRY(e);
    }
    const float ftime = scan_duration > 0.0f ? scan_duration : 1.0f;
    const float tauftime = c->tau * ftime;
    Tables t{c->d_lor, c->d_lor_off, c->d_seg_col, c->d_z, c->nsino, c->nplanes, c->maxrd + 5};
    sings_prepare_kernel<<<NCOLS / PREP_COLS, 256, 0, s>>>(d_singles, c->d_sings);
    bin_scale_kernel<<<(c->nsino + 255) / 256, 256, 0, s>>>(t, c->d_sings, tauftime, c->d_scale);
    DTRY(hipGetLastError());
    const unsigned grid = 8 * ((c->nsino / 8 + COL_BINS - 1) / COL_BINS);
    delays_column_kernel<<<grid, COL_THREADS, 0, s>>>(t, c->d_sings, c->d_scale, tauftime, c->d_cols, cstride);
    DTRY(hipGetLastError());
    column_transpose_kernel<<<dim3((c->nplanes + 64 * TT - 1) / (64 * TT), (c->nsino + 63) / 64), 256, 0, s>>>(c->d_cols, d_delays,
                                                                                               c->nsino, c->nplanes, cstride);
    DTRY(hipGetLastError());
    return HRRT_OK;
}

extern "C" int hrrt_gen_delays(hrrt_delays *c, const int32_t *coins, float scan_duration, float *d_delays,
                               float *singles_out, int *niter, void *stream) {
    if (!c || !coins || !d_delays) return hrrt_dl::fail(HRRT_ERR_ARG, "null argument");
    std::vector<float> sg(NCRYS);
    int r = hrrt_delays_singles(c, coins, scan_duration, sg.data(), niter);
    if (r != HRRT_OK) return r;
    if (singles_out) memcpy(singles_out, sg.data(), sizeof(float) * NCRYS);
    // the singles are staged in the head of the output (nplanes*nsino >= crystals), which the
    // smoothing reads into its transposed copy before its last kernel overwrites the output
    hipStream_t s = (hipStream_t)stream;
    DTRY(hipMemcpyAsync(d_delays, sg.data(), sizeof(float) * NCRYS, hipMemcpyHostToDevice, s));
    DTRY(hipStreamSynchronize(s));
    return hrrt_delays_smooth(c, d_delays, scan_duration, d_delays, stream);
}

extern "C" int hrrt_delays_write(hrrt_delays *c, const float *d_delays, const char *path, void *stream) {
    if (!c || !d_delays || !path) return hrrt_dl::fail(HRRT_ERR_ARG, "null argument");
    hipStream_t s = (hipStream_t)stream;
    const size_t plane = (size_t)c->nsino;
    std::vector<float> h(plane * 64);
    FILE *f = fopen(path, "wb");
    if (!f) return hrrt_dl::fail(HRRT_ERR_ARG, std::string("cannot create ") + path);
    bool ok = true;
    for (int p0 = 0; ok && p0 < c->nplanes; p0 += 64) {
        const size_t n = plane * std::min(64, c->nplanes - p0);
        if (hipMemcpyAsync(h.data(), d_delays + (size_t)p0 * plane, sizeof(float) * n, hipMemcpyDeviceToHost, s) !=
                hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess) {
            fclose(f);
            return hrrt_dl::fail(HRRT_ERR_HIP, "copy of the delays to the host failed");
        }
        ok = fwrite(h.data(), sizeof(float), n, f) == n;
    }
    ok = (fclose(f) == 0) && ok;
    return ok ? HRRT_OK : hrrt_dl::fail(HRRT_ERR_ARG, std::string("write failed: ") + path);
}
