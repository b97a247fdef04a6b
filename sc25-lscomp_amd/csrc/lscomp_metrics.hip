// lscomp_metrics.hip -- error metrics between an original and a decoded volume.
//
// Definitions follow the reference's computePSNR (lsCOMP/src/cuLSZ_utility.cu:887-946):
// mse = sum(err^2)/n, range = max(orig) - min(orig), psnr = 20 log10(range)
// - 10 log10(mse), normErr = sqrt(sum err^2), normErr_norm = normErr /
// sqrt(sum dec^2), nrmse = sqrt(mse)/range; plus the maximum absolute error
// and the maximum pointwise relative error over nonzero originals.  Sums are
// exact 64-bit integers (uint16 data), one partial per workgroup.
// One pass, HBM-bound: 4 bytes read per element pair.  Also the mean SSIM
// of the reference's computeSSIM (cuLSZ_utility.cu:757-886), and the plain
// copy used to measure copy bandwidth and to calibrate the HBM byte counters.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "../../include/lscomp.h"
#include "lscomp_host.h"

namespace lsc {

// 16 bytes at 4-byte alignment (global_load_dwordx4 takes dword alignment).
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), __aligned__(4)));

__device__ __forceinline__ uint32_t pk_max(uint32_t a, uint32_t b)
{
    return as_u32(__builtin_elementwise_max(as_u16x2(a), as_u16x2(b)));
}
__device__ __forceinline__ uint32_t pk_min(uint32_t a, uint32_t b)
{
    return as_u32(__builtin_elementwise_min(as_u16x2(a), as_u16x2(b)));
}
__device__ __forceinline__ uint32_t pk_sub(uint32_t a, uint32_t b) { return as_u32(as_u16x2(a) - as_u16x2(b)); }

constexpr uint32_t kMetricWg = 512, kMetricGrid = 1024;   // threads per workgroup, workgroups at most

// Sums and extrema of one thread, one workgroup or the whole pair of volumes.
// The largest relative error is kept as the fraction rel_e / rel_a: rounding is
// monotone, so the largest rounded quotient is the rounded largest quotient,
// and two fractions of 16-bit values compare exactly by 32-bit products.
struct MetricAcc {
    unsigned long long sum_sq_err, sum_sq_dec;
    uint32_t max_err, min_orig, max_orig;
    uint32_t rel_e, rel_a, pad;

    __device__ __forceinline__ void rel(uint32_t e, uint32_t a)
    {
        e = a ? e : 0u;
        if (e * rel_a > rel_e * a) {
            rel_e = e;
            rel_a = a;
        }
    }
    __device__ __forceinline__ void pair(uint32_t a, uint32_t d)
    {
        const uint32_t e = a > d ? a - d : d - a;
        sum_sq_err += (uint64_t)e * e;
        sum_sq_dec += (uint64_t)d * d;
        max_err = e > max_err ? e : max_err;
        min_orig = a < min_orig ? a : min_orig;
        max_orig = a > max_orig ? a : max_orig;
        rel(e, a);
    }
    __device__ __forceinline__ void merge(const MetricAcc &o)
    {
        sum_sq_err += o.sum_sq_err;
        sum_sq_dec += o.sum_sq_dec;
        max_err = o.max_err > max_err ? o.max_err : max_err;
        min_orig = o.min_orig < min_orig ? o.min_orig : min_orig;
        max_orig = o.max_orig > max_orig ? o.max_orig : max_orig;
        rel(o.rel_e, o.rel_a);
    }
};

__device__ __forceinline__ MetricAcc metric_zero() { return MetricAcc{0, 0, 0, 0xffffu, 0, 0, 1, 0}; }

// Merge over the workgroup's WG threads; thread 0 holds the result.
template <uint32_t WG>
__device__ __forceinline__ void metric_reduce(MetricAcc &m)
{
    __shared__ MetricAcc part[WG / 64];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1)
        m.merge(MetricAcc{__shfl_xor(m.sum_sq_err, o, 64), __shfl_xor(m.sum_sq_dec, o, 64), __shfl_xor(m.max_err, o, 64),
                          __shfl_xor(m.min_orig, o, 64), __shfl_xor(m.max_orig, o, 64), __shfl_xor(m.rel_e, o, 64),
                          __shfl_xor(m.rel_a, o, 64), 0});
    if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0)
        for (uint32_t w = 1; w < WG / 64; w++) m.merge(part[w]);
}

// One pass over both volumes, read-bound: 16-byte loads of `n8` groups of 8
// elements starting at element `head` (both volumes dword aligned there), the
// elements before and after one by one.  A group's arithmetic is on packed
// pairs (absolute difference, extrema, dot products for the squares: their sum
// over 8 elements fits 32 bits while all are below 2^14, otherwise element by
// element).  Each workgroup writes one partial (metrics_finish_kernel merges
// them): six 64- and 32-bit atomics per wave on one line cost 2.37 ms at 512 x
// 1024 x 1024, whatever the size above some thousand waves, against 0.37 ms.
__global__ __launch_bounds__(kMetricWg) void metrics_kernel(const uint16_t *__restrict__ orig,
                                                            const uint16_t *__restrict__ dec, uint64_t n,
                                                            uint32_t head, uint64_t n8, MetricAcc *__restrict__ part)
{
    MetricAcc m = metric_zero();
    const uint64_t stride = (uint64_t)gridDim.x * kMetricWg, first = (uint64_t)blockIdx.x * kMetricWg + threadIdx.x;
    const u32x4_a4 *va = (const u32x4_a4 *)(orig + head), *vd = (const u32x4_a4 *)(dec + head);
    uint32_t mn2 = 0xffffffffu, mx2 = 0, me2 = 0;   // packed extrema
    for (uint64_t i = first; i < n8; i += stride) {
        const u32x4_a4 a = va[i], d = vd[i];
        uint32_t e[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            mn2 = pk_min(mn2, a[k]);
            mx2 = pk_max(mx2, a[k]);
            e[k] = pk_sub(pk_max(a[k], d[k]), pk_min(a[k], d[k]));
            me2 = pk_max(me2, e[k]);
            m.rel(e[k] & 0xffffu, a[k] & 0xffffu);
            m.rel(e[k] >> 16, a[k] >> 16);
        }
        if (((e[0] | e[1] | e[2] | e[3] | d[0] | d[1] | d[2] | d[3]) & 0xc000c000u) == 0) {
            uint32_t se = 0, sd = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                se = dot2(e[k], e[k], se);
                sd = dot2(d[k], d[k], sd);
            }
            m.sum_sq_err += se;
            m.sum_sq_dec += sd;
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t e0 = e[k] & 0xffffu, e1 = e[k] >> 16, d0 = d[k] & 0xffffu, d1 = d[k] >> 16;
                m.sum_sq_err += (uint64_t)(e0 * e0) + (uint64_t)(e1 * e1);
                m.sum_sq_dec += (uint64_t)(d0 * d0) + (uint64_t)(d1 * d1);
            }
        }
    }
    m.max_err = me2 >> 16 > (me2 & 0xffffu) ? me2 >> 16 : me2 & 0xffffu;
    m.max_orig = mx2 >> 16 > (mx2 & 0xffffu) ? mx2 >> 16 : mx2 & 0xffffu;
    m.min_orig = mn2 >> 16 < (mn2 & 0xffffu) ? mn2 >> 16 : mn2 & 0xffffu;
    // the elements before the first group and after the last one
    const uint64_t rest = n - 8 * n8;
    for (uint64_t i = first; i < rest; i += stride) {
        const uint64_t at = i < head ? i : i + 8 * n8;
        m.pair(orig[at], dec[at]);
    }
    metric_reduce<kMetricWg>(m);
    if (threadIdx.x == 0) part[blockIdx.x] = m;
}

__global__ __launch_bounds__(kMetricGrid) void metrics_finish_kernel(const MetricAcc *__restrict__ part, uint32_t np,
                                                                     MetricAcc *__restrict__ out)
{
    MetricAcc m = threadIdx.x < np ? part[threadIdx.x] : metric_zero();
    metric_reduce<kMetricGrid>(m);
    if (threadIdx.x == 0) *out = m;
}

// Plain copy: each workgroup copies one contiguous 16 KiB chunk, four 16-byte
// loads per lane issued before the four stores.
__global__ __launch_bounds__(256) void copy_kernel(uint4 *__restrict__ dst, const uint4 *__restrict__ src,
                                                   uint64_t n16)
{
    const uint64_t base = (uint64_t)blockIdx.x * 1024 + threadIdx.x;
    uint4 v[4];
#pragma unroll
    for (int k = 0; k < 4; k++)
        if (base + 256 * k < n16) v[k] = src[base + 256 * k];
#pragma unroll
    for (int k = 0; k < 4; k++)
        if (base + 256 * k < n16) dst[base + 256 * k] = v[k];
}

__global__ void copy_tail_kernel(uint8_t *dst, const uint8_t *src, uint32_t n)
{
    if (threadIdx.x < n) dst[threadIdx.x] = src[threadIdx.x];
}

// ---------------------------------------------------------------------------
// SSIM (cuLSZ_utility.cu:757-886): the mean over 7x7x7 windows moved by 2
// along every axis of luminance * contrast * structure, with c1 = (0.01 R)^2,
// c2 = (0.03 R)^2 (R: the original's range in the window; 0.01^2 and 0.03^2
// when R = 0) and c3 = c2 / 2.
//
// Separable window sums instead of the reference's two passes over every
// window's 343 points, and the product of the three terms in closed form:
// with c3 = c2 / 2, contrast * structure = (2 cov + c2) / (var_x + var_y + c2)
// (the standard deviations cancel), so a window needs its sums of x, y, xy and
// x^2 + y^2, the original's extrema and one division.  All sums are exact
// integers, and n^2 times each factor's numerator and denominator (n = 343) is
// formed from them in doubles, where the reference rounds a two-pass double
// sum.
//
// ALU-bound, so the mapping is chosen for few operations per window.  A lane
// owns one word (two elements) of its rows and kSsimJ windows along size1, and
// walks planes (size2).  It adds its word's values and products over a
// window's 7 rows, for the pair and for its first element, by packed dot
// products that accumulate; a window of 7 elements is then three pairs and one
// element of lanes i .. i + 3, so a wave's 64 words make 61 windows.  Rows 2 to
// 6 are summed once for both windows.  Along size2 windows overlap by 5 of 7
// planes, so a window is the sum of three disjoint pairs of planes and one
// plane; pairs stay in registers, nothing goes through LDS and there is no
// barrier in the loop.  The next plane's words are loaded before a plane's are
// used.  512 x 1024 x 1024 (values below 2^12): 0.66 ms, against 1.23 ms with
// each lane loading and adding the 7 elements of its rows (4.5 rows of 7
// elements per window and plane, against 4.5 words), and 3.19 ms with one
// window per thread, double sums through LDS, square roots, divisions and three
// barriers per plane; 600 x 1813 x 1558 with 16-bit values 2.1, 4.3 and 10.2
// ms.  Without the narrow sums' packed halves and 32-bit window products 0.77
// ms, without the load ahead 4 % more; 4 waves per SIMD (128 registers) 0.72
// and 2.36 ms.  Vector ALU instructions issue in 93 % of the cycles.
//
// Each workgroup writes one partial sum, reduced in a fixed order (here and in
// ssim_finish_kernel), so the result does not depend on scheduling.
// ---------------------------------------------------------------------------
constexpr uint32_t kSsimJ = 2;                            // windows of a lane along size1
constexpr uint32_t kSsimT0 = 61, kSsimT1 = 4 * kSsimJ;    // windows of a workgroup (4 waves) along size0, size1
constexpr uint32_t kSsimRows = 2 * kSsimJ + 5;            // rows of a lane's windows

// Sums over a 7 x 7 patch of a plane, and over planes; mm = max | (65535 - min) << 16.
struct SsimMom {
    uint32_t sx, sy, mm;
    uint64_t sxy, sqq;
};

__device__ __forceinline__ SsimMom mom_add(const SsimMom &a, const SsimMom &b)
{
    return {a.sx + b.sx, a.sy + b.sy, pk_max(a.mm, b.mm), a.sxy + b.sxy, a.sqq + b.sqq};
}
__device__ __forceinline__ double ssim_of(const SsimMom &m)
{
#pragma clang fp contract(off)
    const double n = 343.0, n2 = n * n;
    const double sx = (double)m.sx, sy = (double)m.sy;
    const double range = (double)((m.mm & 0xffffu) - (0xffffu - (m.mm >> 16)));
    const double r2 = range == 0.0 ? 1.0 : range * range;
    const double c1 = 0.01 * 0.01 * n2 * r2, c2 = 0.03 * 0.03 * n2 * r2;
    // integers below 2^51: exact in doubles
    const double pxy = sx * sy, pqq = sx * sx + sy * sy;
    const double cov = n * (double)m.sxy - pxy, var = n * (double)m.sqq - pqq;
    return ((2.0 * pxy + c1) * (2.0 * cov + c2)) / ((pqq + c1) * (var + c2));
}

// Sums over a lane's word of up to 7 rows: of both elements (p) and of the
// first one (l).  Narrow, every value below 2^12: the values' sums in packed
// halves (7 values), and the products of a window's 49 elements fit 32 bits,
// those of x^2 + y^2 too.
struct SsimCol {
    uint32_t sx2 = 0, sy2 = 0, mx2 = 0, mn2 = 0xffffffffu, pxy = 0, pqq = 0, lxy = 0, lqq = 0;
};
// Any value: the products of the first factor's low bytes in s and those of its
// high bytes in h; 98 products below 2^24 fit 32 bits.
struct SsimProd {
    uint32_t pxy, pqq, lxy, lqq;
};
struct SsimColWide {
    uint32_t px = 0, py = 0, lx = 0, ly = 0, mx2 = 0, mn2 = 0xffffffffu;
    SsimProd s{}, h{};
};

// The product of the low halves, added to c; written out because the compiler
// takes two masks, a 24-bit product and an addition for it.
__device__ __forceinline__ uint32_t mad_low(uint32_t a, uint32_t b, uint32_t c)
{
    uint32_t r;
    asm("v_mad_u32_u16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ void col_row(SsimCol &a, uint32_t x, uint32_t y)
{
    a.sx2 = as_u32(as_u16x2(a.sx2) + as_u16x2(x));
    a.sy2 = as_u32(as_u16x2(a.sy2) + as_u16x2(y));
    a.mx2 = pk_max(a.mx2, x);
    a.mn2 = pk_min(a.mn2, x);
    a.pxy = dot2(x, y, a.pxy);
    a.pqq = dot2(y, y, dot2(x, x, a.pqq));
    a.lxy = mad_low(x, y, a.lxy);
    a.lqq = mad_low(y, y, mad_low(x, x, a.lqq));
}
__device__ __forceinline__ void prod_row(SsimProd &a, uint32_t fx, uint32_t fy, uint32_t x, uint32_t y, uint32_t lx,
                                         uint32_t ly)
{
    a.pxy = dot2(fx, y, a.pxy);
    a.pqq = dot2(fy, y, dot2(fx, x, a.pqq));
    a.lxy = dot2(fx, ly, a.lxy);
    a.lqq = dot2(fy, ly, dot2(fx, lx, a.lqq));
}
__device__ __forceinline__ void col_row(SsimColWide &a, uint32_t x, uint32_t y)
{
    const uint32_t lx = x & 0xffffu, ly = y & 0xffffu;
    a.px = dot2(x, 0x00010001u, a.px);
    a.py = dot2(y, 0x00010001u, a.py);
    a.lx += lx;
    a.ly += ly;
    a.mx2 = pk_max(a.mx2, x);
    a.mn2 = pk_min(a.mn2, x);
    prod_row(a.s, x & 0x00ff00ffu, y & 0x00ff00ffu, x, y, lx, ly);
    prod_row(a.h, perm(0u, x, 0x0c030c01u), perm(0u, y, 0x0c030c01u), x, y, lx, ly);
}

// The next lane's value; 0 in lane 63 (wave_shl:1).
__device__ __forceinline__ uint32_t lane_next(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x130, 0xf, 0xf, true);
}
// A lane's window from the columns of lanes i .. i + 3: three whole words and
// the first element of the last.
__device__ __forceinline__ SsimMom col_window(const SsimCol &a)
{
    const uint32_t nm2 = ~a.mn2;
    const uint32_t ml = perm(nm2, a.mx2, 0x05040100u), mp = pk_max(ml, perm(nm2, a.mx2, 0x07060302u));
    const uint32_t lx = a.sx2 & 0xffffu, ly = a.sy2 & 0xffffu, px = lx + (a.sx2 >> 16), py = ly + (a.sy2 >> 16);
    uint32_t sx = lx, sy = ly, mm = ml, xy = a.lxy, qq = a.lqq;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        sx = px + lane_next(sx);
        sy = py + lane_next(sy);
        mm = pk_max(mp, lane_next(mm));
        xy = a.pxy + lane_next(xy);
        qq = a.pqq + lane_next(qq);
    }
    return {sx, sy, mm, xy, qq};
}
__device__ __forceinline__ SsimMom col_window(const SsimColWide &a)
{
    const uint32_t nm2 = ~a.mn2;
    const uint32_t ml = perm(nm2, a.mx2, 0x05040100u), mp = pk_max(ml, perm(nm2, a.mx2, 0x07060302u));
    uint32_t sx = a.lx, sy = a.ly, mm = ml, xys = a.s.lxy, xyh = a.h.lxy, qqs = a.s.lqq, qqh = a.h.lqq;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        sx = a.px + lane_next(sx);
        sy = a.py + lane_next(sy);
        mm = pk_max(mp, lane_next(mm));
        xys = a.s.pxy + lane_next(xys);
        xyh = a.h.pxy + lane_next(xyh);
        qqs = a.s.pqq + lane_next(qqs);
        qqh = a.h.pqq + lane_next(qqh);
    }
    return {sx, sy, mm, ((uint64_t)xyh << 8) + xys, ((uint64_t)qqh << 8) + qqs};
}

// A lane's word of each of its rows: elements c and c + 1.  Rows past the
// volume repeat its last one; their windows are not counted.
struct SsimWords {
    uint32_t x[kSsimRows], y[kSsimRows];
};

typedef const __attribute__((address_space(1))) uint8_t *GlobalBytes;

// The words from the dword boundary at or before element c0 + `at` bytes of each
// row.  c0 is the workgroup's first element, so the lane's own offset stays
// within a wave's words however long the rows are.
template <bool kOdd>
__device__ __forceinline__ void ssim_load(const uint16_t *ori, const uint16_t *dec, uint64_t plane, uint32_t Y,
                                          uint32_t Z, uint32_t y0, uint32_t c0, uint32_t at, uint32_t odd0, SsimWords &w)
{
    ori += c0;
    dec += c0;
    asm("" : "+v"(at));   // keeps the zero extension beside the loads, which take it as their offset
#pragma unroll
    for (uint32_t r = 0; r < kSsimRows; r++) {
        const uint64_t row = plane + (uint64_t)(y0 + r < Y ? y0 + r : Y - 1u) * Z;
        const uint32_t ox = kOdd ? ((uint32_t)row ^ odd0) & 1u : 0u, oy = kOdd ? ((uint32_t)row ^ odd0 >> 1) & 1u : 0u;
        // the row in scalar registers plus the lane's offset, not a 64-bit vector add per row
        GlobalBytes qx = (GlobalBytes)(ori + row - ox), qy = (GlobalBytes)(dec + row - oy);
        asm("" : "+s"(qx));
        asm("" : "+s"(qy));
        w.x[r] = *(const __attribute__((address_space(1))) uint32_t *)(qx + at);
        w.y[r] = *(const __attribute__((address_space(1))) uint32_t *)(qy + at);
    }
}
// Where a word starts one element before c, the second one comes from the next
// lane's word.
__device__ __forceinline__ void ssim_shift(uint64_t plane, uint32_t Y, uint32_t Z, uint32_t y0, uint32_t odd0,
                                           SsimWords &w)
{
#pragma unroll
    for (uint32_t r = 0; r < kSsimRows; r++) {
        const uint32_t row = (uint32_t)(plane + (uint64_t)(y0 + r < Y ? y0 + r : Y - 1u) * Z);
        w.x[r] = __builtin_amdgcn_alignbit(lane_next(w.x[r]), w.x[r], 16u * ((row ^ odd0) & 1u));
        w.y[r] = __builtin_amdgcn_alignbit(lane_next(w.y[r]), w.y[r], 16u * ((row ^ odd0 >> 1) & 1u));
    }
}
// By elements; an element c + 1 past its row is never used.  Rare, so a rolled
// loop that shifts the words into place: unrolled, its loads cost the kernel 45
// spilled registers.
__device__ __forceinline__ void ssim_words_by_element(const uint16_t *ori, const uint16_t *dec, uint64_t plane,
                                                      uint32_t Y, uint32_t Z, uint32_t y0, uint32_t c, SsimWords &w)
{
    const uint32_t c1 = c + 1u < Z ? c + 1u : Z - 1u;
    w = {};
#pragma unroll 1
    for (uint32_t r = 0; r < kSsimRows; r++) {
        const uint64_t row = plane + (uint64_t)(y0 + r < Y ? y0 + r : Y - 1u) * Z;
#pragma unroll
        for (uint32_t k = 0; k + 1 < kSsimRows; k++) {
            w.x[k] = w.x[k + 1];
            w.y[k] = w.y[k + 1];
        }
        w.x[kSsimRows - 1] = ori[row + c] | (uint32_t)ori[row + c1] << 16;
        w.y[kSsimRows - 1] = dec[row + c] | (uint32_t)dec[row + c1] << 16;
    }
}

// The plane sums of a lane's kSsimJ windows: P[j] over rows 2j .. 2j + 6.
template <class Col>
__device__ __forceinline__ void ssim_plane(const SsimWords &w, SsimMom P[kSsimJ])
{
    static_assert(kSsimJ == 2, "rows 2 .. 6 are those of both windows");
    Col b;
#pragma unroll
    for (uint32_t r = 2; r < 7; r++) col_row(b, w.x[r], w.y[r]);
    Col a = b;
    col_row(a, w.x[0], w.y[0]);
    col_row(a, w.x[1], w.y[1]);
    P[0] = col_window(a);
    col_row(b, w.x[7], w.y[7]);
    col_row(b, w.x[8], w.y[8]);
    P[1] = col_window(b);
}

// One workgroup of 256 threads per (size0 tile, size1 tile, size2 chunk) of
// windows, nb0 * nb1 * nchunks in all, of which the launch runs those from
// `first` on; partial[first + blockIdx.x] = the sum of the SSIM of its windows.  odd0: bit 0 (1) is set when the original (decoded)
// volume starts at 2 mod 4.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void ssim_kernel(
    const uint16_t *__restrict__ ori, const uint16_t *__restrict__ dec, uint32_t X, uint32_t Y, uint32_t Z, uint32_t n0,
    uint32_t n1, uint32_t n2, uint32_t nb0, uint32_t nb1, uint32_t chunk, uint32_t odd0, uint32_t first,
    double *__restrict__ partial)
{
    __shared__ double wsum[4];
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t blk = first + blockIdx.x;
    const uint32_t b0 = blk % nb0;
    blk /= nb0;
    const uint32_t b1 = blk % nb1, b2 = blk / nb1;
    const uint32_t o0 = b0 * kSsimT0 + lane, o1 = b1 * kSsimT1 + wave * kSsimJ, o2 = b2 * chunk;
    const uint32_t nw = n2 - o2 < chunk ? n2 - o2 : chunk;   // windows along size2
    // a lane's word: that of its window, and for the last windows the three words after them
    const uint32_t o = o0 < n0 + 2u ? o0 : n0 + 2u, c = 2u * o, c0 = 2u * (b0 * kSsimT0), at = 4u * (o - b0 * kSsimT0);
    const bool odd = (Z & 1u) || odd0;
    double acc = 0.0;
    if (o1 < n1) {
        // carry: after an odd plane the last three pairs of planes, after an
        // even one that plane; the last two pairs, the last one
        SsimMom carry[kSsimJ] = {}, s2[kSsimJ] = {}, s1[kSsimJ] = {};
        const uint64_t per_plane = (uint64_t)Y * Z;
        uint64_t plane = 2ull * o2 * per_plane;
        const uint64_t last = (X - 1u) * per_plane;
        // a word can leave a volume, by one element, only in its first row (a
        // base at 2 mod 4) and in its last: the first or last plane by
        // elements; its neighbour is loaded in its place
        const bool edge0 = o1 == 0 && odd0, edge1 = 2u * o1 + kSsimRows >= Y;
        const auto safe = [&](uint64_t p) -> uint64_t {
            if (p >= last) return edge1 ? last - per_plane : last;
            return p == 0 && edge0 ? per_plane : p;
        };
        SsimWords next;
        if (odd)
            ssim_load<true>(ori, dec, safe(plane), Y, Z, 2u * o1, c0, at, odd0, next);
        else
            ssim_load<false>(ori, dec, safe(plane), Y, Z, 2u * o1, c0, at, odd0, next);
        // planes 2 o2 .. 2 o2 + 2 nw + 4, the last one at most X - 1
        for (uint32_t i = 0; i < 2u * nw + 5u; i++, plane += per_plane) {
            SsimMom P[kSsimJ];
            SsimWords w = next;
            if (i == 2u * nw + 4u)
                ;
            else if (odd)
                ssim_load<true>(ori, dec, safe(plane + per_plane), Y, Z, 2u * o1, c0, at, odd0, next);
            else
                ssim_load<false>(ori, dec, safe(plane + per_plane), Y, Z, 2u * o1, c0, at, odd0, next);
            if ((plane == 0 && edge0) || (plane == last && edge1))
                ssim_words_by_element(ori, dec, plane, Y, Z, 2u * o1, c, w);
            else if (odd)
                ssim_shift(plane, Y, Z, 2u * o1, odd0, w);
            uint32_t seen = 0;
#pragma unroll
            for (uint32_t r = 0; r < kSsimRows; r++) seen |= w.x[r] | w.y[r];
            if (__ballot((seen & 0xf000f000u) != 0))
                ssim_plane<SsimColWide>(w, P);
            else
                ssim_plane<SsimCol>(w, P);
            if (i & 1u) {
#pragma unroll
                for (uint32_t j = 0; j < kSsimJ; j++) {
                    const SsimMom t = mom_add(carry[j], P[j]);
                    carry[j] = mom_add(s2[j], t);
                    s2[j] = mom_add(s1[j], t);
                    s1[j] = t;
                }
            } else {
                if (i >= 6u) {
#pragma unroll
                    for (uint32_t j = 0; j < kSsimJ; j++) {
                        const double s = ssim_of(mom_add(carry[j], P[j]));
                        acc += lane < kSsimT0 && o0 < n0 && o1 + j < n1 ? s : 0.0;
                    }
                }
#pragma unroll
                for (uint32_t j = 0; j < kSsimJ; j++) carry[j] = P[j];
            }
        }
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if (lane == 0) wsum[wave] = acc;
    __syncthreads();
    if (threadIdx.x == 0) partial[first + blockIdx.x] = ((wsum[0] + wsum[1]) + wsum[2]) + wsum[3];
}

// The sum of np partials in a fixed order: thread t adds t, t + 1024, ...
__global__ __launch_bounds__(1024) void ssim_finish_kernel(const double *__restrict__ partial, uint64_t np,
                                                           double *__restrict__ out)
{
    __shared__ double wsum[16];
    double acc = 0.0;
    for (uint64_t i = threadIdx.x; i < np; i += 1024u) acc += partial[i];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if ((threadIdx.x & 63u) == 0) wsum[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (uint32_t w = 1; w < 16; w++) acc += wsum[w];
        *out = acc;
    }
}

}  // namespace lsc

extern "C" int lscomp_copy_bytes(void *d_dst, const void *d_src, size_t bytes, hipStream_t stream)
{
    using namespace lsc;
    if (bytes == 0) return LSCOMP_OK;
    if (!d_dst || !d_src || (((uintptr_t)d_dst | (uintptr_t)d_src) & 15)) return LSCOMP_ERR_INVALID_ARG;
    const uint8_t *s = (const uint8_t *)d_src;
    uint8_t *d = (uint8_t *)d_dst;
    if (d < s + bytes && s < d + bytes) return LSCOMP_ERR_INVALID_ARG;   // overlap
    const uint64_t n16 = bytes / 16;
    if (n16) {
        const uint64_t blocks = (n16 + 1023) / 1024;   // 16 KiB per workgroup
        if (blocks > 0xffffffffull) return LSCOMP_ERR_INVALID_ARG;
        hipLaunchKernelGGL(copy_kernel, dim3((uint32_t)blocks), dim3(256), 0, stream, (uint4 *)d,
                           (const uint4 *)s, n16);
    }
    const uint32_t tail = (uint32_t)(bytes - 16 * n16);
    if (tail)
        hipLaunchKernelGGL(copy_tail_kernel, dim3(1), dim3(16), 0, stream, d + 16 * n16, s + 16 * n16, tail);
    return hip_fail(hipGetLastError(), "copy launch");
}

extern "C" int lscomp_error_stats_u16(const uint16_t *d_orig, const uint16_t *d_dec, size_t n,
                                      lscomp_error_stats *out, hipStream_t stream)
{
    using namespace lsc;
    if (!d_orig || !d_dec || !out || n == 0 || (((uintptr_t)d_orig | (uintptr_t)d_dec) & 1))
        return LSCOMP_ERR_INVALID_ARG;
    // the first element from which both volumes are dword aligned; volumes of
    // different alignment mod 4 have none and are read by elements
    const uint32_t oa = (uint32_t)((uintptr_t)d_orig >> 1) & 1u, od = (uint32_t)((uintptr_t)d_dec >> 1) & 1u;
    const uint64_t n8 = oa == od && n > oa ? (n - oa) / 8 : 0;
    const uint32_t head = n8 ? oa : 0u;
    const uint64_t work = n8 ? n8 : n;
    uint64_t blocks = (work + kMetricWg - 1) / kMetricWg;
    if (blocks > kMetricGrid) blocks = kMetricGrid;
    AuxLease aux(stream, (kMetricGrid + 1) * sizeof(MetricAcc), sizeof(MetricAcc));
    int st = aux.status();
    if (st) return st;
    MetricAcc *acc = (MetricAcc *)aux.device();
    hipLaunchKernelGGL(metrics_kernel, dim3((uint32_t)blocks), dim3(kMetricWg), 0, stream, d_orig, d_dec, (uint64_t)n,
                       head, n8, acc + 1);
    hipLaunchKernelGGL(metrics_finish_kernel, dim3(1), dim3(kMetricGrid), 0, stream, acc + 1, (uint32_t)blocks, acc);
    st = hip_fail(hipGetLastError(), "metrics launch");
    if (!st) st = aux.read_back(sizeof(MetricAcc));
    if (st) return st;
    const MetricAcc host = *(const MetricAcc *)aux.host();
    std::memset(out, 0, sizeof *out);
    out->n = n;
    out->max_abs_err = host.max_err;
    out->min_orig = host.min_orig;
    out->max_orig = host.max_orig;
    out->sum_sq_err = host.sum_sq_err;
    out->sum_sq_dec = host.sum_sq_dec;
    out->max_rel_err = (float)host.rel_e / (float)host.rel_a;   // a float quotient, as the pointwise ones are defined
    out->mse = (double)host.sum_sq_err / (double)n;
    out->range = (double)host.max_orig - (double)host.min_orig;
    out->psnr = 20.0 * std::log10(out->range) - 10.0 * std::log10(out->mse);   // inf when lossless
    out->norm_err = std::sqrt((double)host.sum_sq_err);
    out->norm_err_norm = out->norm_err / std::sqrt((double)host.sum_sq_dec);
    out->nrmse = std::sqrt(out->mse) / out->range;
    return LSCOMP_OK;
}

extern "C" int lscomp_ssim_u16(const uint16_t *d_orig, const uint16_t *d_dec, lscomp_dim3 dims, double *ssim,
                               hipStream_t stream)
{
    using namespace lsc;
    if (!d_orig || !d_dec || !ssim || (((uintptr_t)d_orig | (uintptr_t)d_dec) & 1)) return LSCOMP_ERR_INVALID_ARG;
    if (dims.x < 7 || dims.y < 7 || dims.z < 7) return LSCOMP_ERR_INVALID_ARG;   // no window fits
    const uint32_t n0 = (dims.z - 7) / 2 + 1, n1 = (dims.y - 7) / 2 + 1, n2 = (dims.x - 7) / 2 + 1;
    const uint32_t nb0 = (n0 + kSsimT0 - 1) / kSsimT0, nb1 = (n1 + kSsimT1 - 1) / kSsimT1;
    // A chunk of k windows along size2 reads 2 k + 5 planes, so as few chunks as
    // fill the chip once (256 CUs hold 3 workgroups each), of 4 to 32 windows:
    // 205 x 553 x 256 89 us in 735 workgroups, 104 in 2625; 100 x 512 x 512 68
    // us in 640, 77 in 2560; 60 x 1813 x 1558 227 us in 1469, 254 in 5876.
    // Longer chunks gain nothing (512 x 1024 x 1024: 653 us at 32, 641 at 40,
    // 684 at 64).
    const uint64_t fill = 768 / ((uint64_t)nb0 * nb1);
    const uint32_t most = (n2 + 3) / 4, least = (n2 + 31) / 32;
    const uint32_t want = fill < least ? least : fill > most ? most : (uint32_t)fill;
    const uint32_t chunk = (n2 + want - 1) / want, nc = (n2 + chunk - 1) / chunk;
    const uint64_t blocks = (uint64_t)nb0 * nb1 * nc;
    if (blocks > 0x7fffffffull) return LSCOMP_ERR_TOO_LARGE;
    AuxLease aux(stream, (blocks + 1) * sizeof(double), sizeof(double));
    int st = aux.status();
    if (st) return st;
    double *partial = (double *)aux.device();
    const uint32_t odd0 = (uint32_t)((uintptr_t)d_orig >> 1 & 1u) | (uint32_t)((uintptr_t)d_dec >> 1 & 1u) << 1;
    // a launch holds fewer than 2^32 threads, so 2^23 workgroups each
    for (uint64_t first = 0; first < blocks; first += 1u << 23) {
        const uint64_t n = blocks - first < 1u << 23 ? blocks - first : 1u << 23;
        hipLaunchKernelGGL(ssim_kernel, dim3((uint32_t)n), dim3(256), 0, stream, d_orig, d_dec, dims.x, dims.y, dims.z,
                           n0, n1, n2, nb0, nb1, chunk, odd0, (uint32_t)first, partial + 1);
    }
    hipLaunchKernelGGL(ssim_finish_kernel, dim3(1), dim3(1024), 0, stream, partial + 1, blocks, partial);
    st = hip_fail(hipGetLastError(), "ssim launch");
    if (!st) st = aux.read_back(sizeof(double));
    if (st) return st;
    const double sum = *(const double *)aux.host();
    *ssim = sum / ((double)n0 * (double)n1 * (double)n2);
    return LSCOMP_OK;
}
