// tt_kernels.hip -- CDNA4 (gfx950) kernels of the trace transform.
//
// Built with -ffp-contract=off: every product and sum that feeds a
// weighted-median index is rounded exactly as in the reference's float code
// (no FMA), so median and sort indices are bit-identical to the reference's
// arithmetic.  Denormals are kept (no flush) and sqrtf is correctly rounded,
// as on the reference's x86-64 SSE2 build.  Sums that only feed values (the
// T1-T5 and P integrals) use explicit fma and, where it buys accuracy against
// the FP64 oracle, double accumulators.
#include "tt_internal.hpp"

#include <math.h>
#include <type_traits>

namespace ttk {

namespace {

// 16-byte load from an 8-byte aligned address (legal for global memory on
// CDNA): two neighbouring pixel pairs; 8-byte load from a 4-byte aligned one:
// two neighbouring pixels.
typedef float f4p __attribute__((ext_vector_type(4), aligned(8)));
typedef float f2p __attribute__((ext_vector_type(2), aligned(4)));

// A pointer every lane of the wave holds, made visibly wave-uniform (its
// two halves read from the first lane), so that loads from it can take the
// scalar-base form.
__device__ __forceinline__ const float *uniform_ptr(const float *p)
{
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<const float *>(((uint64_t)hi << 32) | lo);
}

// Load at a 32-bit byte offset from a wave-uniform base in global memory:
// the scalar-base + vector-offset form of global loads (no 64-bit VALU
// math, no flat addressing).
template <class V> __device__ __forceinline__ V ldb(const float *base, uint32_t byte_off)
{
    typedef const char __attribute__((address_space(1))) *gbyte;
    typedef const V __attribute__((address_space(1))) *gv;
    return *(gv)((gbyte)base + byte_off);
}

__device__ __forceinline__ int wave_id()
{
    return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}

// Workgroups are dealt to the 8 XCDs round-robin; give each XCD a contiguous
// range of logical blocks so the lines one XCD works on share its L2.  The
// grid is padded to a multiple of 8 by the launcher.
__device__ __forceinline__ int xcd_block()
{
    const int g8 = gridDim.x / kNumXcd;
    const int b = blockIdx.x;
    return (b % kNumXcd) * g8 + b / kNumXcd;
}

// ---------------------------------------------------------------------------
// Bilinear sample of the rotated image at (row, col), c++/src/auxiliary.cpp
// :223-255 and :182-196.  x = px*c + py*s + o, y = px*(-s) + py*c + o, with
// pxc = px*c and pxns = px*(-s) precomputed per lane (each is one rounded
// product, as in the reference).  Strict bounds 0 <= x,y < n-1; the four
// taps are evaluated left to right with the reference's association.
// PAIRS: src is the pixel-pair copy of the image that the lanes step along: TR
// (along x) pairs of rows, else pairs of columns; the four taps are one 16-byte
// load.  Else src is the image's row-major copy (TR) or the image itself, and
// the taps are two 8-byte loads.  The taps, hence the results, are the same.
// The L1 looks up one line per four lanes of a load whatever the load's width,
// about 25 cycles per load and CU, and two 8-byte loads a sample (one per
// image row) made that the line kernel's bound: 0.87 ms against 0.59 for the
// samples of 1449^2 pixels at 360 angles (a copy of 2 x 2 quads, four times
// the image, reads 0.97: it leaves the L2).
// ---------------------------------------------------------------------------
// A sample whose load is under way: its taps, fractions and whether it lies
// inside the image.
struct Tap {
    f4p q;
    float fx, fy;
    bool in;
};

// CHK: test the position against the image's bounds (without it the caller
// knows that the position is inside).
template <bool TR, bool PAIRS, bool CHK>
__device__ __forceinline__ Tap rot_load(const float *__restrict__ src, int n, float lim,
                                        float o, float pxc, float pxns, float c, float s,
                                        float py)
{
    Tap t;
    float x = pxc + py * s;
    float y = pxns + py * c;
    x = x + o;
    y = y + o;
    // for 0 <= x the integer part is the truncating conversion and the
    // fraction x - floor(x) is exact (modf's split)
    t.fx = __builtin_amdgcn_fractf(x);
    t.fy = __builtin_amdgcn_fractf(y);
    // unsigned 32-bit offsets from a wave-uniform base: global loads in
    // scalar-base + vector-offset form, no 64-bit address arithmetic
    uint32_t X = (uint32_t)x, Y = (uint32_t)y;
    t.in = true;
    if constexpr (CHK) {
        // 0 <= x < lim as one unsigned compare of the bit patterns: x is never
        // -0 (a sum with o > 0 rounds an exact zero to +0), non-negative floats
        // order as their bits, and negative values and NaN compare above lim
        t.in = __float_as_uint(x) < __float_as_uint(lim) &&
               __float_as_uint(y) < __float_as_uint(lim);
        X = t.in ? X : 0u;
        Y = t.in ? Y : 0u;
    }
    const uint32_t un = (uint32_t)n;
    // X, Y < n <= 2730, so X * n fits the 24-bit multiplier
    const uint32_t at = TR ? __umul24(Y, un) + X : __umul24(X, un) + Y;
    if constexpr (PAIRS) {
        t.q = ldb<f4p>(src, at * 8u);
    } else {
        const f2p a = ldb<f2p>(src, at * 4u), b = ldb<f2p>(src, (at + un) * 4u);
        t.q = f4p{a.x, b.x, a.y, b.y};
    }
    return t;
}

template <bool TR, bool CHK>
__device__ __forceinline__ float rot_value(const Tap &t)
{
    const float s00 = t.q.x, s01 = TR ? t.q.z : t.q.y, s10 = TR ? t.q.y : t.q.z, s11 = t.q.w;
    const float ofx = 1.0f - t.fx;
    const float ofy = 1.0f - t.fy;
    const float v = s00 * ofx * ofy + s01 * t.fx * ofy + s10 * ofx * t.fy +
                    s11 * t.fx * t.fy;
    return !CHK || t.in ? v : 0.0f;
}

template <bool TR, bool PAIRS>
__device__ __forceinline__ float rot_sample(const float *__restrict__ src, int n, float lim,
                                            float o, float pxc, float pxns, float c, float s,
                                            float py)
{
    return rot_value<TR, true>(rot_load<TR, PAIRS, true>(src, n, lim, o, pxc, pxns, c, s, py));
}

// Square root of a line sample, correctly rounded.  FS: v_sqrt_f32 and one
// residual test per neighbour (x - s' s against 0 picks the float nearest
// the true root), without the correctly rounded sequence's scaling of small
// inputs and its zero/infinity select.  Equal to that sequence on every
// float except x in (0, 2^-96) and the negative denormals (checked on the
// GPU over all 2^32 inputs); a bilinear sample falls there only if some
// pixel is negative or in (0, 2^-45) (each non-zero tap weight is a product
// of two factors >= 2^-25), which the image's bounding-box pass flags.
template <bool FS>
__device__ __forceinline__ float line_sqrt(float x)
{
    if constexpr (!FS) {
        return sqrtf(x);
    } else {
        const float s = __builtin_amdgcn_sqrtf(x);
        const float sd = __uint_as_float(__float_as_uint(s) - 1u);
        const float su = __uint_as_float(__float_as_uint(s) + 1u);
        const float r = fmaf(-sd, s, x) <= 0.0f ? sd : s;
        return fmaf(-su, s, x) > 0.0f ? su : r;
    }
}

// The line kernel's root: FS: v_rsq_f32, its product with x and one Newton
// step with an exact residual (fma), 7 issue slots of a line_sqrt<true>'s 11.
// Equal to the correctly rounded root on 0 and on every float in
// [2^-96, 2^127) (checked on the GPU over all of them); NaN gives NaN.  The
// image flag rules out samples elsewhere: negative ones, (0, 2^-96), infinite.
template <bool FS>
__device__ __forceinline__ float line_root(float x)
{
    if constexpr (!FS) {
        return sqrtf(x);
    } else {
        // (the addend keeps the reciprocal root of 0 finite and rounds away
        // from 2^-96 on)
        const float y = __builtin_amdgcn_rsqf(x + 0x1p-126f);
        const float g = x * y;
        return fmaf(fmaf(-g, g, x), 0.5f * y, g);
    }
}

// Test hook: line_sqrt<true> against the correctly rounded sqrtf on the
// float bit patterns [lo, lo + count), outside its documented exceptions
// ((0, 2^-96) and the negative denormals).  Counts the patterns whose
// results differ (NaN results compare equal) and keeps the smallest one.
// ROOT: line_root<true> instead, on 0, NaN and [2^-96, 2^127).
template <bool ROOT>
__global__ __launch_bounds__(kBlock) void short_sqrt_check_kernel(uint32_t lo, uint64_t count,
                                                                 unsigned long long *mism,
                                                                 unsigned int *first)
{
    unsigned long long bad = 0;
    unsigned int firstbad = 0xFFFFFFFFu;
    const uint64_t stride = (uint64_t)gridDim.x * kBlock;
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < count; i += stride) {
        const uint32_t b = lo + (uint32_t)i;
        const bool tiny = b > 0u && b < 0x0F800000u;           // (0, 2^-96)
        const bool negden = b > 0x80000000u && b < 0x80800000u;  // negative denormals
        const float x = __uint_as_float(b);
        if (ROOT ? !(x == 0.0f || x != x || (x >= 0x1p-96f && x < 0x1p127f))
                 : tiny || negden)
            continue;
        const float a = ROOT ? line_root<true>(x) : line_sqrt<true>(x);
        const float r = line_sqrt<false>(x);
        const bool same = __float_as_uint(a) == __float_as_uint(r) || (a != a && r != r);
        if (!same) {
            bad++;
            firstbad = b < firstbad ? b : firstbad;
        }
    }
    if (bad) {
        atomicAdd(mism, bad);
        atomicMin(first, firstbad);
    }
}

// ---------------------------------------------------------------------------
// T0..T5 line kernel.  Lane = one column of the rotated image of one angle.
// Pass 1 streams the column and forms Eigen's packet-order sum (8 stride
// accumulators, c++/src/functionals.cpp:22 via Eigen Redux) of x and sqrt(x):
// S_x is T0 and the median threshold; S_sqrt the sqrt-median threshold.
// Pass 2 re-samples the column (the rotated image is never stored), walks
// the sequential float prefix to find findWeightedMedian's first index with
// 2*prefix >= S (c++/src/functionals.cpp:21-30), and from there accumulates
// T1/T2 (c++/src/functionals.cpp:104-129) and T3/T4/T5
// (c++/src/functionals.cpp:200-213) over the same rows as the reference.
// ---------------------------------------------------------------------------
// Wave minimum and maximum as wave-uniform values, by data-parallel moves
// (rows of 16 lanes, then across rows): no LDS traffic.  Every lane of the
// wave must be active.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_i(int v)
{
    return __builtin_amdgcn_update_dpp(v, v, CTRL, ROWS, 0xf, false);
}
template <class Op>
__device__ __forceinline__ int wave_reduce_u(int v, Op op)
{
    v = op(v, dpp_i<0x111, 0xf>(v));  // row_shr 1, 2, 4, 8: lane 15 of each row
    v = op(v, dpp_i<0x112, 0xf>(v));
    v = op(v, dpp_i<0x114, 0xf>(v));
    v = op(v, dpp_i<0x118, 0xf>(v));
    v = op(v, dpp_i<0x142, 0xa>(v));  // row_bcast 15 into rows 1 and 3
    v = op(v, dpp_i<0x143, 0xc>(v));  // row_bcast 31 into rows 2 and 3
    return __builtin_amdgcn_readlane(v, kWave - 1);
}
__device__ __forceinline__ int wave_min_u(int v)
{
    return wave_reduce_u(v, [](int a, int b) { return a < b ? a : b; });
}
__device__ __forceinline__ int wave_max_u(int v)
{
    return wave_reduce_u(v, [](int a, int b) { return a > b ? a : b; });
}

__device__ __forceinline__ int wave_max_i(int v)
{
#pragma unroll
    for (int m = kWave / 2; m > 0; m >>= 1) {
        const int o = __shfl_xor(v, m, kWave);
        v = o > v ? o : v;
    }
    return v;
}

__device__ __forceinline__ int wave_min_i(int v)
{
#pragma unroll
    for (int m = kWave / 2; m > 0; m >>= 1) {
        const int o = __shfl_xor(v, m, kWave);
        v = o < v ? o : v;
    }
    return v;
}

// Rows r with base + (r - o) * slope in [lo_v, hi_v] (exact arithmetic),
// intersected into [*lo, *hi].
__device__ __forceinline__ void slab_rows(double base, double slope, double lo_v,
                                          double hi_v, double o, double *lo, double *hi)
{
    if (fabs(slope) < 1e-30) {
        if (base < lo_v || base > hi_v)
            *lo = 1.0, *hi = 0.0;
        return;
    }
    double r1 = (lo_v - base) / slope + o, r2 = (hi_v - base) / slope + o;
    if (r1 > r2) {
        const double t = r1;
        r1 = r2;
        r2 = t;
    }
    *lo = r1 > *lo ? r1 : *lo;
    *hi = r2 < *hi ? r2 : *hi;
}

// Rows of column col (angle with trig c, s) whose sample can be non-zero:
// the sample at row r reads taps (trunc(x), trunc(y)) + {0,1}^2 with
// x = px c + (r - o) s + o, y = -px s + (r - o) c + o.  Outside the rows
// where the exact x and y lie within 2 pixels of the bounding box of the
// non-zero pixels (float rounding of x, y is below 1e-3 here), every tap
// lies outside that box, so the sample is exactly 0.  Returns [lo, hi]
// (lo > hi when empty); no box means every row.
__device__ __forceinline__ int2 line_rows(const int *bbox, int n, int col, float c, float s)
{
    if (!bbox)
        return int2{0, n - 1};
    const int bx0 = bbox[0], bx1 = bbox[1], by0 = bbox[2], by1 = bbox[3];
    if (bx0 > bx1 || by0 > by1)
        return int2{n, -1};
    const double o = (n - 1) / 2.0, px = (double)col - o;
    double lo = 0.0, hi = (double)(n - 1);
    slab_rows(px * (double)c + o, (double)s, bx0 - 2.0, bx1 + 2.0, o, &lo, &hi);
    slab_rows(-px * (double)s + o, (double)c, by0 - 2.0, by1 + 2.0, o, &lo, &hi);
    if (!(lo <= hi))
        return int2{n, -1};
    return int2{(int)ceil(lo), (int)floor(hi)};
}

// Rows of a line whose sample position lies inside the image with a margin of
// 0.05 pixels, far above the rounding of the positions and of this bound
// (below 0.005 for n <= 2730): their samples need no bounds test.  [lo, hi]
// (lo > hi: none), not clipped to [0, n).
__device__ __forceinline__ int2 inside_rows(int n, int col, float c, float s)
{
    const float o = (float)(n - 1) * 0.5f, px = (float)col - o;
    const float a = 0.05f - o, b = o - 0.05f;  // bounds of position - o
    float lo = -1e6f, hi = 1e6f;
    auto slab = [&](float base, float slope) {
        if (fabsf(slope) < 1e-6f) {
            // the position moves by less than 0.003 over the line
            if (!(base >= a + 0.01f && base <= b - 0.01f))
                hi = -2e6f;
            return;
        }
        const float inv = 1.0f / slope;
        const float p = (a - base) * inv, q = (b - base) * inv;
        lo = fmaxf(lo, fminf(p, q));
        hi = fminf(hi, fmaxf(p, q));
    };
    slab(px * c, s);
    slab(-px * s, c);
    return int2{(int)ceilf(lo + o), (int)floorf(hi + o)};
}

// Outputs in global memory, typed so (pointers from a batch descriptor are
// generic): their stores and loads are global, not flat, operations.
typedef float __attribute__((address_space(1))) *gf32;
typedef int32_t __attribute__((address_space(1))) *gi32;
typedef float f2v __attribute__((ext_vector_type(2)));
typedef f2v __attribute__((address_space(1))) *gf2;

struct LineDst {
    gf32 sino;
    gi32 med_x;
    gi32 med_s;
    gf2 z345;
    gf2 ckpt;  // walk checkpoints (with CK), see sino_line
    int n;
    int A;
    int tabn;
    Slots slot;

    __device__ LineDst(float *sino_, int32_t *med_x_, int32_t *med_s_, float2 *z345_,
                       float2 *ckpt_, int n_, int A_, int tabn_, Slots slot_)
        : sino((gf32)sino_), med_x((gi32)med_x_), med_s((gi32)med_s_), z345((gf2)z345_),
          ckpt((gf2)ckpt_), n(n_), A(A_), tabn(tabn_), slot(slot_)
    {
    }
};

// Row schedule of a wave.  At step v a lane handles row v - d of its line,
// d = rint(col t) + 64 K, t = -s/c for a line with |c| > |s| and c/s
// otherwise (|t| <= 1, from the line's own angle), K a wave-wide integer
// that makes the smallest d of the wave fall in [0, 64).  Lanes of one
// angle and consecutive columns then take samples along one row of the
// image copy the wave reads (TR: y constant, else x), a few cache lines per
// load, instead of spanning one image row per sample when the lanes all
// take the same row.  Each line still sees its rows in increasing order, so
// every sum, prefix and walk is the unskewed one, and d mod 64 depends on
// the line alone, so the 64-step blocks of pass 2 (v in [64 k, 64 k + 64))
// hold the same rows of a line whatever other lines share its wave: the
// results of a line do not depend on the tile that computes it.  Steps run
// from G, the smallest first row plus skew in the wave rounded down to a
// multiple of 8, in groups of 8: slot j of the stride-8 accumulators takes
// the rows of steps 8k + j, i.e. Eigen's accumulator (j - d) mod 8, and the
// slots are rotated back after the pass.  Rows outside [0, n) (and outside
// [0, a8) for the stride-8 accumulators) are masked and positions outside
// the image tested; a group all of whose lanes are inside (steps [va, vb),
// nearly all of them) does neither.  The schedule's bounds are wave-uniform
// scalars, so the loops run on the scalar unit.
//
// The groups whose samples need no test load four rows ahead of the four
// they work on, so that a wave that is nearly alone on its SIMD (a small
// image) does not wait for each load: the samples of two half groups
// alternate in two register sets.
//
// With CK, pass 1 also runs the median walks' sequential prefixes (the
// same float additions in the same row order as the walk) and stores them
// at the start of every 64-step block from G after the first (at most
// sino_ckpt_blocks(n) of them).  When every sample
// a line has before a block is non-negative its prefixes never decrease, so
// a block whose starting prefix fails a lane's test 2 * prefix >= S holds
// none of that lane's earlier passes: pass 2 starts at the last block start
// where no lane has passed yet, from the stored prefixes, and samples only
// the steps from there on.  A negative or NaN sample (S of the square roots
// NaN, or a negative minimum) keeps the full walk.  [lo, hi] is the lane's
// row range that can hold non-zero samples (lo > hi: none).
//
// Pass 2 goes by the same groups.  While some lane has not passed its tests,
// a group's eight samples are walked first (branch-free: the median is a
// select of the row), and its integrals taken only if some lane has passed
// by the group's end; rows before a lane's median enter with distance 0.
// Once every lane has passed, a row is its sample and the multiply-adds.
//
// T0..T5 of 1449^2 pixels at 360 angles, from the two-load form to pairs and
// untested groups: 1440 -> 930 us; of 363^2 at 360 194 -> 138; of 91^2 at 180
// angles, one wave per three SIMDs, 54 -> 43.  Bound by VALU issue (about 24
// half-rate slots a row in pass 1, of which the bilinear sample is 14; adds and
// multiplies issue twice as fast as the rest on this chip) and, in a batch, as
// much by the bytes behind the L2: 256 images of 91 to 725 rows read 53 GB of
// pairs, 5.3 TB/s, half of the lookups hit, the waves wait for memory 28 % of
// their cycles and for an issue slot 30 % (one image of 1449 rows: 2.4 GB, two
// lookups in three hit, 27 and 25 %).
template <bool TR, bool PAIRS, bool NEED_X, bool NEED_S, bool DO345, bool CK, bool FS>
__device__ __forceinline__ void sino_line(const LineDst &p, const float *src,
                                          const float2 *s_tab, int a, int col,
                                          bool active, float c, float s, int lo, int hi)
{
    const int n = __builtin_amdgcn_readfirstlane(p.n);
    src = uniform_ptr(src);
    const float o = (float)((n - 1) / 2.0);
    const float lim = (float)(n - 1);
    const float px = (float)col - o;
    const float pxc = px * c;
    const float pxns = px * (-s);
    const size_t line = (size_t)a * n + col;
    const size_t plane = (size_t)p.A * n;
    constexpr int kNone = 1 << 28;

    // ---- schedule --------------------------------------------------------
    int dl = (int)rintf((float)col * (fabsf(c) > fabsf(s) ? -s / c : c / s));
    dl -= wave_min_u(dl) & ~63;
    const int ncap = sino_ckpt_blocks(n);
    const int a8 = n & ~7;
    const int a4 = n & ~3;
    const int r0 = lo > 0 ? lo : 0;
    const int r1 = hi + 1 < n ? hi + 1 : n;
    const bool any = active && r1 > r0;  // the lanes past the last column follow it
    const int G = wave_min_u(any ? r0 + dl : kNone) & ~7;
    const int V = wave_max_u(any ? r1 + dl : -kNone);
    const int V1 = wave_max_u(any ? (r1 < a8 ? r1 : a8) + dl : -kNone);
    const int2 ins = inside_rows(n, col, c, s);
    const int va = (wave_max_u((ins.x > 0 ? ins.x : 0) + dl) + 7) & ~7;
    const int vb1 = (wave_min_u((ins.y + 1 < a8 ? ins.y + 1 : a8) + dl)) & ~7;  // pass 1
    const int vb2 = (wave_min_u((ins.y + 1 < n ? ins.y + 1 : n) + dl)) & ~7;    // pass 2

    auto load = [&](auto chk, float py) {
        return rot_load<TR, PAIRS, decltype(chk)::value>(src, n, lim, o, pxc, pxns, c, s, py);
    };
    struct Half {
        Tap t[4];
    };
    // samples of the steps v .. v + 3, untested
    auto load_half = [&](int v) {
        Half h;
        const float py0 = (float)(v - dl) - o;
#pragma unroll
        for (int j = 0; j < 4; j++)
            h.t[j] = load(std::false_type{}, py0 + (float)j);
        return h;
    };
    // the eight samples of the group from step v, tested and with the rows
    // outside [0, n) zero
    auto load_masked = [&](int v, float *x) {
        const int rb = v - dl;
        const float py0 = (float)rb - o;
        Tap t[8];
#pragma unroll
        for (int j = 0; j < 8; j++)
            t[j] = load(std::true_type{}, py0 + (float)j);
#pragma unroll
        for (int j = 0; j < 8; j++)
            x[j] = (unsigned)(rb + j) < (unsigned)n ? rot_value<TR, true>(t[j]) : 0.0f;
    };

    // ---- pass 1: Eigen-order sums -------------------------------------
    float rx[8], rs[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        rx[j] = 0.0f;
        rs[j] = 0.0f;
    }
    constexpr bool WALK = CK && (NEED_X || NEED_S);
    float cx = 0.0f, cs = 0.0f, vmin = 0.0f;  // walk prefixes, smallest sample
    auto add = [&](int j, float x, bool chain) {
        const float sv = NEED_S ? line_root<FS>(x) : 0.0f;
        rx[j] += chain ? x : 0.0f;
        if (NEED_S)
            rs[j] += chain ? sv : 0.0f;
        if (WALK && NEED_X)
            cx += x;
        if (WALK && NEED_S)
            cs += sv;
        if (WALK && !NEED_S)
            vmin = fminf(vmin, x);
    };
    auto checkpoint = [&](int v) {
        if (WALK && v > G && ((v - G) & 63) == 0 && (v - G) / 64 <= ncap && active)
            p.ckpt[(size_t)((v - G) / 64 - 1) * plane + line] = f2v{cx, cs};
    };
    // row coordinates py = row - o are integers or half-integers far below
    // 2^23, so stepping them by whole rows is exact
    for (int v = G; v < V1;) {
        if (v >= va && v < vb1) {
            const int ve = V1 < vb1 ? (V1 + 7) & ~7 : vb1;
            const int vl = ve < vb1 ? ve : vb1;  // groups up to here are untested
            Half h0 = load_half(v);
            for (; v < vl; v += 8) {
                checkpoint(v);
                Half h1 = load_half(v + 4);
#pragma unroll
                for (int j = 0; j < 4; j++)
                    add(j, rot_value<TR, false>(h0.t[j]), true);
                // (the last group loads its own rows again)
                h0 = load_half(v + 8 < vl ? v + 8 : v);
#pragma unroll
                for (int j = 0; j < 4; j++)
                    add(4 + j, rot_value<TR, false>(h1.t[j]), true);
            }
        } else {
            checkpoint(v);
            float x[8];
            load_masked(v, x);
#pragma unroll
            for (int j = 0; j < 8; j++)
                add(j, x[j], (unsigned)(v - dl + j) < (unsigned)a8);
            v += 8;
        }
    }
    // slot j holds accumulator (j - d) mod 8: rotate it back
    const int d = (0 - dl) & 7;
#pragma unroll
    for (int b = 1; b < 8; b <<= 1) {
        const bool on = (d & b) != 0;
        float tx[8], ts[8];
#pragma unroll
        for (int m = 0; m < 8; m++) {
            tx[m] = on ? rx[(m - b) & 7] : rx[m];
            ts[m] = on ? rs[(m - b) & 7] : rs[m];
        }
#pragma unroll
        for (int m = 0; m < 8; m++) {
            rx[m] = tx[m];
            rs[m] = ts[m];
        }
    }
    // rows from a8 on: all zero samples (which change no sum) unless some
    // line of the wave has non-zero rows there
    const bool tail = n < 8 || wave_max_u(r1) > a8;
    float Sx, Ss;
    if (a4 == 0) {
        Sx = 0.0f;
        Ss = 0.0f;
        for (int r = 0; r < n; r++) {
            const float v = rot_sample<TR, PAIRS>(src, n, lim, o, pxc, pxns, c, s,
                                           (float)r - o);
            Sx = r == 0 ? v : Sx + v;
            if (NEED_S)
                Ss = r == 0 ? line_root<FS>(v) : Ss + line_root<FS>(v);
        }
    } else {
        float ax[4], as[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            ax[j] = rx[j] + rx[j + 4];
            as[j] = rs[j] + rs[j + 4];
        }
        if (a4 > a8 && tail) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float v = rot_sample<TR, PAIRS>(src, n, lim, o, pxc, pxns, c, s,
                                               (float)(a8 + j) - o);
                const float sv = NEED_S ? line_root<FS>(v) : 0.0f;
                if (n >= 8) {
                    ax[j] += v;
                    as[j] += sv;
                } else {
                    ax[j] = v;
                    as[j] = sv;
                }
            }
        }
        Sx = (ax[0] + ax[2]) + (ax[1] + ax[3]);
        Ss = (as[0] + as[2]) + (as[1] + as[3]);
        for (int r = a4; tail && r < n; r++) {
            const float v = rot_sample<TR, PAIRS>(src, n, lim, o, pxc, pxns, c, s,
                                           (float)r - o);
            Sx += v;
            if (NEED_S)
                Ss += line_root<FS>(v);
        }
    }

    const size_t tstride = plane;
    if (active && p.slot.s[0] >= 0)
        p.sino[p.slot.s[0] * tstride + line] = Sx;
    if (!NEED_X && !NEED_S)
        return;

    // ---- where pass 2 starts: the last checkpoint no lane passes --------
    int start = G;
    float Px = 0.0f, Ps = 0.0f;
    if constexpr (WALK) {
        // NaN sums flag negative (square root NaN) or NaN samples
        const bool bad = (NEED_S && Ss != Ss) || Sx != Sx || vmin < 0.0f;
        int nck = V1 > G ? (V1 - G - 1) / 64 : 0;
        nck = nck < ncap ? nck : ncap;
        int b0 = 0;
        if (nck > 0 && !__builtin_amdgcn_ballot_w64(active && bad)) {
            for (int b = 1; b <= nck; b += 8) {
                f2v ck[8];
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    // (a block past the last reads the last again)
                    const int bu = b + u <= nck ? b + u : nck;
                    ck[u] = active ? p.ckpt[(size_t)(bu - 1) * plane + line] : f2v{0.0f, 0.0f};
                }
                bool stop = false;
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    const bool pass = (NEED_X && 2.0f * ck[u].x >= Sx) ||
                                      (NEED_S && 2.0f * ck[u].y >= Ss);
                    stop = stop || b + u > nck ||
                           __builtin_amdgcn_ballot_w64(active && pass) != 0;
                    if (!stop) {
                        b0 = b + u;
                        Px = ck[u].x;
                        Ps = ck[u].y;
                    }
                }
                if (stop)
                    break;
            }
        }
        start = G + 64 * b0;
    }

    // ---- pass 2: median walk + integrals -----------------------------
    // The walk is the reference's float prefix.  The integrals only feed
    // values: they accumulate with float FMAs over blocks of 64 steps, each
    // block flushed into a double, so they land within ~1e-7 of the FP64
    // oracle instead of inheriting the reference's sequential float error.
    // The blocks are the 64-step grid v in [64 k, 64 k + 64) whatever step
    // pass 2 starts at (every integral starts at or after it), so the
    // integrals depend neither on the checkpoints nor on the wave's other
    // lines.
    double t1 = 0.0, t2 = 0.0;
    double r3 = 0.0, i3 = 0.0, r4 = 0.0, i4 = 0.0, r5 = 0.0, i5 = 0.0;
    float f1 = 0.0f, f2 = 0.0f;
    float f3r = 0.0f, f3i = 0.0f, f4r = 0.0f, f4i = 0.0f, f5r = 0.0f, f5i = 0.0f;
    int m = kNone, sm = kNone;  // not passed yet
    const bool do3 = p.slot.s[3] >= 0, do4 = p.slot.s[4] >= 0, do5 = p.slot.s[5] >= 0;
    if (lo > 0 || lo > hi) {
        // the walk's first row is a zero: it passes there iff S <= 0
        if (NEED_X && 2.0f * 0.0f >= Sx)
            m = 0;
        if (NEED_S && 2.0f * 0.0f >= Ss)
            sm = 0;
    }
    if (!active)  // a copy of another lane's line: nothing waits for it
        m = sm = 0;
    const float4 *tab34 = reinterpret_cast<const float4 *>(s_tab);
    const float2 *tab5 = s_tab + 2 * p.tabn;
    // T1/T2 and T3..T5 of one row: its sample, distance from the x-median and
    // table rows at the distance from the root median (zero at distance 0)
    auto integrate12 = [&](float x, float rr) {
        const float vr = x * rr;
        f1 += vr;
        f2 = fmaf(vr, rr, f2);
    };
    // (all three, whichever are stored: a test per row costs more)
    auto integrate345 = [&](float x, float4 w34, float2 w5) {
        f3r = fmaf(w34.x, x, f3r);
        f3i = fmaf(w34.y, x, f3i);
        f4r = fmaf(w34.z, x, f4r);
        f4i = fmaf(w34.w, x, f4i);
        f5r = fmaf(w5.x, x, f5r);
        f5i = fmaf(w5.y, x, f5i);
    };
    auto flush = [&] {
        if (NEED_X) {
            t1 += f1;
            t2 += f2;
            f1 = f2 = 0.0f;
        }
        if (DO345) {
            r3 += f3r;
            i3 += f3i;
            r4 += f4r;
            i4 += f4i;
            r5 += f5r;
            i5 += f5i;
            f3r = f3i = f4r = f4i = f5r = f5i = 0.0f;
        }
    };
    bool done = false;  // every lane has passed (wave-uniform)
    for (int v = start; v < V;) {
        const bool plain = v >= va && v < vb2;
        if (plain && done) {
            // the untested groups up to the end of this 64-step block
            int ve = (v & ~63) + 64;
            ve = ve < vb2 ? ve : vb2;
            ve = ve < V ? ve : (V + 7) & ~7;
            const int rb = v - dl;
            float rr = (float)(rb - m);
            const float4 *w34 = tab34 + (rb - sm);
            const float2 *w5 = tab5 + (rb - sm);
            auto use = [&](const Half &h, int base) {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float x = rot_value<TR, false>(h.t[j]);
                    if (NEED_X) {
                        integrate12(x, rr);
                        rr += 1.0f;
                    }
                    if (DO345)
                        integrate345(x, w34[base + j], w5[base + j]);
                }
            };
            Half h0 = load_half(v);
            for (; v < ve; v += 8) {
                Half h1 = load_half(v + 4);
                use(h0, 0);
                h0 = load_half(v + 8 < ve ? v + 8 : v);
                use(h1, 4);
                w34 += 8;
                w5 += 8;
            }
        } else {
            float x[8];
            if (plain) {
                const Half h0 = load_half(v), h1 = load_half(v + 4);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    x[j] = rot_value<TR, false>(h0.t[j]);
                    x[4 + j] = rot_value<TR, false>(h1.t[j]);
                }
            } else {
                load_masked(v, x);
            }
            const int rb = v - dl;
            if (!done) {
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const int r = rb + j;
                    const bool row = (unsigned)r < (unsigned)n;
                    if (NEED_X) {
                        Px += x[j];
                        m = row && m == kNone && 2.0f * Px >= Sx ? r : m;
                    }
                    if (NEED_S) {
                        Ps += line_root<FS>(x[j]);
                        sm = row && sm == kNone && 2.0f * Ps >= Ss ? r : sm;
                    }
                }
            }
            const bool passed = (NEED_X && m != kNone) || (NEED_S && sm != kNone);
            if (__builtin_amdgcn_ballot_w64(active && passed)) {
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const int r = rb + j;
                    if (NEED_X)
                        integrate12(x[j], (float)(r > m ? r - m : 0));
                    if (DO345) {
                        int q = r - sm;
                        const float xq = q > 0 ? x[j] : 0.0f;
                        q = q > 0 ? q : 0;
                        q = q < n ? q : 0;  // a row past the last: sample 0
                        integrate345(xq, tab34[q], tab5[q]);
                    }
                }
            }
            if (!done)
                done = !__builtin_amdgcn_ballot_w64((NEED_X && m == kNone) ||
                                                    (NEED_S && sm == kNone));
            v += 8;
        }
        if ((v & 63) == 0)
            flush();
    }
    flush();
    if (m == kNone) {
        m = n - 1;
        t1 = t2 = 0.0;
    }
    if (sm == kNone) {
        sm = n - 1;
        r3 = i3 = r4 = i4 = r5 = i5 = 0.0;
    }
    if (!active)
        return;
    if (NEED_X && p.med_x)
        p.med_x[line] = m;
    if (NEED_S && p.med_s)
        p.med_s[line] = sm;
    if (p.slot.s[1] >= 0)
        p.sino[p.slot.s[1] * tstride + line] = (float)t1;
    if (p.slot.s[2] >= 0)
        p.sino[p.slot.s[2] * tstride + line] = (float)t2;
    if (DO345) {
        if (do3)
            p.sino[p.slot.s[3] * tstride + line] = (float)hypot(r3, i3);
        if (do4)
            p.sino[p.slot.s[4] * tstride + line] = (float)hypot(r4, i4);
        if (do5)
            p.sino[p.slot.s[5] * tstride + line] = (float)hypot(r5, i5);
        if (p.z345) {
            const size_t plane = (size_t)p.A * n;
            p.z345[line] = f2v{(float)r3, (float)i3};
            p.z345[plane + line] = f2v{(float)r4, (float)i4};
            p.z345[2 * plane + line] = f2v{(float)r5, (float)i5};
        }
    }
}

// One line, with the image copy whose fast axis the lanes step along (TR)
// and the square root the image's bounding-box flag allows (FS).
template <bool PAIRS, bool NEED_X, bool NEED_S, bool DO345, bool CK>
__device__ __forceinline__ void sino_line_any(const LineDst &dst, const float *src,
                                              const float *srcT, const int *bbox,
                                              const float2 *s_tab, int a, int col,
                                              bool active, float2 cs, int lo, int hi)
{
    // Lanes step (dx, dy) = (c, -s) per column; one copy for the whole wave
    const bool tr = __builtin_amdgcn_readfirstlane(fabsf(cs.x) > fabsf(cs.y));
    const bool fs = bbox && bbox[4] == 0;
    if (tr && fs)
        sino_line<true, PAIRS, NEED_X, NEED_S, DO345, CK, true>(dst, srcT, s_tab, a, col, active,
                                                                cs.x, cs.y, lo, hi);
    else if (tr)
        sino_line<true, PAIRS, NEED_X, NEED_S, DO345, CK, false>(dst, srcT, s_tab, a, col, active,
                                                                 cs.x, cs.y, lo, hi);
    else if (fs)
        sino_line<false, PAIRS, NEED_X, NEED_S, DO345, CK, true>(dst, src, s_tab, a, col, active,
                                                                 cs.x, cs.y, lo, hi);
    else
        sino_line<false, PAIRS, NEED_X, NEED_S, DO345, CK, false>(dst, src, s_tab, a, col, active,
                                                                  cs.x, cs.y, lo, hi);
}

// LDS copy of the T3..T5 tables ([3][tabn] float2 in global memory) with the
// T3 and T4 entries of a row interleaved as one float4 (rows 0..tabn-1) and
// T5 after them (float2 at 2*tabn + r).
__device__ __forceinline__ void stage_tab345(float2 *s_tab, const float2 *g, int tabn,
                                             int nthreads)
{
    float4 *s4 = reinterpret_cast<float4 *>(s_tab);
    for (int r = threadIdx.x; r < tabn; r += nthreads) {
        const float2 a = g[r], b = g[tabn + r];
        s4[r] = float4{a.x, a.y, b.x, b.y};
        s_tab[2 * tabn + r] = g[2 * tabn + r];
    }
}

template <bool NEED_X, bool NEED_S, bool DO345>
__global__ __launch_bounds__(kBlock) void sino_t05_kernel(SinoParams p)
{
    extern __shared__ __align__(16) float2 s_tab[];
    if (DO345) {
        stage_tab345(s_tab, p.tab345, p.n, kBlock);
        __syncthreads();
    }
    const int item = xcd_block() * (kBlock / kWave) + wave_id();
    if (item >= p.items)
        return;
    const int a = item / p.nb;
    const int cb = item - a * p.nb;
    const int lane = threadIdx.x & (kWave - 1);
    int col = cb * kWave + lane;
    const bool active = col < p.n;
    if (!active)
        col = p.n - 1;
    const float2 cs = p.trig[a];
    const LineDst dst = {p.sino, p.med_x, p.med_s, p.z345, p.ckpt, p.n, p.A, p.n, p.slot};
    const int2 rows = line_rows(p.bbox, p.n, col, cs.x, cs.y);
    sino_line_any<true, NEED_X, NEED_S, DO345, true>(
        dst, reinterpret_cast<const float *>(p.pair), reinterpret_cast<const float *>(p.pairT),
        p.bbox, s_tab, a, col, active, cs, rows.x, rows.y);
}

// ---------------------------------------------------------------------------
// Batched T0..T5: one persistent launch over every (image, angle tile,
// column tile) wave item of a batch of padded images of uneven side.  A
// tile is tile_a consecutive angles by tile_c consecutive columns (64, 32
// or 16): the wave takes it in tile_a tile_c / 64 passes, in each pass lane
// l on column l % tile_c of angle l / tile_c of the pass.  Waves take items
// from a device counter (dynamic load balance; items are ordered largest
// image first) and find their image by binary search over the descriptors'
// first-item offsets.  The counter is zeroed by reset_counter_kernel ahead
// of each launch.  The image copy a pass reads (row- or column-major) is
// the one that suits the angle of its first lane; the results of a line do
// not depend on the tile.
// ---------------------------------------------------------------------------
template <bool PAIRS, bool NEED_X, bool NEED_S, bool DO345>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4)))
void sino_t05_batched_kernel(BatchSinoParams p)
{
    extern __shared__ __align__(16) float2 s_tab[];
    if (DO345) {
        stage_tab345(s_tab, p.tab345, p.tabn, blockDim.x);
        __syncthreads();
    }
    const int lane = threadIdx.x & (kWave - 1);
    const int sub = kWave / p.tile_c;  // angles per pass
    const int lc = lane & (p.tile_c - 1), la = lane / p.tile_c;
    // one pass per iteration (an item's passes in a row): no loop nested
    // inside the item loop, whose invariants would stay live across the
    // line code
    int item = 0, pass = 0, passes = 0;
    for (;;) {
        if (pass == passes) {
            unsigned int v = 0;
            if (lane == 0)
                v = atomicAdd(p.counter, 1u);
            item = __builtin_amdgcn_readfirstlane(__shfl(v, 0, kWave));
            if (item >= p.items)
                break;
            pass = 0;
        }
        int lo = 0, hi = p.nimg - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (p.images[mid].item0 <= item)
                lo = mid;
            else
                hi = mid - 1;
        }
        const BatchImage im = p.images[lo];
        const int local = item - im.item0;
        const int at = local / im.nb;
        const int cb = local - at * im.nb;
        const int a_first = at * p.tile_a;
        const int a_end = a_first + p.tile_a < p.A ? a_first + p.tile_a : p.A;
        passes = (a_end - a_first + sub - 1) / sub;
        int a = a_first + pass * sub + la;
        pass++;
        int col = cb * p.tile_c + lc;
        const bool active = col < im.n && a < a_end;
        col = col < im.n ? col : im.n - 1;
        a = a < a_end ? a : a_end - 1;
        const float2 cs = p.trig[a];
        const LineDst dst = {im.sino, im.med_x, im.med_s, im.z345, im.ckpt, im.n, p.A, p.tabn,
                             p.slot};
        const int2 rows = line_rows(im.bbox, im.n, col, cs.x, cs.y);
        const float *src = PAIRS ? reinterpret_cast<const float *>(im.pair) : im.img;
        const float *srcT = PAIRS ? reinterpret_cast<const float *>(im.pairT) : im.imgT;
        sino_line_any<PAIRS, NEED_X, NEED_S, DO345, true>(dst, src, srcT, im.bbox, s_tab, a, col,
                                                          active, cs, rows.x, rows.y);
    }
}

__global__ void reset_counter_kernel(unsigned int *c)
{
    if (threadIdx.x == 0)
        c[0] = 0u;
}

__global__ void reset_counters_kernel(unsigned int *c, int count)
{
    if ((int)threadIdx.x < count)
        c[threadIdx.x] = 0u;
}

// The pixel pairs (PAIRS) or the row-major copy of an n x n column-major image
// and the box of its non-zero pixels (launch_image_pairs): block `block` of
// nblocks takes 32 x 32 tiles through LDS (33 x 33, the pairs' second pixels
// included) and leaves its box in box[0..4].
template <bool PAIRS>
__device__ __forceinline__ void image_pairs_block(const float *img, int n, float2 *pair,
                                                  float2 *pairT, float *imgT, int block,
                                                  int nblocks, int *box)
{
    constexpr int S = PAIRS ? 33 : 32;  // pixels of a tile each way
    __shared__ float tile[33][35];
    __shared__ int s_b[5][kBlock / kWave];
    const int tiles = (n + 31) / 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    int x0 = n, x1 = -1, y0 = n, y1 = -1;
    bool narrow = false;  // a pixel that is not 0 or in [2^-45, 2^120]
    for (int t = block; t < tiles * tiles; t += nblocks) {
        const int bx = (t % tiles) * 32, by = (t / tiles) * 32;
        for (int i = threadIdx.x; i < S * S; i += kBlock) {
            const int k = i / S, r = i - S * k;
            const int col = bx + k, row = by + r;
            const bool in = col < n && row < n;
            const float v = in ? img[(size_t)col * n + row] : 0.0f;
            tile[k][r] = v;
            narrow = narrow || !(v == 0.0f || (v >= 0x1p-45f && v <= 0x1p120f));
            if (v != 0.0f) {
                x0 = col < x0 ? col : x0;
                x1 = col > x1 ? col : x1;
                y0 = row < y0 ? row : y0;
                y1 = row > y1 ? row : y1;
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = ty; k < 32; k += 8) {
            const int col = bx + k, row = by + tx;
            const int rowT = by + k, colT = bx + tx;
            if constexpr (PAIRS) {
                if (col < n && row < n)
                    pair[(size_t)col * n + row] = float2{tile[k][tx], tile[k + 1][tx]};
                if (colT < n && rowT < n)
                    pairT[(size_t)rowT * n + colT] = float2{tile[tx][k], tile[tx][k + 1]};
            } else {
                if (colT < n && rowT < n)
                    imgT[(size_t)rowT * n + colT] = tile[tx][k];
            }
        }
        __syncthreads();
    }
    if (PAIRS && block == 0 && threadIdx.x < 2) {  // what a sample's second pair may load
        pair[(size_t)n * n + threadIdx.x] = float2{0.0f, 0.0f};
        pairT[(size_t)n * n + threadIdx.x] = float2{0.0f, 0.0f};
    }
    x0 = wave_min_i(x0);
    x1 = wave_max_i(x1);
    y0 = wave_min_i(y0);
    y1 = wave_max_i(y1);
    const int nw = __ballot(narrow) != 0;
    const int w = threadIdx.x / kWave;
    if ((threadIdx.x & (kWave - 1)) == 0) {
        s_b[0][w] = x0;
        s_b[1][w] = x1;
        s_b[2][w] = y0;
        s_b[3][w] = y1;
        s_b[4][w] = nw;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int nr = s_b[4][0];
        for (int k = 1; k < kBlock / kWave; k++) {
            x0 = s_b[0][k] < x0 ? s_b[0][k] : x0;
            x1 = s_b[1][k] > x1 ? s_b[1][k] : x1;
            y0 = s_b[2][k] < y0 ? s_b[2][k] : y0;
            y1 = s_b[3][k] > y1 ? s_b[3][k] : y1;
            nr |= s_b[4][k];
        }
        box[0] = x0;
        box[1] = x1;
        box[2] = y0;
        box[3] = y1;
        box[4] = nr;
    }
}

// bb[0..4] = the union of the blocks' boxes at bb + 8 (1 + block), by one wave.
__device__ __forceinline__ void image_box_reduce(int n, int nblocks, int *bb)
{
    const int lane = threadIdx.x & (kWave - 1);
    int x0 = n, x1 = -1, y0 = n, y1 = -1, nr = 0;
    for (int k = lane; k < nblocks; k += kWave) {
        const int *b = bb + 8 * (1 + k);
        x0 = b[0] < x0 ? b[0] : x0;
        x1 = b[1] > x1 ? b[1] : x1;
        y0 = b[2] < y0 ? b[2] : y0;
        y1 = b[3] > y1 ? b[3] : y1;
        nr |= b[4];
    }
    x0 = wave_min_i(x0);
    x1 = wave_max_i(x1);
    y0 = wave_min_i(y0);
    y1 = wave_max_i(y1);
    const int narrow = __ballot(nr != 0) != 0;
    if (lane == 0) {
        bb[0] = x0;
        bb[1] = x1;
        bb[2] = y0;
        bb[3] = y1;
        bb[4] = narrow;
    }
}

__global__ __launch_bounds__(kBlock) void image_pairs_kernel(const float *img, int n,
                                                             float2 *pair, float2 *pairT,
                                                             int *bb)
{
    image_pairs_block<true>(img, n, pair, pairT, nullptr, blockIdx.x, gridDim.x,
                            bb + 8 * (1 + blockIdx.x));
}

__global__ void image_box_kernel(int n, int nblocks, int *bb)
{
    image_box_reduce(n, nblocks, bb);
}

// Every image of a batch: grid.y walks the images.  The grid is wide enough
// for the largest; an image's surplus blocks end at once and leave no box
// (with 256 images of 95 to 725 rows two blocks in three had no tile, and
// each reduced and stored an empty box: 298 -> 248 us).
template <bool PAIRS>
__global__ __launch_bounds__(kBlock) void image_pairs_batched_kernel(const BatchImage *images)
{
    const BatchImage &im = images[blockIdx.y];
    const int blocks = pair_blocks(im.n);
    if ((int)blockIdx.x >= blocks)
        return;
    image_pairs_block<PAIRS>(im.img, im.n, im.pair, im.pairT, im.imgT, blockIdx.x, blocks,
                             im.bbox + 8 * (1 + blockIdx.x));
}

__global__ void image_box_batched_kernel(const BatchImage *images, unsigned int *counter)
{
    const BatchImage &im = images[blockIdx.x];
    image_box_reduce(im.n, pair_blocks(im.n), im.bbox);
    if (blockIdx.x == 0 && threadIdx.x == 0)
        *counter = 0u;
}

// ---------------------------------------------------------------------------
// Helper: pad.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void pad_kernel(const float *in, int rows,
                                                     int cols, float *out,
                                                     int n, int dfx, int dfy)
{
    const size_t total = (size_t)n * n;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < total;
         i += (size_t)gridDim.x * kBlock) {
        const int R = (int)(i % n), Cc = (int)(i / n);
        const int r = R - dfy, c = Cc - dfx;
        float v = 0.0f;
        if (r >= 0 && r < rows && c >= 0 && c < cols)
            v = in[(size_t)c * rows + r];
        out[i] = v;
    }
}

// ---------------------------------------------------------------------------
// Block-wide helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ float wave_sum(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        v += __shfl_xor(v, o, kWave);
    return v;
}

__device__ __forceinline__ float block_sum(float v, float *s_red)
{
    v = wave_sum(v);
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0)
        s_red[w] = v;
    __syncthreads();
    float r = 0.0f;
#pragma unroll
    for (int i = 0; i < kBlock / kWave; i++)
        r += s_red[i];
    return r;
}

__device__ __forceinline__ double block_sum_d(double v, double *s_red)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        v += __shfl_xor(v, o, kWave);
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0)
        s_red[w] = v;
    __syncthreads();
    double r = 0.0;
#pragma unroll
    for (int i = 0; i < kBlock / kWave; i++)
        r += s_red[i];
    return r;
}

// findWeightedMedian's walk over x[0..n) in LDS (c++/src/functionals.cpp
// :21-30): first i with 2 * (sequential float prefix) >= S.  One thread;
// x must be 16-byte aligned so the rows come in four at a time.
__device__ int weighted_median_walk(const float *x, int n, float S)
{
    float integral = 0.0f;
    int i = 0;
    for (; i + 4 <= n; i += 4) {
        const float4 v = *reinterpret_cast<const float4 *>(x + i);
        integral += v.x;
        if (2.0f * integral >= S)
            return i;
        integral += v.y;
        if (2.0f * integral >= S)
            return i + 1;
        integral += v.z;
        if (2.0f * integral >= S)
            return i + 2;
        integral += v.w;
        if (2.0f * integral >= S)
            return i + 3;
    }
    for (; i < n; i++) {
        integral += x[i];
        if (2.0f * integral >= S)
            return i;
    }
    return n - 1;
}

// Eigen packet-order sum of x[0..n) in LDS: threads 0..7 run the eight
// stride-8 chains, thread 0 combines (c++/src/functionals.cpp:22 via Eigen
// Redux).  Result broadcast through *s_out.  Must be called by the block.
__device__ void eigen_sum_block(const float *x, int n, float *s_chain, float *s_out)
{
    const int a4 = n & ~3, a8 = n & ~7;
    if (threadIdx.x < 8 && n >= 8) {
        float r = 0.0f;
        for (int i = threadIdx.x; i < a8; i += 8)
            r += x[i];
        s_chain[threadIdx.x] = r;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float res;
        if (a4 == 0) {
            res = n > 0 ? x[0] : 0.0f;
            for (int i = 1; i < n; i++)
                res += x[i];
        } else {
            float ax[4];
            for (int j = 0; j < 4; j++)
                ax[j] = n >= 8 ? s_chain[j] + s_chain[j + 4] : x[j];
            if (n >= 8 && a4 > a8)
                for (int j = 0; j < 4; j++)
                    ax[j] += x[a8 + j];
            res = (ax[0] + ax[2]) + (ax[1] + ax[3]);
            for (int i = a4; i < n; i++)
                res += x[i];
        }
        *s_out = res;
    }
    __syncthreads();
}

// Ascending bitonic sort of s[0..m) (m a power of two) by the whole block.
__device__ void bitonic_sort_lds(float *s, int m)
{
    for (int k = 2; k <= m; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = threadIdx.x; i < m; i += kBlock) {
                const int ixj = i ^ j;
                if (ixj > i) {
                    const bool up = (i & k) == 0;
                    const float a = s[i], b = s[ixj];
                    if ((a > b) == up) {
                        s[i] = b;
                        s[ixj] = a;
                    }
                }
            }
            __syncthreads();
        }
    }
}

// ---------------------------------------------------------------------------
// P-functionals, one workgroup per sinogram column (c++/src/circus.cpp
// :104-177): P1 (functionals.cpp:287-296), P2 (:303-311), P3 (:332-360),
// Hermite (:369-386).
// ---------------------------------------------------------------------------
// LDS layout of one circus workgroup for columns of height up to nmax.
struct CircusLds {
    float *x;      // nmax4
    float *sort;   // pow2 >= nmax
    float *mod;    // nmax4
};

__device__ __forceinline__ CircusLds circus_lds(float *smem, int nmax)
{
    const int n4 = (nmax + 3) & ~3;
    int m2 = 1;
    while (m2 < nmax)
        m2 <<= 1;
    CircusLds l;
    l.x = smem;
    l.sort = l.x + n4;
    l.mod = l.sort + m2;
    return l;
}

// All P-functionals of one sinogram column x[0..n) (already in L.x; P3 reads
// the column's half spectrum spec: real parts, then imaginary parts from
// spec_h on).  Result q goes to out[q * out_stride].
__device__ void circus_column(const CircusLds &L, int n, int np, const int *code,
                              const int *herm, const double *herm_w, float *out,
                              size_t out_stride, int32_t *p2rank,
                              const float *spec, int spec_h, bool wave_done)
{
    __shared__ float s_red[kBlock / kWave];
    __shared__ double s_red_d[kBlock / kWave];
    __shared__ float s_chain[8];
    __shared__ float s_sum;
    __shared__ int s_rank;
    int m2 = 1;
    while (m2 < n)
        m2 <<= 1;
    for (int q = 0; q < np; q++) {
        const int cd = code[q];
        if (cd != 0 && wave_done)
            continue;  // written by circus_wave_kernel
        float res = 0.0f;
        if (cd == 1) {
            float acc = 0.0f;
            for (int i = 1 + threadIdx.x; i < n; i += kBlock)
                acc += fabsf(L.x[i - 1] - L.x[i]);
            res = block_sum(acc, s_red);
        } else if (cd == 0) {
            const double *w = herm_w + (size_t)herm[q] * n;
            double acc = 0.0;
            for (int i = threadIdx.x; i < n; i += kBlock)
                acc = fma((double)L.x[i], w[i], acc);
            res = (float)block_sum_d(acc, s_red_d);
        } else if (cd == 2) {
            for (int i = threadIdx.x; i < m2; i += kBlock)
                L.sort[i] = i < n ? L.x[i] : INFINITY;
            __syncthreads();
            bitonic_sort_lds(L.sort, m2);
            eigen_sum_block(L.sort, n, s_chain, &s_sum);
            if (threadIdx.x == 0)
                s_rank = weighted_median_walk(L.sort, n, s_sum);
            __syncthreads();
            res = L.sort[s_rank];
            if (p2rank && threadIdx.x == 0)
                p2rank[q * out_stride] = s_rank;
        } else {
            // P3 from the column's half spectrum (tt_dft.hip):
            // pow(hypot(Re/N, Im/N), 4) in double, mirrored onto k > N/2,
            // and the trapz sum over the reference's float abscissae
            // lin[p] = -1 + 2p/(N-1) (c++/src/functionals.cpp:53-60, 332-360)
            const int half = n / 2;
            for (int k = threadIdx.x; k <= half; k += kBlock) {
                const double hy = hypot((double)spec[k] / n, (double)spec[spec_h + k] / n);
                const double h2 = hy * hy;
                L.mod[k] = (float)(h2 * h2);
            }
            __syncthreads();
            for (int k = half + 1 + threadIdx.x; k < n; k += kBlock)
                L.mod[k] = L.mod[n - k];
            __syncthreads();
            float acc = 0.0f;
            for (int i = threadIdx.x; i < n - 1; i += kBlock) {
                const float l0 = (float)(-1 + i * 2.0 / (n - 1));
                const float l1 = (float)(-1 + (i + 1) * 2.0 / (n - 1));
                acc += (l1 - l0) * (L.mod[i + 1] + L.mod[i]);
            }
            res = (float)(block_sum(acc, s_red) * 0.5);
        }
        if (threadIdx.x == 0)
            out[q * out_stride] = res;
        __syncthreads();
    }
}

__global__ __launch_bounds__(kBlock) void circus_kernel(CircusParams p)
{
    extern __shared__ __align__(16) float smem[];
    const int n = p.n;
    const CircusLds L = circus_lds(smem, n);
    const int colg = blockIdx.x;   // column over all sinograms
    const int sg = colg / p.ncols;
    const int col = colg - sg * p.ncols;
    const float *x = p.sino + (size_t)colg * n;
    for (int i = threadIdx.x; i < n; i += kBlock)
        L.x[i] = x[i];
    __syncthreads();
    const size_t o = (size_t)sg * p.np * p.ncols + col;
    circus_column(L, n, p.np, p.code, p.herm, p.herm_w, p.out + o, p.ncols,
                  p.p2rank ? p.p2rank + o : nullptr,
                  p.p3_spec ? p.p3_spec + (size_t)colg * 2 * p.p3_h : nullptr, p.p3_h,
                  p.wave_done != 0);
}

// Every sinogram column of a batch; the image is found by binary search over
// the descriptors' first-column offsets.  P3 reads the image's half spectra
// (im.spec, formed by the DFT GEMM as in the single-image path).
__global__ __launch_bounds__(kBlock) void circus_batched_kernel(BatchCircusParams p)
{
    extern __shared__ __align__(16) float smem[];
    const CircusLds L = circus_lds(smem, p.nmax);
    const int colg = blockIdx.x;
    int lo = 0, hi = p.nimg - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (p.images[mid].col0 <= colg)
            lo = mid;
        else
            hi = mid - 1;
    }
    const BatchImage im = p.images[lo];
    const int n = im.n;
    const int lc = colg - im.col0;
    const int t = lc / p.A;
    const int a = lc - t * p.A;
    const float *x = im.sino + ((size_t)t * p.A + a) * n;
    for (int i = threadIdx.x; i < n; i += kBlock)
        L.x[i] = x[i];
    __syncthreads();
    const int herm_none[kMaxP] = {};
    const int h = n / 2 + 1;
    circus_column(L, n, p.np, p.code, herm_none, nullptr,
                  im.circus + (size_t)t * p.np * p.A + a, p.A, nullptr,
                  im.spec ? im.spec + (size_t)lc * 2 * h : nullptr, h, false);
}

// ---------------------------------------------------------------------------
// Sort-based T-functionals T6 (c++/src/functionals.cpp:226-255) and T7
// (:262-276).  One workgroup per line, persistent over lines.  The line's
// column is sampled into LDS with lanes along rows; the medians m and sm come
// from the T0..T5 kernel, which ran first on the same stream.  Sorting is an
// LDS bitonic sort over 64-bit keys (orderable float bits << 32 | index), a
// total order equal to the stable order glibc's merge-sort qsort_r gives
// compareFloat; T7 sorts values only (equal keys are equal values).
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t ord_key(float f)
{
    if (f == 0.0f)
        f = 0.0f;  // -0 and +0 compare equal in compareFloat
    const uint32_t b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

__device__ __forceinline__ float ord_val(uint32_t k)
{
    const uint32_t b = (k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k;
    return __uint_as_float(b);
}

template <class K>
__device__ void bitonic_lds(K *s, int m)
{
    for (int k = 2; k <= m; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = threadIdx.x; i < m; i += kBlock) {
                const int ixj = i ^ j;
                if (ixj > i) {
                    const bool up = (i & k) == 0;
                    const K a = s[i], b = s[ixj];
                    if ((a > b) == up) {
                        s[i] = b;
                        s[ixj] = a;
                    }
                }
            }
            __syncthreads();
        }
    }
}

// 64-bit broadcast from one lane.
// Values of one lane given a wave-uniform lane index (v_readlane: no LDS
// round trip, unlike a shuffle).
__device__ __forceinline__ int lane_int(int v, int l)
{
    return __builtin_amdgcn_readlane(v, l);
}

__device__ __forceinline__ float lane_float(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

__device__ __forceinline__ uint64_t lane_u64(uint64_t v, int l)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), l);
    return ((uint64_t)hi << 32) | lo;
}

// 64-bit shuffle (two 32-bit halves).
__device__ __forceinline__ uint64_t shfl_xor64(uint64_t v, int m)
{
    const int lo = __shfl_xor((int)(uint32_t)v, m, kWave);
    const int hi = __shfl_xor((int)(uint32_t)(v >> 32), m, kWave);
    return ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo;
}

// The sort's keys: float (any values but NaN, -0 as +0) or uint64_t
// (tail_key: the bits of a non-negative float, then an index).  The 64-bit
// keys order as the doubles of the same bits (finite: the high word is at most
// a float infinity, exponent field 0x7F8), so a compare-exchange of two keys of
// either kind is a minimum and a maximum, the 64-bit ones at the rate of the
// 32-bit ones on this chip (an integer compare of 64 bits needs four selects
// more).  Written in assembly: the compiler's fmin would first quiet NaNs
// that cannot occur.
__device__ __forceinline__ uint64_t key_min(uint64_t a, uint64_t b)
{
    uint64_t r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ uint64_t key_max(uint64_t a, uint64_t b)
{
    uint64_t r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float key_min(float a, float b)
{
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float key_max(float a, float b)
{
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// A key that no other sorts after.
template <class Key>
__device__ __forceinline__ Key key_last()
{
    if constexpr (sizeof(Key) == 8)
        return 0x7FEFFFFFFFFFFFFFull;
    else
        return INFINITY;
}
// Float key of a value that is not NaN.
__device__ __forceinline__ float key_of(float v) { return v == 0.0f ? 0.0f : v; }

// Value of lane l ^ LX (LX = 1, 2, 4, 8) by data-parallel moves: full-rate
// VALU instructions (two for 4), where a shuffle is an LDS access at a fifth of
// that rate through one unit per CU.
template <int LX>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v)
{
    static_assert(LX == 1 || LX == 2 || LX == 4 || LX == 8, "within a row of 16 lanes");
    const int x = (int)v;
    if constexpr (LX == 1)
        return (uint32_t)__builtin_amdgcn_mov_dpp(x, 0xB1, 0xf, 0xf, true);  // quad 1 0 3 2
    else if constexpr (LX == 2)
        return (uint32_t)__builtin_amdgcn_mov_dpp(x, 0x4E, 0xf, 0xf, true);  // quad 2 3 0 1
    else if constexpr (LX == 8)
        return (uint32_t)__builtin_amdgcn_mov_dpp(x, 0x128, 0xf, 0xf, true);  // row_ror 8
    // mirrored within 8 lanes (l ^ 7), then within 4 (l ^ 3)
    const int h = __builtin_amdgcn_mov_dpp(x, 0x141, 0xf, 0xf, true);
    return (uint32_t)__builtin_amdgcn_mov_dpp(h, 0x1B, 0xf, 0xf, true);
}

// The values of the two lanes of the pair {l, l ^ LX}, the lower lane's first,
// on both lanes (LX = 16 or 32): the swap of row halves with itself.
template <int LX>
__device__ __forceinline__ uint2 lane_pair(uint32_t v)
{
    static_assert(LX == 16 || LX == 32, "across rows of 16 lanes");
    if constexpr (LX == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return uint2{r[0], r[1]};
    } else {
        const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return uint2{r[0], r[1]};
    }
}

// One bitonic exchange between lanes l and l ^ LX, the lower lane keeping the
// smaller key.  LX < 16: the upper lanes hold their keys negated, so that
// both sides are the minimum of the own key and the negated other one.
template <int LX>
__device__ __forceinline__ void exchange(uint64_t &v, bool lower)
{
    const uint32_t lo = (uint32_t)v, hi = (uint32_t)(v >> 32);
    if constexpr (LX >= 16) {
        const uint2 pl = lane_pair<LX>(lo), ph = lane_pair<LX>(hi);
        const uint64_t a = ((uint64_t)ph.x << 32) | pl.x, b = ((uint64_t)ph.y << 32) | pl.y;
        const bool less = __longlong_as_double((long long)a) < __longlong_as_double((long long)b);
        v = less == lower ? a : b;
    } else {
        const uint64_t b = ((uint64_t)lane_xor<LX>(hi) << 32) | lane_xor<LX>(lo);
        asm("v_min_f64 %0, %0, -%1" : "+v"(v) : "v"(b));
    }
}
template <int LX>
__device__ __forceinline__ void exchange(float &v, bool lower)
{
    if constexpr (LX >= 16) {
        const uint2 p = lane_pair<LX>(__float_as_uint(v));
        // the median with -inf is the minimum, with +inf the maximum
        asm("v_med3_f32 %0, %1, %2, %3"
            : "=v"(v)
            : "v"(p.x), "v"(p.y), "v"(lower ? -INFINITY : INFINITY));
    } else {
        const uint32_t b = lane_xor<LX>(__float_as_uint(v));
        asm("v_min_f32 %0, %0, -%1" : "+v"(v) : "v"(b));
    }
}

// Negates the keys of the lanes where the sign state changes.
template <int KPL>
__device__ __forceinline__ void key_sign(uint64_t (&k)[KPL], bool &neg, bool next)
{
    const uint64_t flip = neg != next ? 1ull << 63 : 0ull;
#pragma unroll
    for (int r = 0; r < KPL; r++)
        k[r] ^= flip;
    neg = next;
}
template <int KPL>
__device__ __forceinline__ void key_sign(float (&k)[KPL], bool &neg, bool next)
{
    const uint32_t flip = neg != next ? 1u << 31 : 0u;
#pragma unroll
    for (int r = 0; r < KPL; r++)
        k[r] = __uint_as_float(__float_as_uint(k[r]) ^ flip);
    neg = next;
}

// Strides LX, LX / 2, .. 1 lanes of a merge; down: the lane's block descends,
// i.e. ascends in its negated keys.
template <int LX, int KPL, class Key>
__device__ __forceinline__ void merge_lanes(Key (&k)[KPL], int lane, bool down, bool &neg)
{
    const bool lower = (lane & LX) == 0;
    key_sign(k, neg, LX >= 16 ? down : down == lower);
#pragma unroll
    for (int r = 0; r < KPL; r++)
        exchange<LX>(k[r], lower);
    if constexpr (LX > 1)
        merge_lanes<LX / 2>(k, lane, down, neg);
}

// In-lane strides S, S / 2, .. 1, ascending.
template <int S, int KPL, class Key>
__device__ __forceinline__ void merge_regs(Key (&k)[KPL])
{
#pragma unroll
    for (int r = 0; r < KPL; r++) {
        const int r2 = r ^ S;
        if (r2 > r) {
            const Key a = k[r], b = k[r2];
            k[r] = key_min(a, b);
            k[r2] = key_max(a, b);
        }
    }
    if constexpr (S > 1)
        merge_regs<S / 2>(k);
}

// Merges of LM lanes' keys, then of 2 LM, .. up to the wave.
template <int LM, int KPL, class Key>
__device__ __forceinline__ void merge_levels(Key (&k)[KPL], int lane, bool neg)
{
    const bool down = (lane & LM) != 0;
    merge_lanes<LM / 2>(k, lane, down, neg);
    if constexpr (KPL > 1 || LM == kWave)
        key_sign(k, neg, down);
    if constexpr (KPL > 1)
        merge_regs<KPL / 2>(k);
    if constexpr (LM < kWave)
        merge_levels<2 * LM>(k, lane, neg);
}

// Ascending bitonic sort of 64*KPL keys (float or uint64_t) held by one
// wave in registers, blocked layout: lane l holds positions l*KPL ..
// l*KPL+KPL-1.  Merge sizes up to KPL stay inside a lane and are unrolled
// with their directions known at compile time; for larger sizes the
// direction depends on the lane only, strides of KPL and more exchange with
// lane l ^ (stride / KPL).  Descending blocks (and, across lanes, the upper
// lane of a pair) hold their keys negated, so every exchange is the same
// minimum and maximum on all lanes.  Wave-synchronous: no barriers; every lane
// of the wave must be active.
//
// No exchange goes through LDS: shuffles (a ds_bpermute a word, 5.5 times a
// VALU instruction's slot at full occupancy) were what the sorts of T6/T7
// waited for.  T6/T7 of 1449^2 pixels at 360 angles 5.2 -> 3.8 ms, P2 of the
// 276480 columns of 256 images 1.81 -> 1.35 ms; bound by VALU issue now (3.5
// slots per 64-bit key and stride across lanes, 1 within a lane).
template <int KPL, class Key>
__device__ __forceinline__ void wave_bitonic_sort(Key (&k)[KPL], int lane)
{
#pragma unroll
    for (int size = 2; size < KPL; size <<= 1) {
#pragma unroll
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
#pragma unroll
            for (int r = 0; r < KPL; r++) {
                const int r2 = r ^ stride;
                if (r2 > r) {
                    const Key a = k[r], b = k[r2];
                    const bool up = (r & size) == 0;
                    k[r] = up ? key_min(a, b) : key_max(a, b);
                    k[r2] = up ? key_max(a, b) : key_min(a, b);
                }
            }
        }
    }
    bool neg = false;
    if constexpr (KPL > 1) {
        key_sign(k, neg, (lane & 1) != 0);  // direction of the size-KPL merge
        merge_regs<KPL / 2>(k);
    }
    merge_levels<2>(k, lane, neg);
}

// Wave-wide reductions.
__device__ __forceinline__ uint64_t wave_max_u64(uint64_t v)
{
#pragma unroll
    for (int m = kWave / 2; m > 0; m >>= 1) {
        const uint64_t o = shfl_xor64(v, m);
        v = o > v ? o : v;
    }
    return v;
}

__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// The sorted square roots of a tail of length L as a compact LDS array c of
// its Le non-trailing entries: position j of the full sequence holds c[j]
// for j < ins, 0 for ins <= j < ins + zt, and c[j - zt] beyond.
struct TailView {
    const float *c;
    int ins, zt, L;
    __device__ __forceinline__ float at(int j) const
    {
        return j < ins ? c[j] : (j < ins + zt ? 0.0f : c[j - zt]);
    }
};

// Sequential float sum of c[i0], c[i0 + 8], ... (i < i1), added to acc.
__device__ __forceinline__ float chain_sum(const float *c, int i0, int i1, float acc)
{
    int i = i0;
    for (; i + 24 < i1; i += 32) {
        const float v0 = c[i], v1 = c[i + 8], v2 = c[i + 16], v3 = c[i + 24];
        acc += v0;
        acc += v1;
        acc += v2;
        acc += v3;
    }
    for (; i < i1; i += 8)
        acc += c[i];
    return acc;
}

// Eigen packet-order sum of a TailView's full sequence (as eigen_sum_block),
// for G = 1 or 2 views at once: lanes 8g .. 8g + 7 run the stride-8 chains
// of the view they pass (group g), lane 8g combines them; the sum of group g
// is returned on lane 8g (other lanes: unspecified).  Adding the zero run's +0 leaves a chain of non-negative
// values unchanged, so chain r sums the compact entries before the run
// (positions r, r + 8, ... below ins) and after it (positions congruent to r
// from ins + zt on, entry = position - zt) and skips the run.
template <int G>
__device__ __forceinline__ float eigen_sum_group(const TailView &v, int lane)
{
    const bool active = lane < 8 * G;
    const int n = v.L;
    const int a4 = n & ~3, a8 = n & ~7;
    const int ch_i = lane & 7;
    float r = 0.0f;
    if (active && n >= 8) {
        const int e1 = v.ins < a8 ? v.ins : a8;
        r = chain_sum(v.c, ch_i, e1, r);
        const int q0 = v.ins + v.zt;
        const int p0 = q0 + ((ch_i - q0) & 7);  // first position >= q0 in chain ch_i
        if (p0 < a8)
            r = chain_sum(v.c, p0 - v.zt, a8 - v.zt, r);
    }
    float ch[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        ch[j] = lane_float(r, j);
        if (G == 2 && lane >= 8)
            ch[j] = lane_float(r, 8 + j);
    }
    float res = 0.0f;
    if (active && ch_i == 0) {
        if (a4 == 0) {
            res = n > 0 ? v.at(0) : 0.0f;
            for (int i = 1; i < n; i++)
                res += v.at(i);
        } else {
            float ax[4];
            for (int j = 0; j < 4; j++)
                ax[j] = n >= 8 ? ch[j] + ch[j + 4] : v.at(j);
            if (n >= 8 && a4 > a8)
                for (int j = 0; j < 4; j++)
                    ax[j] += v.at(a8 + j);
            res = (ax[0] + ax[2]) + (ax[1] + ax[3]);
            for (int i = a4; i < n; i++)
                res += v.at(i);
        }
    }
    return res;
}

// The same for one view (lanes 0..7), the sum returned to every lane.
__device__ __forceinline__ float eigen_sum_view(const TailView &v, int lane)
{
    return lane_float(eigen_sum_group<1>(v, lane), 0);
}

// findWeightedMedian's sequential walk over a TailView (one lane).  Adding
// the zero run leaves the prefix unchanged, so the test can first pass there
// only at its first position (when nothing before it passed, that is only
// possible with ins == 0 and S <= 0).
// Walks c[j0..j1); returns the first passing j + off, or -1 with the prefix
// carried in *integral.  A block of 8 is summed first (the same additions in
// the same order as the element walk, so the same prefixes); when none of its
// values is negative or NaN the prefix does not decrease inside it, so a
// block whose last prefix fails the test holds no passing position and is
// skipped.  Any other block is walked element by element.  NONNEG: every c
// is known to be >= 0 (square roots of non-negative samples), which drops
// the per-block sign test.
template <bool NONNEG>
__device__ __forceinline__ int walk_segment(const float *c, int j0, int j1, int off, float S,
                                            float *integral)
{
    float acc = *integral;
    int j = j0;
    for (; j + 8 <= j1; j += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++)
            v[u] = c[j + u];
        float t = acc;
        bool mono = true;
#pragma unroll
        for (int u = 0; u < 8; u++) {
            t += v[u];
            if (!NONNEG)
                mono = mono & (v[u] >= 0.0f);
        }
        if (mono && !(2.0f * t >= S)) {
            acc = t;
            continue;
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            acc += v[u];
            if (2.0f * acc >= S)
                return j + u + off;
        }
    }
    for (; j < j1; j++) {
        acc += c[j];
        if (2.0f * acc >= S)
            return j + off;
    }
    *integral = acc;
    return -1;
}

template <bool NONNEG>
__device__ __forceinline__ int weighted_median_walk_view(const TailView &v, int Le, float S)
{
    float integral = 0.0f;
    int k = walk_segment<NONNEG>(v.c, 0, v.ins, 0, S, &integral);
    if (k >= 0)
        return k;
    if (v.zt > 0 && 2.0f * integral >= S)
        return v.ins;
    k = walk_segment<NONNEG>(v.c, v.ins, Le, v.zt, S, &integral);
    return k >= 0 ? k : v.L - 1;
}

// Sorted tail of one line for T6 (T6 = true) or T7, given the tail's first
// Le samples in xs[0..Le), no sample negative or NaN, and every sample at
// i >= Le zero (the line has left the rotated image).  Only the first Le keys
// are sorted (K keys per lane, 64*K >= Le); the L - Le trailing zeros are
// placed without sorting: for T7 (value keys) they are the smallest values
// and lead the order; for T6 (w = float(i) * x keys) they have w = 0 and the
// largest indices, so they follow the zero-w keys of the sorted part (stable
// order: ties by ascending index).  Replaces xs[0..Le) by the square roots
// of the sorted part, takes the Eigen-order sum and the sequential walk over
// the full sequence, and returns the key at the weighted-median position k.
template <bool IDX>
using TailKey = typename std::conditional<IDX, uint64_t, float>::type;

// Sort key of tail sample i: T6 w = float(i) * x with the index (stable
// order, and the source row is an output); T7 the value x, with the index
// when its source row is asked for (IDX7), else alone (equal values are
// interchangeable).  Only tails without a negative or NaN sample are sorted,
// so the bits of a float order as its value.  Counts the zero keys of the
// index-carrying kinds.
template <bool T6, bool IDX7>
__device__ __forceinline__ TailKey<T6 || IDX7> tail_key(const float *xs, int i, bool *zero)
{
    const float x = xs[i];
    const float kv = T6 ? (float)i * x : x;
    *zero = kv == 0.0f;
    if constexpr (T6 || IDX7)  // (-0 as +0, as ord_key)
        return ((uint64_t)(__float_as_uint(kv) & 0x7FFFFFFFu) << 32) | (uint32_t)i;
    else
        return key_of(kv);
}

// Highest lane index whose flag is set plus base, or `prev` when none is:
// the largest row index of a 64-row step (consecutive lanes on consecutive
// rows) from one ballot, no cross-lane reduction.
__device__ __forceinline__ int last_set(bool flag, int base, int prev)
{
    const unsigned long long b = __ballot(flag);
    return b ? base + 63 - __clzll(b) : prev;
}

// The key at position k of a tail's full sequence (L = Le + zt entries,
// the zt trailing zeros at ins .. ins + zt - 1), the sorted part's keys in
// blocked layout with KO per lane (a power of two); returned to every lane as
// (orderable value << 32) | index (index 0 for value-only keys).
template <int KR, bool IDX>
__device__ __forceinline__ uint64_t tail_key_at(const TailKey<IDX> (&key)[KR], int KO, int k,
                                                int ins, int zt, int Le)
{
    if (k >= ins && k < ins + zt)  // a trailing zero: w (or x) = +0, index Le + ...
        return ((uint64_t)ord_key(0.0f) << 32) | (uint32_t)(Le + (k - ins));
    const int pos = k < ins ? k : k - zt;
    // KO is a power of two (a network width): shift and mask, no division
    const int sh = __builtin_ctz((unsigned)KO);
    const int pr = pos & (KO - 1), pl = pos >> sh;
    TailKey<IDX> kk = 0;
#pragma unroll
    for (int r = 0; r < KR; r++)
        kk = (r == pr) ? key[r] : kk;
    if constexpr (IDX)  // the orderable form of a non-negative value
        return lane_u64(kk, pl) | (1ull << 63);
    else  // value key in the high word (no index asked for)
        return (uint64_t)ord_key(lane_float(kk, pl)) << 32;
}

// Second half of a sorted tail's median: the sorted part's keys are in
// blocked layout (lane l holds positions l*KO .. l*KO + KO - 1, KO <= KR),
// ins is where the trailing zeros go.  Replaces xs[0..Le) by the square
// roots of the sorted samples, takes the Eigen-order sum and the sequential
// walk over the full sequence, and returns the key at the weighted-median
// position k.
template <int KR, bool T6, bool IDX7>
__device__ __forceinline__ uint64_t tail_finish(const TailKey<T6 || IDX7> (&key)[KR], int KO,
                                                int ins, float *xs, int L, int Le, int lane,
                                                int *k_out, bool fs)
{
    constexpr bool IDX = T6 || IDX7;
    const int zt = L - Le;
    // gather the sorted samples before overwriting the slice with roots
    float sq[KR];
    auto roots = [&](auto fsc) {
        constexpr bool FS = decltype(fsc)::value;
#pragma unroll
        for (int r = 0; r < KR; r++) {
            const int pos = lane * KO + r;
            sq[r] = 0.0f;
            if (r < KO && pos < Le) {
                if constexpr (T6)
                    sq[r] = line_sqrt<FS>(xs[(uint32_t)key[r]]);
                else if constexpr (IDX7)
                    sq[r] = line_sqrt<FS>(__uint_as_float((uint32_t)(key[r] >> 32)));
                else
                    sq[r] = line_sqrt<FS>(key[r]);
            }
        }
    };
    if (fs)
        roots(std::true_type{});
    else
        roots(std::false_type{});
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < KR; r++) {
        const int pos = lane * KO + r;
        if (r < KO && pos < Le)
            xs[pos] = sq[r];
    }
    wave_lds_sync();
    const TailView view = {xs, ins, zt, L};
    const float S = eigen_sum_view(view, lane);
    int k = 0;
    if (lane == 0)
        k = weighted_median_walk_view<true>(view, Le, S);
    k = lane_int(k, 0);
    *k_out = k;
    return tail_key_at<KR, IDX>(key, KO, k, ins, zt, Le);
}

// Sorted tail of one line for T6 (T6 = true) or T7, given the tail's first
// Le samples in xs[0..Le), no sample negative or NaN, and every sample at
// i >= Le zero (the line has left the rotated image).  Only the first Le keys
// are sorted (K keys per lane, 64*K >= Le); the L - Le trailing zeros are
// placed without sorting: for T7 (value keys) they are the smallest values
// and lead the order; for T6 (w = float(i) * x keys) they have w = 0 and the
// largest indices, so they follow the zero-w keys of the sorted part (stable
// order: ties by ascending index).
template <int K, bool T6, bool IDX7>
__device__ __forceinline__ uint64_t sorted_tail_median(float *xs, int L, int Le, int lane,
                                                       int *k_out, bool fs)
{
    constexpr bool IDX = T6 || IDX7;
    using Key = TailKey<IDX>;
    Key key[K];
    int zin = 0;  // zero keys of the sorted part (a popcount per slot)
#pragma unroll
    for (int r = 0; r < K; r++) {
        const int i = r * kWave + lane;  // any placement: the sort orders them
        key[r] = key_last<Key>();
        bool z = false;
        if (i < Le)
            key[r] = tail_key<T6, IDX7>(xs, i, &z);
        if constexpr (IDX)
            zin += __popcll(__ballot(z));
    }
    wave_bitonic_sort<K>(key, lane);
    // where the trailing zeros go: after the sorted part's zero keys in the
    // stable (index) order, or first when the order of equal values is free
    const int ins = IDX ? zin : 0;
    return tail_finish<K, T6, IDX7>(key, K, ins, xs, L, Le, lane, k_out, fs);
}

// The sorted tail with the smallest register network that holds its Le
// sorted keys (at least KMIN, at most KMAX per lane; the networks below
// KMIN are not instantiated).
template <int KMAX, int KMIN, bool T6, bool IDX7>
__device__ __forceinline__ uint64_t sorted_tail_dispatch(float *xs, int L, int Le, int lane,
                                                         int *k, bool fs)
{
    const int kneed = (Le + kWave - 1) / kWave;
    if constexpr (KMIN <= 1)
        if (kneed <= 1 || KMAX == 1)
            return sorted_tail_median<1, T6, IDX7>(xs, L, Le, lane, k, fs);
    if constexpr (KMAX >= 2 && KMIN <= 2)
        if (kneed <= 2 || KMAX == 2)
            return sorted_tail_median<2, T6, IDX7>(xs, L, Le, lane, k, fs);
    if constexpr (KMAX >= 4 && KMIN <= 4)
        if (kneed <= 4 || KMAX == 4)
            return sorted_tail_median<4, T6, IDX7>(xs, L, Le, lane, k, fs);
    if constexpr (KMAX >= 8 && KMIN <= 8)
        if (kneed <= 8 || KMAX == 8)
            return sorted_tail_median<8, T6, IDX7>(xs, L, Le, lane, k, fs);
    if constexpr (KMAX >= 16 && KMIN <= 16)
        if (kneed <= 16 || KMAX == 16)
            return sorted_tail_median<16, T6, IDX7>(xs, L, Le, lane, k, fs);
    if constexpr (KMAX >= 32)
        return sorted_tail_median<32, T6, IDX7>(xs, L, Le, lane, k, fs);
    return 0;  // not reached: kneed <= KMAX
}

// Keys per lane of the network for Le keys: KMIN, 2 KMIN, ... up to KMAX.
template <int KMAX, int KMIN = 1>
__device__ __forceinline__ int keys_per_lane(int Le)
{
    int K = KMIN;
    while (K < KMAX && K * kWave < Le)
        K <<= 1;
    return K;
}

// Sorts the first K of KMAX keys per lane (the rest hold the largest key)
// with the K-per-lane network (K a power of two from KMIN up to KMAX).
template <int KMAX, int KMIN = 1, class Key>
__device__ __forceinline__ void sort_prefix(Key (&k)[KMAX], int K, int lane)
{
    if constexpr (KMIN <= 1)
        if (K <= 1 || KMAX == 1) {
            wave_bitonic_sort<1>(reinterpret_cast<Key(&)[1]>(k), lane);
            return;
        }
    if constexpr (KMAX >= 2 && KMIN <= 2)
        if (K <= 2 || KMAX == 2) {
            wave_bitonic_sort<2>(reinterpret_cast<Key(&)[2]>(k), lane);
            return;
        }
    if constexpr (KMAX >= 4 && KMIN <= 4)
        if (K <= 4 || KMAX == 4) {
            wave_bitonic_sort<4>(reinterpret_cast<Key(&)[4]>(k), lane);
            return;
        }
    if constexpr (KMAX >= 8 && KMIN <= 8)
        if (K <= 8 || KMAX == 8) {
            wave_bitonic_sort<8>(reinterpret_cast<Key(&)[8]>(k), lane);
            return;
        }
    if constexpr (KMAX >= 16)
        wave_bitonic_sort<16>(reinterpret_cast<Key(&)[16]>(k), lane);
}

// P2 of one sinogram column per wave, columns of up to kP2Max rows
// (functionals.cpp:303-311, the weighted median of the sorted column with
// the values as weights, :21-30): the column sorted in the wave's registers
// (value keys: equal values are interchangeable), the sorted values
// into the wave's LDS row, the Eigen-order sum on lanes 0..7 and the
// sequential walk on lane 0.  Entry q of the P list; four columns per
// workgroup.
constexpr int kP2Max = 2048;

// Source row of P2's element (the adjoint's one-hot): the stable order of
// compareFloat (c++/src/functionals.cpp:32-43, ties by ascending index, -0
// equal to +0) puts the r-th occurrence in column order of the value v at
// rank lo + r, lo the number of elements below v.  -1 when v occurs nowhere
// (a NaN median).  Wave-uniform result.
__device__ __forceinline__ int p2_source(const float *x, int n, float v, int k, int lane)
{
    int lo = 0;
    for (int i0 = 0; i0 < n; i0 += kWave) {
        const int i = i0 + lane;
        lo += __popcll(__ballot(i < n && x[i] < v));
    }
    int r = k - lo;
    for (int i0 = 0; i0 < n; i0 += kWave) {
        const int i = i0 + lane;
        uint64_t eq = __ballot(i < n && x[i] == v);
        const int c = __popcll(eq);
        if (r < c) {
            for (int j = 0; j < r; j++)
                eq &= eq - 1;
            return i0 + __ffsll((unsigned long long)eq) - 1;
        }
        r -= c;
    }
    return -1;
}

// P2 of the column x[0..n) (n <= kP2Max) by one wave, sorted values in xs;
// the value and its rank are valid on lane 0, and with src its source row
// (every lane).
template <int KMAX>
__device__ __forceinline__ void p2_wave(const float *x, int n, float *xs, int lane,
                                        float *res, int *rank, int *src = nullptr)
{
    const int K = keys_per_lane<KMAX>(n);
    float key[KMAX];
    bool nan = false;
#pragma unroll
    for (int r = 0; r < KMAX; r++) {
        const int i = r * kWave + lane;
        const float c = r < K && i < n ? x[i] : INFINITY;
        nan = nan || c != c;
        key[r] = key_of(c);
    }
    if (__builtin_amdgcn_ballot_w64(nan)) {
        // a NaN sum: no prefix passes, the last position's value is the
        // largest in the order of ord_key (a positive NaN where there is one)
        uint32_t best = 0;
        for (int i = lane; i < n; i += kWave) {
            const uint32_t o = ord_key(x[i]);
            best = o > best ? o : best;
        }
        best = (uint32_t)wave_max_u64(best);
        *res = ord_val(best);
        *rank = n - 1;
        if (src)
            *src = p2_source(x, n, *res, n - 1, lane);
        return;
    }
    if constexpr (KMAX <= 16) {
        sort_prefix<KMAX>(key, K, lane);
    } else {
        if (K <= 16)
            sort_prefix<16>(reinterpret_cast<float(&)[16]>(key), K, lane);
        else
            wave_bitonic_sort<KMAX>(key, lane);
    }
#pragma unroll
    for (int r = 0; r < KMAX; r++) {
        const int pos = lane * K + r;
        if (r < K && pos < n)
            xs[pos] = key[r];
    }
    wave_lds_sync();
    const TailView v = {xs, 0, 0, n};
    const float S = eigen_sum_view(v, lane);
    int k = 0;
    if (lane == 0)
        k = weighted_median_walk_view<false>(v, n, S);
    k = lane_int(k, 0);
    *res = xs[k];
    *rank = k;
    if (src)
        *src = p2_source(x, n, xs[k], k, lane);
}

// P1 of the column x[0..n) (n >= 2) by one wave: the sum of
// |x[i - 1] - x[i]|, a lane's terms in row order.  Long columns with the loads
// of eight terms under way together: one after the other their latency was the
// time of a few such columns (45 of 2048 rows: 6.2 -> 4.0 us; 4.5 by a
// workgroup a column).  Short ones have no eight terms a lane (270000 columns
// of 33 rows: 71 us with the eight loads, 62 without).
__device__ __forceinline__ float p1_wave(const float *x, int n, int lane)
{
    constexpr int kDeep = 8;
    float acc = 0.0f;
    if (n <= kDeep * kWave) {
        for (int i = 1 + lane; i < n; i += kWave)
            acc += fabsf(x[i - 1] - x[i]);
        return wave_sum(acc);
    }
    for (int i = 1 + lane; i < n; i += kDeep * kWave) {
        float a[kDeep], b[kDeep];
#pragma unroll
        for (int u = 0; u < kDeep; u++) {
            // (a row past the last reads the last again)
            const int j = min(i + u * kWave, n - 1);
            a[u] = x[j - 1];
            b[u] = x[j];
        }
#pragma unroll
        for (int u = 0; u < kDeep; u++)
            acc += i + u * kWave < n ? fabsf(a[u] - b[u]) : 0.0f;
    }
    return wave_sum(acc);
}

// P3 from a column's half spectrum (tt_dft.hip) by one wave, mod in LDS (n / 2
// + 1 floats): (|X| / N)^4 in double (c++/src/functionals.cpp:332-360 takes
// pow(hypot(Re/N, Im/N), 4)), mirrored onto k > N/2, and the trapz sum over
// the reference's float abscissae lin[p] = -1 + 2p/(N-1) (:53-60; the
// quotient corrected by its remainder, the division's own result).
__device__ __forceinline__ float p3_wave(const float *spec, int h, int n, float *mod, int lane)
{
    const int half = n / 2;
    const double inv_n = 1.0 / (double)n, den = (double)(n - 1), inv_d = 1.0 / den;
    for (int k = lane; k <= half; k += kWave) {
        const double re = (double)spec[k] * inv_n, im = (double)spec[h + k] * inv_n;
        const double m2 = fma(re, re, im * im);
        mod[k] = (float)(m2 * m2);
    }
    wave_lds_sync();
    auto lin = [&](int i) {
        const double a = 2.0 * (double)i, q = a * inv_d;
        return (float)(-1.0 + fma(fma(-q, den, a), inv_d, q));
    };
    float acc = 0.0f;
    for (int i = lane; i < n - 1; i += kWave) {
        const int m0 = i <= half ? i : n - i, m1 = i < half ? i + 1 : n - i - 1;
        acc += (lin(i + 1) - lin(i)) * (mod[m1] + mod[m0]);
    }
    const float r = (float)(wave_sum(acc) * 0.5);
    wave_lds_sync();
    return r;
}

// P1, P2 and P3 of one sinogram column by one wave (xs: the wave's 64 KMAX
// floats of LDS), results q of the P list at out[q * stride] (out may be
// null: only the source row is wanted), P2's rank and source row where asked
// for.  Hermite entries are left to the workgroup kernel.
template <int KMAX>
__device__ __forceinline__ void circus_wave_column(const float *x, int n, float *xs, int lane,
                                                   int np, const int *code, float *out,
                                                   size_t stride, int32_t *p2rank,
                                                   int32_t *p2src, const float *spec, int h)
{
    float r1 = 0.0f, r2 = 0.0f, r3 = 0.0f;
    int rank = 0, src = -1;
    bool p1 = false, p2 = p2src != nullptr, p3 = false;
    for (int q = 0; out && q < np; q++) {
        p1 = p1 || code[q] == 1;
        p2 = p2 || code[q] == 2;
        p3 = p3 || code[q] == 3;
    }
    if (p3)
        r3 = p3_wave(spec, h, n, xs, lane);
    if (p1)
        r1 = p1_wave(x, n, lane);
    if (p2)
        p2_wave<KMAX>(x, n, xs, lane, &r2, &rank, p2src ? &src : nullptr);
    if (lane != 0)
        return;
    for (int q = 0; out && q < np; q++) {
        if (code[q] == 0)
            continue;
        out[q * stride] = code[q] == 1 ? r1 : code[q] == 2 ? r2 : r3;
        if (p2rank && code[q] == 2)
            p2rank[q * stride] = rank;
    }
    if (p2src)
        *p2src = src;
}

// One wave per sinogram column of up to 64 KMAX rows, four columns per
// workgroup.  KMAX is the smallest of 8, 16 and 32 that holds the longest
// column: the keys set the registers, hence the waves in flight that hide the
// sequential walk.  One pass over the columns for all three
// functionals, where P1 and P3 took a workgroup per column in a launch of
// their own: P1-P3 of the 276480 columns (avg 407 rows) of 256 images
// 2.23 -> 1.28 ms.
template <int KMAX>
__global__ __launch_bounds__(kBlock) void circus_wave_kernel(CircusParams p)
{
    __shared__ float s_x[kBlock / kWave][kWave * KMAX];
    const int w = wave_id(), lane = threadIdx.x & (kWave - 1);
    const int colg = blockIdx.x * (kBlock / kWave) + w;
    if (colg >= p.ncols * p.nsino)
        return;
    const int sg = colg / p.ncols, col = colg - sg * p.ncols;
    const size_t o = (size_t)sg * p.np * p.ncols + col;
    circus_wave_column<KMAX>(p.sino + (size_t)colg * p.n, p.n, s_x[w], lane, p.np, p.code,
                             p.out + o, p.ncols, p.p2rank ? p.p2rank + o : nullptr, nullptr,
                             p.p3_spec ? p.p3_spec + (size_t)colg * 2 * p.p3_h : nullptr,
                             p.p3_h);
}

// P2's source row of every sinogram column (the adjoint's one-hot), columns
// up to 64 KMAX rows: src[colg] for the n-row columns of sino.
template <int KMAX>
__global__ __launch_bounds__(kBlock) void p2_source_kernel(const float *sino, int n, int cols,
                                                           int32_t *src)
{
    __shared__ float s_x[kBlock / kWave][kWave * KMAX];
    const int w = wave_id(), lane = threadIdx.x & (kWave - 1);
    const int colg = blockIdx.x * (kBlock / kWave) + w;
    if (colg >= cols)
        return;
    circus_wave_column<KMAX>(sino + (size_t)colg * n, n, s_x[w], lane, 0, nullptr, nullptr, 0,
                             nullptr, src + colg, nullptr, 0);
}

// The same over every sinogram column of a batch (image found by binary
// search over the descriptors' first-column offsets; every n <= 64 KMAX).
// Writes the circus values (with_circus) and P2's source row (into the
// image's p2src [nt][A], when set).
template <int KMAX>
__global__ __launch_bounds__(kBlock) void circus_wave_batched_kernel(BatchCircusParams p)
{
    __shared__ float s_x[kBlock / kWave][kWave * KMAX];
    const int w = wave_id(), lane = threadIdx.x & (kWave - 1);
    const int colg = blockIdx.x * (kBlock / kWave) + w;
    if (colg >= p.cols)
        return;
    int lo = 0, hi = p.nimg - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (p.images[mid].col0 <= colg)
            lo = mid;
        else
            hi = mid - 1;
    }
    const BatchImage &im = p.images[lo];
    const int n = im.n, h = n / 2 + 1;
    const int lc = colg - im.col0;
    const int t = lc / p.A;
    const int a = lc - t * p.A;
    circus_wave_column<KMAX>(im.sino + ((size_t)t * p.A + a) * n, n, s_x[w], lane, p.np, p.code,
                             p.with_circus ? im.circus + (size_t)t * p.np * p.A + a : nullptr,
                             p.A, nullptr, im.p2src ? im.p2src + lc : nullptr,
                             im.spec ? im.spec + (size_t)lc * 2 * h : nullptr, h);
}

// findWeightedMedian of one column per wave (columns up to kP2Max rows, in
// their own order, c++/src/circus.cpp:74-78): the column into the wave's LDS
// row, the Eigen-order sum on lanes 0..7 and the walk on lane 0.
__global__ __launch_bounds__(kBlock) void column_median_wave_kernel(const float *in, int n,
                                                                    int cols, int32_t *med)
{
    __shared__ float s_x[kBlock / kWave][kP2Max];
    const int w = wave_id(), lane = threadIdx.x & (kWave - 1);
    const int col = blockIdx.x * (kBlock / kWave) + w;
    if (col >= cols)
        return;
    const float *x = in + (size_t)col * n;
    float *xs = s_x[w];
    for (int i = lane; i < n; i += kWave)
        xs[i] = x[i];
    wave_lds_sync();
    const TailView v = {xs, 0, 0, n};
    const float S = eigen_sum_view(v, lane);
    if (lane == 0)
        med[col] = weighted_median_walk_view<false>(v, n, S);
}

// The largest key of a tail whose first Ls samples are in xs (the rest of
// its L are zero): with a negative or NaN sample, sqrt makes the Eigen sum
// NaN, no prefix passes the test and findWeightedMedian returns the last
// position, i.e. the largest key.
__device__ __forceinline__ uint64_t tail_max_key(const float *xs, int Ls, int L, bool t6,
                                                 int lane)
{
    // the unsampled zeros' largest key: (0, L - 1)
    uint64_t kmax = Ls < L ? (((uint64_t)ord_key(0.0f) << 32) | (uint32_t)(L - 1)) : 0ull;
    for (int i = lane; i < Ls; i += kWave) {
        const float x = xs[i];
        const float kv = t6 ? (float)i * x : x;
        const uint64_t kk = ((uint64_t)ord_key(kv) << 32) | (uint32_t)i;
        kmax = kk > kmax ? kk : kmax;
    }
    return wave_max_u64(kmax);
}

// Lane 0 stores one tail's result: the value, its rank k and source row.
template <bool IDX7>
__device__ __forceinline__ void store_tail_result(const SortTParams &p, int line, int which,
                                                  uint64_t res, int k, int base, int lane)
{
    if (lane != 0)
        return;
    const int slotw = which == 0 ? p.slot6 : p.slot7;
    p.sino[(size_t)slotw * p.A * p.n + line] = ord_val((uint32_t)(res >> 32));
    if (which == 0) {
        if (p.t6_rank)
            p.t6_rank[line] = k;
        if (p.t6_src)
            p.t6_src[line] = (int)(uint32_t)res;
    } else {
        if (p.t7_rank)
            p.t7_rank[line] = k;
        if (IDX7)
            p.t7_src[line] = base + (int)(uint32_t)res;
    }
}

// T6 (which = 0, tail from the sqrt-median sm) or T7 (which = 1, tail from
// the median m) of one line by one wave.  The wave samples the tail into its
// LDS slice, then
//   * if any sample is negative, sqrt makes the Eigen sum NaN, no prefix
//     passes the test and findWeightedMedian returns the last position: the
//     result is the largest key (no sort needed);
//   * otherwise it sorts the part before the trailing zeros with the
//     smallest register network that holds it (K = 1..KMAX keys per lane).
// With DEFER, an entry whose sorted part needs more than KMAX keys per lane
// is left for a wider pass: sort_line then returns true (nothing written).
template <int KMAX, int KMIN, bool DEFER, bool IDX7>
__device__ __forceinline__ bool sort_line(const SortTParams &p, int line, int which,
                                          float *xs, int lane)
{
    constexpr int M = kWave * KMAX;  // capacity of the wave's LDS slice
    const int n = p.n;
    const int slotw = which == 0 ? p.slot6 : p.slot7;
    if (slotw < 0)
        return false;
    const float o = (float)((n - 1) / 2.0);
    const float lim = (float)(n - 1);
    const int a = line / n;
    const int col = line - a * n;
    const float2 cs = p.trig[a];
    const float px = (float)col - o;
    const float pxc = px * cs.x, pxns = px * (-cs.y);
    const bool tr = fabsf(cs.y) > fabsf(cs.x);
    const float *src = reinterpret_cast<const float *>(tr ? p.pairT : p.pair);
    const bool t6 = which == 0;
    const int base = t6 ? p.med_s[line] : p.med_x[line];
    const int L = n - base;
    // rows past the line's last possibly non-zero row sample exactly 0
    const int2 rows = line_rows(p.bbox, n, col, cs.x, cs.y);
    const int Ls = rows.y + 1 - base < L ? rows.y + 1 - base : L;
    // a sampled part longer than the slice cannot sort here: queue it for a
    // wider pass before sampling (its sorted part may turn out shorter;
    // the wider pass then sorts it with the smaller network)
    if (DEFER && Ls > M)
        return true;
    // consecutive lanes take consecutive rows (neighbouring taps)
    int last_nz = -1;
    bool bad = false;
    // (a longer sampled part is queued before sampling, or cannot occur)
    auto sample_tail = [&](auto trc) {
        constexpr bool TRC = decltype(trc)::value;
        float pyo = (float)(base + lane) - o;  // exact steps of 64 rows
        for (int i = lane; i < Ls; i += kWave, pyo += (float)kWave) {
            const float x = rot_sample<TRC, true>(src, n, lim, o, pxc, pxns, cs.x, cs.y, pyo);
            if (i < M)
                xs[i] = x;
            last_nz = last_set(x != 0.0f, i - lane, last_nz);
            bad |= !(x >= 0.0f);  // negative or NaN
        }
    };
    if (tr)
        sample_tail(std::true_type{});
    else
        sample_tail(std::false_type{});
    int k = L - 1;
    uint64_t res;
    if (__any(bad)) {
        wave_lds_sync();
        res = tail_max_key(xs, Ls < M ? Ls : M, L, t6, lane);
    } else {
        // lane 0 took part in every step of the loop: its copy is complete
        const int Le = __builtin_amdgcn_readfirstlane(last_nz) + 1;
        const int kneed = (Le + kWave - 1) / kWave;
        if (DEFER && kneed > KMAX)
            return true;
        wave_lds_sync();
        const bool fs = p.bbox && p.bbox[4] == 0;
        res = t6 ? sorted_tail_dispatch<KMAX, KMIN, true, false>(xs, L, Le, lane, &k, fs)
                 : sorted_tail_dispatch<KMAX, KMIN, false, IDX7>(xs, L, Le, lane, &k, fs);
    }
    store_tail_result<IDX7>(p, line, which, res, k, base, lane);
    return false;
}

// T6 and T7 of one line by one wave (a first pass, both requested).  The
// tails [sm, n) and [m, n) share their rows from max(sm, m) on, so the wave
// samples the union [min(sm, m), E) once into xs (E: the row after the
// line's last possibly non-zero row), sorts both tails' keys, writes the T6
// roots into xs2 and the T7 roots over xs, and runs the two Eigen sums on
// lanes 0..7 and 8..15 and the two walks on lanes 0 and 1 together.
// Returns the entries left for a wider pass (bit 0: T6, bit 1: T7; nothing
// written for them).  A pair whose union exceeds the slice goes entry by
// entry; so do the tails of a pair with a negative or NaN sample (largest
// key), from the shared samples.
template <int KMAX, int KMIN, bool DEFER, bool IDX7>
__device__ __forceinline__ int sort_pair(const SortTParams &p, int line, float *xs, float *xs2,
                                         int lane)
{
    constexpr int M = kWave * KMAX;
    const int n = p.n;
    const float o = (float)((n - 1) / 2.0);
    const float lim = (float)(n - 1);
    const int a = line / n;
    const int col = line - a * n;
    const float2 cs = p.trig[a];
    const float px = (float)col - o;
    const float pxc = px * cs.x, pxns = px * (-cs.y);
    const bool tr = fabsf(cs.y) > fabsf(cs.x);
    const float *src = reinterpret_cast<const float *>(tr ? p.pairT : p.pair);
    const int sm = p.med_s[line], m = p.med_x[line];
    const bool fs = p.bbox && p.bbox[4] == 0;  // short square roots (line_sqrt)
    const int L6 = n - sm, L7 = n - m;
    const int2 rows = line_rows(p.bbox, n, col, cs.x, cs.y);
    const int E = rows.y + 1 < n ? rows.y + 1 : n;
    const int Ls6 = E - sm, Ls7 = E - m;  // sampled lengths (<= 0: no sample)
    int deferred = 0;
    if (DEFER)
        deferred = (Ls6 > M ? 1 : 0) | (Ls7 > M ? 2 : 0);
    const int b0 = sm < m ? sm : m;
    const int Lu = E - b0;
    if (deferred || Lu > M) {
        for (int which = 0; which < 2; which++) {
            if (!((deferred >> which) & 1) &&
                sort_line<KMAX, KMIN, DEFER, IDX7>(p, line, which, xs, lane))
                deferred |= 1 << which;
            wave_lds_sync();
        }
        return deferred;
    }
    int last_nz = -1, last_bad = -1;
    auto sample_union = [&](auto trc) {
        constexpr bool TRC = decltype(trc)::value;
        float pyo = (float)(b0 + lane) - o;  // exact steps of 64 rows
        for (int i = lane; i < Lu; i += kWave, pyo += (float)kWave) {
            const float x = rot_sample<TRC, true>(src, n, lim, o, pxc, pxns, cs.x, cs.y, pyo);
            xs[i] = x;
            last_nz = last_set(x != 0.0f, i - lane, last_nz);
            last_bad = last_set(!(x >= 0.0f), i - lane, last_bad);  // negative or NaN
        }
    };
    if (tr)
        sample_union(std::true_type{});
    else
        sample_union(std::false_type{});
    const int o6 = sm - b0, o7 = m - b0;
    // lane 0 took part in every step of the loop: its copies are complete
    const int lnz = __builtin_amdgcn_readfirstlane(last_nz);
    const int lbad = __builtin_amdgcn_readfirstlane(last_bad);
    const int Le6 = lnz + 1 - o6 > 0 ? lnz + 1 - o6 : 0;
    const int Le7 = lnz + 1 - o7 > 0 ? lnz + 1 - o7 : 0;
    wave_lds_sync();
    if (lbad >= o6 || lbad >= o7) {
        // the bad tails read the shared samples first; then at most one
        // good tail sorts (and overwrites them)
        const bool bad6 = lbad >= o6, bad7 = lbad >= o7;
        uint64_t r6 = 0, r7 = 0;
        int k6 = L6 - 1, k7 = L7 - 1;
        if (bad6)
            r6 = tail_max_key(xs + o6, Ls6, L6, true, lane);
        if (bad7)
            r7 = tail_max_key(xs + o7, Ls7, L7, false, lane);
        wave_lds_sync();
        if (!bad6)
            r6 = sorted_tail_dispatch<KMAX, KMIN, true, false>(xs + o6, L6, Le6, lane, &k6, fs);
        if (!bad7)
            r7 = sorted_tail_dispatch<KMAX, KMIN, false, IDX7>(xs + o7, L7, Le7, lane, &k7, fs);
        store_tail_result<IDX7>(p, line, 0, r6, k6, sm, lane);
        store_tail_result<IDX7>(p, line, 1, r7, k7, m, lane);
        return 0;
    }
    using Key7 = TailKey<IDX7>;
    const int K6 = keys_per_lane<KMAX, KMIN>(Le6), K7 = keys_per_lane<KMAX, KMIN>(Le7);
    // T6 first: keys, sort, its samples gathered by index, roots into xs2
    // (the samples in xs stay for T7's keys, so the two key sets are never
    // both being sorted)
    uint64_t key6[KMAX];
    int ins6 = 0;  // zero keys (a popcount per slot)
#pragma unroll
    for (int r = 0; r < KMAX; r++) {
        const int i = r * kWave + lane;  // < 64 * K: within the first K slots
        bool z = false;
        key6[r] = key_last<uint64_t>();
        if (i < Le6)
            key6[r] = tail_key<true, false>(xs + o6, i, &z);
        ins6 += __popcll(__ballot(z));
    }
    sort_prefix<KMAX, KMIN>(key6, K6, lane);
    auto roots6 = [&](auto fsc) {
        constexpr bool FS = decltype(fsc)::value;
#pragma unroll
        for (int r = 0; r < KMAX; r++) {
            const int p6 = lane * K6 + r;
            if (r < K6 && p6 < Le6)
                xs2[p6] = line_sqrt<FS>(xs[o6 + (uint32_t)key6[r]]);
        }
    };
    if (fs)
        roots6(std::true_type{});
    else
        roots6(std::false_type{});
    // T7: keys, sort, roots from the key values over xs (after every lane
    // has read its samples)
    Key7 key7[KMAX];
    int ins7 = 0;  // zero keys when the order of equal values matters
#pragma unroll
    for (int r = 0; r < KMAX; r++) {
        const int i = r * kWave + lane;
        bool z = false;
        key7[r] = key_last<Key7>();
        if (i < Le7)
            key7[r] = tail_key<false, IDX7>(xs + o7, i, &z);
        if constexpr (IDX7)
            ins7 += __popcll(__ballot(z));
    }
    sort_prefix<KMAX, KMIN>(key7, K7, lane);
    wave_lds_sync();
    auto roots7 = [&](auto fsc) {
        constexpr bool FS = decltype(fsc)::value;
#pragma unroll
        for (int r = 0; r < KMAX; r++) {
            const int p7 = lane * K7 + r;
            if (r < K7 && p7 < Le7) {
                if constexpr (IDX7)
                    xs[p7] = line_sqrt<FS>(__uint_as_float((uint32_t)(key7[r] >> 32)));
                else
                    xs[p7] = line_sqrt<FS>(key7[r]);
            }
        }
    };
    if (fs)
        roots7(std::true_type{});
    else
        roots7(std::false_type{});
    wave_lds_sync();
    const TailView v6 = {xs2, ins6, L6 - Le6, L6}, v7 = {xs, ins7, L7 - Le7, L7};
    const float sg = eigen_sum_group<2>(lane >= 8 ? v7 : v6, lane);
    const float S6 = lane_float(sg, 0), S7 = lane_float(sg, 8);
    int kw = 0;
    if (lane < 2)  // lane 0 walks T6, lane 1 T7
        kw = weighted_median_walk_view<true>(lane ? v7 : v6, lane ? Le7 : Le6, lane ? S7 : S6);
    const int k6 = lane_int(kw, 0), k7 = lane_int(kw, 1);
    const uint64_t r6 = tail_key_at<KMAX, true>(key6, K6, k6, ins6, L6 - Le6, Le6);
    const uint64_t r7 = tail_key_at<KMAX, IDX7>(key7, K7, k7, ins7, L7 - Le7, Le7);
    store_tail_result<IDX7>(p, line, 0, r6, k6, sm, lane);
    store_tail_result<IDX7>(p, line, 1, r7, k7, m, lane);
    return 0;
}

// Persistent waves take work items from the counter p.work (zeroed ahead of
// the launch), p.chunk at a time: a line (T6 and T7) or, with p.defer_in
// set, a queued line item (line << 2 | mask, mask bit 0 for T6 and bit 1
// for T7).  One counter serialises its atomics across the device (tens of
// nanoseconds each), so the cheap items of the first pass go in chunks of
// several lines.  With DEFER, tails whose sorted part needs more than KMAX
// keys per lane are queued in p.defer_out for a wider pass (a wide network's
// VGPR budget would otherwise set the occupancy of every wave); a wave
// collects a chunk's queued items in one register (lane i holds the i-th)
// and queues them with one atomic.  Kernels of at most 16 keys per lane take
// the two tails of a line together when both are requested.  The passes over
// queued items (KMIN = KMAX) build only their widest network: a smaller code
// and fewer spills than one network per width.  The occupancy hints are the
// measured best: the 8-key pass over 1449^2 pixels at 360 angles takes 1.64 ms
// at 4 waves per SIMD (56 bytes spilled), 1.79 at 5 (more spills), 1.82 at 3;
// the 16-key one 2.05 at 3 (none), 2.66 at 2.
template <int KMAX, int KMIN, bool DEFER, bool IDX7>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(KMAX <= 4 ? 4 : KMAX <= 8 ? 4 : KMAX <= 16 ? 3 : 1)))
void sino_sort_kernel(SortTParams p)
{
    constexpr int M = kWave * KMAX;
    // pairing kernels hold two slices per wave
    constexpr bool PAIR = KMAX <= 16;
    constexpr int W = PAIR ? 2 * M : M;
    __shared__ __align__(16) float s_all[(kBlock / kWave) * W];
    const int lane = threadIdx.x & (kWave - 1);
    float *xs = s_all + wave_id() * W;
    const int total = p.defer_in ? (int)*p.defer_in_count : p.A * p.n;
    const int chunk = p.chunk;  // at most 64: one queued item per line fits a wave
    for (;;) {
        int j0 = 0;
        if (lane == 0)
            j0 = (int)atomicAdd(p.work, (unsigned int)chunk);
        j0 = __builtin_amdgcn_readfirstlane(j0);
        if (j0 >= total)
            break;
        const int j1 = j0 + chunk < total ? j0 + chunk : total;
        int queued = 0, nq = 0;
        for (int j = j0; j < j1; j++) {
            int line = j, mask = 3;
            if (p.defer_in) {
                const int e = p.defer_in[j];
                line = e >> 2;
                mask = e & 3;
            }
            mask &= (p.slot6 >= 0 ? 1 : 0) | (p.slot7 >= 0 ? 2 : 0);
            int d = 0;
            if (PAIR && mask == 3) {
                d = sort_pair<KMAX, KMIN, DEFER, IDX7>(p, line, xs, xs + M, lane);
                wave_lds_sync();
            } else {
                for (int which = 0; which < 2; which++) {
                    if (((mask >> which) & 1) &&
                        sort_line<KMAX, KMIN, DEFER, IDX7>(p, line, which, xs, lane))
                        d |= 1 << which;
                    wave_lds_sync();
                }
            }
            if (d) {
                queued = lane == nq ? (line << 2) | d : queued;
                nq++;
            }
        }
        if (DEFER && nq > 0) {
            unsigned int at = 0;
            if (lane == 0)
                at = atomicAdd(p.defer_out_count, (unsigned int)nq);
            at = __builtin_amdgcn_readfirstlane(at);
            if (lane < nq)
                p.defer_out[at + lane] = queued;
        }
    }
}

// ---------------------------------------------------------------------------
// Adjoint kernels.  The medians, the T3..T5 integrals and the sample
// positions are those of a forward recompute on the same image (held fixed,
// as the medians are piecewise constant in the image).
// ---------------------------------------------------------------------------

// One LineRecord per (angle, column): folds the sinogram gradient of every
// requested T0..T5 into the coefficients of G(row); the T6/T7 one-sample
// terms go to a LineRecord67 when those functionals are requested.
__device__ __forceinline__ void make_record(const float *dsino, const int32_t *med_x,
                                            const int32_t *med_s, const int32_t *t6_src,
                                            const int32_t *t7_src, const float2 *z345,
                                            size_t plane, size_t line, Slots slot,
                                            LineRecord *out, LineRecord67 *out67)
{
    LineRecord r = {};
    r.m = med_x ? med_x[line] : 0;
    r.sm = med_s ? med_s[line] : 0;
    if (slot.s[0] >= 0)
        r.g0 = dsino[slot.s[0] * plane + line];
    if (slot.s[1] >= 0)
        r.g1 = dsino[slot.s[1] * plane + line];
    if (slot.s[2] >= 0)
        r.g2 = dsino[slot.s[2] * plane + line];
    for (int k = 0; k < 3; k++) {
        const int sl = slot.s[3 + k];
        if (sl < 0)
            continue;
        const float2 z = z345[k * plane + line];
        const float mag = hypotf(z.x, z.y);
        if (mag > 0.0f) {
            const float g = dsino[sl * plane + line] / mag;
            r.ab[2 * k] = g * z.x;
            r.ab[2 * k + 1] = g * z.y;
        }
    }
    out[line] = r;
    if (out67) {
        LineRecord67 q = {-1, -1, 0.0f, 0.0f};
        if (slot.s[6] >= 0 && t6_src) {
            const int s6 = t6_src[line];
            q.r6 = r.sm + s6;
            q.c6 = dsino[slot.s[6] * plane + line] * (float)s6;
        }
        if (slot.s[7] >= 0 && t7_src) {
            q.r7 = t7_src[line];
            q.c7 = dsino[slot.s[7] * plane + line];
        }
        out67[line] = q;
    }
}

__global__ __launch_bounds__(kBlock) void records_kernel(RecordParams p)
{
    const size_t lines = (size_t)p.A * p.n;
    for (size_t line = (size_t)blockIdx.x * kBlock + threadIdx.x; line < lines;
         line += (size_t)gridDim.x * kBlock)
        make_record(p.dsino, p.med_x, p.med_s, p.t6_src, p.t7_src, p.z345, lines, line,
                    p.slot, p.rec, p.rec67);
}

template <class F>
__device__ __forceinline__ int find_image(const BatchImage *images, int nimg, int v, F key)
{
    int lo = 0, hi = nimg - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (key(images[mid]) <= v)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

__global__ __launch_bounds__(kBlock) void records_batched_kernel(BatchAdjointParams p)
{
    for (int g = blockIdx.x * kBlock + threadIdx.x; g < p.lines; g += gridDim.x * kBlock) {
        const int k = find_image(p.images, p.nimg, g,
                                 [](const BatchImage &b) { return b.line0; });
        const BatchImage &im = p.images[k];
        const size_t plane = (size_t)p.A * im.n;
        const size_t line = (size_t)(g - im.line0);
        make_record(im.dsino, im.med_x, im.med_s, nullptr, nullptr, im.z345, plane, line,
                    p.slot, im.rec, nullptr);
    }
}

// ---------------------------------------------------------------------------
// Transposed bilinear rotation (the adjoint of rotate + interpolate,
// c++/src/auxiliary.cpp:223-255 and :182-196) as a scatter into a pixel tile
// held in LDS, one wave per tile.
//
// For every angle the wave visits the rotated samples (col, row) whose taps
// can touch its pixel tile: those whose exact source position lies in the
// tile grown by one pixel, a rectangle turned by the angle.  Each column's
// rows are cut by both of the rectangle's slabs, and the lanes take them
// without gaps: a work item is three consecutive rows of a column, starting
// at a multiple of three, and the items of every third column (a column
// class) are numbered through.  A lane finds the column of its item by
// counting the bits of a wave-uniform mask of column starts.  Lanes laid out
// as 16 columns x 4 rows of a parallelogram cut by one slab had 1.7 to 2.5
// slots per sample; this has 1.1 (48 images x 720 angles, T0 and T3..T5:
// 76.5 -> 58.6 ms; VALU issue is 74 % of that and the LDS busy 78 %, half of
// it bank conflicts of the scattered accumulators).  Each sample is evaluated
// exactly as the forward evaluates it
// (rot_sample's float operations: coordinates, strict bounds, truncated taps
// and modf fractions), its rotated-domain gradient G(row) comes from its
// column's line record, and G times each of the four tap weights is added
// into the tile's accumulators (LDS, with a halo that is discarded: those
// pixels belong to the neighbouring tiles).
//
// Determinism without atomics: two samples whose lattice positions agree
// modulo 3 in both coordinates are at least 3 apart, more than the 2 sqrt 2
// that two samples with overlapping 2x2 tap footprints can be apart.  The
// samples are visited one residue class (column mod 3, row mod 3) at a
// time, so the 64 lanes of a step read, add to and write back 256 distinct
// accumulators, and a pixel's additions follow program order.  Only the
// owning wave touches a tile's accumulators, so each pixel's sum is formed
// in one fixed order.  Every kGatherFlush angles the float accumulators are
// added into per-lane doubles and cleared.
// ---------------------------------------------------------------------------
constexpr int kGatherFlush = 4;
constexpr int kGatherTile = 32;
constexpr int kGatherTabWords = 6;  // LDS floats per row of the T3..T5 tables
constexpr int kGatherCols = 48;     // staged columns per angle, 16 a class

// Tile class T (16 or 32) in pixels: the items of a column class, about
// (TX + 1) (TY + 1) / 9 plus two thirds per column, just fill one or two
// waves (30 x 32: 123 items in the middle, 132 in 99 of 100, 144 at right
// angles, 1.5 % of the classes above 128; a 32 x 32 tile would need a third
// pass for nine classes in ten).  The bound of ITEMS: the grown tile's chords
// along every third column add up to at most a third of its area and the
// longest chord, a chord of length L holds at most L + 1 rows, and r
// consecutive rows lie in at most (r + 4) / 3 items.
template <int T>
struct GatherShape {
    static constexpr int TX = gather_tx(T), TY = gather_ty(T);
    static constexpr int P = TY + 5;                            // odd accumulator stride
    static constexpr int ACC = (((TX + 4) * P + 3) / 4) * 4;    // floats, halo of two cells
    static constexpr int NPIX = TX * TY / kWave;                // interior pixels per lane
    static constexpr int NIT = T == 16 ? 2 : 3;                 // passes over a class at most
    static constexpr int DIAG = T == 16 ? 31 : 46;              // of the grown tile, rounded up
    static constexpr int COLS = (DIAG + 2) / 3;                 // columns of a class
    static constexpr int ITEMS = (int)(((TX + 1.02) * (TY + 1.02) / 3 + DIAG + 5 * COLS) / 3);
    static_assert(T == 16 || T == 32, "tile classes 16 and 32");
    static_assert(TX * TY % kWave == 0, "whole pixels per lane");
    static_assert((TX + 1.02) * (TX + 1.02) + (TY + 1.02) * (TY + 1.02) < DIAG * DIAG &&
                      DIAG <= kGatherCols - 2 && COLS <= 16,
                  "a footprint's columns have their places");
    static_assert(ITEMS < kWave * NIT, "a class's items lie inside NIT passes");
};

// LDS words of one wave: accumulators, the staged column data (per column:
// (g0, sm, first row, row range), (ab0..ab3), (ab4, ab5), and with T1/T2
// (g1, g2, m, -), with T6/T7 (r6, r7, c6, c7)), and the marks of the columns'
// first items.
template <int T>
__host__ __device__ constexpr int gather_words(bool do12, bool do67)
{
    return GatherShape<T>::ACC + kGatherCols * (4 + 4 + 2 + (do12 ? 4 : 0) + (do67 ? 4 : 0)) +
           kWave * GatherShape<T>::NIT;
}
__host__ __device__ constexpr int gather_wave_words(int T, bool do12, bool do67)
{
    return T == 16 ? gather_words<16>(do12, do67) : gather_words<32>(do12, do67);
}

struct GatherImg {
    const LineRecord *rec;      // [A][n]
    const LineRecord67 *rec67;  // [A][n] or null
    float *out;                 // n x n (or this angle group's partial)
    int n;
};

template <int T, bool DO345, bool DO12>
__device__ __forceinline__ void gather_tile_wave(const GatherImg &im, const float2 *trig,
                                                 const float2 *s_tab, int tabn, int a0,
                                                 int a1, int X0, int Y0, float *wl)
{
    constexpr bool do12 = DO12;
    using S = GatherShape<T>;
    constexpr int P = S::P, TX = S::TX, TY = S::TY, NIT = S::NIT;
    const int lane = threadIdx.x & (kWave - 1);
    const int n = im.n;
    const bool do67 = im.rec67 != nullptr;
    float *acc = wl;
    float4 *sA = reinterpret_cast<float4 *>(wl + S::ACC);
    float4 *sB = sA + kGatherCols;
    float4 *sD = sB + kGatherCols;
    float4 *sE = sD + (do12 ? kGatherCols : 0);
    float2 *sC = reinterpret_cast<float2 *>(sE + (do67 ? kGatherCols : 0));
    uint32_t *mark = reinterpret_cast<uint32_t *>(sC + kGatherCols);  // a byte per class
    const float o = (float)((n - 1) / 2.0);
    const float lim = (float)(n - 1);
    // the tile grown by one pixel, plus a margin far above the float
    // rounding of any sample position (< 1e-3 for n <= 2730), relative to o
    const float dm = 0.01f;
    const int X0m = X0 - 2, Y0m = Y0 - 2;  // accumulator cell 0 (the halo)
    const bool interior = X0 >= 2 && X0 + TX <= n - 2 && Y0 >= 2 && Y0 + TY <= n - 2;
    const float xa = (float)(X0 - 1) - o - dm, xb = (float)(X0 + TX) - o + dm;
    const float ya = (float)(Y0 - 1) - o - dm, yb = (float)(Y0 + TY) - o + dm;
    const float4 z4 = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int i = lane; i < S::ACC / 4; i += kWave)
        reinterpret_cast<float4 *>(acc)[i] = z4;
#pragma unroll
    for (int it = 0; it < NIT; it++)
        mark[it * kWave + lane] = 0;
    double accd[S::NPIX];
#pragma unroll
    for (int i = 0; i < S::NPIX; i++)
        accd[i] = 0.0;
    wave_lds_sync();

    // Footprint of angle a: the columns [c_lo, c_lo + K) the grown tile
    // spans, px = c (x - o) - s (y - o) over its corners.  Lane l stages the
    // column kl = l % 16 of class cc = l / 16 (column index mod 3 == cc), its
    // k-th of the footprint.
    struct Foot {
        float c, s;
        int c_lo, K, k;
    };
    const int scc = lane >> 4;
    auto footprint = [&](int a) {
        Foot f;
        const float2 cs = trig[a];
        f.c = cs.x;
        f.s = cs.y;
        const float p1 = f.c * xa - f.s * ya, p2 = f.c * xb - f.s * ya;
        const float p3 = f.c * xa - f.s * yb, p4 = f.c * xb - f.s * yb;
        const float pmin = fminf(fminf(p1, p2), fminf(p3, p4));
        const float pmax = fmaxf(fmaxf(p1, p2), fmaxf(p3, p4));
        int c_lo = (int)ceilf(pmin + o), c_hi = (int)floorf(pmax + o);
        c_lo = c_lo < 0 ? 0 : c_lo;
        c_hi = c_hi > n - 1 ? n - 1 : c_hi;
        // the diagonal of the grown tile bounds the span: at most 46 columns
        // (16 a class), so the clamp never drops one
        const int K = c_hi - c_lo + 1;
        f.c_lo = c_lo;
        f.K = K > kGatherCols - 2 ? kGatherCols - 2 : K;
        const int koff = scc - c_lo % 3;
        f.k = 3 * (lane & 15) + (koff < 0 ? koff + 3 : koff);
        f.k = scc < 3 && f.k < f.K ? f.k : -1;
        return f;
    };
    // this lane's column record of angle a (f.k >= 0), loaded ahead (global
    // address space: the loads do not wait on LDS traffic)
    typedef const float __attribute__((address_space(1))) *GF;
    auto ld4 = [](GF q) { return float4{q[0], q[1], q[2], q[3]}; };
    float4 pa4 = z4, pb4 = z4, pd4 = z4, pe4 = z4;
    auto prefetch = [&](const Foot &f, int a) {
        if (f.k >= 0) {
            const size_t line = (size_t)a * n + f.c_lo + f.k;
            GF r = (GF)(im.rec + line);
            pa4 = ld4(r);
            if (DO345 || do12)
                pb4 = ld4(r + 4);
            if (do12)
                pd4 = ld4(r + 8);
            if (do67)
                pe4 = ld4((GF)(im.rec67 + line));
        }
    };
    Foot fn = footprint(a0);
    prefetch(fn, a0);
    for (int a = a0; a < a1; a++) {
        const Foot f = fn;
        const float c = f.c, s = f.s;
        // This lane's column: the rows of both slabs (ya <= -s px + c py <= yb
        // and xa <= c px + s py <= xb; a slab along the column cuts nothing),
        // and the number of items they lie in (one that is masked for a
        // column without rows, so that every column has a first item).
        int rlo = 0x3fffff, len = 0, first = 0, cnt = 0;
        if (f.k >= 0) {
            const float px = (float)(f.c_lo + f.k) - o;
            float lo = -o, hi = lim - o;
            if (fabsf(c) > 1e-5f) {
                const float inv = 1.0f / c;
                const float u = (ya + s * px) * inv, v = (yb + s * px) * inv;
                lo = fmaxf(lo, fminf(u, v));
                hi = fminf(hi, fmaxf(u, v));
            }
            if (fabsf(s) > 1e-5f) {
                const float inv = 1.0f / s;
                const float u = (xa - c * px) * inv, v = (xb - c * px) * inv;
                lo = fmaxf(lo, fminf(u, v));
                hi = fminf(hi, fmaxf(u, v));
            }
            cnt = 1;
            if (lo <= hi) {
                const int r0 = max((int)ceilf(lo + o), 0), r1 = min((int)floorf(hi + o), n - 1);
                if (r0 <= r1) {
                    // (thirds of numbers below 2^16)
                    const int b0 = (int)(((uint32_t)r0 * 0xAAABu) >> 17);
                    const int b1 = (int)(((uint32_t)r1 * 0xAAABu) >> 17);
                    rlo = r0;
                    len = r1 - r0;
                    first = 3 * b0;
                    cnt = b1 - b0 + 1;
                }
            }
        }
        // items before this column's in its class (16 lanes)
        int incl = cnt;
        incl += __builtin_amdgcn_update_dpp(0, incl, 0x111, 0xf, 0xf, true);
        incl += __builtin_amdgcn_update_dpp(0, incl, 0x112, 0xf, 0xf, true);
        incl += __builtin_amdgcn_update_dpp(0, incl, 0x114, 0xf, 0xf, true);
        incl += __builtin_amdgcn_update_dpp(0, incl, 0x118, 0xf, 0xf, true);
        const int start = incl - cnt;
        if (f.k >= 0) {
            // (inside NIT passes: GatherShape's ITEMS)
            reinterpret_cast<unsigned char *>(mark)[4 * start + scc] = 1;
            sA[lane] = float4{pa4.x, pa4.y, __int_as_float(first - 3 * start),
                              __int_as_float((rlo << 8) | len)};
            if (DO345) {
                sB[lane] = float4{pa4.z, pa4.w, pb4.x, pb4.y};
                sC[lane] = float2{pb4.z, pb4.w};
            }
            if (do12)
                sD[lane] = pd4;
            if (do67)
                sE[lane] = pe4;
        }
        wave_lds_sync();
        uint32_t mk[NIT];
#pragma unroll
        for (int it = 0; it < NIT; it++)
            mk[it] = mark[it * kWave + lane];
#pragma unroll
        for (int it = 0; it < NIT; it++)
            mark[it * kWave + lane] = 0;
        if (a + 1 < a1) {
            fn = footprint(a + 1);
            prefetch(fn, a + 1);
        }
        // CHK: test the sample positions against the image bounds.  A tile
        // at least 2 pixels inside the image on every side can skip it: its
        // samples lie in the tile grown by a pixel and the margin, inside the
        // image.  There the accumulators reach as far as the samples' taps,
        // so nothing else is tested but the column's row range.
        auto classes = [&](auto chk) {
            constexpr bool CHK = decltype(chk)::value;
            const int clo3 = f.c_lo % 3;
            // one column class (col mod 3) at a time, and in it one row class
            // (row mod 3) after the other over all its items: samples of one
            // residue class are pairwise at least 3 apart, so their 2x2 tap
            // footprints are disjoint and every read-add-write of the class
            // has its own four targets, whatever the lanes' order; the order
            // of the classes is the same for every tiling.
            for (int cc = 0; cc < 3; cc++) {
                const int N = __builtin_amdgcn_readlane(incl, 16 * cc + 15);
                const int koff = cc >= clo3 ? cc - clo3 : cc - clo3 + 3;
                const float pxc0 = (float)(f.c_lo + koff) - o;
                uint64_t mask[NIT];
#pragma unroll
                for (int it = 0; it < NIT; it++)
                    mask[it] = __builtin_amdgcn_ballot_w64(((mk[it] >> (8 * cc)) & 1) != 0);
                struct Item {
                    float g0, pxc, pxns, py;
                    int d, len, q, row;  // d: row - first row of the range
                    float4 eb, ed, ee;
                    float2 ec;
                };
                auto load = [&](int it) {
                    Item t = {};
                    uint64_t m = mask[0];
                    int before = 0;
#pragma unroll
                    for (int j = 1; j < NIT; j++)
                        if (it >= j) {
                            before += __builtin_popcountll(m);
                            m = mask[j];
                        }
                    const uint64_t up = m >> 1;
                    const int kl = __builtin_amdgcn_mbcnt_hi(
                        (uint32_t)(up >> 32),
                        __builtin_amdgcn_mbcnt_lo((uint32_t)up, before + (int)(m & 1) - 1));
                    const int at = 16 * cc + kl;
                    const float4 ea = sA[at];
                    const int w = __float_as_int(ea.w);
                    t.g0 = ea.x;
                    t.row = __float_as_int(ea.z) + 3 * (it * kWave + lane);
                    t.len = w & 255;
                    t.d = t.row - (w >> 8);
                    t.q = t.row - __float_as_int(ea.y);
                    // the forward's sample position (rot_sample), bit for bit;
                    // coordinates relative to o are integers or half-integers
                    // far below 2^23: exact
                    const float px = fmaf(3.0f, (float)kl, pxc0);
                    t.pxc = px * c;
                    t.pxns = px * (-s);
                    t.py = (float)t.row - o;
                    if (DO345) {
                        t.eb = sB[at];
                        t.ec = sC[at];
                    }
                    if (do12)
                        t.ed = sD[at];
                    if (do67)
                        t.ee = sE[at];
                    return t;
                };
                auto add = [&](const Item &t, int rc) {
                    const bool in_range = (unsigned)(t.d + rc) <= (unsigned)t.len;
                    const float py = t.py + (float)rc;
                    const int row = t.row + rc, q = t.q + rc;
                    float x = t.pxc + py * s;
                    float y = t.pxns + py * c;
                    x = x + o;
                    y = y + o;
                    const int Xb = (int)(uint32_t)x, Yb = (int)(uint32_t)y;
                    const bool use = in_range &&
                                     (!CHK || (__float_as_uint(x) < __float_as_uint(lim) &&
                                               __float_as_uint(y) < __float_as_uint(lim)));
                    const float fx = __builtin_amdgcn_fractf(x);
                    const float fy = __builtin_amdgcn_fractf(y);
                    // G(row): g0 + [row >= m] (g1 d + g2 d^2)
                    //   + [row > sm] sum_t (alpha_t W_t.re + beta_t W_t.im)[row - sm]
                    //   + [row == r6] c6 + [row == r7] c7
                    float G = t.g0;
                    if (do12) {
                        const int m = __float_as_int(t.ed.z);
                        const float d = (float)(row - m);
                        const float hh = fmaf(d, fmaf(t.ed.y, d, t.ed.x), G);
                        G = row >= m ? hh : G;
                    }
                    // (a wave whose active lanes all sit at or before their
                    // sm skips the term: a uniform branch)
                    if (DO345 && __builtin_amdgcn_ballot_w64(use && q > 0) != 0) {
                        // table entry 0 is zero, so rows at or before sm add
                        // nothing; q <= n - 1 < tabn in the rows that count
                        const int qc = min(max(q, 0), tabn - 1);
                        const float4 w34 = reinterpret_cast<const float4 *>(s_tab)[qc];
                        const float2 w5 = s_tab[2 * tabn + qc];
                        G = fmaf(t.eb.x, w34.x, G);
                        G = fmaf(t.eb.y, w34.y, G);
                        G = fmaf(t.eb.z, w34.z, G);
                        G = fmaf(t.eb.w, w34.w, G);
                        G = fmaf(t.ec.x, w5.x, G);
                        G = fmaf(t.ec.y, w5.y, G);
                    }
                    if (do67) {
                        G += row == __float_as_int(t.ee.x) ? t.ee.z : 0.0f;
                        G += row == __float_as_int(t.ee.y) ? t.ee.w : 0.0f;
                    }
                    const float ofx = 1.0f - fx, ofy = 1.0f - fy;
                    const float ga = G * ofx, gb = G * fx;
                    if (use) {
                        // cell (Xb - X0m) P + Yb - Y0m: a 24-bit multiply,
                        // which the compiler would otherwise widen to a
                        // quarter-rate 32-bit one
                        int xp;
                        asm volatile("v_mul_u32_u24 %0, %1, %2" : "=v"(xp) : "n"(4 * P), "v"(Xb));
                        float *ca = reinterpret_cast<float *>(
                            reinterpret_cast<char *>(acc) +
                            (xp + 4 * Yb - 4 * (X0m * P + Y0m)));
                        const float a00 = ca[0], a01 = ca[1], a10 = ca[P], a11 = ca[P + 1];
                        ca[0] = a00 + ga * ofy;
                        ca[1] = a01 + ga * fy;
                        ca[P] = a10 + gb * ofy;
                        ca[P + 1] = a11 + gb * fy;
                    }
                };
                if (N <= kWave) {
                    if (N > 0) {
                        const Item t0 = load(0);
#pragma unroll
                        for (int rc = 0; rc < 3; rc++)
                            add(t0, rc);
                    }
                } else if (N <= 2 * kWave) {
                    const Item t0 = load(0), t1 = load(1);
#pragma unroll
                    for (int rc = 0; rc < 3; rc++) {
                        add(t0, rc);
                        add(t1, rc);
                    }
                } else {
                    for (int rc = 0; rc < 3; rc++)
                        for (int it = 0; it * kWave < N && it < NIT; it++)
                            add(load(it), rc);
                }
            }
        };
        if (interior)
            classes(std::false_type{});
        else
            classes(std::true_type{});
        wave_lds_sync();  // staged columns are read; the next angle rewrites them
        if ((a - a0) % kGatherFlush == kGatherFlush - 1 || a == a1 - 1) {
            // flush the float accumulators of these angles into the doubles
#pragma unroll
            for (int i = 0; i < S::NPIX; i++) {
                const int p = lane + kWave * i;
                accd[i] += (double)acc[(p / TY + 2) * P + p % TY + 2];
            }
            wave_lds_sync();
            for (int i = lane; i < S::ACC / 4; i += kWave)
                reinterpret_cast<float4 *>(acc)[i] = z4;
            wave_lds_sync();
        }
    }
#pragma unroll
    for (int i = 0; i < S::NPIX; i++) {
        const int p = lane + kWave * i;
        const int X = X0 + p / TY, Y = Y0 + p % TY;
        if (X < n && Y < n)
            im.out[(size_t)X * n + Y] = (float)accd[i];
    }
}

// Stages the T3..T5 tables into the workgroup's LDS (every wave helps; T3
// and T4 of a row as one float4, T5 after them, as stage_tab345), then
// returns this wave's slice of the dynamic LDS.
__device__ __forceinline__ float *gather_lds(float *smem, const float2 *tab345, int tabn,
                                             bool do345, int wave_words)
{
    const int tab_words = do345 ? kGatherTabWords * tabn : 0;
    if (do345)
        stage_tab345(reinterpret_cast<float2 *>(smem), tab345, tabn, blockDim.x);
    __syncthreads();
    return smem + ((tab_words + 3) & ~3) + wave_id() * wave_words;
}

template <bool DO345, bool DO12>
__global__ __launch_bounds__(1024) void gather_kernel(GatherParams p)
{
    constexpr int T = kGatherTile;
    extern __shared__ float4 smem4[];
    float *smem = reinterpret_cast<float *>(smem4);
    const int words = gather_wave_words(T, DO12, p.rec67 != nullptr);
    float *wl = gather_lds(smem, p.tab345, p.n, DO345, words);
    const int waves = blockDim.x / kWave;
    const int item = blockIdx.x * waves + wave_id();
    const int tiles = gather_tiles(p.n, T);
    if (item >= tiles * p.groups)
        return;
    const int g = item / tiles, tile = item - g * tiles;
    const int tny = (p.n + gather_ty(T) - 1) / gather_ty(T);
    const int a0 = (int)((long long)p.A * g / p.groups);
    const int a1 = (int)((long long)p.A * (g + 1) / p.groups);
    GatherImg im;
    im.rec = p.rec;
    im.rec67 = p.rec67;
    im.out = p.groups > 1 ? p.part + (size_t)g * p.n * p.n : p.dimg;
    im.n = p.n;
    gather_tile_wave<T, DO345, DO12>(im, p.trig, reinterpret_cast<const float2 *>(smem), p.n,
                                     a0, a1, tile / tny * gather_tx(T),
                                     tile % tny * gather_ty(T), wl);
}

// dimg = sum over angle groups of the partial images, in group order.
__global__ __launch_bounds__(kBlock) void gather_reduce_kernel(const float *part, int groups,
                                                               size_t npix, float *dimg)
{
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < npix;
         i += (size_t)gridDim.x * kBlock) {
        double acc = 0.0;
        for (int g = 0; g < groups; g++)
            acc += (double)part[g * npix + i];
        dimg[i] = (float)acc;
    }
}

template <int T, bool DO345, bool DO12>
__global__ __launch_bounds__(1024) void gather_batched_kernel(BatchAdjointParams p)
{
    extern __shared__ float4 smem4[];
    float *smem = reinterpret_cast<float *>(smem4);
    const int words = gather_wave_words(T, DO12, false);
    float *wl = gather_lds(smem, p.tab345, p.tabn, DO345, words);
    const int waves = blockDim.x / kWave;
    const int item = blockIdx.x * waves + wave_id();
    if (item >= p.tiles)
        return;
    const int k = find_image(p.images, p.nimg, item,
                             [](const BatchImage &b) { return b.tile0; });
    const BatchImage &bi = p.images[k];
    const int n = bi.n;
    const int tny = (n + gather_ty(T) - 1) / gather_ty(T);
    const int tile = item - bi.tile0;
    GatherImg im;
    im.rec = bi.rec;
    im.rec67 = nullptr;
    im.out = bi.dimg;
    im.n = n;
    gather_tile_wave<T, DO345, DO12>(im, p.trig, reinterpret_cast<const float2 *>(smem),
                                     p.tabn, 0, p.A, tile / tny * gather_tx(T),
                                     tile % tny * gather_ty(T), wl);
}

// dS = J_P^T dC for every sinogram column (P1: sign differences; P2: one-hot
// at the source of the weighted-median rank of the stable sort; P3: the
// derivative of sum_p w_p |X_q(p)|^4 / N^4, an inverse-DFT-shaped sum;
// Hermite: its weights).
// LDS layout of one circus-VJP workgroup for columns of height up to nmax.
// (sq and key only where P2's source row is found by sorting here)
struct VjpLds {
    float *x;       // nmax4
    float *ds;      // nmax4
    float *sq;      // nmax4
    uint64_t *key;  // pow2 >= nmax
};

__device__ __forceinline__ VjpLds vjp_lds(unsigned char *smem, int nmax)
{
    const int n4 = (nmax + 3) & ~3;
    VjpLds l;
    l.x = reinterpret_cast<float *>(smem);
    l.ds = l.x + n4;
    l.sq = l.ds + n4;
    l.key = reinterpret_cast<uint64_t *>(l.sq + n4);
    return l;
}

// J_P^T dC for the column x[0..n) already in L.x; dc[q * dc_stride] is the
// upstream gradient of P-functional q at this column.  P3's part comes from
// the DFT GEMMs (tt_dft.hip) and is already in out (folded) when p3_done; the P1, P2
// and Hermite parts are added to it and the sum written back to out.
__device__ void circus_vjp_column(const VjpLds &L, int n, int np, const int *code,
                                  const int *herm, const double *herm_w,
                                  const float *dc, size_t dc_stride, float *out,
                                  bool p3_done, const int32_t *p2src)
{
    __shared__ float s_chain[8];
    __shared__ float s_sum;
    __shared__ int s_src;
    int m2 = 1;
    while (m2 < n)
        m2 <<= 1;
    for (int i = threadIdx.x; i < n; i += kBlock)
        L.ds[i] = p3_done ? dft_unfold(out, n, i) : 0.0f;
    __syncthreads();
    for (int q = 0; q < np; q++) {
        const float g = dc[q * dc_stride];
        const int cd = code[q];
        if (cd == 1) {
            for (int j = threadIdx.x; j < n; j += kBlock) {
                float d = 0.0f;
                if (j >= 1) {
                    const float u = L.x[j - 1] - L.x[j];
                    d -= (float)((u > 0.0f) - (u < 0.0f));
                }
                if (j <= n - 2) {
                    const float u = L.x[j] - L.x[j + 1];
                    d += (float)((u > 0.0f) - (u < 0.0f));
                }
                L.ds[j] += g * d;
            }
        } else if (cd == 0) {
            const double *w = herm_w + (size_t)herm[q] * n;
            for (int j = threadIdx.x; j < n; j += kBlock)
                L.ds[j] += (float)((double)g * w[j]);
        } else if (cd == 2 && p2src) {
            // the source row found by the P2 wave kernel (stable order)
            const int sr = *p2src;
            if (threadIdx.x == 0 && sr >= 0)
                L.ds[sr] += g;
        } else if (cd == 2) {
            for (int i = threadIdx.x; i < m2; i += kBlock)
                L.key[i] = i < n ? (((uint64_t)ord_key(L.x[i]) << 32) | (uint32_t)i)
                                 : ~0ull;
            __syncthreads();
            bitonic_lds(L.key, m2);
            for (int i = threadIdx.x; i < n; i += kBlock)
                L.sq[i] = L.x[(int)(uint32_t)L.key[i]];
            __syncthreads();
            eigen_sum_block(L.sq, n, s_chain, &s_sum);
            if (threadIdx.x == 0) {
                const int m = weighted_median_walk(L.sq, n, s_sum);
                s_src = (int)(uint32_t)L.key[m];
            }
            __syncthreads();
            if (threadIdx.x == 0)
                L.ds[s_src] += g;
        }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < n; i += kBlock)
        out[i] = L.ds[i];
}

// dS = J_P^T dC for every sinogram column: P1 sign differences, P2 one-hot
// at the source of the weighted-median rank of the stable sort, Hermite its
// weights, added to P3's part (the derivative of sum_p w_p |X_q(p)|^4 / N^4,
// from the DFT GEMMs) when p3_done.
__global__ __launch_bounds__(kBlock) void circus_vjp_kernel(CircusVjpParams p)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int n = p.n;
    const VjpLds L = vjp_lds(smem_raw, n);
    const int colg = blockIdx.x;
    const int sg = colg / p.ncols;
    const int col = colg - sg * p.ncols;
    const float *x = p.sino + (size_t)colg * n;
    for (int i = threadIdx.x; i < n; i += kBlock)
        L.x[i] = x[i];
    __syncthreads();
    circus_vjp_column(L, n, p.np, p.code, p.herm, p.herm_w,
                      p.dcircus + (size_t)sg * p.np * p.ncols + col, p.ncols,
                      p.dsino + (size_t)colg * n, p.p3_done != 0,
                      p.p2src ? p.p2src + colg : nullptr);
}

__global__ __launch_bounds__(kBlock) void circus_vjp_batched_kernel(BatchAdjointParams p)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const VjpLds L = vjp_lds(smem_raw, p.nmax);
    const int colg = blockIdx.x;
    const int k = find_image(p.images, p.nimg, colg,
                             [](const BatchImage &b) { return b.col0; });
    const BatchImage &im = p.images[k];
    const int n = im.n;
    const int lc = colg - im.col0;       // t * A + a
    const int t = lc / p.A;
    const int a = lc - t * p.A;
    const float *x = im.sino + (size_t)lc * n;
    for (int i = threadIdx.x; i < n; i += kBlock)
        L.x[i] = x[i];
    __syncthreads();
    const int herm_none[kMaxP] = {};
    circus_vjp_column(L, n, p.np, p.code, herm_none, nullptr,
                      im.dcircus + (size_t)t * p.np * p.A + a, p.A,
                      im.dsino + (size_t)lc * n, p.p3_done != 0,
                      im.p2src ? im.p2src + lc : nullptr);
}

// ---------------------------------------------------------------------------
// Steps either side of the path.
// ---------------------------------------------------------------------------

// c++/src/auxiliary.cpp:198-221 (resize): interior pixels sample the input at
// ((col,row) + 0.5) * diag(in_rows/rows, in_cols/cols) - 0.5 with the
// reference's float operations; the one-pixel border stays zero.  Negative
// coordinates (upscaling) keep modf's semantics: integer part -0 -> index 0,
// negative fraction.
__global__ __launch_bounds__(kBlock) void resize_kernel(const float *in, int in_rows,
                                                        int in_cols, float *out,
                                                        int rows, int cols)
{
    const size_t total = (size_t)rows * cols;
    const float t00 = (float)in_rows / (float)rows;
    const float t11 = (float)in_cols / (float)cols;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < total;
         i += (size_t)gridDim.x * kBlock) {
        const int row = (int)(i % rows), col = (int)(i / rows);
        float v = 0.0f;
        if (row >= 1 && row < rows - 1 && col >= 1 && col < cols - 1) {
            const float px = (float)col + 0.5f, py = (float)row + 0.5f;
            float x = px * t00 + py * 0.0f;
            float y = px * 0.0f + py * t11;
            x = x - 0.5f;
            y = y - 0.5f;
            const float xi = __builtin_truncf(x), yi = __builtin_truncf(y);
            const float fx = x - xi, fy = y - yi;
            const int X = (int)xi, Y = (int)yi;
            // The reference scales the column coordinate by the row ratio
            // (and vice versa), so a non-square input reaches past the
            // matrix; those taps read 0 here.
            auto tap = [&](int r, int c) {
                return (r >= 0 && r < in_rows && c >= 0 && c < in_cols)
                           ? in[(size_t)c * in_rows + r]
                           : 0.0f;
            };
            const float s00 = tap(Y, X), s01 = tap(Y, X + 1);
            const float s10 = tap(Y + 1, X), s11 = tap(Y + 1, X + 1);
            v = s00 * (1 - fx) * (1 - fy) + s01 * fx * (1 - fy) +
                s10 * (1 - fx) * fy + s11 * fx * fy;
        }
        out[i] = v;
    }
}

// c++/src/auxiliary.cpp:277-318 (zscore): float mean from a sequential float
// sum, variance in double over float differences, float result.  One
// workgroup per vector.  The sequential sum is the time: its entries come
// from LDS, 16 ahead of the additions (one load from memory per addition took
// 17.8 us for 360 entries, where the launch alone takes about 4).
constexpr int kZscoreChunk = 2048;  // entries staged at a time

__global__ __launch_bounds__(kBlock) void zscore_kernel(const float *in, int n,
                                                        float *out)
{
    __shared__ float4 s_x4[kZscoreChunk / 4];
    __shared__ float s_mean;
    __shared__ double s_red[kBlock / kWave];
    float *s_x = reinterpret_cast<float *>(s_x4);
    const float *x = in + (size_t)blockIdx.x * n;
    float *y = out + (size_t)blockIdx.x * n;
    float sum = 0.0f;
    for (int c0 = 0; c0 < n; c0 += kZscoreChunk) {
        // whole groups of 16, the last filled up with zeros (a sum that began
        // at +0 is never -0, so they change nothing)
        const int m = min(n - c0, kZscoreChunk), m16 = (m + 15) & ~15;
        if (c0 > 0)
            __syncthreads();
        for (int i = threadIdx.x; i < m16; i += kBlock)
            s_x[i] = i < m ? x[c0 + i] : 0.0f;
        __syncthreads();
        if (threadIdx.x < kWave) {
            float4 v[4];
#pragma unroll
            for (int k = 0; k < 4; k++)
                v[k] = s_x4[k];
            for (int i = 4; i <= m16 / 4; i += 4) {
                float4 w[4];
                const int at = i < m16 / 4 ? i : 0;  // (the last group loads nothing new)
#pragma unroll
                for (int k = 0; k < 4; k++)
                    w[k] = s_x4[at + k];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    sum += v[k].x;
                    sum += v[k].y;
                    sum += v[k].z;
                    sum += v[k].w;
                    v[k] = w[k];
                }
            }
        }
    }
    if (threadIdx.x == 0)
        s_mean = sum / (float)n;
    __syncthreads();
    const float mean = s_mean;
    const bool staged = n <= kZscoreChunk;
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += kBlock) {
        const double d = (double)((staged ? s_x[i] : x[i]) - mean);
        acc = fma(d, d, acc);
    }
    const double var = block_sum_d(acc, s_red);
    const float stdev = (float)sqrt(var / (double)(n - 1));
    for (int i = threadIdx.x; i < n; i += kBlock)
        y[i] = ((staged ? s_x[i] : x[i]) - mean) / stdev;
}

// findWeightedMedian of every column of an n x cols matrix (one workgroup per
// column), as nearest_orthonormal_sinogram uses it (c++/src/circus.cpp:74-78).
__global__ __launch_bounds__(kBlock) void column_median_kernel(const float *in, int n,
                                                               int32_t *med)
{
    extern __shared__ __align__(16) float s_col[];
    __shared__ float s_chain[8];
    __shared__ float s_sum;
    const float *x = in + (size_t)blockIdx.x * n;
    for (int i = threadIdx.x; i < n; i += kBlock)
        s_col[i] = x[i];
    __syncthreads();
    eigen_sum_block(s_col, n, s_chain, &s_sum);
    if (threadIdx.x == 0)
        med[blockIdx.x] = weighted_median_walk(s_col, n, s_sum);
}

// Smallest and largest of a sinogram's column medians med[0 .. cols), for
// every thread of the block.
__device__ __forceinline__ int2 block_min_max(const int32_t *med, int cols)
{
    __shared__ int s_mm[2][kBlock / kWave];
    int mn = 1 << 30, mx = -(1 << 30);
    for (int c = threadIdx.x; c < cols; c += kBlock) {
        mn = min(mn, med[c]);
        mx = max(mx, med[c]);
    }
    mn = wave_min_i(mn);
    mx = wave_max_i(mx);
    if ((threadIdx.x & (kWave - 1)) == 0) {
        s_mm[0][threadIdx.x / kWave] = mn;
        s_mm[1][threadIdx.x / kWave] = mx;
    }
    __syncthreads();
    mn = s_mm[0][0];
    mx = s_mm[1][0];
    for (int w = 1; w < kBlock / kWave; w++) {
        mn = min(mn, s_mm[0][w]);
        mx = max(mx, s_mm[1][w]);
    }
    return int2{mn, mx};
}

// aligned(max + row - med[col], col) = in(row, col), zero elsewhere
// (c++/src/circus.cpp:85-93), in double for the SVD, for a batch: grid y =
// sinogram t (sinograms of n x cols back to back, medians med[t * cols + c],
// aligned matrices mstride doubles apart), max the largest median of
// sinogram t.
__global__ __launch_bounds__(kBlock) void align_batched_kernel(const float *in, int n, int cols,
                                                               const int32_t *med,
                                                               int rows_out, size_t mstride,
                                                               double *out)
{
    const int t = blockIdx.y;
    const int32_t *off = med + (size_t)t * cols;
    const int maxoff = block_min_max(off, cols).y;
    const float *src_t = in + (size_t)t * cols * n;
    double *out_t = out + (size_t)t * mstride;
    const size_t total = (size_t)rows_out * cols;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < total;
         i += (size_t)gridDim.x * kBlock) {
        const int r = (int)(i % rows_out), c = (int)(i / rows_out);
        const int src = r - (maxoff - off[c]);
        out_t[i] = (src >= 0 && src < n) ? (double)src_t[(size_t)c * n + src] : 0.0;
    }
}

// Float copy of the aligned rows of a batch of matrices (grid y = matrix t,
// column major with leading dimension ld, mstride doubles apart in, ostride
// floats apart out, leading dimension the matrix's rows): matrix t keeps its
// aligned height n + |max - sc| + |min - sc| of its medians' offsets from
// sc.
__global__ __launch_bounds__(kBlock) void to_float_batched_kernel(const double *in, int ld,
                                                                  size_t mstride, int cols,
                                                                  const int32_t *med, int n,
                                                                  int sc, float *out,
                                                                  size_t ostride)
{
    const int t = blockIdx.y;
    const int2 mm = block_min_max(med + (size_t)t * cols, cols);
    const int rows = n + abs(mm.y - sc) + abs(mm.x - sc);
    const double *in_t = in + (size_t)t * mstride;
    float *out_t = out + (size_t)t * ostride;
    const size_t total = (size_t)rows * cols;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < total;
         i += (size_t)gridDim.x * kBlock) {
        const int r = (int)(i % rows), c = (int)(i / rows);
        out_t[i] = (float)in_t[(size_t)c * ld + r];
    }
}

// out(i, j) = v(i, j) / sqrt(lambda_j) for count column-major k x k matrices
// (eigenvectors v, eigenvalues lambda, k per matrix).
__global__ __launch_bounds__(kBlock) void scale_eigvec_kernel(const double *v,
                                                             const double *lambda, int k,
                                                             int count, double *out)
{
    const size_t kk = (size_t)k * k, total = kk * count;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < total;
         i += (size_t)gridDim.x * kBlock) {
        const size_t m = i / kk;
        const int j = (int)((i - m * kk) / k);
        out[i] = v[i] / sqrt(lambda[m * k + j]);
    }
}

// x <- 1.5 I - 0.5 x for count k x k matrices (one Newton-Schulz factor).
__global__ __launch_bounds__(kBlock) void newton_schulz_factor_kernel(double *x, int k,
                                                                     int count)
{
    const size_t kk = (size_t)k * k, total = kk * count;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < total;
         i += (size_t)gridDim.x * kBlock) {
        const size_t e = i % kk;
        const int r = (int)(e % k), c = (int)(e / k);
        x[i] = (r == c ? 1.5 : 0.0) - 0.5 * x[i];
    }
}

// Polar iteration of the nearest orthonormal sinogram (X <- X q(X^T X)).
// The Gram matrices come from a GEMM split over row chunks: S_m = sum over
// c < chunks of part[m * chunks + c], summed in chunk order (deterministic).
__global__ __launch_bounds__(kBlock) void nos_reduce_kernel(const double *part, int chunks,
                                                           size_t kk, int count, double *S)
{
    const size_t total = kk * count;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < total;
         i += (size_t)gridDim.x * kBlock) {
        const size_t m = i / kk, e = i - m * kk;
        const double *p = part + m * chunks * kk + e;
        double acc = p[0];
        for (int c = 1; c < chunks; c++)
            acc += p[c * kk];
        S[i] = acc;
    }
}

// Per-slice partial reductions of each k x k matrix (grid: kNosSlices x
// count): sum of squares (WHAT = 0) or max |S - I| (WHAT = 1, NaN
// propagates), into part[m * kNosSlices + slice].
template <int WHAT>
__global__ __launch_bounds__(kBlock) void nos_slice_kernel(const double *S, int k, double *part)
{
    __shared__ double s_red[kBlock / kWave];
    const size_t kk = (size_t)k * k;
    const double *M = S + kk * blockIdx.y;
    const size_t per = (kk + gridDim.x - 1) / gridDim.x;
    const size_t i0 = per * blockIdx.x, i1 = i0 + per < kk ? i0 + per : kk;
    double acc = 0.0;
    for (size_t i = i0 + threadIdx.x; i < i1; i += kBlock) {
        if (WHAT == 0) {
            acc += M[i] * M[i];
        } else {
            const double v = fabs(M[i] - ((i % k) == (i / k) ? 1.0 : 0.0));
            acc = (v > acc || v != v) ? v : acc;
        }
    }
    if (WHAT == 0) {
        acc = block_sum_d(acc, s_red);
    } else {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const double v = __shfl_xor(acc, o, kWave);
            acc = (v > acc || v != v) ? v : acc;
        }
        __syncthreads();
        if ((threadIdx.x & 63) == 0)
            s_red[threadIdx.x >> 6] = acc;
        __syncthreads();
        acc = s_red[0];
        for (int w = 1; w < kBlock / kWave; w++)
            acc = (s_red[w] > acc || s_red[w] != s_red[w]) ? s_red[w] : acc;
    }
    if (threadIdx.x == 0)
        part[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = acc;
}

// Scales of the first step from the Gram matrices' squared Frobenius norms
// f2 (sums of the slices, in order): s = ||G||_F^-1 normalises S_0 = s G
// (every eigenvalue in [0, 1]) and r = ||G||_F^(-1/2) scales X_0 = A r; both
// 0 for a zero matrix, which then never converges.
__global__ void nos_scales_kernel(const double *part, int slices, int count, double *s,
                                  double *r)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m < count) {
        double f2 = 0.0;
        for (int j = 0; j < slices; j++)
            f2 += part[(size_t)m * slices + j];
        const double f = sqrt(f2);
        s[m] = f > 0.0 ? 1.0 / f : 0.0;
        r[m] = f > 0.0 ? 1.0 / sqrt(f) : 0.0;
    }
}

// The elementwise part of Q = q(S) = c0 I + c1 S + c2 S^2 + c3 S^3 + c4 S^4
// (Paterson-Stockmeyer: Q = (c0 I + c1 S + c2 S^2) + S^2 (c3 S + c4 S^2),
// the product added by a GEMM).  In the first step S and S2 hold G and G G
// unnormalised, S_0 = s G, and Q is scaled by r (X_1 = A r q(S_0)):
// a = s S, b = s^2 S2, Q = r (c0 I + c1 a + c2 b) and T = s^2 r (c3 a +
// c4 b), so that S2 T = S_0^2 r (c3 S_0 + c4 S_0^2).  Later steps: s = r = 1
// (null pointers).
__global__ __launch_bounds__(kBlock) void nos_poly_kernel(const double *S, const double *S2,
                                                         int k, int count, PolarStep c,
                                                         const double *scale, const double *r,
                                                         double *T, double *Q)
{
    const size_t kk = (size_t)k * k, total = kk * count;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < total;
         i += (size_t)gridDim.x * kBlock) {
        const size_t m = i / kk, e = i - m * kk;
        const double sc = scale ? scale[m] : 1.0, rr = r ? r[m] : 1.0;
        const double a = sc * S[i], b = sc * sc * S2[i];
        const double d = (e % k) == (e / k) ? c.c[0] : 0.0;
        T[i] = sc * sc * rr * (c.c[3] * a + c.c[4] * b);
        Q[i] = rr * (d + c.c[1] * a + c.c[2] * b);
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
hipError_t launch_pad(const float *in, int rows, int cols, float *out, int n,
                      int dfx, int dfy, hipStream_t s)
{
    size_t total = (size_t)n * n;
    int blocks = (int)((total + kBlock - 1) / kBlock);
    if (blocks > 4096)
        blocks = 4096;
    pad_kernel<<<blocks, kBlock, 0, s>>>(in, rows, cols, out, n, dfx, dfy);
    return hipGetLastError();
}

hipError_t launch_sino_t05(const SinoParams &p, bool need_x, bool need_s,
                           bool do345, hipStream_t s)
{
    const int wpb = kBlock / kWave;
    int blocks = (p.items + wpb - 1) / wpb;
    blocks = (blocks + kNumXcd - 1) / kNumXcd * kNumXcd;
    const size_t shm = do345 ? sizeof(float2) * 3 * (size_t)p.n : 0;
#define TT_LAUNCH(X, S, D)                                                     \
    sino_t05_kernel<X, S, D><<<blocks, kBlock, shm, s>>>(p)
    if (need_x && need_s && do345)
        TT_LAUNCH(true, true, true);
    else if (need_x && need_s)
        TT_LAUNCH(true, true, false);
    else if (need_x)
        TT_LAUNCH(true, false, false);
    else if (need_s && do345)
        TT_LAUNCH(false, true, true);
    else if (need_s)
        TT_LAUNCH(false, true, false);
    else
        TT_LAUNCH(false, false, false);
#undef TT_LAUNCH
    return hipGetLastError();
}

static size_t circus_shm(int nmax)
{
    int m2 = 1;
    while (m2 < nmax)
        m2 <<= 1;
    const size_t n4 = ((size_t)nmax + 3) & ~(size_t)3;
    return sizeof(float) * (2 * n4 + m2);
}

// Calls f with the key width of columns of up to n (<= kP2Max) rows.
template <class F>
static void with_key_width(int n, F f)
{
    if (n <= 8 * kWave)
        f(std::integral_constant<int, 8>{});
    else if (n <= 16 * kWave)
        f(std::integral_constant<int, 16>{});
    else
        f(std::integral_constant<int, 32>{});
}

static int wave_blocks(int cols)
{
    const int wpb = kBlock / kWave;
    return (cols + wpb - 1) / wpb;
}

hipError_t launch_circus(const CircusParams &p, hipStream_t s)
{
    // P1..P3 of columns up to kP2Max rows: one wave per column; Hermite
    // entries, and every entry of longer columns: one workgroup per column.
    // A list with Hermite entries has that second launch anyway, which takes
    // its P1 and P3 along unless P2's sort needs the wave (P1 and one Hermite
    // entry of 45 columns of 725 rows: 12.5 us in two launches, 9.6 in one;
    // of 2880 columns of 2048 rows 27.6 and 13.4).
    CircusParams c = p;
    const int cols = p.ncols * p.nsino;
    bool p2 = false, herm = false, other = false;
    for (int q = 0; q < p.np; q++) {
        p2 = p2 || p.code[q] == 2;
        herm = herm || p.code[q] == 0;
        other = other || p.code[q] != 0;
    }
    const bool wave = other && p.n <= kP2Max && (p2 || !herm);
    const bool block = herm || (other && !wave);
    c.wave_done = wave;
    if (wave)
        with_key_width(p.n, [&](auto K) {
            circus_wave_kernel<decltype(K)::value><<<wave_blocks(cols), kBlock, 0, s>>>(c);
        });
    if (block)
        circus_kernel<<<cols, kBlock, circus_shm(p.n), s>>>(c);
    return hipGetLastError();
}

hipError_t launch_p2_source(const float *sino, int n, int cols, int32_t *src, hipStream_t s)
{
    if (n > kP2Max)
        return hipErrorInvalidValue;
    with_key_width(n, [&](auto K) {
        p2_source_kernel<decltype(K)::value>
            <<<wave_blocks(cols), kBlock, 0, s>>>(sino, n, cols, src);
    });
    return hipGetLastError();
}

static void launch_circus_wave_batched(const BatchCircusParams &p, hipStream_t s)
{
    with_key_width(p.nmax, [&](auto K) {
        circus_wave_batched_kernel<decltype(K)::value>
            <<<wave_blocks(p.cols), kBlock, 0, s>>>(p);
    });
}

hipError_t launch_p2_source_batched(const BatchCircusParams &p, hipStream_t s)
{
    if (p.nmax > kP2Max)
        return hipErrorInvalidValue;
    BatchCircusParams c = p;
    c.with_circus = 0;
    launch_circus_wave_batched(c, s);
    return hipGetLastError();
}

hipError_t launch_circus_batched(const BatchCircusParams &p, hipStream_t s)
{
    // as launch_circus (no Hermite entries in a batch)
    if (p.nmax <= kP2Max)
        launch_circus_wave_batched(p, s);
    else
        circus_batched_kernel<<<p.cols, kBlock, circus_shm(p.nmax), s>>>(p);
    return hipGetLastError();
}

hipError_t launch_image_pairs(const float *img, int n, float2 *pair, float2 *pairT, int *bbox,
                              hipStream_t s)
{
    const int blocks = pair_blocks(n);
    image_pairs_kernel<<<blocks, kBlock, 0, s>>>(img, n, pair, pairT, bbox);
    image_box_kernel<<<1, kWave, 0, s>>>(n, blocks, bbox);
    return hipGetLastError();
}

hipError_t launch_image_pairs_batched(const BatchImage *images, int nimg, int nmax, bool pairs,
                                      unsigned int *counter, hipStream_t s)
{
    const dim3 grid(pair_blocks(nmax), nimg);
    if (pairs)
        image_pairs_batched_kernel<true><<<grid, kBlock, 0, s>>>(images);
    else
        image_pairs_batched_kernel<false><<<grid, kBlock, 0, s>>>(images);
    image_box_batched_kernel<<<nimg, kWave, 0, s>>>(images, counter);
    return hipGetLastError();
}

hipError_t launch_reset_counter(unsigned int *counter, hipStream_t s)
{
    reset_counter_kernel<<<1, kWave, 0, s>>>(counter);
    return hipGetLastError();
}

hipError_t launch_sino_t05_batched(const BatchSinoParams &p, bool need_x,
                                   bool need_s, bool do345, int waves_per_block,
                                   int blocks, hipStream_t s)
{
    if (!line_tile_ok(p.tile_a, p.tile_c))
        return hipErrorInvalidValue;
    const int threads = kWave * waves_per_block;
    const size_t shm = do345 ? sizeof(float2) * 3 * (size_t)p.tabn : 0;
#define TT_LAUNCH(P, X, S, D)                                                  \
    sino_t05_batched_kernel<P, X, S, D><<<blocks, threads, shm, s>>>(p)
#define TT_LAUNCH_P(P)                                                         \
    do {                                                                       \
        if (need_x && need_s && do345)                                         \
            TT_LAUNCH(P, true, true, true);                                    \
        else if (need_x && need_s)                                             \
            TT_LAUNCH(P, true, true, false);                                   \
        else if (need_x)                                                       \
            TT_LAUNCH(P, true, false, false);                                  \
        else if (need_s && do345)                                              \
            TT_LAUNCH(P, false, true, true);                                   \
        else if (need_s)                                                       \
            TT_LAUNCH(P, false, true, false);                                  \
        else                                                                   \
            TT_LAUNCH(P, false, false, false);                                 \
    } while (0)
    if (p.pairs)
        TT_LAUNCH_P(true);
    else
        TT_LAUNCH_P(false);
#undef TT_LAUNCH_P
#undef TT_LAUNCH
    return hipGetLastError();
}

// Workgroups of one sort pass that fit on the device at once (the waves are
// persistent, so more would only wait).
template <int KMAX, int KMIN, bool DEFER, bool IDX7>
static int sort_blocks(int cus, int items = 0x7fffffff)
{
    static int per_cu = 0;
    if (per_cu == 0) {
        int b = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &b, sino_sort_kernel<KMAX, KMIN, DEFER, IDX7>, kBlock, 0) != hipSuccess || b < 1)
            b = 2;
        per_cu = b;
    }
    const int need = (int)(((long long)items + kBlock / kWave - 1) / (kBlock / kWave));
    return cus * per_cu < need ? cus * per_cu : need;
}

template <bool IDX7>
static hipError_t sino_sort_passes(const SortTParams &p_in, int32_t *queue_a,
                            int32_t *queue_b, unsigned int *counts, hipStream_t s)
{
    SortTParams p = p_in;
    p.defer_in = nullptr;
    p.defer_in_count = nullptr;
    if (p.n > 2048 || !counts)
        return hipErrorInvalidValue;
    const int lines = p.A * p.n;
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) == hipSuccess)
        (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    // counts: [0], [1] queue lengths, [2..4] the passes' work counters
    reset_counters_kernel<<<1, kWave, 0, s>>>(counts, kSortCounters);
    p.work = counts + 2;
    p.chunk = 8;
    if (p.n <= 512) {
#define TT_SORT(K) sino_sort_kernel<K, 1, false, IDX7><<<sort_blocks<K, 1, false, IDX7>(cus, lines), kBlock, 0, s>>>(p)
        if (p.n <= 64)
            TT_SORT(1);
        else if (p.n <= 128)
            TT_SORT(2);
        else if (p.n <= 256)
            TT_SORT(4);
        else
            TT_SORT(8);
#undef TT_SORT
        return hipGetLastError();
    }
    // sorted parts up to 512 keys in the first pass, up to 1024 in the
    // second, the rest in the third; each pass queues what it cannot hold
    if (!queue_a || !queue_b)
        return hipErrorInvalidValue;
    p.defer_out = queue_a;
    p.defer_out_count = counts;
    sino_sort_kernel<8, 1, true, IDX7><<<sort_blocks<8, 1, true, IDX7>(cus, lines), kBlock, 0, s>>>(p);
    p.defer_in = queue_a;
    p.defer_in_count = counts;
    p.work = counts + 3;
    p.chunk = 2;
    if (p.n <= 1024) {
        sino_sort_kernel<16, 16, false, IDX7><<<sort_blocks<16, 16, false, IDX7>(cus), kBlock, 0, s>>>(p);
        return hipGetLastError();
    }
    p.defer_out = queue_b;
    p.defer_out_count = counts + 1;
    sino_sort_kernel<16, 16, true, IDX7><<<sort_blocks<16, 16, true, IDX7>(cus), kBlock, 0, s>>>(p);
    p.defer_in = queue_b;
    p.defer_in_count = counts + 1;
    p.work = counts + 4;
    p.chunk = 1;
    sino_sort_kernel<32, 32, false, IDX7><<<sort_blocks<32, 32, false, IDX7>(cus), kBlock, 0, s>>>(p);
    return hipGetLastError();
}

hipError_t launch_sino_sort(const SortTParams &p, int32_t *queue_a, int32_t *queue_b,
                            unsigned int *counts, hipStream_t s)
{
    return p.t7_src ? sino_sort_passes<true>(p, queue_a, queue_b, counts, s)
                    : sino_sort_passes<false>(p, queue_a, queue_b, counts, s);
}

}  // namespace ttk

namespace ttk {

hipError_t launch_records(const RecordParams &p, hipStream_t s)
{
    const size_t lines = (size_t)p.A * p.n;
    int blocks = (int)((lines + kBlock - 1) / kBlock);
    if (blocks > 8192)
        blocks = 8192;
    records_kernel<<<blocks, kBlock, 0, s>>>(p);
    return hipGetLastError();
}

size_t gather_lds_bytes(int tile, int waves, int tabn, bool do345, bool do12, bool do67)
{
    const size_t tab = do345 ? (size_t)kGatherTabWords * tabn : 0;
    return sizeof(float) * (tab + (size_t)waves * gather_wave_words(tile, do12, do67));
}

hipError_t launch_gather(const GatherParams &p, hipStream_t s)
{
    if (p.tile != kGatherTile || p.waves < 1 || p.waves > 16 || p.groups < 1 ||
        (p.groups > 1 && !p.part))
        return hipErrorInvalidValue;
    const int items = gather_tiles(p.n, p.tile) * p.groups;
    const int blocks = (items + p.waves - 1) / p.waves;
    const size_t shm = gather_lds_bytes(p.tile, p.waves, p.n, p.do345, p.do12,
                                        p.rec67 != nullptr);
    const dim3 block(kWave * p.waves);
    if (p.do345) {
        if (p.do12)
            gather_kernel<true, true><<<blocks, block, shm, s>>>(p);
        else
            gather_kernel<true, false><<<blocks, block, shm, s>>>(p);
    } else {
        if (p.do12)
            gather_kernel<false, true><<<blocks, block, shm, s>>>(p);
        else
            gather_kernel<false, false><<<blocks, block, shm, s>>>(p);
    }
    if (p.groups > 1) {
        const size_t npix = (size_t)p.n * p.n;
        size_t gb = (npix + kBlock - 1) / kBlock;
        gb = gb > 4096 ? 4096 : gb;
        gather_reduce_kernel<<<(int)gb, kBlock, 0, s>>>(p.part, p.groups, npix, p.dimg);
    }
    return hipGetLastError();
}

// sort: some P2 source row is found in the kernel (columns above kP2Max).
static size_t vjp_shm(int nmax, bool sort)
{
    int m2 = 1;
    while (m2 < nmax)
        m2 <<= 1;
    const size_t n4 = ((size_t)nmax + 3) & ~(size_t)3;
    return sort ? sizeof(uint64_t) * m2 + sizeof(float) * 3 * n4 : sizeof(float) * 2 * n4;
}

hipError_t launch_circus_vjp(const CircusVjpParams &p, hipStream_t s)
{
    circus_vjp_kernel<<<p.ncols * p.nsino, kBlock, vjp_shm(p.n, !p.p2src), s>>>(p);
    return hipGetLastError();
}

hipError_t launch_circus_vjp_batched(const BatchAdjointParams &p, hipStream_t s)
{
    // (the batch's P2 source rows come from the wave kernel up to kP2Max rows)
    circus_vjp_batched_kernel<<<p.cols, kBlock, vjp_shm(p.nmax, p.nmax > kP2Max), s>>>(p);
    return hipGetLastError();
}

hipError_t launch_records_batched(const BatchAdjointParams &p, hipStream_t s)
{
    int blocks = (p.lines + kBlock - 1) / kBlock;
    if (blocks > 8192)
        blocks = 8192;
    records_batched_kernel<<<blocks, kBlock, 0, s>>>(p);
    return hipGetLastError();
}

hipError_t launch_gather_batched(const BatchAdjointParams &p, int tile, int waves,
                                 hipStream_t s)
{
    if ((tile != 32 && tile != 16) || waves < 1 || waves > 16)
        return hipErrorInvalidValue;
    const bool do12 = p.slot.s[1] >= 0 || p.slot.s[2] >= 0;
    const size_t shm = gather_lds_bytes(tile, waves, p.tabn, p.do345, do12, false);
    const int blocks = (p.tiles + waves - 1) / waves;
    const dim3 block(kWave * waves);
#define TT_LAUNCH(T)                                                                   \
    do {                                                                               \
        if (p.do345 && do12)                                                           \
            gather_batched_kernel<T, true, true><<<blocks, block, shm, s>>>(p);        \
        else if (p.do345)                                                              \
            gather_batched_kernel<T, true, false><<<blocks, block, shm, s>>>(p);       \
        else if (do12)                                                                 \
            gather_batched_kernel<T, false, true><<<blocks, block, shm, s>>>(p);       \
        else                                                                           \
            gather_batched_kernel<T, false, false><<<blocks, block, shm, s>>>(p);      \
    } while (0)
    if (tile == 32)
        TT_LAUNCH(32);
    else
        TT_LAUNCH(16);
#undef TT_LAUNCH
    return hipGetLastError();
}

}  // namespace ttk

namespace ttk {

static int grid_for(size_t total)
{
    size_t b = (total + kBlock - 1) / kBlock;
    return (int)(b > 4096 ? 4096 : (b < 1 ? 1 : b));
}

hipError_t launch_short_sqrt_check(bool root, uint32_t lo, uint64_t count,
                                   unsigned long long *mism, unsigned int *first, hipStream_t s)
{
    if (root)
        short_sqrt_check_kernel<true><<<8192, kBlock, 0, s>>>(lo, count, mism, first);
    else
        short_sqrt_check_kernel<false><<<8192, kBlock, 0, s>>>(lo, count, mism, first);
    return hipGetLastError();
}

hipError_t launch_resize(const float *in, int in_rows, int in_cols, float *out,
                         int rows, int cols, hipStream_t s)
{
    resize_kernel<<<grid_for((size_t)rows * cols), kBlock, 0, s>>>(in, in_rows, in_cols,
                                                                   out, rows, cols);
    return hipGetLastError();
}

hipError_t launch_zscore(const float *in, int n, int count, float *out, hipStream_t s)
{
    zscore_kernel<<<count, kBlock, 0, s>>>(in, n, out);
    return hipGetLastError();
}

hipError_t launch_column_medians(const float *in, int n, int cols, int32_t *med,
                                 hipStream_t s)
{
    if (n <= kP2Max) {
        const int wpb = kBlock / kWave;
        column_median_wave_kernel<<<(cols + wpb - 1) / wpb, kBlock, 0, s>>>(in, n, cols, med);
        return hipGetLastError();
    }
    const size_t shm = sizeof(float) * (((size_t)n + 3) & ~(size_t)3);
    column_median_kernel<<<cols, kBlock, shm, s>>>(in, n, med);
    return hipGetLastError();
}

hipError_t launch_scale_eigvec(const double *v, const double *lambda, int k, int count,
                               double *out, hipStream_t s)
{
    scale_eigvec_kernel<<<grid_for((size_t)k * k * count), kBlock, 0, s>>>(v, lambda, k,
                                                                          count, out);
    return hipGetLastError();
}

hipError_t launch_newton_schulz_factor(double *x, int k, int count, hipStream_t s)
{
    newton_schulz_factor_kernel<<<grid_for((size_t)k * k * count), kBlock, 0, s>>>(x, k,
                                                                                  count);
    return hipGetLastError();
}

hipError_t launch_nos_reduce(const double *part, int chunks, int k, int count, double *S,
                             hipStream_t s)
{
    const size_t kk = (size_t)k * k;
    nos_reduce_kernel<<<grid_for(kk * count), kBlock, 0, s>>>(part, chunks, kk, count, S);
    return hipGetLastError();
}

hipError_t launch_nos_scales(const double *G, int k, int count, double *part, double *scale,
                             double *r, hipStream_t s)
{
    nos_slice_kernel<0><<<dim3(kNosSlices, count), kBlock, 0, s>>>(G, k, part);
    nos_scales_kernel<<<(count + kWave - 1) / kWave, kWave, 0, s>>>(part, kNosSlices, count,
                                                                    scale, r);
    return hipGetLastError();
}

hipError_t launch_nos_deviation(const double *S, int k, int count, double *part,
                                hipStream_t s)
{
    nos_slice_kernel<1><<<dim3(kNosSlices, count), kBlock, 0, s>>>(S, k, part);
    return hipGetLastError();
}

hipError_t launch_nos_poly(const double *S, const double *S2, int k, int count,
                           const PolarStep &c, const double *scale, const double *r, double *T,
                           double *Q, hipStream_t s)
{
    nos_poly_kernel<<<grid_for((size_t)k * k * count), kBlock, 0, s>>>(S, S2, k, count, c,
                                                                       scale, r, T, Q);
    return hipGetLastError();
}


hipError_t launch_align_batched(const float *in, int n, int cols, const int32_t *med,
                                int count, int rows_out, size_t mstride, double *out,
                                hipStream_t s)
{
    const int bx = (grid_for((size_t)rows_out * cols) + count - 1) / count;
    align_batched_kernel<<<dim3(bx, count), kBlock, 0, s>>>(in, n, cols, med, rows_out,
                                                             mstride, out);
    return hipGetLastError();
}

hipError_t launch_to_float_batched(const double *in, int ld, size_t mstride, int cols,
                                   const int32_t *med, int n, int sc, int count, int rows_max,
                                   float *out, size_t ostride, hipStream_t s)
{
    const int bx = (grid_for((size_t)rows_max * cols) + count - 1) / count;
    to_float_batched_kernel<<<dim3(bx, count), kBlock, 0, s>>>(in, ld, mstride, cols, med, n,
                                                                sc, out, ostride);
    return hipGetLastError();
}


}  // namespace ttk
