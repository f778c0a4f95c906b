// dsx_lines.hip -- zero-width line rasterisation (glyphs/line.py, line_width == 0).
//
// General layouts: one work item per segment.  Each item clips its segment to the view (Liang-Barsky,
// line.py:734-800), snaps both ends to pixels (map_onto_pixel_snap, 688-720) and walks
// the integer Bresenham path (986-1031), appending every pixel to the accumulator
// planes.  The arithmetic follows the reference's numba typing: coordinates promote to
// float64 except the segment delta x1 - x0, which a float32 column computes in float32.
#include "dsx_common.h"

namespace dsx {

struct LineArgs {
    int64_t nlines, nverts;
    const void *x, *y, *val;
    const double *mean;  // squared-deviation mode (var / std second pass)
    Cat cat;
    int64_t xls, xvs, yls, yvs;
    int32_t axis, plot_start;
    int32_t W, H, xlog, ylog;
    double sx, tx, sy, ty, xmin, xmax, ymin, ymax;
    int64_t xxmax, yymax;
};

// _clipt, line.py:783-800
__device__ __forceinline__ bool clipt(double p, double q, double &t0, double &t1) {
    if (p < 0 && q < 0) {
        const double r = q / p;
        if (r > t1) return false;
        if (r > t0) t0 = r;
    } else if (p > 0 && q < p) {
        const double r = q / p;
        if (r < t0) return false;
        if (r < t1) t1 = r;
    } else if (q < 0) {
        return false;
    }
    return true;
}

template <typename TV, bool HAS_VAL, bool SQDEV = false>
struct Sink {
    const Planes *p;
    const double *mean;
    int64_t W, H, ncat, c;
    TV v;
    __device__ __forceinline__ void operator()(int64_t x, int64_t y) const {
        if (x < 0) x += W;  // numba's negative-index wraparound
        if (y < 0) y += H;
        if ((uint64_t)x >= (uint64_t)W || (uint64_t)y >= (uint64_t)H) return;
        const int64_t cell = (y * W + x) * ncat + c;
        if constexpr (SQDEV) {
            if (v != v) return;
            const double d = (double)v - mean[cell];
            unsafeAtomicAdd(p->sum + cell, d * d);
        } else {
            append<TV, HAS_VAL>(*p, cell, v);
        }
    }
    template <typename I>
    __device__ __forceinline__ void walk(bool start, I x0, I x1, I y0, I y1, bool clipped) const;
};

// _bresenham, line.py:986-1031, in integer type I (the ends passed in are within one
// pixel of the canvas, so 32 bits hold every intermediate of the walk)
template <typename I, typename S>
__device__ __forceinline__ void bresenham(const S &put, bool segment_start, I x0, I x1, I y0,
                                          I y1, bool clipped) {
    I dx = x1 - x0;
    const I ix = (dx > 0) - (dx < 0);
    dx = (dx < 0 ? -dx : dx) * 2;
    I dy = y1 - y0;
    const I iy = (dy > 0) - (dy < 0);
    dy = (dy < 0 ? -dy : dy) * 2;
    if (!clipped && !(dx | dy)) {
        put(x0, y0);
        return;
    }
    if (segment_start) put(x0, y0);
    if (dx >= dy) {
        I err = 2 * dy - dx;
        while (x0 != x1) {
            if (err >= 0 && (err || ix > 0)) {
                err -= 2 * dx;
                y0 += iy;
            }
            err += 2 * dy;
            x0 += ix;
            put(x0, y0);
        }
    } else {
        I err = 2 * dx - dy;
        while (y0 != y1) {
            if (err >= 0 && (err || iy > 0)) {
                err -= 2 * dy;
                x0 += ix;
            }
            err += 2 * dx;
            y0 += iy;
            put(x0, y0);
        }
    }
}

template <typename TV, bool HAS_VAL, bool SQDEV>
template <typename I>
__device__ __forceinline__ void Sink<TV, HAS_VAL, SQDEV>::walk(bool start, I x0, I x1, I y0,
                                                              I y1, bool clipped) const {
    bresenham<I>(*this, start, x0, x1, y0, y1, clipped);
}

__device__ __forceinline__ int64_t snap1(double v, double s, double t, int64_t vmax,
                                         int32_t log) {
    const int64_t vv = (int64_t)__dadd_rn(__dmul_rn(axis_map(v, log), s), t);
    return vv == vmax ? vv - 1 : vv;
}

// For a segment with both ends in [lo, hi], starting at v0 with the delta d its column's
// precision gives: whether _clipt leaves it whole.  Its q are then >= 0, so only the
// `p > 0 and q < p` branch could act, for (p, q) = (-d, v0 - lo) and (d, hi - v0).  (The
// exact q is never less than the exact delta, but a float32 delta that rounds away from
// zero can exceed it when a vertex lies on a bound.)
__device__ __forceinline__ bool unclipped(double v0, double d, double lo, double hi) {
    return __dsub_rn(v0, lo) >= -d && __dsub_rn(hi, v0) >= d;
}

// The pixels a segment is drawn between, what is left of it in the view.
struct Ends {
    int32_t x0, y0, x1, y1;
    bool start, clipped;
};

// draw_segment, line.py:1045-1095, up to its _bresenham call, for coordinates of column
// types TX / TY: false where nothing is drawn.
template <typename TX, typename TY>
__device__ __forceinline__ bool segment_ends(const LineArgs &a, bool segment_start, TX x0c, TX x1c,
                                             TY y0c, TY y1c, Ends &e) {
    double x0 = (double)x0c, x1 = (double)x1c, y0 = (double)y0c, y1 = (double)y1c;
    bool skip = (x0 != x0) || (y0 != y0) || (x1 != x1) || (y1 != y1);
    if (x0 < a.xmin && x1 < a.xmin) skip = true;
    else if (x0 > a.xmax && x1 > a.xmax) skip = true;
    else if (y0 < a.ymin && y1 < a.ymin) skip = true;
    else if (y0 > a.ymax && y1 > a.ymax) skip = true;
    double t0 = 0.0, t1 = 1.0;
    const double dx1 = (double)(TX)(x1c - x0c);  // column precision (numba typing)
    const double dy1 = (double)(TY)(y1c - y0c);
    // Both ends inside the view and no _clipt call able to shorten the segment: (t0, t1)
    // stays (0, 1) and the four calls, with their divisions, are skipped.
    const bool inside = a.xmin <= x0 && x0 <= a.xmax && a.xmin <= x1 && x1 <= a.xmax &&
                        a.ymin <= y0 && y0 <= a.ymax && a.ymin <= y1 && y1 <= a.ymax &&
                        unclipped(x0, dx1, a.xmin, a.xmax) && unclipped(y0, dy1, a.ymin, a.ymax);
    if (!inside) {
        if (!clipt(-dx1, __dsub_rn(x0, a.xmin), t0, t1)) skip = true;
        if (!clipt(dx1, __dsub_rn(a.xmax, x0), t0, t1)) skip = true;
        if (!clipt(-dy1, __dsub_rn(y0, a.ymin), t0, t1)) skip = true;
        if (!clipt(dy1, __dsub_rn(a.ymax, y0), t0, t1)) skip = true;
    }
    if (skip) return false;
    e.start = segment_start;
    e.clipped = false;
    if (t1 < 1) {
        e.clipped = true;
        x1 = __dadd_rn(x0, __dmul_rn(t1, dx1));
        y1 = __dadd_rn(y0, __dmul_rn(t1, dy1));
    }
    if (t0 > 0) {
        e.clipped = true;
        e.start = true;
        x0 = __dadd_rn(x0, __dmul_rn(t0, dx1));
        y0 = __dadd_rn(y0, __dmul_rn(t0, dy1));
    }
    const int64_t px0 = snap1(x0, a.sx, a.tx, a.xxmax, a.xlog);
    const int64_t py0 = snap1(y0, a.sy, a.ty, a.yymax, a.ylog);
    const int64_t px1 = snap1(x1, a.sx, a.tx, a.xxmax, a.xlog);
    const int64_t py1 = snap1(y1, a.sy, a.ty, a.yymax, a.ylog);
    e.x0 = (int32_t)px0; e.y0 = (int32_t)py0; e.x1 = (int32_t)px1; e.y1 = (int32_t)py1;
    // Clipped ends project into [0, W] x [0, H] (one pixel of rounding slack either
    // side); anything else comes from a degenerate view (infinite or NaN scale) and
    // would make the walk unbounded, so such a segment is not drawn.
    return !(px0 < -1 || px0 > a.W + 1 || px1 < -1 || px1 > a.W + 1 || py0 < -1 ||
             py0 > a.H + 1 || py1 < -1 || py1 > a.H + 1);
}

template <typename TX, typename TY, typename I, typename S>
__device__ __forceinline__ void draw_segment(const LineArgs &a, const S &put, bool segment_start,
                                             TX x0c, TX x1c, TY y0c, TY y1c) {
    Ends e;
    if (segment_ends<TX, TY>(a, segment_start, x0c, x1c, y0c, y1c, e))
        put.template walk<I>(e.start, (I)e.x0, (I)e.x1, (I)e.y0, (I)e.y1, e.clipped);
}

template <typename TX, typename TY, typename TV, bool HAS_VAL, bool SQDEV>
__global__ __launch_bounds__(256) void lines_kernel(LineArgs a, Planes p) {
    const int64_t nseg = a.nverts - 1;
    const int64_t total = a.nlines * nseg;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const TX *X = reinterpret_cast<const TX *>(a.x);
    const TY *Y = reinterpret_cast<const TY *>(a.y);
    for (int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; s < total; s += stride) {
        const int64_t l = s / nseg, k = s - l * nseg;
        if (k == 0 && a.axis == 0 && a.plot_start == DSX_PLOT_CONTEXT) continue;  // context vertex
        const TX x0 = X[l * a.xls + k * a.xvs], x1 = X[l * a.xls + (k + 1) * a.xvs];
        const TY y0 = Y[l * a.yls + k * a.yvs], y1 = Y[l * a.yls + (k + 1) * a.yvs];
        bool start;
        if (k == 0) {
            start = a.axis == 0 ? (a.plot_start != 0) : true;
        } else {
            const TX xp = X[l * a.xls + (k - 1) * a.xvs];
            const TY yp = Y[l * a.yls + (k - 1) * a.yvs];
            start = (xp != xp) || (yp != yp);
        }
        const int64_t row = a.axis == 0 ? k : l;
        Sink<TV, HAS_VAL, SQDEV> put;
        put.p = &p; put.mean = a.mean; put.W = a.W; put.H = a.H; put.ncat = a.cat.ncat;
        put.v = TV(0);
        put.c = category(a.cat, row);
        if (put.c < 0) continue;
        if constexpr (HAS_VAL) put.v = reinterpret_cast<const TV *>(a.val)[row];
        draw_segment<TX, TY, int64_t>(a, put, start, x0, x1, y0, y1);
    }
}

// ---- count only: rasterising into LDS ------------------------------------------------
// The lines of a count (no value column, no categorizer) are drawn into a box of the
// canvas held in LDS, and the box's non-zero cells are added to the count plane with one
// global atomic each; a pixel outside the box goes straight to the global plane, so the
// result never depends on the box.  Random LDS u32 atomics run at 5.1 T/s here, global
// ones at 14-27 G/s.
constexpr int kBoxThreads = 1024;
constexpr int kBoxLds = 160 * 1024 - 1024;  // a run's box, less 1 KB for the kernel's own words

// The box's counters in the workgroup's dynamic LDS.
extern __shared__ uint32_t box_cells[];

using lds_u32 = __attribute__((address_space(3))) uint32_t;

// Count one pixel at an LDS address (32-bit, from Box::at): an address the walk steps
// itself, so that no base is added to it again for every pixel.
__device__ __forceinline__ void box_add(uint32_t addr) {
    __hip_atomic_fetch_add((lds_u32 *)(uintptr_t)addr, 1u, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Columns [c0, c0 + cols) and rows [r0, r0 + rows) of the canvas; odd row pitch, so that a
// column's cells spread over the LDS banks.
struct Box {
    int32_t c0, r0, cols, rows, pitch;
    __device__ __forceinline__ bool has(int32_t x, int32_t y) const {
        return (uint32_t)(x - c0) < (uint32_t)cols && (uint32_t)(y - r0) < (uint32_t)rows;
    }
    __device__ __forceinline__ uint32_t at(int32_t x, int32_t y) const {
        return (uint32_t)(uintptr_t)(lds_u32 *)box_cells + (uint32_t)((y - r0) * pitch + (x - c0)) * 4u;
    }
};

// _bresenham for a segment whose ends (so all its pixels) lie in the box; first: whether
// its first pixel is drawn.  With n steps along the major axis and m <= n along the minor
// one, the reference's error term has moved the minor axis floor((2 m i + n - b) / 2 n)
// times after i steps, b = 1 where the major axis runs backwards (its tie rule), else 0.
// Short segments hold that quotient, moved up by 1 / 4n -- half of its distance to the next
// value above --, in fixed point with 20 fractional bits: n steps of a slope that is off by
// less than 1.5 * 2^-20 stay within 1 / 4n for n < kDdaMax, so the floor is exact.  A step
// is then an add, a shift, a multiply-add and an add, with no compare or select.  Long ones
// keep the error term (its half, less b, so that the reference's
// `err >= 0 && (err || i > 0)` is err >= 0), and so do the short ones of a wave that has a
// long one: their loops would run one after the other (100k x 256 samples of white noise,
// where nearly every wave has both and a clipped one, into 2048 x 1024: 19.9 ms with a loop
// for each kind, 5.0 with one).
// common: a number of steps that every active lane takes (uniform), so that those run
// without a lane mask.
constexpr int32_t kDdaMax = 256;

__device__ __forceinline__ void box_walk(uint32_t at, int32_t dx, int32_t dy, uint32_t pitch4,
                                         bool first, int32_t common) {
    const int32_t ax = dx < 0 ? -dx : dx, ay = dy < 0 ? -dy : dy;
    const bool xm = ax >= ay;
    const int32_t n = xm ? ax : ay, m = xm ? ay : ax;
    if (first) box_add(at);
    const int32_t ox = dx < 0 ? -4 : 4, oy = dy < 0 ? -(int32_t)pitch4 : (int32_t)pitch4;
    const int32_t o1 = xm ? ox : oy, o2 = xm ? oy : ox;  // along the major axis; the minor
    const bool fwd = (xm ? dx : dy) > 0;
    if (!__any(n >= kDdaMax)) {
        const float rn = __builtin_amdgcn_rcpf((float)n);  // (n = 0: nothing is read of it)
        const uint32_t slope = (uint32_t)((float)m * rn * 1048576.0f);
        const int32_t quarter = (int32_t)(rn * 262144.0f);
        uint32_t acc = 524288u + (uint32_t)(fwd ? quarter : -quarter);
        int32_t i = 0;
        auto step = [&]() {
            acc += slope;
            at += (uint32_t)o1;
            box_add((uint32_t)(__mul24((int32_t)(acc >> 20), o2) + (int32_t)at));
        };
#pragma unroll 4
        for (; i < common; ++i) step();
        uint32_t left = (uint32_t)(n - i);
        while (!__builtin_sub_overflow(left, 1u, &left)) step();
        return;
    }
    const int32_t e1 = 2 * m, e2 = 2 * (m - n);
    int32_t err = e1 - n - (fwd ? 0 : 1);
    for (int32_t i = n; i > 0; --i) {
        const bool both = err >= 0;
        at += (uint32_t)(both ? o1 + o2 : o1);
        err += both ? e2 : e1;
        box_add(at);
    }
}

struct BoxSink {
    uint32_t *count;
    int32_t W, H;
    Box box;
    __device__ __forceinline__ void operator()(int32_t x, int32_t y) const {
        if (x < 0) x += W;  // numba's negative-index wraparound
        if (y < 0) y += H;
        if ((uint32_t)x >= (uint32_t)W || (uint32_t)y >= (uint32_t)H) return;
        if (box.has(x, y)) box_add(box.at(x, y));
        else atomicAdd(count + (int64_t)y * W + x, 1u);
    }
    template <typename I>
    __device__ __forceinline__ void walk(bool start, I x0, I x1, I y0, I y1, bool clipped) const {
        bresenham<I>(*this, start, x0, x1, y0, y1, clipped);
    }
};

// Pixel of a coordinate (snap1 in 32 bits).  A value far off the canvas (a degenerate view)
// saturates, so it is in no box; NaN becomes pixel 0, as in snap1 -- the callers draw nothing
// of a segment with a missing vertex, so only a view's NaN scale gets there.
// vmax: snap_max of the axis's last pixel.
template <bool LOG>
__device__ __forceinline__ int32_t snap_in(double v, double s, double t, int32_t vmax, int32_t log) {
    const double d = __dadd_rn(__dmul_rn(LOG ? axis_map(v, log) : v, s), t);
    int32_t p;
    asm("v_cvt_i32_f64 %0, %1" : "=v"(p) : "v"(d));  // truncates and saturates
    return p == vmax ? p - 1 : p;
}
__device__ __forceinline__ int32_t snap_max(int64_t vmax) {  // (no pixel is the lowest integer)
    return vmax == (int64_t)(int32_t)vmax ? (int32_t)vmax : INT32_MIN;
}

__device__ __forceinline__ void box_flush(const Box &b, uint32_t *count, int32_t W, int32_t H) {
    for (int i = threadIdx.x; i < b.rows * b.pitch; i += kBoxThreads) {
        const uint32_t v = box_cells[i];
        if (!v) continue;
        const int32_t r = i / b.pitch, c = i - r * b.pitch;
        const int32_t x = b.c0 + c, y = b.r0 + r;
        if (c < b.cols && x < W && y < H) atomicAdd(count + (int64_t)y * W + x, v);
    }
}

// ---- x-constant series, count only: LDS strips ---------------------------------------
// Lines of an axis-1 frame whose x is shared (x_line_stride == 0, LinesAxis1XConstant,
// line.py:334-380) put segment j of every line between the same two x values, so the
// pixels of segments [j0, j0 + k) of all lines fall in one narrow band of columns.
// Workgroup (s, b) rasterises segments [s*k, s*k + k) of lines [b*L, b*L + L) into an
// LDS copy of that band (all H rows).
//
// Bound by instruction issue (2.3 G pixel updates of 1M x 256 series: 0.45 ms of LDS
// atomics, 1.03 GB of columns: 0.2 ms).  So what all lines share -- the snapped x of each
// vertex, whether it is in the view -- is worked out once per workgroup, each vertex's y is
// projected once (not once per segment it ends), in 32 bits, and only segments that
// clipping could shorten take draw_segment: telling those by an inexact float32 delta sent
// a lane of nearly every wave there (values near zero), 2.21 against 1.54 ms.  The
// fixed-point walk, its common steps without a lane mask: 1.54 -> 1.13 ms.  Before all of
// it 2.89 ms (2048 x 1024).
constexpr int kStripMaxK = 8;        // segments per strip
// The band alone takes the LDS; what the lanes share is in scalar registers.  (A few words of
// it in LDS cost the band two columns at some heights, whose pixels then take global atomics:
// 0.7M x 32 series into 1812 x 803, segments wider than the band, 9.9 ms against 8.2.)
constexpr int kStripLds = 160 * 1024;

enum : int32_t {
    SEG_FAST = 1,   // both ends in the view and in the band's columns, unclipped in x
    SEG_SKIP = 2,   // nothing of it can be drawn (an end missing, or both outside)
    SEG_START = 4   // the x before it is missing
};

// Line l's samples j0 .. j0 + K (the last one repeated past nv), and whether sample j0 - 1
// is missing.
template <typename TY, int K>
struct StripRow {
    TY y[K + 1];
    TY prev;
    __device__ __forceinline__ void load(const LineArgs &a, int64_t j0, int nv, int64_t l) {
        const TY *Y = reinterpret_cast<const TY *>(a.y) + l * a.yls;
#pragma unroll
        for (int q = 0; q <= K; ++q) y[q] = Y[(j0 + (q < nv ? q : nv - 1)) * a.yvs];
        prev = Y[(j0 > 0 ? j0 - 1 : 0) * a.yvs];
    }
};

template <typename TX, typename TY, int K, bool LOG>
__global__ __launch_bounds__(kBoxThreads) void lines_xconst_strip_kernel(LineArgs a,
                                                                         uint32_t *count,
                                                                         int32_t k,
                                                                         int32_t pitch,
                                                                         int64_t lpb) {
    const TX *X = reinterpret_cast<const TX *>(a.x);
    const int64_t nseg = a.nverts - 1;
    const int64_t j0 = (int64_t)blockIdx.x * k;
    const int64_t j1 = j0 + k < nseg ? j0 + k : nseg;  // segments [j0, j1)
    const int ns = (int)(j1 - j0), nv = ns + 1;
    const int64_t l0 = (int64_t)blockIdx.y * lpb;
    const int64_t l1 = l0 + lpb < a.nlines ? l0 + lpb : a.nlines;
    const int tid = threadIdx.x;
    // first column of the band: the leftmost snapped vertex of the strip, with x clamped
    // to the view as clipping would (a clipped end lies between its vertices)
    int64_t lo = a.W;
    for (int64_t j = j0; j <= j1; ++j) {
        double x = (double)X[j * a.xvs];
        if (x != x) continue;
        x = x < a.xmin ? a.xmin : (x > a.xmax ? a.xmax : x);
        const int64_t c = snap1(x, a.sx, a.tx, a.xxmax, a.xlog);
        lo = c < lo ? c : lo;
    }
    BoxSink put;
    put.count = count; put.W = a.W; put.H = a.H;
    put.box.c0 = __builtin_amdgcn_readfirstlane((int32_t)(lo < 0 ? 0 : (lo > a.W ? a.W : lo)));
    put.box.r0 = 0;
    put.box.cols = pitch; put.box.rows = a.H; put.box.pitch = pitch;
    for (int i = tid; i < a.H * pitch; i += kBoxThreads) box_cells[i] = 0u;
    const int32_t xxmax = snap_max(a.xxmax), yymax = snap_max(a.yymax);
    // Lane q of every wave works out vertex q's column in the band and segment q's flags;
    // then they are uniform values (16 bits a column: those of a segment outside the band are
    // not read).
    uint64_t cols_a, cols_b;  // vertices 0-3, 4-7
    uint32_t col_c, flags_all = 0u;
    {
        const int q = tid & 63, q0 = q < ns ? q : ns, q1 = q + 1 < ns ? q + 1 : ns;
        const TX x0c = X[(j0 + q0) * a.xvs], x1c = X[(j0 + q1) * a.xvs];
        const TX xp = X[(j0 + q0 > 0 ? j0 + q0 - 1 : 0) * a.xvs];
        const double x0 = (double)x0c, x1 = (double)x1c;
        const int32_t px0 = snap_in<LOG>(x0, a.sx, a.tx, xxmax, a.xlog);
        const int32_t px1 = snap_in<LOG>(x1, a.sx, a.tx, xxmax, a.xlog);
        const auto in_band = [&](int32_t c) {
            return c >= 0 && c < a.W && (uint32_t)(c - put.box.c0) < (uint32_t)pitch;
        };
        int32_t f = 0;
        if (a.xmin <= x0 && x0 <= a.xmax && a.xmin <= x1 && x1 <= a.xmax && in_band(px0) &&
            in_band(px1) && unclipped(x0, (double)(TX)(x1c - x0c), a.xmin, a.xmax))
            f |= SEG_FAST;
        if (x0 != x0 || x1 != x1 || (x0 < a.xmin && x1 < a.xmin) || (x0 > a.xmax && x1 > a.xmax))
            f |= SEG_SKIP;
        if (j0 + q0 > 0 && xp != xp) f |= SEG_START;
        const int32_t c = (px0 - put.box.c0) & 0xFFFF;
        uint32_t cl[9];
#pragma unroll
        for (int i = 0; i <= kStripMaxK; ++i) cl[i] = (uint32_t)__builtin_amdgcn_readlane(c, i);
#pragma unroll
        for (int i = 0; i < kStripMaxK; ++i)
            flags_all |= (uint32_t)__builtin_amdgcn_readlane(f, i) << (4 * i);
        cols_a = (uint64_t)(cl[0] | cl[1] << 16) | (uint64_t)(cl[2] | cl[3] << 16) << 32;
        cols_b = (uint64_t)(cl[4] | cl[5] << 16) | (uint64_t)(cl[6] | cl[7] << 16) << 32;
        col_c = cl[8];
    }
    __syncthreads();
    const uint32_t pitch4 = (uint32_t)pitch * 4u;
    // the next line's samples are loaded while this line is drawn
    StripRow<TY, K> row, far;
    const int64_t lt = l0 + tid;
    if (lt < l1) row.load(a, j0, nv, lt);
    for (int64_t l = lt; l < l1; l += kBoxThreads) {
        far.load(a, j0, nv, l + kBoxThreads < l1 ? l + kBoxThreads : l);
        // one vertex per step: its place in the view and its pixel row, once
        bool gap = j0 == 0 || row.prev != row.prev;  // the sample before is missing
        double y0 = (double)row.y[0];
        bool in0 = a.ymin <= y0 && y0 <= a.ymax;
        // (a log10 of nothing in the view is not worked out)
        int32_t py0 = !LOG || in0 ? snap_in<LOG>(y0, a.sy, a.ty, yymax, a.ylog) : -1;
        uint64_t ca = cols_a, cb = cols_b;
        uint32_t cc = col_c, fl = flags_all;
        // segments drawn from the front of a shifting register window (a rolled loop with
        // constant register indices: one copy of the rasteriser, no indexed registers)
#pragma unroll 1
        for (int q = 0; q < ns; ++q) {
            const int32_t px0 = put.box.c0 + (int32_t)(ca & 0xFFFFu), flags = (int32_t)(fl & 15u);
            ca = ca >> 16 | cb << 48;
            cb = cb >> 16 | (uint64_t)cc << 48;
            cc = 0u;
            fl >>= 4;
            const int32_t px1 = put.box.c0 + (int32_t)(ca & 0xFFFFu);
            const TY y0c = row.y[0], y1c = row.y[1];
            const double y1 = (double)y1c;
            const bool in1 = a.ymin <= y1 && y1 <= a.ymax;
            const int32_t py1 = !LOG || in1 ? snap_in<LOG>(y1, a.sy, a.ty, yymax, a.ylog) : -1;
            const bool start = gap || (flags & SEG_START) != 0;
            const bool fast = in0 & in1 & ((uint32_t)py0 < (uint32_t)a.H) &
                              ((uint32_t)py1 < (uint32_t)a.H) &
                              unclipped(y0, (double)(TY)(y1c - y0c), a.ymin, a.ymax) &
                              ((flags & SEG_FAST) != 0);
            const bool first = start || (px0 == px1 && py0 == py1);
            // (a copy of its own, so that the x side of the walk stays in scalar registers: 1M x
            // 256 series 1.20 ms with the ends in the vector registers of the other, 1.12 so)
            if (__all(fast)) {
                const int32_t dx = px1 - px0;
                box_walk(put.box.at(px0, py0), dx, py1 - py0, pitch4, first, dx < 0 ? -dx : dx);
            } else {
                // each lane's own pixels or what clipping leaves of them, then one walk for
                // the lanes of either kind
                Ends e{px0, py0, px1, py1, first, false};
                bool draw = fast;
                if (!fast && !(flags & SEG_SKIP)) {
                    // (both ends beyond one bound, or one missing: nothing is drawn)
                    const bool none = y0 != y0 || y1 != y1 || (y0 < a.ymin && y1 < a.ymin) ||
                                      (y0 > a.ymax && y1 > a.ymax);
                    if (!none && segment_ends<TX, TY>(a, start, X[(j0 + q) * a.xvs],
                                                      X[(j0 + q + 1) * a.xvs], y0c, y1c, e)) {
                        draw = put.box.has(e.x0, e.y0) && put.box.has(e.x1, e.y1) && e.x0 < a.W &&
                               e.x1 < a.W;
                        if (!draw) put.walk<int32_t>(e.start, e.x0, e.x1, e.y0, e.y1, e.clipped);
                        e.start = e.start || (!e.clipped && e.x0 == e.x1 && e.y0 == e.y1);
                    }
                }
                if (draw)
                    box_walk(put.box.at(e.x0, e.y0), e.x1 - e.x0, e.y1 - e.y0, pitch4, e.start, 0);
            }
            gap = y0 != y0;
            y0 = y1;
            in0 = in1;
            py0 = py1;
#pragma unroll
            for (int i = 0; i < K; ++i) row.y[i] = row.y[i + 1];
        }
        row = far;
    }
    __syncthreads();
    box_flush(put.box, count, a.W, a.H);
}

// ---- axis 0, count only: runs of one line through a moving LDS box ----------------------
// Consecutive vertices of a line are near each other (a time series, a track), so a run of
// its segments draws in a small box of the canvas.  Workgroup (l, g) takes `per`
// consecutive segments of line l, kRunSegs at a time: it projects every vertex, reduces
// the round's pixel bounds, and if they leave the current box adds the box to the count
// plane and places a new one around them, grown to the LDS capacity (so that the next
// rounds fit too).  Bounds larger than the capacity keep the box where it is (or, at
// first, are covered around their centre) and the pixels outside it take global atomics.
// 10M vertices of a noisy series into 900 x 525: 6.97 ms with a global atomic a pixel,
// 0.14 ms through the boxes (0.16 GB of vertices: 0.03 ms; the rest is the walk, whose
// lanes differ in length); the call around it, with its automatic ranges, 0.24 ms.
constexpr int kRunU = 4;                          // segments per thread and round
constexpr int kRunSegs = kBoxThreads * kRunU;

// A box of at most cap cells around pixel bounds [x0, x1] x [y0, y1] of the canvas: it
// holds them when their own box fits, and is grown in proportion to fill cap.
__device__ __forceinline__ Box place_box(int32_t x0, int32_t x1, int32_t y0, int32_t y1, int32_t W,
                                         int32_t H, int32_t cap) {
    const int32_t bw = x1 - x0 + 1, bh = y1 - y0 + 1;
    const float f = sqrtf((float)cap / ((float)bw * (float)bh));
    int32_t w = (int32_t)fminf((float)bw * f, (float)(W < cap ? W : (cap - 1)));
    w = w < 1 ? 1 : w;
    if (cap / (w | 1) < bh && (int64_t)(bw | 1) * bh <= cap) w = bw;
    int32_t h = cap / (w | 1);
    if (h > H) {  // full height: the rest of the capacity as width
        h = H;
        int32_t w2 = cap / H;
        w2 = (w2 & 1) || w2 == 0 ? w2 : w2 - 1;  // (an odd pitch)
        w2 = w2 > W ? W : w2;
        w = w2 > w ? w2 : w;
    }
    Box b;
    b.cols = w; b.rows = h; b.pitch = w | 1;
    b.c0 = x0 - (w - bw) / 2;
    b.r0 = y0 - (h - bh) / 2;
    b.c0 = b.c0 < 0 ? 0 : (b.c0 > W - w ? W - w : b.c0);
    b.r0 = b.r0 < 0 ? 0 : (b.r0 > H - h ? H - h : b.r0);
    return b;
}

template <typename TX, typename TY, bool LOG>
__global__ __launch_bounds__(kBoxThreads) void lines_run_kernel(LineArgs a, uint32_t *count,
                                                                int32_t cap, int64_t per,
                                                                int64_t groups) {
    // a round's pixel bounds: -x0, x1, -y0, y1 (maxima), after the box in dynamic LDS
    int32_t(*s_bb)[4] = reinterpret_cast<int32_t(*)[4]>(box_cells + cap);
    const int tid = threadIdx.x;
    const int64_t nseg = a.nverts - 1;
    const int64_t l = blockIdx.x / groups, g = blockIdx.x - l * groups;
    const int64_t s0 = g * per, s1 = s0 + per < nseg ? s0 + per : nseg;
    const TX *X = reinterpret_cast<const TX *>(a.x) + l * a.xls;
    const TY *Y = reinterpret_cast<const TY *>(a.y) + l * a.yls;
    constexpr int32_t kNone = -(1 << 30);
    if (tid < 12) s_bb[tid >> 2][tid & 3] = kNone;
    __syncthreads();
    BoxSink put;
    put.count = count; put.W = a.W; put.H = a.H;
    put.box = Box{0, 0, 0, 0, 1};
    const int32_t xxmax = snap_max(a.xxmax), yymax = snap_max(a.yymax);
    int r = 0;
    for (int64_t base = s0; base < s1; base += kRunSegs) {
        TX x0c[kRunU], x1c[kRunU], xpc[kRunU];
        TY y0c[kRunU], y1c[kRunU], ypc[kRunU];
#pragma unroll
        for (int u = 0; u < kRunU; ++u) {  // a segment past the run re-reads its last one
            int64_t k = base + u * kBoxThreads + tid;
            k = k < s1 ? k : s1 - 1;
            x0c[u] = X[k * a.xvs]; x1c[u] = X[(k + 1) * a.xvs];
            y0c[u] = Y[k * a.yvs]; y1c[u] = Y[(k + 1) * a.yvs];
            const int64_t kp = k > 0 ? k - 1 : 0;
            xpc[u] = X[kp * a.xvs]; ypc[u] = Y[kp * a.yvs];
        }
        int32_t px0[kRunU], px1[kRunU], py0[kRunU], py1[kRunU];
        uint32_t todo = 0u, whole = 0u;  // bit u: segment u draws; it needs no clipping
        int32_t bb[4] = {kNone, kNone, kNone, kNone};
#pragma unroll
        for (int u = 0; u < kRunU; ++u) {
            const int64_t k = base + u * kBoxThreads + tid;
            const double x0 = (double)x0c[u], x1 = (double)x1c[u];
            const double y0 = (double)y0c[u], y1 = (double)y1c[u];
            const bool none = x0 != x0 || x1 != x1 || y0 != y0 || y1 != y1 ||
                              (x0 < a.xmin && x1 < a.xmin) || (x0 > a.xmax && x1 > a.xmax) ||
                              (y0 < a.ymin && y1 < a.ymin) || (y0 > a.ymax && y1 > a.ymax) ||
                              (k == 0 && a.plot_start == DSX_PLOT_CONTEXT);
            if (k >= s1 || none) continue;
            // the ends moved into the view bound what clipping can leave of the segment
            const auto in_view = [](double v, double lo, double hi) { return v < lo ? lo : (v > hi ? hi : v); };
            const double cx0 = in_view(x0, a.xmin, a.xmax), cx1 = in_view(x1, a.xmin, a.xmax);
            const double cy0 = in_view(y0, a.ymin, a.ymax), cy1 = in_view(y1, a.ymin, a.ymax);
            px0[u] = snap_in<LOG>(cx0, a.sx, a.tx, xxmax, a.xlog);
            px1[u] = snap_in<LOG>(cx1, a.sx, a.tx, xxmax, a.xlog);
            py0[u] = snap_in<LOG>(cy0, a.sy, a.ty, yymax, a.ylog);
            py1[u] = snap_in<LOG>(cy1, a.sy, a.ty, yymax, a.ylog);
            todo |= 1u << u;
            if (a.xmin <= x0 && x0 <= a.xmax && a.xmin <= x1 && x1 <= a.xmax &&
                a.ymin <= y0 && y0 <= a.ymax && a.ymin <= y1 && y1 <= a.ymax &&
                unclipped(x0, (double)(TX)(x1c[u] - x0c[u]), a.xmin, a.xmax) &&
                unclipped(y0, (double)(TY)(y1c[u] - y0c[u]), a.ymin, a.ymax))
                whole |= 1u << u;
            const auto cl = [](int32_t p, int32_t n) { return p < 0 ? 0 : (p >= n ? n - 1 : p); };
            const int32_t xa = cl(px0[u], a.W), xb = cl(px1[u], a.W);
            const int32_t ya = cl(py0[u], a.H), yb = cl(py1[u], a.H);
            bb[0] = max(bb[0], max(-xa, -xb)); bb[1] = max(bb[1], max(xa, xb));
            bb[2] = max(bb[2], max(-ya, -yb)); bb[3] = max(bb[3], max(ya, yb));
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) bb[i] = max(bb[i], __shfl_xor(bb[i], off, 64));
            if ((tid & 63) == 0 && bb[i] != kNone) atomicMax(&s_bb[r][i], bb[i]);
        }
        __syncthreads();  // the round's bounds; the last round is drawn
        const int32_t bx0 = -s_bb[r][0], bx1 = s_bb[r][1], by0 = -s_bb[r][2], by1 = s_bb[r][3];
        const int r2 = r == 0 ? 2 : r - 1;  // read before this barrier, written after the next
        if (tid < 4) s_bb[r2][tid] = kNone;
        r = r == 2 ? 0 : r + 1;
        if (bx1 == kNone) continue;  // uniform: nothing to draw
        const bool holds = put.box.has(bx0, by0) && put.box.has(bx1, by1);
        const bool fits = (int64_t)((bx1 - bx0 + 1) | 1) * (by1 - by0 + 1) <= cap;
        if (!holds && (fits || put.box.rows == 0)) {  // uniform
            if (put.box.rows) {
                box_flush(put.box, count, a.W, a.H);
                __syncthreads();
            }
            // (the last round's box is no larger than its bounds: cleared and added whole, one of
            // the LDS's size costs some 5 us, for a track of 100k vertices a third of the kernel)
            const int32_t bw = bx1 - bx0 + 1, bh = by1 - by0 + 1;
            put.box = fits && base + kRunSegs >= s1 ? Box{bx0, by0, bw, bh, bw | 1}
                                                    : place_box(bx0, bx1, by0, by1, a.W, a.H, cap);
            for (int i = tid; i < put.box.rows * put.box.pitch; i += kBoxThreads) box_cells[i] = 0u;
            __syncthreads();
        }
        const uint32_t pitch4 = (uint32_t)put.box.pitch * 4u;
#pragma unroll
        for (int u = 0; u < kRunU; ++u) {
            if (!(todo >> u & 1u)) continue;
            const bool start = base + u * kBoxThreads + tid == 0
                                   ? a.plot_start != 0
                                   : (xpc[u] != xpc[u]) || (ypc[u] != ypc[u]);
            if ((whole >> u & 1u) && put.box.has(px0[u], py0[u]) && put.box.has(px1[u], py1[u]))
                box_walk(put.box.at(px0[u], py0[u]), px1[u] - px0[u], py1[u] - py0[u], pitch4,
                         start || (px0[u] == px1[u] && py0[u] == py1[u]), 0);
            else
                draw_segment<TX, TY, int32_t>(a, put, start, x0c[u], x1c[u], y0c[u], y1c[u]);
        }
    }
    __syncthreads();
    if (put.box.rows) box_flush(put.box, count, a.W, a.H);
}

static int cu_count() {
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) == hipSuccess) {
        int c = 0;
        if (hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && c > 0)
            cus = c;
    }
    return cus;
}

template <typename TX, typename TY>
static int launch_strips(const LineArgs &a, uint32_t *count, int64_t nstrips, int64_t nblocks,
                         int64_t k, int64_t pitch, int64_t lpb, hipStream_t s) {
    const size_t lds = (size_t)4 * a.H * pitch;
    // (two band sizes, so that few registers hold samples a strip does not have)
    auto kern = k <= 4 ? lines_xconst_strip_kernel<TX, TY, 4, false>
                       : lines_xconst_strip_kernel<TX, TY, kStripMaxK, false>;
    if (a.xlog || a.ylog) kern = lines_xconst_strip_kernel<TX, TY, kStripMaxK, true>;
    const hipError_t e = hipFuncSetAttribute((const void *)kern,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) { record_hip_error(e); return DSX_ERR_HIP; }
    hipLaunchKernelGGL(kern, dim3((unsigned)nstrips, (unsigned)nblocks), dim3(kBoxThreads), lds, s, a,
                       count, (int32_t)k, (int32_t)pitch, lpb);
    return launch_status();
}

template <typename TX, typename TY>
static int launch_runs(const LineArgs &a, uint32_t *count, hipStream_t s) {
    const int64_t nseg = a.nverts - 1;
    // at most one workgroup per CU (its box takes the CU's LDS), of at least 256 segments (20k
    // segments: 1024 each 61.9 us a call, 256 each 59.8).  Where the lines alone are more
    // than that, a last round of few workgroups leaves the chip idle: lines are then split
    // as long as that shortens the rounds' sum and a workgroup keeps half a round of segments
    // (300 lines of 12000 noisy vertices, 300 workgroups on 256 CUs: 15.9 ms, 6.3
    // split; one global atomic a pixel 13.6).
    const int64_t cus = cu_count();
    int64_t groups = cus / a.nlines;
    const int64_t most = (nseg + 255) / 256;
    groups = groups > most ? most : groups;
    if (groups < 1) {
        groups = 1;
        const auto rounds = [&](int64_t g) { return (a.nlines * g + cus - 1) / cus; };
        for (int64_t g = 2; g <= 8 && nseg >= g * (kRunSegs / 2); ++g)
            if (rounds(g) * groups < rounds(groups) * g) groups = g;
    }
    const int64_t per = (nseg + groups - 1) / groups;
    auto kern = a.xlog || a.ylog ? lines_run_kernel<TX, TY, true> : lines_run_kernel<TX, TY, false>;
    constexpr int lds = kBoxLds + 64;  // the box and a round's bounds
    const hipError_t e = hipFuncSetAttribute((const void *)kern,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) { record_hip_error(e); return DSX_ERR_HIP; }
    hipLaunchKernelGGL(kern, dim3((unsigned)(a.nlines * groups)), dim3(kBoxThreads), lds, s, a, count,
                       (int32_t)(kBoxLds / 4), per, groups);
    return launch_status();
}

template <typename TX, typename TY>
static void launch_lines(const LineArgs &a, const Planes &p, int32_t vdt, int grid, int block,
                         hipStream_t s) {
    if (!a.val) lines_kernel<TX, TY, float, false, false><<<grid, block, 0, s>>>(a, p);
    else if (a.mean && vdt == DSX_F32) lines_kernel<TX, TY, float, true, true><<<grid, block, 0, s>>>(a, p);
    else if (a.mean) lines_kernel<TX, TY, double, true, true><<<grid, block, 0, s>>>(a, p);
    else if (vdt == DSX_F32) lines_kernel<TX, TY, float, true, false><<<grid, block, 0, s>>>(a, p);
    else lines_kernel<TX, TY, double, true, false><<<grid, block, 0, s>>>(a, p);
}

}  // namespace dsx

using namespace dsx;

extern "C" int dsx_lines_agg(const dsx_lines_desc *d, const dsx_view *v, const dsx_planes *acc,
                             void *stream) {
    if (!d || !v || !acc) return DSX_ERR_NULL;
    if (d->nlines < 0 || d->nverts < 0 || v->width <= 0 || v->height <= 0) return DSX_ERR_SHAPE;
    if (d->axis != 0 && d->axis != 1) return DSX_ERR_SHAPE;
    if ((d->x_dtype != DSX_F32 && d->x_dtype != DSX_F64) ||
        (d->y_dtype != DSX_F32 && d->y_dtype != DSX_F64))
        return DSX_ERR_DTYPE;
    if (d->val && d->val_dtype != DSX_F32 && d->val_dtype != DSX_F64) return DSX_ERR_DTYPE;
    const int cst = check_cat(d->cat);
    if (cst) return cst;
    if (acc->mean) return DSX_ERR_ACCUM;  // lines accumulate: a mean is finalized afterwards
    const bool needs_val = acc->countv || acc->sum || acc->min || acc->max;
    if (needs_val && !d->val) return DSX_ERR_ACCUM;
    if (d->mean && (!d->val || !acc->sum || acc->count || acc->countv || acc->min || acc->max))
        return DSX_ERR_ACCUM;
    if (d->nlines == 0 || d->nverts < 2) return DSX_OK;
    if (!d->x || !d->y) return DSX_ERR_NULL;
    LineArgs a;
    a.nlines = d->nlines; a.nverts = d->nverts;
    a.x = d->x; a.y = d->y; a.val = d->val; a.cat = cat_of(d->cat); a.mean = d->mean;
    a.xls = d->x_line_stride; a.xvs = d->x_vert_stride;
    a.yls = d->y_line_stride; a.yvs = d->y_vert_stride;
    a.axis = d->axis; a.plot_start = d->plot_start;
    a.W = v->width; a.H = v->height; a.xlog = v->xlog; a.ylog = v->ylog;
    a.sx = v->sx; a.tx = v->tx; a.sy = v->sy; a.ty = v->ty;
    a.xmin = v->xmin; a.xmax = v->xmax; a.ymin = v->ymin; a.ymax = v->ymax;
    a.xxmax = v->xxmax; a.yymax = v->yymax;
    const Planes p = planes_of(acc);
    hipStream_t s = as_stream(stream);
    const bool x32 = d->x_dtype == DSX_F32, y32 = d->y_dtype == DSX_F32;
    // x-constant series with count / any only: LDS strips
    int64_t pitch = kStripLds / (4 * (int64_t)v->height);
    if (pitch % 2 == 0) --pitch;
    const bool counts = !d->val && d->cat.kind == DSX_CAT_NONE && acc->count && !needs_val;
    if (counts && d->axis == 1 && d->x_line_stride == 0 && pitch >= 5) {
        const int64_t nseg = d->nverts - 1;
        int64_t k = (pitch - 2) * nseg / v->width;  // segments whose band fits, for x spread evenly
        k = k < 1 ? 1 : (k > kStripMaxK ? kStripMaxK : k);
        const int64_t nstrips = (nseg + k - 1) / k;
        const int cus = cu_count();
        int64_t nblocks = (cus + nstrips - 1) / nstrips;
        if (nblocks > d->nlines) nblocks = d->nlines;
        if (nblocks < 1) nblocks = 1;
        if (nstrips <= 65535 && nblocks <= 65535) {
            const int64_t lpb = (d->nlines + nblocks - 1) / nblocks;
            return x32 ? (y32 ? launch_strips<float, float>(a, p.count, nstrips, nblocks, k, pitch, lpb, s)
                              : launch_strips<float, double>(a, p.count, nstrips, nblocks, k, pitch, lpb, s))
                       : (y32 ? launch_strips<double, float>(a, p.count, nstrips, nblocks, k, pitch, lpb, s)
                              : launch_strips<double, double>(a, p.count, nstrips, nblocks, k, pitch, lpb, s));
        }
    }
    // axis 0 with count / any only: runs of segments through an LDS box, from the size where the
    // middle of a time series is drawn sooner so than by a global atomic a pixel (kernels, 762 x
    // 426: 20k vertices 12.8 against 16.6 us, 30k 17.6 against 14.9, 100k 26.7 against 15.9; all
    // of the series 30k 13.0 against 9.2, 200k 58 against 10; 10M into 900 x 525 6.1 against
    // 0.24 ms a call).  A smooth track has few pixels a segment and stays with the atomics' time
    // longer (100k vertices 8.5 against 9.0 us, the middle of it 6.0 against 11.4), which the host
    // part of a call hides.  Lines shorter than a workgroup would each clear and add a box for
    // few segments.
    if (counts && d->axis == 0 && d->nverts > kBoxThreads && d->nlines <= 65535 &&
        d->nlines * (d->nverts - 1) >= 32768)
        return x32 ? (y32 ? launch_runs<float, float>(a, p.count, s) : launch_runs<float, double>(a, p.count, s))
                   : (y32 ? launch_runs<double, float>(a, p.count, s) : launch_runs<double, double>(a, p.count, s));
    const int block = 256;
    const int grid = grid_for(d->nlines * (d->nverts - 1), block);
    if (x32 && y32) launch_lines<float, float>(a, p, d->val_dtype, grid, block, s);
    else if (x32) launch_lines<float, double>(a, p, d->val_dtype, grid, block, s);
    else if (y32) launch_lines<double, float>(a, p, d->val_dtype, grid, block, s);
    else launch_lines<double, double>(a, p, d->val_dtype, grid, block, s);
    return launch_status();
}
