// lt_delense_tile.h -- the delensing scan's test of a tile of cells against a source, for the device
// kernel and for host checks of the same code.
//
// The scan has to find every (cell, source) pair for which cell_hit() (lt_delense_geom.h) is not 0, and a
// tile of 8 x 8 cells holds none for nearly every source. skip() proves that for a whole tile from
// numbers that cost a few instructions per vertex: each vertex is mapped to the source plane with the
// smallest and the largest D_ls/D_s of the sample's sources (lo, hi), and the tile keeps the boxes of
// both mappings and the range of three determinants per triangle.
//
// Why it is exact. For dr = (1 - t) lo + t hi a vertex maps to (1 - t) v(lo) + t v(hi), so
//   * every mapped vertex lies in the box (1 - t) box(lo) + t box(hi), and
//   * the determinant of a triangle with edges e, f at lo and e', f' at hi is
//     (1 - t)^2 e x f + t (1 - t) (e x f' + e' x f) + t^2 e' x f',
//     at least the smallest of b0 = e x f, b1 = (e x f' + e' x f) / 2, b2 = e' x f' (Bernstein form).
// With M a bound on the coordinates of pixels and mapped vertices, on dr |g| <= |p| + |v| and on the
// sources, each value computed here is within 2e-13 M^2 (determinants) or 1e-14 M (boxes) of the exact
// one of the corners that cell_hit() forms (their coordinates differ from these by a few roundings of
// M). If b0, 2 b1, b2 of both triangles of every cell exceed tau = 2e-10 M^2 in one sign, each |det| is
// above 9e-11 M^2 for every dr of the range, more than the 8 E / eps = 3.2e-11 M^2 of the proof in
// lt_delense_geom.h with eps = 1e-3 (E = 4e-15 M^2 bounds the rounding of a computed determinant). That proof needs a
// source at a distance m > eps / 2 times the diameter D of each triangle: m is at least the distance to
// the box along one axis, and D at most the box's width plus its height, so a source farther from the box
// than s = 1e-3 (width + height) + 1e-9 M is a miss for every triangle. Values that are not finite, or
// beyond 1e100, switch the test off: minima and maxima drop NaN, but a sum over the vertices
// holds it, and an infinity reaches the boxes or the sum.
#pragma once

#include <hip/hip_runtime.h>

#include "lt_delense_geom.h"

namespace lt {

// A vertex mapped with both ends of the D_ls/D_s range.
struct Vertex2 {
    double xl, yl, xh, yh;
};

__host__ __device__ inline Vertex2 map_vertex(double x, double y, double gx, double gy, double lo, double hi)
{
    return {__builtin_fma(-lo, gx, x), __builtin_fma(-lo, gy, y), __builtin_fma(-hi, gx, x), __builtin_fma(-hi, gy, y)};
}

__host__ __device__ inline Vertex2 edge(const Vertex2& a, const Vertex2& b)
{
    return {b.xl - a.xl, b.yl - a.yl, b.xh - a.xh, b.yh - a.yh};
}

struct TileBound {
    double lo[4], hi[4];  // smallest and largest x, y at lo and x, y at hi
    double dmin, dmax;    // range of b0, 2 b1, b2 over the triangles
    double sum;           // of the vertices: not finite when one is not
};

__host__ __device__ inline TileBound empty_tile()
{
    TileBound t;
    for (int k = 0; k < 4; ++k) {
        t.lo[k] = __builtin_inf();
        t.hi[k] = -__builtin_inf();
    }
    t.dmin = __builtin_inf();
    t.dmax = -__builtin_inf();
    t.sum = 0.;
    return t;
}

__host__ __device__ inline void add_vertices(TileBound& t, const Vertex2& a, const Vertex2& b)
{
    const double av[4] = {a.xl, a.yl, a.xh, a.yh}, bv[4] = {b.xl, b.yl, b.xh, b.yh};
    for (int k = 0; k < 4; ++k) {
        t.lo[k] = __builtin_fmin(t.lo[k], __builtin_fmin(av[k], bv[k]));
        t.hi[k] = __builtin_fmax(t.hi[k], __builtin_fmax(av[k], bv[k]));
    }
    t.sum += (a.xl + a.yl) + (b.xl + b.yl);
}

// a triangle with edges e and f from one vertex
__host__ __device__ inline void add_triangle(TileBound& t, const Vertex2& e, const Vertex2& f)
{
    const double b0 = __builtin_fma(e.xl, f.yl, -(e.yl * f.xl));
    const double b2 = __builtin_fma(e.xh, f.yh, -(e.yh * f.xh));
    const double b1 = __builtin_fma(e.xl, f.yh, -(e.yl * f.xh)) + __builtin_fma(e.xh, f.yl, -(e.yh * f.xl));
    t.dmin = __builtin_fmin(t.dmin, __builtin_fmin(b0, __builtin_fmin(b1, b2)));
    t.dmax = __builtin_fmax(t.dmax, __builtin_fmax(b0, __builtin_fmax(b1, b2)));
}

// What the test needs of a tile: pmax bounds |coordinates| of its pixels and of the sample's sources (NaN when a source is
// not finite), `finite` says that t.sum was finite in each part of the tile.
struct TileTest {
    double lo[4], hi[4], s;
    bool boxed;   // the boxes hold: a source outside them misses every triangle whose |det| is known to exceed tau
    bool det_ok;  // every triangle's does
};

__host__ __device__ inline TileTest tile_test(const TileBound& t, double pixmax, double srcmax, bool finite)
{
    TileTest r;
    double v = 0., w0 = 0., w1 = 0.;
    for (int k = 0; k < 4; ++k) {
        r.lo[k] = t.lo[k];
        r.hi[k] = t.hi[k];
        v = __builtin_fmax(v, __builtin_fmax(__builtin_fabs(t.lo[k]), __builtin_fabs(t.hi[k])));
        if (k < 2) w0 += t.hi[k] - t.lo[k];
        else w1 += t.hi[k] - t.lo[k];
    }
    const double m = __builtin_fmax(pixmax + v, srcmax) * 1.000001;
    r.s = __builtin_fma(1e-3, __builtin_fmax(w0, w1), 1e-9 * m);
    r.boxed = finite && srcmax <= 1e100 && m <= 1e100 && m >= 1e-50;
    const double tau = 2e-10 * m * m;
    r.det_ok = r.boxed && (t.dmin > tau || t.dmax < -tau);
    return r;
}

// How far source (px, py), with D_ls/D_s a share t of the way from lo to hi, is beyond the distance s from
// the tile's box: positive when outside. Never positive for a NaN.
__host__ __device__ inline double box_margin(const TileTest& r, double px, double py, double t)
{
    const double x0 = __builtin_fma(t, r.lo[2] - r.lo[0], r.lo[0]), x1 = __builtin_fma(t, r.hi[2] - r.hi[0], r.hi[0]);
    const double y0 = __builtin_fma(t, r.lo[3] - r.lo[1], r.lo[1]), y1 = __builtin_fma(t, r.hi[3] - r.hi[1], r.hi[1]);
    const double ex = __builtin_fmax(x0 - px, px - x1), ey = __builtin_fmax(y0 - py, py - y1);
    return __builtin_fmax(ex, ey) - r.s;
}

// the share t of a source's D_ls/D_s (lo <= dr <= hi)
__host__ __device__ inline double range_share(double dr, double lo, double hi)
{
    return hi > lo ? (dr - lo) / (hi - lo) : 0.;
}

}  // namespace lt
