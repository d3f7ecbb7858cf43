// lt_delense.hip -- image-plane -> source-plane delensing and the chi^2 of multiple-image families,
// batched over lens-model samples (blockIdx.z / one thread per sample where the work is serial).
//
//   source barycentres  src/chi_CPU_barycenter.cpp:173-210
//   delensing           src/delense_CPU.cpp:6-138, src/delense_CPU_utils.hpp:81-214
//   chi^2               src/chi_computation.cpp:10-195
//
// The geometry and the chi^2 are FP64 with contraction off, operation for operation as the
// reference expressions, so that for the same gradient planes the found images (and their order:
// the reference's single-thread row-major scan order) and the chi^2 are bit-identical to the CPU
// path. Hits are collected with atomics and then put back into scan order by a per-source sort.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "lenstool_hip/lt_status.h"
#include "lt_delense.h"
#include "lt_delense_geom.h"
#include "lt_delense_tile.h"
#include "lt_device.h"
#include "lt_math.h"

namespace lt {

// ------------------------------------------------------------------------------------------------
// source barycentres: one thread per (sample, family); images in order, sum then divide
// ------------------------------------------------------------------------------------------------
__global__ void k_barycentres(const double* __restrict__ img_gx, const double* __restrict__ img_gy,
                              DelenseDesc d)
{
#pragma clang fp contract(off)
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const int s = blockIdx.y;
    if (k >= d.nsets) return;
    const int first = d.first_image[k], ni = d.nimages[k];
    double sx = 0., sy = 0.;
    for (int i = first; i < first + ni; ++i) {
        const int64_t j = (int64_t)s * d.nimg_total + i;
        sx += d.img_x[i] - d.img_dr[i] * img_gx[j];
        sy += d.img_y[i] - d.img_dr[i] * img_gy[j];
    }
    const int64_t o = (int64_t)s * d.nsets + k;
    d.src_x[o] = sx / ni;
    d.src_y[o] = sy / ni;
    d.src_dr[o] = d.img_dr[first];
}

// corners of cell (xid, yid) of a sample's gradient planes, image-plane coordinates as the reference
// forms them (src/delense_CPU.cpp:64-85)
__device__ __forceinline__ CellCorners load_corners(const double* __restrict__ gx, const double* __restrict__ gy,
                                                    const DelenseDesc& d, int xid, int yid)
{
#pragma clang fp contract(off)
    const int n = d.n;
    const int64_t g = (int64_t)yid * n + xid;
    CellCorners c;
    c.xp = d.xmin + xid * d.dx;
    c.yp = d.ymin + yid * d.dy;
    c.xq = c.xp + d.dx;
    c.yq = c.yp + d.dy;
    c.g0x = gx[g];
    c.g0y = gy[g];
    c.g1x = gx[g + n];
    c.g1y = gy[g + n];
    c.g2x = gx[g + 1];
    c.g2y = gy[g + 1];
    c.g3x = gx[g + n + 1];
    c.g3y = gy[g + n + 1];
    return c;
}

// ------------------------------------------------------------------------------------------------
// per-sample bounds of the sources for the scan's cull: max |x|, |y| and the range of D_ls/D_s; a
// non-finite source makes the bounds NaN, which switches the cull off for the whole sample. One wavefront per
// sample, which also clears the sample's counters.
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(64) void k_source_bounds(DelenseDesc d)
{
    const int s = blockIdx.x, lane = threadIdx.x;
    double pmax = 0., lo = __builtin_inf(), hi = -__builtin_inf();
    bool finite = true;  // fmin / fmax drop NaN
    for (int k = lane; k < d.nsets; k += 64) {
        const int64_t sk = (int64_t)s * d.nsets + k;
        const double x = fabs(d.src_x[sk]), y = fabs(d.src_y[sk]), r = d.src_dr[sk];
        finite = finite && x <= 1e100 && y <= 1e100 && fabs(r) <= 1e100;
        pmax = fmax(pmax, fmax(x, y));
        lo = fmin(lo, r);
        hi = fmax(hi, r);
        d.count[sk] = 0;
    }
    finite = __ballot(!finite) == 0;
    pmax = wave_max64(pmax);
    lo = -wave_max64(-lo);
    hi = wave_max64(hi);
    if (lane == 0) {
        const double nan = __builtin_nan("");
        d.src_bound[3 * (int64_t)s] = finite ? pmax : nan;
        d.src_bound[3 * (int64_t)s + 1] = finite ? lo : nan;
        d.src_bound[3 * (int64_t)s + 2] = finite ? hi : nan;
        d.nitems[s] = 0;
        d.status[s] = 0;
    }
}

// append a hit of source k of sample s in cell `cell` (0 = none, 1 upper, 2 lower triangle)
__device__ __forceinline__ void record_hit(const DelenseDesc& d, int s, int k, int cell, int hit)
{
    if (!hit) return;
    const int64_t sk = (int64_t)s * d.nsets + k;
    const int slot = atomicAdd(&d.count[sk], 1);
    if (slot < DELENSE_CAP) d.hits[sk * DELENSE_CAP + slot] = cell * 2 + (hit - 1);
}

// ------------------------------------------------------------------------------------------------
// delensing scan: a wavefront takes 64 columns of 8 rows of cells, eight tiles of 8 x 8. Each lane walks
// down its column with the vertices on both sides of it, mapped to the source plane at both ends of the
// sample's D_ls/D_s range, and keeps their box and the range of the cells' determinants; eight lanes'
// make a tile (lt_delense_tile.h), which its lanes test against the sources, staged in LDS. Only
// (tile, source) pairs that the test leaves open go through the reference's triangle test, in k_delense_open: a
// wavefront's lanes take the 64 cells of the tile; tiles with a cell near a critical line (or values that are not
// finite) take each cell's own bounds on the determinant (lt_delense_geom.h).
// Bound by reading the planes: 1024 samples of 512 x 512 pixels in 1.31 ms, 3.7 TB/s with the rows that two
// wavefronts share, and about 70 VALU instructions per row of 64 cells. With a cell a lane, each bounding its own
// corners' distances and determinants, 300 of set-up per 64 cells took 4.18 ms. 152 registers, three wavefronts a
// SIMD, hold the nine rows' loads in flight; held to 128 it spills and takes 1.41 ms.
// ------------------------------------------------------------------------------------------------
constexpr int SCAN_BLOCK = 256;  // threads per block (4 wavefronts: 64 x 32 cells); also the sources staged in LDS per pass
constexpr int SCAN_WAVES = SCAN_BLOCK / 64;

// smallest / largest value over the eight lanes of a tile, in each of them
__device__ __forceinline__ double tile_min(double v)
{
    v = __builtin_fmin(v, dpp_move64<0xB1>(v));     // quad_perm [1, 0, 3, 2]
    v = __builtin_fmin(v, dpp_move64<0x4E>(v));     // quad_perm [2, 3, 0, 1]
    return __builtin_fmin(v, dpp_move64<0x141>(v));  // row_half_mirror
}

__device__ __forceinline__ double tile_max(double v) { return -tile_min(-v); }

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_or(uint32_t v)
{
    return v | (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, false);
}

__device__ __forceinline__ uint64_t tile_or(uint64_t v)
{
    const uint32_t lo = dpp_or<0x141>(dpp_or<0x4E>(dpp_or<0xB1>((uint32_t)v)));
    const uint32_t hi = dpp_or<0x141>(dpp_or<0x4E>(dpp_or<0xB1>((uint32_t)(v >> 32))));
    return ((uint64_t)hi << 32) | lo;
}

__global__ __launch_bounds__(SCAN_BLOCK) void k_delense(const double* __restrict__ gx, const double* __restrict__ gy,
                                                        DelenseDesc d)
{
    __shared__ double lsx[SCAN_BLOCK], lsy[SCAN_BLOCK], lst[SCAN_BLOCK];
    const int n = d.n;
    const int lane = (int)threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int s = blockIdx.z;
    const int x0 = blockIdx.x * 64, y0 = (blockIdx.y * SCAN_WAVES + wv) * SCAN_TILE;
    const bool rows = y0 < n - 1;  // a wavefront past the grid only stages sources
    const double* const px = gx + (int64_t)s * d.grid_stride;
    const double* const py = gy + (int64_t)s * d.grid_stride;
    const double* sb = d.src_bound + 3 * (int64_t)s;
    const double pmax = sb[0], lo = sb[1], hi = sb[2];

    TileTest tt = {};
    if (rows) {
        const int xid = min(x0 + lane, n - 2);  // lanes past the grid repeat its last column
        const int ncells = min(SCAN_TILE, n - 1 - y0);
        const double xa = d.xmin + xid * d.dx, xb = xa + d.dx;
        double ga[SCAN_TILE + 1][4];
#pragma unroll
        for (int k = 0; k <= SCAN_TILE; ++k) {
            const int64_t at = (int64_t)min(y0 + k, n - 1) * n + xid;
            ga[k][0] = px[at];
            ga[k][1] = py[at];
            ga[k][2] = px[at + 1];
            ga[k][3] = py[at + 1];
        }
        TileBound t = empty_tile();
        Vertex2 a, b, top;
#pragma unroll
        for (int k = 0; k <= SCAN_TILE; ++k) {
            if (k > ncells) continue;
            const double y = d.ymin + (y0 + k) * d.dy;
            const Vertex2 na = map_vertex(xa, y, ga[k][0], ga[k][1], lo, hi), nb = map_vertex(xb, y, ga[k][2], ga[k][3], lo, hi);
            const Vertex2 bottom = edge(na, nb);
            add_vertices(t, na, nb);
            if (k) {
                add_triangle(t, edge(a, na), top);
                add_triangle(t, edge(b, nb), bottom);
            }
            a = na;
            b = nb;
            top = bottom;
        }
        const uint64_t fin = __ballot(__builtin_fabs(t.sum) <= 1e100);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            t.lo[k] = tile_min(t.lo[k]);
            t.hi[k] = tile_max(t.hi[k]);
        }
        t.dmin = tile_min(t.dmin);
        t.dmax = tile_max(t.dmax);
        const double ya = d.ymin + y0 * d.dy, yb = d.ymin + (y0 + ncells) * d.dy;
        const double pix = tile_max(__builtin_fmax(__builtin_fmax(__builtin_fabs(xa), __builtin_fabs(xb)),
                                                   __builtin_fmax(__builtin_fabs(ya), __builtin_fabs(yb))));
        tt = tile_test(t, pix, pmax, ((fin >> (lane & 56)) & 0xff) == 0xff);
    }
    const bool inside = rows && x0 + (lane & 56) < n - 1;  // a tile of the grid
    const int64_t cap = scan_items(n, d.nsets);

    for (int k0 = 0; k0 < d.nsets; k0 += SCAN_BLOCK) {
        const int cnt = min(SCAN_BLOCK, d.nsets - k0);
        __syncthreads();  // the previous pass is done with the staged sources
        if ((int)threadIdx.x < cnt) {
            const int64_t sk = (int64_t)s * d.nsets + k0 + threadIdx.x;
            lsx[threadIdx.x] = d.src_x[sk];
            lsy[threadIdx.x] = d.src_y[sk];
            lst[threadIdx.x] = range_share(d.src_dr[sk], lo, hi);
        }
        __syncthreads();
        if (!rows) continue;
        for (int c0 = 0; c0 < cnt; c0 += SCAN_CHUNK) {
            // lane j of a tile tests sources j, j + 8, ..: bit 8 j + i of the tile's word is source 8 i + j
            uint32_t bits = 0;
            const int most = min(SCAN_CHUNK, cnt - c0);
            for (int i = 0; i * SCAN_TILE < most; ++i) {
                const int j = i * SCAN_TILE + (lane & 7), at = c0 + min(j, most - 1);
                const bool miss = tt.boxed && box_margin(tt, lsx[at], lsy[at], lst[at]) > 0.;
                if (j < most && !miss) bits |= 1u << i;
            }
            const uint64_t open = tile_or((uint64_t)bits << (8 * (lane & 7)));
            const bool item = inside && (lane & 7) == 0 && (open || !tt.det_ok);
            const uint64_t all = __ballot(item);
            if (!all) continue;
            int base = 0;
            if (lane == 0) base = atomicAdd(&d.nitems[s], __builtin_popcountll(all));
            base = __builtin_amdgcn_readfirstlane(base);
            if (item) {
                ScanItem it;
                it.open = open;
                it.tile = (y0 / SCAN_TILE) * scan_tiles(n) + (x0 + lane) / SCAN_TILE;
                it.chunk = ((k0 + c0) / SCAN_CHUNK) * 2 + (tt.det_ok ? 1 : 0);
                d.items[s * cap + base + __builtin_popcountll(all & ((1ull << lane) - 1))] = it;
            }
        }
    }
}

// The tiles that k_delense left open, one wavefront per tile and 64 sources, a lane per cell. In a kernel of their
// own: they lie along the critical lines and around the images, and a wavefront of the scan that met eight of them
// took longer than all others together (both in one kernel: 45 us for one sample of 40 sources on 512 x 512, 3561 for
// 1024; apart 7 + 10 and 1312 + 773). Bound by the cells' set-up along the critical lines.
__global__ __launch_bounds__(SCAN_BLOCK) void k_delense_open(const double* __restrict__ gx, const double* __restrict__ gy,
                                                             DelenseDesc d)
{
    const int n = d.n;
    const int s = blockIdx.y;
    const int lane = (int)threadIdx.x & 63;
    const int64_t cap = scan_items(n, d.nsets);
    const int nitems = d.nitems[s], step = (int)gridDim.x * SCAN_WAVES;
    const double* sb = d.src_bound + 3 * (int64_t)s;
    for (int i = blockIdx.x * SCAN_WAVES + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); i < nitems; i += step) {
        const ScanItem it = d.items[s * cap + i];
        const int xid = (it.tile % scan_tiles(n)) * SCAN_TILE + (lane & 7), yid = (it.tile / scan_tiles(n)) * SCAN_TILE + (lane >> 3);
        const bool active = xid < n - 1 && yid < n - 1;
        const int cell = yid * (n - 1) + xid;
        const CellCorners c = load_corners(gx + (int64_t)s * d.grid_stride, gy + (int64_t)s * d.grid_stride, d, min(xid, n - 2), min(yid, n - 2));
        const int k0 = (it.chunk >> 1) * SCAN_CHUNK;
        const int64_t s0 = (int64_t)s * d.nsets + k0;
        // the chunk's sources, one a lane: taken from there without a wait on memory
        const int64_t mine = s0 + min(lane, min(SCAN_CHUNK, d.nsets - k0) - 1);
        const double lx = d.src_x[mine], ly = d.src_y[mine], ldr = d.src_dr[mine];
        if (it.chunk & 1) {
            uint64_t open = it.open;
            while (open) {
                const int p = __builtin_ctzll(open), k = (p & 7) * 8 + (p >> 3);
                open &= open - 1;
                if (active) record_hit(d, s, k0 + k, cell, cell_hit(c, read_lane64(lx, k), read_lane64(ly, k), read_lane64(ldr, k)));
            }
            continue;
        }
        const CellFilter f = cell_filter(c, sb[0], sb[1], sb[2]);
        for (int k = 0; k < min(SCAN_CHUNK, d.nsets - k0); ++k) {
            // outside the tile's box a cell needs its own determinants only
            const double sx = read_lane64(lx, k), sy = read_lane64(ly, k), dr = read_lane64(ldr, k);
            const double du = __builtin_fma(dr, __builtin_fma(dr, f.c2u, f.c1u), f.c0);
            const double dl = __builtin_fma(dr, __builtin_fma(dr, f.c2l, f.c1l), f.c0);
            const bool out = !((it.open >> ((k & 7) * 8 + (k >> 3))) & 1);
            const bool miss = out & f.on & (__builtin_fmin(abs_d(du), abs_d(dl)) > f.tau);
            if (active && !miss && !far_from_cell(f, c, sx, sy, dr)) record_hit(d, s, k0 + k, cell, cell_hit(c, sx, sy, dr));
        }
    }
}

// ------------------------------------------------------------------------------------------------
// back to scan order, barycentres of the first MAXIMPERSOURCE hits: one thread per (sample, source)
// ------------------------------------------------------------------------------------------------
__global__ void k_delense_finish(const double* __restrict__ gx, const double* __restrict__ gy, DelenseDesc d)
{
#pragma clang fp contract(off)
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const int s = blockIdx.y;
    if (k >= d.nsets) return;
    const int64_t sk = (int64_t)s * d.nsets + k;
    int cnt = d.count[sk];
    int status = LT_OK;
    if (cnt > LT_MAXIMPERSOURCE) status = LT_ERR_OVERFLOW;
    int* h = d.hits + sk * DELENSE_CAP;
    if (cnt > DELENSE_CAP) {
        // the slots hold an arbitrary subset of the hits: take the first MAXIMPERSOURCE in scan order
        // again, serially (an error case: the status says the source overflowed)
        const int64_t base = (int64_t)s * d.grid_stride;
        int got = 0;
        for (int yid = 0; yid < d.n - 1 && got < LT_MAXIMPERSOURCE; ++yid)
            for (int xid = 0; xid < d.n - 1 && got < LT_MAXIMPERSOURCE; ++xid) {
                const int hit = cell_hit(load_corners(gx + base, gy + base, d, xid, yid), d.src_x[sk], d.src_y[sk],
                                         d.src_dr[sk]);
                if (hit) h[got++] = (yid * (d.n - 1) + xid) * 2 + (hit - 1);
            }
        cnt = got;
    }
    const int kept = cnt;
    for (int i = 1; i < kept; ++i) {  // insertion sort: cell-major, upper before lower
        int v = h[i], j = i - 1;
        while (j >= 0 && h[j] > v) {
            h[j + 1] = h[j];
            --j;
        }
        h[j + 1] = v;
    }
    const int nout = kept < LT_MAXIMPERSOURCE ? kept : LT_MAXIMPERSOURCE;
    for (int i = 0; i < nout; ++i) {
        const int code = h[i];
        const int cell = code >> 1;
        const int yid = cell / (d.n - 1), xid = cell % (d.n - 1);
        const double xp = d.xmin + xid * d.dx;
        const double yp = d.ymin + yid * d.dy;
        double bx, by;
        if ((code & 1) == 0) {  // upper (x,y) (x,y+dy) (x+dx,y)
            bx = (xp + xp + (xp + d.dx)) / 3.;
            by = (yp + (yp + d.dy) + yp) / 3.;
        } else {  // lower (x+dx,y+dy) (x+dx,y) (x,y+dy)
            bx = ((xp + d.dx) + (xp + d.dx) + xp) / 3.;
            by = ((yp + d.dy) + yp + (yp + d.dy)) / 3.;
        }
        d.pos_x[sk * LT_MAXIMPERSOURCE + i] = bx;
        d.pos_y[sk * LT_MAXIMPERSOURCE + i] = by;
    }
    d.loc[sk] = nout;
    if (status != LT_OK) atomicMax(&d.status[s], status);
}

// ------------------------------------------------------------------------------------------------
// chi^2 matching (src/chi_computation.cpp:10-195, with its two early-stopping loop conditions at
// :110 and :118): a wavefront per sample, a lane per source writes the per-image chi terms; the wavefront
// then sums them in the reference's order, 64 terms loaded at a time (one thread that loaded each as it
// summed took 15 us for a sample of 120 images, 36 for 1024 samples). The matching is a serial chain on what it indexes by
// image, so that lies in LDS: 14 us a sample with the sum, 20 from private arrays in memory.
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ double pdist(double ax, double ay, double bx, double by)
{
#pragma clang fp contract(off)
    double x = ax - bx, y = ay - by;
    return sqrt(x * x + y * y);
}

// Per lane: the family's observed and found images and the matching's state, in LDS (indexed by image: in private
// arrays they live in memory).
struct ChiLds {
    double ox[LT_MAXIMPERSOURCE][64], oy[LT_MAXIMPERSOURCE][64], fx[LT_MAXIMPERSOURCE][64], fy[LT_MAXIMPERSOURCE][64];
    double tx[LT_MAXIMPERSOURCE][64], ty[LT_MAXIMPERSOURCE][64], dist[LT_MAXIMPERSOURCE][64];
    int nfound[LT_MAXIMPERSOURCE][64];
};

__device__ __forceinline__ void chi_match(const DelenseDesc& d, int s, int k, int nf, ChiLds& m)
{
#pragma clang fp contract(off)
    const int l = threadIdx.x;
    const int64_t sk = (int64_t)s * d.nsets + k;
    const int first = d.first_image[k], ni = d.nimages[k];
#pragma unroll 4
    for (int i = 0; i < ni; ++i) {
        m.ox[i][l] = d.img_x[first + i];
        m.oy[i][l] = d.img_y[first + i];
        m.tx[i][l] = m.ty[i][l] = 0.;
        m.nfound[i][l] = 0;
    }
#pragma unroll 4
    for (int i = 0; i < nf; ++i) {
        m.fx[i][l] = d.pos_x[sk * LT_MAXIMPERSOURCE + i];
        m.fy[i][l] = d.pos_y[sk * LT_MAXIMPERSOURCE + i];
    }
    for (int ii = 0; ii < nf; ++ii) {
        const double px = m.fx[ii][l], py = m.fy[ii][l];
        int idx = 0;
        double least = pdist(px, py, m.ox[0][l], m.oy[0][l]);
        m.dist[0][l] = least;
        for (int i = 1; i < ni; i++) {
            const double v = pdist(px, py, m.ox[i][l], m.oy[i][l]);
            m.dist[i][l] = v;
            if (v < least) {
                idx = i;
                least = v;
            }
        }
        if (m.nfound[idx][l] == 0) {
            m.tx[idx][l] = px;
            m.ty[idx][l] = py;
            m.nfound[idx][l]++;
        } else if (m.nfound[idx][l] > 0) {
            double tmpx, tmpy;
            if (least < pdist(m.ox[idx][l], m.oy[idx][l], m.tx[idx][l], m.ty[idx][l])) {
                tmpx = m.tx[idx][l];
                tmpy = m.ty[idx][l];
                m.tx[idx][l] = px;
                m.ty[idx][l] = py;
            } else {
                tmpx = px;
                tmpy = py;
            }
            int second = 0;
            for (int i = 1; i < ni && (i != idx); i++)
                if (m.dist[i][l] > m.dist[second][l]) second = i;
            for (int i = 0; i < ni && m.nfound[i][l] == 0; i++) {
                if (m.dist[i][l] < m.dist[second][l]) {
                    second = i;
                    idx = i;
                    m.tx[idx][l] = tmpx;
                    m.ty[idx][l] = tmpy;
                }
            }
            m.nfound[idx][l]++;
        }
    }
    for (int i = 0; i < ni; i++) {
        double term;
        if (m.nfound[i][l] > 0) {
            double p1 = m.ox[i][l] - m.tx[i][l];
            double p2 = m.oy[i][l] - m.ty[i][l];
            term = p1 * p1 + p2 * p2;
        } else {
            term = 1000. * ni;
        }
        d.terms[(int64_t)s * d.nimg_total + first + i] = term;
    }
}

__global__ __launch_bounds__(64) void k_chi(DelenseDesc d)
{
#pragma clang fp contract(off)
    __shared__ ChiLds lds;
    const int s = blockIdx.x, lane = threadIdx.x;
    int found = 0;
    for (int k = lane; k < d.nsets; k += 64) {
        const int nf = d.loc[(int64_t)s * d.nsets + k];
        chi_match(d, s, k, nf, lds);
        found += nf;
    }
    __syncthreads();  // the terms are written
    const double* const terms = d.terms + (int64_t)s * d.nimg_total;
    double chi = 0.;
    for (int i = 0; i < d.nimg_total; i += 64) {
        const int n = min(64, d.nimg_total - i);
        const double t = terms[i + min(lane, n - 1)];
        for (int j = 0; j < n; ++j) chi += read_lane64(t, j);
    }
#pragma unroll
    for (int m = 32; m; m >>= 1) found += __shfl_xor(found, m);
    if (lane == 0) {
        d.chi[s] = chi;
        d.found[s] = found;
    }
}

// ------------------------------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------------------------------
hipError_t launch_barycentres(const double* img_gx, const double* img_gy, const DelenseDesc& d, hipStream_t s)
{
    hipLaunchKernelGGL(k_barycentres, dim3((d.nsets + 63) / 64, d.nsamples), dim3(64), 0, s, img_gx, img_gy, d);
    return hipGetLastError();
}

hipError_t launch_delense(const double* gx, const double* gy, const DelenseDesc& d, hipStream_t s)
{
    hipLaunchKernelGGL(k_source_bounds, dim3((unsigned)d.nsamples), dim3(64), 0, s, d);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    dim3 blk(SCAN_BLOCK);
    constexpr int rows = SCAN_WAVES * SCAN_TILE;
    dim3 grd((unsigned)((d.n - 1 + 63) / 64), (unsigned)((d.n - 1 + rows - 1) / rows), (unsigned)d.nsamples);
    hipLaunchKernelGGL(k_delense, grd, blk, 0, s, gx, gy, d);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    // open tiles: about 4096 work-groups over the samples, at most 256 (as many tiles as 512 x 512 pixels leave) and at
    // least 8 of them for a sample
    const int groups = std::min(256, std::max(8, 4096 / d.nsamples));
    hipLaunchKernelGGL(k_delense_open, dim3((unsigned)groups, (unsigned)d.nsamples), blk, 0, s, gx, gy, d);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_delense_finish, dim3((d.nsets + 63) / 64, d.nsamples), dim3(64), 0, s, gx, gy, d);
    return hipGetLastError();
}

hipError_t launch_chi(const DelenseDesc& d, hipStream_t s)
{
    hipLaunchKernelGGL(k_chi, dim3((unsigned)d.nsamples), dim3(64), 0, s, d);
    return hipGetLastError();
}

}  // namespace lt
