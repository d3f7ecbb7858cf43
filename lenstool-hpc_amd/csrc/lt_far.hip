// lt_far.hip -- halo sums on large grids by tile expansions: the halos far from a tile of pixels are
// summed once at 16 x 16 Chebyshev nodes of the tile and interpolated to its pixels, the near ones are
// summed at every pixel as in lt_kernels64.hip.
//
// Why it is the same sum. A halo's gradient, Hessian and potential are analytic functions of x and of y;
// their only complex singularities lie where w^2 = r^2 + a^2 x^2 + b^2 y^2 = 0 (halo frame; r the smaller
// of its radii; SIS: R^2 = 0) or where the deflection's Q = 0, which is never closer than the halo's
// centre. For one real and one complex coordinate the distance from (x0, y0) to the former is at least
// w(x0, y0) / b. Chebyshev interpolation of order 16 on [-h, h] of a function whose nearest singularity
// is K h away from the middle has an error of about (K + sqrt(K^2 - 1))^-16 of it. A halo is far from a
// tile of half side h when w(centre) >= 6 b h, so K >= 5 along both axes wherever the other coordinate
// lies in the tile: measured in 80-bit arithmetic over ellipticities up to 0.6 (potential), cores from
// zero to the tile's distance, all directions, the error is at most 2.5e-15 of the halo's own term for a
// halo just outside the bound (1e-17 in the median) and below 1e-16 from 1.2 times the bound on. That is
// the rounding of the direct sum (which takes each term with reciprocals good to 2^-48); the nodes use
// the fully corrected ones, so a map's error against the extended oracle is no larger than the direct
// kernel's.
//
// Geometry. The levels halve: LV = 3: a work-group of 16 waves takes a root of 4 UNIT pixels a side; halos
// far from all of it are summed at the root's nodes, a sixteenth of them by each wave. Each of its four subs
// (2 UNIT) starts from the root's coefficients shifted to it (T_k(+-1/2 + t/2) in T_m(t)) and adds the
// halos near the root but far from the sub, a quarter of them by each of four waves; each of the four units
// of a sub goes to one wave. LV = 2: a work-group of 4 waves, one sub as its root. Units of 64 pixels are
// expanded and then worked off in quarters of 32; at 32 pixels (units or quarters) the halos between it and
// its parent are expanded where there are kFarRefine of them and otherwise summed with the near ones.
// Everything is aligned to the grid's own pixel indices (col + istart, row + jstart), so a sub-grid gets the
// same squares, the same sets and the same values bit for bit.
//
// The pixels: out = Ty^T C Tx with C the 16 x 16 coefficients and T the Chebyshev polynomials at the pixels'
// own rounded coordinates, as FP64 matrix instructions (16 x 16 x 4). D's layout (lane 16 q + j, register
// s: row 4 s + q, column j) is the A operand's layout of the transposed matrix for step s, so products
// chain in registers, and a lane's four node values enter the first transform as they are.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include "lenstool_hip/lt_status.h"
#include "lt_cheb_tables.h"
#include "lt_device.h"
#include "lt_far.h"
#include "lt_kernels.h"
#define LT_HORNER_COEF "s"
#include "lt_math.h"
#include "lt_terms64.h"

namespace lt {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int FP = 16;                     // nodes per axis
constexpr int FN = FP * FP;
constexpr int FWORDS = kFarMaxHalos / 64;  // words of a halo mask
constexpr double kFarBound2 = 36.0;        // (K + 1)^2
constexpr int kFarIlp = 2;                  // pixels or nodes whose terms are interleaved
constexpr int kFarRefine = 3;               // halos between a tile and a quarter from which the quarter is expanded

// waves of a work-group and pixels of its side
constexpr int far_waves(int lv) { return lv == 3 ? 16 : 4; }
constexpr int far_side(int lv, int unit) { return (lv == 3 ? 4 : 2) * unit; }


template <int FAM>
constexpr int fields_of()
{
    return FAM == FAM_HESSIAN ? 3 : FAM == FAM_GRADIENT ? 2 : 1;
}

__device__ __forceinline__ d4 mfma64(double a, double b, d4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// a wave-uniform 64-bit word in scalar registers
__device__ __forceinline__ uint64_t uniform64(uint64_t v)
{
    const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}

// the halos [start, end) of word w as a mask
__device__ __forceinline__ uint64_t run_bits(int w, int start, int end)
{
    const int lo = start - w * 64, hi = end - w * 64;
    uint64_t m = ~0ull;
    if (lo > 0) m &= ~0ull << lo;
    if (hi < 64) m &= ~(~0ull << hi);
    return m;
}

// one halo's term at NP offsets (tx, ty[k]) added to acc[field][k]; FULL: as for the nodes
template <int FAM, int TYPE, bool CIRC, bool FULL, int NP>
__device__ __forceinline__ void add_halo(const HaloRec& h, double tx, const double* ty, double (*acc)[NP], double* mn)
{
#pragma unroll
    for (int k = 0; k < NP; ++k) {
        if (k && k % kFarIlp == 0) __builtin_amdgcn_sched_barrier(0);
        if constexpr (FAM == FAM_HESSIAN) {
            if constexpr (TYPE == TYPE_DPIE) hess_piemd_at<true, FULL>(h, tx, ty[k], acc[0][k], acc[1][k], acc[2][k]);
            else if constexpr (TYPE == TYPE_PIEMD) hess_piemd_at<false, FULL>(h, tx, ty[k], acc[0][k], acc[1][k], acc[2][k]);
            else if constexpr (TYPE == TYPE_SIS && CIRC) hess_sis_circ_at<FULL>(h, tx, ty[k], acc[0][k], acc[1][k], acc[2][k]);
            else if constexpr (TYPE == TYPE_SIS) hess_sis_at<FULL>(h, tx, ty[k], acc[0][k], acc[1][k], acc[2][k]);
            else {
                acc[0][k] += h.h14a + h.h14c;
                acc[1][k] += h.h14a - h.h14c;
                acc[2][k] += h.h14b;
            }
        } else if constexpr (FAM == FAM_TRACE) {
            double d = 0., b = 0.;  // unused: the compiler drops them with everything that only they need
            if constexpr (TYPE == TYPE_DPIE) hess_piemd_at<true, FULL>(h, tx, ty[k], acc[0][k], d, b);
            else if constexpr (TYPE == TYPE_PIEMD) hess_piemd_at<false, FULL>(h, tx, ty[k], acc[0][k], d, b);
            else if constexpr (TYPE == TYPE_SIS && CIRC) hess_sis_circ_at<FULL>(h, tx, ty[k], acc[0][k], d, b);
            else if constexpr (TYPE == TYPE_SIS) hess_sis_at<FULL>(h, tx, ty[k], acc[0][k], d, b);
            else acc[0][k] += h.h14a + h.h14c;
        } else if constexpr (FAM == FAM_GRADIENT) {
            if constexpr (TYPE == TYPE_DPIE) grad_piemd_at<true, FULL>(h, tx, ty[k], acc[0][k], acc[1][k]);
            else if constexpr (TYPE == TYPE_PIEMD) grad_piemd_at<false, FULL>(h, tx, ty[k], acc[0][k], acc[1][k]);
            else if constexpr (CIRC) grad_sis_circ_at(h, tx, ty[k], acc[0][k], acc[1][k]);
            else grad_sis_at(h, tx, ty[k], acc[0][k], acc[1][k]);
        } else {
            add_pot_halo<FULL>(h, TYPE, tx, ty[k], acc[0][k], mn[k]);
        }
    }
}

// The halos of a set, run by run with the run's weight, at the offsets (cx - xh) + ox, (cy - yh) + oy[k]: the
// node offsets are added to the square's offset from the halo, so a node's position carries no rounding of the
// field's own coordinates (as the direct sum's pixel - centre). For pixels cx = cy = 0 and ox, oy are the
// pixel. A set is mask words in LDS (wave-uniform; `pick` restricts them to every n-th bit) over the halos
// (list NULL) or over the positions of a list of halo indices; a run is a range of bits.
struct HaloSet {
    const uint64_t* words;
    const uint16_t* list;
    const int* bounds;  // list: positions where the runs start, nruns + 1 of them
};

template <int FAM, int TYPE, bool CIRC, bool FULL, int NP, bool LIST>
__device__ __forceinline__ void sum_type(const HaloRec* __restrict__ halos, const HaloSet& set, uint64_t pick,
                                         int start, int end, double cx, double cy, double ox, const double* oy,
                                         double (*acc)[NP], double* mn)
{
    for (int w = start >> 6; w <= (end - 1) >> 6; ++w) {
        uint64_t m = uniform64(set.words[w]) & pick & run_bits(w, start, end);
        while (m) {
            int i = w * 64 + __builtin_ctzll(m);
            m &= m - 1;
            if constexpr (LIST) i = __builtin_amdgcn_readfirstlane(set.list[i]);
            const HaloRec& h = halos[i];
            double ty[NP];
#pragma unroll
            for (int k = 0; k < NP; ++k) ty[k] = FULL ? (cy - h.yh) + oy[k] : oy[k] - h.yh;
            add_halo<FAM, TYPE, CIRC, FULL, NP>(h, FULL ? (cx - h.xh) + ox : ox - h.xh, ty, acc, mn);
        }
    }
}

template <int FAM, bool FULL, int NP, bool LIST>
__device__ __forceinline__ void sum_halos(const HaloRec* __restrict__ halos, const Run* __restrict__ runs, int nruns,
                                          const HaloSet& set, uint64_t pick, double cx, double cy, double ox,
                                          const double* oy, double (*tot)[NP], double* mn)
{
    constexpr int NF = fields_of<FAM>();
    for (int r = 0; r < nruns; ++r) {
        const Run run = runs[r];
        const int start = LIST ? __builtin_amdgcn_readfirstlane(set.bounds[r]) : run.start;
        const int end = LIST ? __builtin_amdgcn_readfirstlane(set.bounds[r + 1]) : run.start + run.count;
        if (start >= end) continue;
        double acc[NF][NP];
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int k = 0; k < NP; ++k) acc[f][k] = 0.;
        if (run.type == TYPE_DPIE)
            sum_type<FAM, TYPE_DPIE, false, FULL, NP, LIST>(halos, set, pick, start, end, cx, cy, ox, oy, acc, mn);
        else if (run.type == TYPE_PIEMD)
            sum_type<FAM, TYPE_PIEMD, false, FULL, NP, LIST>(halos, set, pick, start, end, cx, cy, ox, oy, acc, mn);
        else if (run.type == TYPE_SIS && run.circ && FAM != FAM_POTENTIAL)
            sum_type<FAM, TYPE_SIS, true, FULL, NP, LIST>(halos, set, pick, start, end, cx, cy, ox, oy, acc, mn);
        else if (run.type == TYPE_SIS)
            sum_type<FAM, TYPE_SIS, false, FULL, NP, LIST>(halos, set, pick, start, end, cx, cy, ox, oy, acc, mn);
        else if constexpr (FAM == FAM_HESSIAN || FAM == FAM_TRACE)
            sum_type<FAM, TYPE_SHEAR, false, FULL, NP, LIST>(halos, set, pick, start, end, cx, cy, ox, oy, acc, mn);
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int k = 0; k < NP; ++k) tot[f][k] = __builtin_fma(run.weight, acc[f][k], tot[f][k]);
    }
}

__device__ __forceinline__ int floor_div(int a, int b)
{
    const int q = a / b;
    return q * b > a ? q - 1 : q;
}

// One axis of a root tile: centre c and half side h (signed as the pixel step) with c, c +- h/2 exact:
// h is the side rounded up to 24 bits, c a multiple of h 2^-20; the pixels lie inside [c - h, c + h].
struct Axis {
    double c, h;
};

__device__ __forceinline__ Axis root_axis(double xmin, double d, int i0, int side)
{
    Axis a;
    a.h = (double)(float)(0.5 * (double)side * d * (1. + 1e-6));
    const double q = a.h * 0x1p-20;
    a.c = __builtin_rint((xmin + ((double)i0 + 0.5 * (double)(side - 1)) * d) / q) * q;
    return a;
}

// a copy of v that the compiler cannot form ahead of this point (keeps table loads out of the registers of
// the halo loops before it)
__device__ __forceinline__ int opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// T_{4 s + q}(t), s = 0 .. 3, for this lane's q: T_{n + 4} = 2 T_4 T_n - T_{n - 4}
__device__ __forceinline__ d4 cheb4(double t, int q)
{
    const double t2 = __builtin_fma(2. * t, t, -1.);
    const double t3 = __builtin_fma(2. * t, t2, -t);
    const double t4 = __builtin_fma(2. * t2, t2, -1.);
    const bool hi = q & 2, lo = q & 1;
    const double n0 = hi ? (lo ? t3 : t2) : (lo ? t : 1.);    // T_q
    const double nm = hi ? (lo ? t : t2) : (lo ? t3 : t4);    // T_{4 - q}
    d4 r;
    r[0] = n0;
    r[1] = __builtin_fma(2. * t4, n0, -nm);
    r[2] = __builtin_fma(2. * t4, r[1], -n0);
    r[3] = __builtin_fma(2. * t4, r[2], -r[1]);
    return r;
}

// Chebyshev coefficients M N M^T of the node values n (register s of lane 16 q + j: node row 4 s + q, column
// j) added to c (same layout)
__device__ __forceinline__ d4 transform(const d4& n, int j, int q, d4 c)
{
    const int at = opaque(j * FP + q);
    d4 t = {0., 0., 0., 0.};
#pragma unroll
    for (int s = 0; s < 4; ++s) t = mfma64(n[s], kDct[at + 4 * s], t);
#pragma unroll
    for (int s = 0; s < 4; ++s) c = mfma64(t[s], kDct[at + 4 * s], c);
    return c;
}

// S_y C S_x^T: the coefficients c of a parent on its half (sx, sy)
__device__ __forceinline__ d4 shift_half(const d4& c, int sx, int sy, int q, int j)
{
    const int at = opaque(j * FP + q);
    d4 t = {0., 0., 0., 0.}, r = {0., 0., 0., 0.};
#pragma unroll
    for (int s = 0; s < 4; ++s) t = mfma64(c[s], kShift[sy * FN + at + 4 * s], t);
#pragma unroll
    for (int s = 0; s < 4; ++s) r = mfma64(t[s], kShift[sx * FN + at + 4 * s], r);
    return r;
}

// far from the square at (cx, cy): w(centre)^2 >= 36 b^2 h^2 = bound b^2; a NaN makes the halo near. A potential's
// halo whose centre may lie in the square is near however large its core: a pixel on a PIEMD centre is NaN, which
// only its own sum can tell (X^2 + Y^2 <= d^2, and d <= sqrt(2) h inside).
template <int FAM>
__device__ __forceinline__ bool is_far(const FarRec& h, double cx, double cy, float bound)
{
    const float tx = (float)(cx - h.xh), ty = (float)(cy - h.yh);
    const float X = __builtin_fmaf(tx, h.a, ty * h.b);
    const float Y = __builtin_fmaf(ty, h.c, -(tx * h.d));
    const float d2 = __builtin_fmaf(X, X, Y * Y);
    return d2 + h.f >= bound && (FAM != FAM_POTENTIAL || d2 > bound * (2.1f / 36.f));
}

// The halos of `from` (mask words over the list) far from the square at (cx, cy), the others to `near`. Words
// first, first + step, .. of nwords.
template <int FAM>
__device__ __forceinline__ void split_sets(const FarRec* __restrict__ recs, const uint16_t* list, int count, int first,
                                           int step, const uint64_t* from, double cx, double cy, double bound,
                                           uint64_t* far, uint64_t* near)
{
    const int lane = threadIdx.x & 63;
    for (int w = first; w * 64 < count; w += step) {
        uint64_t f = run_bits(w, 0, count), m = 0;
        if (from) f = from[w];
        f = uniform64(f);
        if (f) m = __ballot(is_far<FAM>(recs[list[min(w * 64 + lane, count - 1)]], cx, cy, (float)bound)) & f;
        if (lane == 0) {
            far[w] = m;
            near[w] = f & ~m;
        }
    }
}

// sums of the halos of `set` (every `pick`ed one) at this lane's four nodes of the square at (cx, cy)
template <int FAM, bool LIST>
__device__ __forceinline__ void node_sums(const HaloRec* __restrict__ halos, const Run* __restrict__ runs, int nruns,
                                          const HaloSet& set, uint64_t pick, double cx, double cy, double hx,
                                          double hy, d4* out)
{
    constexpr int NF = fields_of<FAM>();
    const int lane = threadIdx.x & 63;
    double acc[NF][4], oy[4], unused[4] = {1., 1., 1., 1.};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        oy[k] = hy * kNode[4 * k + (lane >> 4)];
#pragma unroll
        for (int f = 0; f < NF; ++f) acc[f][k] = 0.;
    }
    sum_halos<FAM, true, 4, LIST>(halos, runs, nruns, set, pick, cx, cy, hx * kNode[lane & 15], oy, acc, unused);
#pragma unroll
    for (int f = 0; f < NF; ++f) out[f] = d4{acc[f][0], acc[f][1], acc[f][2], acc[f][3]};
}

__device__ __forceinline__ d4 load4(const double* p, int lane)
{
    return d4{p[lane], p[64 + lane], p[128 + lane], p[192 + lane]};
}

__device__ __forceinline__ void store4(double* p, int lane, const d4& v)
{
#pragma unroll
    for (int k = 0; k < 4; ++k) p[64 * k + lane] = v[k];
}

// Bound by the FP64 pipes: VALU issue (70 % of the cycles on the 503-halo 4096^2 fields, 88 % on the 2048^2 potential) and,
// for light models, matrix instructions beside it (38 % and 26 % on 256 maps of 11 halos). Work-groups of 4 waves are held to
// three waves a SIMD (168 registers): 256 magnitude maps of 2048^2 in 7.1 ms, 8.7 with two, 8.8 with four, which spills
// (7.3 with the logarithm that carries its remainders). The logarithm's and arctangent's coefficients stay in scalar
// registers, 36 vector registers less: the potential 2048^2, 503 halos, roots of 128, 825 -> 800 us, displacement
// 701 x 643, 160 mixed halos, 152 -> 146.
// PARTS 2 and 4: the halves or the subs of a root go to a work-group each, all of which sum its nodes: a map of fewer than
// 128 roots would leave the other CUs idle (displacement 701 x 643, 160 mixed halos, 121 roots: 147 us, halved 87).
template <int FAM, int KIND, int LV, int UNIT, int PARTS>
__global__ __launch_bounds__(WAVE* far_waves(LV) / PARTS, LV == 3 && PARTS < 4 ? 4 : 3) void k_far(const HaloRec* __restrict__ halos,
                                                                                     const FarRec* __restrict__ recs,
                                                                                     const Run* __restrict__ runs,
                                                                                     int nruns, int nhalos, GridDesc g,
                                                                                     OutDesc o)
{
    constexpr int NF = fields_of<FAM>();
    constexpr int NW = far_waves(LV) / PARTS, NS = NW / 4;  // waves = units, subs
    constexpr int SIDE = far_side(LV, UNIT);
    __shared__ double part[NW][NF][FN];  // node sums of each wave; later the coefficients that it expands
    __shared__ double rootc[LV == 3 ? NF : 1][FN], subc[NS][NF][FN];
    __shared__ double rootref[NF], subref[NS][NF];
    // halo sets: far from the root (the sub, for LV 2) over all halos; the others as a list, and masks over the
    // list's positions
    __shared__ uint64_t top[FWORDS], sfar[LV == 3 ? NS : 1][FWORDS], snear[LV == 3 ? NS : 1][FWORDS];
    __shared__ uint64_t ufar[UNIT > 16 ? NW : 1][FWORDS], unear[UNIT > 16 ? NW : 1][FWORDS];
    __shared__ uint64_t qnear[UNIT == 64 ? NW : 1][FWORDS];
    __shared__ uint16_t list[kFarMaxHalos];
    __shared__ int first[FWORDS + 1], bounds[kFarMaxRuns + 1];

    halos = select_sample(g, halos, o);
    recs += (int64_t)blockIdx.z * g.halo_stride;
    const int lane = threadIdx.x & 63, q = lane >> 4, j = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), sub = wave >> 2, wv = wave & 3;
    const int place = sub + (int)blockIdx.y % PARTS * NS;  // of the sub in the root
    const int nwords = (nhalos + 63) >> 6;
    const int i0 = (floor_div(g.istart, SIDE) + (int)blockIdx.x) * SIDE;
    const int j0 = (floor_div(g.jstart, SIDE) + (int)blockIdx.y / PARTS) * SIDE;
    if constexpr (PARTS > 1) {  // a part past the grid
        const int down = j0 - g.jstart + (place >> 1) * (SIDE / 2), across = PARTS == 4 ? i0 - g.istart + (place & 1) * (SIDE / 2) : 0;
        if (down + SIDE / 2 <= 0 || down >= g.ny || across + SIDE / 2 <= 0 || across >= g.nx) return;
    }
    const Axis ax = root_axis(g.xmin, g.dx, i0, SIDE), ay = root_axis(g.ymin, g.dy, j0, SIDE);
    // centre and half sides (signed as the pixel steps) of the wave's sub
    const double shx = LV == 3 ? 0.5 * ax.h : ax.h, shy = LV == 3 ? 0.5 * ay.h : ay.h;
    const double scx = LV == 3 ? ax.c + ((place & 1) ? shx : -shx) : ax.c;
    const double scy = LV == 3 ? ay.c + ((place >> 1) ? shy : -shy) : ay.c;
    const double hm = __builtin_fmax(__builtin_fabs(shx), __builtin_fabs(shy)), sb2 = kFarBound2 * hm * hm;

    // ---- root and sub: sets, node sums by all waves, then one wave per field transforms. The value at a
    // middle node is taken off first and added to the pixels last, so that the transforms round only the
    // field's variation over the square
    const double tcx = LV == 3 ? ax.c : scx, tcy = LV == 3 ? ay.c : scy;
    for (int w = wave; w < nwords; w += NW) {
        const uint64_t f = run_bits(w, 0, nhalos);
        const uint64_t m =
            __ballot(is_far<FAM>(recs[min(w * 64 + lane, nhalos - 1)], tcx, tcy, (float)(LV == 3 ? 4. * sb2 : sb2))) & f;
        if (lane == 0) {
            top[w] = m;
            first[w] = nwords > 1 ? __builtin_popcountll(f & ~m) : 0;
            if (nwords == 1) first[1] = __builtin_popcountll(f & ~m);
        }
    }
    __syncthreads();
    // the list: positions by a prefix sum over the words, kept in halo order
    if (nwords > 1) {
        if (wave == 0) {
            int v = lane < nwords ? first[lane] : 0, sum = v;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int t = __shfl_up(sum, d);
                if (lane >= d) sum += t;
            }
            if (lane < nwords) first[lane] = sum - v;
            if (lane == 63) first[nwords] = sum;
        }
        __syncthreads();
    }
    for (int w = wave; w < nwords; w += NW) {
        const uint64_t m = run_bits(w, 0, nhalos) & ~uniform64(top[w]);
        if ((m >> lane) & 1) list[first[w] + __builtin_popcountll(m & ((1ull << lane) - 1))] = (uint16_t)(w * 64 + lane);
    }
    if ((int)threadIdx.x <= nruns) {
        const int at = (int)threadIdx.x < nruns ? runs[threadIdx.x].start : nhalos, w = at >> 6;
        bounds[threadIdx.x] = at < nhalos ? first[w] + __builtin_popcountll(~top[w] & ((1ull << (at & 63)) - 1)) : first[nwords];
    }
    __syncthreads();
    const int nlist = __builtin_amdgcn_readfirstlane(first[nwords]);
    d4 n[NF];
    if constexpr (LV == 3) {
        split_sets<FAM>(recs, list, nlist, wv, 4, nullptr, scx, scy, sb2, sfar[sub], snear[sub]);
        node_sums<FAM, false>(halos, runs, nruns, HaloSet{top, nullptr, nullptr}, (NW == 4 ? 0x1111111111111111ull : NW == 8 ? 0x0101010101010101ull : 0x0001000100010001ull) << wave, ax.c, ay.c,
                              ax.h, ay.h, n);
#pragma unroll
        for (int f = 0; f < NF; ++f) store4(part[wave][f], lane, n[f]);
        __syncthreads();
        if (wave < NF) {
            d4 v = {0., 0., 0., 0.};
            for (int p = 0; p < NW; ++p) v += load4(part[p][wave], lane);
            const double r = read_lane64(v[2], 8);
            store4(rootc[wave], lane, transform(v - r, j, q, d4{0., 0., 0., 0.}));
            if (lane == 0) rootref[wave] = r;
        }
        __syncthreads();
        node_sums<FAM, true>(halos, runs, nruns, HaloSet{sfar[sub], list, bounds}, 0x1111111111111111ull << wv, scx, scy,
                             shx, shy, n);
    } else {
        node_sums<FAM, false>(halos, runs, nruns, HaloSet{top, nullptr, nullptr}, 0x1111111111111111ull << wv, scx, scy,
                              shx, shy, n);
    }
#pragma unroll
    for (int f = 0; f < NF; ++f) store4(part[wave][f], lane, n[f]);
    __syncthreads();
    if (wv < NF) {
        d4 v = (load4(part[4 * sub][wv], lane) + load4(part[4 * sub + 1][wv], lane)) +
               (load4(part[4 * sub + 2][wv], lane) + load4(part[4 * sub + 3][wv], lane));
        double r = read_lane64(v[2], 8);
        v -= r;
        d4 c = {0., 0., 0., 0.};
        if constexpr (LV == 3) {
            c = shift_half(load4(rootc[wv], lane), place & 1, place >> 1, q, j);
            r += rootref[wv];
        }
        store4(subc[sub][wv], lane, transform(v, j, q, c));
        if (lane == 0) subref[sub][wv] = r;
    }
    __syncthreads();

    // ---- the wave's unit; no work-group barrier from here on
    const int urow = j0 + (place >> 1) * 2 * UNIT + (wv >> 1) * UNIT - g.jstart;
    const int ucol = i0 + (place & 1) * 2 * UNIT + (wv & 1) * UNIT - g.istart;
    if (urow + UNIT - 1 < 0 || urow >= g.ny || ucol + UNIT - 1 < 0 || ucol >= g.nx) return;
    const double uhx = 0.5 * shx, uhy = 0.5 * shy;
    const double ucx = scx + ((wv & 1) ? uhx : -uhx), ucy = scy + ((wv >> 1) ? uhy : -uhy);
    uint64_t *const uf = ufar[UNIT > 16 ? wave : 0], *const un = UNIT > 16 ? unear[wave] : snear[sub];
    if constexpr (UNIT > 16) {
        split_sets<FAM>(recs, list, nlist, 0, 1, LV == 3 ? snear[sub] : nullptr, ucx, ucy, 0.25 * sb2, uf, un);
        wave_sync();
    }
    double (*const own)[FN] = part[wave];
    d4 uc[NF];          // UNIT 64: the unit's coefficients
    double uref[NF];
    if constexpr (UNIT == 64) {
        node_sums<FAM, true>(halos, runs, nruns, HaloSet{uf, list, bounds}, ~0ull, ucx, ucy, uhx, uhy, n);
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            const double r = read_lane64(n[f][2], 8);
            uref[f] = subref[sub][f] + r;
            uc[f] = transform(n[f] - r, j, q, shift_half(load4(subc[sub][f], lane), wv & 1, wv >> 1, q, j));
        }
    }
#pragma unroll 1
    for (int u = 0; u < (UNIT == 64 ? 4 : 1); ++u) {
        // the square of 32 x 32 pixels, its parent, and the half of the parent that it is
        const int hx = UNIT == 64 ? u & 1 : wv & 1, hy = UNIT == 64 ? u >> 1 : wv >> 1;
        const int row0 = UNIT == 64 ? urow + 32 * hy : urow, col0 = UNIT == 64 ? ucol + 32 * hx : ucol;
        if (UNIT == 64 && (row0 + 31 < 0 || row0 >= g.ny || col0 + 31 < 0 || col0 >= g.nx)) continue;
        const double phx = UNIT == 64 ? uhx : shx, phy = UNIT == 64 ? uhy : shy;
        const double pcx = UNIT == 64 ? ucx : scx, pcy = UNIT == 64 ? ucy : scy;
        const double qcx = pcx + (hx ? 0.5 : -0.5) * phx, qcy = pcy + (hy ? 0.5 : -0.5) * phy;
        uint64_t* const qn = UNIT == 64 ? qnear[wave] : un;
        if constexpr (UNIT == 64) {
            split_sets<FAM>(recs, list, nlist, 0, 1, un, qcx, qcy, 0.0625 * sb2, uf, qn);
            wave_sync();
        }
        bool refine = false;  // units of 16 pixels: expanded from their sub
        if constexpr (UNIT > 16) {
            int between = 0;
            for (int w = 0; w * 64 < nlist; ++w) between += __builtin_popcountll(uniform64(uf[w]));
            refine = between >= kFarRefine;
        }
        double ref[NF];
        if (refine)
            node_sums<FAM, true>(halos, runs, nruns, HaloSet{uf, list, bounds}, ~0ull, qcx, qcy, 0.5 * phx, 0.5 * phy, n);
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            d4 c = UNIT == 64 ? uc[f] : load4(subc[sub][f], lane);
            ref[f] = UNIT == 64 ? uref[f] : subref[sub][f];
            if (refine) {
                const double r = read_lane64(n[f][2], 8);
                ref[f] += r;
                c = transform(n[f] - r, j, q, shift_half(c, hx, hy, q, j));
            }
            store4(own[f], lane, c);
        }
        if (UNIT > 16 && !refine)
            for (int w = lane; w * 64 < nlist; w += 64) qn[w] |= uf[w];
        wave_sync();
        const double ecx = refine ? qcx : pcx, ecy = refine ? qcy : pcy;
        const double iex = (refine ? 2. : 1.) / phx, iey = (refine ? 2. : 1.) / phy;
#pragma unroll 1
        for (int rb = 0; rb < (UNIT > 16 ? 2 : 1); ++rb) {
            // coefficients in x of 16 rows: register s of lane 16 q + j: order 4 s + q of row j
            d4 gk[NF];
            {
                const d4 ty = cheb4((pixel_coord(g.ymin, row0 + 16 * rb + j + g.jstart, g.dy) - ecy) * iey, q);
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    gk[f] = d4{0., 0., 0., 0.};
#pragma unroll
                    for (int s = 0; s < 4; ++s) gk[f] = mfma64(own[f][64 * s + lane], ty[s], gk[f]);
                }
            }
            double py[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) py[k] = pixel_coord(g.ymin, row0 + 16 * rb + 4 * k + q + g.jstart, g.dy);
#pragma unroll 1
            for (int cb = 0; cb < (UNIT > 16 ? 2 : 1); ++cb) {
                const int col = col0 + 16 * cb + j;
                const double px = pixel_coord(g.xmin, col + g.istart, g.dx);
                const d4 tx = cheb4((px - ecx) * iex, q);
                double v[NF][4];
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    d4 d = {0., 0., 0., 0.};
#pragma unroll
                    for (int s = 0; s < 4; ++s) d = mfma64(gk[f][s], tx[s], d);
#pragma unroll
                    for (int k = 0; k < 4; ++k) v[f][k] = d[k] + ref[f];
                }
                double mn[4] = {1., 1., 1., 1.};
                sum_halos<FAM, false, 4, true>(halos, runs, nruns, HaloSet{qn, list, bounds}, ~0ull, 0., 0., px, py, v, mn);
                if (col >= 0 && col < g.nx) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        __builtin_amdgcn_sched_barrier(0);
                        const int row = row0 + 16 * rb + 4 * k + q;
                        if (row < 0 || row >= g.ny) continue;
                        const int64_t idx = (int64_t)row * g.pitch + col;
                        if constexpr (FAM == FAM_HESSIAN) {
                            hess_epilogue<KIND>(o, idx, v[0][k], v[1][k], v[2][k]);
                        } else if constexpr (FAM == FAM_TRACE) {
                            hess_epilogue<KIND>(o, idx, v[0][k], 0., 0.);
                        } else if constexpr (FAM == FAM_GRADIENT) {
                            const double m = o.kind == LT_MAP_DPL ? o.r : 1.0;
                            o.p0[idx] = v[0][k] * m;
                            o.p1[idx] = v[1][k] * m;
                        } else {
                            // a pixel on a PIEMD centre: the reference's potential is 0/0 there
                            o.p0[idx] = mn[k] == 0. ? __builtin_nan("") : v[0][k] * o.mult;
                        }
                    }
                }
            }
        }
        wave_sync();  // the next quarter reuses the wave's sets and coefficients
    }
}

// ------------------------------------------------------------------------------------------------
// the rule
// ------------------------------------------------------------------------------------------------
FarStats far_stats(int nhalos, const std::vector<Run>& runs)
{
    FarStats st;
    st.nhalos = nhalos;
    st.nruns = (int)runs.size();
    st.cost = model_cost(runs);
    return st;
}

double halo_density(const HaloRec* recs, const std::vector<Run>& runs)
{
    double x0 = INFINITY, x1 = -INFINITY, y0 = INFINITY, y1 = -INFINITY, sum = 0;
    int n = 0;
    for (const Run& r : runs) {
        if (r.type == TYPE_SHEAR) continue;  // constant: far everywhere
        for (int i = r.start; i < r.start + r.count; ++i) {
            const HaloRec& h = recs[i];
            x0 = std::min(x0, h.xh);
            x1 = std::max(x1, h.xh);
            y0 = std::min(y0, h.yh);
            y1 = std::max(y1, h.yh);
            // ellipse X^2 + Y^2 < bound, X and Y the scaled frame
            sum += M_PI * kFarBound2 * h.kx * (h.cs * h.cs + h.sn * h.sn) / std::fabs(h.csx * h.csy + h.snx * h.sny);
            ++n;
        }
    }
    if (!n) return 0.;
    const double area = (x1 - x0) * (y1 - y0);
    return area > 0. ? std::exp2(0.25 * std::rint(4. * std::log2(sum / n / area))) : INFINITY;
}

void far_records(const HaloRec* recs, int nhalos, FarRec* out)
{
    for (int i = 0; i < nhalos; ++i) {
        const HaloRec& h = recs[i];
        FarRec& r = out[i];
        r = FarRec{};
        r.xh = h.xh;
        r.yh = h.yh;
        r.f = 3.0e38f;       // type 14, a constant: far from everything
        if (!(h.kx > 0.)) continue;
        // W^2 / a^2, in units of b^2 h^2 after W = cx1 w, cx1 b = a. (The halo frame is the caller's cos and sin: where
        // they are not of norm 1 it is as much larger than the lab frame, and so is the square in it.)
        const double n2 = h.cs * h.cs + h.sn * h.sn, s = 1. / std::sqrt(h.kx * n2);
        r.a = (float)(s * h.csx);
        r.b = (float)(s * h.snx);
        r.c = (float)(s * h.csy);
        r.d = (float)(s * h.sny);
        r.f = (float)std::fmin(h.far0 / (h.kx * n2), 1.0e38);
    }
}

static unsigned tiles_over(int start, int n, int side);

// Tile expansions cost, per pixel, the halos near its 32-pixel square, 256 nodes over the area of a square for each
// halo first expanded there, and the expansion itself (72 matrix instructions per 1024 pixels and three fields,
// in VALU issue slots). From that count and the number of work-groups follows a time in cycles of a CU (four
// instructions a cycle and 64 lanes), with the efficiencies and fixed shares that were measured: a root of 64 pixels
// takes 1.15 times its count and about 100 000 cycles beside it (its barriers and the longest wave), a half or a
// quarter of one 1.25 and 1.5 times its share, the root's nodes included, and about half as much. Over 176 maps (20 to 1000 halos, four kinds, 240^2 to 2100^2)
// the shape taken is 2 % behind the best of the six in the mean. Some of them, us (direct, 4 waves, 16, halves, quarters):
//   dpl 672 x 635, 160 mixed halos: 233, 174, 158, 100; fields 450 x 413, 258 dPIE: 129, 214, 174, 110;
//   potential 450 x 413, 1000 dPIE: 1638, 2409, 2262, 1300; fields 900 x 863, 258: 498, 118, 101, 121.
//   light models (1 dPIE + 10 SIS): 256 maps of 2048^2 in 7.1 ms with 4 waves, 17.6 with 16.
//   503 halos, 4096^2: root 128 565 us, root 64 1145; 2000 on 8192^2: root 256 2.6 ms, root 128 5.3.
// Where roots of 128 pixels halve the count of 64 with these shares added (fine pixels, many halos), the shape depends on
// the steps and the lens alone, so that a part of a map takes the same form as the whole; roots of 256 again have to halve
// the count of 128: their
// work-groups are few and uneven (a 300 x 200 part of the 4096^2 map: 271 us, 111 with 128, 183 directly).
// Elsewhere the quickest shape is taken, or the direct sum.
FarShape far_shape(const FarStats& st, double density, int kind, int precision, const GridDesc& g, double* cost)
{
    const int fam = family_of(kind);
    const double d = st.cost.px[fam], direct = direct_cost(st.cost, kind, precision);
    if (cost) *cost = direct;
    if (st.nhalos < 1 || st.nhalos > kFarMaxHalos || st.nruns > kFarMaxRuns) return FarShape::Direct;
    const double dx = std::fabs(g.dx), dy = std::fabs(g.dy);
    // (the far tests square lengths in FP32)
    if (!(std::fmin(dx, dy) > 0.) || !(std::fmax(dx, dy) >= 1e-15) || !(std::fmax(dx, dy) <= 1e15)) return FarShape::Direct;
    // pixel coordinates must resolve the squares: |coordinate| <= 2^30 steps
    const double cx = std::fabs(g.xmin) + (std::fabs((double)g.istart) + g.nx) * dx;
    const double cy = std::fabs(g.ymin) + (std::fabs((double)g.jstart) + g.ny) * dy;
    if (!(cx <= 0x1p30 * dx) || !(cy <= 0x1p30 * dy)) return FarShape::Direct;
    // share of the halos near a square of n pixels a side
    auto near = [&](double n) {
        const double h = 0.5 * n * std::fmax(dx, dy);
        return std::fmin(1., density * h * h);
    };
    auto per_px = [&](int side) {
        double nodes = 0., above = 1.;  // the halos not yet expanded
        for (int m = side; m >= 32; m /= 2) {
            nodes += (above - near(m)) * FN / ((double)m * m);
            above = near(m);
        }
        return d * (nodes + near(32)) + (fam == FAM_HESSIAN ? 80. : fam == FAM_GRADIENT ? 55. : 30.);
    };
    auto tiles = [&](int side) {
        return (double)tiles_over(g.istart, g.nx, side) * (double)tiles_over(g.jstart, g.ny, side);
    };
    const double c64 = per_px(64), c128 = per_px(128), c256 = per_px(256);
    if (2. * (c128 + 280.) <= c64 + 100. && 1.25 * c128 < direct) {
        const bool wide = 2. * c256 <= c128;
        if (cost) *cost = wide ? c256 : c128;
        return wide ? FarShape::Root256 : FarShape::Root128;
    }
    const double npix = (double)g.nx * (double)g.ny;
    double best = npix * direct / (64. * 256. * 0.62) + 15e3;
    FarShape shape = FarShape::Direct;
    auto offer = [&](FarShape f, double t, double c) {
        if (t >= best) return;
        best = t;
        shape = f;
        if (cost) *cost = c;
    };
    const double n64 = tiles(64), n128 = tiles(128);
    const double root = d * (1. - near(64)) * FN / 4096., fixed = fam == FAM_POTENTIAL ? 130e3 : 100e3;
    const auto rounds = [](double groups) { return groups <= 256. ? 1. : std::fmin(std::ceil(groups / 256.), 1.35 * groups / 256.); };
    offer(FarShape::Root64, n64 < 512. ? 1.2 * 64. * c64 * rounds(n64) + fixed : n64 / 256. * (c64 * 64. / 0.55 + 8e3), c64);
    offer(FarShape::Root64Wide, 1.15 * 64. * c64 * rounds(n64) + fixed, c64);
    offer(FarShape::Root64Half, 1.25 * 32. * (c64 + root) * rounds(2. * n64) + 0.55 * fixed, c64);
    offer(FarShape::Root64Quarter, 1.5 * 16. * (c64 + 3. * root) * rounds(4. * n64) + 0.45 * fixed, c64);
    offer(FarShape::Root128, rounds(n128) * 1.4 * c128 * 256. + 160e3, c128);
    return shape;
}

// tiles of side `side` that cover n pixels from global index start
static unsigned tiles_over(int start, int n, int side)
{
    const auto fd = [side](int64_t v) { return v >= 0 ? v / side : -((-v + side - 1) / side); };
    return (unsigned)(fd((int64_t)start + n - 1) - fd(start) + 1);
}

template <int FAM, int KIND, int LV, int UNIT, int PARTS = 1>
static void launch_far_shape(const HaloRec* halos, const FarRec* recs, const Run* runs, int nruns, int nhalos, const GridDesc& g,
                             const OutDesc& o, hipStream_t s)
{
    constexpr int side = far_side(LV, UNIT);
    const dim3 grd(tiles_over(g.istart, g.nx, side), PARTS * tiles_over(g.jstart, g.ny, side),
                   (unsigned)(g.nsamples > 0 ? g.nsamples : 1));
    hipLaunchKernelGGL((k_far<FAM, KIND, LV, UNIT, PARTS>), grd, dim3(WAVE * far_waves(LV) / PARTS), 0, s, halos, recs, runs, nruns,
                       nhalos, g, o);
}

template <int FAM, int KIND>
static hipError_t launch_far_kind(const HaloRec* halos, const FarRec* recs, const Run* runs, int nruns, int nhalos, const GridDesc& g,
                                  const OutDesc& o, FarShape shape, hipStream_t s)
{
    switch (shape) {
    case FarShape::Root64: launch_far_shape<FAM, KIND, 2, 32>(halos, recs, runs, nruns, nhalos, g, o, s); break;
    case FarShape::Root64Wide: launch_far_shape<FAM, KIND, 3, 16>(halos, recs, runs, nruns, nhalos, g, o, s); break;
    case FarShape::Root64Half: launch_far_shape<FAM, KIND, 3, 16, 2>(halos, recs, runs, nruns, nhalos, g, o, s); break;
    case FarShape::Root64Quarter: launch_far_shape<FAM, KIND, 3, 16, 4>(halos, recs, runs, nruns, nhalos, g, o, s); break;
    case FarShape::Root128: launch_far_shape<FAM, KIND, 3, 32>(halos, recs, runs, nruns, nhalos, g, o, s); break;
    case FarShape::Root256: launch_far_shape<FAM, KIND, 3, 64>(halos, recs, runs, nruns, nhalos, g, o, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_far(const HaloRec* halos, const FarRec* recs, const Run* runs, int nruns, int nhalos, const GridDesc& g,
                      const OutDesc& o, FarShape shape, hipStream_t s)
{
    switch (o.kind) {
    case LT_MAP_GRADIENT:
    case LT_MAP_DPL: return launch_far_kind<FAM_GRADIENT, LT_MAP_GRADIENT>(halos, recs, runs, nruns, nhalos, g, o, shape, s);
    case LT_MAP_POT: return launch_far_kind<FAM_POTENTIAL, LT_MAP_POT>(halos, recs, runs, nruns, nhalos, g, o, shape, s);
    case LT_MAP_FIELDS: return launch_far_kind<FAM_HESSIAN, LT_MAP_FIELDS>(halos, recs, runs, nruns, nhalos, g, o, shape, s);
    case LT_MAP_AMPLI: return launch_far_kind<FAM_HESSIAN, LT_MAP_AMPLI>(halos, recs, runs, nruns, nhalos, g, o, shape, s);
    case LT_MAP_SHEAR: return launch_far_kind<FAM_HESSIAN, LT_MAP_SHEAR>(halos, recs, runs, nruns, nhalos, g, o, shape, s);
    case LT_MAP_MASS: return launch_far_kind<FAM_TRACE, LT_MAP_MASS>(halos, recs, runs, nruns, nhalos, g, o, shape, s);
    default: return launch_far_kind<FAM_HESSIAN, LT_MAP_HESSIAN>(halos, recs, runs, nruns, nhalos, g, o, shape, s);
    }
}

}  // namespace lt
