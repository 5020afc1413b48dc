// FP64 short-range pair force -- the plain path.
//
// Every target's sum runs over its neighbour cells in the reference's order:
// ix, iy, iz ascending over
//   [(int)(fac*(x-rcut)+M)-M, (int)(fac*(x+rcut))]  (gravlist.cpp:233-243),
// and inside a cell the particles in stable-sorted order
// (gravlist_kernel.cu:195-213).  With x-major keys the cells of one (ix,iy)
// column are contiguous in the sorted array, so each column is one or two
// contiguous j ranges (two when the z range wraps), read straight from the
// CSR offsets.  Columns and z cells that cannot hold a particle within rcut
// are skipped; that only removes pairs whose r^2 exceeds rcut^2, so the
// summation order of the surviving terms equals the reference loop's.
// Three ways of walking share the targets of a clustered box (plan, below);
// each adds the same terms in the same order, so which one takes a target does
// not show in its bits.
//
// Measured (pair force alone, kernel times; one target per lane throughout,
// then shared by three walks in x-major order, now): 128^3 halo particles
// 62.7, 55.5, 45.6 ms; 100003 on a 90 mesh 11.3, 3.1, 2.1; active sets of a
// 64^3 timeline 21, 7.7, 5.0.  Bound by the vector unit: at 128^3 the teams
// and the list issue vector instructions in 71% of the cycles, and all
// walks together take 73 of them for 64 ordered pairs inside the cut
// (counters over the whole launches, their ends included).
//
// The pair law is gravlist.cpp:279-327 (with the source mass), evaluated in
// the same operation order as the C source; this file is compiled with
// -ffp-contract=off, so no multiply-add is fused and the FP64 result is
// bit-identical to the CPU restatement.
#include <algorithm>

#include "internal.h"

namespace cuco {

namespace {

constexpr int kThreads = 256;

// sqrt(x) and n / d for the ranges pair terms take, correctly rounded
// without the extreme-exponent scaling and special-value selects a general
// sqrt and divide need.  sqrt_pair: 2^-767 <= x < 2^1023 (0 gives NaN; the
// pairs inside h, the only ones it can come from, take it back); half_inv:
// 1 / (2 sqrt(x)) to 2^-46, from the same iteration.
__device__ inline double sqrt_pair(double x, double &half_inv)
{
    double y = __builtin_amdgcn_rsq(x);
    double g = x * y;
    double h = y * 0.5;
    const double e = fma(-h, g, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    double d = fma(-g, g, x);
    g = fma(d, h, g);
    d = fma(-g, g, x);
    g = fma(d, h, g);
    half_inv = h;
    return g;
}

// Normal n and d whose quotient and reciprocal stay normal (masses over
// cubed distances, the spline's 0.06667 / u^3 with u >= 0.5).  y: 1 / d to
// 2^-44 or better; one step makes it 1 / d to half an ulp and 2^-88, which is
// the nearest double unless 1 / d lies within 2^-88 of the middle of two (one
// d in 2^34).  With the nearest y the quotient is the nearest too (Markstein's
// theorem on q + r y); with the other neighbour it can only differ where n / d
// itself is within 3 units of 2^-106 of a middle (at most a few n in 2^52 for
// each such d).
__device__ inline double div_from(double n, double d, double y)
{
    const double e = fma(-d, y, 1.0);
    y = fma(y, e, y);
    const double q = n * y;
    const double r = fma(-d, q, n);
    return fma(r, y, q);
}

__device__ inline double div_pair(double n, double d)
{
    const double y = __builtin_amdgcn_rcp(d);
    return div_from(n, d, fma(y, fma(-d, y, 1.0), y));
}

// m / (r2 r) with r = sqrt_pair(r2, h): the reciprocal starts from 8 h^3
// (three times the error of h, 2^-44.4, and four roundings) instead of a
// second quarter-rate instruction and its step.
__device__ inline double over_cube(double m, double r2, double r, double h)
{
    return div_from(m, r2 * r, h * h * (h * 8.0));
}

// Cell pruning only has to keep every cell that can hold a pair inside
// rcut: cells it keeps beyond rcut contribute nothing (their pairs fail the
// r^2 test) and do not change the order of the others.  So it runs in FP32
// with margins far above FP32 rounding of coordinates below 2^12 cells.
//
// Squared distance in cell units from u to the cell interval [c, c+1), made
// smaller by the margin.
__device__ inline float gap_cells(float u, int c)
{
    float g = fmaxf(0.0f, fmaxf((float)c - u, u - (float)(c + 1)));
    g = fmaxf(0.0f, g - 1e-2f);
    return g * g;
}

__device__ inline int wave_min_i(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
    return __builtin_amdgcn_readfirstlane(v);
}

__device__ inline int wave_max_i(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    return __builtin_amdgcn_readfirstlane(v);
}

// z cells of column (ix, iy) that can hold a pair inside rcut for the target
// at cell coordinate uz: [za, zb] inside the reference range [zl, zr], or
// za > zb.  gxy: squared gap to the column in cells (both widened by the
// margin).
__device__ inline void z_window(float uz, float gxy, float rc2, int zl, int zr, int &za, int &zb)
{
    const float zext = sqrtf(fmaxf(rc2 - gxy, 0.0f)) + 1e-2f;
    za = max(zl, (int)floorf(uz - zext));
    zb = min(zr, (int)floorf(uz + zext));
}

// Part h of the z window [za, zb] of a column: 0 before the wrap (all of it
// when it does not wrap), 1 after.  [z0, z1], empty when z0 > z1.
__device__ inline void window_part(int za, int zb, int M, int h, int &z0, int &z1)
{
    const int wrap = za < 0 ? 0 : M;  // first z past the wrap
    z0 = h == 0 ? za : max(za, wrap);
    z1 = h == 0 ? min(zb, wrap - 1) : zb;
}

// Image shift of a neighbour cell index c (unwrapped) on a mesh of M.
__device__ inline double image_shift(int c, int M, double L)
{
    return c < 0 ? -L : (c >= M ? L : 0.0);
}

// The reference's neighbour cell range of one target (gravlist.cpp:233-243,
// unwrapped) and what the pruning needs.
struct Reach {
    int xl, xr, yl, yr, zl, zr;
    float ux, uy, uz, rc2;
};

__device__ inline Reach reach_of(const PairParams &pp, const double4 &p)
{
    const int M = pp.M;
    const double fac = pp.fac;
    Reach t;
    t.xl = (int)(fac * (p.x - pp.rcut) + M) - M;
    t.xr = (int)(fac * (p.x + pp.rcut));
    t.yl = (int)(fac * (p.y - pp.rcut) + M) - M;
    t.yr = (int)(fac * (p.y + pp.rcut));
    t.zl = (int)(fac * (p.z - pp.rcut) + M) - M;
    t.zr = (int)(fac * (p.z + pp.rcut));
    t.ux = (float)(fac * p.x);
    t.uy = (float)(fac * p.y);
    t.uz = (float)(fac * p.z);
    t.rc2 = (float)(pp.rcut * fac * pp.rcut * fac) * (1.0f + 1e-4f);
    return t;
}

__device__ inline bool in_box(const PairParams &pp, const double4 &p)
{
    return p.x >= 0 && p.x < pp.L && p.y >= 0 && p.y < pp.L && p.z >= 0 && p.z < pp.L;
}

// Union of the live lanes' cell ranges, and whether the wave's targets sit
// within a handful of z cells of one column (compact: the uniform walk where
// no plan has weighed it).
struct Union {
    int XL, XR, YL, YR, ZL, ZR;
    bool any, fits, compact;  // fits: less than a mesh wide, so no cell twice
};

__device__ inline Union wave_union(const Reach &t, bool live, int M)
{
    constexpr int kBig = 1 << 30;
    Union u;
    u.XL = wave_min_i(live ? t.xl : kBig);
    u.XR = wave_max_i(live ? t.xr : -kBig);
    u.YL = wave_min_i(live ? t.yl : kBig);
    u.YR = wave_max_i(live ? t.yr : -kBig);
    u.ZL = wave_min_i(live ? t.zl : kBig);
    u.ZR = wave_max_i(live ? t.zr : -kBig);
    u.any = u.XL <= u.XR;
    u.fits = u.XR - u.XL < M && u.YR - u.YL < M && u.ZR - u.ZL < M;
    const bool near = u.XR - u.XL <= (t.xr - t.xl) + 1 && u.YR - u.YL <= (t.yr - t.yl) + 1 &&
                      u.ZR - u.ZL <= (t.zr - t.zl) + 8;
    u.compact = u.fits &&
                __builtin_amdgcn_readfirstlane((uint32_t)(__ballot(live && !near) == 0ull)) != 0u;
    return u;
}

// The wave-uniform walk: the candidates of a compact wave's 64 targets
// together, in the reference order (ix, iy, z ascending, unwrapped).  The
// column pieces (a piece: the part of one (ix, iy) column in one z image,
// one contiguous run of sorted particles) are enumerated one per lane from
// the box around the targets; the non-empty ones, compacted into lanes
// 0..nr-1, are then read back as scalars.  A lane needs no window of its
// own: what it must not count lies beyond rcut, except that a pair within
// rounding of rcut is checked against the lane's own cell range (in_cut).
// One wave-wide reduction per column instead took longer than the pairs of
// a column of 30.
struct WalkBox {
    float ux0, ux1, uy0, uy1, uz0, uz1;  // box of the targets, in cells
    int XL, YL, ZL, ZR;                  // union of the cell ranges
    uint32_t ny, halves, npieces;
    float rc2;
};

__device__ inline float wave_min_f(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

__device__ inline float wave_max_f(float v) { return -wave_min_f(-v); }

__device__ inline WalkBox walk_box(const Reach &t, const Union &un, bool live, int M)
{
    const float inf = __builtin_huge_valf();
    WalkBox w;
    w.ux0 = wave_min_f(live ? t.ux : inf);
    w.ux1 = wave_max_f(live ? t.ux : -inf);
    w.uy0 = wave_min_f(live ? t.uy : inf);
    w.uy1 = wave_max_f(live ? t.uy : -inf);
    w.uz0 = wave_min_f(live ? t.uz : inf);
    w.uz1 = wave_max_f(live ? t.uz : -inf);
    w.XL = un.XL;
    w.YL = un.YL;
    w.ZL = un.ZL;
    w.ZR = un.ZR;
    w.ny = (uint32_t)(un.YR - un.YL + 1);
    w.halves = un.ZL < 0 || un.ZR >= M ? 2u : 1u;
    w.npieces = (uint32_t)(un.XR - un.XL + 1) * w.ny * w.halves;
    w.rc2 = t.rc2;
    return w;
}

// Squared distance in cells from the interval [u0, u1] to the cell interval
// [c, c+1), made smaller by the margin.
__device__ inline float gap_box(float u0, float u1, int c)
{
    float g = fmaxf(0.0f, fmaxf((float)c - u1, u0 - (float)(c + 1)));
    g = fmaxf(0.0f, g - 1e-2f);
    return g * g;
}

__device__ inline uint32_t incl_scan(uint32_t v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}

__device__ inline uint32_t uni(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ inline int image_code(int c, int M) { return c < 0 ? 0 : (c >= M ? 2 : 1); }

// Up to 64 pieces of the walk.  Lane k < nr: piece k holds the candidates
// numbered up to end (exclusive; from the piece before's), candidate f being
// sorted particle first + f; code: the image per axis, 2 bits each.
struct Batch {
    uint32_t first, end, code;
    uint32_t nr, total;  // wave-uniform
};

__device__ inline void push(uint32_t &v, int to)
{
    v = (uint32_t)__builtin_amdgcn_ds_permute(to * 4, (int)v);
}

__device__ inline void walk_batch(const WalkBox &w, uint32_t b,
                                  const uint32_t *__restrict__ off, int M, Batch &o)
{
    const int lane = threadIdx.x & 63;
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const uint32_t k = b + (uint32_t)lane;
    uint32_t js = 0, c = 0;
    o.code = 0;
    if (k < w.npieces) {
        const uint32_t col = w.halves == 2u ? k >> 1 : k;
        const uint32_t qx = col / w.ny;
        const int ix = w.XL + (int)qx, iy = w.YL + (int)(col - qx * w.ny);
        const float gxy = gap_box(w.ux0, w.ux1, ix) + gap_box(w.uy0, w.uy1, iy);
        if (gxy <= w.rc2) {
            const float zext = sqrtf(fmaxf(w.rc2 - gxy, 0.0f)) + 1e-2f;
            const int za = max(w.ZL, (int)floorf(w.uz0 - zext));
            const int zb = min(w.ZR, (int)floorf(w.uz1 + zext));
            // The union range spans less than M cells: at most two images.
            const int wrap = w.ZL < 0 ? 0 : M;
            int z0 = za, z1 = zb;
            if (w.halves == 2u) {
                if (k & 1u) z0 = max(za, wrap);
                else z1 = min(zb, wrap - 1);
            }
            if (z0 <= z1) {
                const uint32_t base =
                    ((uint32_t)wrap_index(ix, M) * M + wrap_index(iy, M)) * (uint32_t)M;
                const int zw = wrap_index(z0, M);
                js = off[base + zw];
                c = off[base + zw + (z1 - z0) + 1] - js;
                o.code = (uint32_t)(image_code(ix, M) | image_code(iy, M) << 2 |
                                    image_code(z0, M) << 4);
            }
        }
    }
    const uint64_t bal = __ballot(c > 0);
    o.nr = (uint32_t)__popcll(bal);
    o.end = incl_scan(c);
    o.total = (uint32_t)__builtin_amdgcn_readlane(o.end, 63);
    o.first = js - (o.end - c);
    const int to = c > 0 ? __popcll(bal & lt) : (int)o.nr + __popcll(~bal & lt);
    push(o.first, to);
    push(o.end, to);
    push(o.code, to);
}

constexpr uint32_t kInside = 0x15u;  // code of no image

// Image shifts of a code: -L, 0 or L (exact).
__device__ inline void code_shift(const PairParams &pp, uint32_t code, double &sx, double &sy,
                                  double &sz)
{
    sx = (double)((int)(code & 3u) - 1) * pp.L;
    sy = (double)((int)((code >> 2) & 3u) - 1) * pp.L;
    sz = (double)((int)((code >> 4) & 3u) - 1) * pp.L;
}

// A pair whose r^2 is within rounding of rcut^2 counts only when j's
// (unwrapped) cell lies in the target's own range, as in the reference loop.
__device__ inline bool in_range(const PairParams &pp, const Reach &t, const double4 &q,
                                uint32_t code)
{
    const int M = pp.M;
    const int x = cell_coord(pp.fac, q.x, M) + ((int)(code & 3u) - 1) * M;
    const int y = cell_coord(pp.fac, q.y, M) + ((int)((code >> 2) & 3u) - 1) * M;
    const int z = cell_coord(pp.fac, q.z, M) + ((int)((code >> 4) & 3u) - 1) * M;
    return x >= t.xl && x <= t.xr && y >= t.yl && y <= t.yr && z >= t.zl && z <= t.zr;
}

// rcut^2 less far more than the rounding of positions, cell edges and r^2.
__device__ inline double edge_r2(const PairParams &pp) { return pp.rcut2 * (1.0 - 1e-9); }

// Minimum image.  WRAP: the reference's per-pair tests.  Otherwise the
// caller passes the image shift of j's cell (sx, sy, sz: -L for a cell
// index below 0, +L above M-1, else 0): when rcut plus one cell stays below
// half the box (cell_images), a pair in an image cell is exactly one the
// tests would wrap and no other pair is, and dx + (-L) is the same IEEE
// operation as dx -= L (dx + 0.0 leaves dx unchanged), so the result is
// bit-identical.
// EDGE: the caller's walk holds pairs outside the target's own cell range;
// they lie beyond rcut up to rounding (in_range).
template <bool WRAP, bool EDGE>
__device__ inline void pair64(const PairParams &pp, const double *__restrict__ tab,
                              double px, double py, double pz, double4 q,
                              double sx, double sy, double sz,
                              double &ax, double &ay, double &az,
                              uint32_t &in_count, double edge2, const Reach *reach,
                              uint32_t code)
{
    double dx = q.x - px;
    double dy = q.y - py;
    double dz = q.z - pz;
    if (WRAP) {
        if (dx > pp.boxhalf) dx -= pp.L;
        if (dx < -pp.boxhalf) dx += pp.L;
        if (dy > pp.boxhalf) dy -= pp.L;
        if (dy < -pp.boxhalf) dy += pp.L;
        if (dz > pp.boxhalf) dz -= pp.L;
        if (dz < -pp.boxhalf) dz += pp.L;
    } else {
        dx += sx;
        dy += sy;
        dz += sz;
    }
    double r2 = dx * dx + dy * dy + dz * dz;
    if (r2 > pp.rcut2) return;
    if (EDGE && r2 > edge2 && !in_range(pp, *reach, q, code)) return;
    ++in_count;
    double hi;
    double r = sqrt_pair(r2, hi);
    double fac;
    if (r >= pp.h) {
        fac = over_cube(q.w, r2, r, hi);
    } else {
        if (r2 == 0.0) r = 0.0;
        double u = r * pp.h_inv;
        if (u < 0.5)
            fac = q.w * pp.h3_inv * (10.66667 + u * u * (32.0 * u - 38.4));
        else
            fac = q.w * pp.h3_inv *
                  (21.33333 - 48.0 * u + 38.4 * u * u - 10.66667 * u * u * u -
                   div_pair(0.06667, u * u * u));  // u >= 0.5
    }
    int tabindex = (int)(pp.asmthfac * r);
    if (tabindex < kNTab) {
        fac *= tab[tabindex];
        ax += dx * fac;
        ay += dy * fac;
        az += dz * fac;
    }
}

// Candidates of a target in its column (ix, iy): those of the z window.
__device__ inline uint32_t column_count(const Reach &t, int ix, int iy,
                                        const uint32_t *__restrict__ off, int M)
{
    const float gx = gap_cells(t.ux, ix);
    if (gx > t.rc2) return 0u;
    const float gxy = gx + gap_cells(t.uy, iy);
    if (gxy > t.rc2) return 0u;
    int za, zb;
    z_window(t.uz, gxy, t.rc2, t.zl, t.zr, za, zb);
    if (za > zb) return 0u;
    const uint32_t col = ((uint32_t)wrap_index(ix, M) * M + wrap_index(iy, M)) * (uint32_t)M;
    // [za, zb] wrapped: the span, or all of the column but a gap.
    const int a = wrap_index(za, M), b = wrap_index(zb, M);
    uint32_t c = off[col + b + 1] - off[col + a];
    if (a > b) c += off[col + M] - off[col];
    return c;
}

// ------------------------------------------------------------------ plan
// A box where no target has many candidates (plain_most64) is one whose walks
// all last about as long: one target per lane, in sorted order, takes it
// whole, and neither the order nor the split below is made.  k_target_keys
// decides that from one target of each wave.
//
// In the other boxes: which kernel takes which wave of 64 targets.  Targets
// are taken in the order of a Morton key two levels finer than the cells,
// those outside the active set behind the others: 64 of them then fill a box of
// few cells, or of a part of a cell in a halo core, whichever way the mesh
// runs, so that fewer of a wave's candidates are out of reach of its targets
// (sorted by cells alone, x-major, every third one was), and an active set
// fills its waves.  The sort is 60-150 us; 128^3 halo particles 48.0 -> 44.5
// ms, timeline steps of 64^3 6.8 -> 6.3.  The order decides only which targets share a wave; each
// target's sum keeps its own.
//
//  k_pp64       one target per lane.  Each lane's sum is one serial chain, so
//               a wave lasts as long as its busiest target however idle the
//               chip is, and lanes without a target (an active set) or with
//               few pairs wait for it.
//  the team     the same wave-uniform walk shared by the eight waves of a
//               workgroup: for dense waves that alone would outlast the
//               evaluation.
//  the list     one target per wave at a time, its candidates across the
//               lanes: even work whatever the counts, at a higher cost per
//               pair than a dense wave's, where a candidate is loaded once
//               for 64 targets.
//
// k_pp64_plan counts each target's candidates (the same columns and z
// windows the walks visit) and those of the wave-uniform walk, and takes the
// cheapest of three by modelled SIMD cycles: the uniform walk, the walk of
// each lane by itself, the list.  The wave sums of the cheapest give the
// evaluation's total; a walk whose serial chain would last longer than an
// eighth of the whole evaluation goes to a team (uniform) or to the list
// (per lane) instead.  Cycles measured on 1024 SIMDs at 2.1 GHz at 128^3 and
// 256^3 halo particles: the uniform walk and the team 5.4 per pair and lane
// (80 vector instructions, FP64 ones at 4 cycles), the per-lane walk 830 per
// candidate of the busiest lane, the list 11 per candidate and the
// enumeration of a target's columns.
constexpr uint32_t kUniformCycles = 345;  // per candidate of the wave
constexpr uint32_t kLaneCycles = 830;     // per candidate of the busiest lane
constexpr uint32_t kListPair = 11;        // per candidate
constexpr uint32_t kListTarget = 2500;    // per target
constexpr uint32_t kChainCycles = 2500;   // per candidate of a walk, wall time among 8 waves

// stats of a wave: candidates in its walk's serial chain, modelled cycles,
// the cheapest kind.
enum : uint32_t { kUniform = 0, kPerLane = 1, kList = 2, kTeam = 3 };

__device__ inline uint32_t wave_kind(const Plan64 &plan, uint32_t wave)
{
    const uint4 st = plan.stats[wave];
    const unsigned long long total = plan.total[0];
    const bool heavy = (unsigned long long)st.x * kChainCycles > total >> 13;  // 1024 SIMDs, an eighth
    const uint32_t k = !heavy ? st.z : st.z == kUniform ? (uint32_t)kTeam : (uint32_t)kList;
    return __builtin_amdgcn_readfirstlane(k);
}

// Whether the plan shares the box's targets.
__device__ inline bool shared_box(const Plan64 &plan)
{
    return !plan.split || __builtin_amdgcn_readfirstlane(plan.split[0]) != 0u;
}

// Sorted index of target number il of the box: the plan's order, or (without
// a plan) the sorted order itself.

__device__ inline uint32_t target_at(const Plan64 &plan, uint32_t i0, uint32_t n, uint32_t il)
{
    const uint32_t k = i0 + min(il, n - 1);
    return plan.order ? plan.order[k] : k;
}

__global__ __launch_bounds__(kThreads) void k_pp64_plan(
    const double4 *__restrict__ spos, const uint32_t *__restrict__ perm,
    const uint32_t *__restrict__ off, uint32_t i0, uint32_t n, PairParams pp,
    const int32_t *__restrict__ active_end, int32_t ti_current, Plan64 plan)
{
    if (!shared_box(plan)) return;
    const uint32_t il = blockIdx.x * kThreads + threadIdx.x;
    const uint32_t i = target_at(plan, i0, n, il);
    bool live = il < n;
    if (live && active_end && active_end[perm[i]] != ti_current) live = false;
    const double4 p = spos[i];
    live = live && in_box(pp, p);
    const int M = pp.M;
    const Reach t = reach_of(pp, p);
    const Union un = wave_union(t, live, M);
    uint32_t count = 0;
    if (live) {
        for (int ix = t.xl; ix <= t.xr; ++ix) {
            if (gap_cells(t.ux, ix) > t.rc2) continue;
            for (int iy = t.yl; iy <= t.yr; ++iy) count += column_count(t, ix, iy, off, M);
        }
    }
    unsigned long long sum = count;
    uint32_t most = count;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        sum += __shfl_xor(sum, o, 64);
        most = max(most, (uint32_t)__shfl_xor((int)most, o, 64));
    }
    const uint32_t nlive = (uint32_t)__popcll(__ballot(live));
    const unsigned long long lane_cost = (unsigned long long)most * kLaneCycles;
    const unsigned long long list_cost =
        sum * kListPair + (unsigned long long)nlive * kListTarget;
    unsigned long long best = min(lane_cost, list_cost);
    uint32_t kind = lane_cost <= list_cost ? (uint32_t)kPerLane : (uint32_t)kList, chain = most;
    // The uniform walk's candidates, counted until it is not the cheapest.
    if (un.any && un.fits) {
        const WalkBox wb = walk_box(t, un, live, M);
        unsigned long long cand = 0;
        for (uint32_t b = 0; b < wb.npieces && cand * kUniformCycles < best; b += 64) {
            Batch bt;
            walk_batch(wb, b, off, M, bt);
            cand += bt.total;
        }
        if (cand * kUniformCycles < best) {
            best = cand * kUniformCycles;
            kind = kUniform;
            chain = (uint32_t)cand;
        }
    }
    if ((threadIdx.x & 63) == 0 && il < n) {
        plan.stats[il >> 6] = make_uint4(chain, 0u, kind, 0u);
        if (nlive) atomicAdd(plan.total, best);
    }
}

// The work lists: live targets of the list's waves (a wave's stay together)
// and the team's waves.  Long ones are put at the front, the others at the
// back from the end down, and taken in that order, so that no long one
// starts last.  Otherwise the order does not matter to any result.
__device__ inline uint32_t list_slot(uint32_t at, uint32_t front, uint32_t size)
{
    return at < front ? at : size - 1u - (at - front);
}

__global__ __launch_bounds__(kThreads) void k_pp64_gather(
    const double4 *__restrict__ spos, const uint32_t *__restrict__ perm, uint32_t i0,
    uint32_t n, PairParams pp, const int32_t *__restrict__ active_end, int32_t ti_current,
    Plan64 plan)
{
    if (!shared_box(plan)) return;
    const uint32_t il = blockIdx.x * kThreads + threadIdx.x;
    if ((il & ~63u) >= n) return;
    const uint32_t wave = il >> 6, kind = wave_kind(plan, wave);
    if (kind != kTeam && kind != kList) return;
    const int lane = threadIdx.x & 63;
    // Long: a chain over twice what makes a walk heavy.
    const bool lng = (unsigned long long)plan.stats[wave].x * kChainCycles > plan.total[0] >> 12;
    if (kind == kTeam) {
        const uint32_t nwaves = (n + 63u) / 64u;
        if (lane == 0) {
            if (lng) plan.teams[atomicAdd(&plan.nteams[0], 1u)] = wave;
            else plan.teams[nwaves - 1u - atomicAdd(&plan.nteams[1], 1u)] = wave;
        }
        return;
    }
    const uint32_t i = target_at(plan, i0, n, il);
    bool live = il < n;
    if (live && active_end && active_end[perm[i]] != ti_current) live = false;
    live = live && in_box(pp, spos[i]);
    const uint64_t bal = __ballot(live);
    uint32_t at = 0;
    if (lane == 0 && bal) at = atomicAdd(&plan.nlist[lng ? 0 : 1], (uint32_t)__popcll(bal));
    at = __builtin_amdgcn_readfirstlane(at);
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    at += (uint32_t)__popcll(bal & lt);
    if (live) plan.list[lng ? at : n - 1u - at] = i;
}

// ------------------------------------------------------------------ terms
// pair64's term of kN candidates at once (independent chains), the same
// operations on the same values; a zero where has is false or the pair is
// outside the cut (adding a zero leaves a sum as it is: it starts at 0.0 and
// so is never -0.0).  (dx, dy, dz): the
// imaged separation in, the term out.  A pair above edge2 counts only where
// keep(its number) holds.
template <int kN, typename F>
__device__ inline void pair_terms(const PairParams &pp, const double *__restrict__ tab,
                                  const bool (&has)[kN], double (&dx)[kN], double (&dy)[kN],
                                  double (&dz)[kN], const double (&m)[kN], double edge2, F keep)
{
    double r[kN], fac[kN], r2[kN];
    bool in[kN], edge[kN], near = false, any_edge = false;
#pragma unroll
    for (int q = 0; q < kN; ++q) {
        r2[q] = dx[q] * dx[q] + dy[q] * dy[q] + dz[q] * dz[q];
        in[q] = has[q] && !(r2[q] > pp.rcut2);
        edge[q] = in[q] && r2[q] > edge2;
        any_edge |= edge[q];
        double hi;
        r[q] = sqrt_pair(r2[q], hi);
        fac[q] = over_cube(m[q], r2[q], r[q], hi);  // unused inside h
        near |= in[q] && !(r[q] >= pp.h);
    }
    if (__ballot(any_edge) != 0ull) {
#pragma unroll
        for (int q = 0; q < kN; ++q)
            if (edge[q]) in[q] = keep(q);
    }
    if (__ballot(near) != 0ull) {
#pragma unroll
        for (int q = 0; q < kN; ++q) {
            if (in[q] && !(r[q] >= pp.h)) {
                if (r2[q] == 0.0) r[q] = 0.0;
                const double u = r[q] * pp.h_inv;
                if (u < 0.5)
                    fac[q] = m[q] * pp.h3_inv * (10.66667 + u * u * (32.0 * u - 38.4));
                else
                    fac[q] = m[q] * pp.h3_inv *
                             (21.33333 - 48.0 * u + 38.4 * u * u - 10.66667 * u * u * u -
                              div_pair(0.06667, u * u * u));  // u >= 0.5
            }
        }
    }
#pragma unroll
    for (int q = 0; q < kN; ++q) {
        // r is NaN at r2 = 0 (the target itself, a slot without a candidate),
        // which fmin answers with the bound: in range for the conversion and
        // for the table, and outside the cut.
        const int tabindex = table_index64(pp.asmthfac * r[q]);
        const double t = fac[q] * tab[tabindex];
        const double f = in[q] && tabindex < kNTab ? t : 0.0;
        dx[q] *= f;
        dy[q] *= f;
        dz[q] *= f;
    }
}

// j's separation from the target, imaged.  Shifts of zero are left out when
// the whole wave has none: dx + 0.0 differs from dx only for dx = -0.0, and
// a term of either zero leaves a sum as it is.
template <bool WRAP>
__device__ inline void separation(const double4 &p, const double4 &q, const PairParams &pp,
                                  uint32_t code, double &dx, double &dy, double &dz)
{
    dx = q.x - p.x;
    dy = q.y - p.y;
    dz = q.z - p.z;
    if (WRAP) {
        if (dx > pp.boxhalf) dx -= pp.L;
        if (dx < -pp.boxhalf) dx += pp.L;
        if (dy > pp.boxhalf) dy -= pp.L;
        if (dy < -pp.boxhalf) dy += pp.L;
        if (dz > pp.boxhalf) dz -= pp.L;
        if (dz < -pp.boxhalf) dz += pp.L;
    } else if (__ballot(code != kInside) != 0ull) {
        double sx, sy, sz;
        code_shift(pp, code, sx, sy, sz);
        dx += sx;
        dy += sy;
        dz += sz;
    }
}

// ------------------------------------------------------------------ team
// A workgroup walks one wave's 64 targets (lane = target in every wave).
// The walk's candidates go through a filter first, kTeamList at a time: those
// further than rcut from the box around the targets (a quarter of a halo
// core's, the walk being whole cells) contribute nothing to any target and
// are left out, the others keep their order in LDS.  The waves take kTeamJ
// listed candidates a step, two each, and put the terms into one of two LDS
// buffers; after a barrier the first three waves add one component each, in
// candidate order, while the next candidates are computed into the other
// buffer.  The terms and the order of their additions are k_pp64's, so the
// bits are the same.
constexpr int kTeamWaves = 8;
constexpr int kTeamJ = 2 * kTeamWaves;
constexpr int kTeamWin = 2;                            // windows of 64 per wave and fill
constexpr int kTeamList = 64 * kTeamWaves * kTeamWin;

struct TeamShared {
    double term[2][kTeamJ][3][64];
    uint32_t j[kTeamList];
    uint8_t code[kTeamList];
    uint32_t count[kTeamWaves * kTeamWin];
    uint32_t item;
};

// Distance in cells, less the margin, of coordinate u from [u0, u1].
__device__ inline float gap_point(float u0, float u1, float u)
{
    return fmaxf(0.0f, fmaxf(u - u1, u0 - u) - 1e-2f);
}

// Candidates [c0, c0 + kTeamList) of a batch through the filter into the
// list; returns their number.  All waves of the workgroup.
template <bool WRAP>
__device__ inline uint32_t team_fill(TeamShared &sh, const WalkBox &w, const Batch &bt, uint32_t c0,
                                     const double4 *__restrict__ spos, const PairParams &pp, int wv)
{
    const int lane = threadIdx.x & 63;
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const float Mf = (float)pp.M;
    const uint32_t ends = (uint32_t)lane < bt.nr ? bt.end : 0xffffffffu;
    uint32_t j[kTeamWin], code[kTeamWin];
    uint64_t bal[kTeamWin];
#pragma unroll
    for (int v = 0; v < kTeamWin; ++v) {
        const uint32_t f = c0 + (uint32_t)((v * kTeamWaves + wv) * 64 + lane);
        bool ok = f < bt.total;
        // The piece of candidate f: the first that ends past it.
        int k = 0;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
            if ((uint32_t)__shfl((int)ends, k + o - 1, 64) <= f) k += o;
        k = min(k, 63);
        j[v] = (uint32_t)__shfl((int)bt.first, k, 64) + f;
        code[v] = (uint32_t)__shfl((int)bt.code, k, 64);
        // With the reference's per-pair image tests a pair's distance is not
        // that of its cell's image: no filter.
        if (!WRAP && ok) {
            const double4 q = spos[j[v]];
            const float x = (float)(pp.fac * q.x) + (float)((int)(code[v] & 3u) - 1) * Mf;
            const float y = (float)(pp.fac * q.y) + (float)((int)((code[v] >> 2) & 3u) - 1) * Mf;
            const float z = (float)(pp.fac * q.z) + (float)((int)((code[v] >> 4) & 3u) - 1) * Mf;
            const float gx = gap_point(w.ux0, w.ux1, x), gy = gap_point(w.uy0, w.uy1, y),
                        gz = gap_point(w.uz0, w.uz1, z);
            ok = gx * gx + gy * gy + gz * gz <= w.rc2;
        }
        bal[v] = __ballot(ok);
        if (lane == 0) sh.count[v * kTeamWaves + wv] = (uint32_t)__popcll(bal[v]);
    }
    __syncthreads();
    const uint32_t inc = incl_scan(lane < kTeamWaves * kTeamWin ? sh.count[lane] : 0u);
#pragma unroll
    for (int v = 0; v < kTeamWin; ++v) {
        const int win = v * kTeamWaves + wv;
        const uint32_t before =
            (uint32_t)__builtin_amdgcn_readlane(inc, win) - (uint32_t)__popcll(bal[v]);
        if ((bal[v] >> lane) & 1ull) {
            const uint32_t at = before + (uint32_t)__popcll(bal[v] & lt);
            sh.j[at] = j[v];
            sh.code[at] = (uint8_t)code[v];
        }
    }
    __syncthreads();
    return (uint32_t)__builtin_amdgcn_readlane(inc, 63);
}

template <bool WRAP>
__device__ inline void team_items(
    TeamShared &sh, const double *__restrict__ tab, const double4 *__restrict__ spos,
    const uint32_t *__restrict__ perm, const uint32_t *__restrict__ off, uint32_t i0, uint32_t n,
    const PairParams &pp, double4 *__restrict__ acc, const int32_t *__restrict__ active_end,
    int32_t ti_current, const Plan64 &plan)
{
    const uint32_t front = __builtin_amdgcn_readfirstlane(plan.nteams[0]);
    const uint32_t nteams = front + __builtin_amdgcn_readfirstlane(plan.nteams[1]);
    if (nteams == 0) return;
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int M = pp.M;
    const double edge2 = edge_r2(pp);
    for (;;) {
        if (threadIdx.x == 0) sh.item = atomicAdd(plan.team_work, 1u);
        __syncthreads();  // also: the buffers of the last item
        const uint32_t item = __builtin_amdgcn_readfirstlane(sh.item);
        __syncthreads();
        if (item >= nteams) break;
        const uint32_t il = plan.teams[list_slot(item, front, (n + 63u) / 64u)] * 64u + (uint32_t)lane;
        const uint32_t i = target_at(plan, i0, n, il);
        bool live = il < n;
        if (live && active_end && active_end[perm[i]] != ti_current) live = false;
        const double4 p = spos[i];
        live = live && in_box(pp, p);
        const Reach rch = reach_of(pp, p);
        const Union un = wave_union(rch, live, M);
        const WalkBox wb = walk_box(rch, un, live, M);
        double sum = 0.0;  // waves 0..2: one component each
        int buf = 0;
        for (uint32_t b = 0; b < wb.npieces; b += 64) {
            Batch bt;
            walk_batch(wb, b, off, M, bt);
            for (uint32_t c0 = 0; c0 < bt.total; c0 += (uint32_t)kTeamList) {
                const uint32_t nl = team_fill<WRAP>(sh, wb, bt, c0, spos, pp, wv);
                // This wave's two candidates of a step, loaded a step ahead
                // (a barrier each step would wait for the slowest load) into
                // scalar registers: the vector unit is the bound (scalar
                // loads 35.3 ms, vector loads 37.8, 128^3 halo particles).
                struct Pair {
                    double4 q[2];
                    uint32_t j[2], code[2];
                };
                auto fetch = [&](uint32_t f0, Pair &c) {
                    if (f0 >= nl) return;
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const uint32_t f = min(f0 + (uint32_t)u, nl - 1u);
                        c.j[u] = sh.j[f];
                        c.code[u] = sh.code[f];
                    }
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        c.j[u] = uni(c.j[u]);
                        c.code[u] = uni(c.code[u]);
                        c.q[u] = spos[c.j[u]];
                    }
                };
                auto step = [&](uint32_t fb, const Pair &c, Pair &next) {
                    const uint32_t f0 = fb + 2u * (uint32_t)wv;
                    fetch(f0 + kTeamJ, next);
                    if (f0 < nl) {
                        // A last odd candidate comes twice; only one is added.
                        bool has[2];
                        double dx[2], dy[2], dz[2], m[2];
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            has[u] = c.j[u] != i;
                            separation<WRAP>(p, c.q[u], pp, c.code[u], dx[u], dy[u], dz[u]);
                            m[u] = c.q[u].w;
                        }
                        pair_terms<2>(pp, tab, has, dx, dy, dz, m, edge2,
                                      [&](int u) { return in_range(pp, rch, c.q[u], c.code[u]); });
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            sh.term[buf][2 * wv + u][0][lane] = dx[u];
                            sh.term[buf][2 * wv + u][1][lane] = dy[u];
                            sh.term[buf][2 * wv + u][2][lane] = dz[u];
                        }
                    }
                    __syncthreads();
                    if (wv < 3) {
                        const int nj = (int)min((uint32_t)kTeamJ, nl - fb);
                        if (nj == kTeamJ) {
                            // All loads before the chain of additions.
                            double v[kTeamJ];
#pragma unroll
                            for (int j = 0; j < kTeamJ; ++j) v[j] = sh.term[buf][j][wv][lane];
                            asm volatile("" ::: "memory");
#pragma unroll
                            for (int j = 0; j < kTeamJ; ++j) sum += v[j];
                        } else {
                            for (int j = 0; j < nj; ++j) sum += sh.term[buf][j][wv][lane];
                        }
                    }
                    buf ^= 1;
                };
                Pair even, odd;
                fetch(2u * (uint32_t)wv, even);
                for (uint32_t fb = 0; fb < nl; fb += 2u * kTeamJ) {
                    step(fb, even, odd);
                    if (fb + kTeamJ < nl) step(fb + kTeamJ, odd, even);
                }
                __syncthreads();  // the list is read, the counts are free
            }
        }
        __syncthreads();
        if (wv < 3) sh.term[0][0][wv][lane] = sum;
        __syncthreads();
        if (wv == 0 && live)
            acc[perm[i]] = make_double4(sh.term[0][0][0][lane] * pp.G, sh.term[0][0][1][lane] * pp.G,
                                        sh.term[0][0][2][lane] * pp.G, 0.0);
    }
}

// ------------------------------------------------------------------ list
// One wave takes kGroup targets of the list at a time.  In a round, each
// unfinished target gets its next 64 candidates, one per lane: their pair
// terms (three doubles, 0.0 for a pair outside the cut -- adding it leaves
// a sum as it is) go to LDS, and then one lane per target and component
// adds its 64 terms in candidate order.  So a target's terms are added in
// the reference's order, one rounding each, as in k_pp64, and the bits are
// the same; only the terms are computed side by side.
//
// Candidates: the (ix, iy) columns of a target, in order, 64 column pieces a
// batch (a lane each; a z window that wraps is two pieces), the non-empty
// pieces compacted into LDS with the prefix of their lengths.  Candidate
// slot -> piece as in the FP32 kernel's staging: a window's piece starts are
// marked with one permute and counted below each lane.
constexpr int kGroup = 4;
constexpr int kListWaves = 8;
constexpr int kTermPitch = 66;  // even (16-byte reads), spreads the rows over the banks

struct ListWave {
    double term[kGroup * 3][kTermPitch];
    uint32_t start[kGroup][64];
    uint32_t pre[kGroup][64];   // slots before the piece
    uint8_t code[kGroup][64];   // image of the piece: 2 bits per axis (0 below, 1 inside, 2 above)
    // Per target: sorted index, next batch, batches, pieces and slots of the
    // current batch, first slot of the next window, piece holding it.
    uint32_t target[kGroup], batch[kGroup], pieces[kGroup], slots[kGroup], next[kGroup],
        piece[kGroup];
};

// Next non-empty batch of target t's column pieces; false when it has none.
__device__ inline bool next_batch(ListWave &w, int t, const double4 *__restrict__ spos,
                                  const uint32_t *__restrict__ off, const PairParams &pp)
{
    const int lane = threadIdx.x & 63;
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const int M = pp.M;
    const Reach r = reach_of(pp, spos[w.target[t]]);
    const uint32_t ny = (uint32_t)(r.yr - r.yl + 1);
    const uint32_t halves = r.zl < 0 || r.zr >= M ? 2u : 1u;
    const uint32_t pieces = uni((uint32_t)(r.xr - r.xl + 1) * ny * halves);
    uint32_t b = uni(w.batch[t]);
    while (b < pieces) {
        const uint32_t k = b + (uint32_t)lane;
        b += 64;
        uint32_t js = 0, c = 0, code = 0;
        if (k < pieces) {
            const uint32_t col = halves == 2u ? k >> 1 : k;
            const uint32_t qx = col / ny;
            const int ix = r.xl + (int)qx, iy = r.yl + (int)(col - qx * ny);
            const float gx = gap_cells(r.ux, ix);
            const float gxy = gx + gap_cells(r.uy, iy);
            if (gx <= r.rc2 && gxy <= r.rc2) {
                int za, zb;
                z_window(r.uz, gxy, r.rc2, r.zl, r.zr, za, zb);
                int z0, z1;
                window_part(za, zb, M, halves == 2u ? (int)(k & 1u) : 0, z0, z1);
                if (z0 <= z1) {
                    const uint32_t base =
                        ((uint32_t)wrap_index(ix, M) * M + wrap_index(iy, M)) * (uint32_t)M;
                    const int zw = wrap_index(z0, M);
                    js = off[base + zw];
                    c = off[base + zw + (z1 - z0) + 1] - js;
                    code = (uint32_t)(image_code(ix, M) | image_code(iy, M) << 2 |
                                      image_code(z0, M) << 4);
                }
            }
        }
        const uint64_t bal = __ballot(c > 0);
        if (bal == 0ull) continue;
        const uint32_t inc = incl_scan(c);
        if (c > 0) {
            const int at = __popcll(bal & lt);
            w.start[t][at] = js;
            w.pre[t][at] = inc - c;
            w.code[t][at] = (uint8_t)code;
        }
        if (lane == 0) {
            w.batch[t] = b;
            w.pieces[t] = (uint32_t)__popcll(bal);
            w.next[t] = 0;
            w.piece[t] = 0;
        }
        if (lane == 63) w.slots[t] = inc;
        wave_sync();
        return true;
    }
    if (lane == 0) {
        w.batch[t] = b;
        w.slots[t] = 0;
        w.next[t] = 0;
    }
    wave_sync();
    return false;
}

// Target t's next 64 candidates, one per lane: the separation (imaged) and
// mass of this lane's, and whether it has one other than the target itself.
template <bool WRAP>
__device__ inline bool next_candidate(ListWave &w, int t, const double4 *__restrict__ spos,
                                      const PairParams &pp, double &dx, double &dy, double &dz,
                                      double &m)
{
    const int lane = threadIdx.x & 63;
    const uint32_t f0 = uni(w.next[t]), rc = uni(w.piece[t]), nr = uni(w.pieces[t]);
    const uint32_t f = f0 + (uint32_t)lane;
    const bool ok = f < uni(w.slots[t]);
    const uint32_t i = uni(w.target[t]);
    // Pieces rc+1.. start at strictly increasing slots after f0.
    const uint32_t rn = rc + 1 + (uint32_t)lane;
    const uint32_t st = rn < nr ? w.pre[t][rn] - f0 : 0xffffffffu;
    const bool mark = st < 64u;
    const int got = __builtin_amdgcn_ds_permute(mark ? (int)(st * 4u) : 0, mark ? 1 : 0);
    const uint64_t starts = __ballot(got != 0);
    const uint32_t at = rc +
                        __builtin_amdgcn_mbcnt_hi((uint32_t)(starts >> 32),
                                                  __builtin_amdgcn_mbcnt_lo((uint32_t)starts, 0u)) +
                        (got != 0 ? 1u : 0u);
    const uint32_t past = (uint32_t)__popcll(__ballot(st <= 64u));
    const uint32_t j = ok ? w.start[t][at] + (f - w.pre[t][at]) : i;
    const uint32_t code = ok ? w.code[t][at] : kInside;
    const double4 p = spos[i], q = spos[j];
    wave_sync();  // every lane has read the cursor
    if (lane == 0) {
        w.next[t] = f0 + 64;
        w.piece[t] = rc + past;
    }
    wave_sync();
    separation<WRAP>(p, q, pp, code, dx, dy, dz);
    m = q.w;
    return ok && j != i;
}

template <bool WRAP>
__device__ inline void list_items(ListWave *s_w, const double *__restrict__ tab,
                                  const double4 *__restrict__ spos,
                                  const uint32_t *__restrict__ perm,
                                  const uint32_t *__restrict__ off, const PairParams &pp,
                                  double4 *__restrict__ acc, uint32_t n, const Plan64 &plan)
{
    const uint32_t front = uni(plan.nlist[0]);
    const uint32_t ntarget = front + uni(plan.nlist[1]);
    if (ntarget == 0) return;
    const int lane = threadIdx.x & 63;
    ListWave &w = s_w[threadIdx.x >> 6];
    for (;;) {
        // Every lane takes part in the atomic (lane 0 adds, the rest add 0).
        uint32_t g = atomicAdd(plan.list_work, lane == 0 ? (uint32_t)kGroup : 0u);
        g = __builtin_amdgcn_readlane(g, 0);
        if (g >= ntarget) break;
        const int nt = (int)min((uint32_t)kGroup, ntarget - g);
        if (lane < kGroup) {
            w.target[lane] = plan.list[list_slot(g + (uint32_t)min(lane, nt - 1), front, n)];
            w.batch[lane] = 0;
            w.slots[lane] = 0;
            w.next[lane] = 0;
        }
        wave_sync();
        uint32_t left = (1u << nt) - 1u;  // unfinished targets
        double sum = 0.0;                 // lane 3t + c: component c of target t
        while (uni(left)) {
            // The targets with candidates left, each with a window ready.
            for (int t = 0; t < nt; ++t) {
                if (!((left >> t) & 1u)) continue;
                if (uni(w.next[t]) >= uni(w.slots[t]) && !next_batch(w, t, spos, off, pp))
                    left &= ~(1u << t);
            }
            for (int t = 0; t < nt; t += 2) {
                const uint32_t two = (left >> t) & 3u;
                if (two == 0u) continue;
                bool has[2] = {false, false};
                double dx[2], dy[2], dz[2], m[2];
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    dx[q] = dy[q] = dz[q] = m[q] = 0.0;
                    if ((two >> q) & 1u)
                        has[q] = next_candidate<WRAP>(w, t + q, spos, pp, dx[q], dy[q], dz[q], m[q]);
                }
                // The pieces are the target's own windows: no pair to drop.
                pair_terms<2>(pp, tab, has, dx, dy, dz, m, pp.rcut2, [](int) { return true; });
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    if (t + q >= kGroup) break;
                    w.term[3 * (t + q)][lane] = dx[q];
                    w.term[3 * (t + q) + 1][lane] = dy[q];
                    w.term[3 * (t + q) + 2][lane] = dz[q];
                }
            }
            wave_sync();
            if (lane < 3 * kGroup && ((left >> (lane / 3)) & 1u)) {
                const double2 *row = reinterpret_cast<const double2 *>(w.term[lane]);
#pragma unroll 8
                for (int k = 0; k < 32; ++k) {
                    const double2 v = row[k];
                    sum += v.x;
                    sum += v.y;
                }
            }
            wave_sync();
        }
        const double y = __shfl_down(sum, 1, 64), z = __shfl_down(sum, 2, 64);
        if (lane < 3 * nt && lane % 3 == 0)
            acc[perm[w.target[lane / 3]]] = make_double4(sum * pp.G, y * pp.G, z * pp.G, 0.0);
        wave_sync();  // the targets have been read before the next group's
    }
}

// The team's items, then the list's, in one launch: the list's short items
// fill the chip while the last teams' serial sums end.  One launch each: 2.28
// ms where this takes 1.59 (100003 halo particles), 6.06 against 4.62
// (timeline steps of 64^3).  Sixteen waves a team with the CU to itself take
// 47.8 ms at 128^3 where eight take 40.3: two workgroups fill each other's
// barriers.
template <bool WRAP>
__global__ __launch_bounds__(64 * kTeamWaves, 4) void k_pp64_shared(
    const double4 *__restrict__ spos, const uint32_t *__restrict__ perm,
    const uint32_t *__restrict__ off, uint32_t i0, uint32_t n, PairParams pp,
    const float *__restrict__ table, double4 *__restrict__ acc,
    const int32_t *__restrict__ active_end, int32_t ti_current, Plan64 plan)
{
    static_assert(kTeamWaves == kListWaves, "one workgroup does both");
    __shared__ double tab[kNTab + 1];
    __shared__ union {
        TeamShared team;
        ListWave list[kListWaves];
    } sh;
    if (!shared_box(plan) ||
        uni(plan.nteams[0] + plan.nteams[1] + plan.nlist[0] + plan.nlist[1]) == 0u)
        return;
    for (int k = threadIdx.x; k <= kNTab; k += 64 * kTeamWaves)
        tab[k] = k < kNTab ? (double)table[k] : 0.0;
    __syncthreads();
    team_items<WRAP>(sh.team, tab, spos, perm, off, i0, n, pp, acc, active_end, ti_current, plan);
    // The last item of every workgroup ended on a barrier.
    list_items<WRAP>(sh.list, tab, spos, perm, off, pp, acc, n, plan);
}

// Eight waves per SIMD (at most 64 VGPRs, a few spilled): each lane's pair
// loop is a long dependent FP64 chain (correctly rounded sqrt and divide),
// so more resident waves hide more of it (441 ms at the register
// allocation's natural 5 waves, 400 ms at 8, halo256).
template <bool COUNT, bool WRAP>
__global__ __launch_bounds__(kThreads, 8) void k_pp64(
    const double4 *__restrict__ spos, const uint32_t *__restrict__ perm,
    const uint32_t *__restrict__ off, uint32_t i0, uint32_t n, PairParams pp,
    const float *__restrict__ table, double4 *__restrict__ acc,
    unsigned long long *__restrict__ counter,
    const int32_t *__restrict__ active_end, int32_t ti_current, Plan64 plan)
{
    __shared__ double tab[kNTab];
    for (int k = threadIdx.x; k < kNTab; k += kThreads) tab[k] = (double)table[k];
    __syncthreads();
    if (plan.stats && !shared_box(plan)) {
        plan.stats = nullptr;
        plan.order = nullptr;
    }
    const uint32_t il = blockIdx.x * kThreads + threadIdx.x;
    const uint32_t i = target_at(plan, i0, n, il);
    // Lanes past the end or outside the active set compute nothing but stay
    // for the wave-wide decisions below.
    bool live = il < n;
    if (live && active_end && active_end[perm[i]] != ti_current) live = false;

    const int M = pp.M;
    const double4 p = spos[i];
    if (live && !in_box(pp, p)) {
        // Positions are wrapped on upload and by every drift; anything else
        // is left without a short-range force rather than indexing wildly.
        acc[perm[i]] = make_double4(0.0, 0.0, 0.0, 0.0);
        live = false;
    }
    // Waves the plan gave to another kernel.
    uint32_t kind = kPerLane;
    if (plan.stats) {
        if ((il & ~63u) >= n) return;
        kind = wave_kind(plan, il >> 6);
        if (kind != kUniform && kind != kPerLane) return;
    }
    const Reach rch = reach_of(pp, p);
    const int xl = rch.xl, xr = rch.xr, yl = rch.yl, yr = rch.yr, zl = rch.zl, zr = rch.zr;
    const float ux = rch.ux, uy = rch.uy, uz = rch.uz, rc2 = rch.rc2;

    double ax = 0, ay = 0, az = 0;
    uint32_t in_count = 0;

    // Wave-uniform walk when the wave's targets are close together: the wave
    // visits the union of its lanes' windows in the reference order (ix, iy,
    // z ascending, unwrapped) with uniform loop bounds and uniform j loads,
    // and every lane takes only the j of its own window -- the pairs and
    // their order for each target are exactly those of the per-lane walk
    // below.
    const Union un = wave_union(rch, live, M);
    if (!un.any) return;  // no live lane
    if (plan.stats ? kind == kUniform : un.compact) {
        const WalkBox wb = walk_box(rch, un, live, M);
        const double edge2 = edge_r2(pp);
        for (uint32_t b = 0; b < wb.npieces; b += 64) {
            Batch bt;
            walk_batch(wb, b, off, M, bt);
            uint32_t f = 0;
            for (uint32_t k = 0; k < bt.nr; ++k) {
                const uint32_t first = __builtin_amdgcn_readlane(bt.first, k);
                const uint32_t end = __builtin_amdgcn_readlane(bt.end, k);
                const uint32_t code = __builtin_amdgcn_readlane(bt.code, k);
                double sx, sy, sz;
                code_shift(pp, code, sx, sy, sz);
                for (; f < end; ++f) {
                    const uint32_t j = first + f;
                    const double4 q = spos[j];
                    if (live && j != i)
                        pair64<WRAP, true>(pp, tab, p.x, p.y, p.z, q, sx, sy, sz, ax, ay, az,
                                           in_count, edge2, &rch, code);
                }
            }
        }
    } else if (live) {
        for (int ix = xl; ix <= xr; ++ix) {
            const float gx = gap_cells(ux, ix);
            if (gx > rc2) continue;
            const int iix = wrap_index(ix, M);
            const double sx = image_shift(ix, M, pp.L);
            for (int iy = yl; iy <= yr; ++iy) {
                const float gxy = gx + gap_cells(uy, iy);
                if (gxy > rc2) continue;
                const int iiy = wrap_index(iy, M);
                const double sy = image_shift(iy, M, pp.L);
                int za, zb;
                z_window(uz, gxy, rc2, zl, zr, za, zb);
                if (za > zb) continue;
                const uint32_t col = ((uint32_t)iix * M + iiy) * (uint32_t)M;
                // Up to two contiguous runs in reference order (wrapped part
                // first when the range starts below 0): z cells za..zb, the
                // second run starting at the wrap.
                for (int z0 = za; z0 <= zb;) {
                    const int zw = wrap_index(z0, M);
                    const int z1 = min(zb, z0 + (M - 1 - zw));  // last z before a wrap
                    const double sz = image_shift(z0, M, pp.L);
                    const uint32_t js = off[col + zw];
                    const uint32_t je = off[col + zw + (z1 - z0) + 1];
                    for (uint32_t j = js; j < je; ++j) {
                        if (j == i) continue;
                        pair64<WRAP, false>(pp, tab, p.x, p.y, p.z, spos[j], sx, sy, sz, ax,
                                            ay, az, in_count, 0.0, nullptr, 0u);
                    }
                    z0 = z1 + 1;
                }
            }
        }
    }
    if (!live) return;
    acc[perm[i]] = make_double4(ax * pp.G, ay * pp.G, az * pp.G, 0.0);
    if (COUNT) atomicAdd(counter, (unsigned long long)in_count);
}

}  // namespace

// One box: its sorted particles are [i0, i0+n) and off points at the cell
// table entry of the box's first key (entries are global sorted indices).
namespace {

// Also sets split of the boxes whose targets the plan is to share: of each
// wave of 64 sorted targets one has its candidates counted, and a wave with
// less than half of its targets active asks for the plan too.
__global__ __launch_bounds__(256) void k_target_keys(
    const double4 *__restrict__ spos, const uint32_t *__restrict__ perm,
    const uint32_t *__restrict__ off, BoxView v, const BoxDev *__restrict__ xmajor, int finer,
    const int32_t *__restrict__ active_end, int32_t ti_current, uint32_t *__restrict__ keys,
    uint32_t *__restrict__ split)
{
    int bi;
    uint32_t lb;
    if (!box_block(v, bi, lb)) return;
    const BoxDev &bx = v.box[bi];
    const uint32_t il = lb * blockDim.x + threadIdx.x;
    if ((il & ~63u) >= bx.n) return;
    const bool own = il < bx.n;
    const uint32_t i = bx.p0 + min(il, bx.n - 1u);
    const GridInfo &g = bx.g;
    const double4 p = spos[i];
    const bool active = own && (!active_end || active_end[perm[i]] == ti_current);
    const int lane = threadIdx.x & 63;
    const uint64_t act = __ballot(active);
    if (bx.plain_most != 0u && act != 0ull) {
        bool share = 2 * __popcll(act) < __popcll(__ballot(own));
        if (!share) {
            PairParams pp;
            pp.L = g.L;
            pp.M = g.M;
            pp.fac = g.fac;
            pp.rcut = bx.rcut;
            const int who = __ffsll((unsigned long long)act) - 1;
            double4 q;
            q.x = __shfl(p.x, who, 64);
            q.y = __shfl(p.y, who, 64);
            q.z = __shfl(p.z, who, 64);
            uint32_t count = 0;
            if (in_box(pp, q)) {
                const Reach t = reach_of(pp, q);
                const int ny = t.yr - t.yl + 1, cols = (t.xr - t.xl + 1) * ny;
                for (int k = lane; k < cols; k += 64)
                    count += column_count(t, t.xl + k / ny, t.yl + k % ny, off + xmajor[bi].key_base,
                                          g.M);
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) count += (uint32_t)__shfl_xor((int)count, o, 64);
            share = count > bx.plain_most;
        }
        if (share && lane == 0) split[bi] = split[v.nboxes] = 1u;
    }
    if (!own) return;
    // The key space of the box ends on its last key, which inactive targets
    // share with the far corner of a mesh of a power of two.
    uint32_t key = (g.nkeys << (3 * finer)) - 1u;
    if (active) {
        const int sub = 1 << finer;
        const double x[3] = {p.x, p.y, p.z};
        int c[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const int cell = cell_coord(g.fac, x[d], g.M);
            const int s = (int)((g.fac * x[d] - cell) * sub);
            c[d] = (cell << finer) | min(max(s, 0), sub - 1);
        }
        key = cell_key(g, c[0], c[1], c[2]);
    }
    keys[i] = (bx.key_base << (3 * finer)) + key;
}

}  // namespace

// Where every target of a box has about as many candidates as a uniform box
// would give it (u), the plain walk's serial chains are all alike and short,
// and no sort, plan or list pays once the box has the waves to fill the chip.
// Whole evaluation in us, by the plan -> by the plain walk:
//   u   n (lattice, or uniform at random)
//   17  32768 418 -> 307   262144 1407 -> 450   1000000 4605 -> 990
//  136  65536 516 -> 465    262144 1219 -> 632   1000000 3917 -> 1412
// 1085  131072 1200 -> 1250  262144 2033 -> 1313  1000000 6574 -> 3592
// They cross at n0 below (8000-12000, 50000-60000 and 150000-200000
// particles; 16000 of u = 34: 358 -> 309, 8000 of u = 17 at random 298 -> 317).  A wave whose lanes meet clumps in different columns waits for
// each, so the more the targets differ, the more waves it takes to make up
// for it (the largest count met: 300 of u = 136, 1.7 n0 particles: 670 by
// the plan, 970 by the walk; 4 n0: 1275 and 1003; 400, 15 n0: 4571 and 2446).
uint32_t plain_most64(const PairParams &pp, uint32_t n)
{
    const double reach = pp.rcut * pp.fac + 0.75;  // whole cells
    const double u = n / ((double)pp.M * pp.M * pp.M) * (4.0 * M_PI / 3.0) * reach * reach * reach;
    const double n0 = std::min(450.0 * u, 5500.0 * sqrt(u));
    if (n == 0 || n < n0) return 0u;
    return (uint32_t)std::min(u * std::min(1.25 + 0.35 * n / n0, 4.5) + 32.0, 1e9);
}

int order_targets64(const double4 *spos, const uint32_t *perm, const uint32_t *off,
                    const BoxSet &bs, uint32_t n,
                    int key_bits, int max_bits, const int32_t *active_end, int32_t ti_current,
                    uint32_t *scratch, const SortScratch &counters, uint32_t *split, bool always,
                    hipStream_t s, const uint32_t **order)
{
    // Two levels, or what 32 bits of key and 10 bits per coordinate leave.
    const int finer = std::max(0, std::min({2, (32 - key_bits) / 3, 10 - max_bits}));
    k_target_keys<<<xcd_grid(bs.total[kMapPart]), 256, 0, s>>>(
        spos, perm, off, bs.view(kKeyMorton, kMapPart), bs.dev[kKeyXMajor], finer, active_end,
        ti_current, scratch, split);
    CUCO_LAUNCH_CHECK();
    SortScratch sc = counters;
    sc.keys_tmp = scratch + n;
    sc.vals_tmp = scratch + 2 * (size_t)n;
    uint32_t *keys = nullptr, *vals = nullptr;
    const uint32_t *need = always ? nullptr : split + bs.nboxes;
    const int rc = radix_sort_pairs(scratch, scratch + 3 * (size_t)n, true, n,
                                    key_bits + 3 * finer, sc, s, &keys, &vals, need);
    *order = vals;
    return rc;
}

int launch_pp64(const double4 *spos, const uint32_t *perm, const uint32_t *off,
                uint32_t i0, uint32_t n, const PairParams &pp, const float *table,
                double4 *acc, unsigned long long *pair_counter,
                const int32_t *active_end, int32_t ti_current, const Plan64 &plan,
                int num_cu, hipStream_t s)
{
    if (n == 0) return CUCO_OK;
    // Cell-level image shifts are exact when a neighbour cell's pairs all
    // lie within rcut + one cell of the target, below half the box by a
    // margin far above rounding; otherwise the per-pair tests run.
    const bool cell_images = pp.rcut + 1.001 * (pp.L / pp.M) < pp.boxhalf;
    const unsigned grid = grid_for(n, kThreads);
    // Counting pairs is left to the one kernel that does.
    Plan64 pl = pair_counter ? Plan64{} : plan;
    if (pl.stats) {
        k_pp64_plan<<<grid, kThreads, 0, s>>>(spos, perm, off, i0, n, pp, active_end, ti_current, pl);
        CUCO_LAUNCH_CHECK();
        k_pp64_gather<<<grid, kThreads, 0, s>>>(spos, perm, i0, n, pp, active_end, ti_current, pl);
        CUCO_LAUNCH_CHECK();
    }
#define CUCO_PP64(COUNT, WRAP, CTR)                                                      \
    k_pp64<COUNT, WRAP><<<grid, kThreads, 0, s>>>(                                       \
        spos, perm, off, i0, n, pp, table, acc, CTR, active_end, ti_current, pl)
    if (pair_counter) {
        if (cell_images) CUCO_PP64(true, false, pair_counter);
        else CUCO_PP64(true, true, pair_counter);
    } else {
        if (cell_images) CUCO_PP64(false, false, nullptr);
        else CUCO_PP64(false, true, nullptr);
    }
#undef CUCO_PP64
    CUCO_LAUNCH_CHECK();
    if (pl.stats) {
        // Two workgroups of eight waves fill a CU (LDS and registers).
        const unsigned full = 2u * (unsigned)num_cu;
        const unsigned waves = (n + 63) / 64, groups = (n + kGroup - 1) / kGroup;
        const unsigned blocks =
            std::min(std::max(waves, (groups + kListWaves - 1) / kListWaves), full);
#define CUCO_SHARED(WRAP)                                                            \
    k_pp64_shared<WRAP><<<blocks, 64 * kTeamWaves, 0, s>>>(                          \
        spos, perm, off, i0, n, pp, table, acc, active_end, ti_current, pl)
        if (cell_images) CUCO_SHARED(false);
        else CUCO_SHARED(true);
#undef CUCO_SHARED
        CUCO_LAUNCH_CHECK();
    }
    return CUCO_OK;
}

}  // namespace cuco
