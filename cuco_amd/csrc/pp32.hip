// FP32 short-range pair force -- the chosen path.
//
// Same pair law as the reference (gravlist_kernel.cu:20-88 / gravlist.cpp:
// 279-327: minimum image via cell offsets, cut at rcut, spline softening
// inside h, erfc table), re-organised for CDNA4:
//
//  * Particles are sorted by a Morton cell key, so consecutive particles are
//    spatially compact at every density.  A tile is <= 64 consecutive
//    particles: a run of 64 inside one Morton block of 2^s cells per
//    dimension where blocks are dense, several neighbouring sparse blocks of
//    one 2^(s+1) super-block where they are not; one wavefront owns one
//    tile, one lane one target particle.
//  * Positions are FP32 relative to their cell corner (the subtraction is
//    done in FP64 by the reorder kernel).  A tile works in a frame anchored
//    at the corner of its first particle's cell: every coordinate is the
//    cell-relative value plus an integer number of cell sizes, so pair
//    separations are small numbers with small absolute error.
//  * For each tile the wave enumerates the cells within rcut of the tile's
//    bounding box (64 cells per step), reads their ranges from the CSR cell
//    table, and streams the j particles through a filter (distance to the
//    bounding box <= rcut) into an LDS buffer.  Each 64-entry buffer is
//    broadcast to all lanes and evaluated with the erfc table in LDS.
//  * Each lane sums a 64-j chunk in plain FP32 and adds the chunk sum into
//    its total with Kahan compensation.
//  * A persistent grid pulls tiles from an atomic work counter, so dense
//    halo tiles and void tiles balance across the chip.
#include <algorithm>
#include <cmath>

#include "internal.h"
#include "tile_parts.h"

namespace cuco {

namespace {

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kRanges = 128;   // cell ranges per wave before the j stream
constexpr int kJBuf = 128;     // staged j particles per wave
constexpr int kTab = 4096;     // LDS erfc table; zero from the cut bin on
constexpr int kTabSym = 2048;  // its copy in the each-pair-once kernel

__device__ inline float wave_min(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ inline float wave_max(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

// Wave-uniform copies in scalar registers.  Every loop bound and branch
// condition of the tile loop goes through these, so the compiler emits
// uniform (scalar) control flow: a lane-divergent view of an in-fact
// uniform loop exit lets it split the loop into per-lane nests around the
// cross-lane operations, which then read lanes that are not active.
__device__ inline uint32_t uni(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ inline int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ inline float uni(float v)
{
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

__device__ inline uint32_t wave_incl_scan(uint32_t v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}

// Scaled coordinate of a particle relative to its tile's anchor cell: the
// FP32 cell-relative coordinate p times s, plus dq cells.  Targets and
// staged candidates both come through here, as one explicit multiply-add
// (this file is compiled with contraction on, and the two sides written as
// separate expressions were once contracted differently): a target and its
// own copy among the candidates then have bit-identical coordinates, so
// the self pair's separation is exactly zero and its term vanishes.
__device__ inline float rel_coord(float p, int dq, float s, float cellf)
{
    return fmaf(p, s, (float)dq * cellf);
}

__device__ inline uint32_t pack_q(int qx, int qy, int qz)
{
    return ((uint32_t)(qx + 512) << 20) | ((uint32_t)(qy + 512) << 10) |
           (uint32_t)(qz + 512);
}

__device__ inline void unpack_q(uint32_t p, int &qx, int &qy, int &qz)
{
    qx = (int)(p >> 20) - 512;
    qy = (int)((p >> 10) & 1023u) - 512;
    qz = (int)(p & 1023u) - 512;
}

__device__ inline int unwrap_delta(int d, int M)
{
    if (d > M / 2) d -= M;
    if (d < -M / 2) d += M;
    return d;
}

// Newtonian-or-spline factor of one pair (gravlist_kernel.cu:47-56 with
// 1/u^3 = h^3 rinv^3); fac enters as m*rinv^3.
template <bool UNIFORM>
__device__ inline float spline_fac(float r, float fac, float mj, const P32 &pp)
{
    const float u = r * pp.h_inv;
    const float m = UNIFORM ? 1.0f : mj;
    const float lo = m * pp.h3_inv * (10.66667f + u * u * (32.0f * u - 38.4f));
    const float hi = m * pp.h3_inv *
                         (21.33333f - 48.0f * u + 38.4f * u * u - 10.66667f * u * u * u) -
                     0.06667f * fac;
    return r < pp.h ? (u < 0.5f ? lo : hi) : fac;
}

// Byte offset of a pair's table entry, bin floor(r / 4) (lengths are in
// quarter bins).  Far pairs (r >= 1): 2^23 - 0.5 + r, rounded to an
// integer by the multiply-add, is 2^23 + floor(r) (an exact integer r can
// round down by one: the lower bin of an edge), and its mantissa with the
// two low bits cleared is 4 floor(r / 4).  Near pairs, where r may be
// below 1, convert r itself.
__device__ inline uint32_t far_bin_bytes(float r2, float rinv)
{
    return __builtin_bit_cast(uint32_t, fmaf(r2, rinv, 8388607.5f)) & 0x7ffffcu;
}

__device__ inline uint32_t near_bin_bytes(float r) { return (uint32_t)(int)r & ~3u; }

__device__ inline float tab_at(const float *__restrict__ tab, uint32_t bytes)
{
    return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(tab) + bytes);
}

// Pair sum of one lane against cnt staged j particles.
//
// GENERIC=false is the reference configuration: rcut sits on a table bin
// edge (RCUT/ASMTH = 4.5 puts it on bin 750) so the table's zeros do the cut.
// GENERIC keeps the explicit r^2 <= rcut^2 mask and clamps the bin.  CLAMP:
// the tile is wide enough for a candidate to reach past the table (the
// caller's per-tile test), so the bin is clamped.  UNIFORM folds the common
// particle mass into the LDS table.
//
// Candidates go four at a time: the four chains (LDS reads, rsq, table
// lookup) are branch-free and interleave; the softened law is applied in
// one wave-level branch per group, taken only when some lane of the wave
// has a pair inside h.  NEAR=false: no staged j is within h of the tile's
// bounding box (chunk_near), so no pair can be and the test is left out.
template <bool GENERIC, bool UNIFORM, bool NEAR, bool CLAMP>
__device__ inline void interact(const float4 *__restrict__ sj, int cnt,
                                const P32 &pp, const float *__restrict__ tab,
                                float xi, float yi, float zi, float &sx,
                                float &sy, float &sz)
{
    int k = 0;
    for (; k + 4 <= cnt; k += 4) {
        float dx[4], dy[4], dz[4], r[4], fac[4], t[4], r2[4], mj[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 p = sj[k + q];
            dx[q] = p.x - xi;
            dy[q] = p.y - yi;
            dz[q] = p.z - zi;
            mj[q] = p.w;
            // Self and coincident pairs: dx = dy = dz = 0, eps keeps rsq
            // finite and the term is exactly zero (gravlist_kernel.cu:64-69).
            r2[q] = fmaf(dx[q], dx[q], fmaf(dy[q], dy[q], fmaf(dz[q], dz[q], pp.eps)));
            const float rinv = __builtin_amdgcn_rsqf(r2[q]);
            const float rinv3 = rinv * rinv * rinv;
            fac[q] = UNIFORM ? rinv3 : mj[q] * rinv3;
            uint32_t b;
            if (NEAR) {
                r[q] = r2[q] * rinv;
                b = near_bin_bytes(r[q]);
            } else {
                b = far_bin_bytes(r2[q], rinv);
            }
            if (GENERIC || CLAMP) b = min(b, 4u * (kTab - 1));
            t[q] = tab_at(tab, b);
        }
        if (NEAR) {
            const bool close = (r[0] < pp.h) | (r[1] < pp.h) | (r[2] < pp.h) | (r[3] < pp.h);
            if (close) {
#pragma unroll
                for (int q = 0; q < 4; ++q) fac[q] = spline_fac<UNIFORM>(r[q], fac[q], mj[q], pp);
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float tv = t[q];
            if (GENERIC) tv = r2[q] <= pp.rcut2 ? tv : 0.0f;
            const float f = fac[q] * tv;
            sx = fmaf(dx[q], f, sx);
            sy = fmaf(dy[q], f, sy);
            sz = fmaf(dz[q], f, sz);
        }
    }
    for (; k < cnt; ++k) {
        const float4 p = sj[k];
        const float dx = p.x - xi, dy = p.y - yi, dz = p.z - zi;
        const float r2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, pp.eps)));
        const float rinv = __builtin_amdgcn_rsqf(r2);
        const float r = r2 * rinv;
        const float rinv3 = rinv * rinv * rinv;
        float fac = UNIFORM ? rinv3 : p.w * rinv3;
        if (NEAR) fac = spline_fac<UNIFORM>(r, fac, p.w, pp);
        uint32_t b = NEAR ? near_bin_bytes(r) : far_bin_bytes(r2, rinv);
        if (GENERIC || CLAMP) b = min(b, 4u * (kTab - 1));
        float tv = tab_at(tab, b);
        if (GENERIC) tv = r2 <= pp.rcut2 ? tv : 0.0f;
        const float f = fac * tv;
        sx = fmaf(dx, f, sx);
        sy = fmaf(dy, f, sy);
        sz = fmaf(dz, f, sz);
    }
}

__device__ inline void kahan_add(float &sum, float &comp, float v)
{
    const float y = v - comp;
    const float t = sum + y;
    comp = (t - sum) - y;
    sum = t;
}

// ---------------------------------------------------------------------------
// Each pair once (Newton's third law).  A tile takes only the j with a larger
// sorted index than its first particle, and inside the tile only j > i; the
// force on j is minus the pair term, summed over the wave's lanes as it travels with j (DPP)
// and added to j's total in 64-bit fixed point (an integer sum, so the result
// does not depend on the order in which tiles run).

// The j side rides along with j: at step s lane L evaluates the pair with
// staged j number (L + s) mod 64 and subtracts the pair term from its
// accumulator, which then moves one lane down (lane L takes lane L+1's), so
// the accumulator of j is always in the lane that meets j next; after 64
// steps lane L holds the j-side sum of staged j number L.  The move is a
// DPP wave rotation (one full-rate vector instruction per component); a
// backward permute through the LDS crossbar instead takes those three
// instructions off the vector ALU but chains every step on the LDS round
// trip, and measured 70.5 against 47.9 ms at halo256.
__device__ inline float rotate_down(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x134, 0xF, 0xF, false));
}

// Pair sums of one lane against the 64 staged j.  GEN: rcut is not on a
// table bin edge, so pairs past it are masked by r^2 and the bin clamped;
// otherwise the table's zero tail makes the cut.  UNI: the common particle
// mass is folded into the table; otherwise the target side takes j's mass
// (the staged w) and the j side the target's (mi).  With MASKED a pair counts only when j's
// sorted index exceeds i's (iid = 0xffffffff for lanes without a target;
// unused slots carry index 0 and a position inside the tile).
// rot / rotid hold the 64 staged j twice (slots 64..127 repeat 0..63), so
// lane L reads slot L + s with no wrap.
template <bool GEN, bool UNI, bool MASKED, bool NEAR, bool CLAMP>
__device__ inline void interact_sym(const float4 *__restrict__ rot,
                                    const uint32_t *__restrict__ rotid,
                                    const P32 &pp, const float *__restrict__ tab,
                                    float xi, float yi, float zi, float mi, uint32_t iid,
                                    float &sx, float &sy, float &sz, float &jx,
                                    float &jy, float &jz)
{
    const int lane = threadIdx.x & 63;
    const float4 *rl = rot + lane;
    const uint32_t *il = rotid + lane;
    auto group = [&](int s) {
        float dx[4], dy[4], dz[4], r[4], fac[4], t[4], mj[4];
        bool keep[4], inside[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 p = rl[s + q];
            mj[q] = p.w;
            if (MASKED) keep[q] = il[s + q] > iid;
            dx[q] = p.x - xi;
            dy[q] = p.y - yi;
            dz[q] = p.z - zi;
            const float r2 = fmaf(dx[q], dx[q], fmaf(dy[q], dy[q], fmaf(dz[q], dz[q], pp.eps)));
            const float rinv = __builtin_amdgcn_rsqf(r2);
            fac[q] = rinv * rinv * rinv;
            if (GEN) inside[q] = r2 <= pp.rcut2;
            // The table's zero tail from the cut bin on.  CLAMP: bins past
            // the LDS copy read its last (zero) entry; without it the tile's
            // extent keeps every bin inside (the per-tile clamp test).
            uint32_t b;
            if (NEAR) {
                r[q] = r2 * rinv;
                b = near_bin_bytes(r[q]);
            } else {
                b = far_bin_bytes(r2, rinv);
            }
            if (CLAMP || GEN) b = min(b, 4u * (kTabSym - 1));
            t[q] = tab_at(tab, b);
        }
        if (NEAR) {
            const bool close = (r[0] < pp.h) | (r[1] < pp.h) | (r[2] < pp.h) | (r[3] < pp.h);
            if (close) {
#pragma unroll
                for (int q = 0; q < 4; ++q) fac[q] = spline_fac<true>(r[q], fac[q], 1.0f, pp);
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float f = fac[q] * t[q];
            if (MASKED) f = keep[q] ? f : 0.0f;
            if (GEN) f = inside[q] ? f : 0.0f;
            const float fi = UNI ? f : f * mj[q];
            const float fj = UNI ? f : f * mi;
            sx = fmaf(dx[q], fi, sx);
            sy = fmaf(dy[q], fi, sy);
            sz = fmaf(dz[q], fi, sz);
            jx = rotate_down(fmaf(-dx[q], fj, jx));
            jy = rotate_down(fmaf(-dy[q], fj, jy));
            jz = rotate_down(fmaf(-dz[q], fj, jz));
        }
    };
    // The common case (no masks, far, no clamp) is unrolled whole: the LDS
    // reads then take their offsets from the instruction and the loop keeps
    // no counter (1-3% at halo256).
    if (!MASKED && !NEAR && !CLAMP) {
#pragma unroll
        for (int s = 0; s < 64; s += 4) group(s);
    } else {
        for (int s = 0; s < 64; s += 4) group(s);
    }
}

// Two targets per lane (a tile of up to 128): at each step the staged j
// meets both, its position and index are read once, and the j-side sum
// takes both terms before the one rotation -- 20.5 vector instructions per
// pair slot instead of 22.  Same masks and laws as interact_sym.
template <bool GEN, bool UNI, bool MASKED, bool NEAR, bool CLAMP>
__device__ inline void interact_sym2(const float4 *__restrict__ rot,
                                     const uint32_t *__restrict__ rotid, const P32 &pp,
                                     const float *__restrict__ tab, float xa, float ya, float za,
                                     float ma, uint32_t iida, float xb, float yb, float zb,
                                     float mb, uint32_t iidb, float &sxa, float &sya,
                                     float &sza, float &sxb, float &syb, float &szb,
                                     float &jx, float &jy, float &jz)
{
    const int lane = threadIdx.x & 63;
    const float4 *rl = rot + lane;
    const uint32_t *il = rotid + lane;
    auto group = [&](int s) {
        float dxa[2], dya[2], dza[2], ra[2], fa[2], ta[2];
        float dxb[2], dyb[2], dzb[2], rb[2], fb[2], tb[2], mj[2];
        bool keepa[2], keepb[2], ina[2], inb[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const float4 p = rl[s + q];
            mj[q] = p.w;
            if (MASKED) {
                const uint32_t id = il[s + q];
                keepa[q] = id > iida;
                keepb[q] = id > iidb;
            }
            dxa[q] = p.x - xa;
            dya[q] = p.y - ya;
            dza[q] = p.z - za;
            dxb[q] = p.x - xb;
            dyb[q] = p.y - yb;
            dzb[q] = p.z - zb;
            const float r2a = fmaf(dxa[q], dxa[q], fmaf(dya[q], dya[q], fmaf(dza[q], dza[q], pp.eps)));
            const float r2b = fmaf(dxb[q], dxb[q], fmaf(dyb[q], dyb[q], fmaf(dzb[q], dzb[q], pp.eps)));
            const float rinva = __builtin_amdgcn_rsqf(r2a);
            const float rinvb = __builtin_amdgcn_rsqf(r2b);
            fa[q] = rinva * rinva * rinva;
            fb[q] = rinvb * rinvb * rinvb;
            if (GEN) {
                ina[q] = r2a <= pp.rcut2;
                inb[q] = r2b <= pp.rcut2;
            }
            uint32_t ba, bb;
            if (NEAR) {
                ra[q] = r2a * rinva;
                rb[q] = r2b * rinvb;
                ba = near_bin_bytes(ra[q]);
                bb = near_bin_bytes(rb[q]);
            } else {
                ba = far_bin_bytes(r2a, rinva);
                bb = far_bin_bytes(r2b, rinvb);
            }
            if (CLAMP || GEN) {
                ba = min(ba, 4u * (kTabSym - 1));
                bb = min(bb, 4u * (kTabSym - 1));
            }
            ta[q] = tab_at(tab, ba);
            tb[q] = tab_at(tab, bb);
        }
        if (NEAR) {
            const bool close = (ra[0] < pp.h) | (ra[1] < pp.h) | (rb[0] < pp.h) | (rb[1] < pp.h);
            if (close) {
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    fa[q] = spline_fac<true>(ra[q], fa[q], 1.0f, pp);
                    fb[q] = spline_fac<true>(rb[q], fb[q], 1.0f, pp);
                }
            }
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            float f1 = fa[q] * ta[q], f2 = fb[q] * tb[q];
            if (MASKED) {
                f1 = keepa[q] ? f1 : 0.0f;
                f2 = keepb[q] ? f2 : 0.0f;
            }
            if (GEN) {
                f1 = ina[q] ? f1 : 0.0f;
                f2 = inb[q] ? f2 : 0.0f;
            }
            const float fia = UNI ? f1 : f1 * mj[q], fja = UNI ? f1 : f1 * ma;
            const float fib = UNI ? f2 : f2 * mj[q], fjb = UNI ? f2 : f2 * mb;
            sxa = fmaf(dxa[q], fia, sxa);
            sya = fmaf(dya[q], fia, sya);
            sza = fmaf(dza[q], fia, sza);
            sxb = fmaf(dxb[q], fib, sxb);
            syb = fmaf(dyb[q], fib, syb);
            szb = fmaf(dzb[q], fib, szb);
            jx = rotate_down(fmaf(-dxb[q], fjb, fmaf(-dxa[q], fja, jx)));
            jy = rotate_down(fmaf(-dyb[q], fjb, fmaf(-dya[q], fja, jy)));
            jz = rotate_down(fmaf(-dzb[q], fjb, fmaf(-dza[q], fja, jz)));
        }
    };
    if (!MASKED && !NEAR && !CLAMP) {
#pragma unroll
        for (int s = 0; s < 64; s += 2) group(s);
    } else {
        for (int s = 0; s < 64; s += 2) group(s);
    }
}

// True when some staged j (lanes with in set) lies within h of the tile's
// bounding box; otherwise every pair of the chunk has r >= h and takes the
// plain law.  Called with h = max(softening, 1 quarter bin), so a far
// chunk's pairs also have r >= 1, which far_bin_bytes needs.  Wave-uniform.
__device__ inline bool chunk_near(float4 q, bool in, float bminx, float bminy, float bminz,
                                  float bmaxx, float bmaxy, float bmaxz, float h)
{
    const float gx = fmaxf(0.f, fmaxf(bminx - q.x, q.x - bmaxx));
    const float gy = fmaxf(0.f, fmaxf(bminy - q.y, q.y - bmaxy));
    const float gz = fmaxf(0.f, fmaxf(bminz - q.z, q.z - bmaxz));
    const bool near = in && gx * gx + gy * gy + gz * gz < h * h;
    return __builtin_amdgcn_readfirstlane((uint32_t)(__ballot(near) != 0ull)) != 0u;
}

// The box around a tile's targets (scaled, in the tile's frame).
struct TileBox {
    float minx, miny, minz, maxx, maxy, maxz;
};

// Units of cells that can hold a candidate of the tile.
struct TileUnits {
    int ux0, uy0, uz0, nux, nuy, nuz;  // first one (absolute, unwrapped), and how many
    uint32_t total;
    bool coarse;
};

__device__ inline TileUnits tile_units(const TileBox &b, const P32 &pp, int c0x, int c0y, int c0z,
                                       float coarse_cells)
{
    TileUnits t;
    const int M = pp.M;
    const int lqx = (int)floorf((b.minx - pp.rcut) * pp.inv_cellf - 0.01f);
    const int lqy = (int)floorf((b.miny - pp.rcut) * pp.inv_cellf - 0.01f);
    const int lqz = (int)floorf((b.minz - pp.rcut) * pp.inv_cellf - 0.01f);
    const int nqx = (int)floorf((b.maxx + pp.rcut) * pp.inv_cellf + 0.01f) - lqx + 1;
    const int nqy = (int)floorf((b.maxy + pp.rcut) * pp.inv_cellf + 0.01f) - lqy + 1;
    const int nqz = (int)floorf((b.maxz + pp.rcut) * pp.inv_cellf + 0.01f) - lqz + 1;
    // A tile spans at most one Morton super-block plus the cut on each
    // side; anything larger means non-finite input and the tile is
    // skipped.
    const bool sane = nqx > 0 && nqy > 0 && nqz > 0 && nqx <= 2 * M &&
                      nqy <= 2 * M && nqz <= 2 * M;
    // Enumeration unit: one cell, or for a wide tile (a merge of sparse
    // blocks) an aligned 2x2x2-cell Morton block, whose cells form one
    // contiguous key range: eight times fewer units to test, and the
    // staging takes each candidate's cell from the low bits of its key.
    // Blocks need an even mesh (they wrap onto blocks) and a reach of at
    // most M cells per axis; coarse_cells is the tile extent (in cells)
    // from which they are used (both variants).
    const float ext = fmaxf(b.maxx - b.minx, fmaxf(b.maxy - b.miny, b.maxz - b.minz));
    t.coarse = uni((uint32_t)(sane && (M & 1) == 0 && nqx <= M && nqy <= M && nqz <= M &&
                              ext >= coarse_cells * pp.cellf)) != 0u;
    const int lv = t.coarse ? 1 : 0;
    // Units (absolute, unwrapped) covering cells c0 + lq .. c0 + lq + nq - 1.
    t.ux0 = (c0x + lqx) >> lv;
    t.uy0 = (c0y + lqy) >> lv;
    t.uz0 = (c0z + lqz) >> lv;
    t.nux = ((c0x + lqx + nqx - 1) >> lv) - t.ux0 + 1;
    t.nuy = ((c0y + lqy + nqy - 1) >> lv) - t.uy0 + 1;
    t.nuz = ((c0z + lqz + nqz - 1) >> lv) - t.uz0 + 1;
    t.total = uni(sane ? (uint32_t)t.nux * t.nuy * t.nuz : 0u);
    return t;
}

// Every candidate lies within sqrt(filter2) of the tile's box, so a
// pair's distance is at most that plus the box diagonal; below the
// last bin of the LDS table (with margin for rounding) the bin needs
// no clamp.
template <int kT>
__device__ inline bool tile_clamps(const TileBox &b, const P32 &pp)
{
    const float ex = b.maxx - b.minx, ey = b.maxy - b.miny, ez = b.maxz - b.minz;
    return !(sqrtf(ex * ex + ey * ey + ez * ez) + sqrtf(pp.filter2) + 1.0f < 4.0f * (kT - 2));
}

// A tile's count word: targets (bits 0-7), parts less one (8-17), and
// kListed when the list of parts holds it (k_fill_tiles).
constexpr uint32_t kListed = 1u << 18;

// Tiles of all boxes form one work list; tv.map holds each box's first
// tile, p32s[b] the scaled constants of box b.
// SYM: each pair once (section above); the tile's own sums go to iacc
// (sorted order, unscaled) and the j side to jacc (three 64-bit fixed-point
// planes of n_sorted entries); a second kernel combines them.
// TPL = 2 (each pair once only): a tile holds up to 128 targets, lane L
// targets L and 64 + L.
template <bool GENERIC, bool UNIFORM, bool SYM, int TPL>
__global__ __launch_bounds__(kThreads, SYM ? (TPL == 2 ? 4 : 5) : 1) void k_pp32(
    const float4 *__restrict__ spos, const uint32_t *__restrict__ skeys,
    const uint32_t *__restrict__ perm, const uint32_t *__restrict__ off,
    BoxView tv, const P32 *__restrict__ p32s, float mass,
    const float *__restrict__ table32,
    const uint32_t *__restrict__ tstart, const uint32_t *__restrict__ tcount,
    uint32_t *__restrict__ counters, float4 *__restrict__ acc,
    unsigned long long *__restrict__ cand,
    const int32_t *__restrict__ active_end, int32_t ti_current,
    float4 *__restrict__ iacc, unsigned long long *__restrict__ jacc,
    uint32_t n_sorted, const uint32_t *__restrict__ tlist, float coarse_cells,
    const uint2 *__restrict__ parts, uint32_t max_parts)
{
    // SYM trades half of the range list for the doubled rotation buffer.
    constexpr int kR = SYM ? kRanges / 2 : kRanges;
    constexpr int kT = SYM ? kTabSym : kTab;
    __shared__ float s_tab[kT];
    __shared__ uint32_t s_rs[kWaves][kR];
    __shared__ uint32_t s_rp[kWaves][kR + 1];
    __shared__ uint32_t s_rq[kWaves][kR];
    __shared__ float4 s_j[kWaves][kJBuf];
    __shared__ uint32_t s_jid[kWaves][SYM ? kJBuf : 1];
    __shared__ float4 s_rot[kWaves][SYM ? 128 : 1];
    __shared__ uint32_t s_rotid[kWaves][SYM ? 128 : 1];

    for (int k = threadIdx.x; k < kT; k += kThreads)
        s_tab[k] = k < kTabPadded ? (UNIFORM ? mass * table32[k] : table32[k]) : 0.0f;
    __syncthreads();

    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t *rs = s_rs[w];
    uint32_t *rp = s_rp[w];
    uint32_t *rq = s_rq[w];
    float4 *sj = s_j[w];
    uint32_t *sjid = s_jid[w];
    float4 *rot = s_rot[w];
    uint32_t *rotid = s_rotid[w];
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    // Work items: the parts of long tiles, the tiles of middling length
    // (from the end of the list down), then the other tiles.
    const uint32_t nparts = SYM ? min(counters[2], max_parts) : 0u;
    const uint32_t nmid = SYM ? min(counters[3], max_parts - nparts) : 0u;
    const uint32_t nlisted = uni(nparts + nmid), nitems = uni(nlisted + counters[0]);
    const float inf = __builtin_huge_valf();

    for (;;) {
        // Every lane takes part in the atomic (lane 0 adds 1, the rest 0), so
        // the loop header carries no lane-divergent branch; lane 0's return
        // value is the item whatever order the adds are applied in.  An item
        // is drawn when it can be started: one drawn ahead, or given to a
        // workgroup by its number, waits behind what the wave or the CU is
        // at (8.9 instead of 8.0 ms at 128^3 halo particles).
        uint32_t item = atomicAdd(&counters[1], lane == 0 ? 1u : 0u);
        item = __builtin_amdgcn_readlane(item, 0);
        if (item >= nitems) break;
        uint32_t t = item - nlisted, part = 0;
        if (SYM && item < nlisted) {
            const uint2 pt = parts[item < nparts ? item : max_parts - 1u - (item - nparts)];
            t = uni(pt.x);
            part = uni(pt.y);
        }
        // Targets, parts less one, and whether the list has the tile.
        const uint32_t word = uni(tcount[t]);
        if (SYM && item >= nlisted && (word & kListed)) continue;

        const int bi = find_box(tv.map, tv.nboxes, t);
        const P32 pp = p32s[bi];
        const GridInfo &g = tv.box[bi].g;
        const uint32_t key_base = tv.box[bi].key_base;
        const int M = pp.M;
        const uint32_t i0 = tstart[t];
        const uint32_t cnt = word & 255u, nsplit = ((word >> 8) & (kPartMost - 1u)) + 1u;
        const bool valid = (uint32_t)lane < cnt;
        // tlist: the tile is a run of the active-target list (ia: its first
        // target, the anchor); else a run of the sorted particles.
        const uint32_t ia = tlist ? tlist[i0] : i0;
        const uint32_t i = tlist ? tlist[i0 + (valid ? (uint32_t)lane : 0u)]
                                 : i0 + (valid ? (uint32_t)lane : 0u);
        // Active set: a tile without an active target is skipped; in the
        // others every lane computes and only active lanes store.
        bool act = valid;
        if (active_end) act = valid && active_end[perm[i]] == ti_current;
        if (uni((uint32_t)(__ballot(act) != 0ull)) == 0u) continue;

        int c0x, c0y, c0z, cx, cy, cz;
        key_cell(g, skeys[ia] - key_base, c0x, c0y, c0z);
        key_cell(g, skeys[i] - key_base, cx, cy, cz);
        const float4 pi = spos[i];
        const float xi = rel_coord(pi.x, unwrap_delta(cx - c0x, M), pp.s, pp.cellf);
        const float yi = rel_coord(pi.y, unwrap_delta(cy - c0y, M), pp.s, pp.cellf);
        const float zi = rel_coord(pi.z, unwrap_delta(cz - c0z, M), pp.s, pp.cellf);
        // The lane's second target (TPL = 2): 64 + L of the tile.
        const bool valid2 = TPL == 2 && (uint32_t)lane + 64u < cnt;
        const uint32_t i2 = valid2 ? i0 + 64u + (uint32_t)lane : i;
        float xi2 = xi, yi2 = yi, zi2 = zi, mi2 = pi.w;
        if (TPL == 2) {
            int cx2, cy2, cz2;
            key_cell(g, skeys[i2] - key_base, cx2, cy2, cz2);
            const float4 p2 = spos[i2];
            xi2 = rel_coord(p2.x, unwrap_delta(cx2 - c0x, M), pp.s, pp.cellf);
            yi2 = rel_coord(p2.y, unwrap_delta(cy2 - c0y, M), pp.s, pp.cellf);
            zi2 = rel_coord(p2.z, unwrap_delta(cz2 - c0z, M), pp.s, pp.cellf);
            mi2 = p2.w;
        }

        const float bminx = uni(wave_min(fminf(valid ? xi : inf, valid2 ? xi2 : inf)));
        const float bminy = uni(wave_min(fminf(valid ? yi : inf, valid2 ? yi2 : inf)));
        const float bminz = uni(wave_min(fminf(valid ? zi : inf, valid2 ? zi2 : inf)));
        const float bmaxx = uni(wave_max(fmaxf(valid ? xi : -inf, valid2 ? xi2 : -inf)));
        const float bmaxy = uni(wave_max(fmaxf(valid ? yi : -inf, valid2 ? yi2 : -inf)));
        const float bmaxz = uni(wave_max(fmaxf(valid ? zi : -inf, valid2 ? zi2 : -inf)));

        const TileBox box{bminx, bminy, bminz, bmaxx, bmaxy, bmaxz};
        const TileUnits tu = tile_units(box, pp, c0x, c0y, c0z, coarse_cells);
        const bool coarse = tu.coarse;
        const int lv = coarse ? 1 : 0;
        const int ux0 = tu.ux0, uy0 = tu.uy0, uz0 = tu.uz0;
        const int nux = tu.nux, nuy = tu.nuy, nuz = tu.nuz;
        const uint32_t total_q = tu.total;

        float ax = 0.f, ay = 0.f, az = 0.f, kx = 0.f, ky = 0.f, kz = 0.f;
        float ax2 = 0.f, ay2 = 0.f, az2 = 0.f, kx2 = 0.f, ky2 = 0.f, kz2 = 0.f;
        const bool clamp = tile_clamps<kT>(box, pp);
        // SYM: the j side of one staged chunk, added to jacc (fixed point).
        const uint32_t iid = valid ? i : 0xffffffffu;
        const uint32_t iid2 = valid2 ? i2 : 0xffffffffu;
        auto eval_sym = [&](int nj, float &sx_, float &sy_, float &sz_, float &sx2_, float &sy2_,
                            float &sz2_) {
            float jx = 0.f, jy = 0.f, jz = 0.f;
            // Copy the chunk twice into the rotation buffer; unused slots of a
            // partial chunk get index 0 (always masked) and a position one
            // quarter bin below the tile's box (a bounded far-pair bin).
            float4 mine = make_float4(bminx - 1.0f, bminy, bminz, 0.f);
            uint32_t mid = 0u;
            if (lane < nj) {
                mine = sj[lane];
                mid = sjid[lane];
            }
            rot[lane] = mine;
            rot[lane + 64] = mine;
            rotid[lane] = mid;
            rotid[lane + 64] = mid;
            wave_sync();
            // Pairs inside the tile, lanes without a target, unused slots:
            // mask by index.
            const bool inside = __ballot(lane < nj && mid < i0 + cnt) != 0ull;
            const bool near = chunk_near(mine, lane < nj, bminx, bminy, bminz, bmaxx, bmaxy,
                                         bmaxz, pp.hnear);
            const bool masked = nj < 64 || cnt < 64u * TPL || inside;
#define CUCO_SYM(MK, NR, CL)                                                                    \
    if (TPL == 2)                                                                               \
        interact_sym2<GENERIC, UNIFORM, MK, NR, CL>(rot, rotid, pp, s_tab, xi, yi, zi, pi.w, iid, \
                                                    xi2, yi2, zi2, mi2, iid2, sx_, sy_, sz_,    \
                                                    sx2_, sy2_, sz2_, jx, jy, jz);              \
    else                                                                                        \
        interact_sym<GENERIC, UNIFORM, MK, NR, CL>(rot, rotid, pp, s_tab, xi, yi, zi, pi.w, iid, \
                                                   sx_, sy_, sz_, jx, jy, jz)
            if (clamp) {
                if (masked) {
                    if (near) {
                        CUCO_SYM(true, true, true);
                    } else {
                        CUCO_SYM(true, false, true);
                    }
                } else if (near) {
                    CUCO_SYM(false, true, true);
                } else {
                    CUCO_SYM(false, false, true);
                }
            } else {
                if (masked) {
                    if (near) {
                        CUCO_SYM(true, true, false);
                    } else {
                        CUCO_SYM(true, false, false);
                    }
                } else if (near) {
                    CUCO_SYM(false, true, false);
                } else {
                    CUCO_SYM(false, false, false);
                }
            }
#undef CUCO_SYM
            if ((uint32_t)lane < (uint32_t)nj) {
                const uint32_t j = mid;
                atomicAdd(&jacc[j], (unsigned long long)__double2ll_rn((double)jx * pp.jscale));
                atomicAdd(&jacc[(size_t)n_sorted + j], (unsigned long long)__double2ll_rn((double)jy * pp.jscale));
                atomicAdd(&jacc[2 * (size_t)n_sorted + j], (unsigned long long)__double2ll_rn((double)jz * pp.jscale));
            }
        };
        auto eval_default = [&](int nj, float &sx_, float &sy_, float &sz_) {
            const float4 mine = lane < nj ? sj[lane] : make_float4(0.f, 0.f, 0.f, 0.f);
            const bool near =
                chunk_near(mine, lane < nj, bminx, bminy, bminz, bmaxx, bmaxy, bmaxz, pp.hnear);
#define CUCO_DEF(NR, CL) \
    interact<GENERIC, UNIFORM, NR, CL>(sj, nj, pp, s_tab, xi, yi, zi, sx_, sy_, sz_)
            if (clamp) {
                if (near) CUCO_DEF(true, true);
                else CUCO_DEF(false, true);
            } else if (near) {
                CUCO_DEF(true, false);
            } else {
                CUCO_DEF(false, false);
            }
#undef CUCO_DEF
        };
        uint32_t jc = 0;
        uint32_t cursor = 0;
        uint32_t seen = 0;  // candidate slots of the batches before
        unsigned long long ncand = 0;

        // Unit number cursor + lane as digits (dx, dy, dz) of the mixed radix
        // (nux, nuy, nuz), advanced by the digits of 64 each round (no
        // division per unit); wx0.. = the wrapped unit of digit 0.
        uint32_t dz = 0, dy = 0, dx = 0, sz = 0, sy = 0, sx = 0;
        uint32_t wx0 = 0, wy0 = 0, wz0 = 0;
        const int Mb = M >> lv;
        if (total_q) {
            const uint32_t nz = (uint32_t)nuz, ny = (uint32_t)nuy;
            dz = (uint32_t)lane % nz;
            dy = ((uint32_t)lane / nz) % ny;
            dx = ((uint32_t)lane / nz) / ny;
            sz = 64u % nz;
            sy = (64u / nz) % ny;
            sx = (64u / nz) / ny;
            wx0 = (uint32_t)((ux0 % Mb + Mb) % Mb);
            wy0 = (uint32_t)((uy0 % Mb + Mb) % Mb);
            wz0 = (uint32_t)((uz0 % Mb + Mb) % Mb);
        }
        // A digit is below nu <= 2 Mb + 1 (cells: nq <= 2M; blocks: nq <= M),
        // so two conditional subtractions wrap.
        const uint32_t Mu = (uint32_t)Mb;
        auto wrap2 = [Mu](uint32_t u) {
            u = u >= Mu ? u - Mu : u;
            return u >= Mu ? u - Mu : u;
        };
        // First cell of digit 0 relative to the anchor cell, and the unit's
        // width: cells, and scaled length.
        const int qbx = (ux0 << lv) - c0x, qby = (uy0 << lv) - c0y, qbz = (uz0 << lv) - c0z;
        const int ub = 1 << lv;
        const float uw = (float)ub * pp.cellf;
        const uint32_t span = 1u << (3 * lv);  // keys per unit
        // SYM: a unit whose keys all precede the tile's first particle's
        // holds only particles before it (keys ascend in sorted order).
        const uint32_t key_first = skeys[ia];

        while (cursor < total_q) {
            // Enumerate cells into the range list.
            uint32_t nr = 0;
            // Wide tiles keep filling the range list while a whole round
            // fits (a round that does not fit is redone for the next batch):
            // their rounds find few non-empty units each.
            while (cursor < total_q && (coarse || nr + 64 <= (uint32_t)kR)) {
                bool ok = cursor + lane < total_q;
                uint32_t s = 0, c = 0, packed = 0;
                if (ok) {
                    const int qz = (int)dz * ub + qbz;
                    const int qy = (int)dy * ub + qby;
                    const int qx = (int)dx * ub + qbx;
                    const float lx = qx * pp.cellf, ly = qy * pp.cellf, lz = qz * pp.cellf;
                    const float gx = fmaxf(0.f, fmaxf(lx - bmaxx, bminx - (lx + uw)));
                    const float gy = fmaxf(0.f, fmaxf(ly - bmaxy, bminy - (ly + uw)));
                    const float gz = fmaxf(0.f, fmaxf(lz - bmaxz, bminz - (lz + uw)));
                    ok = gx * gx + gy * gy + gz * gz <= pp.filter2;
                    // FP32 keys are Morton keys; a block's key is its cells'
                    // keys without their 3 low bits.
                    const uint32_t key = key_base + (((spread3(wrap2(wx0 + dx)) << 2) |
                                                      (spread3(wrap2(wy0 + dy)) << 1) |
                                                      spread3(wrap2(wz0 + dz))) << (3 * lv));
                    if (SYM) ok = ok && key + span > key_first;
                    if (ok) {
                        uint32_t e1;
                        if (coarse) {
                            s = off[key];
                            e1 = off[key + 8];
                        } else {
                            load_range(off, key, s, e1);
                        }
                        c = e1 - s;
                        if (SYM) {
                            // only j after the tile's first particle
                            const uint32_t e = s + c, lo = i0 + 1;
                            s = max(s, lo);
                            c = e > s ? e - s : 0u;
                        }
                        ok = c > 0;
                        packed = pack_q(qx, qy, qz);
                    }
                }
                const uint64_t bal = __ballot(ok);
                const uint32_t nnew = uni((uint32_t)__popcll(bal));
                if (nr + nnew > (uint32_t)kR) break;
                if (ok) {
                    const uint32_t pos = nr + (uint32_t)__popcll(bal & lt);
                    rs[pos] = s;
                    rp[pos] = c;
                    rq[pos] = packed;
                }
                nr += nnew;
                cursor += 64;
                dz += sz;
                const uint32_t carry_z = dz >= (uint32_t)nuz ? 1u : 0u;
                dz -= carry_z * (uint32_t)nuz;
                dy += sy + carry_z;
                const uint32_t carry_y = dy >= (uint32_t)nuy ? 1u : 0u;
                dy -= carry_y * (uint32_t)nuy;
                dx += sx + carry_y;
            }
            wave_sync();
            // Exclusive prefix of the range lengths.
            uint32_t carry = 0;
            for (uint32_t b0 = 0; b0 < nr; b0 += 64) {
                const uint32_t idx = b0 + lane;
                const uint32_t v = idx < nr ? rp[idx] : 0u;
                const uint32_t inc = wave_incl_scan(v);
                if (idx < nr) rp[idx] = carry + inc - v;
                carry = uni(carry + (uint32_t)__builtin_amdgcn_readlane(inc, 63));
            }
            if (lane == 0) rp[nr] = carry;
            wave_sync();
            const uint32_t total_j = carry;

            // Stream, filter and evaluate.  Candidate slots are taken 64 at a
            // time; rc is the range holding the window's first slot f0.
            // Ranges are non-empty, so the ranges rc+1.. start at strictly
            // increasing slots after f0: lane L looks up where range rc+1+L
            // starts, marks that slot of the window (a permute: each lane
            // sends a 1 to the lane of its start slot; lanes without a
            // start in the window send 0 to slot 0, which no range after rc
            // can start at), and slot s then lies in range rc + (number of
            // marks at or below s).
            // A split tile's parts go by the number of the window in the whole
            // tile, so that where a batch ends does not matter: its windows
            // start before the batch does where that ended inside one.
            uint32_t rc = 0;
            const uint32_t skew = nsplit > 1u ? seen & 63u : 0u;
            for (uint32_t g = 0; g < total_j + skew; g += 64) {
                // Part p of a split tile takes every nsplit-th window.
                const bool mine = nsplit == 1u || ((seen + g) >> 6) % nsplit == part;
                const uint32_t f0 = g - skew;  // wraps below 0: no slot of this batch
                const uint32_t f = f0 + lane;
                bool ok = f < total_j;
                const uint32_t rn = rc + 1 + (uint32_t)lane;
                const uint32_t st = rn < nr ? rp[rn] - f0 : 0xffffffffu;
                const bool mark = st < 64u;
                const int got = __builtin_amdgcn_ds_permute(mark ? (int)(st * 4u) : 0, mark ? 1 : 0);
                const uint64_t starts = __ballot(got != 0);
                const uint32_t lo =
                    rc + __builtin_amdgcn_mbcnt_hi((uint32_t)(starts >> 32),
                                                   __builtin_amdgcn_mbcnt_lo((uint32_t)starts, 0u)) +
                    (got != 0 ? 1u : 0u);
                rc = uni(rc + (uint32_t)__popcll(__ballot(st <= 64u)));
                if (SYM && !mine) continue;
                float4 qj = make_float4(0.f, 0.f, 0.f, 0.f);
                uint32_t jsorted = 0;
                if (ok) {
                    const uint32_t j = rs[lo] + (f - rp[lo]);
                    jsorted = j;
                    int qx, qy, qz;
                    unpack_q(rq[lo], qx, qy, qz);
                    if (coarse) {
                        // the cell inside the 2x2x2 block: the key's low bits
                        const uint32_t kj = skeys[j];
                        qx += (int)((kj >> 2) & 1u);
                        qy += (int)((kj >> 1) & 1u);
                        qz += (int)(kj & 1u);
                    }
                    const float4 pj = spos[j];
                    qj = make_float4(rel_coord(pj.x, qx, pp.s, pp.cellf),
                                     rel_coord(pj.y, qy, pp.s, pp.cellf),
                                     rel_coord(pj.z, qz, pp.s, pp.cellf), pj.w);
                    const float gx = fmaxf(0.f, fmaxf(bminx - qj.x, qj.x - bmaxx));
                    const float gy = fmaxf(0.f, fmaxf(bminy - qj.y, qj.y - bmaxy));
                    const float gz = fmaxf(0.f, fmaxf(bminz - qj.z, qj.z - bmaxz));
                    ok = gx * gx + gy * gy + gz * gz <= pp.filter2;
                }
                const uint64_t bal = __ballot(ok);
                if (ok) {
                    const uint32_t slot = jc + (uint32_t)__popcll(bal & lt);
                    sj[slot] = qj;
                    if (SYM) sjid[slot] = jsorted;
                }
                jc = uni(jc + (uint32_t)__popcll(bal));
                wave_sync();
                if (jc >= 64) {
                    float sx = 0.f, sy = 0.f, sz = 0.f, sx2 = 0.f, sy2 = 0.f, sz2 = 0.f;
                    if (SYM) {
                        eval_sym(64, sx, sy, sz, sx2, sy2, sz2);
                    } else {
                        eval_default(64, sx, sy, sz);
                    }
                    kahan_add(ax, kx, sx);
                    kahan_add(ay, ky, sy);
                    kahan_add(az, kz, sz);
                    if (TPL == 2) {
                        kahan_add(ax2, kx2, sx2);
                        kahan_add(ay2, ky2, sy2);
                        kahan_add(az2, kz2, sz2);
                    }
                    if (cand) ncand += 64ull * cnt;
                    const uint32_t rem = jc - 64;
                    float4 tmp = make_float4(0.f, 0.f, 0.f, 0.f);
                    uint32_t tid = 0;
                    if ((uint32_t)lane < rem) {
                        tmp = sj[64 + lane];
                        if (SYM) tid = sjid[64 + lane];
                    }
                    wave_sync();
                    if ((uint32_t)lane < rem) {
                        sj[lane] = tmp;
                        if (SYM) sjid[lane] = tid;
                    }
                    jc = rem;
                    wave_sync();
                }
            }
            seen += total_j;
        }
        if (jc > 0) {
            float sx = 0.f, sy = 0.f, sz = 0.f, sx2 = 0.f, sy2 = 0.f, sz2 = 0.f;
            if (SYM) {
                eval_sym((int)jc, sx, sy, sz, sx2, sy2, sz2);
            } else {
                eval_default((int)jc, sx, sy, sz);
            }
            kahan_add(ax, kx, sx);
            kahan_add(ay, ky, sy);
            kahan_add(az, kz, sz);
            if (TPL == 2) {
                kahan_add(ax2, kx2, sx2);
                kahan_add(ay2, ky2, sy2);
                kahan_add(az2, kz2, sz2);
            }
            if (cand) ncand += (unsigned long long)jc * cnt;
            jc = 0;
        }
        wave_sync();
        if (SYM) {
            // Part 0 stores the tile's own sums, the others add theirs to the
            // fixed-point sums of the j side (exact, so in any order).
            auto add_fixed = [&](uint32_t k, float vx, float vy, float vz) {
                atomicAdd(&jacc[k], (unsigned long long)__double2ll_rn((double)vx * pp.jscale));
                atomicAdd(&jacc[(size_t)n_sorted + k], (unsigned long long)__double2ll_rn((double)vy * pp.jscale));
                atomicAdd(&jacc[2 * (size_t)n_sorted + k], (unsigned long long)__double2ll_rn((double)vz * pp.jscale));
            };
            if (part == 0u) {
                if (valid) iacc[i] = make_float4(ax, ay, az, 0.f);
                if (TPL == 2 && valid2) iacc[i2] = make_float4(ax2, ay2, az2, 0.f);
            } else {
                if (valid) add_fixed(i, ax, ay, az);
                if (TPL == 2 && valid2) add_fixed(i2, ax2, ay2, az2);
            }
        } else if (act) {
            acc[perm[i]] = make_float4(ax * pp.out_scale, ay * pp.out_scale,
                                       az * pp.out_scale, 0.f);
        }
        if (cand) atomicAdd(cand, lane == 0 ? ncand : 0ull);
    }
}

// ---------------------------------------------------------------------------
// Small launches: a tile per workgroup.  With fewer tiles than the chip has
// SIMDs a wave alone on its SIMD waits out every load of the enumeration, one
// round of 64 units after another (32^3 lattice particles: 512 tiles, 87 us,
// of which the pairs are about 20).  Here the eight waves of a workgroup enumerate
// 512 units a round, filter eight windows of candidates at a time into one
// list in LDS, and take a chunk of 64 of it each; the chunks' sums are added
// in the order of the chunks.  Candidates, chunks, their evaluation and the
// order of every sum are k_pp32's, so which kernel takes a launch does not
// show in the bits (an ensemble's large launch gives each box what a launch of
// its own does).
constexpr int kTeam = 8;                   // waves
constexpr int kTeamRanges = 1024;          // cell ranges before the windows
constexpr int kTeamList = 1024;            // filtered candidates before the chunks
constexpr int kTeamChunks = kTeamList / 64;
// Launches of up to as many particles (about three tiles a SIMD).  Measured,
// pair force and its clears, a tile a wave -> a tile a workgroup, us: lattice
// 24^3 94 -> 35, 32^3 96 -> 46, 48^3 158 -> 90, 56^3 215 -> 182, 64^3 230 ->
// 179; halos 24^3 241 -> 68, 32^3 361 -> 121, 48^3 571 -> 381, 56^3 766 -> 735,
// 64^3 956 -> 988.  The host knows a launch's particles, not how clustered
// they are: the line lies where halos stop gaining, below the last lattice
// that still would.
constexpr uint32_t kTeamParticles = 200000;

struct Team32 {
    float tab[kTabSym];
    uint32_t rs[kTeamRanges], rp[kTeamRanges], rq[kTeamRanges];
    float4 q[kTeamList];
    uint32_t id[kTeamList];
    float4 rot[kTeam][128];
    uint32_t rotid[kTeam][128];
    float sum[kTeamChunks][3][64];
    uint32_t count[2][kTeam], slots[2][kTeam];
    uint32_t item;
};

// Exclusive prefix over the waves of one value each, and the total.  The two
// buffers take turns, so that one barrier between write and read is enough.
__device__ inline uint32_t team_prefix(const uint32_t (&buf)[2][kTeam], int turn, int w,
                                       uint32_t &total)
{
    uint32_t before = 0;
    total = 0;
#pragma unroll
    for (int k = 0; k < kTeam; ++k) {
        const uint32_t c = buf[turn][k];
        before += k < w ? c : 0u;
        total += c;
    }
    before = uni(before);
    total = uni(total);
    return before;
}

template <bool GENERIC, bool UNIFORM>
__global__ __launch_bounds__(64 * kTeam, 4) void k_pp32_team(
    const float4 *__restrict__ spos, const uint32_t *__restrict__ skeys,
    const uint32_t *__restrict__ off, BoxView tv, const P32 *__restrict__ p32s, float mass,
    const float *__restrict__ table32, const uint32_t *__restrict__ tstart,
    const uint32_t *__restrict__ tcount, uint32_t *__restrict__ counters,
    float4 *__restrict__ iacc, unsigned long long *__restrict__ jacc, uint32_t n_sorted,
    float coarse_cells, const uint2 *__restrict__ parts, uint32_t max_parts)
{
    __shared__ Team32 sh;
    for (int k = threadIdx.x; k < kTabSym; k += 64 * kTeam)
        sh.tab[k] = k < kTabPadded ? (UNIFORM ? mass * table32[k] : table32[k]) : 0.0f;
    const int lane = threadIdx.x & 63, w = (int)uni(threadIdx.x >> 6);
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const uint32_t nparts = min(counters[2], max_parts);
    const uint32_t nmid = min(counters[3], max_parts - nparts);
    const uint32_t nlisted = uni(nparts + nmid), nitems = uni(nlisted + counters[0]);
    const float inf = __builtin_huge_valf();
    float4 *rot = sh.rot[w];
    uint32_t *rotid = sh.rotid[w];

    for (;;) {
        __syncthreads();  // the last item is done with; the table
        if (threadIdx.x == 0) sh.item = atomicAdd(&counters[1], 1u);
        __syncthreads();
        const uint32_t item = uni(sh.item);
        if (item >= nitems) break;
        uint32_t t = item - nlisted, part = 0;
        if (item < nlisted) {
            const uint2 pt = parts[item < nparts ? item : max_parts - 1u - (item - nparts)];
            t = uni(pt.x);
            part = uni(pt.y);
        }
        const uint32_t word = uni(tcount[t]);
        if (item >= nlisted && (word & kListed)) continue;

        const int bi = find_box(tv.map, tv.nboxes, t);
        const P32 pp = p32s[bi];
        const GridInfo &g = tv.box[bi].g;
        const uint32_t key_base = tv.box[bi].key_base;
        const int M = pp.M;
        const uint32_t i0 = uni(tstart[t]);
        const uint32_t cnt = word & 255u, nsplit = ((word >> 8) & (kPartMost - 1u)) + 1u;
        const bool valid = (uint32_t)lane < cnt;
        const uint32_t i = i0 + (valid ? (uint32_t)lane : 0u);
        const uint32_t key_first = skeys[i0];
        int c0x, c0y, c0z, cx, cy, cz;
        key_cell(g, key_first - key_base, c0x, c0y, c0z);
        key_cell(g, skeys[i] - key_base, cx, cy, cz);
        const float4 pi = spos[i];
        const float xi = rel_coord(pi.x, unwrap_delta(cx - c0x, M), pp.s, pp.cellf);
        const float yi = rel_coord(pi.y, unwrap_delta(cy - c0y, M), pp.s, pp.cellf);
        const float zi = rel_coord(pi.z, unwrap_delta(cz - c0z, M), pp.s, pp.cellf);
        TileBox box;
        box.minx = uni(wave_min(valid ? xi : inf));
        box.miny = uni(wave_min(valid ? yi : inf));
        box.minz = uni(wave_min(valid ? zi : inf));
        box.maxx = uni(wave_max(valid ? xi : -inf));
        box.maxy = uni(wave_max(valid ? yi : -inf));
        box.maxz = uni(wave_max(valid ? zi : -inf));
        const TileUnits tu = tile_units(box, pp, c0x, c0y, c0z, coarse_cells);
        const bool clamp = tile_clamps<kTabSym>(box, pp);
        const uint32_t iid = valid ? i : 0xffffffffu;
        const int lv = tu.coarse ? 1 : 0;
        const int ub = 1 << lv;
        const uint32_t Mu = (uint32_t)(M >> lv);
        auto wrap2 = [Mu](uint32_t u) {
            u = u >= Mu ? u - Mu : u;
            return u >= Mu ? u - Mu : u;
        };
        const uint32_t wx0 = (uint32_t)((tu.ux0 % (int)Mu + (int)Mu) % (int)Mu);
        const uint32_t wy0 = (uint32_t)((tu.uy0 % (int)Mu + (int)Mu) % (int)Mu);
        const uint32_t wz0 = (uint32_t)((tu.uz0 % (int)Mu + (int)Mu) % (int)Mu);
        const int qbx = (tu.ux0 << lv) - c0x, qby = (tu.uy0 << lv) - c0y, qbz = (tu.uz0 << lv) - c0z;
        const float uw = (float)ub * pp.cellf;
        const uint32_t span = 1u << (3 * lv);

        // Kahan sums: wave 0 x, wave 1 y, wave 2 z.
        float acc = 0.f, comp = 0.f;
        uint32_t jc = 0;      // candidates in the list
        uint32_t cursor = 0;  // unit
        uint32_t seen = 0;    // candidate slots of the batches before
        int turn = 0;

        // The list's chunks (the last one in part, at the end): evaluated,
        // their sums added, what is left moved to the front.
        auto evaluate = [&](bool all) {
            __syncthreads();  // the list is written
            const uint32_t nfull = jc / 64u, nc = all ? (jc + 63u) / 64u : nfull;
            for (uint32_t c = (uint32_t)w; c < nc; c += kTeam) {
                const int nj = (int)min(64u, jc - 64u * c);
                float sx = 0.f, sy = 0.f, sz = 0.f, jx = 0.f, jy = 0.f, jz = 0.f;
                // As k_pp32's eval_sym.
                float4 mine = make_float4(box.minx - 1.0f, box.miny, box.minz, 0.f);
                uint32_t mid = 0u;
                if (lane < nj) {
                    mine = sh.q[64u * c + lane];
                    mid = sh.id[64u * c + lane];
                }
                rot[lane] = mine;
                rot[lane + 64] = mine;
                rotid[lane] = mid;
                rotid[lane + 64] = mid;
                wave_sync();
                const bool inside = __ballot(lane < nj && mid < i0 + cnt) != 0ull;
                const bool near = chunk_near(mine, lane < nj, box.minx, box.miny, box.minz, box.maxx,
                                             box.maxy, box.maxz, pp.hnear);
                const bool masked = nj < 64 || cnt < 64u || inside;
#define CUCO_SYM(MK, NR, CL)                                                                     \
    interact_sym<GENERIC, UNIFORM, MK, NR, CL>(rot, rotid, pp, sh.tab, xi, yi, zi, pi.w, iid, sx, \
                                               sy, sz, jx, jy, jz)
                if (clamp) {
                    if (masked) {
                        if (near) CUCO_SYM(true, true, true);
                        else CUCO_SYM(true, false, true);
                    } else if (near) {
                        CUCO_SYM(false, true, true);
                    } else {
                        CUCO_SYM(false, false, true);
                    }
                } else {
                    if (masked) {
                        if (near) CUCO_SYM(true, true, false);
                        else CUCO_SYM(true, false, false);
                    } else if (near) {
                        CUCO_SYM(false, true, false);
                    } else {
                        CUCO_SYM(false, false, false);
                    }
                }
#undef CUCO_SYM
                if (lane < nj) {
                    atomicAdd(&jacc[mid], (unsigned long long)__double2ll_rn((double)jx * pp.jscale));
                    atomicAdd(&jacc[(size_t)n_sorted + mid], (unsigned long long)__double2ll_rn((double)jy * pp.jscale));
                    atomicAdd(&jacc[2 * (size_t)n_sorted + mid], (unsigned long long)__double2ll_rn((double)jz * pp.jscale));
                }
                sh.sum[c][0][lane] = sx;
                sh.sum[c][1][lane] = sy;
                sh.sum[c][2][lane] = sz;
                wave_sync();
            }
            const uint32_t left = all ? 0u : jc - 64u * nfull;
            float4 tmp = make_float4(0.f, 0.f, 0.f, 0.f);
            uint32_t tid = 0;
            if (w == kTeam - 1 && (uint32_t)lane < left) {
                tmp = sh.q[64u * nfull + lane];
                tid = sh.id[64u * nfull + lane];
            }
            __syncthreads();
            if (w < 3)
                for (uint32_t c = 0; c < nc; ++c) kahan_add(acc, comp, sh.sum[c][w][lane]);
            if (w == kTeam - 1 && (uint32_t)lane < left) {
                sh.q[lane] = tmp;
                sh.id[lane] = tid;
            }
            jc = left;
            __syncthreads();
        };

        while (cursor < tu.total) {
            // Enumerate units into the range list, rp: slots before the range.
            uint32_t nr = 0, total_j = 0;
            while (cursor < tu.total && nr + 64u * kTeam <= (uint32_t)kTeamRanges) {
                const uint32_t u = cursor + 64u * (uint32_t)w + (uint32_t)lane;
                bool ok = u < tu.total;
                uint32_t first = 0, c = 0, packed = 0;
                if (ok) {
                    const uint32_t r = u / (uint32_t)tu.nuz, dz = u - r * (uint32_t)tu.nuz;
                    const uint32_t dx = r / (uint32_t)tu.nuy, dy = r - dx * (uint32_t)tu.nuy;
                    const int qz = (int)dz * ub + qbz;
                    const int qy = (int)dy * ub + qby;
                    const int qx = (int)dx * ub + qbx;
                    const float lx = qx * pp.cellf, ly = qy * pp.cellf, lz = qz * pp.cellf;
                    const float gx = fmaxf(0.f, fmaxf(lx - box.maxx, box.minx - (lx + uw)));
                    const float gy = fmaxf(0.f, fmaxf(ly - box.maxy, box.miny - (ly + uw)));
                    const float gz = fmaxf(0.f, fmaxf(lz - box.maxz, box.minz - (lz + uw)));
                    const uint32_t key = key_base + (((spread3(wrap2(wx0 + dx)) << 2) |
                                                      (spread3(wrap2(wy0 + dy)) << 1) |
                                                      spread3(wrap2(wz0 + dz))) << (3 * lv));
                    ok = gx * gx + gy * gy + gz * gz <= pp.filter2 && key + span > key_first;
                    if (ok) {
                        // only j after the tile's first particle
                        const uint32_t end = off[key + span];
                        first = max(off[key], i0 + 1);
                        c = end > first ? end - first : 0u;
                        ok = c > 0;
                        packed = pack_q(qx, qy, qz);
                    }
                }
                const uint64_t bal = __ballot(ok);
                const uint32_t inc = wave_incl_scan(c);
                if (lane == 63) {
                    sh.count[turn][w] = (uint32_t)__popcll(bal);
                    sh.slots[turn][w] = inc;
                }
                __syncthreads();
                uint32_t nnew, jnew;
                const uint32_t at = nr + team_prefix(sh.count, turn, w, nnew) +
                                    (uint32_t)__popcll(bal & lt);
                const uint32_t slot = total_j + team_prefix(sh.slots, turn, w, jnew) + inc - c;
                turn ^= 1;
                if (ok) {
                    sh.rs[at] = first;
                    sh.rp[at] = slot;
                    sh.rq[at] = packed;
                }
                nr += nnew;
                total_j += jnew;
                cursor += 64u * kTeam;
            }
            __syncthreads();
            // The part's windows of the batch (numbered over the tile), one
            // per wave at a time.
            const uint32_t skew = nsplit > 1u ? seen & 63u : 0u;
            const uint32_t nwin = (total_j + skew + 63u) / 64u;
            const uint32_t ahead = nsplit > 1u ? (part + nsplit - (seen >> 6) % nsplit) % nsplit : 0u;
            for (uint32_t k0 = ahead; k0 < nwin; k0 += nsplit * kTeam) {
                if (jc + 64u * kTeam > (uint32_t)kTeamList) evaluate(false);
                const uint32_t f = 64u * (k0 + nsplit * (uint32_t)w) - skew + (uint32_t)lane;
                bool ok = f < total_j;
                float4 qj = make_float4(0.f, 0.f, 0.f, 0.f);
                uint32_t j = 0;
                if (ok) {
                    // The range that holds slot f: the last that starts at or before it.
                    uint32_t r = 0;
                    for (uint32_t o = kTeamRanges / 2; o > 0; o >>= 1)
                        if (r + o < nr && sh.rp[r + o] <= f) r += o;
                    j = sh.rs[r] + (f - sh.rp[r]);
                    int qx, qy, qz;
                    unpack_q(sh.rq[r], qx, qy, qz);
                    if (tu.coarse) {
                        // the cell inside the 2x2x2 block: the key's low bits
                        const uint32_t kj = skeys[j];
                        qx += (int)((kj >> 2) & 1u);
                        qy += (int)((kj >> 1) & 1u);
                        qz += (int)(kj & 1u);
                    }
                    const float4 pj = spos[j];
                    qj = make_float4(rel_coord(pj.x, qx, pp.s, pp.cellf),
                                     rel_coord(pj.y, qy, pp.s, pp.cellf),
                                     rel_coord(pj.z, qz, pp.s, pp.cellf), pj.w);
                    const float gx = fmaxf(0.f, fmaxf(box.minx - qj.x, qj.x - box.maxx));
                    const float gy = fmaxf(0.f, fmaxf(box.miny - qj.y, qj.y - box.maxy));
                    const float gz = fmaxf(0.f, fmaxf(box.minz - qj.z, qj.z - box.maxz));
                    ok = gx * gx + gy * gy + gz * gz <= pp.filter2;
                }
                const uint64_t bal = __ballot(ok);
                if (lane == 0) sh.count[turn][w] = (uint32_t)__popcll(bal);
                __syncthreads();
                uint32_t nnew;
                const uint32_t at = jc + team_prefix(sh.count, turn, w, nnew) +
                                    (uint32_t)__popcll(bal & lt);
                turn ^= 1;
                if (ok) {
                    sh.q[at] = qj;
                    sh.id[at] = j;
                }
                jc += nnew;
            }
            seen += total_j;
            __syncthreads();  // the range list is read
        }
        evaluate(true);
        if (w < 3) sh.sum[0][w][lane] = acc;
        __syncthreads();
        if (w == 0 && valid) {
            const float ax = sh.sum[0][0][lane], ay = sh.sum[0][1][lane], az = sh.sum[0][2][lane];
            if (part == 0u) {
                iacc[i] = make_float4(ax, ay, az, 0.f);
            } else {
                atomicAdd(&jacc[i], (unsigned long long)__double2ll_rn((double)ax * pp.jscale));
                atomicAdd(&jacc[(size_t)n_sorted + i], (unsigned long long)__double2ll_rn((double)ay * pp.jscale));
                atomicAdd(&jacc[2 * (size_t)n_sorted + i], (unsigned long long)__double2ll_rn((double)az * pp.jscale));
            }
        }
    }
}

// Tiles of one super-block: the 8 Morton blocks (2^shift cells a side) of
// one block a level up.  Consecutive blocks whose particles add up to at
// most run (64, or 128 for two targets per lane) share a tile (in sparse
// regions a block alone would leave most of the wave idle); a block with
// more than run particles is cut into runs of that length.  A tile is a
// contiguous range of sorted particles inside one super-block.  One wave per
// super-block: lane l <= 8 holds its l-th block offset o; calls
// emit(first block, last block, start, particles, run length) for each group
// of blocks, where a group longer than the run length is cut.
template <typename F>
__device__ inline void super_groups(uint32_t o, uint32_t run, F emit)
{
    uint32_t gs = __builtin_amdgcn_readlane(o, 0), gn = 0;
    int g0 = 0;
    for (int k = 0; k < 8; ++k) {
        const uint32_t bs = __builtin_amdgcn_readlane(o, k);
        const uint32_t c = __builtin_amdgcn_readlane(o, k + 1) - bs;
        if (gn + c > run) {
            if (gn) emit(g0, k - 1, gs, gn);
            gn = 0;
        }
        if (c > run) {
            emit(k, k, bs, c);
        } else if (c) {
            if (gn == 0) {
                gs = bs;
                g0 = k;
            }
            gn += c;
        }
    }
    if (gn) emit(g0, 7, gs, gn);
}

__device__ inline uint32_t super_offsets(const uint32_t *__restrict__ off, uint32_t sb, int shift3)
{
    const int l = min((int)(threadIdx.x & 63u), 8);
    return off[((size_t)sb << (shift3 + 3)) + ((size_t)l << shift3)];
}

// Box of super-block sb, through the map of 16^3-cell bricks (boxes start on
// super-block and brick boundaries: a box's key range is 8^bits, bits > shift
// and >= 4).
__device__ inline int super_box(const BoxView &bricks, uint32_t sb, int shift3)
{
    return uni(find_box(bricks.map, bricks.nboxes, (uint32_t)(((size_t)sb << (shift3 + 3)) >> 12)));
}

__device__ inline uint32_t wave_sum(uint32_t v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += (uint32_t)__shfl_xor((int)v, o, 64);
    return uni(v);
}

// Parts of long tiles (each-pair-once kernel).  A tile in a halo core meets
// thousands of candidates; one wave per tile left the launch waiting for the
// longest of them (300007 halo particles: 3.0 ms for 0.6 ms of pairs).  Such
// a tile is taken by several waves, each every nsplit-th window of 64
// candidates.  Only the box's own particles decide, so a box gives the same
// forces, bit for bit, alone and in an ensemble.
//
// k_super_tiles estimates a tile's candidates as the particles of its aligned
// Morton block of 2^eb cells a side (eb = 3, or the tiles' own block shift
// where that is 4) and of the blocks around it, less the blocks before it
// (they hold only earlier particles); for a tile of several blocks, all the
// blocks in and around its super-block.  The tiles' sum is the box's work.
// k_fill_tiles cuts at a kPartShare-th
// of it, but not below kPartMin candidates, where a part's own enumeration of
// the tile's cells and its last, partly filled chunk would show, nor below
// what tiles of a nearly uniform box come to, where none stands out.  Parts are
// taken first and whole tiles of over a kPartMid-th of a part and twice the
// box's average next, so that the launch ends on short items.  Measured (pair
// kernel): 300007 halo particles 2.97 -> 1.19 ms, 128^3 10.0 -> 7.9, 256^3 in
// tiles of 128 47.3 -> 39.9; at a 16384-th 8.0 and 40.3, at a 65536-th 8.0
// and 40.5; at 8192 candidates at least the 300007 take 1.44 ms.
constexpr uint32_t kPartMid = 4;
constexpr int kSuperEst = 9;     // per super-block: its 8 blocks, all
constexpr int kSuperWaves = 16;  // super-blocks of a workgroup (one add to the box's sum)

__global__ __launch_bounds__(64 * kSuperWaves) void k_super_tiles(
    const uint32_t *__restrict__ off, uint32_t nsuper, int shift, uint32_t run, BoxView bricks,
    uint32_t *__restrict__ super_count,
    uint32_t *__restrict__ est, unsigned long long *__restrict__ work,
    uint32_t *__restrict__ counters)
{
    if (blockIdx.x == 0 && threadIdx.x < 2) counters[2 + threadIdx.x] = 0u;
    const int lane = threadIdx.x & 63;
    const int shift3 = 3 * shift, eb = max(3, shift);
    const int nb = shift + 1 > eb ? 2 : 1;  // estimate blocks of a super-block per axis
    __shared__ unsigned long long s_work[kSuperWaves];
    __shared__ int s_box[kSuperWaves];
    const int wv = (int)uni(threadIdx.x >> 6);
    const uint32_t sb = blockIdx.x * (uint32_t)kSuperWaves + (uint32_t)wv;
    unsigned long long w = 0;
    int bi = -1;
    if (sb < nsuper) {
        const uint32_t o = super_offsets(off, sb, shift3);
        uint32_t count = 0;
        // An empty super-block (voids, and the padding of a Morton key space
        // around a mesh that is not a power of two) has no tiles.
        if (__builtin_amdgcn_readlane(o, 8) != __builtin_amdgcn_readlane(o, 0)) {
            bi = super_box(bricks, sb, shift3);
            const GridInfo &g = bricks.box[bi].g;
            const uint32_t kb = bricks.box[bi].key_base;
            // Lane (x, y, z) of 4^3: the block at the super-block's first one
            // plus (x, y, z) - 1, periodic; a whole turn at most.
            const int last = (g.M - 1) >> eb, turn = last + 1;
            const uint32_t own = ((sb << (shift3 + 3)) - kb) >> (3 * eb);
            int bx, by, bz;
            key_cell(g, own, bx, by, bz);
            const int x = lane >> 4, y = (lane >> 2) & 3, z = lane & 3;
            const int most = min(nb + 2, turn);
            uint32_t occ = 0, blk = 0;
            if (x < most && y < most && z < most) {
                int q[3] = {bx - 1 + x, by - 1 + y, bz - 1 + z};
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    q[k] = q[k] < 0 ? q[k] + turn : q[k];
                    q[k] = q[k] > last ? q[k] - turn : q[k];
                }
                blk = cell_key(g, q[0], q[1], q[2]);
                const uint32_t key = kb + (blk << (3 * eb));
                occ = off[key + (1u << (3 * eb))] - off[key];
            }
            const uint32_t all = wave_sum(blk >= own ? occ : 0u);
            uint32_t mine = all;  // lane k < 8: block k's estimate, else all
            if (all >= 2u * kPartMin && nb == 2) {
                for (int k = 0; k < 8; ++k) {
                    const int dx = x - ((k >> 2) & 1), dy = y - ((k >> 1) & 1), dz = z - (k & 1);
                    const bool around = most < 4 || ((unsigned)dx < 3u && (unsigned)dy < 3u &&
                                                     (unsigned)dz < 3u);
                    const uint32_t e = wave_sum(around && blk >= own + (uint32_t)k ? occ : 0u);
                    if (lane == k) mine = e;
                }
            }
            if (lane < kSuperEst) est[(size_t)sb * kSuperEst + lane] = mine;
            // The tiles, and the box's work: their estimates.
            super_groups(o, run, [&](int b0, int b1, uint32_t, uint32_t n) {
                const uint32_t nt = (n + run - 1) / run;
                count += nt;
                w += (unsigned long long)nt * (uint32_t)__builtin_amdgcn_readlane(mine, b0 == b1 ? b0 : kSuperEst - 1);
            });
        }
        if (lane == 0) super_count[sb] = count;
    }
    // One add per workgroup and box.
    if (lane == 0) {
        s_work[wv] = w;
        s_box[wv] = bi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long sum = 0;
        int box = -1;
        for (int k = 0; k < kSuperWaves; ++k) {
            if (s_box[k] < 0) continue;
            if (s_box[k] != box) {
                if (sum) atomicAdd(&work[box], sum);
                sum = 0;
                box = s_box[k];
            }
            sum += s_work[k];
        }
        if (sum) atomicAdd(&work[box], sum);
    }
}

// First tile of each box: the scanned tile offset of its first super-block.
__device__ inline uint32_t first_tile(int b, const uint32_t *__restrict__ tile_off,
                                      const BoxView &bricks, int shift3,
                                      const uint32_t *__restrict__ counters)
{
    return b < bricks.nboxes ? tile_off[((size_t)bricks.map[b] << 12) >> (shift3 + 3)]
                             : counters[0];
}

__global__ __launch_bounds__(256) void k_fill_tiles(
    const uint32_t *__restrict__ off, const uint32_t *__restrict__ tile_off, uint32_t nsuper,
    int shift3, uint32_t run, BoxView bricks,
    const uint32_t *__restrict__ est, const unsigned long long *__restrict__ work,
    uint32_t *__restrict__ tstart, uint32_t *__restrict__ tcount, uint32_t *__restrict__ counters,
    uint2 *__restrict__ parts, uint32_t max_parts, uint32_t *__restrict__ tile_map)
{
    const uint32_t id = blockIdx.x * 256u + threadIdx.x;
    if (id <= (uint32_t)bricks.nboxes)
        tile_map[id] = first_tile((int)id, tile_off, bricks, shift3, counters);
    const int lane = threadIdx.x & 63;
    const uint32_t sb = uni(id >> 6);
    if (sb >= nsuper) return;
    const uint32_t o = super_offsets(off, sb, shift3);
    if (__builtin_amdgcn_readlane(o, 8) == __builtin_amdgcn_readlane(o, 0)) return;
    const int bi = super_box(bricks, sb, shift3);
    const uint32_t es = lane < kSuperEst ? est[(size_t)sb * kSuperEst + lane] : 0u;
    const unsigned long long total = work[bi];
    const unsigned long long ntiles = first_tile(bi + 1, tile_off, bricks, shift3, counters) -
                                      first_tile(bi, tile_off, bricks, shift3, counters);
    // What the estimate of a tile is at most in a uniform box (4 blocks a side).
    const GridInfo &g = bricks.box[bi].g;
    const float reach = (float)(4 << max(3, shift3 / 3)) / (float)g.M;
    const float uniform = (float)bricks.box[bi].n * reach * reach * reach;
    const uint32_t size = tile_part_size(total, (uint32_t)fminf(1.5f * uniform, 1e9f));
    uint32_t t = uni(tile_off[sb]);
    super_groups(o, run, [&](int b0, int b1, uint32_t start, uint32_t n) {
        const uint32_t e = __builtin_amdgcn_readlane(es, b0 == b1 ? b0 : kSuperEst - 1);
        const uint32_t nt = (n + run - 1) / run, np = uni(tile_parts(e, size));
        const bool mid = np == 1u && e > size / kPartMid && e * ntiles > 2ull * total;
        const uint32_t word = np > 1u ? ((np - 1u) << 8) | kListed : mid ? kListed : 0u;
        for (uint32_t k = lane; k < nt; k += 64u) {
            tstart[t + k] = start + k * run;
            tcount[t + k] = min(run, n - k * run) | word;
        }
        if (word) {
            // tile_parts_bound keeps both ends of the list apart.
            uint32_t at = 0;
            if (lane == 0) at = atomicAdd(&counters[np > 1u ? 2 : 3], nt * np);
            at = uni(at);
            for (uint32_t k = lane; k < nt * np; k += 64u)
                if (at + k < max_parts)
                    parts[np > 1u ? at + k : max_parts - 1u - (at + k)] = make_uint2(t + k / np, k % np);
        }
        t += nt;
    });
}

__global__ void k_box_tiles(const uint32_t *__restrict__ tile_off, BoxView bricks,
                            int shift3, const uint32_t *__restrict__ counters,
                            uint32_t *__restrict__ tile_map)
{
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b <= (uint32_t)bricks.nboxes)
        tile_map[b] = first_tile((int)b, tile_off, bricks, shift3, counters);
}

// Active targets of an integer-timeline step, packed into their own tiles.
// flag: 1 where the particle at sorted index s is active; scanned in place
// (exclusive, scan[n] = total), scan[s+1] - scan[s] is that flag again.
__global__ void k_act_flags(const uint32_t *__restrict__ perm,
                            const int32_t *__restrict__ active_end, int32_t ti_current,
                            uint32_t n, uint32_t *__restrict__ flag)
{
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < n) flag[s] = active_end[perm[s]] == ti_current ? 1u : 0u;
}

__global__ void k_act_list(const uint32_t *__restrict__ scan, uint32_t n,
                           uint32_t *__restrict__ list)
{
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < n && scan[s + 1] > scan[s]) list[scan[s]] = s;
}

// Active targets of super-block sb: list positions [a0, a0 + count).
__device__ inline uint32_t super_active(const uint32_t *__restrict__ off,
                                        const uint32_t *__restrict__ scan, uint32_t sb,
                                        int shift3, uint32_t &a0)
{
    const size_t base = (size_t)sb << (shift3 + 3);
    a0 = scan[off[base]];
    return scan[off[base + ((size_t)1 << (shift3 + 3))]] - a0;
}

__global__ void k_block_tiles_act(const uint32_t *__restrict__ off,
                                  const uint32_t *__restrict__ scan, uint32_t nsuper,
                                  int shift3, uint32_t *__restrict__ super_count)
{
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nsuper) return;
    uint32_t a0;
    super_count[b] = (super_active(off, scan, b, shift3, a0) + 63u) / 64u;
}

__global__ void k_fill_tiles_act(const uint32_t *__restrict__ off,
                                 const uint32_t *__restrict__ scan,
                                 const uint32_t *__restrict__ tile_off, uint32_t nsuper,
                                 int shift3, uint32_t *__restrict__ tstart,
                                 uint32_t *__restrict__ tcount)
{
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nsuper) return;
    uint32_t a0;
    const uint32_t c = super_active(off, scan, b, shift3, a0);
    uint32_t t = tile_off[b];
    for (uint32_t p = 0; p < c; p += 64u, ++t) {
        tstart[t] = a0 + p;
        tcount[t] = min(64u, c - p);
    }
}

// Before an each-pair-once launch: the j sums at zero, the next item to take
// the first.
__global__ __launch_bounds__(256) void k_sym_clear(uint4 *__restrict__ jacc, size_t n16,
                                                   uint32_t *__restrict__ next_item)
{
    const size_t i = blockIdx.x * (size_t)256 + threadIdx.x;
    if (i == 0) *next_item = 0u;
    if (i < n16) jacc[i] = make_uint4(0u, 0u, 0u, 0u);
}

// Each-pair-once result: own sums plus the fixed-point j sums, scaled to
// accelerations and scattered to original order.
__global__ void k_pp32_combine(const float4 *__restrict__ iacc,
                               const unsigned long long *__restrict__ jacc,
                               uint32_t n_sorted, const uint32_t *__restrict__ perm,
                               BoxView v, const P32 *__restrict__ p32s,
                               float4 *__restrict__ acc)
{
    int bi;
    uint32_t lb;
    if (!box_block(v, bi, lb)) return;
    const BoxDev &bx = v.box[bi];
    const uint32_t il = lb * 256 + threadIdx.x;
    if (il >= bx.n) return;
    const uint32_t i = bx.p0 + il;
    const double inv = p32s[bi].jinv;
    const float sc = p32s[bi].out_scale;
    const float4 a = iacc[i];
    const float x = a.x + (float)((double)(long long)jacc[i] * inv);
    const float y = a.y + (float)((double)(long long)jacc[(size_t)n_sorted + i] * inv);
    const float z = a.z + (float)((double)(long long)jacc[2 * (size_t)n_sorted + i] * inv);
    acc[perm[i]] = make_float4(x * sc, y * sc, z * sc, 0.f);
}

}  // namespace

namespace {

int build_active_tiles(const uint32_t *off, const uint32_t *perm, const int32_t *active_end,
                       int32_t ti_current, uint32_t n, const BoxSet &bs,
                       const ActiveTiles &at, hipStream_t s)
{
    const int shift3 = 3 * at.t.block_shift;
    const uint32_t nsuper = at.nkeys >> (shift3 + 3);
    if (nsuper == 0 || nsuper > at.t.nblocks || n > at.capacity) {
        set_error("active tiles: %u super-blocks / %u particles exceed capacity", nsuper, n);
        return CUCO_ERR_INVALID_ARG;
    }
    k_act_flags<<<grid_for(n, 256), 256, 0, s>>>(perm, active_end, ti_current, n, at.scan);
    CUCO_LAUNCH_CHECK();
    int rc = exclusive_scan_u32(at.scan, at.scan, n, at.nscratch, at.scan + n, s);
    if (rc) return rc;
    k_act_list<<<grid_for(n, 256), 256, 0, s>>>(at.scan, n, at.list);
    CUCO_LAUNCH_CHECK();
    k_block_tiles_act<<<grid_for(nsuper, 256), 256, 0, s>>>(off, at.scan, nsuper, shift3,
                                                            at.t.block_tiles);
    CUCO_LAUNCH_CHECK();
    rc = exclusive_scan_u32(at.t.block_tiles, at.t.block_tiles, nsuper, at.t.scan_scratch,
                            at.t.counters, s);
    if (rc) return rc;
    k_fill_tiles_act<<<grid_for(nsuper, 256), 256, 0, s>>>(off, at.scan, at.t.block_tiles,
                                                           nsuper, shift3, at.t.tile_start,
                                                           at.t.tile_count);
    CUCO_LAUNCH_CHECK();
    k_box_tiles<<<grid_for(bs.nboxes + 1, 64), 64, 0, s>>>(
        at.t.block_tiles, bs.view(kKeyMorton, kMapBrick), shift3, at.t.counters, at.tile_map);
    CUCO_LAUNCH_CHECK();
    return CUCO_OK;
}

}  // namespace

int launch_build_tiles(const uint32_t *off, uint32_t n, const BoxSet &bs, uint32_t nkeys,
                       TileInfo &t, hipStream_t s)
{
    const int shift3 = 3 * t.block_shift;
    const uint32_t nsuper = nkeys >> (shift3 + 3);
    // t.nblocks is the capacity (blocks of the smallest tunable shift).
    if (nsuper == 0 || nsuper > t.nblocks) {
        set_error("tile build: %u Morton super-blocks exceed capacity %u", nsuper, t.nblocks);
        return CUCO_ERR_INVALID_ARG;
    }
    if (t.run != 64u && t.run != 128u) {
        set_error("tile build: run length %u (64 or 128)", t.run);
        return CUCO_ERR_INVALID_ARG;
    }
    k_super_tiles<<<grid_for(nsuper, kSuperWaves), 64 * kSuperWaves, 0, s>>>(
        off, nsuper, t.block_shift, t.run, bs.view(kKeyMorton, kMapBrick), t.block_tiles, t.est,
        t.work, t.counters);
    CUCO_LAUNCH_CHECK();
    const int rc = exclusive_scan_u32(t.block_tiles, t.block_tiles, nsuper, t.scan_scratch,
                                      t.counters, s);
    if (rc) return rc;
    // One wave per super-block, and a thread for each of nboxes + 1 entries
    // (every box has a super-block).
    k_fill_tiles<<<grid_for(nsuper, 4), 256, 0, s>>>(
        off, t.block_tiles, nsuper, shift3, t.run, bs.view(kKeyMorton, kMapBrick), t.est, t.work,
        t.tile_start, t.tile_count, t.counters, t.parts, t.max_parts, bs.tile_map);
    CUCO_LAUNCH_CHECK();
    // A super-block of c particles has at most c / run + 8 tiles.
    t.most_tiles =
        (uint32_t)std::min<uint64_t>(t.max_tiles, (uint64_t)n / t.run + 8ull * nsuper);
    return CUCO_OK;
}

P32 make_p32(const PairParams &pp, const GridInfo &g, double uniform_mass,
             double mass_max, uint32_t n_box)
{
    const double sc = 4.0 * pp.asmthfac;  // quarter bins
    P32 p;
    p.s = (float)sc;
    p.rcut = (float)(pp.rcut * sc);
    p.rcut2 = (float)(pp.rcut2 * sc * sc);
    p.filter2 = (float)(pp.rcut2 * sc * sc * (1.0 + 1e-4));
    p.h = (float)(pp.h * sc);
    p.h_inv = (float)(1.0 / (pp.h * sc));
    p.h3_inv = p.h_inv * p.h_inv * p.h_inv;
    p.hnear = std::max(p.h, 1.0f);
    p.cellf = (float)(g.cell * sc);
    p.inv_cellf = (float)(1.0 / (g.cell * sc));
    p.eps = 1e-12f;
    p.out_scale = (float)(pp.G * sc * sc);
    p.mass = (float)uniform_mass;
    p.M = g.M;
    // Fixed-point scale of the each-pair-once j sums: a pair term is at most
    // m_max * 10.67 / h^2 (scaled units; the spline's peak, the table is <= 1),
    // so n such terms stay below 2^62 / scale.
    const double pair_max = std::max(mass_max, 1e-30) * 10.67 / ((double)p.h * p.h);
    const double bound = std::max(1.0, (double)n_box) * pair_max;
    int e2 = 0;
    std::frexp(std::ldexp(1.0, 62) / bound, &e2);
    p.jscale = (float)std::ldexp(1.0, std::min(e2 - 1, 126));
    p.jinv = 1.0f / p.jscale;
    return p;
}

bool pp32_table_cut(const PairParams &pp)
{
    // The table alone can make the cut when rcut sits on a bin edge; bins a
    // wide tile's candidates could reach past the LDS table are clamped per
    // tile in the kernel.
    const double edge = pp.asmthfac * pp.rcut;
    return fabs(edge - nearbyint(edge)) < 1e-9 * edge;
}

int launch_pp32(const float4 *spos, const uint32_t *skeys,
                const uint32_t *perm, const uint32_t *off, const BoxSet &bs,
                const P32 *p32s, bool table_cut, double uniform_mass,
                const float *table32, const TileInfo &t, float4 *acc,
                unsigned long long *cand_counter, int num_workgroups,
                const int32_t *active_end, int32_t ti_current,
                const PairSym &sym, const ActiveTiles *at, uint32_t n_sorted,
                hipStream_t s)
{
    if (bs.total[kMapPart] == 0) return CUCO_OK;
    const bool generic = !table_cut;
    const bool uniform = uniform_mass > 0;
    const float mass = (float)uniform_mass;
    const BoxView tv{bs.dev[kKeyMorton], bs.tile_map, bs.nboxes};
    int rc = CUCO_OK;
    const uint32_t full = num_workgroups > 0 ? (uint32_t)num_workgroups : 2048u;
    const uint32_t nwg = wave_tile_workgroups(t.most_tiles, kWaves, full);
    // Each pair once: all targets (not an active set).
    const bool symmetric = sym.on && sym.iacc && sym.jacc && !active_end;
    if (symmetric) {
        // Three planes of n_sorted 8-byte sums, rounded up to 16 bytes (the
        // allocation is).
        const size_t n16 = ((size_t)3 * sym.n_sorted + 1) / 2;
        k_sym_clear<<<(unsigned)((n16 + 255) / 256), 256, 0, s>>>(
            reinterpret_cast<uint4 *>(sym.jacc), n16, t.counters + 1);
        CUCO_LAUNCH_CHECK();
#define CUCO_SYM32(GENERIC, UNIFORM, TPL)                                               \
    k_pp32<GENERIC, UNIFORM, true, TPL><<<nwg, kThreads, 0, s>>>(                       \
        spos, skeys, perm, off, tv, p32s, mass, table32, t.tile_start, t.tile_count,    \
        t.counters, acc, cand_counter, nullptr, 0, sym.iacc, sym.jacc, sym.n_sorted,   \
        nullptr, t.coarse_cells, t.parts, t.max_parts)
        if (t.run == 64u && !cand_counter && n_sorted <= kTeamParticles) {
#define CUCO_TEAM32(GENERIC, UNIFORM)                                                   \
    k_pp32_team<GENERIC, UNIFORM><<<team_tile_workgroups(t.most_tiles, full), 64 * kTeam, 0, s>>>( \
        spos, skeys, off, tv, p32s, mass, table32, t.tile_start, t.tile_count,          \
        t.counters, sym.iacc, sym.jacc, sym.n_sorted, t.coarse_cells, t.parts, t.max_parts)
            if (generic) {
                if (uniform) CUCO_TEAM32(true, true); else CUCO_TEAM32(true, false);
            } else {
                if (uniform) CUCO_TEAM32(false, true); else CUCO_TEAM32(false, false);
            }
#undef CUCO_TEAM32
        } else if (t.run == 128u) {
            if (generic) {
                if (uniform) CUCO_SYM32(true, true, 2); else CUCO_SYM32(true, false, 2);
            } else {
                if (uniform) CUCO_SYM32(false, true, 2); else CUCO_SYM32(false, false, 2);
            }
        } else {
            if (generic) {
                if (uniform) CUCO_SYM32(true, true, 1); else CUCO_SYM32(true, false, 1);
            } else {
                if (uniform) CUCO_SYM32(false, true, 1); else CUCO_SYM32(false, false, 1);
            }
        }
#undef CUCO_SYM32
        CUCO_LAUNCH_CHECK();
        k_pp32_combine<<<xcd_grid(bs.total[kMapPart]), 256, 0, s>>>(
            sym.iacc, sym.jacc, sym.n_sorted, perm, bs.view(kKeyMorton, kMapPart), p32s, acc);
        CUCO_LAUNCH_CHECK();
        return CUCO_OK;
    }
    // Active set with its own tiles: every listed target is active.
    const bool packed = active_end && at;
    const TileInfo &tt = packed ? at->t : t;
    // The kernel that visits every ordered pair holds one target per lane.
    if (tt.run != 64u) {
        set_error("pair force: tiles of %u targets need the each-pair-once kernel", tt.run);
        return CUCO_ERR_INVALID_ARG;
    }
    if (!packed) {
        rc = launch_fill_u32(t.counters + 1, 0u, 1, s);
        if (rc) return rc;
    }
    const BoxView tva{bs.dev[kKeyMorton], packed ? at->tile_map : bs.tile_map, bs.nboxes};
    const int32_t *ae = packed ? nullptr : active_end;
    const uint32_t *tl = packed ? at->list : nullptr;
    if (packed) {
        rc = build_active_tiles(off, perm, active_end, ti_current, n_sorted, bs, *at, s);
        if (rc) return rc;
        rc = launch_fill_u32(at->t.counters + 1, 0u, 1, s);
        if (rc) return rc;
    }
#define CUCO_PP32(GENERIC, UNIFORM)                                                     \
    k_pp32<GENERIC, UNIFORM, false, 1><<<nwg, kThreads, 0, s>>>(                        \
        spos, skeys, perm, off, tva, p32s, mass, table32, tt.tile_start, tt.tile_count, \
        tt.counters, acc, cand_counter, ae, ti_current, nullptr, nullptr, 0u, tl, t.coarse_cells, nullptr, 0u)
    if (generic) {
        if (uniform) CUCO_PP32(true, true); else CUCO_PP32(true, false);
    } else {
        if (uniform) CUCO_PP32(false, true); else CUCO_PP32(false, false);
    }
#undef CUCO_PP32
    CUCO_LAUNCH_CHECK();
    return CUCO_OK;
}

}  // namespace cuco
