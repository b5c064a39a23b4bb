/*
 * near_lists.h -- neighbour lists of a wave's particles, built by the wave.
 *
 * The neighbour passes give a wave 64 / GL particles with GL lanes each.
 * Walking the cell boxes lane by lane leaves two lanes in three idle: cells
 * hold different numbers of particles and boxes different numbers of cells,
 * and every walk pays for the cell table and the addresses again.  Here the
 * wave first walks the union of its particles' boxes once, 64 candidates at
 * a time with every lane busy, tests each candidate against the particles
 * (their positions and radii are wave-uniform, in scalar registers) and
 * appends the slots inside a particle's radius to that particle's list in
 * LDS.  The passes then work on the lists, whose entries are dealt evenly to
 * the particle's lanes.
 */
#ifndef NEAR_LISTS_H
#define NEAR_LISTS_H

#include "sph_internal.h"

#include <type_traits>

struct Cells {
    const uint2* cell_se;
    float cell_size;
    int mask;
    /* the same for blocks of 2^3 and 4^3 cells, whose slots are consecutive
     * too (null where the grid has no such blocks) */
    const uint2* block_se[2];
};

/* One of the cell table's levels: cells (0) or blocks of 2^3 or 4^3. */
struct Level {
    const uint2* se;
    float size, inv;
    int mask;
};
constexpr int kLevels = 3;
__device__ __forceinline__ Level cell_level(const Cells& c, int level) {
    const float size = c.cell_size * (float)(1 << level);
    return Level{level == 0 ? c.cell_se : c.block_se[level - 1], size, 1.f / size, c.mask >> level};
}
/* The level to walk for a list of radius `reach`: blocks of at most about
 * three quarters of it, so that a box holds a few hundred cells or blocks at
 * most (a wave looks 64 up at a time) without many more candidates. */
__device__ __forceinline__ int near_level(const Cells& c, float reach) {
    const bool one = c.block_se[0] && reach >= 2.6f * c.cell_size;
    return one ? (c.block_se[1] && reach >= 5.2f * c.cell_size ? 2 : 1) : 0;
}

constexpr int kPerLane = 16; /* list entries per lane */

/* Data movement between lanes without LDS (DPP); lanes without a source,
 * or outside ROWS, read `old`. */
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ int dpp(int old, int v) {
    return __builtin_amdgcn_update_dpp(old, v, CTRL, ROWS, 0xF, false);
}
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ float dppf(float old, float v) {
    return __int_as_float(dpp<CTRL, ROWS>(__float_as_int(old), __float_as_int(v)));
}
constexpr int kQuadXor1 = 0xB1, kQuadXor2 = 0x4E, kHalfMirror = 0x141, kRowRor8 = 0x128;
constexpr int kRowShr1 = 0x111, kRowShr2 = 0x112, kRowShr4 = 0x114, kRowShr8 = 0x118;
constexpr int kBcast15 = 0x142, kBcast31 = 0x143;

/* Sum and maximum over a particle's GL lanes (8, 16, 32, 64), the same bits
 * in each. */
template <int GL>
__device__ __forceinline__ float lanes_sum(float v) {
    v += dppf<kQuadXor1>(0.f, v);
    v += dppf<kQuadXor2>(0.f, v);
    v += dppf<kHalfMirror>(0.f, v);
    if constexpr (GL >= 16) v += dppf<kRowRor8>(0.f, v);
    if constexpr (GL >= 32) v += __shfl_xor(v, 16, 64);
    if constexpr (GL >= 64) v += __shfl_xor(v, 32, 64);
    return v;
}
template <int GL>
__device__ __forceinline__ int lanes_sum(int v) {
    v += dpp<kQuadXor1>(0, v);
    v += dpp<kQuadXor2>(0, v);
    v += dpp<kHalfMirror>(0, v);
    if constexpr (GL >= 16) v += dpp<kRowRor8>(0, v);
    if constexpr (GL >= 32) v += __shfl_xor(v, 16, 64);
    if constexpr (GL >= 64) v += __shfl_xor(v, 32, 64);
    return v;
}
template <int GL>
__device__ __forceinline__ float lanes_max(float v) {
    v = fmaxf(v, dppf<kQuadXor1>(v, v));
    v = fmaxf(v, dppf<kQuadXor2>(v, v));
    v = fmaxf(v, dppf<kHalfMirror>(v, v));
    if constexpr (GL >= 16) v = fmaxf(v, dppf<kRowRor8>(v, v));
    if constexpr (GL >= 32) v = fmaxf(v, __shfl_xor(v, 16, 64));
    if constexpr (GL >= 64) v = fmaxf(v, __shfl_xor(v, 32, 64));
    return v;
}
/* Minimum over the wave of a value that is the same in each aligned group
 * of 8 lanes, as a wave-uniform scalar. */
__device__ __forceinline__ float groups_min(float v) {
    v = fminf(v, dppf<kRowRor8>(v, v));
    v = fminf(v, dppf<kBcast15, 0xA>(v, v));
    v = fminf(v, dppf<kBcast31, 0xC>(v, v));
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
__device__ __forceinline__ int groups_min_i(int v) {
    v = min(v, dpp<kRowRor8>(v, v));
    v = min(v, dpp<kBcast15, 0xA>(v, v));
    v = min(v, dpp<kBcast31, 0xC>(v, v));
    return __builtin_amdgcn_readlane(v, 63);
}
/* Inclusive sum and maximum (of values >= 0) over the lanes up to this one. */
__device__ __forceinline__ int scan_add(int v) {
    v += dpp<kRowShr1>(0, v);
    v += dpp<kRowShr2>(0, v);
    v += dpp<kRowShr4>(0, v);
    v += dpp<kRowShr8>(0, v);
    v += dpp<kBcast15, 0xA>(0, v);
    return v + dpp<kBcast31, 0xC>(0, v);
}
__device__ __forceinline__ int scan_max(int v) {
    v = max(v, dpp<kRowShr1>(0, v));
    v = max(v, dpp<kRowShr2>(0, v));
    v = max(v, dpp<kRowShr4>(0, v));
    v = max(v, dpp<kRowShr8>(0, v));
    v = max(v, dpp<kBcast15, 0xA>(0, v));
    return max(v, dpp<kBcast31, 0xC>(0, v));
}
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float lane_f(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
/* LDS accesses of one wave complete in order: this only keeps the compiler
 * from moving them. */
__device__ __forceinline__ void lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

/* The walk's: marks of a window, and a queue of cells that hold particles. */
struct WalkLds {
    int32_t mark[64];
    uint2 se[128];
    int32_t tag[128];
};

/* The lists of P particles with GL lanes each (P = 64 / GL, or 1: every group
 * of lanes works on the same one).  S = 0: kPerLane entries per lane, and 64
 * more places that a window may spill into.  S > 0 (the cell walk's order,
 * deal_bins): GL S bins, S of them a lane's; a bin's first kRows entries are
 * kept in registers; the others, up to kBin, are read again for every scan
 * (where a box is 8 cells wide in z, say, a bin of 8 is a slab of the box and
 * may hold a third of the list). */
struct NoWalk {};
template <int GL, int S, int P, bool BINS = (S > 0), bool WALK = true>
struct NearLds {
    static constexpr int kCap = GL * kPerLane, kRows = kPerLane;
    int32_t slot[P][kCap + 64];
    typename std::conditional<WALK, WalkLds, NoWalk>::type walk;
};
template <int GL, int S, int P, bool WALK>
struct NearLds<GL, S, P, true, WALK> {
    static constexpr int kCap = P == 1 ? 768 : (GL <= 8 ? 160 : 224);
    static constexpr int kRows = (P == 1 ? 64 : (S <= 1 ? 28 : 32)) / S; /* (a multiple of 4) */
    static constexpr int kBin = P == 1 ? 192 / S : (S <= 1 ? 64 : (S > 2 ? 14 : (GL > 8 ? 24 : 40)));
    /* one bin of each lane's may hold so many more: where the cells are wide
     * (3 h or more) most of a particle's neighbours lie in a few of them */
    static constexpr int kOver = P > 1 && (S > 2 || (S == 2 && GL > 8)) ? 40 : 0;
    using Place = typename std::conditional<(kCap > 255), uint16_t, uint8_t>::type;
    int32_t slot[P][kCap];
    /* the entries' cells, 5 bits an axis, counted from the walk's first */
    uint16_t cell[P][kCap];
    union {
        struct {
            /* the entries' bins (a byte each, in an order that turns a byte
             * compare into a mask of entries), and each bin's entries in list
             * order */
            uint32_t bin[P][kCap / 4];
            Place row[S * kBin + kOver][64];
        };
        typename std::conditional<WALK, WalkLds, NoWalk>::type walk; /* while the lists are built */
    };
};

/* A candidate's place in a list of c entries, for the lanes of m. */
__device__ __forceinline__ int list_place(uint64_t m, int c) {
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, (unsigned)c));
}

/* A cell's place counted from a walk's first, 5 bits an axis. */
__device__ __forceinline__ int cell_place(int ix, int iy, int iz) { return (ix & 31) | (iy & 31) << 5 | (iz & 31) << 10; }

/* From this many cells on the walk queues those with particles.  The queue
 * costs a trip through LDS per 64 cells; without it every 64 cells take a
 * window of their own, however few particles they hold.  The density and
 * acceleration pass with and without, ms, at 2e4 (80 look-ups of 64 cells per
 * wave) 0.30 + 0.20 and 0.41 + 0.30, at 1e5 (24) 0.82 + 0.30 and 0.87 + 0.35, at
 * 1e6 (4) 6.19 + 1.07 and 5.80 + 1.01. */
constexpr int kQueueFrom = 512;

/* Calls body(k, record, valid, tag) with a candidate slot, its record and
 * its cell's tag per lane for every particle of nx x ny x nz cells from mn on,
 * 64 at a time in cell order.  tag_of(ix, iy, iz), counted from mn, is a
 * cell's tag, or negative to drop it.  The lanes look 64 cells up and a queue
 * keeps those that hold particles; for 64 of them a prefix sum of their counts
 * and a running maximum over marks at their first candidates tell each lane
 * which cell its candidate is of, so that the candidates of any number of
 * cells of any size fill the wave.  The next window's records are requested
 * before body works on this one's. */
template <class Tag, class Body>
__device__ __forceinline__ void wave_candidates(const Level& cells, const float4* __restrict__ spos, const int mn[3], int nx,
                                                int ny, int nz, WalkLds& lds, Tag tag_of, Body body) {
    const int lane = (int)(threadIdx.x & 63);
    const int ncell = nx * ny * nz;
    const float inz = 1.f / (float)nz, iny = 1.f / (float)ny;
    const bool small = ncell <= 1 << 18;
    int next_tag = -1;
    uint2 next_se = make_uint2(0xFFFFFFFFu, 0u);
    auto look_up = [&](int c) {
        /* the divisions through FP32 are exact while the rounding of the
         * quotient, 2^-22 of it, stays under half a step, 1 / (2 n) */
        const int t = small ? (int)(((float)c + 0.5f) * inz) : c / nz, iz = c - t * nz;
        const int ix = small ? (int)(((float)t + 0.5f) * iny) : t / ny, iy = t - ix * ny;
        next_se = make_uint2(0xFFFFFFFFu, 0u);
        next_tag = c < ncell ? tag_of(ix, iy, iz) : -1;
        if (next_tag >= 0)
            next_se = cells.se[dev_expand_bits((uint32_t)((mn[0] + ix) & cells.mask)) |
                               (dev_expand_bits((uint32_t)((mn[1] + iy) & cells.mask)) << 1) |
                               (dev_expand_bits((uint32_t)((mn[2] + iz) & cells.mask)) << 2)];
    };
    const bool queue = ncell > kQueueFrom;
    int head = 0, queued = 0; /* the queue's first cell and its length */
    look_up(lane);
    for (int base = 0; base < ncell || queued > 0; base += 64) {
        /* the next cells' ranges are requested before these are used */
        uint2 se = next_se;
        int own = next_tag;
        if (base + 64 < ncell) look_up(base + 64 + lane);
        bool some = se.x != 0xFFFFFFFFu && base < ncell;
        if (queue) {
            const uint64_t m = __ballot(some);
            if (some) {
                const int at = (head + queued + list_place(m, 0)) & 127;
                lds.se[at] = se;
                lds.tag[at] = own;
            }
            queued += (int)__popcll(m);
            if (queued < 64 && base + 64 < ncell) continue;
            lds_order();
            const int at = (head + lane) & 127;
            some = lane < queued;
            se = lds.se[at];
            own = lds.tag[at];
            head += 64;
            queued = max(queued - 64, 0);
        }
        const int cnt = some ? (int)(se.y - se.x + 1u) : 0;
        const int incl = scan_add(cnt), excl = incl - cnt;
        const int total = __builtin_amdgcn_readlane(incl, 63);
        if (total == 0) continue;
        const int shift = (int)se.x - excl; /* slot = flat index + shift of its cell's lane */
        int tag;
        auto slot_at = [&](int w) {
            lds.mark[lane] = 0;
            lds_order();
            const int at = max(excl - w, 0);
            if (cnt > 0 && incl > w && at < 64) lds.mark[at] = lane;
            lds_order();
            const int src = scan_max(lds.mark[lane]);
            lds_order();
            /* the lanes past the last candidate repeat it */
            const int f = min(w + lane, total - 1);
            tag = __builtin_amdgcn_ds_bpermute(4 * src, own);
            return f + __builtin_amdgcn_ds_bpermute(4 * src, shift);
        };
        int k = slot_at(0);
        float4 q = spos[k];
        for (int w = 0; w < total; w += 64) {
            const int k0 = k, tag0 = tag;
            const float4 q0 = q;
            if (w + 64 < total) {
                k = slot_at(w + 64);
                q = spos[k];
            }
            body(k0, q0, w + lane < total, tag0);
        }
    }
}

/* The cells that hold every particle within `reach` of some particle of the
 * lanes with `mine`, and which of them to keep. */
struct NearBox {
    int mn[3], nc[3];
    float inlo[3], inhi[3], rr, cs;
    bool whole;
    __device__ __forceinline__ int tag(int ix, int iy, int iz) const {
        const int cx = mn[0] + ix, cy = mn[1] + iy, cz = mn[2] + iz;
        const float gx = fmaxf(fmaxf(inlo[0] - (float)(cx + 1) * cs, (float)cx * cs - inhi[0]), 0.f);
        const float gy = fmaxf(fmaxf(inlo[1] - (float)(cy + 1) * cs, (float)cy * cs - inhi[1]), 0.f);
        const float gz = fmaxf(fmaxf(inlo[2] - (float)(cz + 1) * cs, (float)cz * cs - inhi[2]), 0.f);
        return whole || gx * gx + gy * gy + gz * gz <= rr ? cell_place(ix, iy, iz) : -1;
    }
};
__device__ __forceinline__ NearBox near_box(const Level& cells, bool mine, float x, float y, float z, float reach, float& ratio) {
    const float big = 3.0e38f;
    const float dim = (float)(cells.mask + 1);
    const float rmax = -groups_min(mine ? -reach : big), rmin = groups_min(mine ? reach : big);
    const float xyz[3] = {x, y, z};
    NearBox b;
    b.cs = cells.size;
    b.rr = rmax * rmax * 1.0002f;
    b.whole = false;
    const float iown = 1.f / fminf(2.f * rmax * cells.inv + 2.f, dim);
    ratio = 1.f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float lo = groups_min(mine ? xyz[k] - reach : big), hi = -groups_min(mine ? -(xyz[k] + reach) : big);
        /* the pad covers the rounding of the coordinates that the cells were
         * assigned by; the particles lie in [inlo, inhi] */
        const float pad = 1e-3f * cells.size + 5e-7f * (fabsf(lo) + fabsf(hi));
        b.mn[k] = uniform((int)floorf((lo - pad) * cells.inv));
        b.nc[k] = uniform((int)floorf((hi + pad) * cells.inv)) - b.mn[k] + 1;
        if (b.nc[k] > cells.mask + 1) { /* the periodic grid once */
            b.nc[k] = cells.mask + 1;
            b.whole = true;
        }
        ratio *= (float)b.nc[k] * iown;
        b.inlo[k] = lo + rmin - pad;
        b.inhi[k] = hi - rmin + pad;
    }
    return b;
}

/* Calls body(k, record, valid, place) for every candidate near one particle,
 * at a wave-uniform (x, y, z): every particle within `reach`, and others. */
template <class Body>
__device__ __forceinline__ NearBox wave_near(const Level& cells, const float4* __restrict__ spos, float x, float y, float z,
                                             float reach, WalkLds& lds, Body body) {
    float ratio;
    const NearBox b = near_box(cells, true, x, y, z, reach, ratio);
    wave_candidates(cells, spos, b.mn, b.nc[0], b.nc[1], b.nc[2], lds,
                    [&](int ix, int iy, int iz) { return b.tag(ix, iy, iz); }, body);
    return b;
}

/* Neighbour lists of the wave's P particles: particle p, of lane GL p, sits at
 * (x, y, z); the slots of the candidates within `reach` go to
 * l.slot[p][0..cnt[p]), in the order of the level's cells (cnt[p] may exceed
 * kCap: then only the first kCap are sure to be there).  A particle with
 * reach < 0 keeps its list and count.  A particle's list depends on its
 * position, reach and level alone, not on the particles that share its wave.
 * The particles are built together from the union of their boxes; when they
 * are spread out, each from its own: a candidate of the union costs about 25
 * instructions and 10 per particle, so that eight boxes alone cost less from
 * a union of 2.5 of them on.  S > 0 also keeps the candidates' cells, counted
 * from `first` (set for the lanes of the built particles); a box as wide as
 * the periodic grid, where a cell has two places, counts as too long. */
template <int GL, int S, int P>
__device__ __forceinline__ void build_near_lists(const Level& cells, const float4* __restrict__ spos, float x, float y,
                                                 float z, float reach, NearLds<GL, S, P>& l, int (&cnt)[P],
                                                 int (&first)[3]) {
    constexpr int kCap = NearLds<GL, S, P>::kCap;
    const uint64_t asked = __ballot(reach >= 0.f);
    auto append = [&](int p, bool hit, int k, int cell, int& c) {
        const uint64_t m = __ballot(hit);
        if constexpr (S == 0) {
            const int at = list_place(m, min(c, kCap));
            if (hit) l.slot[p][at] = k;
        } else {
            const int at = list_place(m, c);
            if (hit && at < kCap) {
                l.slot[p][at] = k;
                l.cell[p][at] = (uint16_t)cell;
            }
        }
        c += (int)__popcll(m);
    };
    float ratio;
    const NearBox b = near_box(cells, reach >= 0.f, x, y, z, reach, ratio);
    const float reach2 = reach * reach;
    if ((S == 0 && P == 1) || (ratio <= 2.5f && !b.whole)) {
        float px[P], py[P], pz[P], pr2[P];
#pragma unroll
        for (int p = 0; p < P; ++p) {
            px[p] = lane_f(x, GL * p);
            py[p] = lane_f(y, GL * p);
            pz[p] = lane_f(z, GL * p);
            pr2[p] = lane_f(reach2, GL * p);
            if ((asked >> (GL * p)) & 1ull) cnt[p] = 0;
        }
        wave_candidates(cells, spos, b.mn, b.nc[0], b.nc[1], b.nc[2], l.walk,
                        [&](int ix, int iy, int iz) { return b.tag(ix, iy, iz); },
                        [&](int k, float4 q, bool valid, int cell) {
            if (!valid) q.x = 3.0e38f;
#pragma unroll
            for (int p = 0; p < P; ++p) {
                if (((asked >> (GL * p)) & 1ull) == 0ull) continue;
                const float dx = q.x - px[p], dy = q.y - py[p], dz = q.z - pz[p];
                append(p, fmaf(dx, dx, fmaf(dy, dy, dz * dz)) <= pr2[p], k, cell, cnt[p]);
            }
        });
        if (S > 0 && reach >= 0.f)
#pragma unroll
            for (int j = 0; j < 3; ++j) first[j] = b.mn[j];
    } else {
        for (int p = 0; p < P; ++p) {
            if (((asked >> (GL * p)) & 1ull) == 0ull) continue;
            const float px = lane_f(x, GL * p), py = lane_f(y, GL * p), pz = lane_f(z, GL * p);
            const float rp = lane_f(reach, GL * p), rp2 = lane_f(reach2, GL * p);
            int c = 0;
            const NearBox own = wave_near(cells, spos, px, py, pz, rp, l.walk, [&](int k, float4 q, bool valid, int cell) {
                const float dx = q.x - px, dy = q.y - py, dz = q.z - pz;
                append(p, valid && fmaf(dx, dx, fmaf(dy, dy, dz * dz)) <= rp2, k, cell, c);
            });
            if (S > 0 && own.whole) c = kCap + 1;
#pragma unroll
            for (int j = 0; j < P; ++j) cnt[j] = j == p ? c : cnt[j];
            if (S > 0 && (P == 1 || (int)(threadIdx.x & 63) / GL == p))
#pragma unroll
                for (int j = 0; j < 3; ++j) first[j] = own.mn[j];
        }
    }
    lds_order();
}

/* Whether a candidate is no pair of a particle's (beyond 2 h of both, or the
 * particle itself): the acceleration walk's own test, form for form. */
__device__ __forceinline__ bool pair_skip(float4 q, float px, float py, float pz, float pi2x4, float qj2x4) {
    const float dx = px - q.x, dy = py - q.y, dz = pz - q.z;
    const float r2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
    return (r2 > pi2x4 && r2 > qj2x4) || r2 < 1e-12f;
}

/* Lists of the pairs of the acceleration pass for the wave's P particles of
 * LANES lanes each: the candidates of the particle's own cell box [mn, mx]
 * (empty: none) within 2 h of either side, in the order of the cells.  The
 * union of the boxes is walked once where it is less than 2.5 of the largest
 * (and no wider than the periodic grid), each box alone otherwise.  ny, nz and
 * off are those of deal_bins for the lane's particle. */
template <int LANES, int P, class Lds>
__device__ __forceinline__ void build_pair_lists(const Level& cells, const float4* __restrict__ s_posh, float4 xi,
                                                 const int mn[3], const int mx[3], Lds& l, WalkLds& walk, int (&cnt)[P], int& ny,
                                                 int& nz, int& off) {
    constexpr int kCap = Lds::kCap;
    constexpr bool kSpill = sizeof(l.slot[0]) / sizeof(l.slot[0][0]) > kCap;
    int nc[3];
    float own = 1.f, ratio = 1.f;
    int umn[3], unc[3];
    const bool some = mx[0] >= mn[0] && mx[1] >= mn[1] && mx[2] >= mn[2];
    bool wide = false;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        nc[k] = mx[k] - mn[k] + 1;
        own *= (float)nc[k];
        umn[k] = groups_min_i(some ? mn[k] : 0x7FFFFFFF);
        unc[k] = -groups_min_i(some ? -mx[k] : 0x7FFFFFFF) - umn[k] + 1;
        wide = wide || unc[k] > cells.mask + 1;
        ratio *= (float)unc[k];
    }
    const uint64_t asked = __ballot(some);
#pragma unroll
    for (int p = 0; p < P; ++p) cnt[p] = 0;
    ny = nc[1];
    nz = nc[2];
    off = 0;
    if (asked == 0ull) return;
    const float hi2x4 = xi.w * xi.w * 4.f;
    auto append = [&](int p, bool hit, int k, int place, int& c) {
        const uint64_t m = __ballot(hit);
        const int at = list_place(m, kSpill ? min(c, kCap) : c);
        if (hit && (kSpill || at < kCap)) {
            l.slot[p][at] = k;
            if constexpr (!kSpill) l.cell[p][at] = (uint16_t)place;
        }
        c += (int)__popcll(m);
    };
    if (!wide && ratio <= -2.5f * groups_min(some ? -own : 0.f)) {
        float px[P], py[P], pz[P], ph[P];
        int pmn[P][3], pnc[P][3];
#pragma unroll
        for (int p = 0; p < P; ++p) {
            px[p] = lane_f(xi.x, LANES * p);
            py[p] = lane_f(xi.y, LANES * p);
            pz[p] = lane_f(xi.z, LANES * p);
            ph[p] = lane_f(hi2x4, LANES * p);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                pmn[p][k] = __builtin_amdgcn_readlane(mn[k], LANES * p) - umn[k];
                pnc[p][k] = __builtin_amdgcn_readlane(some ? nc[k] : 0, LANES * p);
            }
        }
        wave_candidates(cells, s_posh, umn, unc[0], unc[1], unc[2], walk,
                        [&](int ix, int iy, int iz) {
            int m = 0;
#pragma unroll
            for (int p = 0; p < P; ++p)
                m |= ((unsigned)(ix - pmn[p][0]) < (unsigned)pnc[p][0] && (unsigned)(iy - pmn[p][1]) < (unsigned)pnc[p][1] &&
                      (unsigned)(iz - pmn[p][2]) < (unsigned)pnc[p][2]) ? 1 << p : 0;
            return m == 0 ? -1 : m << 15 | cell_place(ix, iy, iz);
        }, [&](int k, float4 q, bool valid, int tag) {
            const float qj2x4 = q.w * q.w * 4.f;
            if (!valid) tag = 0;
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const bool in = (tag & (1 << (15 + p))) != 0;
                if (__any(in)) append(p, in && !pair_skip(q, px[p], py[p], pz[p], ph[p], qj2x4), k, tag & 0x7FFF, cnt[p]);
            }
        });
        off = ((umn[0] - mn[0]) * ny + (umn[1] - mn[1])) * nz + (umn[2] - mn[2]);
    } else {
        for (int p = 0; p < P; ++p) {
            if (((asked >> (LANES * p)) & 1ull) == 0ull) continue;
            const float px = lane_f(xi.x, LANES * p), py = lane_f(xi.y, LANES * p), pz = lane_f(xi.z, LANES * p);
            const float ph = lane_f(hi2x4, LANES * p);
            int m[3], n[3], c = 0;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                m[k] = __builtin_amdgcn_readlane(mn[k], LANES * p);
                n[k] = __builtin_amdgcn_readlane(nc[k], LANES * p);
            }
            wave_candidates(cells, s_posh, m, n[0], n[1], n[2], walk, cell_place,
                            [&](int k, float4 q, bool valid, int tag) {
                append(p, valid && !pair_skip(q, px, py, pz, ph, q.w * q.w * 4.f), k, tag, c);
            });
#pragma unroll
            for (int j = 0; j < P; ++j) cnt[j] = j == p ? c : cnt[j];
        }
    }
    lds_order();
}

/* The row of the e-th entry of a lane's k-th bin. */
template <int S, class Lds>
__device__ __forceinline__ int bin_row(int k, int e) {
    return Lds::kOver > 0 && e >= Lds::kBin ? (S - 1) * Lds::kBin + e : k * Lds::kBin + e;
}

/* The order of the sums of the cell walk with G = GL S lanes per particle:
 * there lane b sums the candidates of cells b, b + G, ... of the particle's
 * box in order, and the lanes' sums are added in a fixed tree.  This deals a
 * list's entries to the same G bins, bins b, b + GL, ... to the particle's
 * lane b, so that the same terms are added in the same order, bit for bit.
 * The bin of an entry is its cell's position in the box, modulo G, which
 * changes with the box: `ny`, `nz` are the box's cells in y and z and `off`
 * the position, in it, of the cell that the list's cells are counted from.
 * (An entry outside the box is beyond 2h: it adds 0 to whichever bin.)
 * n[k] = entries of the lane's k-th bin, all of them kept (bin_row); 0 for a
 * bin with more than there is room for, of which nothing may be read, and then
 * true. */
template <int GL, int S, int P, class Lds>
__device__ __forceinline__ bool deal_bins(Lds& l, int have, int longest, int ny, int nz, int off, int (&n)[S]) {
    constexpr uint32_t kNone = 0x40u, kMask = GL * S - 1;
    static_assert(GL * S <= 32, "cells are kept modulo 32");
    const int lane = (int)(threadIdx.x & 63), gl = lane % GL, g = P == 1 ? 0 : lane / GL;
    uint8_t* bytes = reinterpret_cast<uint8_t*>(l.bin[g]);
    /* entry 32 W + p in byte p / 8 of word 8 W + p % 8 */
    auto byte_at = [](int i) { return (i & ~31) + ((i & 7) << 2) + ((i >> 3) & 3); };
    const int words = (longest + 31) / 32;
    const int sx = (ny * nz) & kMask, sy = nz & kMask;
#pragma unroll 4
    for (int i = gl; i < words * 32; i += GL) {
        uint32_t bin = kNone;
        if (i < have) {
            const int c = l.cell[g][i];
            bin = (uint32_t)(__mul24(c & 31, sx) + __mul24((c >> 5) & 31, sy) + (c >> 10) + off) & kMask;
        }
        bytes[byte_at(i)] = (uint8_t)bin;
    }
    lds_order();
    uint32_t c = 0; /* entries of the lane's bins so far, a byte each */
    [[maybe_unused]] int over = -1; /* the bin that goes on past the others' rows */
    constexpr uint32_t kLane = (kNone | (GL - 1)) * 0x01010101u;
    const uint32_t mine = (uint32_t)gl * 0x01010101u;
    for (int w = 0; w < words; ++w) {
        uint32_t m = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const uint32_t v = (l.bin[g][8 * w + k] ^ mine) & kLane; /* zero byte: a bin of this lane's */
            m |= (~(v + 0x7F7F7F7Fu) & 0x80808080u) >> (7 - k);
        }
        while (__any(m != 0u)) {
            if (m != 0u) {
                const int i = 32 * w + __ffs((int)m) - 1;
                m &= m - 1u;
                const int k = S > 1 ? (int)(bytes[byte_at(i)] / GL) : 0;
                const int at = (int)((c >> (8 * k)) & 255u);
                if (at < Lds::kBin) l.row[k * Lds::kBin + at][lane] = (typename Lds::Place)i;
                else if constexpr (Lds::kOver > 0) {
                    if (over < 0) over = k;
                    if (over == k && at < Lds::kBin + Lds::kOver)
                        l.row[(S - 1) * Lds::kBin + at][lane] = (typename Lds::Place)i;
                }
                if (at < 255) c += 1u << (8 * k);
            }
        }
    }
    lds_order();
    bool full = false;
#pragma unroll
    for (int k = 0; k < S; ++k) {
        n[k] = (int)((c >> (8 * k)) & 255u);
        if (n[k] > Lds::kBin + (over == k ? Lds::kOver : 0)) {
            n[k] = 0;
            full = true;
        }
    }
    return full;
}

/* The cell walk's tree over its G = GL S lanes (distances G/2, ..., 1); no
 * product is drawn into its additions. */
template <int GL, int S>
__device__ __forceinline__ float bins_sum(const float (&v)[S]) {
#pragma clang fp contract(off)
    float t = S == 4 ? (v[0] + v[2 % S]) + (v[1 % S] + v[3 % S]) : (S == 2 ? v[0] + v[1 % S] : v[0]);
    if constexpr (GL == 16) t += dppf<kRowRor8>(0.f, t);
    /* lanes 4 apart within 8: up for the low half, down for the high */
    const float x = dppf<0x104>(0.f, t), y = dppf<0x114>(0.f, t); /* row_shl 4, row_shr 4 */
    t += (threadIdx.x & 4) ? y : x;
    t += dppf<kQuadXor2>(0.f, t);
    return t + dppf<kQuadXor1>(0.f, t);
}
/* Maximum over the wave of a value >= 0. */
__device__ __forceinline__ int wave_max(int v) { return __builtin_amdgcn_readlane(scan_max(v), 63); }

#endif
