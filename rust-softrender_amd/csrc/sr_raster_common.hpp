// sr_raster_common.hpp — device helpers shared by the raster kernels
// (sr_raster.hip, sr_raster_fmt.hip): the reference's screen tile grid,
// uniform loads through the scalar cache, and the triangle record as the
// per-triangle loop reads it.
#pragma once

#include "sr_device.hpp"

namespace sr {

// Screen tile grid of the reference (fragment.rs:188-216): column j spans
// [j*tw, min((j+1)*tw, W-1)], rows likewise; both ends inclusive.
__device__ __forceinline__ void sem_range(uint32_t lo_px, uint32_t hi_px, uint32_t t, uint32_t n,
                                          uint32_t& jlo, uint32_t& jhi) {
    // tiles whose inclusive span meets [lo_px, hi_px]
    const uint32_t a = (lo_px + t - 1) / t;  // ceil(lo/t)
    jlo = a > 0 ? a - 1 : 0;
    jhi = hi_px / t;
    if (jhi > n - 1) jhi = n - 1;
}

// Loads through the constant address space: read-only for the kernel's
// lifetime, so a wave-uniform address becomes an s_load into SGPRs.
__device__ __forceinline__ uint32_t load_item(const uint32_t* base, uint32_t i) {
#if defined(__HIP_DEVICE_COMPILE__)
    return ((const __attribute__((address_space(4))) uint32_t*)base)[i];
#else
    return base[i];
#endif
}

// 64 consecutive item ids, lane k holding the id at position c0 + k, the
// position clamped into [beg, end) (beg < end) so every lane loads.
__device__ __forceinline__ uint32_t load_ids(const uint32_t* items, uint32_t c0, uint32_t beg,
                                             uint32_t end, int lane) {
    const uint32_t c = min(max(c0 + (uint32_t)lane, beg), end - 1);
#if defined(__HIP_DEVICE_COMPILE__)
    return ((const __attribute__((address_space(1))) uint32_t*)items)[c];
#else
    return items[c];
#endif
}

// Execution tiles per bin, and tile `t` of a draw (tiles numbered bin by bin,
// row-major within a bin): its bin and its first pixel.
template <int ETS>
struct BinTiles {
    static constexpr uint32_t PER_ROW = BIN_EDGE / ETS, N = PER_ROW * PER_ROW;
};
template <int ETS>
__device__ __forceinline__ void tile_origin(const RasterParams& P, uint32_t t, uint32_t& bin, uint32_t& x,
                                            uint32_t& y) {
    constexpr uint32_t R = BinTiles<ETS>::PER_ROW;
    bin = t / BinTiles<ETS>::N;
    const uint32_t sub = t % BinTiles<ETS>::N;
    x = (bin % P.nbx) * BIN_EDGE + (sub % R) * ETS;
    y = (bin / P.nbx) * BIN_EDGE + (sub / R) * ETS;
}

// The key bits of the 8x8 tiles in a region of rw x rh pixels at (x, y)
// inside one bin.
__device__ __forceinline__ uint32_t region_bits(int x, int y, int rw, int rh) {
    const uint32_t cols = ((1u << (rw / 8)) - 1u) << ((x >> 3) & 3);
    uint32_t m = 0;
    for (int r = 0; r < rh / 8; r++) m |= cols << (4 * (((y >> 3) & 3) + r));
    return m;
}

// 256 consecutive values, lane k holding those at positions c0 + 4k .. + 3
// (c0 a multiple of 4; whole 16-byte words, the last at or before the one
// that holds position end - 1).
__device__ __forceinline__ uint4 load_ids4(const uint32_t* items, uint32_t c0, uint32_t end, int lane) {
    const uint32_t q = min((c0 >> 2) + (uint32_t)lane, (end - 1u) >> 2);
#if defined(__HIP_DEVICE_COMPILE__)
    typedef uint32_t V4 __attribute__((ext_vector_type(4)));
    const V4 v = ((const __attribute__((address_space(1))) V4*)items)[q];
    return make_uint4(v.x, v.y, v.z, v.w);
#else
    return ((const uint4*)items)[q];
#endif
}

// The fields of a triangle record the raster loop reads.
struct RecLane {
    double R;
    uint32_t zs;  // bit 0: strip flag; the rest: depth bound key (TriRec::zs)
    float x3, y3, e23y, e23x, e31y, e31x, z1, z2, z3;
    int X0, X1, Y0, Y1;
};

__device__ __forceinline__ uint32_t lane_u32(uint32_t v, int k) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, k);
}
__device__ __forceinline__ float lane_f32(uint32_t v, int k) {
    return __builtin_bit_cast(float, lane_u32(v, k));
}

// Record `id` through the scalar cache: `id` is wave-uniform, so these
// become scalar loads into SGPRs.
__device__ __forceinline__ RecLane rec_s(const TriRec* tris, uint32_t id) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef const __attribute__((address_space(4))) TriRec CRec;
    const CRec* p = (const CRec*)tris + id;
    RecLane r;
    r.R = p->R;
    r.zs = p->zs;
    r.x3 = p->x3; r.y3 = p->y3;
    r.e23y = p->e23y; r.e23x = p->e23x; r.e31y = p->e31y; r.e31x = p->e31x;
    r.z1 = p->z1; r.z2 = p->z2; r.z3 = p->z3;
    r.X0 = p->X0; r.X1 = p->X1; r.Y0 = p->Y0; r.Y1 = p->Y1;
    return r;
#else
    const TriRec& t = tris[id];
    return RecLane{t.R, t.zs, t.x3, t.y3, t.e23y, t.e23x, t.e31y, t.e31x, t.z1, t.z2, t.z3, t.X0, t.X1, t.Y0, t.Y1};
#endif
}

// The box of record `id` into rc (scalar loads).
__device__ __forceinline__ void rec_box(const TriRec* tris, uint32_t id, RecLane& rc) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef const __attribute__((address_space(4))) TriRec CRec;
    const CRec* p = (const CRec*)tris + id;
    rc.X0 = p->X0; rc.X1 = p->X1; rc.Y0 = p->Y0; rc.Y1 = p->Y1;
#else
    const TriRec& t = tris[id];
    rc.X0 = t.X0; rc.X1 = t.X1; rc.Y0 = t.Y0; rc.Y1 = t.Y1;
#endif
}

// Lane k copies bytes 0-47 of record ids[k] into stage chunks 0-2 (stage[c
// * 64 + k]) by three 16-byte LDS DMA loads (no registers in between).
__device__ __forceinline__ void stage_records(const TriRec* tris, uint32_t id, uint4* stage) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(3))) void LVoid;
    const char* src = (const char*)(tris + id);
#pragma unroll
    for (int c = 0; c < 3; c++)
        __builtin_amdgcn_global_load_lds((const void*)(src + 16 * c), (LVoid*)(stage + 64 * c), 16, 0, 0);
#else
    for (int c = 0; c < 3; c++) stage[64 * c] = ((const uint4*)(tris + id))[c];
#endif
}

// s_waitcnt vmcnt(0) (expcnt and lgkmcnt left alone): every vector memory
// operation of the wave, LDS DMA loads included, has completed.
__device__ __forceinline__ void wait_vm_all() {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt [3:0] = 0, expcnt [6:4] = 7, lgkmcnt [11:8] = 15, vmcnt [15:14] = 0
#endif
}

// Record k of the stage; the box is left unset.
__device__ __forceinline__ RecLane rec_stage_lane(const uint4* stage, uint32_t k) {
    const uint4 a = stage[k], b = stage[64 + k], c = stage[128 + k];
    RecLane r;
    r.R = __builtin_bit_cast(double, ((uint64_t)a.y << 32) | a.x);
    r.zs = a.z;
    r.x3 = __uint_as_float(a.w);
    r.y3 = __uint_as_float(b.x); r.e23y = __uint_as_float(b.y); r.e23x = __uint_as_float(b.z);
    r.e31y = __uint_as_float(b.w);
    r.e31x = __uint_as_float(c.x); r.z1 = __uint_as_float(c.y); r.z2 = __uint_as_float(c.z);
    r.z3 = __uint_as_float(c.w);
    r.X0 = r.X1 = r.Y0 = r.Y1 = 0;
    return r;
}
// The same record for every lane (broadcast reads): zs goes to an SGPR, the
// raster branches on it.
__device__ __forceinline__ RecLane rec_stage(const uint4* stage, int k) {
    RecLane r = rec_stage_lane(stage, (uint32_t)k);
    r.zs = (uint32_t)__builtin_amdgcn_readfirstlane((int)r.zs);
    return r;
}

// Triangles between refreshes of the hierarchical depth key.
#ifndef SR_HIZ_PERIOD
#define SR_HIZ_PERIOD 8u
#endif

__device__ __forceinline__ void wave_sync_lds() {
    // LDS written by one lane and read by another within the same wave
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The four 4x4 pixel groups of an 8x8 region (lanes 16 g .. 16 g + 15 own
// group g): bit g = the triangle may cover a pixel centre of group g.  The
// maxima of u, v and w (linear in the pixel) over a group sit at its corners
// by the signs of the coefficients; a group is left out only when one of
// them lies below minus a bound of what the f32 test may be off: with T_u =
// (|e23y| |dx| + |e23x| |dy|) |R| over the region (T_v likewise), |u_f32 -
// u| <= 2^-22 T_u + 2^-149 |R| + 2^-150 (a difference, two products, a sum
// and the rounded quotient, denormals included) and w = (1 - u) - v adds
// less than 2^-22 (T_u + T_v + 1); the margins here are 2^-18 of the same
// sums and more than the f64 rounding.  A NaN keeps the group.
__device__ __forceinline__ uint32_t group_cover(const RecLane& r, int x, int y) {
    const double R = r.R;
    const double ua = (double)r.e23y * R, ub = (double)r.e23x * R, va = (double)r.e31y * R, vb = (double)r.e31x * R;
    const double dx = ((double)x + 0.5) - (double)r.x3, dy = ((double)y + 0.5) - (double)r.y3;
    const double X = fmax(fabs(dx), fabs(dx + 7.0)), Y = fmax(fabs(dy), fabs(dy + 7.0));
    const double tu = fabs(ua) * X + fabs(ub) * Y, tv = fabs(va) * X + fabs(vb) * Y;
    const double tiny = 0x1p-100 + 0x1p-140 * fabs(R);
    const double u0 = ua * dx + ub * dy, v0 = va * dx + vb * dy;
    const double wa = -(ua + va), wb = -(ub + vb);
    auto best = [](double a, double b) { return 3.0 * (fmax(a, 0.0) + fmax(b, 0.0)); };
    const double u = (u0 + best(ua, ub)) + (0x1p-18 * tu + tiny);
    const double v = (v0 + best(va, vb)) + (0x1p-18 * tv + tiny);
    const double w = (((1.0 - u0) - v0) + best(wa, wb)) + (0x1p-18 * (tu + tv + 1.0) + tiny);
    uint32_t m = 0;
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const double ox = (g & 1) ? 4.0 : 0.0, oy = (g & 2) ? 4.0 : 0.0;
        const bool out = (u + (ua * ox + ub * oy) < 0.0) | (v + (va * ox + vb * oy) < 0.0) | (w + (wa * ox + wb * oy) < 0.0);
        m |= out ? 0u : 1u << g;
    }
    return m;
}

// The lanes (4x4 groups) whose pixels of the 8x8 region lie in the box
// [x0, x1] x [y0, y1], given relative to the region.
__device__ __forceinline__ uint64_t box_lanes(int x0, int x1, int y0, int y1) {
    x0 = max(x0, 0); x1 = min(x1, 7);
    y0 = max(y0, 0); y1 = min(y1, 7);
    if (x0 > x1 || y0 > y1) return 0;
    const uint32_t cols = (0xFFu >> (7 - x1)) & (0xFFu << x0), rows = (0xFFu >> (7 - y1)) & (0xFFu << y0);
    // a group's 16 lanes: its four rows' bits spread to nibbles, its four columns' bits in each
    auto spread = [](uint32_t r) { return ((r | r << 3 | r << 6 | r << 9) & 0x1111u) * 0xFu; };
    const uint32_t r0 = spread(rows & 0xFu), r1 = spread(rows >> 4);
    const uint32_t c0 = (cols & 0xFu) * 0x1111u, c1 = (cols >> 4) * 0x1111u;
    return (uint64_t)((r1 & c1) << 16 | (r1 & c0)) << 32 | ((r0 & c1) << 16 | (r0 & c0));
}

// The least depth key of each 4x4 group's pixels in `in` (rotations within
// the rows of 16 lanes).
__device__ __forceinline__ void group_min_keys(float dep, bool in, uint32_t (&key)[4]) {
    uint32_t m = in ? depth_key(__float_as_uint(dep)) : 0xFFFFFFFFu;
    m = min(m, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)m, 0x128, 0xf, 0xf, false));  // row_ror:8
    m = min(m, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)m, 0x124, 0xf, 0xf, false));  // row_ror:4
    m = min(m, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)m, 0x122, 0xf, 0xf, false));  // row_ror:2
    m = min(m, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)m, 0x121, 0xf, 0xf, false));  // row_ror:1
#pragma unroll
    for (int g = 0; g < 4; g++) key[g] = (uint32_t)__builtin_amdgcn_readlane((int)m, 16 * g);
}

// A value that is the same in every lane, kept in an SGPR where the compiler
// cannot see that it is (it went through a loop whose exit it thinks differs
// by lane).
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

// ballot64 of a single comparison is the comparison's own mask in SGPRs;
// conditions are combined as masks (scalar instructions), because a ballot of
// a combined condition costs a select and another comparison.  in_mask turns
// a mask back into a lane condition.
__device__ __forceinline__ uint64_t ballot64(bool p) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ballot_w64(p);
#else
    return p;
#endif
}
__device__ __forceinline__ bool in_mask(uint64_t m) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_inverse_ballot_w64(m);
#else
    return m != 0;
#endif
}

// Whether a triangle's box, or the pixels beyond it that a strip triangle may
// reach, meets [x0, x1] x [y0, y1].
__device__ __forceinline__ bool box_meets(const TriRec& r, int x0, int y0, int x1, int y1) {
    return (r.zs & 1u) != 0u || (r.X0 <= x1 && r.X1 >= x0 && r.Y0 <= y1 && r.Y1 >= y0);
}

// Fragments that passed the depth test and wait to be shaded, one pixel a
// lane: RING_SLOTS of them in LDS in passing order for the whole wave (the
// first waiting position and the number waiting are the same for all lanes),
// and each lane's own as up to RING_DEPTH ring positions in a register (low
// byte first).
constexpr uint32_t RING_SLOTS = 128, RING_DEPTH = 8;

struct FragRing {
    uint32_t head = 0, count = 0, own = 0;
    uint64_t queue = 0;

    __device__ __forceinline__ void put(float4* ring, uint64_t pm, uint32_t tri, float u, float v) {
        if (in_mask(pm)) {
            const uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(pm >> 32),
                                                          __builtin_amdgcn_mbcnt_lo((uint32_t)pm, head + count)) &
                                (RING_SLOTS - 1);
            ring[at] = make_float4(__uint_as_float(tri), u, v, 0.0f);
            queue |= (uint64_t)at << (8u * own);
            own++;
        }
        count += (uint32_t)__popcll(pm);
    }
    // (one more step adds at most 64 fragments, one a lane)
    __device__ __forceinline__ bool full() const { return count >= 64u || ballot64(own == RING_DEPTH) != 0; }
    // The first min(count, 64) fragments: shade(position), one a lane, then
    // blend(position), each pixel its own in order.
    template <class Shade, class Blend>
    __device__ __forceinline__ void flush(int lane, Shade&& shade, Blend&& blend) {
        const uint32_t n = min(count, 64u);
        wave_sync_lds();
        if ((uint32_t)lane < n) shade((head + (uint32_t)lane) & (RING_SLOTS - 1));
        wave_sync_lds();
        for (;;) {
            const uint32_t at = (uint32_t)queue & (RING_SLOTS - 1);
            const bool mine = own != 0u && ((at - head) & (RING_SLOTS - 1)) < n;
            if (!ballot64(mine)) break;
            if (mine) {
                blend(at);
                queue >>= 8;
                own--;
            }
        }
        head = (head + n) & (RING_SLOTS - 1);
        count -= n;
        wave_sync_lds();
    }
};

// The items [sb, se) of a bin that a wave's region may need, in order, up to
// 64 at a time: 256 items are read a step (four a lane, the next step's while
// this one's wait) and those of the region (by the key bits, or by the boxes
// where the keys hold none) join the survivors in LDS.  Every word read is
// one of [sb, se)'s, so every id kept is a valid triangle.
struct BinWalk {
    const RasterParams& P;
    const uint32_t sb, se, bits;
    const int x0, y0, x1, y1, lane;
    uint32_t* const surv;  // 320 words of LDS
    uint32_t c0, waiting = 0, head = 0;
    uint4 id, key;

    __device__ __forceinline__ BinWalk(const RasterParams& P_, uint32_t sb_, uint32_t se_, uint32_t bits_, int x0_,
                                       int y0_, int x1_, int y1_, int lane_, uint32_t* surv_)
        : P(P_), sb(sb_), se(se_), bits(bits_), x0(x0_), y0(y0_), x1(x1_), y1(y1_), lane(lane_), surv(surv_),
          c0(sb_ & ~3u), key(make_uint4(0u, 0u, 0u, 0u)) {
        load();
    }
    __device__ __forceinline__ void load() {
        id = load_ids4(P.items, c0, se, lane);
        if (P.keys) key = load_ids4(P.keys, c0, se, lane);
    }
    // The next survivors: lane k < n holds the k-th one's id (the other lanes
    // the last one's); false at the end.
    __device__ __forceinline__ bool next(uint32_t& cid, uint32_t& n) {
        if (waiting < 64u && c0 < se) {
            if (head) {  // those waiting move to the front
                const uint32_t v = surv[head + lane];
                wave_sync_lds();
                surv[lane] = v;
                head = 0;
            }
            do {
                const uint32_t pos = c0 + 4u * (uint32_t)lane;
                if (P.packed) {
                    key = id;
                    id = make_uint4(id.x >> 16, id.y >> 16, id.z >> 16, id.w >> 16);
                }
                const uint32_t idj[4] = {id.x, id.y, id.z, id.w}, keyj[4] = {key.x, key.y, key.z, key.w};
                uint64_t km[4];  // the lanes whose item j stays
                uint32_t at = waiting;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    km[j] = ballot64(pos + j >= sb) & ballot64(pos + j < se);
                    if (P.keys || P.packed) km[j] &= ballot64((keyj[j] & bits) != 0u);
                    else if (!P.exhaustive)
                        km[j] = ballot64(in_mask(km[j]) && box_meets(P.tris[idj[j]], x0, y0, x1, y1));
                    at = __builtin_amdgcn_mbcnt_hi((uint32_t)(km[j] >> 32),
                                                   __builtin_amdgcn_mbcnt_lo((uint32_t)km[j], at));
                    waiting += (uint32_t)__popcll(km[j]);
                }
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    if (in_mask(km[j])) surv[at++] = idj[j];
                }
                c0 += 256;
                if (c0 < se) load();
            } while (waiting < 64u && c0 < se);
            wave_sync_lds();
        }
        if (waiting == 0u) return false;
        n = min(waiting, 64u);
        cid = surv[head + min((uint32_t)lane, n - 1u)];
        head += n;
        waiting -= n;
        return true;
    }
};

struct ScreenTile {
    int x0, x1, y0, y1;  // inclusive
};

// A block of nblk survivors (lane k's id in cid, its record staged) against
// an 8x8 region with a 4x4 pixel group per 16 lanes (lane's pixel px, py):
// survivor k's groups by its planes, then per group the survivors it may
// cover in front of the group's least depth key hz_g; each group's lanes
// walk their own list (a record per 16 lanes from the stage) and the wave
// steps as often as its longest one.  Every SR_HIZ_PERIOD steps refresh()
// renews hz_g and what is left is filtered by it.  test(record, id, lanes)
// is one step, after() follows it; inM: the lanes of the screen tile T.
// On the 1080p frame of 1M small triangles a step serves 2.6 (triangle, group)
// pairs; all lanes on one triangle at a time took 303 us instead of 238 (4K
// terrain 305 instead of 235).
template <class Refresh, class Test, class After>
__device__ __forceinline__ void walk_groups(const RasterParams& P, uint32_t cid, uint32_t nblk, uint4* stage, int lane,
                                            int wx0, int wy0, int px, int py, const ScreenTile& T, uint64_t inM,
                                            uint32_t (&hz_g)[4], uint32_t& hz_n, Refresh&& refresh, Test&& test,
                                            After&& after) {
    const RecLane mine = rec_stage_lane(stage, (uint32_t)lane);
    const uint32_t zsk = mine.zs | 1u;
    const uint64_t inblk = nblk == 64u ? ~0ull : (1ull << nblk) - 1ull;
    uint64_t gm[4];
#pragma unroll
    for (int g = 0; g < 4; g++) gm[g] = inblk & ballot64(zsk >= hz_g[g]);
    if ((gm[0] | gm[1] | gm[2] | gm[3]) == 0) return;  // all hidden: their planes cost more than the rest
    const uint64_t strips = ballot64((mine.zs & 1u) != 0u);
    // (the key word is read; the stage holds the id in its place)
    ((uint32_t*)&stage[lane])[2] = cid;
    wave_sync_lds();
    const uint32_t gc = group_cover(mine, wx0, wy0);
    // v[lane >> 4], by masks (all ones where bit 4, bit 5 of the lane is set)
    const uint32_t b0 = 0u - ((uint32_t)lane >> 4 & 1u), b1 = 0u - ((uint32_t)lane >> 5 & 1u);
    auto pick1 = [&](uint32_t v0, uint32_t v1, uint32_t v2, uint32_t v3) {
        const uint32_t a = v0 ^ ((v0 ^ v1) & b0), b = v2 ^ ((v2 ^ v3) & b0);
        return a ^ ((a ^ b) & b1);
    };
    auto pick = [&](const uint64_t (&v)[4]) {
        const uint32_t lo = pick1((uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]);
        const uint32_t hi = pick1((uint32_t)(v[0] >> 32), (uint32_t)(v[1] >> 32), (uint32_t)(v[2] >> 32),
                                  (uint32_t)(v[3] >> 32));
        return (uint64_t)hi << 32 | lo;
    };
#pragma unroll
    for (int g = 0; g < 4; g++) gm[g] &= ballot64((gc >> g & 1u) != 0u);
    uint64_t left = pick(gm);
    for (;;) {
        if (--hz_n == 0u) {
            hz_n = SR_HIZ_PERIOD;
            refresh();
            uint64_t zm[4];
#pragma unroll
            for (int g = 0; g < 4; g++) zm[g] = ballot64(zsk >= hz_g[g]);
            left &= pick(zm);
        }
        const uint64_t has = ballot64(left != 0);
        if (has == 0) break;
        // the lowest set bit (the last slot, which always holds a record,
        // where there is none: a count of zeros in 0 is undefined), then cleared
        const uint32_t k = (uint32_t)__builtin_ctzll(left | 1ull << 63);
        left &= left - 1;
        const RecLane rc = rec_stage_lane(stage, k);
        const uint32_t cur = rc.zs;
        uint64_t okm = inM & has;
        if (strips != 0) {
            // strip triangles in the block: those only in their box clamped
            // into the screen tile (triangle.rs:66-78)
            bool in = true;
            if (strips >> k & 1u) {
                const TriRec& t = P.tris[cur];
                in = px >= min(max(t.X0, T.x0), T.x1) && px <= min(max(t.X1, T.x0), T.x1) &&
                     py >= min(max(t.Y0, T.y0), T.y1) && py <= min(max(t.Y1, T.y0), T.y1);
            }
            okm &= ballot64(in);
        }
        test(rc, cur, okm);
        after();
    }
}

}  // namespace sr
