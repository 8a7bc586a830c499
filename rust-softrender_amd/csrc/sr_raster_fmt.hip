// sr_raster_fmt.hip — the raster for every framebuffer format
// (sr_fb_create_ex: up to four colour planes of RGBA8 or RGBAF32 colour, f32
// or f64 depth, u8 or `()` stencil), for the multi-output program and for
// the normalised over-blend, with each lane owning one pixel of an 8x8 tile.
// Two kernels: the binned one walks and shades as the main raster does; the
// other one runs the reference's per-pixel sequence (triangle.rs:82-155)
// triangle by triangle -- stencil test and op in order, coverage, depth, then
// the fragment program and the blend of every plane at once -- for the
// exhaustive mode, for a stencil whose values follow the order of things and
// for a few blended triangles.
#include "sr_kernels.hpp"
#include "sr_raster_common.hpp"

namespace sr {

template <int FP>
__device__ __forceinline__ void shade_varyings(const RasterParams& P, uint32_t tri, float u, float v,
                                               float* k) {
    constexpr int KV = fp_varyings<FP>();
    if constexpr (KV > 0) {
        uint32_t i0 = 3u * tri, i1 = i0 + 1u, i2 = i0 + 2u;  // no indices: 3t, 3t+1, 3t+2
        if (P.vids) {
            const TriVid& r = P.vids[tri];
            i0 = r.i0; i1 = r.i1; i2 = r.i2;
        }
        const float w = (1.0f - u) - v;
        const float *r0 = P.verts.var(i0), *r1 = P.verts.var(i1), *r2 = P.verts.var(i2);
#pragma unroll
        for (int c = 0; c < KV; c++) k[c] = ((r0[c] * u) + (r1[c] * v)) + (r2[c] * w);  // interpolate.rs:43-64
    }
}

template <int FP, int BLEND>
__global__ __launch_bounds__(64) void k_raster_fmt(RasterParams P, FmtParams F) {
    __shared__ float lut_s[256];
    if (P.skip_if && ((load_item(P.skip_if, 0) & 1u) | load_item(P.skip_if, 4))) return;  // NaN, overflow
    for (int i = threadIdx.x; i < 256; i += 64) lut_s[i] = (float)i / 255.0f;
    __syncthreads();
    const Lut lut{lut_s};
    const uint32_t tile = xcd_deal<BinTiles<8>::N>(blockIdx.x, gridDim.x);
    uint32_t bin, tx0, ty0;
    tile_origin<8>(P, tile, bin, tx0, ty0);
    if (tx0 >= P.W || ty0 >= P.H) return;
    const uint32_t bits = region_bits((int)tx0, (int)ty0, 8, 8);
    const uint32_t beg = load_item(P.tile_start, bin), end = bin_end(beg, load_item(P.tile_end, bin), bits);
    if (beg >= end) return;
    const int lane = threadIdx.x;
    const int wx0 = (int)tx0, wy0 = (int)ty0;
    const int wx1 = min(wx0 + 7, (int)P.W - 1), wy1 = min(wy0 + 7, (int)P.H - 1);
    const int px = wx0 + (lane & 7), py = wy0 + (lane >> 3);
    const bool live = px < (int)P.W && py < (int)P.H;
    const size_t idx = live ? (size_t)py * P.W + px : 0;

    // the pixel's planes; an RGBA8 plane keeps its packed value in c[p][0]
    float c[SR_MAX_COLOR_PLANES][4] = {};
#pragma unroll
    for (int p = 0; p < SR_MAX_COLOR_PLANES; p++) {
        if (p >= (int)F.n_color || !live) continue;
        if (F.color_fmt[p] == SR_COLOR_RGBAF32) {
            const float4 v = ((const float4*)F.planes[p])[idx];
            c[p][0] = v.x; c[p][1] = v.y; c[p][2] = v.z; c[p][3] = v.w;
        } else {
            c[p][0] = __builtin_bit_cast(float, ((const uint32_t*)F.planes[p])[idx]);
        }
    }
    double dep = live ? (F.depth64 ? F.depth64[idx] : (double)P.depth[idx]) : 0.0;
    uint32_t st = (live && F.has_stencil) ? P.stencil[idx] : 0u;
    const float fx = (float)px + 0.5f, fy = (float)py + 0.5f;  // triangle.rs:104-105

    uint32_t jlo, jhi, ilo, ihi;
    sem_range((uint32_t)wx0, (uint32_t)wx1, P.tw, P.scols, jlo, jhi);
    sem_range((uint32_t)wy0, (uint32_t)wy1, P.th, P.srows, ilo, ihi);
    const uint32_t xmax = P.W - 1, ymax = P.H - 1;
    for (uint32_t si = ilo; si <= ihi; si++) {
        const int Ty0 = (int)(si * P.th), Ty1 = (int)min(si * P.th + P.th, ymax);
        for (uint32_t sj = jlo; sj <= jhi; sj++) {
            const int Tx0 = (int)(sj * P.tw), Tx1 = (int)min(sj * P.tw + P.tw, xmax);
            if (max(wx0, Tx0) > min(wx1, Tx1) || max(wy0, Ty0) > min(wy1, Ty1)) continue;
            const bool inT = live && px >= Tx0 && px <= Tx1 && py >= Ty0 && py <= Ty1;
            for (uint32_t c0 = beg; c0 < end; c0 += 64) {
                // 64 items of the bin at a time, those of this tile among them
                uint32_t id64 = load_ids(P.items, c0, beg, end, lane), key = ~0u;
                if (P.keys) key = load_ids(P.keys, c0, beg, end, lane);
                if (P.packed) {
                    key = id64;
                    id64 >>= 16;
                }
                uint64_t m = __ballot(c0 + (uint32_t)lane < end && (key & bits) != 0u);
                for (; m != 0; m &= m - 1) {
                    const uint32_t id = lane_u32(id64, __builtin_amdgcn_readfirstlane(__builtin_ctzll(m)));
                    const RecLane rc = rec_s(P.tris, id);
                    int cx0 = rc.X0, cx1 = rc.X1, cy0 = rc.Y0, cy1 = rc.Y1;
                    if (P.exhaustive || (rc.zs & 1u)) {  // every box, or one a pixel outside may pass
                        if (rc.X0 > rc.X1) continue;  // culled or invalid
                        // clamp_as_int! into the screen tile, triangle.rs:66-78
                        cx0 = min(max(rc.X0, Tx0), Tx1); cx1 = min(max(rc.X1, Tx0), Tx1);
                        cy0 = min(max(rc.Y0, Ty0), Ty1); cy1 = min(max(rc.Y1, Ty0), Ty1);
                    }
                    bool ok = inT && px >= cx0 && px <= cx1 && py >= cy0 && py <= cy1;
                    if (F.track_stencil) {  // stencil before coverage, triangle.rs:90-99
                        const bool sp = ok && stencil_test(P.s_test, st, P.s_ref);
                        st = sp ? stencil_op(P.s_op, P.s_wrap, st, P.s_ref) : st;
                        ok = sp;
                    }
                    if (ballot64(ok) == 0) continue;  // the box meets no pixel here
                    const float dx = fx - rc.x3, dy = fy - rc.y3;
                    const float un = (rc.e23y * dx) + (rc.e23x * dy);  // triangle.rs:108
                    const float vn = (rc.e31y * dx) + (rc.e31x * dy);  // triangle.rs:109
                    const float u = quot(un, rc.R), v = quot(vn, rc.R);
                    const float w = (1.0f - u) - v;                    // triangle.rs:110
                    const float z = ((rc.z1 * u) + (rc.z2 * v)) + (rc.z3 * w);
                    // Depth::from_scalar(z) is exact for f64 (depth.rs:26-41), so
                    // z >= dt compares the same values either way
                    if (!(ok && !(u < 0.0f) && !(v < 0.0f) && !(w < 0.0f) && z < 0.0f && (double)z >= dep)) continue;
                    dep = (double)z;
                    float k[8];
                    shade_varyings<FP>(P, id, u, v, k);
                    float o[FP == SR_FP_GBUFFER ? 4 : 1][4];
                    constexpr int NO = FP == SR_FP_GBUFFER ? 4 : 1;
                    fragment_rgba<FP>(P, k, lut, o);
#pragma unroll
                    for (int p = 0; p < SR_MAX_COLOR_PLANES; p++) {
                        if (p >= (int)F.n_color) continue;
                        const float* src = o[p < NO ? p : NO - 1];
                        if (F.color_fmt[p] == SR_COLOR_RGBAF32) {
                            float out[4];
                            blend_f32<BLEND>(src, c[p], out);
#pragma unroll
                            for (int q = 0; q < 4; q++) c[p][q] = out[q];
                        } else {
                            const uint32_t d = __builtin_bit_cast(uint32_t, c[p][0]);
                            c[p][0] = __builtin_bit_cast(float, blend<BLEND>(pack_q(src), d, lut));
                        }
                    }
                }
            }
        }
    }
    if (!live) return;
#pragma unroll
    for (int p = 0; p < SR_MAX_COLOR_PLANES; p++) {
        if (p >= (int)F.n_color) continue;
        if (F.color_fmt[p] == SR_COLOR_RGBAF32)
            ((float4*)F.planes[p])[idx] = make_float4(c[p][0], c[p][1], c[p][2], c[p][3]);
        else
            ((uint32_t*)F.planes[p])[idx] = __builtin_bit_cast(uint32_t, c[p][0]);
    }
    if (F.depth64) F.depth64[idx] = dep;
    else P.depth[idx] = (float)dep;
    if (F.has_stencil) P.stencil[idx] = (uint8_t)st;
}

// Binned draws whose stencil takes no part.  Bound by the triangle tests and
// the shading (VALU issue): the tests are the main raster's (4x4 groups,
// hierarchical depth), the shading is dense.  `()` blend: only a pixel's last
// fragment shades, once.  OVER and its normalised form: a ring of fragments,
// shaded 64 at a time, each pixel's blended in order.  At 900p, 60k
// triangles into four planes (`()`): 57 us instead of 165; 720p with
// normalised OVER into RGBAF32: 43 instead of 220.
// z is a float, so z >= dt for an f64 depth dt is z >= the least float not
// below dt: the depth is tested as that float, and it is written (as z) only
// where a fragment passed.
// NP: colour planes the kernel holds (1, or up to SR_MAX_COLOR_PLANES).
template <int FP, int BLEND, int NP>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(NP == 1 ? 5 : 4, 8))) void k_raster_fmt_bins(RasterParams P, FmtParams F) {
    constexpr bool RING = BLEND != SR_BLEND_REPLACE;
    constexpr int NO = FP == SR_FP_GBUFFER ? 4 : 1;
    __shared__ float4 ring[RING ? NO : 1][RING ? RING_SLOTS : 1];  // [0]: (triangle, u, v) until shaded
    __shared__ uint4 stage[3 * 64];
    __shared__ uint32_t surv[320];
    __shared__ float lut_s[256];
    if (P.skip_if && ((load_item(P.skip_if, 0) & 1u) | load_item(P.skip_if, 4))) return;  // NaN, overflow
    const uint32_t tile = xcd_deal<BinTiles<8>::N>(blockIdx.x, gridDim.x);
    uint32_t bin, tx0, ty0;
    tile_origin<8>(P, tile, bin, tx0, ty0);
    if (tx0 >= P.W || ty0 >= P.H) return;
    const uint32_t bits = region_bits((int)tx0, (int)ty0, 8, 8);
    const uint32_t beg = load_item(P.tile_start, bin), end = bin_end(beg, load_item(P.tile_end, bin), bits);
    if (beg >= end) return;
    const int lane = threadIdx.x;
    for (int i = lane; i < 256; i += 64) lut_s[i] = unorm8((float)i);
    wave_sync_lds();
    const Lut lut{lut_s};
    const int wx0 = (int)tx0, wy0 = (int)ty0;
    const int wx1 = min(wx0 + 7, (int)P.W - 1), wy1 = min(wy0 + 7, (int)P.H - 1);
    const int px = wx0 + ((lane >> 2) & 4) + (lane & 3), py = wy0 + ((lane >> 3) & 4) + ((lane >> 2) & 3);
    const bool live = px < (int)P.W && py < (int)P.H;
    const size_t idx = live ? (size_t)py * P.W + px : 0;
    const float fx = (float)px + 0.5f, fy = (float)py + 0.5f;  // triangle.rs:104-105

    // a pixel outside the framebuffer: see the main raster
    float dep = __uint_as_float(0x7FFFFFFFu);
    if (live) {
        if (F.depth64) {
            const double d = F.depth64[idx];
            dep = (float)d;
            if ((double)dep < d) dep = __uint_as_float(__float_as_uint(dep) + (dep < 0.0f ? ~0u : 1u));
        } else {
            dep = P.depth[idx];
        }
    }
    // the pixel's planes where they are blended; an RGBA8 plane keeps its
    // packed value in c[p][0]
    float c[RING ? NP : 1][4] = {};
    if constexpr (RING) {
#pragma unroll
        for (int p = 0; p < NP; p++) {
            if (NP > 1 && p >= (int)F.n_color) continue;
            if (F.color_fmt[p] == SR_COLOR_RGBAF32) {
                const float4 v = ((const float4*)F.planes[p])[idx];
                c[p][0] = v.x; c[p][1] = v.y; c[p][2] = v.z; c[p][3] = v.w;
            } else {
                c[p][0] = __builtin_bit_cast(float, ((const uint32_t*)F.planes[p])[idx]);
            }
        }
    }
    uint64_t have = 0;  // the lanes where a fragment passed
    uint32_t last = 0;  // `()` blend: the last one
    float last_u = 0.0f, last_v = 0.0f;
    FragRing waiting;
    auto shade = [&](uint32_t tri, float u, float v, float (&o)[NO][4]) __attribute__((always_inline)) {
        float k[8];
        shade_varyings<FP>(P, tri, u, v, k);
        fragment_rgba<FP>(P, k, lut, o);
    };
    auto flush = [&]() __attribute__((always_inline)) {
        waiting.flush(
            lane,
            [&](uint32_t at) __attribute__((always_inline)) {
                const float4 f = ring[0][at];
                float o[NO][4];
                shade(__float_as_uint(f.x), f.y, f.z, o);
#pragma unroll
                for (int q = 0; q < NO; q++) ring[q][at] = make_float4(o[q][0], o[q][1], o[q][2], o[q][3]);
            },
            [&](uint32_t at) __attribute__((always_inline)) {
#pragma unroll
                for (int p = 0; p < NP; p++) {
                    if (NP > 1 && p >= (int)F.n_color) continue;
                    const float4 f = ring[p < NO ? p : NO - 1][at];
                    const float src[4] = {f.x, f.y, f.z, f.w};
                    if (F.color_fmt[p] == SR_COLOR_RGBAF32) {
                        float out[4];
                        blend_f32<BLEND>(src, c[p], out);
#pragma unroll
                        for (int q = 0; q < 4; q++) c[p][q] = out[q];
                    } else {
                        const uint32_t d = __builtin_bit_cast(uint32_t, c[p][0]);
                        c[p][0] = __builtin_bit_cast(float, blend<BLEND>(pack_q(src), d, lut));
                    }
                }
            });
    };

    uint32_t jlo, jhi, ilo, ihi;
    sem_range((uint32_t)wx0, (uint32_t)wx1, P.tw, P.scols, jlo, jhi);
    sem_range((uint32_t)wy0, (uint32_t)wy1, P.th, P.srows, ilo, ihi);
    const uint32_t xmax = P.W - 1, ymax = P.H - 1;
    for (uint32_t si = ilo; si <= ihi; si++) {
        const int Ty0 = (int)(si * P.th), Ty1 = (int)min(si * P.th + P.th, ymax);
        for (uint32_t sj = jlo; sj <= jhi; sj++) {
            const int Tx0 = (int)(sj * P.tw), Tx1 = (int)min(sj * P.tw + P.tw, xmax);
            if (max(wx0, Tx0) > min(wx1, Tx1) || max(wy0, Ty0) > min(wy1, Ty1)) continue;
            const bool inT = live && px >= Tx0 && px <= Tx1 && py >= Ty0 && py <= Ty1;
            const uint64_t inM = ballot64(inT);
            // (a bound for this screen tile's pixels: see the main raster)
            uint32_t hz_n = 1u, hz_g[4] = {0u, 0u, 0u, 0u};
            BinWalk items(P, beg, end, bits, wx0, wy0, wx1, wy1, lane, surv);
            uint32_t cid, nblk;
            while (items.next(cid, nblk)) {
                stage_records(P.tris, cid, stage);
                wait_vm_all();  // the stage has landed
                walk_groups(
                    P, cid, nblk, stage, lane, wx0, wy0, px, py, ScreenTile{Tx0, Tx1, Ty0, Ty1}, inM, hz_g, hz_n,
                    [&]() { group_min_keys(dep, inT, hz_g); },
                    [&](const RecLane& rc, uint32_t cur, uint64_t okm) {
                        const float dx = fx - rc.x3, dy = fy - rc.y3;
                        const float un = (rc.e23y * dx) + (rc.e23x * dy);  // triangle.rs:108
                        const float vn = (rc.e31y * dx) + (rc.e31x * dy);  // triangle.rs:109
                        const float u = quot(un, rc.R), v = quot(vn, rc.R);
                        const float w = (1.0f - u) - v;                    // triangle.rs:110
                        const float z = ((rc.z1 * u) + (rc.z2 * v)) + (rc.z3 * w);  // :115-117
                        // :113 inside, :120-126 depth
                        const uint64_t pm = okm & ballot64(!(u < 0.0f)) & ballot64(!(v < 0.0f)) &
                                            ballot64(!(w < 0.0f)) & ballot64(z < 0.0f) & ballot64(z >= dep);
                        const bool pass = in_mask(pm);
                        dep = pass ? z : dep;
                        have |= pm;
                        if constexpr (RING) {
                            waiting.put(ring[0], pm, cur, u, v);
                        } else {
                            last = pass ? cur : last;
                            last_u = pass ? u : last_u;
                            last_v = pass ? v : last_v;
                        }
                    },
                    [&]() {
                        if constexpr (RING) {
                            while (waiting.full()) flush();
                        }
                    });
            }
        }
    }
    if constexpr (RING) {
        while (waiting.count) flush();
    }
    if (!in_mask(have)) return;
    float o[NO][4];
    if constexpr (!RING) shade(last, last_u, last_v, o);
#pragma unroll
    for (int p = 0; p < NP; p++) {
        if (NP > 1 && p >= (int)F.n_color) continue;
        const float* src = RING ? c[RING ? p : 0] : o[p < NO ? p : NO - 1];
        if (F.color_fmt[p] == SR_COLOR_RGBAF32)
            ((float4*)F.planes[p])[idx] = make_float4(src[0], src[1], src[2], src[3]);
        else
            ((uint32_t*)F.planes[p])[idx] = RING ? __builtin_bit_cast(uint32_t, src[0]) : pack_q(src);
    }
    if (F.depth64) F.depth64[idx] = (double)dep;
    else P.depth[idx] = dep;
}

// Blended draws of up to this many triangles go triangle by triangle: with so
// few the walk's setup costs more than its denser shading gives (900p,
// textured, normalised OVER, full-screen layers of two triangles: one layer 71
// us by triangle, 86 binned; two 90, 104; eight 198, 197; 32: 605, 584).
constexpr uint32_t FMT_FEW_TRIS = 16;

template <int FP, int BLEND>
static void raster_fmt(const RasterParams& P, const FmtParams& F, uint32_t ntris, uint32_t ntiles, hipStream_t s) {
    const dim3 g(ntiles), b(64);
    if (P.exhaustive || F.track_stencil || (BLEND != SR_BLEND_REPLACE && ntris <= FMT_FEW_TRIS))
        hipLaunchKernelGGL((k_raster_fmt<FP, BLEND>), g, b, 0, s, P, F);
    else if (F.n_color == 1) hipLaunchKernelGGL((k_raster_fmt_bins<FP, BLEND, 1>), g, b, 0, s, P, F);
    else hipLaunchKernelGGL((k_raster_fmt_bins<FP, BLEND, SR_MAX_COLOR_PLANES>), g, b, 0, s, P, F);
}

template <int FP>
static void raster_fmt_blend(const RasterParams& P, const FmtParams& F, uint32_t ntris, uint32_t ntiles,
                             hipStream_t s) {
    if (P.blend == SR_BLEND_OVER) raster_fmt<FP, SR_BLEND_OVER>(P, F, ntris, ntiles, s);
    else if (P.blend == SR_BLEND_OVER_NORMALIZED) raster_fmt<FP, SR_BLEND_OVER_NORMALIZED>(P, F, ntris, ntiles, s);
    else raster_fmt<FP, SR_BLEND_REPLACE>(P, F, ntris, ntiles, s);
}

void launch_raster_fmt(const RasterParams& P, const FmtParams& F, uint32_t ntris, uint32_t ntiles, hipStream_t s) {
    if (!ntiles) return;
    switch (P.fp) {
        case SR_FP_BLINN_PHONG: raster_fmt_blend<SR_FP_BLINN_PHONG>(P, F, ntris, ntiles, s); break;
        case SR_FP_TEX_LAMBERT: raster_fmt_blend<SR_FP_TEX_LAMBERT>(P, F, ntris, ntiles, s); break;
        case SR_FP_UV_COLOR: raster_fmt_blend<SR_FP_UV_COLOR>(P, F, ntris, ntiles, s); break;
        case SR_FP_GBUFFER: raster_fmt_blend<SR_FP_GBUFFER>(P, F, ntris, ntiles, s); break;
        case SR_FP_FRESNEL4: raster_fmt_blend<SR_FP_FRESNEL4>(P, F, ntris, ntiles, s); break;
        case SR_FP_INT_PALETTE: raster_fmt_blend<SR_FP_INT_PALETTE>(P, F, ntris, ntiles, s); break;
        default: raster_fmt_blend<SR_FP_FLAT>(P, F, ntris, ntiles, s); break;
    }
}

}  // namespace sr
