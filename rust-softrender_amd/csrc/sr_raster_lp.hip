// sr_raster_lp.hip — raster work-groups for line plots and points.
//
// One work-group per 16x16 execution tile.  Each plot (or point) is one
// stencil/depth/shade/blend step on one pixel.  Per pixel those steps must run
// in the reference's order: screen tile by screen tile (row-major,
// fragment.rs:250-253), then line by line, then plot by plot.
#include "sr_device.hpp"
#include "sr_kernels.hpp"
#include "sr_raster_common.hpp"

namespace sr {

constexpr int LP_ETS = 16;
static_assert(LP_ETS == LINE_STEP, "a tile's edge is a sample's place");

__device__ __forceinline__ float lp_hypot(float a, float b) {
    // glibc hypotf: sqrt(x*x + y*y) in double, rounded once to float
    if (__builtin_isinf(a) || __builtin_isinf(b)) return __builtin_inff();
    const double x = (double)a, y = (double)b;
    return (float)sqrt(x * x + y * y);
}

__device__ __forceinline__ uint32_t block_min_256(uint32_t v, uint32_t* lds4) {
    // (the steps of wave_excl_scan; lane 63 ends with the minimum)
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x111, 0xf, 0xf, false));
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x112, 0xf, 0xf, false));
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x114, 0xf, 0xf, false));
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x118, 0xf, 0xf, false));
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x142, 0xa, 0xf, false));
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x143, 0xc, 0xf, false));
    if ((threadIdx.x & 63) == 63) lds4[threadIdx.x >> 6] = v;
    __syncthreads();
    const uint32_t r = min(min(lds4[0], lds4[1]), min(lds4[2], lds4[3]));
    __syncthreads();
    return r;
}

// Runs `apply(rank)` for every pending rank in this chunk, same-pixel ranks
// in increasing order.
template <class F>
__device__ __forceinline__ void ordered_rounds(bool pending, int lp, uint32_t rank, uint32_t* claim,
                                               F&& apply) {
    while (__syncthreads_or(pending)) {
        if (pending) atomicMin(&claim[lp], rank);
        __syncthreads();
        const bool mine = pending && claim[lp] == rank;
        if (mine) {
            apply();
            pending = false;
        }
        __syncthreads();
        if (mine) claim[lp] = 0xFFFFFFFFu;
        __syncthreads();
    }
}

// Exclusive prefix sums of two values over the work-group's 256 threads (in
// thread order), and their totals.
__device__ __forceinline__ void lp_scan2(uint32_t& a, uint32_t& b, uint32_t& total_a, uint32_t& total_b, uint32_t (*lds)[4]) {
    const uint32_t wave = threadIdx.x >> 6;
    uint32_t ta, tb;
    a = wave_excl_scan(a, ta);
    b = wave_excl_scan(b, tb);
    if ((threadIdx.x & 63) == 0) {
        lds[0][wave] = ta;
        lds[1][wave] = tb;
    }
    __syncthreads();
    total_a = total_b = 0;
#pragma unroll
    for (uint32_t w = 0; w < 4; w++) {
        const uint32_t qa = lds[0][w], qb = lds[1][w];
        if (w < wave) {
            a += qa;
            b += qb;
        }
        total_a += qa;
        total_b += qb;
    }
    __syncthreads();
}

// Lines: per screen tile (ascending), the tile's line items are staged in
// LDS (256 at a time, list = line order) with what their plots need, and
// the concatenated plot sequence of the staged items is processed LINE_PASS
// plots per pass: plot g belongs to the first staged item whose plot-count
// prefix exceeds g.  A pass has two halves.  Plot by plot, two neighbours a
// thread (a Wu pair mostly, which shares the walk's state): its depth, and its
// colour if the pixel's depth lets it pass (depths only grow, and no program
// looks at the pixel), left in LDS, with the plot's bit set in its pixel's
// mask.  Then pixel by pixel, a thread each with the pixel in registers: the
// plots of the pixel's mask in bit order, which is the reference's
// line-then-plot order.  Bound by instruction issue (57% of the time at 4K)
// and the work-group's barriers: the second half steps as often as a wave's
// busiest pixel, so a pass is as long as five work-groups a CU leave LDS for
// where the plots fill it, and half as long where they don't.  4K with 200,000
// lines: 466 us (550 when the threads of a pass took turns on shared pixels
// and shaded in their turn; 617 with 512 plots always, 544 with 256); 720p with
// the face normals of a sphere of 39,600 triangles, whose poles share few
// tiles: 207 (432; 205, 253).
constexpr uint32_t LINE_PASS = 512;
constexpr uint32_t LINE_STAGE = 128;  // items staged at a time

template <int FP, int BLEND>
__global__ __launch_bounds__(256) void k_raster_lines(RasterParams P) {
    constexpr int KV = fp_varyings<FP>();
    constexpr bool OVER = BLEND == SR_BLEND_OVER;
    constexpr uint32_t MW = LINE_PASS / 64;  // mask words
    __shared__ uint64_t mask[MW][256];  // per pixel: the pass's plots on it, in order
    __shared__ uint32_t words[256];     // per pixel: the mask's words that are not zero
    __shared__ uint2 src[LINE_PASS];    // per plot: its depth (0: it cannot pass) and colour
    __shared__ float s_dep[256], slut[256];
    __shared__ uint32_t lds4[4], lds8[2][4];
    __shared__ float i_cx1[LINE_STAGE], i_cy1[LINE_STAGE], i_dlen[LINE_STAGE], i_zs[LINE_STAGE], i_ze[LINE_STAGE];
    __shared__ uint32_t i_v0[LINE_STAGE], i_v1[LINE_STAGE], i_off[LINE_STAGE], i_end[LINE_STAGE];  // i_end: inclusive plot prefix
    __shared__ uint32_t i_skip[LINE_STAGE];  // interior plots before this tile's (ranged items)
    // sampled items: minor coordinate and major coordinate of the first
    // interior pair in the tile, and the gradient
    __shared__ double i_y[LINE_STAGE], i_grad[LINE_STAGE];
    __shared__ int i_x[LINE_STAGE];
    __shared__ uint8_t i_kind[LINE_STAGE];  // bit 0: sampled, 1: steep, 2, 3: the first, second endpoint's plots may be in the tile
    const int t = threadIdx.x;
    const uint32_t tile = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t etx = tile % P.ntx, ety = tile / P.ntx;
    const uint32_t beg = P.tile_start[tile], end = P.tile_end[tile];
    if (beg >= end) return;
    const int gx = (int)(etx * LP_ETS) + (t % LP_ETS), gy = (int)(ety * LP_ETS) + (t / LP_ETS);
    const bool live = (uint32_t)gx < P.W && (uint32_t)gy < P.H;
    const size_t idx = (size_t)gy * P.W + gx;
    uint32_t col = live ? P.color[idx] : 0u, st = live ? P.stencil[idx] : 0u;
    float dep = live ? P.depth[idx] : 0.0f;
    float dst[4];
#pragma unroll
    for (int q = 0; q < 4; q++) dst[q] = unorm8((float)(col >> (8 * q) & 0xFFu));
    bool shaded = false;
    slut[t] = unorm8((float)t);
    s_dep[t] = dep;
#pragma unroll
    for (uint32_t w = 0; w < MW; w++) mask[w][t] = 0;
    words[t] = 0;
    __syncthreads();
    const Lut lut{slut};
    const int ex0 = (int)(etx * LP_ETS), ey0 = (int)(ety * LP_ETS);
    const bool counts = P.s_op != SR_STENCIL_KEEP;  // a plot that cannot pass the depth test still counts

    // screen tiles in ascending (row-major) order; a list that fits one
    // staging step stays in registers
    LineItem it{};
    const bool once = end - beg <= LINE_STAGE;
    if (once && t < (int)(end - beg)) it = P.line_items[P.items[beg + t]];
    bool first = true;
    uint32_t prev = 0;
    for (;;) {
        uint32_t best = 0xFFFFFFFFu;
        if (once) {
            if (t < (int)(end - beg) && (first || it.tile > prev)) best = it.tile;
        } else {
            for (uint32_t i = beg + t; i < end; i += 256) {
                const uint32_t T = P.line_items[P.items[i]].tile;
                if ((first || T > prev) && T < best) best = T;
            }
        }
        best = block_min_256(best, lds4);
        if (best == 0xFFFFFFFFu) break;
        for (uint32_t ib = beg; ib < end; ib += LINE_STAGE) {
            // stage this screen tile's items among the next of the list
            const uint32_t i = ib + (uint32_t)t;
            const bool have = t < (int)LINE_STAGE && i < end;
            if (!once && have) it = P.line_items[P.items[i]];
            const bool mine = have && it.tile == best && it.plot_cnt > 0;
            // plots to scan: all, or for a ranged Wu item the 4 endpoint
            // plots and the interior pairs whose major coordinate lies in
            // this tile's span (the others fall outside the tile)
            uint32_t scan = mine ? it.plot_cnt : 0u, skip = 0, kind = 0;
            double y0 = 0.0, grad = 0.0;
            int x0 = 0;
            const bool steep = (it.flags & LINE_STEEP) != 0;
            if (mine && (it.flags & LINE_RANGED)) {
                const int64_t M0 = steep ? ey0 : ex0, M1 = M0 + LP_ETS - 1;
                const int64_t nint = (int64_t)(it.plot_cnt - 4) / 2;
                int64_t lo = max<int64_t>(M0 - it.major0, 0);
                int64_t hi = max<int64_t>(min<int64_t>(M1 - it.major0 + 1, nint), lo);
                scan = 4u + 2u * (uint32_t)(hi - lo);
                skip = 2u * (uint32_t)lo;
                if (it.flags & LINE_SAMPLED) {
                    // plots past the right edge land in the first column: there the whole walk is scanned
                    const bool all = (it.flags & LINE_WRAPS) && etx == 0;
                    if (all) {
                        lo = 0;
                        hi = nint;
                    }
                    // an end whose plots (within two pixels of it) lie outside the tile is not scanned
                    auto near = [&](float x, float y) {
                        return all || (x >= (float)(ex0 - 2) && x <= (float)(ex0 + LP_ETS + 2) && y >= (float)(ey0 - 2) &&
                               y <= (float)(ey0 + LP_ETS + 2));
                    };
                    const bool swapped = steep ? it.cy1 > it.cy2 : it.cx1 > it.cx2;  // the walk's first end
                    const bool a = swapped ? near(it.cx2, it.cy2) : near(it.cx1, it.cy1);
                    const bool b = swapped ? near(it.cx1, it.cy1) : near(it.cx2, it.cy2);
                    scan = (a ? 2u : 0u) + (b ? 2u : 0u) + 2u * (uint32_t)(hi - lo);
                    kind = 1u | (steep ? 2u : 0u) | (a ? 4u : 0u) | (b ? 8u : 0u);
                    if (hi > lo) {
                        const double* samples = (const double*)(P.plots + it.plot_off + 4);
                        grad = samples[0];
                        x0 = it.major0 + (int)lo;  // major0, or the tile's edge: a sample's place
                        y0 = samples[1 + x0 / (int)LINE_STEP - it.major0 / (int)LINE_STEP];
                    }
                }
            }
            uint32_t nstaged, total;
            uint32_t slot = scan ? 1u : 0u, pstart = scan;
            lp_scan2(slot, pstart, nstaged, total, lds8);
            if (nstaged == 0) continue;  // uniform
            // plots a thread: one where the pass is short
            const uint32_t ept = total > 256u ? 2u : 1u;
            if (scan) {
                const uint32_t v0 = P.line_v ? P.line_v[2 * it.line] : 2 * it.line;
                const uint32_t v1 = P.line_v ? P.line_v[2 * it.line + 1] : 2 * it.line + 1;
                i_cx1[slot] = it.cx1;
                i_cy1[slot] = it.cy1;
                i_dlen[slot] = it.dlen;
                i_zs[slot] = it.zs;
                i_ze[slot] = it.ze;
                i_v0[slot] = v0;
                i_v1[slot] = v1;
                i_off[slot] = it.plot_off;
                i_skip[slot] = skip;
                i_end[slot] = pstart + scan;
                i_kind[slot] = (uint8_t)kind;
                i_y[slot] = y0;
                i_grad[slot] = grad;
                i_x[slot] = x0;
            }
            __syncthreads();
            for (uint32_t c = 0; c < total; c += 256u * ept) {
                const uint32_t g = c + ept * (uint32_t)t;
                if (g < total) {
                    uint32_t si = 0, hi = nstaged - 1;  // first staged item with i_end > g
                    while (si < hi) {
                        const uint32_t m = (si + hi) >> 1;
                        if (i_end[m] > g) hi = m;
                        else si = m + 1;
                    }
                    double y = 0.0;  // a sampled item's minor coordinate at pair yq
                    uint32_t yq = ~0u;
#pragma unroll
                    for (uint32_t e = 0; e < 2u; e++) {
                        if (e >= ept || g + e >= total) break;
                        if (g + e >= i_end[si]) {  // the next item's first plot
                            si++;
                            yq = ~0u;
                        }
                        uint32_t j = g + e - (si ? i_end[si - 1] : 0u);
                        const uint32_t kind = i_kind[si];
                        bool stored = true;
                        if (kind & 1u) {
                            const uint32_t na = kind >> 1 & 2u, nb = kind >> 2 & 2u;
                            stored = j < na + nb;
                            j = stored ? (j < na ? j : j + 2u - na) : j - na - nb;
                        } else {
                            j = j < 4u ? j : j + i_skip[si];
                        }
                        Plot pl;
                        if (stored) {
                            pl = P.plots[i_off[si] + j];
                        } else {  // an interior plot by the walk's additions
                            if (yq != j >> 1) {
                                yq = j >> 1;
                                y = i_y[si];
                                const double grad = i_grad[si];
                                for (uint32_t q = yq; q != 0; q--) y += grad;
                            }
                            const double yt = trunc(y), fr = y - yt;
                            const int minor = (int)yt + (int)(j & 1u), major = i_x[si] + (int)yq;
                            pl.alpha = (j & 1u) ? fr : 1.0 - fr;
                            pl.x = (kind & 2u) ? minor : major;
                            pl.y = (kind & 2u) ? major : minor;
                            const bool wrap = (uint32_t)pl.x == P.W;
                            pl.row = (uint32_t)pl.y + (wrap ? 1u : 0u);
                            pl.index = (wrap ? 0u : (uint32_t)pl.x) + pl.row * P.W;
                        }
                        const int py = (int)pl.row - ey0, px = (int)(pl.index - pl.row * P.W) - ex0;
                        if (!(px >= 0 && px < LP_ETS && py >= 0 && py < LP_ETS && pl.row < P.H)) continue;
                        // the rasterize_fragment closure, line.rs:54-109
                        const int lp = py * LP_ETS + px;
                        const uint32_t k = ept * (uint32_t)t + e;
                        const float xf = (float)pl.x + 0.5f, yf = (float)pl.y + 0.5f;
                        const float tt = lp_hypot(i_cx1[si] - xf, i_cy1[si] - yf) / i_dlen[si];  // :75
                        const float omt = 1.0f - tt;
                        const float z = (omt * i_zs[si]) + (tt * i_ze[si]);                     // :77
                        const bool may = z < 0.0f && z >= s_dep[lp];
                        if (may || counts) {
                            if (!may) src[k].x = 0u;
                            atomicOr((unsigned long long*)&mask[k >> 6][lp], 1ull << (k & 63u));
                            atomicOr(&words[lp], 1u << (k >> 6));
                        }
                        if (may) {
                            float kv[KV > 0 ? KV : 1];
                            const float *r0 = P.verts.var(i_v0[si]), *r1 = P.verts.var(i_v1[si]);
#pragma unroll
                            for (int q = 0; q < KV; q++) kv[q] = (omt * r0[q]) + (tt * r1[q]);
                            src[k] = make_uint2(__float_as_uint(z),
                                                mul_alpha(P.alpha_mode, fragment<FP>(P, kv, lut), pl.alpha));  // :100
                        }
                    }
                }
                __syncthreads();
                uint32_t left = words[t];
                if (left) {
                    words[t] = 0;
                    uint64_t m = 0;
                    uint32_t w = 0;
                    do {  // the pixel's next plot
                        if (m == 0) {
                            w = (uint32_t)__builtin_ctz(left);
                            m = mask[w][t];
                            mask[w][t] = 0;
                            left &= left - 1u;
                        }
                        const uint32_t k = 64u * w + (uint32_t)__builtin_ctzll(m);
                        m &= m - 1;
                        if (stencil_test(P.s_test, st, P.s_ref)) {
                            st = stencil_op(P.s_op, P.s_wrap, st, P.s_ref);
                            const uint2 f = src[k];
                            const float z = __uint_as_float(f.x);
                            if (z < 0.0f && z >= dep) {
                                dep = z;
                                shaded = true;
                                if constexpr (OVER) {  // blend<SR_BLEND_OVER>
                                    const float a = unorm8((float)(f.y >> 24)), ia = 1.0f - a;
                                    dst[0] = unorm8(quant8_unit(unorm8((float)(f.y & 0xFFu)) * a + dst[0] * ia));
                                    dst[1] = unorm8(quant8_unit(unorm8((float)(f.y >> 8 & 0xFFu)) * a + dst[1] * ia));
                                    dst[2] = unorm8(quant8_unit(unorm8((float)(f.y >> 16 & 0xFFu)) * a + dst[2] * ia));
                                    dst[3] = unorm8(quant8_unit(a + dst[3] * ia));
                                } else {
                                    col = f.y;
                                }
                            }
                        }
                    } while (m != 0 || left != 0);
                    s_dep[t] = dep;
                }
                __syncthreads();
            }
        }
        prev = best;
        first = false;
    }
    if (!live) return;
    if (shaded) {
        if constexpr (OVER)
            col = pack4((uint32_t)quant8_unit(dst[0]), (uint32_t)quant8_unit(dst[1]), (uint32_t)quant8_unit(dst[2]),
                        (uint32_t)quant8_unit(dst[3]));
        P.color[idx] = col;
        P.depth[idx] = dep;
    }
    if (counts) P.stencil[idx] = (uint8_t)st;
}

// Points are sparse (a few per tile), so a work-group reads and writes the
// pixels its points land on in place rather than staging the whole tile:
// it alone touches its tile's pixels, and the claim rounds' barriers order
// same-pixel points.
template <int FP, int BLEND>
__global__ __launch_bounds__(256) void k_raster_points(RasterParams P) {
    constexpr int KV = fp_varyings<FP>();
    __shared__ uint32_t claim[256];
    __shared__ float slut[256];
    const int t = threadIdx.x;
    const uint32_t tile = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t etx = tile % P.ntx, ety = tile / P.ntx;
    const uint32_t beg = P.tile_start[tile], end = P.tile_end[tile];
    if (beg >= end) return;
    slut[t] = (float)t / 255.0f;
    claim[t] = 0xFFFFFFFFu;
    __syncthreads();
    const Lut lut{slut};
    const int ex0 = (int)(etx * LP_ETS), ey0 = (int)(ety * LP_ETS);
    // Every point on a pixel belongs to the same screen tile, so list
    // (= point) order is the reference's per-pixel order.
    for (uint32_t b = beg; b < end; b += 256) {
        const uint32_t k = b + t;
        bool pending = false;
        int lp = 0;
        uint32_t v = 0;
        float x = 0.f, y = 0.f;
        size_t idx = 0;
        if (k < end) {
            const uint32_t pt = P.items[k];
            v = P.point_v ? P.point_v[pt] : pt;
            x = P.verts.comp(0)[v];
            y = P.verts.comp(1)[v];
            const uint32_t px = (uint32_t)x, py = (uint32_t)y;                  // point.rs:47
            lp = ((int)py - ey0) * LP_ETS + ((int)px - ex0);
            pending = px < P.W && py < P.H;  // binning keeps only such points
            idx = (size_t)py * P.W + px;
        }
        ordered_rounds(pending, lp, k, claim, [&]() {
            const uint32_t sv = P.stencil[idx];
            if (!stencil_test(P.s_test, sv, P.s_ref)) return;  // point.rs:293
            P.stencil[idx] = (uint8_t)stencil_op(P.s_op, P.s_wrap, sv, P.s_ref);
            const float z = P.verts.comp(2)[v];
            if (!(z < 0.0f && z >= P.depth[idx])) return;        // point.rs:300-306
            float kv[KV > 0 ? KV : 1];
#pragma unroll
            for (int c = 0; c < KV; c++) kv[c] = P.verts.var(v)[c];
            const uint32_t c = fragment<FP>(P, kv, lut);
            P.color[idx] = blend<BLEND>(c, P.color[idx], lut);
            P.depth[idx] = z;
        });
    }
}

#define SR_LP_DISPATCH(KERNEL)                                                                   \
    template <int FP>                                                                            \
    static void KERNEL##_blend(const RasterParams& P, uint32_t n, hipStream_t s) {              \
        if (P.blend == SR_BLEND_OVER)                                                            \
            hipLaunchKernelGGL((KERNEL<FP, SR_BLEND_OVER>), dim3(n), dim3(256), 0, s, P);        \
        else                                                                                     \
            hipLaunchKernelGGL((KERNEL<FP, SR_BLEND_REPLACE>), dim3(n), dim3(256), 0, s, P);     \
    }                                                                                            \
    static void KERNEL##_fp(const RasterParams& P, uint32_t n, hipStream_t s) {                 \
        switch (P.fp) {                                                                          \
            case SR_FP_BLINN_PHONG: KERNEL##_blend<SR_FP_BLINN_PHONG>(P, n, s); break;           \
            case SR_FP_TEX_LAMBERT: KERNEL##_blend<SR_FP_TEX_LAMBERT>(P, n, s); break;           \
            case SR_FP_UV_COLOR: KERNEL##_blend<SR_FP_UV_COLOR>(P, n, s); break;                 \
            default: KERNEL##_blend<SR_FP_FLAT>(P, n, s); break;                                 \
        }                                                                                        \
    }

SR_LP_DISPATCH(k_raster_lines)
SR_LP_DISPATCH(k_raster_points)

void launch_raster_lines(const RasterParams& P, uint32_t ntiles, hipStream_t s) {
    if (ntiles) k_raster_lines_fp(P, ntiles, s);
}
void launch_raster_points(const RasterParams& P, uint32_t ntiles, hipStream_t s) {
    if (ntiles) k_raster_points_fp(P, ntiles, s);
}

}  // namespace sr
