// sr_internal.hpp — types shared by the kernels (sr_kernels.hip) and the
// host runtime (sr_runtime.hip).  Nothing here crosses the C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/softrender_hip.h"

namespace sr {

constexpr int MAXK = 8;          // varyings per vertex
constexpr uint32_t DRAW_WORDS = 8;  // a draw's words in misc: errors, counts, flags
constexpr int SCAN_TILE = 4096;  // elements per scan / radix block (256 threads x 16)

// Triangles are binned to 32x32-pixel bins of the framebuffer (row-major),
// whatever the execution tile of the raster.  A bin pair's key holds the bin
// in its high half and in its low half one bit per 8x8 tile of the bin
// (row-major 4x4): the tiles where the triangle has to be tested.  A raster
// wave picks its own tiles' items out of its bin's list by those bits.  (One
// pair per 8x8 tile, the finer alternative, means 1.8 times the pairs to
// emit and sort on the 1080p frame of 1M small triangles and 11 times on
// triangles of a few thousand pixels.)  Framebuffers of more than
// MAX_MASKED_BINS bins keep the whole key for the bin; the raster then picks
// by the triangles' boxes.
constexpr uint32_t BIN_EDGE = 32;
constexpr uint32_t BIN_LOG2 = 5;
constexpr uint32_t MAX_MASKED_BINS = 65536;
constexpr int BIN_KEY_SHIFT = 16;  // of a masked key
// Every 8x8 tile of a bin that holds anything would read the bin's list and its
// own pixels, where most tiles of a sparse frame have no triangle.  So the end
// of a bin of up to MASK_ITEMS items is written as END_MASKED | their number <<
// 16 | the tiles that one of them has to be tested in (positions are below
// 2^31): in batches and in frames of MASK_BINS bins and more.  8,000 triangles
// of a few pixels each, frame without and with, us: 2560x1440 126, 106; 1080p
// 97, 85.  Smaller frames have less to skip than the masks cost (512x512 sphere
// 103 without, 105 with).
constexpr uint32_t END_MASKED = 1u << 31;
constexpr uint32_t MASK_ITEMS = 16;  // (with 16 triangles of a tile each a third of the tiles has none)
constexpr uint32_t MASK_BINS = 2000;
// A draw of few triangles is binned directly (k_bin_direct): one work-group
// per bin looks through all triangles' bin boxes, so nothing is counted,
// scanned, emitted or sorted.  An item is id << 16 | tile mask in one word,
// and every bin has room for all triangles (DIRECT_WORK words at most), so
// no place is asked for (an atomic add on one word per bin took 20 ns each)
// and nothing overflows.  Every work-group reads every triangle's box, so past
// some number sorting is faster; few bins are few work-groups, which is sooner.
// Frames of triangles of 3, 25 and 50 pixels, us, direct / sorted: 64x64 with
// 8,000 triangles 73, 108, 119 / 93, 107, 115, with 32,000 154, 289, 314 / 134,
// 173, 193; 512x512 with 28,000 85, 142, 148 / 85, 142, 196; 1366x768 with 20,000
// 112, 177, 197 / 110, 164, 236, with 32,000 141, 225, 245 / 116, 181, 248; 4K with
// 3,000 112, 185, 255 / 118, 177, 277, with 4,000 213, 291, 364 / 139, 204, 309.
constexpr uint32_t DIRECT_TRIS = 32768;           // (an id has 16 bits)
constexpr uint64_t DIRECT_WORK = 24ull << 20;     // boxes read by all work-groups
constexpr uint32_t DIRECT_FEW_BINS = 8192, DIRECT_BIN_TRIS = 512;  // at most the one + the other a bin
__host__ __device__ inline bool binned_directly(uint32_t ntris, uint32_t nbins) {
    return ntris <= DIRECT_TRIS && nbins <= MAX_MASKED_BINS && (uint64_t)ntris * nbins <= DIRECT_WORK &&
           ntris <= DIRECT_FEW_BINS + (uint64_t)DIRECT_BIN_TRIS * nbins;
}
static_assert(DIRECT_TRIS <= 65535, "ids of 16 bits");
// Triangles of more than 32 bins ("wide") are listed apart, so that whole
// work-groups emit their pairs; past WIDE_CAP of them one lane emits each.
constexpr uint32_t WIDE_CAP = 65536;
constexpr uint32_t WIDE_BINS = 32;
constexpr uint32_t WIDE_CLAMP_EDGE = 16384;  // framebuffer edge up to which wide BIN_CLAMP triangles are listed

// Screen- (or clip-) space vertices in one allocation: the position as
// four streams (x, y, z, w: the setup and binning passes read x, y, z
// coalesced), then the varyings interleaved per vertex, `kstride` floats a
// row (a shaded fragment reads each of its three vertices' varyings as one
// short contiguous row instead of one word from each of K streams).
//   comp(c)[i] = position component c of vertex i (c < 4)
//   var(i)[k]  = varying k of vertex i (k < kstride)
// stride = capacity in vertices.
struct VertexBuf {
    float* base;
    uint32_t stride;
    uint32_t kstride;
    __host__ __device__ float* comp(int c) const { return base + (size_t)c * stride; }
    __host__ __device__ float* var(uint32_t i) const { return base + 4 * (size_t)stride + (size_t)i * kstride; }
};

// Per-triangle setup record, written once by k_tri_setup and read by every
// raster workgroup whose tile the triangle touches: 64 bytes, one cache
// line, what the raster's per-triangle loop reads (from LDS, where a block's
// records are staged).  The triangle's vertex ids, needed only to shade, are kept apart (TriVid).
struct alignas(64) TriRec {
    // bytes 0-47: what the raster tests every pixel with (staged into LDS
    // 16 bytes at a time); 48-63: the box, read where a mode needs it
    double R;             // RN64(1 / (double)det): f32 quotients are formed as (float)(num * R)
    uint32_t zs;          // bit 0 (strip): a pixel centre outside the box may pass the
                          // coverage test; the raster tests the box clamped into each
                          // screen tile (clamp_as_int!), as the reference does.
                          // Bits 1..31: depth_key(zhi) rounded up to even, zhi an
                          // upper bound of every depth the triangle can write
                          // (depth_bound_key)
    float x3, y3;         // screen position of the third vertex
    float e23y, e23x;     // (y2 - y3), (x3 - x2)   — triangle.rs:108
    float e31y, e31x;     // (y3 - y1), (x1 - x3)   — triangle.rs:109
    float z1, z2, z3;
    int32_t X0, X1, Y0, Y1;  // floor of the f32 bbox, clamped to [-1, W] x [-1, H]
};
static_assert(sizeof(TriRec) == 64, "TriRec layout");

// Order-preserving key of an f32 (a < b  <=>  key(a) < key(b) for all
// non-NaN a, b, with -0 just below +0); a NaN of either sign lies beyond
// the infinity of its sign.
__host__ __device__ __forceinline__ uint32_t depth_key(uint32_t bits) {
    return bits ^ ((uint32_t)((int32_t)bits >> 31) | 0x80000000u);
}

// The vertex ids of a triangle in the screen vertex buffer (the shading
// gathers' addresses).
struct TriVid {
    uint32_t i0, i1, i2;
};
static_assert(sizeof(TriVid) == 12, "TriVid layout");

// Per-triangle binning record: what pair emission reads (the pixel box
// whose execution tiles get the triangle and the coverable-tile mask),
// apart from the full record for culled boxes of more than 32 tiles.
// Kept apart from TriRec so emission streams 24 bytes per triangle
// instead of 88.
enum BinMode : uint32_t {
    BIN_BOX = 0,    // the 8x8 tiles of the box (or of its mask, with culling)
    BIN_REACH = 1,  // every tile of X0..Y1: the box grown to the pixels that may pass
    BIN_CLAMP = 2,  // every bin meeting the box clamped into some screen tile
    BIN_BINS = 3,   // culled, over 32 tiles but at most 32 bins: the bins of the mask
    BIN_ROWS = 4,   // culled, over 32 bins: the covered run of bins of each bin row
};
struct TriBin {
    int32_t X0, X1, Y0, Y1;  // the box, or the reach (BIN_REACH)
    uint32_t tmask;          // BIN_BOX with culling: bit i = i-th 8x8 tile of the box
                             // (row-major) may be covered; BIN_BINS: the same for bins
    uint32_t mode;           // BinMode, | BIN_WIDE when the wide list holds the triangle
};
constexpr uint32_t BIN_WIDE = 8;
static_assert(sizeof(TriBin) == 24, "TriBin layout");

// Per (line, screen tile) work item: the segment clipped to one screen
// tile by liang_barsky_iterative (geometry/line.rs:6-54), as rasterize_line
// receives it (line.rs:51-52).  80 bytes.
struct alignas(16) LineItem {
    uint32_t line;        // primitive index
    uint32_t tile;        // screen tile index (row-major, the reference's tile order)
    uint32_t plot_off;    // first plot record
    uint32_t plot_cnt;    // number of plot records
    float cx1, cy1;       // clipped start
    float cx2, cy2;       // clipped end
    float dlen;           // hypot of the clipped segment, line.rs:52
    int16_t bx0, by0, bx1, by1;  // execution tiles touched by its plots (bx0 > bx1: none)
    // LINE_MASK: the execution tiles that hold a plot, as bits mlo, mhi
    // (row-major, mcols per row) of a window starting at tile (mbx, mby)
    uint16_t mbx, mby, mcols;
    uint16_t flags;       // LineFlags
    // LINE_RANGED: plots 0..3 are the endpoints and plot 4 + 2i + {0, 1} lies
    // on major coordinate major0 + i (the pixel column, or row when steep)
    int32_t major0;
    float zs, ze;         // depths of the line's ends
    uint64_t mlo, mhi;
};
static_assert(sizeof(LineItem) == 80, "LineItem layout");
enum LineFlags : uint16_t {
    LINE_MASK = 1,     // else its tiles are the box's
    LINE_RANGED = 2,   // a Wu walk that is sampled, or dropped and wrapped no plot
    LINE_STEEP = 4,
    LINE_SAMPLED = 8,  // its interior plots are kept as samples (LINE_STEP)
    LINE_WRAPS = 16,   // sampled: some plots wrap to the next row
};

// A Wu walk inside the frame (line_inside) whose plots would take more room
// keeps only its four endpoint plots (row ~0: dropped) and, after them, samples
// of the walk: doubles, the gradient, then the minor coordinate at the first
// interior major coordinate major0 and at each later one that is a multiple of LINE_STEP
// (the edge of the raster's tiles, so a tile's plots follow from one sample by
// the walk's own additions).
constexpr uint32_t LINE_STEP = 16;

// One plot of a line item: framebuffer index (x + y*W, line.rs:56-58), the
// plot coordinates (for the pixel centre in line.rs:72-73) and the
// coverage alpha in f64 as draw_line_xiaolin_wu computes it.
struct alignas(8) Plot {
    double alpha;
    uint32_t index;
    int32_t x, y;
    uint32_t row;  // index / W: the pixel's row (its column is index - row * W)
};
static_assert(sizeof(Plot) == 3 * sizeof(double), "samples are counted in thirds of a Plot");
static_assert(sizeof(Plot) == 24, "Plot layout");

// Everything a raster workgroup needs, passed by value.
struct RasterParams {
    // framebuffer
    uint32_t W, H;
    uint32_t* color;
    float* depth;
    uint8_t* stencil;
    const uint32_t* strip_counts;  // per-pixel stencil visits outside bboxes (or null)
    // screen tiles of the reference (inclusive rectangles, fragment.rs:188-216)
    uint32_t tw, th;
    uint32_t scols, srows;
    // execution tiles
    uint32_t ets, ntx, nty;
    int nwv;                // waves sharing an execution tile (1, 2 or 4)
    const uint32_t* tile_start;
    const uint32_t* tile_end;
    const uint32_t* items;  // sorted item ids per execution tile (triangles: per bin)
    // triangles: tile_start / tile_end are indexed by bin, nbx bins a row;
    // keys[i] is item i's bin key when the bins are masked (else null);
    // packed: items[i] = id << 16 | tile mask (keys null); a bin's end may be
    // END_MASKED
    const uint32_t* keys;
    int packed;
    uint32_t nbx;
    // primitives
    const TriRec* tris;
    const TriVid* vids;     // per triangle, beside tris; null: triangle t's vertices are 3t, 3t+1, 3t+2
    const LineItem* line_items;
    const Plot* plots;
    VertexBuf verts;        // screen-space vertices
    const uint32_t* line_v; // 2 vertex ids per line
    const uint32_t* point_v;// vertex id per point
    uint32_t n_prims;
    int K;
    // programs
    int fp, blend, alpha_mode;
    int s_test, s_op, s_wrap;
    uint32_t s_ref;
    int smode;              // 0: stencil untouched, 1: count visits, 2: track in order, 3: test only
    int exhaustive;         // every triangle in every tile: the box is clamped into each
                            // screen tile exactly as clamp_as_int! does
    const uint32_t* tex;    // RGBA8 texels, or RGBAF32 (4 floats each) when tex_fmt says so
    int tex_fmt;            // SR_COLOR_*
    uint32_t texW, texH;
    int tex_filter, tex_edge;
    uint32_t tex_border;
    float fsu[32];
    // non-null: nothing is drawn when skip_if[0] bit 0 (a NaN screen
    // coordinate) or skip_if[4] (the bins overflowed) is set
    const uint32_t* skip_if;
    // batch: this scene's first global execution tile and bin, and a fused clear
    // (Framebuffer::clear, renderbuffer/mod.rs:125-133) applied on load
    uint32_t tile_base, bin_base;
    int clear;
    uint32_t clear_rgba;
};

// Framebuffers of other formats (sr_fb_create_ex): the colour planes, the
// depth plane of f64 depth, and how stencil behaves.
struct FmtParams {
    void* planes[SR_MAX_COLOR_PLANES];
    int color_fmt[SR_MAX_COLOR_PLANES];
    uint32_t n_color;
    double* depth64;      // f64 depth (else RasterParams::depth)
    int track_stencil;    // u8 stencil with a test or op: tracked per pixel in order
    int has_stencil;      // 0: `()` stencil, no plane
};

// Raster launch: one scene given inline (one work-group per tile), or a
// batch: a table of draws ("scenes") grouped by framebuffer, each group's
// draws consecutive and in item order; the groups' execution tiles (all
// tiles of every bin, bin by bin) are numbered globally
// [group_tile_end[g-1], group_tile_end[g]) and split
// into runs of near-equal cost, one per work-group of a persistent grid.
struct RasterBatch {
    RasterParams one;
    const RasterParams* scenes;      // null: use `one`
    const uint32_t* group_tile_end;  // inclusive prefix of tiles per group
    const uint32_t* group_first;     // first draw of each group; [ngroups] = draw count
    const uint32_t* tri_end;         // per draw: exclusive end of its batch triangle ids
    uint32_t ngroups;
    uint32_t tile0, ntiles;          // global tile range of this launch
    const uint32_t* wg_start;        // run p = tiles [tile0 + wg_start[p], tile0 + wg_start[p+1])
    const uint32_t* overflow;        // [0] binning overflowed, [2] bit 0: a NaN screen coordinate:
                                     // either draws nothing (no fused clear either)
};

}  // namespace sr
