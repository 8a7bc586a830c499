// sr_kernels.hpp — kernel parameter blocks and host-side launchers.
#pragma once

#include "sr_internal.hpp"

namespace sr {

struct VSParams {
    const float *px, *py, *pz, *nx, *ny, *nz, *u, *v;
    const int32_t* ia;  // integer attribute (SR_VP_MVP_INT), or null
    uint32_t n;
    int program;
    int K;
    int normalize;  // 1: run_to_fragment (viewport fused), 0: keep clip space
    sr_viewport viewport;
    float U[48];
    VertexBuf out;
    uint32_t* misc;  // the draw's DRAW_WORDS words to clear, or null
};

struct GSParams {
    VertexBuf in;        // clip-space vertices
    const uint32_t* idx; // mesh indices (null: implicit)
    uint32_t n_in;       // input primitives
    int K;
    uint32_t* counts;    // outputs per input primitive
    const uint32_t* offsets;
    VertexBuf out;       // generated vertices, screen space (finish fused)
    sr_viewport viewport;
    float G[17];         // normal visualisation: projection * view (row-major), length
};

struct SetupParams {
    VertexBuf v;
    const uint32_t* idx;  // null: vertex 3t+k
    uint32_t n;
    int cull;
    uint32_t W, H;
    uint32_t tw, th;  // screen tiles (clamp_as_int!'s boxes)
    TriRec* recs;
    TriBin* bins;
    TriVid* vids;
    uint32_t* counts;
    uint32_t* err;
    uint32_t* wide;    // WIDE_CAP triangle ids, their number in *wide_n
    uint32_t* wide_n;
    int empty_cull;  // bin only what the triangle may cover (no stencil effects)
    // direct binning: per triangle its bins, columns lo | hi << 16 and rows
    // (lo > hi: none), in place of counts and the wide list; else null.  The
    // last work-group reports misc[0] (launch_report).
    uint2* boxes;
    uint32_t* to;
    uint32_t seq;
};

// Direct binning: bin b's items (id << 16 | tile mask, in triangle order) from
// list[b * stride].
struct DirectParams {
    const uint2* boxes;
    const TriRec* recs;
    const TriBin* bins;
    uint32_t n, W, H, nbx, tw, th;
    int empty_cull;
    uint32_t stride;
    uint32_t* list;
    uint32_t* start;  // per bin
    uint32_t* end;
    int masks;        // ends may be END_MASKED
};

struct EmitParams {
    const TriRec* recs;
    const TriBin* bins;
    const uint32_t* counts;
    const uint32_t* offsets;
    uint32_t cap;  // pairs keys/vals hold: a triangle whose pairs would pass it writes none
    uint32_t n, W, H, nbx;
    uint32_t tw, th;  // screen tiles
    const uint32_t* wide;
    const uint32_t* wide_n;
    uint32_t* keys;
    uint32_t* vals;
    int empty_cull;
    int masked;  // keys carry the tile mask (at most MAX_MASKED_BINS bins)
    uint32_t split;  // waves sharing 64 triangles (1 or 4; set at the launch)
};

// One scene of a batch: its vertex program, mesh streams and placement in
// the batch's vertex / triangle / execution-tile numbering.
struct SceneGeom {
    const float *px, *py, *pz, *nx, *ny, *nz, *u, *v;
    const uint32_t* idx;      // null: vertex 3t+k
    uint32_t nv, vbase;       // vertices, first batch vertex
    uint32_t nt, tbase;       // triangles, first batch triangle
    int program, K, cull;
    uint32_t W, H, nbx;
    uint32_t tw, th;  // screen tiles
    int empty_cull;
    sr_viewport viewport;
    float U[48];
};

struct BatchTables {
    const SceneGeom* scenes;
    const uint32_t* vend;  // inclusive prefix of vertices per scene
    const uint32_t* tend;  // inclusive prefix of triangles per scene
    uint32_t nscenes, nv, nt;
};

struct LineSetupParams {
    VertexBuf v;
    const uint32_t* idx;   // null: vertices 2l, 2l+1
    uint32_t n_lines;
    uint32_t W, H, tw, th, scols, srows;
    uint32_t* counts;      // per line: accepted screen tiles
    const uint32_t* offsets;
    LineItem* items;
    uint32_t* err;
    int aa;                // Wu (1) or Bresenham (0) walks
    uint32_t* walk_len;    // pass 1 (optional): per item, a sort key, 255 - its walk length (capped)
    uint32_t* plot_ub;     // pass 1: per item, room for its plots (the walk's plot calls) or its samples
};

struct WalkParams {
    LineItem* items;
    uint32_t n_items;
    uint32_t W, H;
    int aa;
    uint32_t ets, ntx, nty;
    uint32_t tw, th, scols;  // screen tiles
    const uint32_t* order;   // optional: thread t walks item order[t] (items of similar length share a wave)
    const uint32_t* plot_ub;       // per item: room for its plots or samples (an upper bound)
    const uint32_t* plot_offsets;  // per item: first plot slot (exclusive scan of plot_ub)
    uint32_t* bin_counts;    // out: execution tiles per item
    Plot* plots;             // out
    uint32_t* err;
};

struct ItemEmitParams {
    const LineItem* items;
    const uint32_t* counts;
    const uint32_t* offsets;
    uint32_t n, ntx;
    uint32_t* keys;
    uint32_t* vals;
};

struct PointSetupParams {
    VertexBuf v;
    const uint32_t* idx;
    uint32_t n;
    uint32_t W, H, tw, th, scols, ets, ntx;
    uint32_t* counts;   // 0/1
    const uint32_t* offsets;
    uint32_t* keys;
    uint32_t* vals;
    int pass;
};

struct StripParams {
    const TriRec* recs;
    uint32_t n;
    uint32_t W, H, tw, th, scols, srows;
    uint32_t* colL;  // [scols+1][H+1]  rows of column tx0_j, difference along y
    uint32_t* colR;  // [scols+1][H+1]  from the last tile column back
    uint32_t* rowT;  // [srows+1][W+1]
    uint32_t* rowB;  // [srows+1][W+1]  from the last tile row back
    // corners [srows+1][scols+1]: LL, LR, RL, RR (left / right x above / below),
    // and with colS the boxes of one tile
    uint32_t* corners;
    uint32_t* colS;  // [scols][H+1]  boxes of one tile column, for colL and colR, or null
    uint32_t* rowS;  // [srows][W+1]  boxes of one tile row, for rowT and rowB (with colS)
    uint32_t* out;   // per pixel
};

void launch_vertex(const VSParams& P, hipStream_t s);
// clip space -> screen space (finish) for n vertices with K varyings
void launch_finish(const VertexBuf& in, const VertexBuf& out, uint32_t n, int K, const sr_viewport& vp,
                   hipStream_t s);
void launch_gs_count(int mode, int prim, const GSParams& P, hipStream_t s);
void launch_gs_emit(int mode, int prim, const GSParams& P, hipStream_t s);
// normal visualisation on a triangle list: lines (2 vertices each) into P.out,
// 3 per triangle (SR_GS_VERTEX_NORMALS) or 1 (SR_GS_FACE_NORMALS)
void launch_gs_normals(int mode, const GSParams& P, hipStream_t s);
void launch_tri_setup(const SetupParams& P, hipStream_t s);
void launch_tri_emit(const EmitParams& P, hipStream_t s);
void launch_bin_direct(const DirectParams& P, uint32_t nbins, hipStream_t s);
void launch_vertex_batch(const BatchTables& T, const VertexBuf& out, hipStream_t s);
void launch_tri_setup_batch(const BatchTables& T, const VertexBuf& v, TriRec* recs, TriBin* bins, TriVid* vids,
                            uint32_t* counts, uint32_t* err, uint32_t* wide, uint32_t* wide_n, hipStream_t s);
void launch_tri_emit_batch(const BatchTables& T, const TriRec* recs, const TriBin* bins, const uint32_t* counts,
                           const uint32_t* offsets, uint32_t cap, const uint32_t* wide, const uint32_t* wide_n,
                           int masked, uint32_t* keys, uint32_t* vals, uint32_t* overflow, hipStream_t s);
uint32_t scan_tmp_words(uint32_t n);
// exclusive scan of in[0..n) (or of the first *count elements, count <= n)
void launch_scan(const uint32_t* in, uint32_t* out, uint32_t n, uint32_t* tmp, uint32_t* total,
                 hipStream_t s, const uint32_t* count = nullptr);
uint32_t radix_hist_words(uint32_t n);
// returns 1 if the sorted data ended up in the *_tmp buffers
// n_dev (optional): the element count in device memory, at most n; then
// total[1] is used as scratch
// (sorts by bits [shift, shift + key_bits) of the keys)
int radix_sort(uint32_t* keys, uint32_t* vals, uint32_t* keys_tmp, uint32_t* vals_tmp, uint32_t n,
               int shift, int key_bits, uint32_t* hist, uint32_t* scan_tmp, uint32_t* total, hipStream_t s,
               const uint32_t* n_dev = nullptr);

// Segmented sort of a batch's (bin, triangle) pairs: the pairs of each
// framebuffer group are already contiguous and in group order (they are
// emitted triangle by triangle), so each group's run is sorted apart by its
// keys' bins, which are numbered within the group's framebuffer.  That takes
// the passes the largest framebuffer's bin count needs.  `segs` holds
// 3 * ngroups + 2 words of scratch (first, lo, hi); the histograms
// need radix_hist_words(cap) + 256 * (ngroups + 1) words.  Sorts the first
// *live of `cap` pairs; returns 1 if the result is in the *_tmp buffers.
struct BatchGroups {
    const uint32_t* tend;            // per draw: inclusive prefix of triangles
    const uint32_t* group_first;     // per group: first draw (+1 entry)
    uint32_t ngroups, ntris;
};
int radix_sort_groups(uint32_t* keys, uint32_t* vals, uint32_t* keys_tmp, uint32_t* vals_tmp, uint32_t cap,
                      int shift, int key_bits, const BatchGroups& G, const uint32_t* tri_offsets,
                      const uint32_t* live, uint32_t* segs, uint32_t* hist, uint32_t* scan_tmp,
                      uint32_t* total, hipStream_t s);
void launch_fill(uint32_t* p, uint32_t v, uint32_t n, hipStream_t s);
// start/end of tiles [0, nkeys) in keys[0, n) (sorted by key >> shift), by
// binary search: every tile written, no clearing needed.  n_dev: the key
// count on the device (at most n), when only the device knows it.  masks:
// ends may be END_MASKED (masked keys).
void launch_ranges_search(const uint32_t* keys, uint32_t n, uint32_t nkeys, int shift, uint32_t* start,
                          uint32_t* end, hipStream_t s, const uint32_t* n_dev = nullptr, bool masks = false);
// The same for a batch: bin b of nbins belongs to the group g with
// group_bin_end[g-1] <= b < group_bin_end[g], whose keys (numbered within the
// group) lie in [lo[g], hi[g]).
void launch_ranges_groups(const uint32_t* keys, const uint32_t* lo, const uint32_t* hi,
                          const uint32_t* group_bin_end, uint32_t ngroups, uint32_t nbins, int shift, bool masks,
                          uint32_t* start, uint32_t* end, hipStream_t s);
// p[i] = pat[i % period] over n_words 32-bit words (period 1, 2 or 4)
void launch_fill_pattern(void* p, const uint32_t pat[4], uint32_t period, size_t n_words, hipStream_t s);
void launch_iota(uint32_t* p, uint32_t n, hipStream_t s);  // p[i] = i
// misc[live_word] = misc[overflow_word] ? 0 : misc[total_word]
void launch_live_pairs(uint32_t* misc, int overflow_word, int total_word, int live_word, hipStream_t s);
// misc[4] = misc[1] > cap; misc[5] = pairs to sort (0 on overflow or a NaN
// flag in misc[0]); misc[0..2) reported to the host (launch_report)
void launch_bins_live(uint32_t* misc, uint32_t cap, uint32_t* to, uint32_t seq, hipStream_t s);
// misc[0..n) to pinned host memory at `to`, then seq to to[REPORT_SEQ]
constexpr uint32_t REPORT_SEQ = 15;
void launch_report(const uint32_t* misc, uint32_t n, uint32_t* to, uint32_t seq, hipStream_t s);
// the same of one word, the items of bins [0, nbins)
void launch_report_items(const uint32_t* start, const uint32_t* end, uint32_t nbins, uint32_t* to, uint32_t seq,
                         hipStream_t s);
// persistent-raster partition: cost[t] = fixed + an estimate of tile t's
// items from its bin's (bin t >> tpb_log2) for t < n, cost[n] = 0 (scan the
// costs of all classes into a prefix), then G runs of near-equal cost over
// tiles [tile0, tile0 + n): wg_start[0..G]
void launch_tile_cost(const uint32_t* start, const uint32_t* end, uint32_t n, uint32_t tpb_log2, uint32_t fixed,
                      uint32_t* cost, hipStream_t s);
void launch_partition(const uint32_t* prefix, uint32_t tile0, uint32_t n, uint32_t G, uint32_t* wg_start,
                      hipStream_t s);
void launch_fb_clear(uint32_t* color, float* depth, uint8_t* stencil, uint32_t n, uint32_t rgba,
                     float d, uint32_t st, hipStream_t s);
// grid = (tiles per bin) x bins work-groups (inline scene) or a persistent grid (scene table);
// the batch's `one` carries the launch-wide program choice (fp, blend, smode, ets)
void launch_raster_tris(const RasterBatch& P, uint32_t grid, hipStream_t s);
// The raster for other framebuffer formats, the multi-output program and the
// normalised over-blend (sr_raster_fmt.hip): 8x8 execution tiles.
void launch_raster_fmt(const RasterParams& P, const FmtParams& F, uint32_t ntris, uint32_t ntiles, hipStream_t s);
void launch_raster_tris_8(const RasterBatch& P, uint32_t grid, hipStream_t s);
void launch_raster_tris_16(const RasterBatch& P, uint32_t grid, hipStream_t s);
void launch_raster_tris_32(const RasterBatch& P, uint32_t grid, hipStream_t s);

// lines / points / stencil strips
void launch_line_tiles(const LineSetupParams& P, int pass, hipStream_t s);
void launch_line_walk(const WalkParams& P, hipStream_t s);
void launch_item_emit(const ItemEmitParams& P, hipStream_t s);
void launch_point_setup(const PointSetupParams& P, hipStream_t s);
void launch_raster_lines(const RasterParams& P, uint32_t ntiles, hipStream_t s);
void launch_raster_points(const RasterParams& P, uint32_t ntiles, hipStream_t s);
void launch_strips(const StripParams& P, hipStream_t s);

}  // namespace sr
