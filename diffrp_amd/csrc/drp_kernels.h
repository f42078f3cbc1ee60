// Launch descriptors shared by the kernel files and the C-ABI layer.
#pragma once
#include <hip/hip_runtime.h>
#include "drp_common.h"

namespace drp {

// Uneven batches (items of different resolutions and meshes, packed back to
// back): prefix sums over the items of their pixels, vertices, triangles and of
// the tiles each pass uses.  The item a work unit (block, tile, pixel) belongs
// to is the last item whose prefix is <= the unit's index (um_find).  n = 0:
// uniform batch, every image [H, W] of the launch.
struct UnevenMap {
    const long long *pix;   // [n + 1] pixel offsets
    const int *vert;        // [n + 1] vertex offsets
    const int *tri;         // [n + 1] triangle offsets
    const int *bt16;        // [n + 1] 16 x 16 tiles (deterministic backward)
    const int *blk;         // [n + 1] 64 x 8 blocks (antialias)
    const int *hw;          // [2 n] (H, W) per item
    int n;
};

template <typename T>
__device__ __forceinline__ int um_find(const T *pre, int n, T x) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (pre[mid] <= x) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Pixel box of one (image, triangle) from the forward setup: columns c0..c1 in
// cc (c0 | c1 << 16), rows r0..r1 in rr; c0 > c1 when empty.  hit is set by the
// forward when the triangle won at least one pixel of that image.
struct ItemBox {
    int cc, rr, hit;
};

// heavy-tile split of the fine raster: control words after the bin and list
// counters, at most this many split tiles per call
constexpr int kSplitCtl = 4;
constexpr int kSplitSlotsMax = 4096;
inline int split_slots(long long n_tiles) { return (int)(n_tiles < kSplitSlotsMax ? n_tiles : kSplitSlotsMax); }
// per slot: int4 of bookkeeping, a done counter, 63 queued chunks, 256 depth keys
inline size_t split_region_bytes(int slots) { return (size_t)slots * (16 + 4 + 4 * 63 + 8 * 256); }

struct AALaunch;

struct RasterLaunch {
    Batch b;
    const float *pos;
    const int *tri;
    int tile_w, tile_h;
    int *bin_count;   // [n_tiles], immediately followed by list_count [n_img] and split_ctl [kSplitCtl]
    int *list_count;
    char *split_base; // heavy-tile split region (split_region_bytes(split_slots))
    int split_slots;
    int *bins;        // [n_tiles * bin_cap]
    int *lists;       // spill lists
    int4 *setup;      // setup records: two int4 per (image, triangle), at the image's list offset
    ItemBox *boxes;   // optional [n_img, F] pixel box + hit flag per (image, triangle)
    int n_tiles;
    int max_tris;     // largest triangle range of any image
    const float *prev;
    float *rast;
    float *rast_db;
    const AALaunch *aa_prepare;  // optional: the antialias preparation, run beside the fine raster
    int depth_cull;   // fine raster with the depth cull (depth_cull_wanted)
};

// The fine raster culls triangles by depth where bins hold more than
// kCullRounds rounds of a tile's lanes (a bin capacity learnt or tuned from
// the exact counts is the largest count + 15 %, rounded up to a power of two).
constexpr int kCullRounds = 4;
inline int depth_cull_wanted(int bin_cap, int tile_w, int tile_h) {
    return bin_cap > kCullRounds * tile_w * tile_h ? 1 : 0;
}

struct RasterBwdLaunch {
    Batch b;
    const float *pos;
    const int *tri;
    const float *rast, *grad_rast, *grad_db;
    float *grad_pos;
    long long total_pix;
    int pix_per_img;
    // triangle-centric path (all set) or per-pixel atomics (any null)
    const ItemBox *boxes;
    float *partial;          // [n_img, 3F] float4
    void *records;           // tile records (tile_records_bytes(n_img, H, W, 12, n_img * F))
    unsigned char *live;     // [n_img, F]: the partial's written triangles
    const int *inc_off, *inc;
    UnevenMap um;            // uneven batch (um.n > 0): packed items, global vertices
    long long um_tiles;      // uneven batch: 16 x 16 tiles of all items
    int local_ids;           // uneven batch: rast ids count from each item's first triangle (else global)
};

struct InterpLaunch {
    const float *attr;
    int V, C, attr_batched;
    int cv;           // compiled channel variant (0 = generic loop)
    const float *rast;
    const int *tri;
    int F;
    long long total_pix, pix_per_img;
    const float *rast_db;
    const int *diff_idx;
    int n_diff;
    float *out, *out_da;
    const float *grad_out, *grad_da;
    float *grad_attr, *grad_rast, *grad_db;
    // triangle-centric backward (all set) or per-pixel atomics (any null)
    int H, W;
    const ItemBox *boxes;
    float *partial;          // [groups, F, 3, min(C, kMaxPassChannels)]
    unsigned char *live;     // [groups, F]
    void *records;           // tile records of min(C, kMaxPassChannels) channels
    const int *inc_off, *inc;
    int views_per_group;
    UnevenMap um;            // uneven batch (um.n > 0): packed items, global ids and vertices, one group
    long long um_tiles;      // uneven batch: 16 x 16 tiles of all items
};

struct TopoLaunch {
    const int *tri;
    int F;
    unsigned long long *keys;
    int *cnt;
    int2 *slots;
    unsigned mask;
    int *opp;
};

// pixels of an antialias block, and what the forward leaves of it beside its
// list of blending pairs: which pairs are listed (right, up per row) and the
// weights of the pairs that reach in from below and from the left
constexpr int kAAW = 64, kAAH = 8;
struct AAHalo {
    unsigned long long mask[2 * kAAH];
    float below[kAAW], left[kAAH];
};

struct AALaunch {
    const float *color, *rast, *pos;
    const int *tri, *opp;
    int n_img, H, W, C, V, F, pos_batched;
    double2 *proj;               // [n_proj, V] pixel coordinates (NaN: w <= 0)
    signed char *orient;
    unsigned char *silh;
    float *ent_w;                // [2 x pixels] weights of the blending pairs, a run per block
    unsigned *ent_word;          // [2 x pixels] their edges
    AAHalo *halo;                // [blocks]
    int reuse;                   // backward: workspace holds the forward's state
    int prepared;                // forward: drp_antialias_prepare filled the per-vertex / per-triangle state
    float *out;                  // forward (nullptr: the pair lists alone)
    const float *grad_out;
    float *grad_color, *grad_pos;
    float boost;
    UnevenMap um;                // uneven batch (um.n > 0): n_img items, packed; pos / tri global
    int total_blk;               // uneven batch: blocks of all items
    int xcd;                     // blocks per XCD turn (set at launch)
};

struct PartitionLaunch {
    const float *rast;  // one layer of npx pixels, W wide
    long long npx;
    int W;
    const int *stencils;  // [F + 1]
    int F, n_owner;
    int *order, *starts, *ends;
    float *frag;            // [n_frag, 4] or nullptr (then rows and cols are not written either)
    long long n_frag;       // at least npx; the rest is zeroed
    long long *rows, *cols;
};

// channels of one pass of the tile backward (wider attributes take several)
constexpr int kMaxPassChannels = 16;

// tiles of a triangle's pixel box whose record index the tile pass stores
constexpr int kBoxSlots = 4;

struct TriBwdLaunch {
    Batch b;
    const float *pos;
    const int *tri;
    const float *rast, *grad_rast, *grad_db, *grad_out;
    const float *attr;       // attribute mode: attributes (for grad_rast)
    int V, attr_batched;
    int ldc, c0;             // attribute mode: row stride of attr and grad_out, first channel of this pass
    int accum;               // attribute mode: a later chunk of channels, added to grad_rast_out (and grad_db_out)
    float *grad_rast_out;    // attribute mode: grad_rast written by the tile pass (fused mode: null skips it)
    const float *rast_db, *grad_da;  // attribute mode, n_diff > 0: gradients [.., 2 n_diff] of the derivatives
    const int *diff_idx;             //   of channels diff_idx[n_diff]
    int n_diff;
    float *grad_db_out;      // nullable
    const ItemBox *boxes;
    float *partial;
    float *partial_pos;      // fused mode: the position partial [n_img, 3F] float4 (partial: attributes)
    unsigned char *live, *live_pos;  // [groups, F], fused mode [n_img, F]: triangles whose partials are written
    int n_img, F, H, W;
    int views_per_block;     // images summed per partial (attribute mode); 1 for positions
    // per-tile records (16 x 16 tiles): count, triangle, sums
    int *rec_count, *rec_t;
    float *rec_v;
    int *box_slot;           // [boxes, kBoxSlots] record index of the box's first tiles (nullptr: search)
    int tiles_x, tiles_per_img, n_tiles, n_tiles_pad;
    int xcd_tiles;           // tiles per XCD turn
    UnevenMap um;            // uneven batch (um.n > 0): tiles of all items, one group
    int local_ids;           // uneven batch: rast ids count from each item's first triangle (else global)
};

// Fork / join onto the device's auxiliary stream (drp_fork.hip).  fork_begin
// returns false (f.side null) when there is none: run everything on `main`.
struct Fork {
    hipStream_t side;
    hipEvent_t join;
};
bool fork_begin(hipStream_t main, Fork &f);
int fork_end(hipStream_t main, const Fork &f);

// C: channels of the pass, 1 .. 16 (with n_diff > 0: 1 .. 4); a multiple of 4
// only where ldc is one too (16-byte rows)
int launch_tri_bwd_pos(const TriBwdLaunch &L, hipStream_t st);
int launch_tri_bwd_attr(const TriBwdLaunch &L, int C, hipStream_t st);
int launch_tri_bwd_fused(const TriBwdLaunch &L, int C, hipStream_t st);
// partial (and its live triangles) [groups, F, 3, C] added to channels [c0, c0 + C) of grad_attr rows of ldc
// floats; outs outputs, one group each when per_output
int launch_gather_attr(const float *partial, const unsigned char *live, int groups, int F, int V, int C, int ldc,
                       int c0, int outs, int per_output, const int *inc_off, const int *inc, float *grad_attr,
                       hipStream_t st);
int launch_gather_pos(const float *partial, const unsigned char *live, int n_img, int F, int V, int pos_batched,
                      const int *inc_off, const int *inc, float *grad_pos, hipStream_t st);
// both, after launch_tri_bwd_fused(T, C, ..)
int launch_gather_both(const TriBwdLaunch &T, int C, const int *inc_off, const int *inc, float *grad_attr,
                       float *grad_pos, int set_attr, int set_pos, hipStream_t st);
// floats of a tile record with the attribute and position sums
int tile_record_floats(int C, bool attr, bool pos);
// workspace of the tile records for nv floats per record and n_boxes pixel
// boxes (n_img * F for a uniform batch, the triangles of an uneven one), and
// its layout
size_t tile_records_bytes(int n_img, int H, int W, int nv, long long n_boxes);
void tile_records_layout(TriBwdLaunch &T, void *ws, int n_img, int H, int W, long long n_boxes);
// the same for an uneven batch of n_tiles 16 x 16 tiles in all
size_t tile_records_bytes_tiles(long long n_tiles, int nv, long long n_boxes);
void tile_records_layout_tiles(TriBwdLaunch &T, void *ws, long long n_tiles, long long n_boxes);

struct EdgeLaunch {
    const float *grad_out, *rgb, *rast, *frag_xy, *tris_xy;
    float *grad_frag_xy;
    int H, W, C, F;
};

int launch_edge_grad_bwd(const EdgeLaunch &L, hipStream_t st);
int launch_rasterize(const RasterLaunch &L, hipStream_t st);
int launch_rasterize_bwd(const RasterBwdLaunch &L, hipStream_t st);
int launch_interpolate(const InterpLaunch &L, hipStream_t st);
int launch_interpolate_bwd(const InterpLaunch &L, hipStream_t st);
int launch_topology(const TopoLaunch &L, hipStream_t st);
int launch_antialias(const AALaunch &L, hipStream_t st);
int launch_antialias_bwd(const AALaunch &L, hipStream_t st);
int launch_antialias_prepare(const AALaunch &L, hipStream_t st);
size_t incidence_ws_bytes(int V, int F);
size_t stencil_partition_ws_bytes(long long npx, int n_owner);
int launch_sample2d(const float *tex, int H, int W, int C, const float *uv, long long n, int wrap, int mode,
                    float *out, hipStream_t st);
int launch_sample2d_bwd(const float *tex, int H, int W, int C, const float *uv, long long n, int width, int wrap,
                        int mode, const float *gout, float *gtex, float *guv, hipStream_t st);
int launch_sample3d(const float *tex, int D, int H, int W, int C, const float *uvw, long long n, int wrap, int mode,
                    float *out, hipStream_t st);
int launch_sample3d_bwd(const float *tex, int D, int H, int W, int C, const float *uvw, long long n, int wrap,
                        int mode, const float *gout, float *gtex, float *guvw, hipStream_t st);
int launch_stencil_partition(const PartitionLaunch &L, void *ws, hipStream_t st);
int launch_count_covered(const float *rast, int n_img, long long npx, int *counts, hipStream_t st);
int launch_incidence(const int *tri, int F, int V, int *inc_off, int *inc, void *ws, hipStream_t st);
size_t l2_loss_ws_bytes();
int launch_l2_loss(const float *a, const float *b, long long n, float *loss, float *grad_a, void *ws,
                   hipStream_t st);
int launch_l2_loss_scale(float *grad, long long n, const float *grad_loss, hipStream_t st);
int launch_l2_loss_bwd(const float *a, const float *b, long long n, const float *grad_loss, float *ga, float *gb,
                       hipStream_t st);
int launch_clip_fwd(const float *xyz, int V, const float *VP, int n, float *pos, hipStream_t st);
int launch_clip_bwd(const float *grad_pos, int V, const float *VP, int n, float *grad_xyz, hipStream_t st);

// one front-to-back compositing step of n pixels (drp_compose.hip)
int launch_compose_fwd(const float *rgba, const float *rast, const float *out_prev, const float *trans_prev,
                       long long n, float *out, float *trans, hipStream_t st);
int launch_compose_bwd(const float *rgba, const float *rast, const float *trans_prev, long long n,
                       const float *grad_out, const float *grad_trans, float *grad_rgba, float *grad_trans_prev,
                       hipStream_t st);

}  // namespace drp
