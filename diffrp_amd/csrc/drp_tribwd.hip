// Deterministic backward of rasterize (positions): the POS instances of the
// tile passes, and the record workspace all tile passes share.
#include "drp_tribwd.h"

namespace drp {

int launch_tri_bwd_pos(const TriBwdLaunch &L, hipStream_t st) {
    if (L.grad_db) launch_tiles<0, 1, true>(L, st);
    else launch_tiles<0, 1, false>(L, st);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int tile_record_floats(int C, bool attr, bool pos) { return (attr ? (3 * C + 3) / 4 * 4 : 0) + (pos ? 12 : 0); }

// workspace: record counts [tiles], triangles [tiles, 256], box slots
// [n_boxes, kBoxSlots], sums [tiles, 256, nv]; the box slots hold int record
// indices, so they are left out (every tile searched) past 2^31 records
static bool box_slots_fit(long long n_tiles) { return n_tiles * kBTP < (1ll << 31); }

static size_t a256(size_t x) { return (x + 255) & ~(size_t)255; }

size_t tile_records_bytes_tiles(long long n_tiles, int nv, long long n_boxes) {
    const size_t slots = box_slots_fit(n_tiles) ? a256((size_t)n_boxes * kBoxSlots * 4) : 0;
    return a256((size_t)n_tiles * 4) + a256((size_t)n_tiles * kBTP * 4) + slots + a256((size_t)n_tiles * kBTP * nv * 4);
}

size_t tile_records_bytes(int n_img, int H, int W, int nv, long long n_boxes) {
    return tile_records_bytes_tiles((long long)n_img * ((W + kBT - 1) / kBT) * ((H + kBT - 1) / kBT), nv, n_boxes);
}

void tile_records_layout_tiles(TriBwdLaunch &T, void *ws, long long n_tiles, long long n_boxes) {
    T.n_tiles = (int)n_tiles;
    T.xcd_tiles = xcd_group(n_tiles, T.um.n ? 1 : T.n_img, kXcdPixels);
    T.n_tiles_pad = (int)xcd_pad(n_tiles, T.xcd_tiles);
    char *b = (char *)ws;
    T.rec_count = (int *)b;
    b += a256((size_t)n_tiles * 4);
    T.rec_t = (int *)b;
    b += a256((size_t)n_tiles * kBTP * 4);
    T.box_slot = nullptr;
    if (box_slots_fit(n_tiles)) {
        T.box_slot = (int *)b;
        b += a256((size_t)n_boxes * kBoxSlots * 4);
    }
    T.rec_v = (float *)b;
}

void tile_records_layout(TriBwdLaunch &T, void *ws, int n_img, int H, int W, long long n_boxes) {
    T.tiles_x = (W + kBT - 1) / kBT;
    T.tiles_per_img = T.tiles_x * ((H + kBT - 1) / kBT);
    tile_records_layout_tiles(T, ws, (long long)n_img * T.tiles_per_img, n_boxes);
}

}  // namespace drp
