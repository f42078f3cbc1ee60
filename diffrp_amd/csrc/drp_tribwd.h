// Device code of the deterministic backward passes of rasterize (positions)
// and interpolate (attributes), pixel-centric in two kernels (gfx950).
//
// k_tile_reduce, one workgroup per 16 x 16 pixel tile of one image: the tile's
// (triangle, pixel) keys are sorted in LDS, and each run of equal triangles --
// a segment -- is summed in pixel order and written as a record (triangle,
// sums).  The records of a tile come out sorted by triangle.  The pixels stage
// what the sums are made of, not the sums' terms: for the attributes the C
// gradients and (u, v, 1 - u - v), from which one thread per (segment, four
// channels) forms the three corners' terms, so a pixel costs C / 4 + 1 LDS
// rows and not 3 C / 4, and the products live in no register across the sort.
// Tiles without a covered pixel leave before the sort.  64 views of 82k
// triangles at 512^2, C = 8, both sums: 483 us with 36 staged terms per pixel,
// 412 us so, 381 with the sums as FMAs and no z/w chain where none can arrive.
// What remains is instruction issue: the sort, the double chain, the sums.
//
// k_tile_gather, one thread per (image [group], triangle) that won a pixel
// in the forward: the triangle's pixel box names the tiles it touches; the
// tile pass stored the record index of the box's first kBoxSlots tiles per
// box, further tiles' records are binary-searched, and the thread adds them in
// tile order.  All sums run in a fixed order, so results are reproducible bit
// for bit.  (Four lanes per triangle, to read a record in whole lines, repeat
// that search per lane: 150 -> 259 us at 64 views.)
//
//   POS  (12 floats): d rast (u, v, z/w [, db]) -> d clip (x, y, z, w) of the 3
//        corners (double-precision chain, drp_grad.h); partial [n, 3F] float4,
//        summed per vertex by the position gather.
//   ATTR (3 C floats): (u, v, 1-u-v) * g per corner, plus the terms of the
//        screen-space derivatives' gradients where those are wanted; the same
//        pass writes grad_rast = (<g, a0-a2>, <g, a1-a2>, 0, 0) (and grad_db);
//        k_tile_gather sums the views of a group, partial [groups, F, 3, C],
//        summed per vertex by the attribute gather.
//   BOTH (3 C + 12): the attribute sums, then the position sums of the
//        grad_rast just computed, from one sort and one record search.
// C is a compile-time count of 1 .. 16 channels; wider attributes go through
// in chunks of up to 16 (L.c0, L.ldc), the later chunks adding to grad_rast.
#pragma once
#include "drp_common.h"
#include "drp_grad.h"
#include "drp_kernels.h"
#include "drp_wave.h"

namespace drp {

constexpr int kBT = 16;            // backward tile edge
constexpr int kBTP = kBT * kBT;    // pixels (and records) per tile
// Sort keys: triangle << 8 | pixel, 32-bit while triangle ids fit 24 bits,
// else 64-bit; an uncovered pixel's triangle field is all ones.
template <typename K> struct SortKey;
template <> struct SortKey<unsigned> {
    static constexpr unsigned kEmptyT = (1u << 24) - 1;
};
template <> struct SortKey<unsigned long long> {
    static constexpr unsigned long long kEmptyT = (1ull << 40) - 1;
};


// number of entries of the sorted run a[0..64) below k (reads a[0..63] only)
template <typename K>
__device__ __forceinline__ int count_below64(const K *a, K k) {
    int base = 0;
#pragma unroll
    for (int half = 32; half >= 1; half >>= 1)
        if (a[base + half - 1] < k) base += half;
    return base + (a[base] < k ? 1 : 0);
}

// floats of a record: the attribute part (a whole number of quads, so that
// every record is 16-byte aligned), then 12 for the positions
template <int MODE, int C>
constexpr int rec_attr() { return MODE == 0 ? 0 : (3 * C + 3) / 4 * 4; }
template <int MODE, int C>
constexpr int tile_nv() { return rec_attr<MODE, C>() + (MODE == 1 ? 0 : 12); }

// Lanes that share one segment's sum, by the tile's segment count alone (the
// sums' order must not depend on what else a pass adds up): a tile of a few
// large triangles has long segments and few of them, and one thread walking
// 100 pixels is a chain of LDS round trips with the block idle around it.
// Lane s adds pixels s, s + lanes, ... in order, then the lanes' sums are added
// in a fixed tree.  One 512^2 view of 20k triangles, C = 4: 35.3 us with one
// thread per (segment, four channels), 16.4 us so; a crumpled uneven batch 158
// and 87 us.  Tiles of small triangles (64 views of 82k at 512^2: some 60
// segments) keep the merged form.
constexpr int kMergedSegs = 40;  // more segments than this: one thread takes all three corners of its channels
__device__ __forceinline__ int sum_lanes(int nseg) {
    return nseg <= 4 ? 16 : (nseg <= 8 ? 8 : (nseg <= 16 ? 4 : (nseg <= kMergedSegs ? 2 : 1)));
}
__device__ __forceinline__ float lanes_sum(float x, int lanes) {
    for (int o = 1; o < lanes; o <<= 1) x += __shfl_xor(x, o, 64);  // (a + b on one lane, b + a on the other)
    return x;
}

// Attribute sums over the segments' contiguous pixels; w: rows of (u, v,
// 1 - u - v), g: the gradients' quads, k: with DA the quads of the derivative
// terms (first corner's, then second's; the third corner takes minus both).
// Many segments: one thread per (segment, four channels) forms the terms of
// all three corners from one read of g and w.  Few: sum_lanes lanes per
// (segment, four channels, corner).
template <int C, bool DA>
__device__ __forceinline__ void attr_sums(const float4 *w, const float4 *g, const float4 *k, const int *seg_start,
                                          int nseg, float *rec, int nv) {
    constexpr int NQ = (C + 3) / 4;
    if (nseg > kMergedSegs) {
        for (int i = threadIdx.x; i < nseg * NQ; i += kBTP) {
            const int sg = i / NQ, q = i - sg * NQ;
            const int p0 = seg_start[sg], p1 = seg_start[sg + 1];
            const float4 *gr = g + q * kBTP;
            float s[3][4];
#pragma unroll
            for (int j = 0; j < 3; ++j)
#pragma unroll
                for (int c = 0; c < 4; ++c) s[j][c] = 0.f;
            for (int p = p0; p < p1; ++p) {
                const float4 wp = w[p], gp = gr[p];
                const float wv[3] = {wp.x, wp.y, wp.z}, gv[4] = {gp.x, gp.y, gp.z, gp.w};
#pragma unroll
                for (int j = 0; j < 3; ++j)
#pragma unroll
                    for (int c = 0; c < 4; ++c) s[j][c] = fma_(wv[j], gv[c], s[j][c]);
                if (DA) {
                    const float4 a = k[q * kBTP + p], b = k[(NQ + q) * kBTP + p];
                    const float av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        s[0][c] += av[c];
                        s[1][c] += bv[c];
                        s[2][c] -= av[c] + bv[c];
                    }
                }
            }
            float *o = rec + (long long)sg * nv + 4 * q;
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                if (C % 4 == 0) {
                    *reinterpret_cast<float4 *>(o + j * C) = make_float4(s[j][0], s[j][1], s[j][2], s[j][3]);
                } else {
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        if (4 * q + c < C) o[j * C + c] = s[j][c];
                }
            }
        }
        return;
    }
    const int lanes = sum_lanes(nseg), n = nseg * NQ * 3 * lanes;
    for (int i0 = 0; i0 < n; i0 += kBTP) {  // every lane stays for the tree
        const int i = i0 + threadIdx.x, l = i & (lanes - 1), item = i / lanes;
        const bool live = i < n;
        const int sg = live ? item / (3 * NQ) : 0, m = live ? item - sg * 3 * NQ : 0, j = m / NQ, q = m - j * NQ;
        const int p1 = live ? seg_start[sg + 1] : 0;
        const float *wj = reinterpret_cast<const float *>(w) + j;
        const float4 *gr = g + q * kBTP;
        float s[4] = {0.f, 0.f, 0.f, 0.f};
        for (int p = live ? seg_start[sg] + l : 0; p < p1; p += lanes) {
            const float wv = wj[4 * p];
            const float4 gp = gr[p];
            const float gv[4] = {gp.x, gp.y, gp.z, gp.w};
#pragma unroll
            for (int c = 0; c < 4; ++c) s[c] = fma_(wv, gv[c], s[c]);
            if (DA) {
                const float4 a = k[q * kBTP + p], b = k[(NQ + q) * kBTP + p];
                const float av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    if (j == 0) s[c] += av[c];
                    else if (j == 1) s[c] += bv[c];
                    else s[c] -= av[c] + bv[c];
                }
            }
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) s[c] = lanes_sum(s[c], lanes);
        if (!live || l != 0) continue;
        float *o = rec + (long long)sg * nv + j * C + 4 * q;
        if (C % 4 == 0) {
            *reinterpret_cast<float4 *>(o) = make_float4(s[0], s[1], s[2], s[3]);
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (4 * q + c < C) o[c] = s[c];
        }
    }
}

// position sums: sum_lanes lanes per (segment, corner)
__device__ __forceinline__ void pos_sums(const float4 *rows, const int *seg_start, int nseg, float *rec, int nv) {
    const int lanes = sum_lanes(nseg), n = nseg * 3 * lanes;
    for (int i0 = 0; i0 < n; i0 += kBTP) {  // every lane stays for the tree
        const int i = i0 + threadIdx.x, l = i & (lanes - 1), item = i / lanes;
        const bool live = i < n;
        const int sg = live ? item / 3 : 0, q = live ? item - sg * 3 : 0;
        const int p1 = live ? seg_start[sg + 1] : 0;
        const float4 *row = rows + q * kBTP;
        float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int p = live ? seg_start[sg] + l : 0; p < p1; p += lanes) {
            const float4 x = row[p];
            sum.x += x.x; sum.y += x.y; sum.z += x.z; sum.w += x.w;
        }
        sum.x = lanes_sum(sum.x, lanes);
        sum.y = lanes_sum(sum.y, lanes);
        sum.z = lanes_sum(sum.z, lanes);
        sum.w = lanes_sum(sum.w, lanes);
        if (live && l == 0) reinterpret_cast<float4 *>(rec + (long long)sg * nv)[q] = sum;
    }
}

// up to four channels from p: one 16-byte load when C is a multiple of 4 (the
// launcher only takes such C where row stride and base keep it aligned)
template <int C>
__device__ __forceinline__ float4 load_quad(const float *p, int q) {
    if (C % 4 == 0) return reinterpret_cast<const float4 *>(p)[q];
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    x.x = p[4 * q];
    if (4 * q + 1 < C) x.y = p[4 * q + 1];
    if (4 * q + 2 < C) x.z = p[4 * q + 2];
    if (4 * q + 3 < C) x.w = p[4 * q + 3];
    return x;
}

// clip positions of a triangle's corners (indices checked by the caller)
__device__ __forceinline__ void load_corners(const TriBwdLaunch &L, int img, int V, int i0, int i1, int i2,
                                             TriVerts &tv) {
    const float4 *P = reinterpret_cast<const float4 *>(L.pos) + (L.b.pos_batched ? (long long)img * V : 0);
    const float4 a = P[i0], b = P[i1], d = P[i2];
    tv.x[0] = a.x; tv.y[0] = a.y; tv.z[0] = a.z; tv.w[0] = a.w;
    tv.x[1] = b.x; tv.y[1] = b.y; tv.z[1] = b.z; tv.w[1] = b.w;
    tv.x[2] = d.x; tv.y[2] = d.y; tv.z[2] = d.z; tv.w[2] = d.w;
}

// waves per SIMD the register budget is cut for
template <int MODE, int C, bool DB>
constexpr int reduce_waves() { return DB ? 6 : 8; }

// DB: MODE 0: with a gradient of rast_db; MODE 1: with gradients of the
// interpolated screen-space derivatives
template <int MODE, int C, bool DB, typename K>
__global__ void __launch_bounds__(256, (reduce_waves<MODE, C, DB>())) k_tile_reduce(TriBwdLaunch L) {
    constexpr int NA = rec_attr<MODE, C>(), NV = tile_nv<MODE, C>();
    constexpr int NQ = (C + 3) / 4;
    constexpr bool DA = MODE == 1 && DB;
    constexpr K kEmptyT = SortKey<K>::kEmptyT;
    constexpr int kAttrRows = MODE == 0 ? 0 : 1 + NQ * (DA ? 3 : 1), kPosRows = MODE == 1 ? 0 : 3;
    __shared__ float4 rows[(kAttrRows > kPosRows ? kAttrRows : kPosRows) * kBTP];
    __shared__ K key[kBTP];
    __shared__ union {
        K run[kBTP];             // the waves' sorted runs (merge)
        int seg_start[kBTP + 1]; // segment starts (after the merge)
    } U;
    __shared__ int wsum[4];
    __shared__ unsigned char rank[kBTP];  // sorted place of each pixel's key
    __shared__ double spx[kBT], spy[kBT]; // NDC centres of the tile's columns and rows (position chain)
    const int tid = threadIdx.x;
    const int tile = xcd_deal(blockIdx.x, L.xcd_tiles);
    if (tile >= L.n_tiles) return;  // uniform per block
    // the tile's image: arithmetic for a uniform batch, the item map for an uneven one
    int img, lt, H = L.H, W = L.W, tiles_x = L.tiles_x;
    long long pix0;
    if (L.um.n) {
        img = um_find(L.um.bt16, L.um.n, tile);
        lt = tile - L.um.bt16[img];
        H = L.um.hw[2 * img];
        W = L.um.hw[2 * img + 1];
        tiles_x = (W + kBT - 1) / kBT;
        pix0 = L.um.pix[img];
    } else {
        img = tile / L.tiles_per_img;
        lt = tile - img * L.tiles_per_img;
        pix0 = (long long)img * L.H * L.W;
    }
    const int r = (lt / tiles_x) * kBT + (tid >> 4), c = (lt % tiles_x) * kBT + (tid & 15);
    if (MODE != 1) {  // one double division per column and row of the tile, not two per pixel
        if (tid < kBT) spx[tid] = pix_ndc_d((lt % tiles_x) * kBT + tid, W);
        else if (tid < 2 * kBT) spy[tid - kBT] = pix_ndc_d((lt / tiles_x) * kBT + tid - kBT, H);
    }
    const bool in = r < H && c < W;
    const long long pix = pix0 + (long long)r * W + c;
    const int V = MODE == 1 ? L.V : L.b.V;
    int t = -1, i0 = 0, i1 = 0, i2 = 0;
    float u = 0.f, v = 0.f;
    if (in) {
        const float4 rv = reinterpret_cast<const float4 *>(L.rast)[pix];
        u = rv.x;
        v = rv.y;
        if (rv.w > 0.f) {
            int id = float_to_triidx(rv.w);
            if (L.um.n && L.local_ids) id += L.um.tri[img];  // item-local id -> batch triangle + 1
            if (id >= 1 && id <= L.F) t = id - 1;
        }
        if (t >= 0) {
            const int *t3 = L.tri + 3 * (long long)t;
            i0 = t3[0]; i1 = t3[1]; i2 = t3[2];
            if ((unsigned)i0 >= (unsigned)V || (unsigned)i1 >= (unsigned)V || (unsigned)i2 >= (unsigned)V) t = -1;
        }
        // pixels without a fragment bring nothing; their grad_rast is zero
        if (MODE != 0 && t < 0 && (MODE == 1 || L.grad_rast_out) && !L.accum) {
            reinterpret_cast<float4 *>(L.grad_rast_out)[pix] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (DA && L.grad_db_out) reinterpret_cast<float4 *>(L.grad_db_out)[pix] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }
    if (!__syncthreads_or(t >= 0)) {
        if (tid == 0) L.rec_count[tile] = 0;
        return;
    }
    // The gradients of narrow attributes and the corners' positions are asked for
    // before the sort, which hides their latency, as far as the registers go: at
    // C = 8, both sums, 381 us with the gradients at 64 x 512^2, 386 without or with both.
    constexpr bool kEarly = MODE != 0 && C <= 8;
    constexpr bool kEarlyPos = MODE == 0 || (MODE == 2 && C <= 4);
    float4 early_g[kEarly ? NQ : 1];
    TriVerts tv;
    if (t >= 0) {
        if (kEarly) {
#pragma unroll
            for (int q = 0; q < NQ; ++q) early_g[q] = load_quad<C>(L.grad_out + pix * L.ldc + L.c0, q);
        }
        if (kEarlyPos) load_corners(L, img, V, i0, i1, i2, tv);
    }
    // sort the 256 keys (triangle << 8 | pixel; uncovered pixels last, keys unique):
    // each wave sorts its 64 across lanes, then every key's place is its lane
    // plus the keys below it in the other three runs
    {
        K k = wave_sort(((t >= 0 ? (K)t : kEmptyT) << 8) | (K)tid);
        const int wave = tid >> 6;
        U.run[tid] = k;
        __syncthreads();
        int place = tid & 63;
#pragma unroll
        for (int w = 0; w < 4; ++w)
            if (w != wave) place += count_below64<K>(U.run + 64 * w, k);
        key[place] = k;
        rank[(int)(k & 255)] = (unsigned char)place;
        __syncthreads();
    }
    // this pixel's place: every segment's pixels are staged contiguously
    const int my = rank[tid];
    // segments: runs of one triangle in sorted order
    const K sk = key[tid];
    const bool valid = (sk >> 8) != kEmptyT;
    const bool head = valid && (tid == 0 || (key[tid - 1] >> 8) != (sk >> 8));
    int nseg;
    const int seg = block_scan<kBTP>(head ? 1 : 0, wsum, nseg);
    const int nvalid = __syncthreads_count(valid);
    if (head) U.seg_start[seg] = tid;
    if (tid == 0) U.seg_start[nseg] = nvalid;
    const long long rbase = (long long)tile * kBTP;
    if (head) {
        const int st = (int)(sk >> 8);
        L.rec_t[rbase + seg] = st;
        if (L.box_slot) {  // the record's place among the first tiles of st's box
            const long long bi = (L.um.n ? 0ll : (long long)img * L.F) + st;
            const ItemBox b = L.boxes[bi];
            const int tx = lt % tiles_x, ty = lt / tiles_x;
            const int tx0 = (b.cc & 0xffff) / kBT, tx1 = ((unsigned)b.cc >> 16) / kBT, ty0 = (b.rr & 0xffff) / kBT;
            const int k = (ty - ty0) * (tx1 - tx0 + 1) + (tx - tx0);
            if (tx >= tx0 && tx <= tx1 && ty >= ty0 && k < kBoxSlots) L.box_slot[kBoxSlots * bi + k] = (int)(rbase + seg);
        }
    }
    if (tid == 0) L.rec_count[tile] = nseg;
    float *rec = L.rec_v + rbase * NV;
    float4 g = make_float4(0.f, 0.f, 0.f, 0.f), gd = g;
    if (MODE != 0) {
        if (t >= 0) {
            const float *A = L.attr + (L.attr_batched ? (long long)img * L.V * L.ldc : 0) + L.c0;
            const float *a0 = A + (long long)i0 * L.ldc, *a1 = A + (long long)i1 * L.ldc, *a2 = A + (long long)i2 * L.ldc;
            const float *go = L.grad_out + pix * L.ldc + L.c0;
            float su = 0.f, sv = 0.f;
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const float4 gq = kEarly ? early_g[kEarly ? q : 0] : load_quad<C>(go, q), x0 = load_quad<C>(a0, q), x1 = load_quad<C>(a1, q),
                             x2 = load_quad<C>(a2, q);
                rows[(1 + q) * kBTP + my] = gq;
                const float gv[4] = {gq.x, gq.y, gq.z, gq.w}, p0[4] = {x0.x, x0.y, x0.z, x0.w},
                            p1[4] = {x1.x, x1.y, x1.z, x1.w}, p2[4] = {x2.x, x2.y, x2.z, x2.w};
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (4 * q + k < C) {
                        su = fma_(gv[k], p0[k] - p2[k], su);
                        sv = fma_(gv[k], p1[k] - p2[k], sv);
                    }
            }
            rows[my] = make_float4(u, v, (1.f - u) - v, 0.f);
            g = make_float4(su, sv, 0.f, 0.f);
            if (DA) {  // the derivatives' terms, accumulated at this pixel's own place
                const float4 db = reinterpret_cast<const float4 *>(L.rast_db)[pix];
                const float *gda = L.grad_da + pix * 2 * L.n_diff;
#pragma unroll
                for (int q = 0; q < 2 * NQ; ++q) rows[(1 + NQ + q) * kBTP + my] = make_float4(0.f, 0.f, 0.f, 0.f);
                for (int j = 0; j < L.n_diff; ++j) {
                    const int ch = L.diff_idx[j] - L.c0;
                    if ((unsigned)ch >= (unsigned)C) continue;
                    const float gx = gda[2 * j], gy = gda[2 * j + 1];
                    const float d0 = a0[ch] - a2[ch], d1 = a1[ch] - a2[ch];
                    reinterpret_cast<float *>(&rows[(1 + NQ + (ch >> 2)) * kBTP + my])[ch & 3] += gx * db.x + gy * db.y;
                    reinterpret_cast<float *>(&rows[(1 + 2 * NQ + (ch >> 2)) * kBTP + my])[ch & 3] += gx * db.z + gy * db.w;
                    gd.x += gx * d0;
                    gd.y += gy * d0;
                    gd.z += gx * d1;
                    gd.w += gy * d1;
                }
            }
            if (MODE == 1 || L.grad_rast_out) {
                float4 *o = reinterpret_cast<float4 *>(L.grad_rast_out) + pix;
                float4 x = g;
                if (L.accum) {
                    const float4 y = *o;
                    x.x += y.x;
                    x.y += y.y;
                }
                *o = x;
                if (DA && L.grad_db_out) {
                    float4 *od = reinterpret_cast<float4 *>(L.grad_db_out) + pix;
                    float4 z = gd;
                    if (L.accum) {
                        const float4 y = *od;
                        z.x += y.x; z.y += y.y; z.z += y.z; z.w += y.w;
                    }
                    *od = z;
                }
            }
        }
        __syncthreads();
        attr_sums<C, DA>(rows, rows + kBTP, rows + (1 + NQ) * kBTP, U.seg_start, nseg, rec, NV);
    }
    if (MODE != 1) {
        if (t >= 0) {
            if (!kEarlyPos) load_corners(L, img, V, i0, i1, i2, tv);
            if (MODE == 0) {
                g = reinterpret_cast<const float4 *>(L.grad_rast)[pix];
                if (DB) gd = db_grad_scaled(reinterpret_cast<const float4 *>(L.grad_db)[pix], H, W);
            }
        }
        if (MODE == 2) __syncthreads();  // the attribute sums have read the rows
        if (t >= 0) {
            float4 o[3];
            raster_pixel_grad_at<MODE == 0 && DB, MODE == 0>(tv, spx[tid & 15], spy[tid >> 4], g, gd, o);
#pragma unroll
            for (int q = 0; q < 3; ++q) rows[q * kBTP + my] = o[q];
        }
        __syncthreads();
        pos_sums(rows, U.seg_start, nseg, rec + NA, NV);
    }
}

// Records of triangle t in one image, in tile order over its pixel box (box
// index bi).  The first kBoxSlots tiles of the box are looked up through
// box_slot, which the tile pass filled with the record index of every
// (box, tile) it wrote; a slot is trusted only when it points into that tile's
// records and names t there (the workspace is not cleared between calls, so a
// slot of a tile where t won no pixel holds whatever an earlier call left).
// Further tiles, and every tile without box_slot, are binary-searched
// (records sorted by triangle), kSearch at a time in lockstep so that their
// dependent loads overlap.
constexpr int kSearch = 4;

// one image's box of the triangle and its box slots, loaded together
struct BoxLoad {
    ItemBox b;
    int4 s;
};
__device__ __forceinline__ BoxLoad load_box(const TriBwdLaunch &L, long long bi) {
    BoxLoad x;
    x.b = L.boxes[bi];
    x.s = L.box_slot ? *reinterpret_cast<const int4 *>(L.box_slot + kBoxSlots * bi) : make_int4(-1, -1, -1, -1);
    return x;
}

__device__ __forceinline__ bool box_hit(const ItemBox &b) {  // won a pixel, inside its box
    return b.hit && (b.cc & 0xffff) <= (int)((unsigned)b.cc >> 16) && (b.rr & 0xffff) <= (int)((unsigned)b.rr >> 16);
}

// (box_hit holds)
template <int NV, typename Add>
__device__ __forceinline__ void image_records(const TriBwdLaunch &L, int t, const BoxLoad &x, int tile_base,
                                              int tiles_x, Add &&add) {
    const ItemBox &b = x.b;
    const int c0 = b.cc & 0xffff, c1 = (unsigned)b.cc >> 16, r0 = b.rr & 0xffff, r1 = (unsigned)b.rr >> 16;
    const int tx0 = c0 / kBT, tx1 = c1 / kBT, ty0 = r0 / kBT, bw = tx1 - tx0 + 1;
    const int nb = bw * (r1 / kBT - ty0 + 1);
    int k0 = 0;
    if (L.box_slot) {
        const int sv[kBoxSlots] = {x.s.x, x.s.y, x.s.z, x.s.w};
        int idx[kBoxSlots], cnt[kBoxSlots], rt[kBoxSlots], seg[kBoxSlots];
        int tx = tx0, ty = ty0;
#pragma unroll
        for (int j = 0; j < kBoxSlots; ++j) {
            idx[j] = -1;
            cnt[j] = 0;
            rt[j] = -1;
            seg[j] = -1;
            if (j < nb) {
                const int tile = tile_base + ty * tiles_x + tx;
                seg[j] = sv[j] - tile * kBTP;
                if (seg[j] >= 0 && seg[j] < kBTP) {  // inside the tile's records: both loads in bounds
                    cnt[j] = L.rec_count[tile];
                    rt[j] = L.rec_t[sv[j]];
                }
                if (++tx > tx1) {
                    tx = tx0;
                    ++ty;
                }
            }
        }
#pragma unroll
        for (int j = 0; j < kBoxSlots; ++j)
            if (seg[j] >= 0 && seg[j] < cnt[j] && rt[j] == t) idx[j] = sv[j];
#pragma unroll
        for (int j = 0; j < kBoxSlots; ++j)
            if (idx[j] >= 0) add(L.rec_v + (long long)idx[j] * NV);
        k0 = min(nb, kBoxSlots);
    }
    for (int k = k0; k < nb; k += kSearch) {
        long long rb[kSearch];
        int lo[kSearch], hi[kSearch], hit[kSearch];
#pragma unroll
        for (int j = 0; j < kSearch; ++j) {
            rb[j] = 0;
            lo[j] = 0;
            hi[j] = -1;
            hit[j] = -1;
            if (k + j < nb) {
                const int q = (k + j) / bw;
                const int tile = tile_base + (ty0 + q) * tiles_x + tx0 + (k + j - q * bw);
                rb[j] = (long long)tile * kBTP;
                hi[j] = L.rec_count[tile] - 1;
            }
        }
        for (bool more = true; more;) {
            more = false;
#pragma unroll
            for (int j = 0; j < kSearch; ++j) {
                if (hit[j] >= 0 || lo[j] > hi[j]) continue;
                const int mid = (lo[j] + hi[j]) >> 1;
                const int tm = L.rec_t[rb[j] + mid];
                if (tm < t) lo[j] = mid + 1;
                else if (tm > t) hi[j] = mid - 1;
                else hit[j] = mid;
                more = more || (hit[j] < 0 && lo[j] <= hi[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < kSearch; ++j)
            if (hit[j] >= 0) add(L.rec_v + (rb[j] + hit[j]) * NV);
    }
}

// Records of triangle t over images [v0, v1) in (image, tile) order; done(img,
// won a pixel) after each image.  Uniform batch: box of (image, t) at image * F + t, tile
// image * tiles_per_img + ty * tiles_x + tx.  Uneven batch: t's item only, box
// at t, tiles from the item's first.  The next image's box and slots are
// loaded before this image's records are read.
template <int NV, typename Add, typename Done>
__device__ __forceinline__ void triangle_records(const TriBwdLaunch &L, int t, int v0, int v1, Add &&add,
                                                 Done &&done) {
    long long box_stride = L.F;
    int tile_stride = L.tiles_per_img, tiles_x = L.tiles_x, tile_base = 0;
    if (L.um.n) {
        const int item = um_find(L.um.tri, L.um.n, t);
        v0 = 0;
        v1 = 1;
        box_stride = 0;
        tile_stride = 0;
        tile_base = L.um.bt16[item];
        tiles_x = (L.um.hw[2 * item + 1] + kBT - 1) / kBT;
    }
    if (v0 >= v1) return;
    BoxLoad cur = load_box(L, v0 * box_stride + t);
    for (int img = v0; img < v1; ++img) {
        BoxLoad nxt;
        if (img + 1 < v1) nxt = load_box(L, (img + 1) * box_stride + t);
        const bool hit = box_hit(cur.b);
        if (hit) image_records<NV>(L, t, cur, tile_base + img * tile_stride, tiles_x, add);
        done(img, hit);
        if (img + 1 < v1) cur = nxt;
    }
}

template <int NV>
__device__ __forceinline__ void add_record(float *acc, const float *q) {
    static_assert(NV % 4 == 0, "records are whole quads from an aligned base");
#pragma unroll
    for (int j = 0; j < NV; j += 4) {
        const float4 x = *reinterpret_cast<const float4 *>(q + j);
        acc[j] += x.x; acc[j + 1] += x.y; acc[j + 2] += x.z; acc[j + 3] += x.w;
    }
}

template <int NV>
__device__ __forceinline__ bool gather_records(const TriBwdLaunch &L, int t, int v0, int v1, float *acc) {
    bool any = false;
    triangle_records<NV>(
        L, t, v0, v1, [&](const float *q) { add_record<NV>(acc, q); }, [&](int, bool hit) { any = any || hit; });
    return any;
}

// corners of (image, triangle) i: 48 consecutive bytes
__device__ __forceinline__ void store_pos(float *partial, long long i, const float *pos) {
    float4 *P = reinterpret_cast<float4 *>(partial) + 3 * i;
    P[0] = make_float4(pos[0], pos[1], pos[2], pos[3]);
    P[1] = make_float4(pos[4], pos[5], pos[6], pos[7]);
    P[2] = make_float4(pos[8], pos[9], pos[10], pos[11]);
}

// MODE 2: the attribute sums over the group's images (as MODE 1), and per
// image the position sums, written to that image's partial (as MODE 0)
template <int NA>
__device__ __forceinline__ bool gather_records_fused(const TriBwdLaunch &L, int t, int v0, int v1, float *acc) {
    float pos[12];
#pragma unroll
    for (int j = 0; j < 12; ++j) pos[j] = 0.f;
    bool any = false;
    triangle_records<NA + 12>(
        L, t, v0, v1,
        [&](const float *q) {
            add_record<NA>(acc, q);
            add_record<12>(pos, q + NA);
        },
        [&](int img, bool hit) {
            const long long i = (long long)img * L.F + t;
            L.live_pos[i] = hit;
            if (!hit) return;
            any = true;
            store_pos(L.partial_pos, i, pos);
#pragma unroll
            for (int j = 0; j < 12; ++j) pos[j] = 0.f;
        });
    return any;
}

// Waves per SIMD the register budget is cut for: 6 keeps the latency-bound
// searches overlapped; records wider than 16 floats need the accumulators of
// 4 waves (128 VGPRs), beyond 40 floats of 3, to stay out of scratch.
template <int MODE, int C>
constexpr int gather_waves() { return tile_nv<MODE, C>() <= 16 ? 6 : (tile_nv<MODE, C>() <= 40 ? 4 : 3); }

template <int MODE, int C>
__global__ void __launch_bounds__(256, (gather_waves<MODE, C>())) k_tile_gather(TriBwdLaunch L, int xcd) {
    constexpr int NV = tile_nv<MODE, C>();
    // neighbouring triangles, which share their tiles' record lines, on one XCD
    const int lin = xcd_deal(blockIdx.x + gridDim.x * blockIdx.y, xcd);
    const int grp = lin / gridDim.x;
    const int t = (lin - grp * (int)gridDim.x) * blockDim.x + threadIdx.x;
    if (t >= L.F) return;
    float acc[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) acc[j] = 0.f;
    const int VB = L.views_per_block;
    const int v0 = grp * VB, v1 = min(v0 + VB, L.n_img);
    // Only triangles that won a pixel have sums: the others' partials are neither
    // written here nor read by the vertex gathers, which look at one byte each
    // (half of a mesh faces away, and a dense one hides most of the rest): 64
    // views of 82k triangles 255 -> 150 us, one view of 5.2M 920 -> 240 us with
    // the triangles dealt to the XCDs.
    const bool hit = MODE == 2 ? gather_records_fused<rec_attr<MODE, C>()>(L, t, v0, v1, acc)
                               : gather_records<NV>(L, t, v0, v1, acc);
    const long long gt = (long long)grp * L.F + t;
    L.live[gt] = hit;
    if (!hit) return;
    if (MODE == 0) {
        store_pos(L.partial, gt, acc);
    } else {
        constexpr int NA = 3 * C;  // the record's attribute part, without its padding
        float *P = L.partial + gt * NA;
        if (NA % 4 == 0) {
#pragma unroll
            for (int j = 0; j < NA; j += 4)
                *reinterpret_cast<float4 *>(P + j) = make_float4(acc[j], acc[j + 1], acc[j + 2], acc[j + 3]);
        } else {
#pragma unroll
            for (int j = 0; j < NA; ++j) P[j] = acc[j];
        }
    }
}

template <int MODE, int C, bool DB>
inline void launch_tiles(const TriBwdLaunch &L, hipStream_t st) {
    const dim3 grid((unsigned)L.n_tiles_pad);
    if (L.F < (int)SortKey<unsigned>::kEmptyT)
        hipLaunchKernelGGL((k_tile_reduce<MODE, C, DB, unsigned>), grid, dim3(kBTP), 0, st, L);
    else
        hipLaunchKernelGGL((k_tile_reduce<MODE, C, DB, unsigned long long>), grid, dim3(kBTP), 0, st, L);
    const int groups = (L.n_img + L.views_per_block - 1) / L.views_per_block;
    // a row of blocks per group of images, padded so that the turns divide all of them
    const bool eighths = !L.um.n && L.n_img >= 8;
    const long long blocks = (L.F + 255ll) / 256;
    const int few = eighths ? 1 : xcd_group(blocks, 1, kXcdVerts);
    const long long width = xcd_pad(blocks, few);
    hipLaunchKernelGGL((k_tile_gather<MODE, C>), dim3((unsigned)width, groups), dim3(256), 0, st, L,
                       eighths ? (int)(width * groups / 8) : few);
}

}  // namespace drp
