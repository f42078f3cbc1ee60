// Analytic silhouette antialiasing (after Laine et al. 2020, "Modular Primitives
// for High-Performance Differentiable Rendering", sec. 3.3) and the edge ->
// opposite-triangle table it needs.
//
// Per horizontal / vertical pair of pixel centres (a, b) with different
// triangle ids: candidates are the triangles at a and b, nearer z/w first.
// For candidate T seen at `from`, the segment from -> to leaves T through the
// edge with the smallest crossing t_e = f(from) / (f(from) - f(to)) among the
// edges whose half-plane excludes `to`.  If that edge is a silhouette (no
// neighbour, or a neighbour of opposite screen orientation) the pair blends:
// t = clamp(t_e, 0, 1); t < 1/2 moves `from` towards `to` by (1/2 - t),
// otherwise `to` towards `from` by (t - 1/2).  Else the next candidate is tried.
//
// Kernels: k_aa_orient (vertices in pixel coordinates, per-triangle screen
// orientation), k_aa_silhouette (triangles with a possible silhouette edge),
// k_aa_fwd (a block evaluates the pairs that touch its pixels, blends the
// colours in a fixed order and leaves a list of its blending pairs) and
// k_aa_bwd (colour and position gradients of a block from that list).
#include <type_traits>

#include "drp_common.h"
#include "drp_kernels.h"
#include "drp_wave.h"

namespace drp {

// ----------------------------------------------------------------------------
// topology: open-addressing hash of undirected edges -> (up to) two faces
// ----------------------------------------------------------------------------
constexpr unsigned long long kEmpty = ~0ull;

__device__ __forceinline__ unsigned long long edge_key(int a, int b) {
    unsigned lo = (unsigned)min(a, b), hi = (unsigned)max(a, b);
    return ((unsigned long long)lo << 32) | hi;
}
__device__ __forceinline__ unsigned hash64(unsigned long long k) {
    k ^= k >> 33;
    k *= 0xff51afd7ed558ccdull;
    k ^= k >> 33;
    k *= 0xc4ceb9fe1a85ec53ull;
    k ^= k >> 33;
    return (unsigned)k;
}

__global__ void k_topo_clear(unsigned long long *keys, int *cnt, long long n) {
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) { keys[i] = kEmpty; cnt[i] = 0; }
}

__global__ void k_topo_insert(const int *__restrict__ tri, int F, unsigned long long *keys, int *cnt, int2 *slots,
                              unsigned mask) {
    long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= 3ll * F) return;
    int t = (int)(g / 3), e = (int)(g % 3);
    int a = tri[3 * (long long)t + e], b = tri[3 * (long long)t + (e == 2 ? 0 : e + 1)];
    unsigned long long k = edge_key(a, b);
    unsigned h = hash64(k) & mask;
    for (unsigned probe = 0; probe <= mask; ++probe) {
        unsigned long long old = atomicCAS(&keys[h], kEmpty, k);
        if (old == kEmpty || old == k) {
            int s = atomicAdd(&cnt[h], 1);
            if (s == 0) slots[h].x = (int)g;
            else if (s == 1) slots[h].y = (int)g;
            return;
        }
        h = (h + 1) & mask;
    }
}

__global__ void k_topo_lookup(const int *__restrict__ tri, int F, const unsigned long long *__restrict__ keys,
                              const int *__restrict__ cnt, const int2 *__restrict__ slots, unsigned mask,
                              int *__restrict__ opp) {
    long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= 3ll * F) return;
    int t = (int)(g / 3), e = (int)(g % 3);
    int a = tri[3 * (long long)t + e], b = tri[3 * (long long)t + (e == 2 ? 0 : e + 1)];
    unsigned long long k = edge_key(a, b);
    unsigned h = hash64(k) & mask;
    int res = -1;
    for (unsigned probe = 0; probe <= mask; ++probe) {
        unsigned long long kk = keys[h];
        if (kk == k) {
            if (cnt[h] == 2) {
                int2 s = slots[h];
                res = (s.x == (int)g ? s.y : s.x) / 3;
            }
            break;
        }
        if (kk == kEmpty) break;
        h = (h + 1) & mask;
    }
    opp[g] = res;
}

int launch_topology(const TopoLaunch &L, hipStream_t st) {
    if (L.F == 0) return 0;
    long long n = (long long)L.mask + 1;
    hipLaunchKernelGGL(k_topo_clear, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, L.keys, L.cnt, n);
    long long ne = 3ll * L.F;
    dim3 g((unsigned)((ne + 255) / 256));
    hipLaunchKernelGGL(k_topo_insert, g, dim3(256), 0, st, L.tri, L.F, L.keys, L.cnt, L.slots, L.mask);
    hipLaunchKernelGGL(k_topo_lookup, g, dim3(256), 0, st, L.tri, L.F, L.keys, L.cnt, L.slots, L.mask, L.opp);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

// ----------------------------------------------------------------------------
// orientation / silhouette precompute
// ----------------------------------------------------------------------------
__device__ __forceinline__ double dfma(double a, double b, double c) { return __builtin_fma(a, b, c); }

__device__ __forceinline__ int orient3(float4 a, float4 b, float4 c) {
    // sign of det[[x0,x1,x2],[y0,y1,y2],[w0,w1,w2]], in double (edge-on triangles decide silhouettes)
    double m0 = dfma(b.y, c.w, -((double)c.y * b.w));
    double m1 = dfma(a.y, c.w, -((double)c.y * a.w));
    double m2 = dfma(a.y, b.w, -((double)b.y * a.w));
    double d = dfma(a.x, m0, dfma(-(double)b.x, m1, (double)c.x * m2));
    return d > 0.0 ? 1 : (d < 0.0 ? -1 : 0);
}

// Two independent maps in one launch: blocks below n_orient_blk give per-triangle
// orientations, the rest the pixel coordinates of every vertex in double (NaN
// when w <= 0), which the pair search reads for every candidate triangle.
__global__ void k_aa_orient(const float *__restrict__ pos, int V, const int *__restrict__ tri, int F, int n_proj, int H,
                            int W, UnevenMap um, int n_orient_blk, signed char *__restrict__ orient,
                            double2 *__restrict__ proj) {
    if ((int)blockIdx.x >= n_orient_blk) {
        long long g = (long long)(blockIdx.x - n_orient_blk) * blockDim.x + threadIdx.x;
        if (g >= (long long)n_proj * V) return;
        if (um.n) {  // uneven batch: the vertex's item sets the image size
            const int item = um_find(um.vert, um.n, (int)g);
            H = um.hw[2 * item];
            W = um.hw[2 * item + 1];
        }
        float4 p = reinterpret_cast<const float4 *>(pos)[g];
        double2 o;
        if (p.w > 0.f) {
            o.x = ((double)p.x / (double)p.w + 1.0) * ((double)W * 0.5);
            o.y = ((double)p.y / (double)p.w + 1.0) * ((double)H * 0.5);
        } else {
            o.x = __longlong_as_double(0x7ff8000000000000ll);
            o.y = o.x;
        }
        proj[g] = o;
        return;
    }
    // XCD k takes the k-th eighth of the (image, triangle) items: an image's vertices stay in one L2
    long long g = (long long)xcd_remap(blockIdx.x, n_orient_blk) * blockDim.x + threadIdx.x;
    if (g >= (long long)n_proj * F) return;
    int img = (int)(g / F), t = (int)(g % F);
    const int *t3 = tri + 3 * (long long)t;
    int i0 = t3[0], i1 = t3[1], i2 = t3[2];
    signed char o = 0;
    if ((unsigned)i0 < (unsigned)V && (unsigned)i1 < (unsigned)V && (unsigned)i2 < (unsigned)V) {
        const float4 *P = reinterpret_cast<const float4 *>(pos) + (long long)img * V;
        o = (signed char)orient3(P[i0], P[i1], P[i2]);
    }
    orient[g] = o;
}

// silh[img][t]: bit e (e = 0, 1, 2) when edge e -> e+1 of t can be a silhouette
// in that image (no neighbour, or a neighbour of another screen orientation),
// bit 3 when t's screen orientation is negative; 0 for an edge-on triangle.
// A pair whose candidate triangle has no such edge cannot blend through it, and
// the pair search reads the edge test and the orientation from this one byte.
__global__ void k_aa_silhouette(const int *__restrict__ opp, const signed char *__restrict__ orient, int F,
                                int n_proj, unsigned char *__restrict__ silh) {
    long long g = (long long)xcd_remap(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;  // as k_aa_orient
    if (g >= (long long)n_proj * F) return;
    int img = (int)(g / F), t = (int)(g % F);
    const signed char *O = orient + (long long)img * F;
    int o = O[t];
    unsigned char f = 0;
    if (o != 0) {
#pragma unroll
        for (int e = 0; e < 3; ++e) {
            int n = opp[3 * (long long)t + e];
            if (!(n >= 0 && n < F && O[n] == o)) f |= (unsigned char)(1 << e);
        }
        if (f && o < 0) f |= 8;
    }
    silh[g] = f;
}

// ----------------------------------------------------------------------------
// pair evaluation (same arithmetic as the scalar reference of these rules)
// ----------------------------------------------------------------------------
struct PairRes {
    int recv;   // -1 none, 0: a receives, 1: b receives
    float wgt;
    int tri, edge, from_a, clamped;
};

struct AAImg {
    const float4 *rast;         // image rast
    const double2 *proj;        // image's vertices in pixel coordinates (NaN: w <= 0)
    const signed char *orient;  // image's triangle orientations
    const unsigned char *silh;  // image's silhouette-capable triangles
    int V, F, H, W;
};

__device__ __forceinline__ int rast_id_w(float w, int F) {  // triangle + 1 from rast's w, 0 for none
    int id = w > 0.f ? float_to_triidx(w) : 0;
    return id > F ? 0 : id;
}
__device__ __forceinline__ int rast_id(float4 p, int F) { return rast_id_w(p.w, F); }

// Pair (a, b) from the two pixels' rast values and their triangles' silhouette
// bytes (the caller loads them, so the loads of neighbouring pairs overlap).
// Both candidates' corner indices, then both candidates' vertex projections,
// are loaded before either is tested, so the pair waits for two rounds of
// loads, not up to four.
__device__ __forceinline__ PairRes eval_pair(const AAImg &I, const int *__restrict__ tri, float4 pa, float4 pb,
                                             int sa, int sb, int ra, int ca, int rb, int cb) {
    PairRes res;
    res.recv = -1;
    const int ida = rast_id(pa, I.F), idb = rast_id(pb, I.F);
    if (ida == idb) return res;
    int a_first = 1;
    if (ida == 0) a_first = 0;
    else if (idb != 0 && pb.z < pa.z) a_first = 0;
    int tc[2], mc[2], vi[2][3];
    bool ok[2];
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {  // candidate 0 first, then 1
        const int use_a = pass == 0 ? a_first : !a_first;
        const int id = use_a ? ida : idb;
        mc[pass] = use_a ? sa : sb;
        ok[pass] = id != 0 && (mc[pass] & 7);  // a candidate needs a silhouette-capable edge
        tc[pass] = ok[pass] ? id - 1 : 0;
        const int *t3 = tri + 3 * (long long)tc[pass];
        vi[pass][0] = t3[0];
        vi[pass][1] = t3[1];
        vi[pass][2] = t3[2];
    }
    // pair geometry in double: a float clip coordinate fixes a vertex to
    // ~W * 2^-25 pixel, and the crossing needs differences of nearby pixel
    // positions
    double2 q[2][3];
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
        ok[pass] = ok[pass] && (unsigned)vi[pass][0] < (unsigned)I.V && (unsigned)vi[pass][1] < (unsigned)I.V &&
                   (unsigned)vi[pass][2] < (unsigned)I.V;
#pragma unroll
        for (int k = 0; k < 3; ++k) q[pass][k] = ok[pass] ? I.proj[vi[pass][k]] : make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
        if (!ok[pass]) continue;
        const int use_a = pass == 0 ? a_first : !a_first;
        const int t = tc[pass], m = mc[pass];
        double X[3], Y[3];
        bool front = true;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            front = front && !isnan(q[pass][k].x);
            X[k] = q[pass][k].x;
            Y[k] = q[pass][k].y;
        }
        if (!front) continue;
        const int o = (m & 8) ? -1 : 1;
        double fx = (double)(use_a ? ca : cb) + 0.5, fy = (double)(use_a ? ra : rb) + 0.5;
        double tx = (double)(use_a ? cb : ca) + 0.5, ty = (double)(use_a ? rb : ra) + 0.5;
        int best = -1;
        double bt = 0.0;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            int j = k == 2 ? 0 : k + 1;
            double ex = X[j] - X[k], ey = Y[j] - Y[k];
            double ff = dfma(ex, fy - Y[k], -(ey * (fx - X[k])));
            double ft = dfma(ex, ty - Y[k], -(ey * (tx - X[k])));
            if (o < 0) { ff = -ff; ft = -ft; }
            if (!(ft < 0.0)) continue;
            double te = ff / (ff - ft);
            if (best < 0 || te < bt) { best = k; bt = te; }
        }
        if (best < 0 || !((m >> best) & 1)) continue;  // no crossing, or the edge has a same-facing neighbour
        int clamped = 0;
        if (bt < 0.0) { bt = 0.0; clamped = 1; }
        if (bt > 1.0) { bt = 1.0; clamped = 1; }
        res.tri = t;
        res.edge = best;
        res.from_a = use_a;
        res.clamped = clamped;
        if (bt < 0.5) { res.recv = use_a ? 0 : 1; res.wgt = (float)(0.5 - bt); }
        else { res.recv = use_a ? 1 : 0; res.wgt = (float)(bt - 0.5); }
        return res;
    }
    return res;
}

__device__ __forceinline__ AAImg aa_img(const AALaunch &L, int img) {
    AAImg I;
    if (L.um.n) {  // uneven batch: the item's pixels; vertices and triangles are global
        I.rast = reinterpret_cast<const float4 *>(L.rast) + L.um.pix[img];
        I.proj = L.proj;
        I.orient = L.orient;
        I.silh = L.silh;
        I.V = L.V;
        I.F = L.F;
        I.H = L.um.hw[2 * img];
        I.W = L.um.hw[2 * img + 1];
        return I;
    }
    long long npx = (long long)L.H * L.W;
    I.rast = reinterpret_cast<const float4 *>(L.rast) + img * npx;
    int pimg = L.pos_batched ? img : 0;
    I.proj = L.proj + (long long)pimg * L.V;
    I.orient = L.orient + (long long)pimg * L.F;
    I.silh = L.silh + (long long)pimg * L.F;
    I.V = L.V;
    I.F = L.F;
    I.H = L.H;
    I.W = L.W;
    return I;
}

// silhouette byte of the triangle id - 1, without a branch around the load
// (callers guarantee F > 0), so that several of them issue together
__device__ __forceinline__ int silh_at(const AAImg &I, int id) {
    const int s = I.silh[id > 0 ? id - 1 : 0];
    return id > 0 ? s : 0;
}

// ----------------------------------------------------------------------------
// blocks and their pair lists
// ----------------------------------------------------------------------------
// A block owns kAAW x kAAH pixels and, with them, the pairs to their right and
// above; the pairs that reach in from the column to the left and the row below
// are evaluated by this block as well as by their owner (14 % more pair tests),
// so a block blends all its pixels from pairs it holds in LDS.  Pair slots:
// right pairs row * (kAAW + 1) + column + 1 (column -1: from the left), then
// upward pairs (row + 1) * kAAW + column (row -1: from below).
//
// What the backward needs is kept as a list of the owned pairs that blend
// (8 bytes each, on silhouettes only) instead of 16 bytes for every pixel:
// two bit masks per row say which pairs are listed, row by row, right pairs
// before upward pairs, in lane order.  A block's entries start at twice its
// pixels' offset, so the arrays hold every pair of the image if need be.
constexpr int kAARight = (kAAW + 1) * kAAH;              // right-pair slots
constexpr int kAASlots = kAARight + kAAW * (kAAH + 1);   // all pair slots
constexpr int kAAPer = kAAW * kAAH / 256;                // pixels per thread
static_assert(kAAW == 64 && kAAH % 4 == 0, "a wave owns rows of 64 pixels");

// the listed pair's corner * 2 + from_a: corner 3 * triangle + edge (corners are
// 32-bit integers throughout, so 2 * corner + 1 fits)
constexpr unsigned kAANone = 0xffffffffu;     // does not blend
constexpr unsigned kAAClamped = 0xfffffffeu;  // blends with a clamped, hence constant, weight

__device__ __forceinline__ int right_slot(int row, int col) { return row * (kAAW + 1) + col + 1; }
__device__ __forceinline__ int up_slot(int row, int col) { return kAARight + (row + 1) * kAAW + col; }

struct PairPos {
    int row, col, dir;  // pixel a within the block (-1: outside), direction (0 right, 1 up)
};
__device__ __forceinline__ PairPos slot_pos(int m) {
    PairPos p;
    p.dir = m >= kAARight;
    if (p.dir) {
        m -= kAARight;
        p.row = m / kAAW - 1;
        p.col = m % kAAW;
    } else {
        p.row = m / (kAAW + 1);
        p.col = m % (kAAW + 1) - 1;
    }
    return p;
}

struct AABlock {
    int img, r0, c0;
    long long pix0;   // the image's first pixel
    long long ent0;   // the block's first list entry
    AAHalo *halo;
};

// block `lin` of the launch; false past the last one
__device__ __forceinline__ bool aa_block(const AALaunch &L, int lin, AABlock &B) {
    int bx, by, H, W;
    if (L.um.n) {  // uneven batch: every item's blocks in turn
        if (lin >= L.total_blk) return false;
        B.img = um_find(L.um.blk, L.um.n, lin);
        H = L.um.hw[2 * B.img];
        W = L.um.hw[2 * B.img + 1];
        const int lb = lin - L.um.blk[B.img], nbx = (W + kAAW - 1) / kAAW;
        bx = lb % nbx;
        by = lb / nbx;
        B.pix0 = L.um.pix[B.img];
    } else {
        H = L.H;
        W = L.W;
        const int gx = (W + kAAW - 1) / kAAW, gy = (H + kAAH - 1) / kAAH;
        if (lin >= gx * gy * L.n_img) return false;
        bx = lin % gx;
        by = (lin / gx) % gy;
        B.img = lin / (gx * gy);
        B.pix0 = (long long)B.img * H * W;
    }
    B.r0 = by * kAAH;
    B.c0 = bx * kAAW;
    B.ent0 = 2 * (B.pix0 + (long long)B.r0 * W + (long long)min(kAAH, H - B.r0) * B.c0);
    B.halo = L.halo + lin;
    return true;
}

// first entry of each (row, direction) of the list, in lanes 0 .. 2 kAAH - 1
// (lane 2 row + direction holds that mask's bits in m); n: entries in all
__device__ __forceinline__ int mask_starts(unsigned long long m, int &n) {
    const int cnt = (int)(threadIdx.x & 63) < 2 * kAAH ? __popcll(m) : 0;
    const int x = wave_incl_scan(cnt);
    n = __builtin_amdgcn_readlane(x, 2 * kAAH - 1);
    return x - cnt;
}
__device__ __forceinline__ int below_lane(unsigned long long m) {  // set bits below this lane
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
}
__device__ __forceinline__ unsigned long long readlane64(unsigned long long v, int lane) {
    return ((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(v >> 32), lane) << 32) |
           (unsigned)__builtin_amdgcn_readlane((int)v, lane);
}

// Channels handled by one thread: 4 (one float4) when C is a multiple of 4, a whole
// pixel below 8 channels (a wave's accesses still cover whole lines, and the
// pixel's weights are read once: 24 views of 361 x 641 x 3, 126 -> 115 us; 3 of 733 x
// 1019 x 5, 52 -> 37 us forward and 54 -> 44 backward), else 1 (9 channels and more that are
// no whole quads: whole pixels were not tried there).
// CV > 0: compile-time channel count; 0: runtime; kAnyQuads: runtime, a multiple of 4
constexpr int kAnyQuads = -4;
template <int CV>
struct AAChunk {
    static constexpr int CH = CV != 0 && CV % 4 == 0 ? 4 : (CV > 0 && CV < 8 ? CV : 1);
};

// CH floats from p; 16-byte aligned when CH is a multiple of 4
template <int CH>
__device__ __forceinline__ void ld(const float *p, float *x) {
    if constexpr (CH > 0 && CH % 4 == 0) {
        const float4 v = *reinterpret_cast<const float4 *>(p);
        x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
        ld<CH - 4>(p + 4, x + 4);
    } else if constexpr (CH > 0) {
        constexpr int N = CH > 4 ? 4 : CH;
        typedef float vec __attribute__((ext_vector_type(N), aligned(4)));
        const vec v = *reinterpret_cast<const vec *>(p);
#pragma unroll
        for (int i = 0; i < N; ++i) x[i] = v[i];
        if constexpr (CH > 4 && CH < 8) {
            typedef float rest_t __attribute__((ext_vector_type(CH - 4), aligned(4)));
            const rest_t r = *reinterpret_cast<const rest_t *>(p + 4);
#pragma unroll
            for (int i = 4; i < CH; ++i) x[i] = r[i - 4];
        }
    }
}
// streaming (non-temporal) stores: the output is not read again by this pass
template <int CH>
__device__ __forceinline__ void st(float *p, const float *x) {
    if constexpr (CH > 0 && CH % 4 == 0) {
        typedef float v4 __attribute__((ext_vector_type(4)));
        const v4 v = {x[0], x[1], x[2], x[3]};
        __builtin_nontemporal_store(v, reinterpret_cast<v4 *>(p));
        st<CH - 4>(p + 4, x + 4);
    } else if constexpr (CH > 0) {
        constexpr int N = CH > 4 ? 4 : CH;
        typedef float vec __attribute__((ext_vector_type(N), aligned(4)));
        vec v;
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] = x[i];
        __builtin_nontemporal_store(v, reinterpret_cast<vec *>(p));
        if constexpr (CH > 4 && CH < 8) {
            typedef float rest_t __attribute__((ext_vector_type(CH - 4), aligned(4)));
            rest_t r;
#pragma unroll
            for (int i = 4; i < CH; ++i) r[i - 4] = x[i];
            __builtin_nontemporal_store(r, reinterpret_cast<rest_t *>(p + 4));
        }
    }
}

// The block's (pixel, channel chunk) items in memory order, 256 at a time (so
// consecutive threads touch consecutive bytes), G of a thread's items per step.
// A step's own values are loaded ahead (aa_own); the blend then issues all loads
// of an item's neighbours before it waits for any.  Waiting for each neighbour
// where it is used took 16 round trips per step on a folded mesh and 40 % of a
// block's time; a second item's loads in flight cost more in waves than they hide.
template <int CV>
struct AASweep {
    static constexpr int CH = AAChunk<CV>::CH, G = CV == 8 || CV == 16 ? 4 : (CH > 4 ? 1 : 2);
    // byte offsets from the pixel before the block's first in the row below
    typedef std::conditional_t<(CV > 0), unsigned, unsigned long long> off_t;
    int C, nch, steps;  // steps: a multiple of 2
    int lp, k;          // this thread's next item: local pixel, chunk
    float own[G][CH];
    int px[G];          // the step's items: local pixel, -1: outside
    off_t at[G];
    long long org;
    off_t dx, dy;

    __device__ __forceinline__ AASweep(const AALaunch &L, const AABlock &B, int W) {
        C = CV > 0 ? CV : L.C;
        nch = C / CH;
        steps = kAAW * kAAH * nch / 256;
        lp = threadIdx.x / nch;
        k = threadIdx.x - lp * nch;
        dx = (off_t)C * 4;
        dy = (off_t)W * C * 4;
        org = ((B.pix0 + (long long)(B.r0 - 1) * W + B.c0) - 1) * C;
    }
    static __device__ __forceinline__ const float *ptr(const float *base, off_t off) {
        return reinterpret_cast<const float *>(reinterpret_cast<const char *>(base) + off);
    }
    // the next step's own values (step s)
    __device__ __forceinline__ void load(const AABlock &B, int H, int W, const float *src, int s) {
        const int dpx = 256 / nch, dch = 256 - dpx * nch;
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const int row = lp / kAAW, col = lp % kAAW;
            const bool in = s + j < steps && B.c0 + col < W && B.r0 + row < H;
            px[j] = in ? lp : -1;
            at[j] = (off_t)(row + 1) * dy + (off_t)(col + 1) * dx + (off_t)k * (4 * CH);
            if (in) ld<CH>(ptr(src + org, at[j]), own[j]);
            lp += dpx;
            k += dch;
            if (k >= nch) {
                k -= nch;
                ++lp;
            }
        }
    }
    // forward (BWD false): own + sum w (neighbour - own) over the pairs that the
    // pixel receives from; backward: (1 - sum of those w) own + sum w neighbour
    // over the pairs whose other pixel received from it
    template <bool BWD>
    __device__ __forceinline__ void blend(const float *src, float *dst, const float *s_w) {
#pragma unroll
        for (int j = 0; j < G; ++j) {
            if (px[j] < 0) continue;
            const int row = px[j] / kAAW, col = px[j] % kAAW;
            const float wl = s_w[right_slot(row, col - 1)], wr = s_w[right_slot(row, col)];
            const float wd = s_w[up_slot(row - 1, col)], wu = s_w[up_slot(row, col)];
            const float recv[4] = {wl, -wr, wd, -wu};  // > 0: this pixel receives (comparisons drop NaN)
            const off_t nat[4] = {at[j] - dx, at[j] + dx, at[j] - dy, at[j] + dy};
            float w[4], nb[4][CH], o[CH], self = 0.f;
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                if (BWD && recv[d] > 0.f) self += recv[d];
                const float x = BWD ? -recv[d] : recv[d];
                w[d] = x > 0.f ? x : 0.f;
                if (w[d] > 0.f) ld<CH>(ptr(src + org, nat[d]), nb[d]);
            }
#pragma unroll
            for (int i = 0; i < CH; ++i) o[i] = BWD ? own[j][i] - self * own[j][i] : own[j][i];
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                if (!(w[d] > 0.f)) continue;
#pragma unroll
                for (int i = 0; i < CH; ++i) o[i] = fma_(w[d], BWD ? nb[d][i] : nb[d][i] - own[j][i], o[i]);
            }
            st<CH>(const_cast<float *>(ptr(dst + org, at[j])), o);
        }
    }
    // every step, the first one's own values already loaded
    template <bool BWD>
    __device__ __forceinline__ void run(const AABlock &B, int H, int W, const float *src, float *dst, const float *s_w) {
        for (int s = 0;;) {
            blend<BWD>(src, dst, s_w);
            s += G;
            if (s >= steps) break;
            load(B, H, W, src, s);
        }
    }
};

// Forward of one block of kAAW x kAAH pixels, kAAPer rows four apart per thread
// (their loads are in flight together).  Only pairs whose two triangles differ
// and that have a silhouette-capable edge on either side can blend; the block
// queues those in LDS and evaluates the queue densely, so the double-precision
// crossing runs on full waves.  The blend then takes all weights from LDS.
//
// Pairs, blend and list in one kernel: as two passes with 16 bytes of pair
// state per pixel between them, the pair search (waiting on chains of dependent
// loads) and the blend (bandwidth) took their times one after the other:
// 454 us, now 349 at 64 x 512^2 x 8 (1.4 GB; with fewer waves it is slower).
//
// Eight waves per SIMD (64 VGPRs, no spill): more waves hide more of the
// search's waits.
template <int CV>
__global__ void __launch_bounds__(256, 8) k_aa_fwd(AALaunch L) {
    __shared__ unsigned q[kAASlots];  // pair slot | its pixels' silhouette bytes << 16, << 20
    __shared__ float s_w[kAASlots];
    __shared__ unsigned s_word[kAASlots];
    __shared__ unsigned long long s_mask[2 * kAAH];
    __shared__ int q_n;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // one row of blocks, dealt to the XCDs in groups of neighbours
    AABlock B;
    if (!aa_block(L, xcd_deal(blockIdx.x, L.xcd), B)) return;  // uniform per block
    const AAImg I = aa_img(L, B.img);
    const int H = I.H, W = I.W;
    const int c = B.c0 + lane;
    bool in[kAAPer], has_r[kAAPer], has_u[kAAPer], has_l[kAAPer];
    float w0[kAAPer], wr[kAAPer], wu[kAAPer], wl[kAAPer], wd = 0.f;
    const bool has_d = wave == 0 && c < W && B.r0 > 0 && I.F > 0;
#pragma unroll
    for (int j = 0; j < kAAPer; ++j) {
        const int r = B.r0 + wave + 4 * j;
        in[j] = c < W && r < H && I.F > 0;
        const long long g = (long long)r * W + c;
        has_r[j] = in[j] && c + 1 < W;
        has_u[j] = in[j] && r + 1 < H;
        has_l[j] = in[j] && lane == 0 && c > 0;
        w0[j] = wr[j] = wu[j] = wl[j] = 0.f;
        if (in[j]) {  // the neighbours' ids come from rast's w alone; all loads issue before the first wait
            w0[j] = I.rast[g].w;
            wr[j] = I.rast[has_r[j] ? g + 1 : g].w;
            wu[j] = I.rast[has_u[j] ? g + W : g].w;
            if (has_l[j]) wl[j] = I.rast[g - 1].w;
        }
    }
    if (has_d) wd = I.rast[(long long)(B.r0 - 1) * W + c].w;
    for (int m = tid; m < kAASlots; m += 256) {
        s_w[m] = 0.f;
        s_word[m] = kAANone;
    }
    if (tid == 0) q_n = 0;
    // the pairs (pixel, right), (pixel, above), (left, pixel), (below, pixel) that may blend: silhouette bytes of
    // their two pixels << 1 | 1
    int cand[kAAPer][4];
    int nq = 0;
#pragma unroll
    for (int j = 0; j < kAAPer; ++j) {
#pragma unroll
        for (int d = 0; d < 4; ++d) cand[j][d] = 0;
        if (in[j]) {
            const int i0 = rast_id_w(w0[j], I.F), ir = rast_id_w(wr[j], I.F), iu = rast_id_w(wu[j], I.F);
            const int s0 = silh_at(I, i0), sr = silh_at(I, ir), su = silh_at(I, iu);
            if (has_r[j] && ir != i0 && ((s0 | sr) & 7)) cand[j][0] = (s0 | sr << 4) << 1 | 1;
            if (has_u[j] && iu != i0 && ((s0 | su) & 7)) cand[j][1] = (s0 | su << 4) << 1 | 1;
            if (has_l[j]) {
                const int il = rast_id_w(wl[j], I.F), sl = silh_at(I, il);
                if (il != i0 && ((s0 | sl) & 7)) cand[j][2] = (sl | s0 << 4) << 1 | 1;
            }
            if (j == 0 && has_d) {
                const int id = rast_id_w(wd, I.F), sd = silh_at(I, id);
                if (id != i0 && ((s0 | sd) & 7)) cand[j][3] = (sd | s0 << 4) << 1 | 1;
            }
        }
#pragma unroll
        for (int d = 0; d < 4; ++d) nq += cand[j][d] & 1;
    }
    __syncthreads();
    // wave-aggregated append
    const int x = wave_incl_scan(nq);
    int base = 0;
    if (lane == 63 && x > 0) base = atomicAdd(&q_n, x);
    base = __builtin_amdgcn_readlane(base, 63) + x - nq;
#pragma unroll
    for (int j = 0; j < kAAPer; ++j) {
        const int row = wave + 4 * j;
        const int slot[4] = {right_slot(row, lane), up_slot(row, lane), right_slot(row, -1), up_slot(-1, lane)};
#pragma unroll
        for (int d = 0; d < 4; ++d)
            if (cand[j][d]) q[base++] = (unsigned)slot[d] | (unsigned)(cand[j][d] >> 1) << 16;
    }
    __syncthreads();
    const int n = q_n;
    for (int e = tid; e < n; e += 256) {
        const int m = q[e] & 0xffff, sa = (q[e] >> 16) & 15, sb = q[e] >> 20;
        const PairPos pp = slot_pos(m);
        const int ra = B.r0 + pp.row, ca = B.c0 + pp.col, rb = ra + pp.dir, cb = ca + 1 - pp.dir;
        const float4 pa = I.rast[(long long)ra * W + ca], pb = I.rast[(long long)rb * W + cb];
        const PairRes p = eval_pair(I, L.tri, pa, pb, sa, sb, ra, ca, rb, cb);
        if (p.recv < 0) continue;
        s_w[m] = p.recv == 1 ? p.wgt : -p.wgt;  // > 0: b receives from a, < 0: a from b
        s_word[m] = p.clamped ? kAAClamped : 2u * (3u * (unsigned)p.tri + (unsigned)p.edge) + (unsigned)p.from_a;
    }
    __syncthreads();
    AASweep<CV> sweep(L, B, W);
    if (L.out) sweep.load(B, H, W, L.color, 0);
    // the list of the owned pairs
    unsigned long long mr[kAAPer], mu[kAAPer];
#pragma unroll
    for (int j = 0; j < kAAPer; ++j) {
        const int row = wave + 4 * j;
        mr[j] = __ballot(s_word[right_slot(row, lane)] != kAANone);
        mu[j] = __ballot(s_word[up_slot(row, lane)] != kAANone);
        if (lane == 0) {
            s_mask[2 * row] = mr[j];
            s_mask[2 * row + 1] = mu[j];
        }
    }
    if (tid < kAAW) B.halo->below[tid] = s_w[up_slot(-1, tid)];
    else if (tid < kAAW + kAAH) B.halo->left[tid - kAAW] = s_w[right_slot(tid - kAAW, -1)];
    __syncthreads();
    const unsigned long long m = lane < 2 * kAAH ? s_mask[lane] : 0ull;
    if (tid < 2 * kAAH) B.halo->mask[tid] = m;
    int n_ent;
    const int start = mask_starts(m, n_ent);
#pragma unroll
    for (int j = 0; j < kAAPer; ++j) {
        const int row = wave + 4 * j;
        const int er = __builtin_amdgcn_readlane(start, 2 * row) + below_lane(mr[j]);
        const int eu = __builtin_amdgcn_readlane(start, 2 * row + 1) + below_lane(mu[j]);
        if ((mr[j] >> lane) & 1) {
            L.ent_w[B.ent0 + er] = s_w[right_slot(row, lane)];
            L.ent_word[B.ent0 + er] = s_word[right_slot(row, lane)];
        }
        if ((mu[j] >> lane) & 1) {
            L.ent_w[B.ent0 + eu] = s_w[up_slot(row, lane)];
            L.ent_word[B.ent0 + eu] = s_word[up_slot(row, lane)];
        }
    }
    if (!L.out) return;  // the list alone
    sweep.template run<false>(B, H, W, L.color, L.out, s_w);
}

// Per-block accumulation of vertex gradients before the global atomics.
// Device-scope float atomics on a multi-XCD GPU are performed beyond the
// per-XCD L2 caches, so every one is a memory transaction; neighbouring
// silhouette pairs share vertices, and summing them per 64 x 8 block first
// leaves one atomic per distinct vertex and component.
constexpr int kAAHashBits = 9;
// table slots per block: its pairs touch 41 vertices on average at 512^2 with 82k triangles (119 at most), 163 at
// 361 x 641 with 328k (309 at most)
constexpr int kAAHash = 1 << kAAHashBits;

struct VertexAcc {
    int key[kAAHash];
    float gx[kAAHash], gy[kAAHash], gw[kAAHash];
};

__device__ __forceinline__ void vacc_add(VertexAcc &A, float *GP, int v, float gx, float gy, float gw) {
    unsigned h = ((unsigned)v * 2654435761u) >> (32 - kAAHashBits);  // top bits
#pragma unroll 1  // unrolled, the probes fill the instruction cache and spill scalar registers
    for (int probe = 0; probe < 32; ++probe) {
        int k = atomicCAS(&A.key[h], -1, v);
        if (k == -1 || k == v) {
            atomicAdd(&A.gx[h], gx);
            atomicAdd(&A.gy[h], gy);
            atomicAdd(&A.gw[h], gw);
            return;
        }
        h = (h + 1) & (kAAHash - 1);
    }
    float *gp = GP + 4 * (long long)v;  // table crowded: straight to memory
    atomicAdd(gp + 0, gx);
    atomicAdd(gp + 1, gy);
    atomicAdd(gp + 3, gw);
}

// Position gradient of one blending pair: dL/dw (from the receiver's output
// gradient and the colour difference) times dw/dt times dt/d(edge vertices).
// The pair's decisions are the forward's; the derivative is taken in double:
// t = fa / (fa - fb) is ill-conditioned for edges nearly parallel to the pair.
// The edge's vertex loads do not wait for dL/dw, and the result is returned
// rather than added, so the loads of a pixel's two pairs overlap.
struct PairGrad {
    int v[2];
    float gx[2], gy[2], gw[2];
    bool live;
};

__device__ __forceinline__ void edge_vertices(const int *__restrict__ tri, unsigned corner, int &v0, int &v1) {
    v0 = tri[corner];
    v1 = tri[corner % 3u == 2u ? corner - 2u : corner + 1u];
}

// pair from pixel a = (r, c) in direction dir: a or b (recv) receives, through
// edge (v0, v1) of triangle t, left from a's or b's side (from_a)
__device__ __forceinline__ PairGrad pair_pos_grad(const AALaunch &L, const AAImg &I, const float4 *P, long long g,
                                                  int r, int c, int dir, int recv, int from_a, unsigned t, int v0,
                                                  int v1) {
    PairGrad out;
    const int rb = dir ? r + 1 : r, cb = dir ? c : c + 1;
    const long long ga = g, gb = dir ? g + I.W : g + 1;
    const long long gr = recv == 0 ? ga : gb, gs = recv == 0 ? gb : ga;
    out.v[0] = v0;
    out.v[1] = v1;
    const double2 q0 = I.proj[out.v[0]], q1 = I.proj[out.v[1]];
    const float4 pv[2] = {P[out.v[0]], P[out.v[1]]};
    const double so = I.orient[t] < 0 ? -1.0 : 1.0;
    double dLdw = 0.0;
    if ((L.C & 3) == 0) {
        const float4 *g4 = reinterpret_cast<const float4 *>(L.grad_out + gr * L.C);
        const float4 *cs = reinterpret_cast<const float4 *>(L.color + gs * L.C);
        const float4 *cr = reinterpret_cast<const float4 *>(L.color + gr * L.C);
        for (int k4 = 0; k4 < (L.C >> 2); ++k4) {
            float4 a = g4[k4], b = cs[k4], e = cr[k4];
            dLdw += (double)a.x * (b.x - e.x) + (double)a.y * (b.y - e.y) + (double)a.z * (b.z - e.z) +
                    (double)a.w * (b.w - e.w);
        }
    } else {
        for (int ch = 0; ch < L.C; ++ch)
            dLdw += (double)L.grad_out[gr * L.C + ch] * (L.color[gs * L.C + ch] - L.color[gr * L.C + ch]);
    }
    out.live = dLdw != 0.0;
    const bool recv_is_from = (recv == 0) == (from_a != 0);
    const double dLdt = recv_is_from ? -dLdw : dLdw;
    const double fxp = (double)(from_a ? c : cb) + 0.5, fyp = (double)(from_a ? r : rb) + 0.5;
    const double txp = (double)(from_a ? cb : c) + 0.5, typ = (double)(from_a ? rb : r) + 0.5;
    const double ex = q1.x - q0.x, ey = q1.y - q0.y;
    const double fa = so * (ex * (fyp - q0.y) - ey * (fxp - q0.x));
    const double fb = so * (ex * (typ - q0.y) - ey * (txp - q0.x));
    const double den = fa - fb;
    const double dt_dfa = -fb / (den * den), dt_dfb = fa / (den * den);
    const double k = dLdt * so * (double)L.boost;
    double gx2[2], gy2[2];
    gx2[0] = k * (dt_dfa * (q1.y - fyp) + dt_dfb * (q1.y - typ));
    gy2[0] = k * (dt_dfa * (fxp - q1.x) + dt_dfb * (txp - q1.x));
    gx2[1] = k * (dt_dfa * (fyp - q0.y) + dt_dfb * (typ - q0.y));
    gy2[1] = k * (dt_dfa * (q0.x - fxp) + dt_dfb * (q0.x - txp));
    const double hw = (double)I.W * 0.5, hh = (double)I.H * 0.5;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        double iw = 1.0 / (double)pv[m].w;
        double gx = gx2[m] * hw * iw, gy = gy2[m] * hh * iw;
        out.gx[m] = (float)gx;
        out.gy[m] = (float)gy;
        out.gw[m] = (float)(-(gx * pv[m].x + gy * pv[m].y) * iw);
    }
    return out;
}

__device__ __forceinline__ void pair_grad_add(VertexAcc &A, float *GP, const PairGrad &pg) {
    if (!pg.live) return;
#pragma unroll
    for (int m = 0; m < 2; ++m) vacc_add(A, GP, pg.v[m], pg.gx[m], pg.gy[m], pg.gw[m]);
}

// Backward of one block: the forward's list gives the weights of every pair
// that touches its pixels (colour gradients, one pass over them) and, by
// consecutive lanes, the position gradients of its own pairs, summed per vertex
// in the block's table and flushed with one atomic request per vertex.  One
// kernel for both, so that the pairs find output gradients in the caches: 343 us
// at 64 x 512^2 x 8, against 430 for a colour and a position kernel side by side.
// Eight waves per SIMD as the forward (at 16 channels two VGPRs spill for it, 12
// bytes of scratch a lane).
template <int CV>
__global__ void __launch_bounds__(256, 8) k_aa_bwd(AALaunch L) {
    __shared__ VertexAcc A;
    __shared__ float s_w[kAASlots];
    __shared__ unsigned short s_slot[2 * kAAW * kAAH];  // pair slot of each list entry
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    AABlock B;
    if (!aa_block(L, xcd_deal(blockIdx.x, L.xcd), B)) return;  // uniform per block
    const AAImg I = aa_img(L, B.img);
    AASweep<CV> sweep(L, B, I.W);
    sweep.load(B, I.H, I.W, L.grad_out, 0);
    const unsigned long long mask = lane < 2 * kAAH ? B.halo->mask[lane] : 0ull;
    if (tid < kAAW) s_w[up_slot(-1, tid)] = B.halo->below[tid];
    else if (tid < kAAW + kAAH) s_w[right_slot(tid - kAAW, -1)] = B.halo->left[tid - kAAW];
    const bool want_pos = L.grad_pos != nullptr;
    if (want_pos)
        for (int e = tid; e < kAAHash; e += 256) {
            A.key[e] = -1;
            A.gx[e] = 0.f;
            A.gy[e] = 0.f;
            A.gw[e] = 0.f;
        }
    int n;
    const int start = mask_starts(mask, n);
    float w[2 * kAAPer];
    int at[2 * kAAPer];
#pragma unroll
    for (int j = 0; j < 2 * kAAPer; ++j) {  // all loads issue before the first wait (unlisted pairs read entry 0)
        const int i = 2 * (wave + 4 * (j >> 1)) + (j & 1);
        const unsigned long long m = readlane64(mask, i);
        const int e = __builtin_amdgcn_readlane(start, i) + below_lane(m);
        at[j] = (m >> lane) & 1 ? e : -1;
        w[j] = L.ent_w[B.ent0 + max(at[j], 0)];
    }
    // past the list's end nothing was written: its words are not read
    const unsigned word0 = want_pos && tid < n ? L.ent_word[B.ent0 + tid] : kAANone;
#pragma unroll
    for (int j = 0; j < 2 * kAAPer; ++j) {
        const int row = wave + 4 * (j >> 1);
        const int slot = j & 1 ? up_slot(row, lane) : right_slot(row, lane);
        s_w[slot] = at[j] >= 0 ? w[j] : 0.f;
        if (at[j] >= 0) s_slot[at[j]] = (unsigned short)slot;
    }
    __syncthreads();
    // the pair's edge vertices, on their way during the colour gradients
    int v0 = 0, v1 = 0;
    if (word0 < kAAClamped) edge_vertices(L.tri, word0 >> 1, v0, v1);
    sweep.template run<true>(B, I.H, I.W, L.grad_out, L.grad_color, s_w);
    if (!want_pos || n == 0) return;  // uniform across the block
    const float4 *P = reinterpret_cast<const float4 *>(L.pos) + (L.pos_batched ? (long long)B.img * L.V : 0);
    float *GP = L.grad_pos + (L.pos_batched ? (long long)B.img * L.V * 4 : 0);
    for (int e = tid; e < n; e += 256) {
        const unsigned word = e < 256 ? word0 : L.ent_word[B.ent0 + e];
        if (word >= kAAClamped) continue;
        const int m = s_slot[e];
        const PairPos pp = slot_pos(m);
        const float w = s_w[m];
        const int from_a = word & 1;
        const int recv = isnan(w) ? from_a : !signbit(w);  // an undefined crossing moves the far pixel
        const int r = B.r0 + pp.row, c = B.c0 + pp.col;
        if (e >= 256) edge_vertices(L.tri, word >> 1, v0, v1);
        pair_grad_add(A, GP, pair_pos_grad(L, I, P, B.pix0 + (long long)r * I.W + c, r, c, pp.dir, recv, from_a,
                                           (word >> 1) / 3u, v0, v1));
    }
    __syncthreads();
    // four lanes per vertex (x, y, none, w): its components leave as one request
    for (int i = tid; i < 4 * kAAHash; i += 256) {
        const int e = i >> 2, k = i & 3, v = A.key[e];
        if (v < 0 || k == 2) continue;
        atomicAdd(GP + 4 * (long long)v + k, k == 0 ? A.gx[e] : k == 1 ? A.gy[e] : A.gw[e]);
    }
}

#define DRP_AA_CASE(KERNEL, CV) \
    case CV: hipLaunchKernelGGL(KERNEL<CV>, grid, dim3(256), 0, st, L); break;
#define DRP_AA_DISPATCH(KERNEL)                                                                     \
    switch (L.C) {                                                                                  \
        DRP_AA_CASE(KERNEL, 1)                                                                      \
        DRP_AA_CASE(KERNEL, 2)                                                                      \
        DRP_AA_CASE(KERNEL, 3)                                                                      \
        DRP_AA_CASE(KERNEL, 4)                                                                      \
        DRP_AA_CASE(KERNEL, 5)                                                                      \
        DRP_AA_CASE(KERNEL, 6)                                                                      \
        DRP_AA_CASE(KERNEL, 7)                                                                      \
        DRP_AA_CASE(KERNEL, 8)                                                                      \
        DRP_AA_CASE(KERNEL, 16)                                                                     \
        default:                                                                                    \
            if (L.C % 4 == 0) hipLaunchKernelGGL(KERNEL<kAnyQuads>, grid, dim3(256), 0, st, L);     \
            else hipLaunchKernelGGL(KERNEL<0>, grid, dim3(256), 0, st, L);                          \
    }

static void launch_orient(const AALaunch &L, hipStream_t st) {
    int n_proj = L.pos_batched ? L.n_img : 1;
    long long nv = (long long)n_proj * L.V, nf = (long long)n_proj * L.F;
    const long long fblk = (((nf + 255) / 256) + 7) & ~7ll;  // a multiple of 8 blocks (xcd_remap)
    const long long blk = fblk + (nv + 255) / 256;
    if (blk)
        hipLaunchKernelGGL(k_aa_orient, dim3((unsigned)blk), dim3(256), 0, st, L.pos, L.V, L.tri, L.F, n_proj, L.H, L.W,
                           L.um, (int)fblk, L.orient, L.proj);
    if (nf)
        hipLaunchKernelGGL(k_aa_silhouette, dim3((unsigned)fblk), dim3(256), 0, st, L.opp, L.orient, L.F, n_proj, L.silh);
}

// blocks of the launch (and AAHalo records of the workspace)
static long long aa_blocks(const AALaunch &L) {
    return L.um.n ? (long long)L.total_blk
                  : (long long)((L.W + kAAW - 1) / kAAW) * ((L.H + kAAH - 1) / kAAH) * L.n_img;
}

// blocks per XCD turn; the grid they make
static AALaunch with_groups(const AALaunch &L0, dim3 &grid) {
    AALaunch L = L0;
    const long long nblk = aa_blocks(L);
    L.xcd = xcd_group(nblk, L.um.n ? 1 : L.n_img, kXcdPixels);
    grid = dim3((unsigned)xcd_pad(nblk, L.xcd));
    return L;
}

static int launch_pairs(const AALaunch &L0, hipStream_t st) {
    const long long nblk = aa_blocks(L0);
    if (nblk == 0) return 0;
    if (nblk >= (1ll << 31) - 8 * kXcdPixels) return -1;
    if (!L0.prepared) launch_orient(L0, st);
    dim3 grid;
    const AALaunch L = with_groups(L0, grid);
    DRP_AA_DISPATCH(k_aa_fwd)
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_antialias(const AALaunch &L, hipStream_t st) { return launch_pairs(L, st); }

// the per-vertex pixel positions and per-triangle orientation and silhouette
// flags alone, for a forward that follows with L.prepared set
int launch_antialias_prepare(const AALaunch &L, hipStream_t st) {
    if (aa_blocks(L) == 0) return 0;
    launch_orient(L, st);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_antialias_bwd(const AALaunch &L0, hipStream_t st) {
    const long long nblk = aa_blocks(L0);
    if (nblk == 0) return 0;
    if (nblk >= (1ll << 31) - 8 * kXcdPixels) return -1;
    // without the forward's state the pairs are evaluated again, for their list alone
    if (!L0.reuse) {
        if (int rc = launch_pairs(L0, st)) return rc;
    }
    dim3 grid;
    const AALaunch L = with_groups(L0, grid);
    DRP_AA_DISPATCH(k_aa_bwd)
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace drp
