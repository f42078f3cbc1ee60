// Attribute interpolation (forward, screen-space derivatives, backward).
// Pixel formula (diffrp/rendering/interpolator.py:43-45):
//   out = (a0 - a2) * u + ((a1 - a2) * v + a2)
#include "drp_common.h"
#include "drp_kernels.h"

namespace drp {

struct InterpPix {
    bool hit;
    int i0, i1, i2;
    float u, v;
};

__device__ __forceinline__ InterpPix interp_pix(const float4 *__restrict__ rast, const int *__restrict__ tri,
                                                long long pix, int F, int V) {
    InterpPix p;
    p.hit = false;
    float4 r = rast[pix];
    if (!(r.w > 0.f)) return p;
    int t = float_to_triidx(r.w) - 1;
    if (t < 0 || t >= F) return p;
    const int *t3 = tri + 3 * (long long)t;
    p.i0 = t3[0]; p.i1 = t3[1]; p.i2 = t3[2];
    if ((unsigned)p.i0 >= (unsigned)V || (unsigned)p.i1 >= (unsigned)V || (unsigned)p.i2 >= (unsigned)V) return p;
    p.u = r.x;
    p.v = r.y;
    p.hit = true;
    return p;
}

// Lanes per pixel of the forward.  From 12 channels up, a pixel's quads go to
// four consecutive lanes, so that a wave's loads of vertex rows and its stores
// cover whole cache lines: one lane per pixel stored 16 bytes in every 64 at 16
// channels, 81 us for 8 x 512^2, 35 us so.  At 8 channels two lanes are slower
// than one (213 against 194 us for 64 x 512^2).  Counts below 8 are compiled: the
// rows of 5 channels then load in two accesses (3 x 733 x 1019: 29 -> 16 us).
template <int CV, bool QUADS>
constexpr int interp_lanes() { return !QUADS || CV == 4 || CV == 8 ? 1 : 4; }

// CV > 0: compile-time channel count, 0: runtime; QUADS: a multiple of 4, rows
// and output 16-byte aligned
template <int CV, bool QUADS>
__global__ void __launch_bounds__(256) k_interp_fwd(const float *__restrict__ attr, int V, int C, int attr_batched,
                                                    const float4 *__restrict__ rast, const int *__restrict__ tri,
                                                    int F, long long first_pix, long long total_pix,
                                                    long long pix_per_img,
                                                    float *__restrict__ out, const float4 *__restrict__ rast_db,
                                                    const int *__restrict__ diff_idx, int n_diff,
                                                    float *__restrict__ out_da) {
    constexpr int LP = interp_lanes<CV, QUADS>();
    const int NC = CV > 0 ? CV : C;
    // groups of blocks dealt to the XCDs: neighbouring pixels share their vertices' rows in one L2
    const long long gt = (long long)xcd_deal(blockIdx.x, kXcdPixels) * blockDim.x + threadIdx.x;
    const long long gid = first_pix + gt / LP;
    const int lane = (int)(gt % LP);
    if (gid >= total_pix) return;
    InterpPix p = interp_pix(rast, tri, gid, F, V);
    float *o = out + gid * NC;
    typedef float v4 __attribute__((ext_vector_type(4)));
    if (!p.hit) {
        if (QUADS) {
            const v4 z = {0.f, 0.f, 0.f, 0.f};
            for (int ch = 4 * lane; ch < NC; ch += 4 * LP) __builtin_nontemporal_store(z, reinterpret_cast<v4 *>(o + ch));
        } else {
            for (int ch = 0; ch < NC; ++ch) o[ch] = 0.f;
        }
        if (out_da)
            for (int j = lane; j < 2 * n_diff; j += LP) out_da[gid * 2 * n_diff + j] = 0.f;
        return;
    }
    const float *A = attr + (attr_batched ? (gid / pix_per_img) * (long long)V * NC : 0);
    const float *a0 = A + (long long)p.i0 * NC, *a1 = A + (long long)p.i1 * NC, *a2 = A + (long long)p.i2 * NC;
    if (QUADS) {
        for (int ch = 4 * lane; ch < NC; ch += 4 * LP) {
            float4 x0 = *reinterpret_cast<const float4 *>(a0 + ch);
            float4 x1 = *reinterpret_cast<const float4 *>(a1 + ch);
            float4 x2 = *reinterpret_cast<const float4 *>(a2 + ch);
            float4 y;
            y.x = fma_(x0.x - x2.x, p.u, fma_(x1.x - x2.x, p.v, x2.x));
            y.y = fma_(x0.y - x2.y, p.u, fma_(x1.y - x2.y, p.v, x2.y));
            y.z = fma_(x0.z - x2.z, p.u, fma_(x1.z - x2.z, p.v, x2.z));
            y.w = fma_(x0.w - x2.w, p.u, fma_(x1.w - x2.w, p.v, x2.w));
            v4 yy = {y.x, y.y, y.z, y.w};
            __builtin_nontemporal_store(yy, reinterpret_cast<v4 *>(o + ch));
        }
    } else {
        for (int ch = 0; ch < NC; ++ch) {
            float x2 = a2[ch];
            o[ch] = fma_(a0[ch] - x2, p.u, fma_(a1[ch] - x2, p.v, x2));
        }
    }
    if (out_da) {
        float4 db = rast_db[gid];
        float *od = out_da + gid * 2 * n_diff;
        for (int j = lane; j < n_diff; j += LP) {
            int ch = diff_idx[j];
            if ((unsigned)ch >= (unsigned)NC) { od[2 * j] = od[2 * j + 1] = 0.f; continue; }
            float d0 = a0[ch] - a2[ch], d1 = a1[ch] - a2[ch];
            od[2 * j + 0] = fma_(d0, db.x, d1 * db.z);
            od[2 * j + 1] = fma_(d0, db.y, d1 * db.w);
        }
    }
}

// backward: grad_attr scatter (atomics), grad_rast (u, v) written per pixel
template <int CV>
__global__ void __launch_bounds__(256) k_interp_bwd(const float *__restrict__ attr, int V, int C, int attr_batched,
                                                    const float4 *__restrict__ rast, const int *__restrict__ tri,
                                                    int F, long long total_pix, long long pix_per_img,
                                                    const float *__restrict__ grad_out, float *__restrict__ grad_attr,
                                                    float4 *__restrict__ grad_rast, const float4 *__restrict__ rast_db,
                                                    const int *__restrict__ diff_idx, int n_diff,
                                                    const float *__restrict__ grad_da, float4 *__restrict__ grad_db) {
    const int NC = CV > 0 ? CV : C;
    long long gid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= total_pix) return;
    InterpPix p = interp_pix(rast, tri, gid, F, V);
    if (!p.hit) {
        grad_rast[gid] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (grad_db) grad_db[gid] = make_float4(0.f, 0.f, 0.f, 0.f);
        return;
    }
    long long aoff = attr_batched ? (gid / pix_per_img) * (long long)V * NC : 0;
    const float *A = attr + aoff;
    float *GA = grad_attr + aoff;
    const float *a0 = A + (long long)p.i0 * NC, *a1 = A + (long long)p.i1 * NC, *a2 = A + (long long)p.i2 * NC;
    float *g0 = GA + (long long)p.i0 * NC, *g1 = GA + (long long)p.i1 * NC, *g2 = GA + (long long)p.i2 * NC;
    const float *g = grad_out + gid * NC;
    float w2 = (1.f - p.u) - p.v;
    float su = 0.f, sv = 0.f;
    for (int ch = 0; ch < NC; ++ch) {
        float gc = g[ch];
        if (gc != 0.f) {
            atomicAdd(g0 + ch, p.u * gc);
            atomicAdd(g1 + ch, p.v * gc);
            atomicAdd(g2 + ch, w2 * gc);
        }
        float x2 = a2[ch];
        su += gc * (a0[ch] - x2);
        sv += gc * (a1[ch] - x2);
    }
    grad_rast[gid] = make_float4(su, sv, 0.f, 0.f);
    if (grad_da && n_diff > 0) {
        float4 db = rast_db[gid];
        const float *gd = grad_da + gid * 2 * n_diff;
        float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
        for (int j = 0; j < n_diff; ++j) {
            int ch = diff_idx[j];
            if ((unsigned)ch >= (unsigned)NC) continue;
            float gx = gd[2 * j], gy = gd[2 * j + 1];
            float d0 = a0[ch] - a2[ch], d1 = a1[ch] - a2[ch];
            float k0 = gx * db.x + gy * db.y, k1 = gx * db.z + gy * db.w;
            atomicAdd(g0 + ch, k0);
            atomicAdd(g1 + ch, k1);
            atomicAdd(g2 + ch, -(k0 + k1));
            s0 += gx * d0; s1 += gy * d0; s2 += gx * d1; s3 += gy * d1;
        }
        if (grad_db) grad_db[gid] = make_float4(s0, s1, s2, s3);
    } else if (grad_db) {
        grad_db[gid] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
}

#define DRP_INTERP_DISPATCH(KERNEL, ...)                                                          \
    switch (L.cv) {                                                                               \
        case 1: hipLaunchKernelGGL(KERNEL<1>, grid, block, 0, st, __VA_ARGS__); break;            \
        case 2: hipLaunchKernelGGL(KERNEL<2>, grid, block, 0, st, __VA_ARGS__); break;            \
        case 3: hipLaunchKernelGGL(KERNEL<3>, grid, block, 0, st, __VA_ARGS__); break;            \
        case 4: hipLaunchKernelGGL(KERNEL<4>, grid, block, 0, st, __VA_ARGS__); break;            \
        case 8: hipLaunchKernelGGL(KERNEL<8>, grid, block, 0, st, __VA_ARGS__); break;            \
        case 16: hipLaunchKernelGGL(KERNEL<16>, grid, block, 0, st, __VA_ARGS__); break;          \
        default: hipLaunchKernelGGL(KERNEL<0>, grid, block, 0, st, __VA_ARGS__); break;           \
    }

template <int CV, bool QUADS>
static void launch_fwd(const InterpLaunch &L, hipStream_t st) {
    constexpr long long most = kMaxBlocks * 256 / interp_lanes<CV, QUADS>();  // pixels of a launch
    for (long long first = 0; first < L.total_pix; first += most) {
        const long long end = first + most < L.total_pix ? first + most : L.total_pix;
        const long long blocks = ((end - first) * interp_lanes<CV, QUADS>() + 255) / 256;
        hipLaunchKernelGGL((k_interp_fwd<CV, QUADS>), dim3((unsigned)xcd_pad(blocks, kXcdPixels)), dim3(256), 0, st,
                           L.attr, L.V, L.C, L.attr_batched, (const float4 *)L.rast, L.tri, L.F, first, end,
                           L.pix_per_img, L.out, (const float4 *)L.rast_db, L.diff_idx, L.n_diff, L.out_da);
    }
}

int launch_interpolate(const InterpLaunch &L, hipStream_t st) {
    if (L.total_pix == 0) return 0;
    // other multiples of four may come without the alignment their quads need
    const bool aligned = (((uintptr_t)L.attr | (uintptr_t)L.out) & 15) == 0;
    switch (L.cv) {
        case 1: launch_fwd<1, false>(L, st); break;
        case 2: launch_fwd<2, false>(L, st); break;
        case 3: launch_fwd<3, false>(L, st); break;
        case 4: launch_fwd<4, true>(L, st); break;
        case 8: launch_fwd<8, true>(L, st); break;
        case 16: launch_fwd<16, true>(L, st); break;
        default:
            if (L.C == 5) launch_fwd<5, false>(L, st);
            else if (L.C == 6) launch_fwd<6, false>(L, st);
            else if (L.C == 7) launch_fwd<7, false>(L, st);
            else if (L.C % 4 == 0 && aligned) launch_fwd<0, true>(L, st);
            else launch_fwd<0, false>(L, st);
    }
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

// ----------------------------------------------------------------------------
// deterministic backward (no atomics)
//   k_tile_reduce / k_tile_gather (drp_tribwd.h): grad_rast per pixel and,
//       per (view group, triangle), (u, v, 1-u-v) * g per corner
//   k_gather_attr_*: per vertex, sum the corner partials (CSR, fixed order)
// Any channel count and the derivatives' gradients: the per-pixel atomics of
// k_interp_bwd above remain for rast that comes without pixel boxes (range
// mode, a modified rast).
// ----------------------------------------------------------------------------
// channels of the next pass over an attribute of C channels, `left` to go: at
// most `most`, and where the rows are not whole quads no multiple of 4 (those
// passes read 16 bytes at a time)
static int pass_channels(int left, int C, int most) {
    const int k = left < most ? left : most;
    return C % 4 && k % 4 == 0 ? k - 1 : k;
}

static int launch_interp_bwd_tri(const InterpLaunch &L, hipStream_t st) {
    int n_img = L.um.n ? 1 : (int)(L.total_pix / L.pix_per_img);  // an uneven batch sums as one group
    int vpg = L.attr_batched ? 1 : L.views_per_group;
    int groups = (n_img + vpg - 1) / vpg;
    TriBwdLaunch T{};
    T.tri = L.tri;
    T.rast = L.rast;
    T.grad_out = L.grad_out;
    T.attr = L.attr;
    T.V = L.V;
    T.attr_batched = L.attr_batched;
    T.ldc = L.C;
    T.grad_rast_out = L.grad_rast;
    T.rast_db = L.rast_db;
    T.diff_idx = L.diff_idx;
    T.n_diff = L.n_diff;
    T.grad_da = L.grad_da;
    T.grad_db_out = L.grad_db;
    T.boxes = L.boxes;
    T.partial = L.partial;
    T.live = L.live;
    T.n_img = n_img;
    T.F = L.F;
    T.H = L.H;
    T.W = L.W;
    T.views_per_block = vpg;
    if (L.um.n) {
        T.um = L.um;
        T.views_per_block = 1;
        tile_records_layout_tiles(T, L.records, L.um_tiles, L.F);
    } else {
        tile_records_layout(T, L.records, n_img, L.H, L.W, (long long)n_img * L.F);
    }
    const int outs = L.attr_batched ? n_img : 1;
    for (int c0 = 0; c0 < L.C;) {
        const int nc = pass_channels(L.C - c0, L.C, L.n_diff > 0 ? 4 : kMaxPassChannels);
        T.c0 = c0;
        T.accum = c0 > 0;
        if (int rc = launch_tri_bwd_attr(T, nc, st)) return rc;
        if (int rc = launch_gather_attr(L.partial, L.live, groups, L.F, L.V, nc, L.C, c0, outs, L.attr_batched,
                                        L.inc_off, L.inc, L.grad_attr, st))
            return rc;
        c0 += nc;
    }
    return 0;
}

int launch_interpolate_bwd(const InterpLaunch &L, hipStream_t st) {
    if (L.total_pix == 0) return 0;
    if (L.boxes && L.partial && L.records && L.inc_off && L.inc) return launch_interp_bwd_tri(L, st);
    dim3 grid((unsigned)((L.total_pix + 255) / 256)), block(256);
    DRP_INTERP_DISPATCH(k_interp_bwd, L.attr, L.V, L.C, L.attr_batched, (const float4 *)L.rast, L.tri, L.F,
                        L.total_pix, L.pix_per_img, L.grad_out, L.grad_attr, (float4 *)L.grad_rast,
                        (const float4 *)L.rast_db, L.diff_idx, L.n_diff, L.grad_da, (float4 *)L.grad_db)
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace drp
