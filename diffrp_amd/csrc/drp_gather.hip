// Per-vertex sums of the tile backward's per-corner partials: attributes,
// positions, and both in one launch.  A corner's row is read only if its
// triangle is live (won a pixel): the tile gather writes no other.
#include "drp_common.h"
#include "drp_kernels.h"

namespace drp {

struct AttrGather {
    const float *partial;  // [groups, F, 3, nc]
    const unsigned char *live;  // [groups, F]: triangles whose rows are written
    int groups, F, V, nc;
    int ldc, c0;           // channels of grad_attr's rows, first channel of this pass
    int per_output;        // one group per output (else every group sums into output 0)
    int lanes, xcd;        // lanes per (vertex, quad), blocks per XCD turn
    const int *inc_off, *inc;
    float *grad_attr;
    int set;               // write the sums instead of adding them
};
struct PosGather {
    const float4 *partial;  // [n_img, 3 F]
    const unsigned char *live;  // [n_img, F]
    int n_img, F, V, pos_batched, xcd;
    const int *inc_off, *inc;
    float4 *grad_pos;
    int set;
};

// s to *o, or added to it (a caller's gradient buffer may lack 16-byte alignment)
__device__ __forceinline__ void put(float *o, float4 s, int set) {
    o[0] = set ? s.x : o[0] + s.x;
    o[1] = set ? s.y : o[1] + s.y;
    o[2] = set ? s.z : o[2] + s.z;
    o[3] = set ? s.w : o[3] + s.w;
}
__device__ __forceinline__ void put(float4 *o, float4 s, int set) {
    if (!set) {
        const float4 cur = *o;
        s = make_float4(cur.x + s.x, cur.y + s.y, cur.z + s.z, cur.w + s.w);
    }
    *o = s;
}

constexpr int kAttrLanes = 4;

// grad_attr[out][v][c0 ..) += sum over groups g in the output's range and
// incident corners, channel counts that are whole quads, with `lanes` lanes per
// (vertex, four channels) (1, 2 or 4: up to the groups each output sums): lane
// s takes groups s, s + lanes, ... (a group's corner rows in flight together,
// summed in corner order), and the lanes' sums are added in a fixed tree.  (One
// lane per (vertex, quad) left the 64-view grid at barely one wave per SIMD
// waiting on its loads.)
__device__ __forceinline__ void gather_attr_q(const AttrGather &A, int blk, int out) {
    const float *__restrict__ partial = A.partial;
    const int *__restrict__ inc_off = A.inc_off, *__restrict__ inc = A.inc;
    const int n_groups = A.groups, F = A.F, V = A.V, NC = A.nc, lanes = A.lanes, per_output_groups = A.per_output;
    const int NQ = NC / 4;
    const long long tl = (long long)blk * blockDim.x + threadIdx.x;
    const int s = (int)(tl & (lanes - 1));
    const long long tq = tl / lanes;
    const int v = (int)(tq / NQ), q = (int)(tq % NQ);
    if (v >= V) return;  // all lanes of (v, q) together
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    const int i0 = inc_off[v], i1 = inc_off[v + 1], deg = i1 - i0;
    const int g0 = per_output_groups ? out : 0, g1 = per_output_groups ? out + 1 : n_groups;
    const long long gstride = (long long)F * 3 * NC;
    if (deg <= 8) {
        int c[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) c[k] = k < deg ? inc[i0 + k] : 0;
        for (int g = g0 + s; g < g1; g += lanes) {
            const float *P = partial + (long long)g * gstride + 4 * q;
            const unsigned char *live = A.live + (long long)g * F;
            float4 x[8];
            bool on[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) on[k] = k < deg && live[(unsigned)c[k] / 3u];
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (on[k]) x[k] = *reinterpret_cast<const float4 *>(P + (long long)c[k] * NC);
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (on[k]) {
                    acc.x += x[k].x; acc.y += x[k].y; acc.z += x[k].z; acc.w += x[k].w;
                }
        }
    } else {
        for (int g = g0 + s; g < g1; g += lanes) {
            const float *P = partial + (long long)g * gstride + 4 * q;
            const unsigned char *live = A.live + (long long)g * F;
            for (int i = i0; i < i1; i += 4) {  // four corners' loads in flight, summed in corner order
                float4 x[4];
                int c[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) c[k] = i + k < i1 ? inc[i + k] : -1;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (c[k] >= 0 && !live[(unsigned)c[k] / 3u]) c[k] = -1;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (c[k] >= 0) x[k] = *reinterpret_cast<const float4 *>(P + (long long)c[k] * NC);
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (c[k] >= 0) {
                        acc.x += x[k].x; acc.y += x[k].y; acc.z += x[k].z; acc.w += x[k].w;
                    }
            }
        }
    }
    for (int o = 1; o < lanes; o <<= 1) {  // (a + b on one lane, b + a on the other: the same sum)
        acc.x += __shfl_xor(acc.x, o, 64);
        acc.y += __shfl_xor(acc.y, o, 64);
        acc.z += __shfl_xor(acc.z, o, 64);
        acc.w += __shfl_xor(acc.w, o, 64);
    }
    if (s != 0) return;
    float *o = A.grad_attr + ((long long)out * V + v) * A.ldc + A.c0 + 4 * q;
    put(o, acc, A.set);
}

// The same one lane per (vertex, channel), for channel counts that are not
// whole quads: consecutive lanes read consecutive floats of a corner's row;
// four corners' loads in flight, summed in corner order.
__device__ __forceinline__ void gather_attr_c(const AttrGather &A, int blk, int out) {
    const float *__restrict__ partial = A.partial;
    const int *__restrict__ inc_off = A.inc_off, *__restrict__ inc = A.inc;
    const int n_groups = A.groups, F = A.F, V = A.V, NC = A.nc, per_output_groups = A.per_output;
    const long long tl = (long long)blk * blockDim.x + threadIdx.x;
    const int v = (int)(tl / NC), ch = (int)(tl - (long long)v * NC);
    if (v >= V) return;
    const int i0 = inc_off[v], i1 = inc_off[v + 1];
    const int g0 = per_output_groups ? out : 0, g1 = per_output_groups ? out + 1 : n_groups;
    float s = 0.f;
    for (int g = g0; g < g1; ++g) {
        const float *P = partial + (long long)g * F * 3 * NC + ch;
        const unsigned char *live = A.live + (long long)g * F;
        for (int i = i0; i < i1; i += 4) {
            float x[4];
            int c[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) c[k] = i + k < i1 ? inc[i + k] : -1;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (c[k] >= 0 && !live[(unsigned)c[k] / 3u]) c[k] = -1;
#pragma unroll
            for (int k = 0; k < 4; ++k) x[k] = c[k] >= 0 ? P[(long long)c[k] * NC] : 0.f;
#pragma unroll
            for (int k = 0; k < 4; ++k) s += x[k];
        }
    }
    float *o = A.grad_attr + ((long long)out * V + v) * A.ldc + A.c0 + ch;
    *o = A.set ? s : *o + s;
}

// grad_pos[img][v] += sum over incident corners of partial[pimg][corner]
// (pos_batched: one output per image; else all images sum into one buffer): a
// thread per vertex, eight corners' bytes, then their rows, in flight together,
// summed in corner order
__device__ __forceinline__ void gather_pos(const PosGather &G, int blk, int oimg) {
    const int v = blk * blockDim.x + threadIdx.x;
    if (v >= G.V) return;
    const int i0 = G.inc_off[v], i1 = G.inc_off[v + 1];
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    const int ia = G.pos_batched ? oimg : 0, ib = G.pos_batched ? oimg + 1 : G.n_img;
    for (int img = ia; img < ib; ++img) {
        const float4 *P = G.partial + (long long)img * G.F * 3;
        const unsigned char *live = G.live + (long long)img * G.F;
        for (int i = i0; i < i1; i += 8) {
            float4 q[8];
            int c[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) c[k] = i + k < i1 ? G.inc[i + k] : -1;
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (c[k] >= 0 && !live[(unsigned)c[k] / 3u]) c[k] = -1;
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (c[k] >= 0) q[k] = P[c[k]];
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (c[k] >= 0) { s.x += q[k].x; s.y += q[k].y; s.z += q[k].z; s.w += q[k].w; }
        }
    }
    put(G.grad_pos + (long long)oimg * G.V + v, s, G.set);
}

// Neighbouring vertices, whose corners' rows share cache lines, on one XCD.
// (Grid: blocks, outputs, further blocks.)
__global__ void __launch_bounds__(256) k_gather_attr_q(AttrGather A) {
    gather_attr_q(A, xcd_deal(blockIdx.x + gridDim.x * blockIdx.z, A.xcd), blockIdx.y);
}
__global__ void __launch_bounds__(256) k_gather_attr_c(AttrGather A) {
    gather_attr_c(A, xcd_deal(blockIdx.x + gridDim.x * blockIdx.z, A.xcd), blockIdx.y);
}
__global__ void __launch_bounds__(256) k_gather_pos(PosGather G) {
    gather_pos(G, xcd_deal(blockIdx.x, G.xcd), blockIdx.y);
}

// Both gathers for one image of a large mesh: a thread per vertex reads its
// corners and their triangles' bytes once for the position and all NQ quads, and
// leaves a vertex without a live corner alone.  With a lane per quad those reads
// are most of the work: 262 -> 149 us for 2.6M vertices of 16 channels.  Below
// kVertexThreads vertices the lanes are needed to fill the GPU.
constexpr int kVertexThreads = 1 << 18;
template <int NQ>
__global__ void __launch_bounds__(256) k_gather_vertex(AttrGather A, PosGather G) {
    const int v = xcd_deal(blockIdx.x, G.xcd) * (int)blockDim.x + (int)threadIdx.x;
    if (v >= G.V) return;
    const int i0 = G.inc_off[v], i1 = G.inc_off[v + 1];
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f), acc[NQ];
    bool any = false;
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[q] = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int i = i0; i < i1; i += 8) {
        int c[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) c[k] = i + k < i1 ? G.inc[i + k] : -1;
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (c[k] >= 0 && !G.live[(unsigned)c[k] / 3u]) c[k] = -1;
        float4 x[8];
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (c[k] >= 0) {
                x[k] = G.partial[c[k]];
                any = true;
            }
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (c[k] >= 0) { s.x += x[k].x; s.y += x[k].y; s.z += x[k].z; s.w += x[k].w; }
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (c[k] >= 0) x[k] = reinterpret_cast<const float4 *>(A.partial)[(long long)c[k] * NQ + q];
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (c[k] >= 0) {
                    acc[q].x += x[k].x; acc[q].y += x[k].y; acc[q].z += x[k].z; acc[q].w += x[k].w;
                }
        }
    }
    if (!any) return;
    put(G.grad_pos + v, s, 0);
    float *ga = A.grad_attr + (long long)v * (4 * NQ);
#pragma unroll
    for (int q = 0; q < NQ; ++q) put(ga + 4 * q, acc[q], 0);
}

template <typename T>
__global__ void __launch_bounds__(256) k_zero(T *p, long long n) {
    const long long i = ((long long)blockIdx.x * 4) * blockDim.x + threadIdx.x;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (i + k * 256 < n) p[i + k * 256] = T{};
}
// n floats, a multiple of 4
static void zero_floats(float *p, long long n, hipStream_t st) {
    if (((uintptr_t)p & 15) == 0)
        hipLaunchKernelGGL(k_zero<float4>, dim3((unsigned)((n / 4 + 1023) / 1024)), dim3(256), 0, st, (float4 *)p, n / 4);
    else
        hipLaunchKernelGGL(k_zero<float>, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, st, p, n);
}

// Both gathers of the fused backward (one attribute output), the first
// `attr_blocks` blocks for the attributes.  They are independent and each too
// small to fill the GPU on an ordinary mesh; as two launches they needed a second
// stream and four event calls (some 15 us of host time) to overlap.
template <bool QUADS>
__global__ void __launch_bounds__(256) k_gather_both(AttrGather A, PosGather G, int attr_blocks, int pos_blocks) {
    const int blk = blockIdx.x;
    if (blk < attr_blocks) {
        if (QUADS) gather_attr_q(A, xcd_deal(blk, A.xcd), 0);
        else gather_attr_c(A, xcd_deal(blk, A.xcd), 0);
        return;
    }
    const int p = blk - attr_blocks, img = p / pos_blocks;
    gather_pos(G, xcd_deal(p - img * pos_blocks, G.xcd), img);
}

// n_img: images the gathered partials come from (1: an uneven batch)
static AttrGather attr_gather(const float *partial, const unsigned char *live, int groups, int F, int V, int C,
                              int ldc, int c0, int per_output, const int *inc_off, const int *inc, float *grad_attr,
                              int n_img, unsigned &blocks) {
    const int per_out = per_output ? 1 : groups;
    const int lanes = per_out >= kAttrLanes ? kAttrLanes : (per_out >= 2 ? 2 : 1);
    const long long n = ((C % 4 == 0 ? (long long)V * (C / 4) * lanes : (long long)V * C) + 255) / 256;
    const int xcd = xcd_group(n, n_img, kXcdVerts);
    blocks = (unsigned)xcd_pad(n, xcd);
    return {partial, live, groups, F, V, C, ldc, c0, per_output, lanes, xcd, inc_off, inc, grad_attr, 0};
}
static PosGather pos_gather(const float *partial, const unsigned char *live, int n_img, int F, int V, int pos_batched,
                            const int *inc_off, const int *inc, float *grad_pos, unsigned &blocks) {
    const long long n = (V + 255ll) / 256;
    const int xcd = xcd_group(n, n_img, kXcdVerts);
    blocks = (unsigned)xcd_pad(n, xcd);
    return {(const float4 *)partial, live, n_img, F, V, pos_batched, xcd, inc_off, inc, (float4 *)grad_pos, 0};
}

static void launch_attr(const AttrGather &A, unsigned blocks, int outs, hipStream_t st) {
    const unsigned x = blocks < kMaxBlocks ? blocks : (unsigned)kMaxBlocks;
    const dim3 grid(x, outs, (blocks + x - 1) / x);
    if (A.nc % 4 == 0) hipLaunchKernelGGL(k_gather_attr_q, grid, dim3(256), 0, st, A);
    else hipLaunchKernelGGL(k_gather_attr_c, grid, dim3(256), 0, st, A);
}

int launch_gather_attr(const float *partial, const unsigned char *live, int groups, int F, int V, int C, int ldc,
                       int c0, int outs, int per_output, const int *inc_off, const int *inc, float *grad_attr,
                       hipStream_t st) {
    if (V == 0) return 0;
    unsigned blocks;
    const AttrGather A = attr_gather(partial, live, groups, F, V, C, ldc, c0, per_output, inc_off, inc, grad_attr, groups, blocks);
    launch_attr(A, blocks, outs, st);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_gather_pos(const float *partial, const unsigned char *live, int n_img, int F, int V, int pos_batched,
                      const int *inc_off, const int *inc, float *grad_pos, hipStream_t st) {
    if (V == 0) return 0;
    unsigned blocks;
    const PosGather G = pos_gather(partial, live, n_img, F, V, pos_batched, inc_off, inc, grad_pos, blocks);
    hipLaunchKernelGGL(k_gather_pos, dim3(blocks, pos_batched ? n_img : 1), dim3(256), 0, st, G);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_gather_both(const TriBwdLaunch &T, int C, const int *inc_off, const int *inc, float *grad_attr,
                       float *grad_pos, int set_attr, int set_pos, hipStream_t st) {
    if (T.V == 0) return 0;
    const int groups = (T.n_img + T.views_per_block - 1) / T.views_per_block;
    unsigned na, np;
    AttrGather A = attr_gather(T.partial, T.live, groups, T.F, T.V, C, C, 0, 0, inc_off, inc, grad_attr, T.n_img, na);
    PosGather G = pos_gather(T.partial_pos, T.live_pos, T.n_img, T.F, T.V, T.b.pos_batched, inc_off, inc, grad_pos, np);
    A.set = set_attr;
    G.set = set_pos;
    if (C % 4 == 0 && T.n_img == 1 && T.V >= kVertexThreads) {
        // (zeros first: writing the dead vertices' from the gather took 0.1 ms more at 2.6M vertices)
        if (set_attr) zero_floats(grad_attr, (long long)T.V * C, st);
        if (set_pos) zero_floats(grad_pos, (long long)T.V * 4, st);
        const dim3 grid(np);
        switch (C / 4) {
            case 1: hipLaunchKernelGGL((k_gather_vertex<1>), grid, dim3(256), 0, st, A, G); break;
            case 2: hipLaunchKernelGGL((k_gather_vertex<2>), grid, dim3(256), 0, st, A, G); break;
            case 3: hipLaunchKernelGGL((k_gather_vertex<3>), grid, dim3(256), 0, st, A, G); break;
            default: hipLaunchKernelGGL((k_gather_vertex<4>), grid, dim3(256), 0, st, A, G); break;
        }
        return hipGetLastError() == hipSuccess ? 0 : -2;
    }
    const unsigned long long blocks = na + (unsigned long long)np * (T.b.pos_batched ? T.n_img : 1);
    if (blocks >= (unsigned long long)kMaxBlocks) {  // past one launch's blocks
        launch_attr(A, na, 1, st);
        hipLaunchKernelGGL(k_gather_pos, dim3(np, T.b.pos_batched ? T.n_img : 1), dim3(256), 0, st, G);
        return hipGetLastError() == hipSuccess ? 0 : -2;
    }
    const dim3 grid((unsigned)blocks);
    if (C % 4 == 0) hipLaunchKernelGGL((k_gather_both<true>), grid, dim3(256), 0, st, A, G, (int)na, (int)np);
    else hipLaunchKernelGGL((k_gather_both<false>), grid, dim3(256), 0, st, A, G, (int)na, (int)np);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace drp
