// Per-vertex sums of the tile backward's per-corner partials: attributes,
// positions, and both in one launch, with the tables they read.
#include "drp_common.h"
#include "drp_kernels.h"

namespace drp {

struct AttrGather {
    const float *partial;  // [groups, F, 3, nc]
    int groups, F, V, nc;
    int ldc, c0;           // channels of grad_attr's rows, first channel of this pass
    int per_output;        // one group per output (else every group sums into output 0)
    int lanes;
    const int *inc_off, *inc;
    float *grad_attr;
};
struct PosGather {
    const float4 *partial;  // [n_img, 3 F], a vertex's corners adjacent
    int n_img, F, V, pos_batched;
    const int *inc_off;
    float4 *grad_pos;
};

constexpr int kAttrLanes = 4;

// grad_attr[out][v][c0 ..) += sum over groups g in the output's range and
// incident corners, channel counts that are whole quads, with `lanes` lanes per
// (vertex, four channels) (1, 2 or 4: up to the groups each output sums): lane
// s takes groups s, s + lanes, ... (two groups' corner rows in flight together,
// each group's corners summed in order), and the lanes' sums are added in a
// fixed tree.  (One lane per (vertex, quad) left the 64-view grid at barely one
// wave per SIMD waiting on its loads.)
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
        for (int g = g0 + s; g < g1; g += 2 * lanes) {
            float4 x[2][8];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int gh = g + h * lanes;
                const float *P = partial + (long long)gh * gstride + 4 * q;
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    if (gh < g1 && k < deg) x[h][k] = *reinterpret_cast<const float4 *>(P + (long long)c[k] * NC);
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    if (g + h * lanes < g1 && k < deg) {
                        acc.x += x[h][k].x; acc.y += x[h][k].y; acc.z += x[h][k].z; acc.w += x[h][k].w;
                    }
        }
    } else {
        for (int g = g0 + s; g < g1; g += lanes) {
            const float *P = partial + (long long)g * gstride + 4 * q;
            for (int i = i0; i < i1; i += 4) {  // four corners' loads in flight, summed in corner order
                float4 x[4];
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (i + k < i1) x[k] = *reinterpret_cast<const float4 *>(P + (long long)inc[i + k] * NC);
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (i + k < i1) {
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
    o[0] += acc.x;
    o[1] += acc.y;
    o[2] += acc.z;
    o[3] += acc.w;
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
        for (int i = i0; i < i1; i += 4) {
            float x[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) x[k] = i + k < i1 ? P[(long long)inc[i + k] * NC] : 0.f;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (i + k < i1) s += x[k];
        }
    }
    A.grad_attr[((long long)out * V + v) * A.ldc + A.c0 + ch] += s;
}

// vertex gather: grad_pos[img][v] += sum over incident corners of partial[pimg][t][corner]
// (pos_batched: one output per image; else all images sum into one buffer).
// The corners of a block's 256 vertices are one contiguous range of each
// image's partials (CSR order): it is staged in LDS with coalesced loads
// when it fits, and each vertex then sums its slice from there, in corner
// order as the direct loads do.
constexpr int kGatherPosLds = 2048;  // float4 per block (32 KiB)
__device__ __forceinline__ void gather_pos(const PosGather &G, int blk, int oimg, float4 *buf) {
    const float4 *__restrict__ partial = G.partial;
    const int *__restrict__ inc_off = G.inc_off;
    const int n_img = G.n_img, F = G.F, V = G.V, pos_batched = G.pos_batched;
    const int vb = blk * blockDim.x, v = vb + threadIdx.x;
    const int b0 = inc_off[vb], b1 = inc_off[min(vb + (int)blockDim.x, V)];  // (vb < V: the grid covers V)
    const bool staged = b1 - b0 <= kGatherPosLds;  // uniform per block
    const int i0 = v < V ? inc_off[v] : b0, i1 = v < V ? inc_off[v + 1] : b0;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    const int ia = pos_batched ? oimg : 0, ib = pos_batched ? oimg + 1 : n_img;
    for (int img = ia; img < ib; ++img) {
        const float4 *P = partial + (long long)img * F * 3;  // this vertex's corners are P[i0 .. i1)
        if (staged) {
            if (img > ia) __syncthreads();  // the previous image's sums have read the buffer
            for (int i = b0 + (int)threadIdx.x; i < b1; i += blockDim.x) buf[i - b0] = P[i];
            __syncthreads();
            for (int i = i0; i < i1; ++i) {
                const float4 q = buf[i - b0];
                s.x += q.x; s.y += q.y; s.z += q.z; s.w += q.w;
            }
            continue;
        }
        // eight corners' loads in flight at once, summed in corner order
        for (int i = i0; i < i1; i += 8) {
            float4 q[8];
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (i + k < i1) q[k] = P[i + k];
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (i + k < i1) { s.x += q[k].x; s.y += q[k].y; s.z += q[k].z; s.w += q[k].w; }
        }
    }
    if (v >= V) return;
    float4 *o = G.grad_pos + (long long)oimg * V + v;
    float4 cur = *o;
    *o = make_float4(cur.x + s.x, cur.y + s.y, cur.z + s.z, cur.w + s.w);
}

__global__ void __launch_bounds__(256) k_gather_attr_q(AttrGather A) { gather_attr_q(A, blockIdx.x, blockIdx.y); }
__global__ void __launch_bounds__(256) k_gather_attr_c(AttrGather A) { gather_attr_c(A, blockIdx.x, blockIdx.y); }
__global__ void __launch_bounds__(256) k_gather_pos(PosGather G) {
    __shared__ float4 buf[kGatherPosLds];
    gather_pos(G, blockIdx.x, blockIdx.y, buf);
}

// Both gathers of the fused backward (one attribute output), the first
// `attr_blocks` blocks for the attributes.  They are independent and each too
// small to fill the GPU on an ordinary mesh; as two launches they needed a second
// stream and four event calls (some 15 us of host time) to overlap.
template <bool QUADS>
__global__ void __launch_bounds__(256) k_gather_both(AttrGather A, PosGather G, int attr_blocks, int pos_blocks) {
    __shared__ float4 buf[kGatherPosLds];
    const int blk = blockIdx.x;
    if (blk < attr_blocks) {
        if (QUADS) gather_attr_q(A, blk, 0);
        else gather_attr_c(A, blk, 0);
        return;
    }
    const int p = blk - attr_blocks;
    gather_pos(G, p % pos_blocks, p / pos_blocks, buf);
}

// slot[c] = position of corner c in the incidence list (the list's inverse),
// -1 for corners whose vertex index is outside [0, V): those are not listed
__global__ void k_corner_slots(const int *__restrict__ tri, const int *__restrict__ inc,
                               const int *__restrict__ inc_off, int V, long long n, int *__restrict__ slot) {
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if ((unsigned)tri[i] >= (unsigned)V) slot[i] = -1;
    if (i < inc_off[V]) slot[inc[i]] = (int)i;
}

int launch_corner_slots(const int *tri, const int *inc, const int *inc_off, int V, int F, int *slot, hipStream_t st) {
    const long long nc = 3ll * F;
    if (nc == 0) return 0;
    hipLaunchKernelGGL(k_corner_slots, dim3((unsigned)((nc + 255) / 256)), dim3(256), 0, st, tri, inc, inc_off, V, nc,
                       slot);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

static AttrGather attr_gather(const float *partial, int groups, int F, int V, int C, int ldc, int c0, int per_output,
                              const int *inc_off, const int *inc, float *grad_attr) {
    const int per_out = per_output ? 1 : groups;
    const int lanes = per_out >= kAttrLanes ? kAttrLanes : (per_out >= 2 ? 2 : 1);
    return {partial, groups, F, V, C, ldc, c0, per_output, lanes, inc_off, inc, grad_attr};
}
static unsigned attr_blocks(const AttrGather &A) {
    const long long n = A.nc % 4 == 0 ? (long long)A.V * (A.nc / 4) * A.lanes : (long long)A.V * A.nc;
    return (unsigned)((n + 255) / 256);
}

int launch_gather_attr(const float *partial, int groups, int F, int V, int C, int ldc, int c0, int outs,
                       int per_output, const int *inc_off, const int *inc, float *grad_attr, hipStream_t st) {
    if (V == 0) return 0;
    const AttrGather A = attr_gather(partial, groups, F, V, C, ldc, c0, per_output, inc_off, inc, grad_attr);
    const dim3 grid(attr_blocks(A), outs);
    if (C % 4 == 0) hipLaunchKernelGGL(k_gather_attr_q, grid, dim3(256), 0, st, A);
    else hipLaunchKernelGGL(k_gather_attr_c, grid, dim3(256), 0, st, A);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_gather_pos(const float *partial, int n_img, int F, int V, int pos_batched, const int *inc_off,
                      float *grad_pos, hipStream_t st) {
    if (V == 0) return 0;
    const PosGather G{(const float4 *)partial, n_img, F, V, pos_batched, inc_off, (float4 *)grad_pos};
    hipLaunchKernelGGL(k_gather_pos, dim3((V + 255) / 256, pos_batched ? n_img : 1), dim3(256), 0, st, G);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_gather_both(const float *partial_attr, int groups, int C, const float *partial_pos, int n_img,
                       int pos_batched, int F, int V, const int *inc_off, const int *inc, float *grad_attr,
                       float *grad_pos, hipStream_t st) {
    if (V == 0) return 0;
    const AttrGather A = attr_gather(partial_attr, groups, F, V, C, C, 0, 0, inc_off, inc, grad_attr);
    const PosGather G{(const float4 *)partial_pos, n_img, F, V, pos_batched, inc_off, (float4 *)grad_pos};
    const unsigned na = attr_blocks(A), np = (unsigned)((V + 255) / 256);
    const unsigned long long blocks = na + (unsigned long long)np * (pos_batched ? n_img : 1);
    if (blocks >= (1ull << 31)) {  // past one launch's blocks
        if (int rc = launch_gather_attr(partial_attr, groups, F, V, C, C, 0, 1, 0, inc_off, inc, grad_attr, st)) return rc;
        return launch_gather_pos(partial_pos, n_img, F, V, pos_batched, inc_off, grad_pos, st);
    }
    if (C % 4 == 0) hipLaunchKernelGGL((k_gather_both<true>), dim3((unsigned)blocks), dim3(256), 0, st, A, G, (int)na, (int)np);
    else hipLaunchKernelGGL((k_gather_both<false>), dim3((unsigned)blocks), dim3(256), 0, st, A, G, (int)na, (int)np);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace drp
