// Texture sampling for the shading stage after interpolation: diffrp's
// sample2d / sample3d (diffrp/utils/shader_ops.py:198-310), used by
// GLTFSampler (diffrp/materials/gltf_material.py:15-22) and image-based
// lighting, which call torch's grid_sample on a permuted (C, H, W) view.
// Here the texture stays channels-last ([H, W, C] / [D, H, W, C]): a tap is
// C contiguous floats.  The coordinate mapping is diffrp's: uv (0, 0) is the
// bottom-left texel corner (last row), x = 2u - 1, y = 1 - 2v (z = 2w - 1), and
// grid_sample's unnormalisation, border / reflection padding and
// align_corners (latlong) rules; "cyclic" samples the 2 x 2 tiled texture at
// (uv mod 1) / 2 shifted into [1/4, 3/4) with reflection padding, as diffrp
// does.  Forward: one thread per sample.  Backward: the texture gradient is
// scattered with float atomics (as grid_sample's backward; 2-D textures sum a
// block's samples first), the coordinate gradient is written per sample.
#include "drp_common.h"
#include "drp_kernels.h"

namespace drp {

enum : int { kWrapBorder = 0, kWrapReflection = 1, kWrapCyclic = 2, kWrapLatlong = 3 };
enum : int { kModeBilinear = 0, kModeNearest = 1, kModeBicubic = 2 };

// grid_sample's source index for one axis with its derivative d(index)/d(grid)
__device__ __forceinline__ float pad_coord(float x, int size, bool align, bool reflect, float &dg);

__device__ __forceinline__ float source_index(float g, int size, bool align, bool reflect, bool raw, float &dg) {
    float x;
    if (align) {
        x = (g + 1.f) * 0.5f * (float)(size - 1);
        dg = (float)(size - 1) * 0.5f;
    } else {
        x = ((g + 1.f) * (float)size - 1.f) * 0.5f;
        dg = (float)size * 0.5f;
    }
    return raw ? x : pad_coord(x, size, align, reflect, dg);  // bicubic pads each tap instead
}

// border / reflection padding of a source coordinate, with its derivative factor
__device__ __forceinline__ float pad_coord(float x, int size, bool align, bool reflect, float &dg) {
    if (reflect) {
        const float lo = align ? 0.f : -0.5f;  // reflection interval [lo, lo + span]
        const float span = align ? (float)(size - 1) : (float)size;
        if (span <= 0.f) {
            x = 0.f;
            dg = 0.f;
        } else {
            float in = x - lo;
            if (in < 0.f) {
                in = -in;
                dg = -dg;
            }
            const float extra = fmodf(in, span);
            const int flips = (int)floorf(in / span);
            if (flips % 2 == 0) {
                x = extra + lo;
            } else {
                x = span - extra + lo;
                dg = -dg;
            }
        }
    }
    // clip to [0, size - 1] (border padding, and after a reflection)
    if (x <= 0.f) {
        x = 0.f;
        dg = 0.f;
    } else if (x >= (float)(size - 1)) {
        x = (float)(size - 1);
        dg = 0.f;
    }
    return x;
}

struct TexAxis {
    float pos;    // source index
    float dpos;   // d pos / d (texture coordinate)
    int size;     // sampled size (2x for cyclic)
    int period;   // texel period (the texture's size)
};

// texture coordinate -> source index of one axis; flip: y axis (1 - 2v)
__device__ __forceinline__ TexAxis make_axis(float u, int size, int wrap, bool flip, bool raw = false) {
    TexAxis a;
    a.period = size;
    float du = 1.f;
    if (wrap == kWrapCyclic) {
        float m = u - floorf(u);  // remainder(u, 1), derivative 1
        m *= 0.5f;
        if (!(m >= 0.25f)) m += 0.5f;
        u = m;
        du = 0.5f;
        size *= 2;
    }
    float g = flip ? -(u * 2.f - 1.f) : (u * 2.f - 1.f);
    float dg;
    const bool align = wrap == kWrapLatlong;
    const bool reflect = wrap != kWrapBorder;
    a.pos = source_index(g, size, align, reflect, raw, dg);
    a.size = size;
    a.dpos = dg * (flip ? -2.f : 2.f) * du;
    return a;
}

__device__ __forceinline__ int texel(const TexAxis &a, int i) { return a.size == a.period ? i : i % a.period; }

// bicubic (Keys, A = -0.75, as grid_sample): weights of the taps x0 - 1 .. x0 + 2 at
// fraction t, the weights' derivatives with respect to -t, and each tap's padded texel
__device__ __forceinline__ void cubic_weights(float t, float w[4], float dw[4]) {
    const float A = -0.75f;
    float x = t + 1.f;
    w[0] = ((A * x - 5.f * A) * x + 8.f * A) * x - 4.f * A;
    x = t;
    w[1] = ((A + 2.f) * x - (A + 3.f)) * x * x + 1.f;
    x = 1.f - t;
    w[2] = ((A + 2.f) * x - (A + 3.f)) * x * x + 1.f;
    x = 2.f - t;
    w[3] = ((A * x - 5.f * A) * x + 8.f * A) * x - 4.f * A;
    x = -1.f - t;
    dw[0] = (-3.f * A * x - 10.f * A) * x - 8.f * A;
    x = -t;
    dw[1] = (-3.f * (A + 2.f) * x - 2.f * (A + 3.f)) * x;
    x = 1.f - t;
    dw[2] = (3.f * (A + 2.f) * x - 2.f * (A + 3.f)) * x;
    x = 2.f - t;
    dw[3] = (3.f * A * x - 10.f * A) * x + 8.f * A;
}

__device__ __forceinline__ int cubic_tap(const TexAxis &a, int i, int wrap) {
    float dg = 0.f;
    const float x = pad_coord((float)i, a.size, wrap == kWrapLatlong, wrap != kWrapBorder, dg);
    return texel(a, (int)x);
}

template <int CV>
__global__ void __launch_bounds__(256) k_sample2d_fwd(const float *__restrict__ tex, int H, int W, int C,
                                                      const float *__restrict__ uv, long long n, int wrap, int mode,
                                                      float *__restrict__ out) {
    const int Cn = CV > 0 ? CV : C;
    // (neighbouring samples share texels: runs of blocks on one XCD)
    long long i = (long long)xcd_deal(blockIdx.x, kXcdPixels) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const bool raw = mode == kModeBicubic;
    const TexAxis ax = make_axis(uv[2 * i], W, wrap, false, raw), ay = make_axis(uv[2 * i + 1], H, wrap, true, raw);
    float *o = out + i * Cn;
    if (mode == kModeBicubic) {
        const float fx0 = floorf(ax.pos), fy0 = floorf(ay.pos);
        float wx[4], wy[4], dwx[4], dwy[4];
        cubic_weights(ax.pos - fx0, wx, dwx);
        cubic_weights(ay.pos - fy0, wy, dwy);
        int tx[4], ty[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            tx[k] = cubic_tap(ax, (int)fx0 - 1 + k, wrap);
            ty[k] = cubic_tap(ay, (int)fy0 - 1 + k, wrap);
        }
        for (int c = 0; c < Cn; ++c) {
            float rows[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float *row = tex + (long long)ty[k] * W * Cn + c;
                rows[k] = row[tx[0] * Cn] * wx[0] + row[tx[1] * Cn] * wx[1] + row[tx[2] * Cn] * wx[2] +
                          row[tx[3] * Cn] * wx[3];
            }
            o[c] = rows[0] * wy[0] + rows[1] * wy[1] + rows[2] * wy[2] + rows[3] * wy[3];
        }
        return;
    }
    if (mode == kModeNearest) {
        const int x = (int)rintf(ax.pos), y = (int)rintf(ay.pos);
        const bool in = x >= 0 && x < ax.size && y >= 0 && y < ay.size;
        const float *t = tex + ((long long)texel(ay, in ? y : 0) * W + texel(ax, in ? x : 0)) * Cn;
        for (int c = 0; c < Cn; ++c) o[c] = in ? t[c] : 0.f;
        return;
    }
    const int x0 = (int)floorf(ax.pos), y0 = (int)floorf(ay.pos);
    const float fx = ax.pos - (float)x0, fy = ay.pos - (float)y0;
    const float w[4] = {(1.f - fx) * (1.f - fy), fx * (1.f - fy), (1.f - fx) * fy, fx * fy};
    long long off[4];
    bool in[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int x = x0 + (k & 1), y = y0 + (k >> 1);
        in[k] = x >= 0 && x < ax.size && y >= 0 && y < ay.size;
        off[k] = in[k] ? ((long long)texel(ay, y) * W + texel(ax, x)) * Cn : 0;
    }
    if (CV > 0) {  // the four texels' loads in flight together (outside: texel 0, not used)
        float t[4][CV > 0 ? CV : 1];
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int c = 0; c < CV; ++c) t[k][c] = tex[off[k] + c];
#pragma unroll
        for (int c = 0; c < CV; ++c) {
            float s = 0.f;
#pragma unroll
            for (int k = 0; k < 4; ++k) s = in[k] ? s + t[k][c] * w[k] : s;
            o[c] = s;
        }
        return;
    }
    for (int c = 0; c < Cn; ++c) {
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (in[k]) s += tex[off[k] + c] * w[k];
        o[c] = s;
    }
}

// Texture gradients of one block's samples (16 x 16 of an image's samples
// where the caller names its row width, else 256 in a row).  Device-scope
// float atomics are performed beyond the per-XCD L2s, one at a time per
// address: samples that share texels (magnified textures, and every background
// pixel sampling the corner texel) queue up on them.  So a block first takes
// the box of the texels that its non-zero gradients touch:
//   - box of at most kTexTile floats: summed in an LDS copy of the box, then
//     one atomic per non-zero float, consecutive lanes on consecutive floats;
//   - larger (a seam, a minified texture): per tap, runs of lanes on one texel
//     are summed across the wave, one atomic per run and channel.
// Zero contributions (masked background) are never sent.  Four 768^2 views of
// a sphere with a 1024^2 x 3 texture, the background masked: 44.8 ms with one
// atomic per tap and channel, 0.151 ms so.  What remains is the LDS atomics
// (12 per covered sample) and the scattered texel reads of the coordinate
// gradient.
constexpr int kTexTile = 4096;  // floats (16 KiB and the box: the eight blocks that a CU's wave slots hold fit its LDS)

struct TexGrad {
    float *tile;        // LDS box, or nullptr
    float *gtex;
    int x0, y0, bw;     // box origin and width in texels
    int W, C;
};

// one tap of every lane of the wave (wave-uniform call): texel (x, y), x < 0:
// none; g[0 .. C) scaled by w
__device__ __forceinline__ void tex_tap(const TexGrad &T, int x, int y, float w, const float *g) {
    if (T.tile) {
        if (x < 0) return;
        float *t = T.tile + ((y - T.y0) * T.bw + (x - T.x0)) * T.C;
        for (int c = 0; c < T.C; ++c) {
            const float v = w * g[c];
            if (v != 0.f) atomicAdd(t + c, v);
        }
        return;
    }
    const int lane = threadIdx.x & 63;
    const long long at = x < 0 ? -1ll : (long long)y * T.W + x;
    const long long before = __shfl_up(at, 1, 64);
    const unsigned long long heads = __ballot(lane == 0 || before != at);
    const unsigned long long after = lane == 63 ? 0ull : heads >> (lane + 1);
    const int end = after ? lane + __ffsll(after) : 64;  // first lane past this lane's run
    const bool head = (heads >> lane) & 1;
    for (int c = 0; c < T.C; ++c) {
        float v = x < 0 ? 0.f : w * g[c];
        if (heads != ~0ull)  // uniform: some texel is shared
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const float n = __shfl_down(v, o, 64);
                if (lane + o < end) v += n;
            }
        if (head && x >= 0 && v != 0.f) atomicAdd(T.gtex + at * T.C + c, v);
    }
}

// a sample's taps along one axis: texel (-1: outside), weight, and the
// weight's derivative with respect to the source index
constexpr int axis_tap_count(int mode) { return mode == kModeBicubic ? 4 : (mode == kModeNearest ? 1 : 2); }
template <int MODE>
struct AxisTaps {
    static constexpr int N = axis_tap_count(MODE);
    int at[N];
    float w[N], dw[N];
};
template <int MODE>
__device__ __forceinline__ AxisTaps<MODE> axis_taps(const TexAxis &a, int wrap) {
    AxisTaps<MODE> t;
#pragma unroll
    for (int k = 0; k < t.N; ++k) {
        t.at[k] = -1;
        t.w[k] = t.dw[k] = 0.f;
    }
    if constexpr (MODE == kModeBicubic) {
        const float f0 = floorf(a.pos);
        cubic_weights(a.pos - f0, t.w, t.dw);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            t.at[k] = cubic_tap(a, (int)f0 - 1 + k, wrap);
            t.dw[k] = -t.dw[k];  // cubic_weights gives -d w / d t
        }
    } else if constexpr (MODE == kModeNearest) {
        const int x = (int)rintf(a.pos);
        if (x >= 0 && x < a.size) t.at[0] = texel(a, x);
        t.w[0] = 1.f;
    } else {
        const int x = (int)floorf(a.pos);
        const float f = a.pos - (float)x;
        t.w[0] = 1.f - f;
        t.w[1] = f;
        t.dw[0] = -1.f;
        t.dw[1] = 1.f;
        if (x >= 0 && x < a.size) t.at[0] = texel(a, x);
        if (x + 1 >= 0 && x + 1 < a.size) t.at[1] = texel(a, x + 1);
    }
    return t;
}

template <int CV, int MODE>
__global__ void __launch_bounds__(256) k_sample2d_bwd(const float *__restrict__ tex, int H, int W, int C,
                                                      const float *__restrict__ uv, long long n, int width, int wrap,
                                                      const float *__restrict__ gout,
                                                      float *__restrict__ gtex, float *__restrict__ guv) {
    __shared__ float tile[kTexTile];
    __shared__ int box[4];  // min x, min y, max x, max y
    const int Cn = CV > 0 ? CV : C;
    const int tid = threadIdx.x;
    const long long blk = xcd_deal(blockIdx.x, kXcdPixels);  // neighbouring samples share texels
    long long i = blk * blockDim.x + tid;
    bool live = i < n;
    if (width > 0) {  // 16 x 16 samples of an image (rows of all images counted on)
        const int tiles_x = (width + 15) / 16;
        const long long ty = blk / tiles_x;
        const int col = (int)(blk - ty * tiles_x) * 16 + (tid & 15);
        i = (ty * 16 + (tid >> 4)) * width + col;
        live = col < width && i < n;
    }
    const long long il = live ? i : 0;
    const TexAxis ax = make_axis(uv[2 * il], W, wrap, false, MODE == kModeBicubic),
                  ay = make_axis(uv[2 * il + 1], H, wrap, true, MODE == kModeBicubic);
    const AxisTaps<MODE> tx = axis_taps<MODE>(ax, wrap), ty = axis_taps<MODE>(ay, wrap);
    const float *g = gout + il * Cn;
    if (guv && live) {
        float gx = 0.f, gy = 0.f;
        if (MODE == kModeBilinear && CV > 0) {  // the texels' and gradients' loads in flight together
            float t[ty.N * tx.N][CV > 0 ? CV : 1], gr[CV > 0 ? CV : 1];
#pragma unroll
            for (int k = 0; k < ty.N * tx.N; ++k)
#pragma unroll
                for (int c = 0; c < CV; ++c)
                    t[k][c] = tex[((long long)max(ty.at[k / tx.N], 0) * W + max(tx.at[k % tx.N], 0)) * Cn + c];
#pragma unroll
            for (int c = 0; c < CV; ++c) gr[c] = g[c];
#pragma unroll
            for (int k = 0; k < ty.N * tx.N; ++k) {
                const int a = k / tx.N, b = k % tx.N;
                if (ty.at[a] < 0 || tx.at[b] < 0) continue;
                float dot = 0.f;
#pragma unroll
                for (int c = 0; c < CV; ++c) dot += t[k][c] * gr[c];
                gx += tx.dw[b] * ty.w[a] * dot;
                gy += tx.w[b] * ty.dw[a] * dot;
            }
        } else if (MODE != kModeNearest) {
#pragma unroll
            for (int a = 0; a < ty.N; ++a)
#pragma unroll
                for (int b = 0; b < tx.N; ++b) {
                    if (ty.at[a] < 0 || tx.at[b] < 0) continue;
                    const float *t = tex + ((long long)ty.at[a] * W + tx.at[b]) * Cn;
                    float dot = 0.f;
                    for (int c = 0; c < Cn; ++c) dot += t[c] * g[c];
                    gx += tx.dw[b] * ty.w[a] * dot;
                    gy += tx.w[b] * ty.dw[a] * dot;
                }
        }
        guv[2 * i] = MODE == kModeNearest ? 0.f : gx * ax.dpos;
        guv[2 * i + 1] = MODE == kModeNearest ? 0.f : gy * ay.dpos;
    }
    if (!gtex) return;  // uniform
    bool any = false;
    if (live)
        for (int c = 0; c < Cn; ++c) any = any || g[c] != 0.f;
    // the box of the texels that non-zero gradients touch
    int x0 = W, y0 = H, x1 = -1, y1 = -1;
    if (any) {
#pragma unroll
        for (int k = 0; k < tx.N; ++k) {
            if (tx.at[k] >= 0) { x0 = min(x0, tx.at[k]); x1 = max(x1, tx.at[k]); }
            if (ty.at[k] >= 0) { y0 = min(y0, ty.at[k]); y1 = max(y1, ty.at[k]); }
        }
    }
    if (tid < 4) box[tid] = tid < 2 ? 0x7fffffff : -1;
    __syncthreads();
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        x0 = min(x0, __shfl_xor(x0, o, 64));
        y0 = min(y0, __shfl_xor(y0, o, 64));
        x1 = max(x1, __shfl_xor(x1, o, 64));
        y1 = max(y1, __shfl_xor(y1, o, 64));
    }
    if ((tid & 63) == 0) {
        atomicMin(&box[0], x0);
        atomicMin(&box[1], y0);
        atomicMax(&box[2], x1);
        atomicMax(&box[3], y1);
    }
    __syncthreads();
    const int bx = box[0], by = box[1], bw = box[2] - bx + 1, bh = box[3] - by + 1;  // uniform per block
    if (box[2] < 0 || box[3] < 0) return;  // no gradient, or no tap inside the texture
    const long long area = (long long)bw * bh * Cn;
    const bool local = area <= kTexTile;
    TexGrad T{local ? tile : nullptr, gtex, bx, by, bw, W, Cn};
    if (local) {
        for (int e = tid; e < (int)area; e += 256) tile[e] = 0.f;
        __syncthreads();
    }
#pragma unroll
    for (int a = 0; a < ty.N; ++a)
#pragma unroll
        for (int b = 0; b < tx.N; ++b) {
            const bool in = any && ty.at[a] >= 0 && tx.at[b] >= 0;
            tex_tap(T, in ? tx.at[b] : -1, ty.at[a], ty.w[a] * tx.w[b], g);
        }
    if (local) {
        __syncthreads();
        for (int e = tid; e < (int)area; e += 256) {
            const int row = e / (bw * Cn);
            const float v = tile[e];
            if (v != 0.f) atomicAdd(gtex + ((long long)(by + row) * W + bx) * Cn + (e - row * bw * Cn), v);
        }
    }
}

template <int CV>
__global__ void __launch_bounds__(256) k_sample3d_fwd(const float *__restrict__ tex, int D, int H, int W, int C,
                                                      const float *__restrict__ uvw, long long n, int wrap, int mode,
                                                      float *__restrict__ out) {
    const int Cn = CV > 0 ? CV : C;
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const TexAxis ax = make_axis(uvw[3 * i], W, wrap, false), ay = make_axis(uvw[3 * i + 1], H, wrap, true),
                  az = make_axis(uvw[3 * i + 2], D, wrap, false);
    float *o = out + i * Cn;
    if (mode == kModeNearest) {
        const int x = (int)rintf(ax.pos), y = (int)rintf(ay.pos), z = (int)rintf(az.pos);
        const bool in = x >= 0 && x < W && y >= 0 && y < H && z >= 0 && z < D;
        const float *t = tex + (((long long)(in ? z : 0) * H + (in ? y : 0)) * W + (in ? x : 0)) * Cn;
        for (int c = 0; c < Cn; ++c) o[c] = in ? t[c] : 0.f;
        return;
    }
    const int x0 = (int)floorf(ax.pos), y0 = (int)floorf(ay.pos), z0 = (int)floorf(az.pos);
    const float fx = ax.pos - (float)x0, fy = ay.pos - (float)y0, fz = az.pos - (float)z0;
    for (int c = 0; c < Cn; ++c) o[c] = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int x = x0 + (k & 1), y = y0 + ((k >> 1) & 1), z = z0 + (k >> 2);
        if (!(x >= 0 && x < W && y >= 0 && y < H && z >= 0 && z < D)) continue;
        const float w = ((k & 1) ? fx : 1.f - fx) * (((k >> 1) & 1) ? fy : 1.f - fy) * ((k >> 2) ? fz : 1.f - fz);
        const float *t = tex + (((long long)z * H + y) * W + x) * Cn;
        for (int c = 0; c < Cn; ++c) o[c] += t[c] * w;
    }
}

template <int CV>
__global__ void __launch_bounds__(256) k_sample3d_bwd(const float *__restrict__ tex, int D, int H, int W, int C,
                                                      const float *__restrict__ uvw, long long n, int wrap, int mode,
                                                      const float *__restrict__ gout, float *__restrict__ gtex,
                                                      float *__restrict__ guvw) {
    const int Cn = CV > 0 ? CV : C;
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const TexAxis ax = make_axis(uvw[3 * i], W, wrap, false), ay = make_axis(uvw[3 * i + 1], H, wrap, true),
                  az = make_axis(uvw[3 * i + 2], D, wrap, false);
    const float *g = gout + i * Cn;
    if (mode == kModeNearest) {
        const int x = (int)rintf(ax.pos), y = (int)rintf(ay.pos), z = (int)rintf(az.pos);
        if (gtex && x >= 0 && x < W && y >= 0 && y < H && z >= 0 && z < D) {
            float *t = gtex + (((long long)z * H + y) * W + x) * Cn;
            for (int c = 0; c < Cn; ++c) atomicAdd(t + c, g[c]);
        }
        if (guvw) guvw[3 * i] = guvw[3 * i + 1] = guvw[3 * i + 2] = 0.f;
        return;
    }
    const int x0 = (int)floorf(ax.pos), y0 = (int)floorf(ay.pos), z0 = (int)floorf(az.pos);
    const float fx = ax.pos - (float)x0, fy = ay.pos - (float)y0, fz = az.pos - (float)z0;
    float gx = 0.f, gy = 0.f, gz = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int x = x0 + (k & 1), y = y0 + ((k >> 1) & 1), z = z0 + (k >> 2);
        if (!(x >= 0 && x < W && y >= 0 && y < H && z >= 0 && z < D)) continue;
        const float wxs = (k & 1) ? fx : 1.f - fx, wys = ((k >> 1) & 1) ? fy : 1.f - fy, wzs = (k >> 2) ? fz : 1.f - fz;
        const float dx = (k & 1) ? 1.f : -1.f, dy = ((k >> 1) & 1) ? 1.f : -1.f, dz = (k >> 2) ? 1.f : -1.f;
        const float *t = tex + (((long long)z * H + y) * W + x) * Cn;
        float *gt = gtex ? gtex + (((long long)z * H + y) * W + x) * Cn : nullptr;
        float dot = 0.f;
        for (int c = 0; c < Cn; ++c) {
            dot += t[c] * g[c];
            if (gt) atomicAdd(gt + c, wxs * wys * wzs * g[c]);
        }
        gx += dx * wys * wzs * dot;
        gy += wxs * dy * wzs * dot;
        gz += wxs * wys * dz * dot;
    }
    if (guvw) {
        guvw[3 * i] = gx * ax.dpos;
        guvw[3 * i + 1] = gy * ay.dpos;
        guvw[3 * i + 2] = gz * az.dpos;
    }
}

#define DRP_TEX_DISPATCH(KERNEL, ...)                                                          \
    switch (C) {                                                                               \
        case 1: hipLaunchKernelGGL(KERNEL<1>, grid, dim3(256), 0, st, __VA_ARGS__); break;     \
        case 3: hipLaunchKernelGGL(KERNEL<3>, grid, dim3(256), 0, st, __VA_ARGS__); break;     \
        case 4: hipLaunchKernelGGL(KERNEL<4>, grid, dim3(256), 0, st, __VA_ARGS__); break;     \
        default: hipLaunchKernelGGL(KERNEL<0>, grid, dim3(256), 0, st, __VA_ARGS__); break;    \
    }

#define DRP_TEX_DISPATCH_M(MODE, ...)                                                                    \
    switch (C) {                                                                                         \
        case 1: hipLaunchKernelGGL((k_sample2d_bwd<1, MODE>), grid, dim3(256), 0, st, __VA_ARGS__); break; \
        case 3: hipLaunchKernelGGL((k_sample2d_bwd<3, MODE>), grid, dim3(256), 0, st, __VA_ARGS__); break; \
        case 4: hipLaunchKernelGGL((k_sample2d_bwd<4, MODE>), grid, dim3(256), 0, st, __VA_ARGS__); break; \
        default: hipLaunchKernelGGL((k_sample2d_bwd<0, MODE>), grid, dim3(256), 0, st, __VA_ARGS__); break; \
    }

int launch_sample2d(const float *tex, int H, int W, int C, const float *uv, long long n, int wrap, int mode,
                    float *out, hipStream_t st) {
    const long long most = kMaxBlocks * 256;  // samples of a launch
    for (; n > 0; n -= most, uv += 2 * most, out += (long long)C * most) {
        const long long k = n < most ? n : most;
        dim3 grid((unsigned)xcd_pad((k + 255) / 256, kXcdPixels));
        DRP_TEX_DISPATCH(k_sample2d_fwd, tex, H, W, C, uv, k, wrap, mode, out)
    }
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_sample2d_bwd(const float *tex, int H, int W, int C, const float *uv, long long n, int width, int wrap,
                        int mode, const float *gout, float *gtex, float *guv, hipStream_t st) {
    const long long most = kMaxBlocks * 256;  // samples of a launch
    long long tiles = 0;
    // Narrower rows, or fewer of them (a list of points shaped [1, n, 2]), leave most of a 16 x 16 block idle:
    // 2^20 points along a curve, C = 3, both gradients with torch's share: 243 us as one row of blocks, 134 us so.
    const long long rows = width > 0 ? (n + width - 1) / width : 0;
    if (width >= 16 && rows >= 16) {
        tiles = (long long)((width + 15) / 16) * ((rows + 15) / 16);
        if (tiles > kMaxBlocks) tiles = 0;
    }
    if (!tiles) width = 0;
    for (; n > 0; n -= most, uv += 2 * most, gout += (long long)C * most, guv = guv ? guv + 2 * most : nullptr) {
        const long long k = tiles || n < most ? n : most;
        dim3 grid((unsigned)xcd_pad(tiles ? tiles : (k + 255) / 256, kXcdPixels));
        if (mode == kModeBicubic) DRP_TEX_DISPATCH_M(kModeBicubic, tex, H, W, C, uv, k, width, wrap, gout, gtex, guv)
        else if (mode == kModeNearest) DRP_TEX_DISPATCH_M(kModeNearest, tex, H, W, C, uv, k, width, wrap, gout, gtex, guv)
        else DRP_TEX_DISPATCH_M(kModeBilinear, tex, H, W, C, uv, k, width, wrap, gout, gtex, guv)
    }
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_sample3d(const float *tex, int D, int H, int W, int C, const float *uvw, long long n, int wrap, int mode,
                    float *out, hipStream_t st) {
    if (n == 0) return 0;
    dim3 grid((unsigned)((n + 255) / 256));
    DRP_TEX_DISPATCH(k_sample3d_fwd, tex, D, H, W, C, uvw, n, wrap, mode, out)
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_sample3d_bwd(const float *tex, int D, int H, int W, int C, const float *uvw, long long n, int wrap,
                        int mode, const float *gout, float *gtex, float *guvw, hipStream_t st) {
    if (n == 0) return 0;
    dim3 grid((unsigned)((n + 255) / 256));
    DRP_TEX_DISPATCH(k_sample3d_bwd, tex, D, H, W, C, uvw, n, wrap, mode, gout, gtex, guvw)
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace drp
