// Stencil partition of a layer's pixels by owning object, for the
// stencil-masked G-buffer path (diffrp/rendering/surface_deferred.py:283-290,
// interpolator.py:87-97).  diffrp takes owner = stencils[tri_id] per pixel and
// one mask.nonzero() per object, i.e. one host synchronisation per object and
// layer.  Here one stable partition orders every pixel by owner and, within an
// owner, by pixel -- the order nonzero() gives -- with each owner's [start,
// end); the caller reads starts/ends once per layer.  Beside the pixel list it
// writes what the masked interpolator takes from it: the pixels' fragments and
// their row and column indices, as the owners' consecutive runs.
//
// Few owners (a scene of objects): a counting partition of three launches.  A
// block of kPartPix pixels counts its owners, one block scans the (owner,
// block) counts, and the blocks place their pixels, a wave's 64 pixels per
// owner present in one ballot.  512 x 512 pixels of four owners: 92 us in 19
// launches as a radix sort of (owner, pixel) keys, 25 us so.  Counts past
// kScanMax (thousands of owners on a large layer) would make the one-block scan
// the longest part: those are sorted.
#include <rocprim/device/device_radix_sort.hpp>

#include "drp_common.h"
#include "drp_kernels.h"
#include "drp_wave.h"

namespace drp {

constexpr int kPartWave = 512, kPartPix = 4 * kPartWave;  // pixels of a wave, of a block
constexpr int kPartSteps = kPartWave / 64;
constexpr long long kScanMax = 1 << 16;  // (owner, block) counts
constexpr int kPartOwners = 1024;        // owners (LDS counters per wave)

__device__ __forceinline__ int pixel_owner(const float4 *rast, long long p, const int *stencils, int F, int n_owner) {
    const float w = rast[p].w;
    const int id = w > 0.f ? float_to_triidx(w) : 0;  // triangle + 1, 0: background
    const int o = (id >= 0 && id <= F) ? stencils[id] : 0;
    return o < 0 || o > n_owner ? 0 : o;
}

// own[i]: owner of the wave's pixel i * 64 + lane (-1 past the layer); cnt: the
// wave's pixels per owner
__device__ __forceinline__ void wave_owners(const PartitionLaunch &L, long long p0, int (&own)[kPartSteps], int *cnt) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < kPartSteps; ++i) {
        const long long p = p0 + i * 64 + lane;
        own[i] = p < L.npx ? pixel_owner(reinterpret_cast<const float4 *>(L.rast), p, L.stencils, L.F, L.n_owner) : -1;
    }
#pragma unroll
    for (int i = 0; i < kPartSteps; ++i) {
        unsigned long long left = __ballot(own[i] >= 0);
        while (left) {  // once per owner among the 64 pixels
            const int first = __ffsll((long long)left) - 1, o = __builtin_amdgcn_readlane(own[i], first);
            const unsigned long long m = __ballot(own[i] == o);
            if (lane == first) cnt[o] += __popcll(m);
            wave_lds_sync();  // another lane may count this owner next
            left &= ~m;
        }
    }
}

__global__ void __launch_bounds__(256) k_owner_count(PartitionLaunch L, int n_blk, int *__restrict__ counts) {
    extern __shared__ int cnt[];  // [4][n_owner + 1]
    const int no = L.n_owner + 1, wave = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < 4 * no; i += 256) cnt[i] = 0;
    __syncthreads();
    int own[kPartSteps];
    wave_owners(L, (long long)blockIdx.x * kPartPix + wave * kPartWave, own, cnt + wave * no);
    __syncthreads();
    for (int o = threadIdx.x; o < no; o += 256)
        counts[(long long)o * n_blk + blockIdx.x] = cnt[o] + cnt[no + o] + cnt[2 * no + o] + cnt[3 * no + o];
}

// counts -> exclusive prefix, owner by owner; the owners' runs
__global__ void __launch_bounds__(1024) k_owner_scan(int n_owner, int n_blk, int npx, int *__restrict__ counts,
                                                     int *__restrict__ starts, int *__restrict__ ends) {
    __shared__ int wsum[16];
    const int n = (n_owner + 1) * n_blk;
    int base = 0;
    for (int i0 = 0; i0 < n; i0 += 1024) {
        const int i = i0 + (int)threadIdx.x, c = i < n ? counts[i] : 0;
        int total;
        const int ex = block_scan<1024>(c, wsum, total);
        if (i < n) counts[i] = base + ex;
        base += total;
        __syncthreads();
    }
    for (int o = threadIdx.x; o <= n_owner; o += 1024) {
        const int s = counts[o * n_blk], e = o < n_owner ? counts[(o + 1) * n_blk] : npx;
        starts[o] = s < e ? s : 0;
        ends[o] = s < e ? e : 0;
    }
}

__device__ __forceinline__ void place_pixel(const PartitionLaunch &L, long long at, long long p) {
    L.order[at] = (int)p;
    if (!L.frag) return;
    reinterpret_cast<float4 *>(L.frag)[at] = reinterpret_cast<const float4 *>(L.rast)[p];
    const long long r = p / L.W;
    L.rows[at] = r;
    L.cols[at] = p - r * L.W;
}

__global__ void __launch_bounds__(256) k_owner_place(PartitionLaunch L, int n_blk, const int *__restrict__ offsets) {
    extern __shared__ int cnt[];  // [4][n_owner + 1]: counts, then the wave's next position per owner
    if ((int)blockIdx.x >= n_blk) {  // the fragments past the layer's
        const long long at = L.npx + (long long)(blockIdx.x - n_blk) * 256 + threadIdx.x;
        if (at < L.n_frag) reinterpret_cast<float4 *>(L.frag)[at] = make_float4(0.f, 0.f, 0.f, 0.f);
        return;
    }
    const int no = L.n_owner + 1, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int i = threadIdx.x; i < 4 * no; i += 256) cnt[i] = 0;
    __syncthreads();
    int own[kPartSteps];
    const long long p0 = (long long)blockIdx.x * kPartPix + wave * kPartWave;
    wave_owners(L, p0, own, cnt + wave * no);
    __syncthreads();
    for (int o = threadIdx.x; o < no; o += 256) {
        int at = offsets[(long long)o * n_blk + blockIdx.x];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const int c = cnt[w * no + o];
            cnt[w * no + o] = at;
            at += c;
        }
    }
    __syncthreads();
    int *next = cnt + wave * no;
#pragma unroll
    for (int i = 0; i < kPartSteps; ++i) {
        unsigned long long left = __ballot(own[i] >= 0);
        while (left) {
            const int first = __ffsll((long long)left) - 1, o = __builtin_amdgcn_readlane(own[i], first);
            const unsigned long long m = __ballot(own[i] == o);
            const int base = next[o];
            wave_lds_sync();  // read by every lane, then moved on by one
            const int rank = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
            if (own[i] == o) place_pixel(L, base + rank, p0 + i * 64 + lane);
            if (lane == first) next[o] = base + __popcll(m);
            wave_lds_sync();
            left &= ~m;
        }
    }
}

__global__ void k_stencil_keys(PartitionLaunch L, unsigned long long *__restrict__ keys) {
    long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= L.npx) return;
    const int o = pixel_owner(reinterpret_cast<const float4 *>(L.rast), p, L.stencils, L.F, L.n_owner);
    keys[p] = ((unsigned long long)(unsigned)o << 32) | (unsigned long long)p;
}

__global__ void k_stencil_runs(PartitionLaunch L, const unsigned long long *__restrict__ sorted) {
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= L.npx) {
        if (i < L.n_frag) reinterpret_cast<float4 *>(L.frag)[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        return;
    }
    unsigned long long k = sorted[i];
    int o = (int)(k >> 32);
    place_pixel(L, i, (long long)(k & 0xffffffffu));
    if (i == 0 || (int)(sorted[i - 1] >> 32) != o) L.starts[o] = (int)i;
    if (i == L.npx - 1 || (int)(sorted[i + 1] >> 32) != o) L.ends[o] = (int)(i + 1);
}

__global__ void k_zero2_i32(int *a, int *b, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = b[i] = 0;
}

static unsigned owner_end_bit(int n_owner) {
    unsigned b = 0;
    while ((1ull << b) <= (unsigned long long)n_owner) ++b;
    return 32 + (b ? b : 1);
}

static size_t sort_bytes(long long npx, int n_owner) {
    size_t s = 0;
    if (npx <= 0) return 0;
    if (rocprim::radix_sort_keys(nullptr, s, (unsigned long long *)nullptr, (unsigned long long *)nullptr,
                                 (size_t)npx, 0, owner_end_bit(n_owner), (hipStream_t)0) != hipSuccess)
        return 0;
    return s;
}

static size_t a256(size_t x) { return (x + 255) & ~(size_t)255; }

static long long part_blocks(long long npx) { return (npx + kPartPix - 1) / kPartPix; }
static bool counting(long long npx, int n_owner) {
    return n_owner < kPartOwners && (n_owner + 1ll) * part_blocks(npx) <= kScanMax;
}

size_t stencil_partition_ws_bytes(long long npx, int n_owner) {
    if (counting(npx, n_owner)) return a256((size_t)((n_owner + 1ll) * part_blocks(npx)) * 4);
    return 2 * a256((size_t)npx * 8) + a256(sort_bytes(npx, n_owner));
}

int launch_stencil_partition(const PartitionLaunch &L, void *ws, hipStream_t st) {
    const long long extra = L.frag ? L.n_frag - L.npx : 0;
    if (counting(L.npx, L.n_owner)) {
        const int n_blk = (int)part_blocks(L.npx);
        const size_t lds = 4 * sizeof(int) * (size_t)(L.n_owner + 1);
        int *counts = (int *)ws;
        hipLaunchKernelGGL(k_owner_count, dim3(n_blk), dim3(256), lds, st, L, n_blk, counts);
        hipLaunchKernelGGL(k_owner_scan, dim3(1), dim3(1024), 0, st, L.n_owner, n_blk, (int)L.npx, counts, L.starts,
                           L.ends);
        hipLaunchKernelGGL(k_owner_place, dim3((unsigned)(n_blk + (extra + 255) / 256)), dim3(256), lds, st, L, n_blk,
                           (const int *)counts);
        return hipGetLastError() == hipSuccess ? 0 : -2;
    }
    char *b = (char *)ws;
    unsigned long long *keys = (unsigned long long *)b, *sorted = (unsigned long long *)(b + a256((size_t)L.npx * 8));
    void *temp = b + 2 * a256((size_t)L.npx * 8);
    hipLaunchKernelGGL(k_zero2_i32, dim3((unsigned)((L.n_owner + 1 + 255) / 256)), dim3(256), 0, st, L.starts, L.ends,
                       L.n_owner + 1);
    hipLaunchKernelGGL(k_stencil_keys, dim3((unsigned)((L.npx + 255) / 256)), dim3(256), 0, st, L, keys);
    size_t temp_bytes = sort_bytes(L.npx, L.n_owner);
    if (rocprim::radix_sort_keys(temp, temp_bytes, keys, sorted, (size_t)L.npx, 0, owner_end_bit(L.n_owner), st) !=
        hipSuccess)
        return -2;
    hipLaunchKernelGGL(k_stencil_runs, dim3((unsigned)((L.npx + extra + 255) / 256)), dim3(256), 0, st, L,
                       (const unsigned long long *)sorted);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace drp
