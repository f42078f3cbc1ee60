// Cross-lane primitives of a 64-lane wave on the VALU's own data paths (DPP
// and gfx950's row / half swaps), in place of ds_bpermute shuffles: those cost
// an LDS round trip and several address instructions each, and the kernels
// that sort and scan per tile are bound by instruction issue.  Measured (sorts
// and scans of the binning, the fine raster, the antialias queues and the tile
// backward together): 64-view 512^2 step 2.986 -> 2.923 ms, a crumpled uneven
// batch's step 3.118 -> 2.894 ms.
// All of them need every lane of the wave active (wave-uniform control flow).
#pragma once
#include <hip/hip_runtime.h>

namespace drp {

// DPP controls (GFX9): lane ^ 1, lane ^ 2, lane ^ 3 within quads; lane ^ 7 and
// lane ^ 15 (mirrors); rotation by 8 within a row of 16 (lane ^ 8)
enum : int {
    kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppXor3 = 0x1B, kDppXor7 = 0x141, kDppXor15 = 0x140, kDppXor8 = 0x128,
    kDppShr1 = 0x111, kDppShr2 = 0x112, kDppShr4 = 0x114, kDppShr8 = 0x118, kDppBcast15 = 0x142, kDppBcast31 = 0x143
};

template <int CTRL>
__device__ __forceinline__ unsigned dpp_mov(unsigned x) {
    return (unsigned)__builtin_amdgcn_mov_dpp((int)x, CTRL, 0xf, 0xf, true);
}

// x of lane ^ XOR, XOR a power of two
template <int XOR>
__device__ __forceinline__ unsigned lane_xor(unsigned x) {
    static_assert(XOR == 1 || XOR == 2 || XOR == 4 || XOR == 8 || XOR == 16 || XOR == 32, "a power of two");
    if constexpr (XOR == 1) return dpp_mov<kDppXor1>(x);
    else if constexpr (XOR == 2) return dpp_mov<kDppXor2>(x);
    else if constexpr (XOR == 4) return dpp_mov<kDppXor3>(dpp_mov<kDppXor7>(x));
    else if constexpr (XOR == 8) return dpp_mov<kDppXor8>(x);
    else if constexpr (XOR == 16) {  // the odd rows' partners arrive in the first word, the even rows' in the second
        const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        return __builtin_amdgcn_inverse_ballot_w64(0xffff0000ffff0000ull) ? r[0] : r[1];
    } else {
        const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
        return __builtin_amdgcn_inverse_ballot_w64(0xffffffff00000000ull) ? r[0] : r[1];
    }
}
template <int XOR>
__device__ __forceinline__ float lane_xor(float x) {
    return __uint_as_float(lane_xor<XOR>(__float_as_uint(x)));
}

// largest x over aligned groups of N lanes, in every lane of the group
template <int N>
__device__ __forceinline__ float group_max(float x) {
    if constexpr (N >= 2) x = fmaxf(x, lane_xor<1>(x));
    if constexpr (N >= 4) x = fmaxf(x, lane_xor<2>(x));
    if constexpr (N >= 8) x = fmaxf(x, lane_xor<4>(x));
    if constexpr (N >= 16) x = fmaxf(x, lane_xor<8>(x));
    if constexpr (N >= 32) x = fmaxf(x, lane_xor<16>(x));
    if constexpr (N >= 64) x = fmaxf(x, lane_xor<32>(x));
    return x;
}

// LDS words handed from lane to lane within a wave, without a block barrier: the
// loads after see the stores before.  (The hardware keeps a wave's LDS accesses in
// order; the fences keep the compiler to it, which may otherwise move or keep a
// lane's load across another lane's store.)
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// lanes that keep the minimum in the bitonic step (size, stride)
constexpr unsigned long long bitonic_min_mask(int size, int stride) {
    unsigned long long m = 0;
    for (int lane = 0; lane < 64; ++lane)
        if (((lane & stride) == 0) == ((lane & size) == 0)) m |= 1ull << lane;
    return m;
}

// one compare-exchange of the bitonic sort: lane i against lane i ^ STRIDE
template <int SIZE, int STRIDE>
__device__ __forceinline__ unsigned bitonic_step(unsigned k) {
    unsigned a = k, b;
    if constexpr (STRIDE == 32) {  // the swapped pair holds both lanes' keys in either order
        const auto r = __builtin_amdgcn_permlane32_swap(k, k, false, false);
        a = r[0];
        b = r[1];
    } else if constexpr (STRIDE == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(k, k, false, false);
        a = r[0];
        b = r[1];
    } else {
        b = lane_xor<STRIDE>(k);
    }
    const unsigned lo = a < b ? a : b, hi = a < b ? b : a;
    return __builtin_amdgcn_inverse_ballot_w64(bitonic_min_mask(SIZE, STRIDE)) ? lo : hi;
}
template <int SIZE, int STRIDE>
__device__ __forceinline__ unsigned bitonic_merge(unsigned k) {
    k = bitonic_step<SIZE, STRIDE>(k);
    if constexpr (STRIDE > 1) k = bitonic_merge<SIZE, STRIDE / 2>(k);
    return k;
}

// the wave's 64 keys in ascending order by lane
__device__ __forceinline__ unsigned wave_sort(unsigned k) {
    k = bitonic_merge<2, 1>(k);
    k = bitonic_merge<4, 2>(k);
    k = bitonic_merge<8, 4>(k);
    k = bitonic_merge<16, 8>(k);
    k = bitonic_merge<32, 16>(k);
    return bitonic_merge<64, 32>(k);
}
__device__ __forceinline__ unsigned long long wave_sort(unsigned long long k) {  // wide keys: shuffles
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int size = 2; size <= 64; size <<= 1) {
#pragma unroll
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            const unsigned long long o = __shfl_xor(k, stride, 64);
            const bool keep_min = ((lane & stride) == 0) == ((lane & size) == 0);
            k = keep_min ? (o < k ? o : k) : (o > k ? o : k);
        }
    }
    return k;
}

template <int CTRL, int ROWS>
__device__ __forceinline__ int scan_step(int x) {  // lanes without a source add 0
    return x + __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xf, false);
}

// sum over lanes 0 .. this one
__device__ __forceinline__ int wave_incl_scan(int x) {
    x = scan_step<kDppShr1, 0xf>(x);
    x = scan_step<kDppShr2, 0xf>(x);
    x = scan_step<kDppShr4, 0xf>(x);
    x = scan_step<kDppShr8, 0xf>(x);
    x = scan_step<kDppBcast15, 0xa>(x);  // rows 1 and 3 add the last lane of the row before
    return scan_step<kDppBcast31, 0xc>(x);  // rows 2 and 3 add lane 31
}

template <int CTRL, int ROWS>
__device__ __forceinline__ int max_step(int x) {  // lanes without a source keep theirs (x >= 0)
    const int y = __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xf, false);
    return x > y ? x : y;
}

// largest of the non-negative values of lanes 0 .. this one
__device__ __forceinline__ int wave_incl_max(int x) {
    x = max_step<kDppShr1, 0xf>(x);
    x = max_step<kDppShr2, 0xf>(x);
    x = max_step<kDppShr4, 0xf>(x);
    x = max_step<kDppShr8, 0xf>(x);
    x = max_step<kDppBcast15, 0xa>(x);
    return max_step<kDppBcast31, 0xc>(x);
}

// exclusive scan over a block of NT threads; wsum: NT / 64 words of LDS that
// nothing else uses between this call and the block's next barrier
template <int NT>
__device__ __forceinline__ int block_scan(int v, int *wsum, int &total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int x = wave_incl_scan(v);
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    int pre = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
        const int s = wsum[w];
        if (w < wave) pre += s;
        tot += s;
    }
    total = tot;
    return pre + x - v;
}

}  // namespace drp
