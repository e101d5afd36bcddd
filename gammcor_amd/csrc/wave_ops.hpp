// Sums and broadcasts over a wave of 64 lanes on the DPP and lane-swap paths:
// the LDS-crossbar shuffles (ds_bpermute, ds_swizzle) take several times
// their latency, which counts where a sum is on a kernel's critical path.
// Every sum has a fixed order.
#pragma once
#include "common.hpp"

namespace gmc {

// Workgroup barrier for data in LDS only.  __syncthreads also waits for the
// waves' outstanding global accesses, stores included: after a store that has
// to travel to memory (an exchange between workgroups) that is 2-4 us.
__device__ inline void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// v of lane l (uniform), as a scalar.
__device__ inline float read_lane(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ inline double read_lane(double v, int l)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffff), l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

template <int CTRL>
__device__ inline float dpp_mov(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ inline double dpp_mov(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffff), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E, DPP_HALF_MIRROR = 0x141, DPP_MIRROR = 0x140;
// a + b after a's upper half (32 lanes; or a's odd rows of 16, O = 16) and
// b's lower half (even rows) have changed places: the lower lanes get the sum
// of a over both halves, the upper ones that of b
template <int O>
__device__ inline float swap_add(float a, float b)
{
    const auto r = O == 32 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false)
                           : __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
template <int O>
__device__ inline double swap_add(double a, double b)
{
    const unsigned long long x = (unsigned long long)__double_as_longlong(a), y = (unsigned long long)__double_as_longlong(b);
    const auto lo = O == 32 ? __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false)
                            : __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = O == 32 ? __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false)
                            : __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    return __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0])) +
           __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
}
// The sum of v over the wave, in every lane.
template <class T>
__device__ inline T wave_total(T v)
{
    v += dpp_mov<DPP_XOR1>(v);
    v += dpp_mov<DPP_XOR2>(v);
    v += dpp_mov<DPP_HALF_MIRROR>(v);
    v += dpp_mov<DPP_MIRROR>(v);
    v = swap_add<16>(v, v);
    return swap_add<32>(v, v);
}
// One halving step across lane bit O: a lane keeps H of its values and adds
// its partner's share of them; below one value per lane plain sums.
template <int H, int O, int CTRL, int KV, class T>
__device__ inline void half_step(T (&s)[KV], int lane)
{
    if constexpr (H >= 1) {
        const bool up = (lane & O) != 0;
#pragma unroll
        for (int k = 0; k < H; k++) {
            const T send = up ? s[k] : s[k + H], keep = up ? s[k + H] : s[k];
            s[k] = keep + dpp_mov<CTRL>(send);
        }
    } else {
        s[0] += dpp_mov<CTRL>(s[0]);
    }
}
// The sums over the wave of KV values per lane (KV = 4, 8 or 16): the lane
// gets that of column lane >> (6 - log2 KV).
template <int KV, class T>
__device__ inline T wave_col_sums(T (&s)[KV], int lane)
{
    static_assert(KV == 4 || KV == 8 || KV == 16, "columns per reduction");
#pragma unroll
    for (int k = 0; k < KV / 2; k++) s[k] = swap_add<32>(s[k], s[k + KV / 2]);
#pragma unroll
    for (int k = 0; k < KV / 4; k++) s[k] = swap_add<16>(s[k], s[k + KV / 4]);
    half_step<KV / 8, 8, DPP_MIRROR>(s, lane);
    half_step<KV / 16, 4, DPP_HALF_MIRROR>(s, lane);
    half_step<0, 2, DPP_XOR2>(s, lane);
    half_step<0, 1, DPP_XOR1>(s, lane);
    return s[0];
}

}  // namespace gmc
