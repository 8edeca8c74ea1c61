// What the device headers take from HIP, for one lane on the CPU: the
// function attributes and the few intrinsics they call.
#pragma once
#include <math.h>
#include <stdint.h>
#include <string.h>

#include <cmath>

#define __device__
#define __host__
#define __forceinline__ inline
using std::fabs;
using std::fma;
using std::fmin;
using std::sqrt;

inline int __ffs(unsigned x) { return __builtin_ffs((int)x); }
inline int __popc(unsigned x) { return __builtin_popcount(x); }

inline bool __any(bool x) { return x; }

// the hardware's square root and reciprocal are good to one unit in the last
// place: lane_ulp moves a result by -1, 0 or 1 of them, by its argument's bits
extern int lane_ulp;
inline float lane_rounded(float y, float x)
{
    if (!lane_ulp || !(std::fabs(y) < HUGE_VALF) || y == 0.0f) return y;
    uint32_t b;
    memcpy(&b, &x, sizeof b);
    b = (b ^ (b >> 15)) * 0x2c1b3c6du * (uint32_t)lane_ulp;
    b ^= b >> 13;
    const int d = (int)(b % 3u) - 1;
    return d ? std::nextafter(y, d > 0 ? HUGE_VALF : -HUGE_VALF) : y;
}
inline float lane_sqrt(float x) { return lane_rounded(std::sqrt(x), x); }
inline float lane_rcp(float x) { return lane_rounded(1.0f / x, x); }
#define __builtin_amdgcn_sqrtf lane_sqrt
#define __builtin_amdgcn_rcpf lane_rcp
