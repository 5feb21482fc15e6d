// The device declarations that the frame header needs, for a host compiler.
#pragma once
#include <cmath>
#include <cstdint>
#define __device__
#define __forceinline__ inline
struct alignas(16) float4 { float x, y, z, w; };
struct alignas(8) uint2 { uint32_t x, y; };
struct alignas(16) uint4 { uint32_t x, y, z, w; };
inline float4 make_float4(float x, float y, float z, float w) { return {x, y, z, w}; }
inline float rsqrtf(float x) { return 1.0f / std::sqrt(x); }
#define __builtin_amdgcn_rsq(x) (1.0 / std::sqrt(x))
#define __builtin_amdgcn_fmed3f(x, lo, hi) std::fmin(std::fmax(x, lo), hi)
