// Triangle frames: per slot, the triangle in its own plane, so that an FP32 point-triangle distance
// takes no branches (closest-point kernels; the refit and the upload write them).
//
// The base is the longest edge P0 P1 (length L), P2 the apex. With the unit vectors u along the base,
// n normal to the plane and v = n x u, a query r = q - P0 has the plane coordinates x = u.r, y = v.r
// and the height z = n.r, and the squared distance is z^2 plus the squared distance of (x, y) to the
// plane triangle (0, 0), (L, 0), P2: zero inside, else the least over the three edges of
// (t - clamp(t, 0, length))^2 + s^2 with t along the edge and s across it.
//
// kFrameRows float4 per slot (f0 .. f4):
//   f0  P0.x P0.y P0.z  w          f1  u.x u.y u.z  L
//   f2  v.x  v.y  v.z   e1.x       f3  n.x n.y n.z  e1.y
//   f4  L1   e2.x e2.y  L2         (e1, L1: direction and length of P1 P2; e2, L2: of P0 P2)
//
// Error of the FP32 value (k = 2^-24, d the exact distance, rho its part in the plane; second order in
// k left to the slack below). The vectors are rounded from double, r = q - P0 rounds once, each
// coordinate is one product and two fused multiply-adds: |error of x| <= 5 k (|u.x r.x| + |u.y r.y| +
// |u.z r.z|) and alike for y and z, together <= 5 k (5/3) |r| (5/3 bounds the norm of an orthogonal
// matrix's absolute values), and the distance to a fixed triangle is 1-Lipschitz: 8.4 k (d + L). In the plane, t and s of
// P1 P2 (taken from P1, |p - P1| <= rho + L) are each within 3.42 k (rho + L) + k L, the clamp's length
// within k L, t - clamp rounds once: 5.84 k rho + 7.26 k L for that edge and less for the others. The
// squares and sums round three times: 3 k d^2. Inside is decided by the signs of y, s1, s2 and by
// 0 <= x <= L, each within 4.5 k L there; the base being the longest edge, the angles at its ends are
// acute (they alone may be arbitrarily sharp, and the slab 0 <= x <= L cuts the wedges past them) and
// the one at P2 is at least 60 degrees, so a point wrongly called inside is within 2.5 times that of
// the triangle: second order in the square. So
//   |error of d^2| <= 2 d (8.4 k (d + L) + 5.84 k d + 7.26 k L) + 3 k d^2 = 31.5 k d^2 + 31.4 k d L,
// and with d L <= d^2 / 32 + 8 L^2 at most kFrameRel d^2 + |w|, kFrameRel = 34 k, w = 256 k L^2. (A band
// of 128 k, from 2 d L <= d^2 + L^2 and coarser steps, lists six candidates per query instead of two on
// a 256^3 grid over a million-triangle sphere: 317 ms instead of the figures at the kernels.)
//
// A triangle whose apex height is at most 2^-20 L has the frame of its base alone, with any normal: the
// cross product that would give the normal is rounding noise there (for collinear corners u x w has its
// whole value from u's rounding), and a frame from it is not orthogonal. The triangle holds its base and
// lies within that height of it, so its distance is at most that of the base and at least that less the
// height: 2 d h <= 32 k d L more on one side, in all 33.5 k d^2 + 508 k L^2, w = 512 k L^2. With two equal
// corners the triangle is the base and w stays 256 k L^2.
//
// The sign bit of w: the exact step may not reach the triangle's distance, so it may be listed but must not
// bound the search. So where the corners are a, a, c, whose weights on the edge a a are 0 / 0, and where
// three distinct corners are flat: the signs that choose the region are rounding noise then, and the face
// region can divide one noise by another. a, b, b and a, b, a are sure: with d3 = d5 and d4 = d6, or d2 = d4 =
// d6 = 0, one of vb, vc is <= 0 as computed and the edge a b is taken. w is NaN where a corner is not
// finite, and d2 too: every comparison with its bounds fails, and the triangle is left to the exact step.
#pragma once

#include "mbvh_device.h"

namespace mbvh {

constexpr int kFrameRows = 5;
constexpr float kFrameRel = 34.0f * 5.9604644775390625e-08f;

namespace {

struct D3f {
  double x, y, z;
};
__device__ __forceinline__ D3f f_sub(D3f a, D3f b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ double f_dot(D3f a, D3f b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ D3f f_cross(D3f a, D3f b) {
  return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ D3f f_scale(D3f a, double s) { return {a.x * s, a.y * s, a.z * s}; }

// 1 / sqrt(x) to 2^-44 of its value, far below the float rounding of what it scales: the hardware's
// estimate (2^-23) and one Newton step.
__device__ __forceinline__ double f_rsqrt(double x) {
  const double r = __builtin_amdgcn_rsq(x);
  return r * (1.5 - 0.5 * x * r * r);
}

__device__ __forceinline__ void tri_frame(f3 fa, f3 fb, f3 fc, float4* out) {
  const D3f a = {fa.x, fa.y, fa.z}, b = {fb.x, fb.y, fb.z}, c = {fc.x, fc.y, fc.z};
  const D3f ab = f_sub(b, a), bc = f_sub(c, b), ca = f_sub(a, c);
  const double l0 = f_dot(ab, ab), l1 = f_dot(bc, bc), l2 = f_dot(ca, ca);
  D3f p0 = a, base = ab, w = f_sub(c, a);  // base edge, and P2 - P0
  double ll = l0;
  if (l1 > ll) {
    p0 = b;
    base = bc;
    w = f_sub(a, b);
    ll = l1;
  }
  if (l2 > ll) {
    p0 = c;
    base = ca;
    w = f_sub(b, c);
    ll = l2;
  }
  D3f u = {1, 0, 0}, v = {0, 1, 0}, n = {0, 0, 1};
  double L = 0, cx = 0, cy = 0;
  bool flat = true;
  if (!(ll == 0)) {
    const double r = f_rsqrt(ll);
    L = ll * r;
    u = f_scale(base, r);
    n = f_cross(u, w);
    double hh = f_dot(n, n);
    flat = hh <= 9.094947017729282e-13 * ll;  // 2^-40
    if (flat) {
      n = f_cross(u, fabs(u.x) < 0.6 ? D3f{1, 0, 0} : D3f{0, 1, 0});
      hh = f_dot(n, n);
    }
    n = f_scale(n, f_rsqrt(hh));
    v = f_cross(n, u);
    if (!flat) {
      cx = f_dot(u, w);
      cy = f_dot(v, w);
    }
  }
  const double x1 = cx - L, mm1 = x1 * x1 + cy * cy, mm2 = cx * cx + cy * cy;
  double m1 = 0, m2 = 0, e1x = 0, e1y = 1, e2x = 1, e2y = 0;
  if (!(mm1 == 0)) {
    const double r = f_rsqrt(mm1);
    m1 = mm1 * r;
    e1x = x1 * r;
    e1y = cy * r;
  }
  if (!(mm2 == 0)) {
    const double r = f_rsqrt(mm2);
    m2 = mm2 * r;
    e2x = cx * r;
    e2y = cy * r;
  }
  const bool equal = l0 == 0 || l1 == 0 || l2 == 0;
  const float wide = static_cast<float>((flat && !equal ? 512.0 : 256.0) * 5.9604644775390625e-08 * 1.0001 * ll);
  const bool unsure = flat && (equal ? l0 == 0 && l1 != 0 : true);
  const float f0w = l0 + l1 + l2 < 1e300 ? (unsure ? -wide : wide) : __builtin_nanf("");
  // p0 is one of the float vertices: the conversion is exact
  out[0] = make_float4(static_cast<float>(p0.x), static_cast<float>(p0.y), static_cast<float>(p0.z), f0w);
  out[1] = make_float4(static_cast<float>(u.x), static_cast<float>(u.y), static_cast<float>(u.z), static_cast<float>(L));
  out[2] = make_float4(static_cast<float>(v.x), static_cast<float>(v.y), static_cast<float>(v.z), static_cast<float>(e1x));
  out[3] = make_float4(static_cast<float>(n.x), static_cast<float>(n.y), static_cast<float>(n.z), static_cast<float>(e1y));
  out[4] = make_float4(static_cast<float>(m1), static_cast<float>(e2x), static_cast<float>(e2y), static_cast<float>(m2));
}

// The FP32 squared distance from q to the triangle of a frame.
__device__ __forceinline__ float frame_dist2(f3 q, float4 f0, float4 f1, float4 f2, float4 f3_, float4 f4) {
  const float rx = q.x - f0.x, ry = q.y - f0.y, rz = q.z - f0.z;
  const float x = fmaf(f1.z, rz, fmaf(f1.y, ry, f1.x * rx));
  const float y = fmaf(f2.z, rz, fmaf(f2.y, ry, f2.x * rx));
  const float z = fmaf(f3_.z, rz, fmaf(f3_.y, ry, f3_.x * rx));
  const float o0 = x - __builtin_amdgcn_fmed3f(x, 0.0f, f1.w);
  const float xl = x - f1.w;
  const float t1 = fmaf(f2.w, xl, f3_.w * y), s1 = fmaf(f2.w, y, -(f3_.w * xl));
  const float t2 = fmaf(f4.y, x, f4.z * y), s2 = fmaf(f4.z, x, -(f4.y * y));
  const float o1 = t1 - __builtin_amdgcn_fmed3f(t1, 0.0f, f4.x);
  const float o2 = t2 - __builtin_amdgcn_fmed3f(t2, 0.0f, f4.w);
  const float d0 = fmaf(o0, o0, y * y), d1 = fmaf(o1, o1, s1 * s1), d2 = fmaf(o2, o2, s2 * s2);
  const float edge = fminf(fminf(d0, d1), d2);
  const float side = fminf(fminf(fminf(y, s1), s2), -fabsf(o0));
  return fmaf(z, z, side >= 0.0f ? 0.0f : edge);
}

}  // namespace
}  // namespace mbvh
