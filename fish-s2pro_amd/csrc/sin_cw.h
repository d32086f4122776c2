// sin_cw.h -- sin^2 in single precision for the snake activation
// (snake_activation_frame_major, crates/fish_s2_infer/src/codec.rs:2162-2186,
// which evaluates sin with the C library's sinf).
//
// Method: sin^2 has period pi, so Cody & Waite argument reduction by pi (split
// into three floats c1 + c2 + c3, each product exact inside a fused
// multiply-add) to r in [-pi/2, pi/2], then sin^2 r = z Q(z) of z = r^2, Q of
// degree 5 in z - 1.25 fitted here to sin^2 r / r^2.  No quadrant to select: 13
// operations.  Over every float in [2^-6, 1024] the largest absolute error against
// 64 bits is 1.64e-7, the root mean square 3.0e-8 and the largest relative error
// 3.0e-7.  The centre is what keeps it there: |z - 1.25| <= 1.25 carries the
// rounding of the inner coefficients, where powers of z up to 2.47 would (1.8e-7 about
// z = 0).  A sine polynomial on [-pi/2, pi/2], squared, is off by up to 2.5e-7 (12
// operations); sine and cosine polynomials on [-pi/4, pi/4] by quadrant reach
// 1.67e-7, 3.7e-8 and 3.1e-7 (20 operations).  Checked on the host against 64 bits
// where the error is largest, and against glibc sinf squared over |x| <= 1024
// (tests/test_cpu_host.py).
#pragma once

#include <hip/hip_runtime.h>

namespace s2 {

__host__ __device__ inline float sin_sq_cw(float x) {
  const float k = rintf(x * 0.31830987f);  // 1 / pi
  float r = fmaf(-k, 3.14159274f, x);      // c1 = f32(pi)
  r = fmaf(-k, -8.74227766e-08f, r);       // c2 = f32(pi - c1)
  r = fmaf(-k, -3.43024902e-15f, r);       // c3 = f32(pi - c1 - c2)
  const float z = r * r, w = z - 1.25f;
  float q = fmaf(w, -3.62368132e-06f, 1.16671101e-04f);
  q = fmaf(w, q, -2.532396e-03f);
  q = fmaf(w, q, 3.37821245e-02f);
  q = fmaf(w, q, -2.36051396e-01f);
  q = fmaf(w, q, 6.46909177e-01f);
  return z * q;
}

// the reference's guard |a| < 1e-8 -> 1e-8
__host__ __device__ inline float snake_guard(float alpha) { return fabsf(alpha) < 1e-8f ? 1e-8f : alpha; }

// x + sin(a x)^2 / a for a guarded a and inv = 1 / a: the quotient of the
// rounded reciprocal, corrected once by its remainder (a channel's reciprocal
// serves all of its frames; a full division per element cost more than the sine)
__host__ __device__ inline float snake_cw(float x, float a, float inv) {
  const float s = sin_sq_cw(a * x);
  const float q = s * inv;
  return x + fmaf(fmaf(-q, a, s), inv, q);
}
__host__ __device__ inline float snake_cw(float x, float alpha) {
  const float a = snake_guard(alpha);
  return snake_cw(x, a, 1.0f / a);
}

}  // namespace s2
