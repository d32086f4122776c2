// sin_cw.h -- sin^2 in single precision for the snake activation
// (snake_activation_frame_major, crates/fish_s2_infer/src/codec.rs:2162-2186,
// which evaluates sin with the C library's sinf).
//
// Method: sin^2 has period pi, so Cody & Waite argument reduction by pi (split
// into three floats c1 + c2 + c3, each product exact inside a fused
// multiply-add) to r in [-pi/2, pi/2], then one odd polynomial r + r^3 P(r^2),
// P of degree 3 fitted here to sin over that interval (relative error 6.1e-9;
// sin^2 in f32 within 2.4e-7), squared.  No quadrant to select: 12 operations.
// Checked on the host against glibc sinf squared over |x| <= 1024
// (tests/test_cpu_host.py).
#pragma once

#include <hip/hip_runtime.h>

namespace s2 {

__host__ __device__ inline float sin_sq_cw(float x) {
  const float k = rintf(x * 0.31830987f);  // 1 / pi
  float r = fmaf(-k, 3.14159274f, x);      // c1 = f32(pi)
  r = fmaf(-k, -8.74227766e-08f, r);       // c2 = f32(pi - c1)
  r = fmaf(-k, -3.43024902e-15f, r);       // c3 = f32(pi - c1 - c2)
  const float z = r * r;
  const float p = fmaf(fmaf(fmaf(2.6056311526190257e-06f, z, -1.980953966267407e-04f), z, 8.333065547049046e-03f), z,
                       -1.6666659712791443e-01f);
  const float v = fmaf(r * z, p, r);
  return v * v;
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
