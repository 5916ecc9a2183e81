// The SiTU-GLU activation (ml/runtime/model/blocks.py:23-27), shared by the
// element-wise kernel and the few-row projection that forms it on its sums.
#pragma once

#include "common.hpp"

namespace sophia {

// tanh(x) for x = |z| / cap >= 0 as a fraction num / den: with t = e^{-2x},
// (1 - t) / (1 + t); below x = 1/8, where 1 - t cancels, the Taylor series
// x (1 - x^2/3 + 2x^4/15 - 17x^6/315) over 1 (truncation below 2e-9
// relative).  t is returned for the sigmoid (cap 4: e^{-|z|} = t^2).
struct Frac {
  float num, den, t;
};

__device__ __forceinline__ float tanh_series(float x) {
  const float x2 = x * x;
  return x * fmaf(x2, fmaf(x2, fmaf(x2, -17.0f / 315.0f, 2.0f / 15.0f), -1.0f / 3.0f), 1.0f);
}

__device__ __forceinline__ Frac tanh_frac(float x) {
  constexpr float kM2Log2e = -2.0f * 1.44269504088896341f;
  const float t = __builtin_amdgcn_exp2f(kM2Log2e * x);
  const bool small = x < 0.125f;
  return Frac{small ? tanh_series(x) : 1.0f - t, small ? 1.0f : 1.0f + t, t};
}

//   h = cg tanh(g/cg) sigmoid(g) * cu tanh(u/cu)
//     = cg cu sgn(g) sgn(u) num_g num_u s / (den_g den_u (1 + e))
// with e = e^{-|g|} <= 1 and s = 1 (g >= 0) or e (g < 0): every factor of the
// denominator lies in [1, 2], so one reciprocal serves the element.  With the
// reference's gate cap of 4 (CAP4), e = t_g^2 and no third exponential is
// needed.  rcg = 1 / cg, rcu = 1 / cu, scale = cg cu; fu = tanh_frac(|u| rcu).
template <bool CAP4>
__device__ __forceinline__ float situ_value(float g, float u, const Frac &fu, float rcg, float scale) {
  const float ag = fabsf(g);
  const Frac fg = tanh_frac(ag * rcg);
  const float e = CAP4 ? fg.t * fg.t : __builtin_amdgcn_exp2f(-1.44269504088896341f * ag);
  const float s = g >= 0.f ? 1.0f : e;
  const float mag = scale * fg.num * fu.num * s * __builtin_amdgcn_rcpf(fg.den * fu.den * (1.0f + e));
  // sign of g times sign of u, as a flip of the sign bit
  return __uint_as_float(__float_as_uint(mag) ^ ((__float_as_uint(g) ^ __float_as_uint(u)) & 0x80000000u));
}

template <bool CAP4>
__device__ __forceinline__ float situ_value(float g, float u, float rcg, float rcu, float scale) {
  return situ_value<CAP4>(g, u, tanh_frac(fabsf(u) * rcu), rcg, scale);
}

}  // namespace sophia
