// The weight of one ray of the skip walk, sqrt(S) * W / D: S its squared
// length, W the sum of the coefficients over its steps, D its steps less one.
// Included by skip_walk.h, and by itself where the arithmetic is tested.
#pragma once

#ifndef ANACOR_DEVICE
#define ANACOR_DEVICE
#endif

// rsq and rcp estimate 1 / sqrt and 1 / to 2^-22 or better.
//   * Root (Goldschmidt's iteration, P. Markstein, Software division and square
//     root using Goldschmidt's algorithms, 2004): y carries 2^-22, one step
//     2^-43, and the last correction adds the exact remainder S - g^2 times
//     1 / 2g, so g is the correctly rounded root but for ties closer than 2^-33
//     of an ulp.
//   * Quotient: q carries 2^-43 after one step; t + (W - t D) q with the exact
//     remainder W - t D likewise rounds W / D correctly.
// One rounding more follows, of the product.  So a weight has three roundings
// behind S and W, as many as sqrt(S) / D * W by the correctly rounded pair and
// one fewer per label than the stepping kernel's sum of segments: its error is
// 0.69 units of 2^-53 in the mean against 0.72 stepping (voxel edges of 1;
// 0.77 and 0.81 with unequal edges), two million random rays against 113 bits.
// A quotient of the root by a reciprocal rounded to an ulp or two, then times
// W, has 0.80 (0.87).
template <class Rsq, class Rcp>
ANACOR_DEVICE inline double ray_weight(double S, double W, double D, Rsq rsq, Rcp rcp) {
  const double y = rsq(S);
  double g = S * y, h = 0.5 * y;
  const double e = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, e, g);
  h = __builtin_fma(h, e, h);
  g = __builtin_fma(__builtin_fma(-g, g, S), h, g);
  double q = rcp(D);
  q = __builtin_fma(__builtin_fma(-D, q, 1.0), q, q);
  double t = W * q;
  t = __builtin_fma(__builtin_fma(-t, D, W), q, t);
  return S > 0.0 ? g * t : 0.0;       // a ray held on its origin by the clamps
}
