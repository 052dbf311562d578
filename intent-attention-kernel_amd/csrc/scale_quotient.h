// Division by a quantisation scale without the division, for the quantising kernels.
#ifndef IAK_SCALE_QUOTIENT_H
#define IAK_SCALE_QUOTIENT_H

namespace iak {

// x / s as the IEEE float32 division rounds it, from r = RN(1 / s) (once per scale):
// q1 is within one ulp of the quotient, its remainder x - q1 s is exact in the
// fma, and the last fma then rounds correctly (Markstein's theorem). Five operations
// in place of the division's dozen. For s in [2^-30, 2^121] and |x| <= 128 s, except:
// quotients below 2^-12 are only small, and a zero's sign is lost (callers round to
// integers or put the sign back). A NaN or infinite s gives NaN for every x.
__device__ __forceinline__ float scale_quotient(float x, float s, float r) {
  const float q0 = x * r;
  const float q1 = __builtin_fmaf(__builtin_fmaf(-q0, s, x), r, q0);
  return __builtin_fmaf(__builtin_fmaf(-q1, s, x), r, q1);
}

}  // namespace iak

#endif
