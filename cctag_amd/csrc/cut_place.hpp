// Where the samples of a cut lie at a homography, from the cut's two ends
// (used by the grid search's kernels; plain arithmetic, so that it can be
// checked on the CPU as well).
#pragma once

#include <cmath>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define CCTAGX_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define CCTAGX_HOST_DEVICE inline
#endif

namespace cctagx {

// The samples are, up to rounding, the images (homography H) of the
// marker-plane segment t * b, t in [begin, end], b the stop (x, y)
// back-projected by the inverse Hi (homogeneous b = Hi (stop, 1)).  When the
// projective denominator keeps its sign between the ends (it is linear in t)
// the image is the straight segment between the ends' images, so two ends
// 2 px inside the w x h image keep every sample in [0, w-1) x [0, h-1), and
// one end 2 px outside puts its own sample outside.
//
// What rounding does to a sample: its marker-plane position is a running sum
// of at most 127 rounded steps, off by a relative 131 u (u = 2^-24: the sums,
// the step, the start); the map adds 3 u of the terms' magnitudes and the
// quotient u.  With mag the sum of a numerator's term magnitudes and dmag
// that of the denominator d, a position moves by at most
// 139 u (mag / |d|) (1 + dmag / |d|), the ends' own evaluation here included.
// Along the cut both ratios are monotone, so their bounds at the ends --
// `steady`: mag < 2^15 |d|, dmag < 4 |d| -- hold for every sample: at most
// 1.4 px, within the 2.  The window on the denominator keeps div2_rn away from
// the ends of the float range; a row of 2^24 pixels is beyond the sampling's
// 24-bit addresses.  Anything else is kUnsure and gets its samples tested.
enum CutPlace { kInside, kOutside, kUnsure };
CCTAGX_HOST_DEVICE CutPlace cut_place(const float* H, const float* Hi, float sx, float sy,
                                      float begin_sig, float end_sig, int w, int h) {
  const float b0 = Hi[0] * sx + Hi[1] * sy + Hi[2];
  const float b1 = Hi[3] * sx + Hi[4] * sy + Hi[5];
  const float b2 = Hi[6] * sx + Hi[7] * sy + Hi[8];
  bool all_in = w < 1 << 24, out = false;
  float den[2];
  for (int e = 0; e < 2; ++e) {
    const float t = e ? end_sig : begin_sig, p0 = t * b0, p1 = t * b1;
    const float d = H[6] * p0 + H[7] * p1 + H[8] * b2, ad = fabsf(d);
    const float s = d < 0.f ? -1.f : 1.f;
    const float x = s * (H[0] * p0 + H[1] * p1 + H[2] * b2);  // times |d|: the position
    const float y = s * (H[3] * p0 + H[4] * p1 + H[5] * b2);
    const float mag = fmaxf(fabsf(H[0] * p0) + fabsf(H[1] * p1) + fabsf(H[2] * b2),
                            fabsf(H[3] * p0) + fabsf(H[4] * p1) + fabsf(H[5] * b2));
    const float dmag = fabsf(H[6] * p0) + fabsf(H[7] * p1) + fabsf(H[8] * b2);
    const bool steady = ad > 0.25f * dmag && mag < 32768.f * ad && ad > 0x1p-60f * fabsf(b2) &&
                        ad < 0x1p60f * fabsf(b2);
    den[e] = d;
    all_in &= steady && x >= 2.f * ad && x <= (float)(w - 3) * ad && y >= 2.f * ad &&
              y <= (float)(h - 3) * ad;
    out |= steady && (x < -2.f * ad || x > (float)(w + 1) * ad || y < -2.f * ad ||
                      y > (float)(h + 1) * ad);
  }
  if (out) return kOutside;
  return all_in && (den[0] > 0.f) == (den[1] > 0.f) ? kInside : kUnsure;
}

}  // namespace cctagx
