// gfx950 kernels of CCTag identification.
//
// k_select_cuts  identify_step_1: collectCuts + selectCutCheapUniform
//                (Identification.cpp:396-709, 1172-1301); one block per
//                marker, one thread per outer point.  Bit-exact with the
//                reference's serial float arithmetic.
// k_refine_*     refineConicFamilyGlob (Identification.cpp:813-1158): few
//                markers in one launch per grid-search iteration
//                (k_refine_iter), many in one launch with a block per marker
//                (k_refine_search); then the final signals and the per-cut
//                distances to every bank profile of orazioDistanceRobust
//                (:50-160), or the centres alone (k_refine_centers).  The
//                pairwise sum of squared differences is taken per sample, in
//                double, from the sum and the sum of squares over the valid
//                cuts instead of the reference's sequential float sum;
//                everything else (grid, homographies, sampling, the sticky
//                out-of-bounds flag of a cut) follows the reference's float
//                operations.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>

#include "cut_place.hpp"
#include "division.hpp"
#include "ident_device.hpp"

namespace cctagx {
namespace {

__device__ __forceinline__ float sqrt_rn(float x) { return __builtin_sqrtf(x); }

// A pointer the compiler knows to be in device global memory (the loads
// become global rather than flat ones).
typedef const __attribute__((address_space(1))) uint32_t* gptr_u32;

// The frame as quads: word (x, y) holds pixels (x, y), (x+1, y), (x, y+1),
// (x+1, y+1) in bytes 0..3, so a bilinear sample is one aligned load.
struct Img {
  const uint32_t* q;
  int w, h;
  __device__ __forceinline__ uint32_t quad(int x, int y) const { return ((gptr_u32)q)[x + y * w]; }
  // the same for 0 <= x < w, 0 <= y < h: a 24-bit multiply-add and a 32-bit
  // byte offset (an image has less than 2^30 pixels)
  __device__ __forceinline__ uint32_t quad24(uint32_t x, uint32_t y) const {
    const uint32_t off = (__umul24(y, (uint32_t)w) + x) << 2;
    return *(gptr_u32)((const __attribute__((address_space(1))) char*)(gptr_u32)q + off);
  }
};

// Identification.hpp:197-222: the bilinear value at the offset (fx, fy) into
// the quad of its pixel, and half of it at (x, y).
__device__ __forceinline__ float bilinear2(float fx, float fy, uint32_t quad) {
  const float fx1 = 1.0f - fx, fy1 = 1.0f - fy;
  const float w1 = fx1 * fy1, w2 = fx * fy1, w3 = fx1 * fy, w4 = fx * fy;
  const float a = (float)(quad & 255u), b = (float)((quad >> 8) & 255u),
              c = (float)((quad >> 16) & 255u), d = (float)(quad >> 24);
  return a * w1 + b * w2 + c * w3 + d * w4;
}
__device__ __forceinline__ float bilinear_of(float x, float y, uint32_t quad) {
  return bilinear2(x - (int)x, y - (int)y, quad) / 2;
}

__device__ __forceinline__ void apply_h(float& xr, float& yr, const float* H, float x, float y) {
  const float u = H[0] * x + H[1] * y + H[2];
  const float v = H[3] * x + H[4] * y + H[5];
  const float ww = H[6] * x + H[7] * y + H[8];
  xr = u / ww;
  yr = v / ww;
}

__device__ __forceinline__ float cof(const float* m, int i, int j) {
  const int i1 = (i + 1) % 3, i2 = (i + 2) % 3, j1 = (j + 1) % 3, j2 = (j + 2) % 3;
  return m[i1 * 3 + j1] * m[i2 * 3 + j2] - m[i1 * 3 + j2] * m[i2 * 3 + j1];
}

// Adjugate inverse, same operation order as the host's inverse3.
__device__ void inverse3(const float* m, float* out) {
  const float c0 = cof(m, 0, 0), c1 = cof(m, 1, 0), c2 = cof(m, 2, 0);
  const float det = c0 * m[0] + c1 * m[3] + c2 * m[6];
  const float invdet = 1.0f / det;
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) out[i * 3 + j] = cof(m, j, i) * invdet;
}

__device__ __forceinline__ void mul3(const float* a, const float* b, float* r) {
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j)
      r[i * 3 + j] = a[i * 3 + 0] * b[0 * 3 + j] + a[i * 3 + 1] * b[1 * 3 + j] + a[i * 3 + 2] * b[2 * 3 + j];
}

// optimization/conditioner.hpp:66-72.
__device__ __forceinline__ void condition(float& x, float& y, const float* T) {
  const float c0 = T[0] * x + T[1] * y + T[2] * 1.f;
  const float c1 = T[3] * x + T[4] * y + T[5] * 1.f;
  const float c2 = T[6] * x + T[7] * y + T[8] * 1.f;
  x = c0 / c2;
  y = c1 / c2;
}

// x / n, correctly rounded, for a float x and an integer 1 <= n <=
// kMaxSamples, from inv_n = 1/n rounded to double: the double product is
// within 2^-52 (relative) of x/n; x/n, a 24-bit significand over an
// integer below 2^8, is never a midpoint between two floats and lies more
// than 2^-33 (relative) away from every midpoint, so rounding the product to
// float rounds x/n.  The argument needs a result in the normal range: for a
// subnormal one (div_n_tiny) the caller takes the division.
__device__ __forceinline__ double div_n_product(float x, double inv_n) { return (double)x * inv_n; }
__device__ __forceinline__ bool div_n_tiny(double p) { return p != 0.0 && fabs(p) < 0x1p-126; }

// n in float and 1/n in double for n = 0 .. kMaxSamples (1/0 unused).  Every
// lane is at the same count, so these are scalar loads, a batch at a time.
struct CountTable {
  double inv[kMaxSamples + 1];
  float n[kMaxSamples + 1];
  constexpr CountTable() : inv{}, n{} {
    for (int q = 0; q <= kMaxSamples; ++q) {
      inv[q] = q ? 1.0 / (double)q : 0.0;
      n[q] = (float)q;
    }
  }
};
__constant__ const CountTable kCount;

// boost::accumulators immediate mean and variance, one non-negative value at
// a time (at most kMaxSamples; cnt, the same in every lane, counts this one).
// With EXACT false every quotient is a double product.  That is the division
// while no nonzero value or squared deviation is below 2^-100 (the mean and
// the variance then stay above 2^-120 or zero); `low` remembers the smallest
// of them (their bits less one, so that zero is the largest), and the caller
// runs the values again through the dividing form where it was too small:
// the chain itself has no test and no branch.
template <bool EXACT>
struct MeanVar {
  float mean = 0.f, var = 0.f;
  uint32_t low = ~0u;
  __device__ __forceinline__ bool tiny() const { return low < 0x0d800000u; }  // 2^-100
  __device__ __forceinline__ void add(float v, int cnt) {
    const float before = kCount.n[cnt - 1];
    const float xm = mean * before + v;
    if (EXACT) mean = xm / (float)cnt;
    else mean = (float)div_n_product(xm, kCount.inv[cnt]);
    if (cnt > 1) {
      const float t = v - mean;
      const float xa = var * before, xb = t * t;
      if (EXACT) {
        var = xa / (float)cnt + xb / before;
      } else {
        var = (float)div_n_product(xa, kCount.inv[cnt]) + (float)div_n_product(xb, kCount.inv[cnt - 1]);
        low = min(low, min(__float_as_uint(xb) - 1u, __float_as_uint(v) - 1u));
      }
    } else if (!EXACT) {
      low = min(low, __float_as_uint(v) - 1u);
    }
  }
};

// Identification.cpp:396-459: the n samples of a cut, kWalkBatch at a time.
// Positions follow the reference's running sums, which are monotone in x and
// in y: a batch lies inside the image when its last sample (and the cut's
// first) does.  The image reads of a batch are issued together.
constexpr int kWalkBatch = 20;
struct WalkBatch {
  float fx[kWalkBatch], fy[kWalkBatch];
  uint32_t q[kWalkBatch];
  __device__ __forceinline__ float value(int t) const { return bilinear2(fx[t], fy[t], q[t]) / 2; }
};
struct CutWalk {
  float x, y, stepX, stepY;
  bool inside;  // every sample so far
  __device__ __forceinline__ CutWalk(const Img& im, float sx, float sy, float ex, float ey, float begin,
                                     float end, int n) {
    float xe, ye;
    const float diffX = ex - sx, diffY = ey - sy;
    if (begin != 0.f) {
      x = sx + diffX * begin;
      y = sy + diffY * begin;
    } else {
      x = sx;
      y = sy;
    }
    if (end != 1.f) {
      xe = sx + diffX * end;
      ye = sy + diffY * end;
    } else {
      xe = ex;
      ye = ey;
    }
    stepX = (xe - x) / ((float)n - 1.f);
    stepY = (ye - y) / ((float)n - 1.f);
    inside = in(im, x, y);
  }
  static __device__ __forceinline__ bool in(const Img& im, float x, float y) {
    return x >= 1.f && x < (float)(im.w - 1) && y >= 1.f && y < (float)(im.h - 1);
  }
  // The next `live` samples (1 <= live <= kWalkBatch, the same in every
  // lane); nothing is read once a sample was outside.
  __device__ __forceinline__ void fetch(const Img& im, int live, WalkBatch& b) {
    float px[kWalkBatch], py[kWalkBatch];
    float lx = x, ly = y;
#pragma unroll
    for (int t = 0; t < kWalkBatch; ++t) {
      px[t] = t < live ? x : px[0];
      py[t] = t < live ? y : py[0];
      lx = t < live ? x : lx;
      ly = t < live ? y : ly;
      x += stepX;
      y += stepY;
    }
    inside = inside && in(im, lx, ly);
    if (!inside) return;
#pragma unroll
    for (int t = 0; t < kWalkBatch; ++t) {
      b.q[t] = im.quad24((uint32_t)(int)px[t], (uint32_t)(int)py[t]);
      b.fx[t] = __builtin_amdgcn_fractf(px[t]);
      b.fy[t] = __builtin_amdgcn_fractf(py[t]);
    }
  }
};

// The mean and variance of a cut's samples, the next batch's reads in flight
// while one is added up.  False when a sample falls outside the image.
template <bool EXACT>
__device__ __forceinline__ bool cut_stats(const Img& im, float cx, float cy, float sx, float sy,
                                          float begin, int n, MeanVar<EXACT>& mv) {
  CutWalk walk(im, cx, cy, sx, sy, begin, 1.f, n);
  WalkBatch a, b;
  auto take = [&](const WalkBatch& w, int i0) {
    if (i0 + kWalkBatch <= n) {
#pragma unroll
      for (int t = 0; t < kWalkBatch; ++t) mv.add(w.value(t), i0 + t + 1);
    } else {
#pragma unroll
      for (int t = 0; t < kWalkBatch; ++t)
        if (i0 + t < n) mv.add(w.value(t), i0 + t + 1);
    }
  };
  walk.fetch(im, min(kWalkBatch, n), a);
  for (int i0 = 0; i0 < n && walk.inside; i0 += 2 * kWalkBatch) {
    if (i0 + kWalkBatch < n) walk.fetch(im, min(kWalkBatch, n - i0 - kWalkBatch), b);
    if (!walk.inside) return false;
    take(a, i0);
    if (i0 + kWalkBatch >= n) break;
    if (i0 + 2 * kWalkBatch < n) walk.fetch(im, min(kWalkBatch, n - i0 - 2 * kWalkBatch), a);
    if (!walk.inside) return false;
    take(b, i0 + kWalkBatch);
  }
  return walk.inside;
}

constexpr float kRefineKernels[3][9] = {
    {-0.0000f, -0.0003f, -0.1065f, -0.7863f, .0f, 0.7863f, 0.1065f, 0.0003f, 0.0000f},
    {-0.0044f, -0.0540f, -0.2376f, -0.3450f, .0f, 0.3450f, 0.2376f, 0.0540f, 0.0044f},
    {-0.0366f, -0.1113f, -0.1801f, -0.1594f, .0f, 0.1594f, 0.1801f, 0.1113f, 0.0366f}};

// The strongest response of each refinement kernel along a signal of N
// samples (value(i); beyond the ends its first and last), and where
// (Identification.cpp:630-657).  A tap of weight zero adds nothing to a sum
// and is left out.
template <int N, class F>
__device__ __forceinline__ void edge_responses(const F& value, float* key, float* loc) {
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    float best = 0.f;
    int bi = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      float tmp = 0;
#pragma unroll
      for (int j = 0; j < 9; ++j)
        if (kRefineKernels[k][j] != 0.f) {
          const int r = i - 4 + j;
          tmp += value(r < 0 ? 0 : r >= N ? N - 1 : r) * kRefineKernels[k][j];
        }
      if (i == 0 || tmp > best) {
        best = tmp;
        bi = i;
      }
    }
    key[k] = best;
    loc[k] = (float)bi;
  }
}

// (the same for any n, in a loop)
template <class F>
__device__ __forceinline__ void edge_responses_any(int n, const F& value, float* key, float* loc) {
  for (int k = 0; k < 3; ++k) {
    float best = 0.f;
    int bi = 0;
    for (int i = 0; i < n; ++i) {
      float tmp = 0;
      for (int j = 0; j < 9; ++j) {
        const int r = i - 4 + j;
        tmp += value(r < 0 ? 0 : r >= n ? n - 1 : r) * kRefineKernels[k][j];
      }
      if (i == 0 || tmp > best) {
        best = tmp;
        bi = i;
      }
    }
    key[k] = best;
    loc[k] = (float)bi;
  }
}

// One thread per outer point (n <= kMaxOuterPoints = blockDim.x).  The
// counts, the maximum variance and the candidates' ranks come from block
// reductions and a ballot scan; the uniform-stride pick of
// selectCutCheapUniform (Identification.cpp:546-601) is one lane per
// selected cut.  Bound by the statistics' chain, one instruction per 5.3
// cycles from a wavefront alone on its SIMD: with tests and LDS reciprocals
// in the chain 43.6 us at 1920x1080 (55 markers) and 39 at 640x480, without
// them 28 and 23.
constexpr int kSelectBlock = 256;
static_assert(kSelectBlock >= kMaxOuterPoints, "one lane per outer point");

__global__ __launch_bounds__(kSelectBlock) void k_select_cuts(const SelectJobDev* __restrict__ jobs,
                                                              const float4* __restrict__ pts,
                                                              float start_sig, int n_samples, int n_ref,
                                                              int select_max, SelectOutDev* __restrict__ out) {
  constexpr int NW = kSelectBlock / 64;
  __shared__ float4 stop[kMaxOuterPoints];
  __shared__ int idx_of_rank[kMaxOuterPoints];
  __shared__ int w_cnt[NW], w_cand[NW];
  __shared__ float w_max[NW];
  __shared__ float ref_sig[kMaxRefineSamples][kSelectBlock];  // the thread's refinement cut
  const SelectJobDev J = jobs[blockIdx.x];
  const Img im{J.quad, J.iw, J.ih};
  const int n = J.n_outer;
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
  bool valid = false;
  float var = 0.f;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  if (t < n) {
    s = pts[J.pt_offset + t];
    MeanVar<false> mv;
    valid = cut_stats(im, J.cx, J.cy, s.x, s.y, start_sig, n_samples, mv);
    var = mv.var;
    if (valid && mv.tiny()) {  // the same walk again, dividing
      MeanVar<true> me;
      cut_stats(im, J.cx, J.cy, s.x, s.y, start_sig, n_samples, me);
      var = me.var;
    }
  }
  // number of collected cuts and their largest variance
  {
    int c = valid ? 1 : 0;
    float mx = valid ? var : -FLT_MAX;
    for (int o = 32; o > 0; o >>= 1) {
      c += __shfl_xor(c, o, 64);
      mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    }
    if (lane == 0) {
      w_cnt[wid] = c;
      w_max[wid] = mx;
    }
  }
  __syncthreads();
  int nc = 0;
  float var_max = -FLT_MAX;
  for (int w = 0; w < NW; ++w) {
    nc += w_cnt[w];
    var_max = fmaxf(var_max, w_max[w]);
  }
  bool cand = false;
  if (valid) {
    // pointOnEllipse (EllipseFromPoints.cpp:29-49), double like the C cos/sin
    {
      const float x = s.x - J.cx, y = s.y - J.cy;
      float tx = (float)((double)x * J.ca + (double)y * J.sa);
      float ty = (float)(-(double)x * J.sa + (double)y * J.ca);
      const float cs = (float)sqrt((double)(tx * tx / (J.ea * J.ea) + ty * ty / (J.eb * J.eb)));
      tx /= cs;
      ty /= cs;
      s.x = (float)((double)tx * J.ca - (double)ty * J.sa + (double)J.cx);
      s.y = (float)((double)tx * J.sa + (double)ty * J.ca + (double)J.cy);
    }
    // outerEdgeRefinement (Identification.cpp:604-657)
    const float len = (float)(3.0 * 1.4142135623730951 * (double)J.scale);
    const float half = len / 2.f;
    const float gn = sqrt_rn(s.z * s.z + s.w * s.w);
    const float gdx = s.z / gn, gdy = s.w / gn;
    const float hx = half * gdx, hy = half * gdy;
    const float psx = s.x - hx, psy = s.y - hy;
    const float pex = s.x + half * gdx, pey = s.y + half * gdy;
    CutWalk walk(im, psx, psy, pex, pey, 0.f, 1.f, n_ref);
    float key[3], loc[3];
    if (n_ref == kWalkBatch) {
      // (the default: the signal stays in registers)
      WalkBatch w;
      walk.fetch(im, kWalkBatch, w);
      if (walk.inside) {
        float v[kWalkBatch];
#pragma unroll
        for (int i = 0; i < kWalkBatch; ++i) v[i] = w.value(i);
        edge_responses<kWalkBatch>([&](int i) { return v[i]; }, key, loc);
      }
    } else {
      for (int i0 = 0; i0 < n_ref && walk.inside; i0 += kWalkBatch) {
        WalkBatch w;
        walk.fetch(im, min(kWalkBatch, n_ref - i0), w);
        if (!walk.inside) break;
#pragma unroll
        for (int i = 0; i < kWalkBatch; ++i)
          if (i0 + i < n_ref) ref_sig[i0 + i][t] = w.value(i);
      }
      if (walk.inside) edge_responses_any(n_ref, [&](int i) { return ref_sig[i][t]; }, key, loc);
    }
    if (walk.inside) {
      // std::map<float,float> insert (first of equal keys kept), then the largest key
      int b = 0;
      for (int k = 1; k < 3; ++k)
        if (key[k] > key[b]) b = k;
      const float step = len / ((float)n_ref - 1.f);
      s.x = psx + step * loc[b] * gdx;
      s.y = psy + step * loc[b] * gdy;
      cand = var / var_max > 0.5f;
    }
  }
  // rank of each candidate among the collected cuts, in outer-point order
  const uint64_t ball = __ballot(cand);
  const int in_wave = __popcll(ball & ((1ull << lane) - 1ull));
  if (lane == 0) w_cand[wid] = __popcll(ball);
  if (t < n) stop[t] = s;
  __syncthreads();
  int before = 0, ni = 0;
  for (int w = 0; w < NW; ++w) {
    if (w < wid) before += w_cand[w];
    ni += w_cand[w];
  }
  if (cand) idx_of_rank[before + in_wave] = t;
  __syncthreads();
  // uniform stride over the candidates: pick k takes rank (int)(k * step)
  const int select = min(select_max, nc);
  const float step = fmaxf(1.f, (float)ni / (float)select);
  if (t < select) {
    const int at = (int)((float)t * step);
    if (at < ni) out[blockIdx.x].stops[t] = stop[idx_of_rank[at]];
  }
  // (out is host memory: written after the last barrier, which would
  // otherwise wait for the stores to reach the host)
  if (t == 0) {
    int nsel = 0;
    while (nsel < select && (int)((float)nsel * step) < ni) ++nsel;
    out[blockIdx.x].n_collected = nc;
    out[blockIdx.x].n_selected = nsel;
  }
}

// ---------------------------------------------------------------------------
// Centre refinement.  An iteration of the grid search evaluates the grid
// points around the current centre: per point its homography, the samples of
// every selected cut and the residual sum_{k<l} sum_i (s_ki - s_li)^2 over
// its valid cuts, taken per sample as m S2_i - S1_i^2 (S1_i and S2_i the sum
// and the sum of squares of the valid cuts' samples, in double, in cut
// order; summed in sample order by chunks of kRefineChunk).  The centre then
// moves to the first minimum, as the reference's loop does.  A cut that
// leaves the image at a grid point is invalid there and at every later point
// (Identification.cpp:264-273).
//
// The search is bound by the instruction issue of the sampling (per sample
// two quotients, a projective map and a bilinear blend whose rounding is the
// reference's): a cut proven inside the image needs no bounds test, its two
// quotients share one reciprocal (div2_rn) and the halving of the samples is
// left to the end of the sum (an exact power of two).
constexpr int kFinalBlock = 1024;  // one block per marker: every loop of the read-out in one pass
constexpr int kRefineChunk = 10;  // samples of a cut whose image reads are in flight together
constexpr int G2MAX = kMaxGrid * kMaxGrid;
constexpr int kXcds = 8;               // accelerator complex dies of the MI355X

// getNearbyPoints point g + computeHomographyFromEllipseAndImagedCenter
// (Identification.cpp:739-798, 1071-1109) and the inverse.
__device__ void grid_homography(const RefineJobDev& J, float cur_x, float cur_y, float neighbour,
                                int g, int grid_n, float* Hf, float* Hi, float& qx, float& qy) {
  const int i = g / grid_n, j = g - i * grid_n;
  const float ns = neighbour * J.grid_scale;
  float cx = cur_x, cy = cur_y;
  condition(cx, cy, J.cond);
  const float halfWidth = ns / 2.f;
  const float stepSize = ns / (float)(grid_n - 1);
  qx = cx - halfWidth + (float)i * stepSize;
  qy = cy - halfWidth + (float)j * stepSize;
  condition(qx, qy, J.cond_inv);
  float xc, yc;
  apply_h(xc, yc, J.t_can, qx, qy);
  const float Q11 = J.Q11, Q22 = J.Q22, Q33 = J.Q33;
  float H[9];
  H[0] = Q33;              H[1] = Q22 * xc * yc;        H[2] = -Q33 * xc;
  H[3] = 0.f;              H[4] = -Q11 * xc * xc - Q33; H[5] = -Q33 * yc;
  H[6] = -Q11 * xc;        H[7] = Q22 * yc;             H[8] = -Q33;
  const float d0 = sqrt_rn((Q22 * Q33 / Q11 * (Q11 * xc * xc + Q22 * yc * yc + Q33)));
  const float d1 = Q33;
  const float d2 = sqrt_rn(-Q22 * (Q11 * xc * xc + Q33));
  for (int r = 0; r < 3; ++r) {
    H[r * 3 + 0] *= d0;
    H[r * 3 + 1] *= d1;
    H[r * 3 + 2] *= d2;
  }
  mul3(J.t_inv_can, H, Hf);
  inverse3(Hf, Hi);
}

// extractSignalUsingHomography (Identification.cpp:216-280), first part: the
// stop back-projected by Hi, the sample positions from begin*stop to
// end*stop in the marker plane as the reference's running sums.
__host__ __device__ constexpr int chunks_of(int n_samples) {
  return (n_samples + kRefineChunk - 1) / kRefineChunk;
}
// The residual's terms are summed kSumChunk samples at a time, then the sums.
constexpr int kSumChunk = 5;
static_assert(kRefineChunk % kSumChunk == 0, "whole sums per chunk");
__host__ __device__ constexpr int sum_chunks_of(int n_samples) {
  return (n_samples + kSumChunk - 1) / kSumChunk;
}
constexpr int kMaxSumChunks = sum_chunks_of(kMaxSamples);
static_assert(kMaxSumChunks <= kMaxRefineSums, "the work buffer's sums");

// A cut's samples: their number n and 1/(n - 1) in double.
struct Samples {
  int n;
  double inv_steps;
};

// x / (n - 1), correctly rounded (div_n_product).
__device__ __forceinline__ float per_step(float x, const Samples& ns) {
  const double p = div_n_product(x, ns.inv_steps);
  return div_n_tiny(p) ? x / ((float)ns.n - 1.f) : (float)p;
}

// The first sample position and the step.
__device__ __forceinline__ void cut_walk_begin(const float* Hi, float2 stop, float begin_sig,
                                               float end_sig, const Samples& ns, float2& first,
                                               float2& step) {
  float bx, by;
  apply_h(bx, by, Hi, stop.x, stop.y);
  float xs, ys, xe, ye;
  if (begin_sig != 0.f) {
    xs = bx * begin_sig;
    ys = by * begin_sig;
  } else {
    xs = 0;
    ys = 0;
  }
  if (end_sig != 1.f) {
    xe = bx * end_sig;
    ye = by * end_sig;
  } else {
    xe = bx;
    ye = by;
  }
  step.x = per_step(xe - xs, ns);
  step.y = per_step(ye - ys, ns);
  first = make_float2(xs, ys);
}

// Second part for the next N samples of a cut from position p on (advanced
// past them): mapped by H, twice the half-bilinear value into val[].
// kInside cuts only, whole chunks.
template <int N>
__device__ __forceinline__ void sample_inside(const Img& im, const float* H, float2& p, float2 step,
                                              float (&val)[N]) {
  float fx[N], fy[N];
  uint32_t qd[N];
#pragma unroll
  for (int t = 0; t < N; ++t) {
    const float u = H[0] * p.x + H[1] * p.y + H[2];
    const float v = H[3] * p.x + H[4] * p.y + H[5];
    const float ww = H[6] * p.x + H[7] * p.y + H[8];
    float xr, yr;
    div2_rn(u, v, ww, xr, yr);
    qd[t] = im.quad24((uint32_t)(int)xr, (uint32_t)(int)yr);
    fx[t] = __builtin_amdgcn_fractf(xr);  // positions are positive: x - (int)x
    fy[t] = __builtin_amdgcn_fractf(yr);
    p.x += step.x;
    p.y += step.y;
  }
#pragma unroll
  for (int t = 0; t < N; ++t) val[t] = bilinear2(fx[t], fy[t], qd[t]);
}

// The same for any cut and the last, partial chunk (`live` samples left): 0
// for a sample outside the image; returns whether one is.  BATCH samples'
// reads are in flight together.
template <int N, int BATCH>
__device__ __forceinline__ bool sample_any(const Img& im, const float* H, float2& p, float2 step,
                                           int live, float* val) {
  static_assert(N % BATCH == 0, "whole load batches per chunk");
  const float xmax = (float)(im.w - 1), ymax = (float)(im.h - 1);
  bool oob = false;
#pragma unroll
  for (int t0 = 0; t0 < N; t0 += BATCH) {
    float fx[BATCH], fy[BATCH];
    bool in[BATCH];
    uint32_t qd[BATCH];
#pragma unroll
    for (int t = 0; t < BATCH; ++t) {
      float xr, yr;
      apply_h(xr, yr, H, p.x, p.y);
      in[t] = t0 + t < live && xr >= 0.f && xr < xmax && yr >= 0.f && yr < ymax;
      oob |= t0 + t < live && !in[t];
      // an outside sample reads pixel (0, 0), so the loads need no branch
      qd[t] = in[t] ? im.quad((int)xr, (int)yr) : im.quad(0, 0);
      fx[t] = xr - (int)xr;
      fy[t] = yr - (int)yr;
      p.x += step.x;
      p.y += step.y;
    }
#pragma unroll
    for (int t = 0; t < BATCH; ++t) val[t0 + t] = in[t] ? bilinear2(fx[t], fy[t], qd[t]) : 0.f;
  }
  return oob;
}

// Whether a sample of a cut falls outside the image (the kUnsure cuts).
__device__ bool samples_leave(const Img& im, const float* H, const float* Hi, float2 stop,
                              float begin_sig, float end_sig, const Samples& ns) {
  float2 p, step;
  cut_walk_begin(Hi, stop, begin_sig, end_sig, ns, p, step);
  const float xmax = (float)(im.w - 1), ymax = (float)(im.h - 1);
  for (int i = 0; i < ns.n; ++i) {
    float xr, yr;
    apply_h(xr, yr, H, p.x, p.y);
    if (!(xr >= 0.f && xr < xmax && yr >= 0.f && yr < ymax)) return true;
    p.x += step.x;
    p.y += step.y;
  }
  return false;
}

// A grid point's residual from its chunks' sums (those of the doubled
// samples); FLT_MAX (never picked) below two valid cuts.
__device__ __forceinline__ float point_residual(const double* part, int nchunk, int m) {
  double sum = part[0];
#pragma unroll
  for (int c = 1; c < kMaxSumChunks; ++c)
    if (c < nchunk) sum += part[c];
  return m < 2 ? FLT_MAX : (float)(0.25 * sum) / (float)(m * (m - 1) / 2);
}

__device__ __forceinline__ uint32_t cut_bits(int nc) { return nc >= 32 ? ~0u : (1u << nc) - 1u; }

// What the reference's loop does after evaluating a grid, by wavefront 0
// with lane g on grid point g: the first minimum among the points with a
// residual below FLT_MAX becomes the centre, the neighbourhood shrinks;
// without one the marker has failed.  `sticky`: the cuts flagged by the end
// of the iteration.
__device__ __forceinline__ void select_state(bool on, float res, float gx, float gy, uint32_t sticky,
                                             const RefineStateDev& prev, int grid_n,
                                             RefineStateDev& S) {
  const bool pickable = on && res < FLT_MAX;
  float key = pickable ? res : INFINITY;
  int idx = pickable ? (int)threadIdx.x : 64;
  for (int o = 32; o > 0; o >>= 1) {
    const float k2 = __shfl_xor(key, o, 64);
    const int i2 = __shfl_xor(idx, o, 64);
    if (k2 < key || (k2 == key && i2 < idx)) {
      key = k2;
      idx = i2;
    }
  }
  const int b = idx < 64 ? idx : -1;
  const float bx = __shfl(gx, b < 0 ? 0 : b, 64), by = __shfl(gy, b < 0 ? 0 : b, 64);
  if (threadIdx.x == 0) {
    RefineStateDev n = prev;
    n.sticky = sticky;
    if (b < 0) {
      n.ok = 0;
    } else {
      n.ok = 1;
      n.best_g = b;
      n.cx = bx;
      n.cy = by;
      n.neighbour = prev.neighbour / (float)((grid_n - 1) / 2);
      n.min_res = key;
    }
    S = n;
  }
}

__device__ __forceinline__ RefineStateDev first_state(const RefineJobDev& J) {
  RefineStateDev s;
  s.cx = J.c0x;
  s.cy = J.c0y;
  s.neighbour = J.neighbour0;
  s.min_res = FLT_MAX;
  s.ok = 1;
  s.best_g = 0;
  s.sticky = 0;
  s.pad = 0;
  return s;
}

// The state a marker starts iteration `it` with: the job's start for the
// first one, otherwise the selection over the previous launch's records
// (buffers of parity (it - 1) & 1).  In two steps, so that the records are on
// their way while the block reads its job: lane g of wavefront 0 loads grid
// point g's, then the whole block takes the state.
struct PointRecord {
  RefineStateDev prev;
  RefinePointDev point;
  double part[kMaxSumChunks];
};
__device__ __forceinline__ void load_records(int it, int m, int n_jobs, int n_samples, int grid_n,
                                             const RefineWork& W, PointRecord& r) {
  if (it == 0 || threadIdx.x >= 64) return;
  const int pb = (it - 1) & 1, g = (int)threadIdx.x < grid_n * grid_n ? threadIdx.x : 0;
  const size_t at = ((size_t)pb * n_jobs + m) * G2MAX + g;
  const int last = sum_chunks_of(n_samples) - 1;
  r.prev = W.state[(size_t)pb * n_jobs + m];
  r.point = W.points[at];
#pragma unroll
  for (int c = 0; c < kMaxSumChunks; ++c) r.part[c] = W.part[at * kMaxRefineSums + min(c, last)];
}
__device__ void state_at(const RefineJobDev& J, int it, int n_samples, int grid_n,
                         const PointRecord& r, RefineStateDev& S) {
  const int tid = threadIdx.x;
  if (it == 0) {
    if (tid == 0) S = first_state(J);
  } else if (tid < 64) {
    const int G2 = grid_n * grid_n;
    const float res = point_residual(r.part, sum_chunks_of(n_samples),
                                     __popc(~r.point.flagged & cut_bits(J.n_cuts)));
    if (r.prev.ok) {
      select_state(tid < G2, res, r.point.gx, r.point.gy, __shfl(r.point.flagged, G2 - 1, 64),
                   r.prev, grid_n, S);
    } else if (tid == 0) {
      S = r.prev;
    }
  }
  __syncthreads();
}

// A marker's centre, its job's start when no grid point was readable.
__device__ __forceinline__ void put_center(const RefineJobDev& J, bool found, const RefineStateDev& S,
                                           int m, float2* centers, int* found_out) {
  centers[m] = found ? make_float2(S.cx, S.cy) : make_float2(J.c0x, J.c0y);
  if (found_out) found_out[m] = found ? 1 : 0;
}

// Two kernels run the search, with the same results: k_refine_iter, one
// launch per iteration, spreads few markers over the chip; k_refine_search,
// a block per marker, does the least work for many.
//
// k_refine_iter: iteration `it`, block (b, m) on chunks [b * per, (b + 1) *
// per) of marker m's samples -- the residual is a sum over samples, so a
// chunk's share needs no other block.  Every block derives the iteration's
// start from the records the previous launch left (the last selection is the
// read-out kernel's).
//
// A lane takes one cut at one grid point and walks its samples, the grid
// points side by side: the 25 lanes of a cut sample within a pixel or a few
// of each other, so a wavefront's load touches few cache lines.  (With a
// block per grid point the lanes of a load lay on 57 different lines, and
// the L1's tag lookups, one line per cycle, took as long as the arithmetic.)
// The chunk's samples meet in LDS, double-buffered with one barrier per
// chunk; two lanes per grid point and sample then take the sum and the sum
// of squares over the cuts.
constexpr int kMaxRefineBlock = (G2MAX * kMaxCuts + 63) / 64 * 64;

__global__ __launch_bounds__(kMaxRefineBlock) void k_refine_iter(
    const RefineJobDev* __restrict__ jobs, int it, int per, Samples ns, int grid_n, RefineWork W) {
  extern __shared__ float sig_lds[];  // [buffer][cut][grid point][sample of the chunk], doubled samples
  __shared__ float gH[G2MAX][9], gHi[G2MAX][9];
  __shared__ float2 center[G2MAX];
  __shared__ double term[2][G2MAX * kRefineChunk];
  __shared__ RefineStateDev S;
  __shared__ uint32_t oob[G2MAX];
  __shared__ int any_oob;

  const int n_samples = ns.n, tid = threadIdx.x, G2 = grid_n * grid_n, nchunk = chunks_of(n_samples);
  // Workgroups are dealt to the 8 XCDs in turn, each XCD with its own L2:
  // renumber them so that an XCD runs consecutive (chunks, marker) pairs,
  // i.e. whole markers, and each marker's image area is fetched into one L2
  // only.
  const int n_jobs = gridDim.y;
  int b, m;
  {
    const int n = gridDim.x * gridDim.y, hw = blockIdx.y * gridDim.x + blockIdx.x;
    const int x = hw % kXcds, k = hw / kXcds, q = n / kXcds, r = n % kXcds;
    const int logical = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + k;
    b = logical % gridDim.x;
    m = logical / gridDim.x;
  }
  const RefineJobDev& J = jobs[m];
  PointRecord rec;
  load_records(it, m, n_jobs, n_samples, grid_n, W, rec);
  const int k = tid / G2, g = tid - k * G2;  // the lane's cut and grid point
  const float2 stop = J.stops[min(k, kMaxCuts - 1)];
  const int nc = J.n_cuts, n_iter = J.n_iter;
  const Img im{J.quad, J.iw, J.ih};
  const int c0 = b * per, c1 = min(nchunk, c0 + per);
  const int width = G2 * kRefineChunk, buf = nc * width;
  if (it >= n_iter) return;
  state_at(J, it, n_samples, grid_n, rec, S);
  if (b == 0 && tid == 0) W.state[(size_t)(it & 1) * n_jobs + m] = S;
  if (!S.ok) return;
  if (tid < G2) {
    float Hf[9], Hi[9], qx, qy;
    grid_homography(J, S.cx, S.cy, S.neighbour, tid, grid_n, Hf, Hi, qx, qy);
    for (int r = 0; r < 9; ++r) {
      gH[tid][r] = Hf[r];
      gHi[tid][r] = Hi[r];
    }
    center[tid] = make_float2(qx, qy);
    oob[tid] = 0;
    if (b == 0 && it + 1 == J.n_iter) {  // the read-out's, should this point be chosen
      RefineHomDev& GH = W.hom[(size_t)m * G2MAX + tid];
      for (int r = 0; r < 9; ++r) {
        GH.H[r] = Hf[r];
        GH.Hi[r] = Hi[r];
      }
    }
  }
  if (tid == blockDim.x - 1) any_oob = 0;
  __syncthreads();
  // place the cut, and walk it to the block's first chunk
  float H[9];
  float2 p = make_float2(0.f, 0.f), step = p;
  bool on = k < nc, inside = false;
  if (on) {
    float Hi[9];
    for (int r = 0; r < 9; ++r) {
      H[r] = gH[g][r];
      Hi[r] = gHi[g][r];
    }
    CutPlace at = cut_place(H, Hi, stop.x, stop.y, J.begin_sig, J.end_sig, J.iw, J.ih);
    inside = at == kInside;
    if (at == kUnsure && samples_leave(im, H, Hi, stop, J.begin_sig, J.end_sig, ns)) at = kOutside;
    if (at == kOutside) {
      atomicOr(&oob[g], 1u << k);
      any_oob = 1;
      on = false;
    } else {
      cut_walk_begin(Hi, stop, J.begin_sig, J.end_sig, ns, p, step);
      for (int q = 0; q < c0; ++q) {
#pragma unroll
        for (int t = 0; t < kRefineChunk; ++t) {
          p.x += step.x;
          p.y += step.y;
        }
      }
    }
  }
  // the cuts flagged by grid point q: before the iteration, at q or before it
  auto flags = [&](int q) {
    uint32_t f = S.sticky;
    if (any_oob)
      for (int r = 0; r <= q; ++r) f |= oob[r];
    return f;
  };
  auto chunk_sum = [&](int c) {  // lane g: grid point g's share of chunk c
    const double* v = &term[c & 1][tid * kRefineChunk];
    double* out = W.part + (((size_t)(it & 1) * n_jobs + m) * G2MAX + tid) * kMaxRefineSums +
                  c * (kRefineChunk / kSumChunk);
#pragma unroll
    for (int t0 = 0; t0 < kRefineChunk; t0 += kSumChunk) {
      double sum = 0.0;
#pragma unroll
      for (int t = t0; t < t0 + kSumChunk; ++t)
        if (c * kRefineChunk + t < n_samples) sum += v[t];
      if (c * kRefineChunk + t0 < n_samples) out[t0 / kSumChunk] = sum;
    }
  };
  uint32_t valid = 0;
  for (int c = c0; c < c1; ++c) {
    float* sig = sig_lds + (per > 1 ? (c & 1) * buf : 0);
    if (on) {
      const int live = n_samples - c * kRefineChunk;
      float val[kRefineChunk];
      if (inside && live >= kRefineChunk) sample_inside(im, H, p, step, val);
      else sample_any<kRefineChunk, 1>(im, H, p, step, live, val);
      float* out = sig + tid * kRefineChunk;  // (cut, grid point) = lane
#pragma unroll
      for (int t = 0; t < kRefineChunk; ++t) out[t] = val[t];
    }
    __syncthreads();
    if (c > c0 && tid < G2) chunk_sum(c - 1);
    // lanes 2w and 2w + 1: sum and sum of squares at (grid point, sample) w
    // over the valid cuts, in cut order, kRowBatch reads in flight
    constexpr int kRowBatch = 8;
    const int w = tid >> 1;
    const bool squares = tid & 1;
    if (c == c0) valid = ~flags(min(w / kRefineChunk, G2 - 1)) & cut_bits(nc);
    if (w < width) {
      double s = 0.0;
      for (int k0 = 0; k0 < nc; k0 += kRowBatch) {
        float v[kRowBatch];
#pragma unroll
        for (int j = 0; j < kRowBatch; ++j) v[j] = sig[min(k0 + j, nc - 1) * width + w];
#pragma unroll
        for (int j = 0; j < kRowBatch; ++j)
          if (k0 + j < nc && ((valid >> (k0 + j)) & 1u)) {
            const double d = (double)v[j];
            s += squares ? d * d : d;
          }
      }
      const double other = __shfl_xor(s, 1, 64);
      if (squares) term[c & 1][w] = (double)__popc(valid) * s - other * other;
    }
  }
  __syncthreads();
  if (tid < G2) chunk_sum(c1 - 1);
  if (b == 0 && tid < G2)
    W.points[((size_t)(it & 1) * n_jobs + m) * G2MAX + tid] =
        RefinePointDev{center[tid].x, center[tid].y, flags(tid), 0u};
}

// The whole search in one block per marker (at most `iters` iterations; with
// `centers`, the centre reached is all that is kept).  A lane owns one chunk of
// kSumChunk samples at one grid point, the grid points side by side as in
// k_refine_iter, and keeps the sums over the cuts in registers, so no sample
// goes through LDS; B >= grid_n^2 * sum chunks.  The cuts' running sums are
// laid out kSearchCuts cuts at a time, which bounds their LDS.
constexpr int kSearchCuts = 6;

template <int B>
__global__ __launch_bounds__(B) __attribute__((amdgpu_waves_per_eu(6))) void k_refine_search(
    const RefineJobDev* __restrict__ jobs, Samples ns, int grid_n, int iters, RefineWork W,
    float2* __restrict__ centers, int* __restrict__ found) {
  __shared__ float2 start[kSearchCuts][kMaxSumChunks][G2MAX], step[kSearchCuts][G2MAX];
  __shared__ double part[G2MAX][kMaxSumChunks];
  __shared__ float gH[G2MAX][9], gHi[G2MAX][9];
  __shared__ float2 center[G2MAX];
  __shared__ uint32_t oob[G2MAX], unsure[G2MAX];
  __shared__ int any_unsure, any_oob;
  __shared__ RefineStateDev S;
  const int m = blockIdx.x, n_jobs = gridDim.x, tid = threadIdx.x, n_samples = ns.n;
  const RefineJobDev& J = jobs[m];
  const int n_iter = min(J.n_iter, iters), nc = J.n_cuts, G2 = grid_n * grid_n;
  const Img im{J.quad, J.iw, J.ih};
  const int nchunk = sum_chunks_of(n_samples);
  const int c = tid / G2, g = tid - c * G2;  // the lane's chunk and grid point
  const bool on = c < nchunk;
  const int live = n_samples - c * kSumChunk;
  if (tid == 0) S = first_state(J);
  __syncthreads();
  for (int it = 0; it < n_iter; ++it) {
    if (tid < G2) {
      float Hf[9], Hi[9], qx, qy;
      grid_homography(J, S.cx, S.cy, S.neighbour, tid, grid_n, Hf, Hi, qx, qy);
      for (int r = 0; r < 9; ++r) {
        gH[tid][r] = Hf[r];
        gHi[tid][r] = Hi[r];
      }
      center[tid] = make_float2(qx, qy);
      oob[tid] = 0;
      unsure[tid] = 0;
    }
    if (tid == B - 1) any_unsure = any_oob = 0;
    __syncthreads();
    for (int p = tid; p < G2 * nc; p += B) {
      const int k = p / G2, gp = p - k * G2;
      const float2 stop = J.stops[k];
      const CutPlace at =
          cut_place(gH[gp], gHi[gp], stop.x, stop.y, J.begin_sig, J.end_sig, J.iw, J.ih);
      if (at == kUnsure) {
        atomicOr(&unsure[gp], 1u << k);
        any_unsure = 1;
      }
      if (at == kOutside ||
          (at == kUnsure &&
           samples_leave(im, gH[gp], gHi[gp], J.stops[k], J.begin_sig, J.end_sig, ns))) {
        atomicOr(&oob[gp], 1u << k);
        any_oob = 1;
      }
    }
    __syncthreads();
    // the cuts flagged by grid point q: before the iteration, at q or before it
    auto flags = [&](int q) {
      uint32_t f = S.sticky;
      if (any_oob)
        for (int r = 0; r <= q; ++r) f |= oob[r];
      return f;
    };
    uint32_t valid = 0, slow = 0;
    float H[9];
    if (on) {
      valid = ~flags(g) & cut_bits(nc);
      slow = live < kSumChunk ? ~0u : any_unsure ? unsure[g] : 0u;
      for (int r = 0; r < 9; ++r) H[r] = gH[g][r];
    }
    double s1[kSumChunk], s2[kSumChunk];
#pragma unroll
    for (int t = 0; t < kSumChunk; ++t) s1[t] = s2[t] = 0.0;
    for (int k0 = 0; k0 < nc; k0 += kSearchCuts) {
      const int nk = min(kSearchCuts, nc - k0);
      for (int p = tid; p < G2 * nk; p += B) {
        const int k = p / G2, gp = p - k * G2;
        float2 q, d;
        cut_walk_begin(gHi[gp], J.stops[k0 + k], J.begin_sig, J.end_sig, ns, q, d);
        for (int cc = 0; cc < nchunk; ++cc) {
          start[k][cc][gp] = q;
#pragma unroll
          for (int t = 0; t < kSumChunk; ++t) {
            q.x += d.x;
            q.y += d.y;
          }
        }
        step[k][gp] = d;
      }
      __syncthreads();
      if (on) {
        for (int k = 0; k < nk; ++k) {
          if (!((valid >> (k0 + k)) & 1u)) continue;
          float2 p = start[k][c][g];
          float val[kSumChunk];
          if (!((slow >> (k0 + k)) & 1u)) sample_inside(im, H, p, step[k][g], val);
          else sample_any<kSumChunk, 1>(im, H, p, step[k][g], live, val);
#pragma unroll
          for (int t = 0; t < kSumChunk; ++t) {
            const double d = (double)val[t];
            s1[t] += d;
            s2[t] += d * d;
          }
        }
      }
      __syncthreads();
    }
    if (on) {
      const double mv = (double)__popc(valid);
      double sum = 0.0;
#pragma unroll
      for (int t = 0; t < kSumChunk; ++t)
        if (t < live) sum += mv * s2[t] - s1[t] * s1[t];
      part[g][c] = sum;
    }
    __syncthreads();
    if (tid < 64) {
      const int q = tid < G2 ? tid : 0;
      const RefineStateDev prev = S;
      const uint32_t f = flags(q);
      const float res = point_residual(part[q], nchunk, __popc(~f & cut_bits(nc)));
      select_state(tid < G2, res, center[q].x, center[q].y, __shfl(f, G2 - 1, 64), prev, grid_n, S);
    }
    __syncthreads();
    if (!S.ok) break;
  }
  if (centers) {
    if (tid == 0) put_center(J, n_iter >= 1 && S.ok, S, m, centers, found);
    return;
  }
  if (tid == 0) W.state[(size_t)(J.n_iter & 1) * n_jobs + m] = S;
  if (n_iter > 0 && S.ok && tid < 9) {
    RefineHomDev& GH = W.hom[(size_t)m * G2MAX + S.best_g];
    GH.H[tid] = gH[S.best_g][tid];
    GH.Hi[tid] = gHi[S.best_g][tid];
  }
}

// Signals at the last iteration's best grid point, then the per-cut
// statistics and distances of orazioDistanceRobust (Identification.cpp:
// 88-160).
// The identification read-out at one homography per marker: the grid
// search's choice after its last iteration (given == null), or a given
// homography with its centre and score (given: 9 floats per job, centres 2
// per job, scores), whose out-of-bounds cuts are the ones leaving the image
// there.  Signals, median profile, orazio statistics, distance to every
// bank profile.  Led by the statistics' chain as k_select_cuts is: 37 us with
// the tests in it at 1920x1080 (55 markers), 33 without, 30 at 640x480.
__global__ __launch_bounds__(kFinalBlock) void k_refine_final(
    const RefineJobDev* __restrict__ jobs, Samples ns, int grid_n,
    const float* __restrict__ inv_ratio, int bank_rows, int bank_cols, RefineWork W,
    const float* __restrict__ given_H, const float* __restrict__ given_c,
    const double* __restrict__ given_cost, int searched, RefineOutDev* __restrict__ out,
    float* __restrict__ dist) {
  const int n_samples = ns.n;
  __shared__ float sig[kMaxCuts][kMaxSamples + 1];
  __shared__ float ordered[kMaxSamples][kMaxCuts];  // per sample, the valid cuts' values sorted
  __shared__ float bar[kMaxSamples];
  __shared__ int valid_cut[kMaxCuts];
  __shared__ int n_valid;
  __shared__ int oob_at[kMaxCuts];
  __shared__ float sH[9], sHi[9];
  __shared__ float stat_mub[kMaxCuts], stat_muw[kMaxCuts], stat_var[kMaxCuts];
  __shared__ float xs[kMaxSamples];
  __shared__ float ratio[kMaxBankRows * kMaxRatios];
  __shared__ uint8_t parity[kMaxSamples][kMaxBankRows];  // [sample][bank row]
  // a sample's term of the distance, for each ring parity
  __shared__ float term[2][kMaxCuts][kMaxSamples + 1];
  __shared__ RefineStateDev S;
  const int m = blockIdx.x, tid = threadIdx.x, n_jobs = gridDim.x;
  const RefineJobDev& J = jobs[m];
  RefineOutDev& O = out[m];
  const bool given = given_H != nullptr;
  if (!given && J.n_iter == 0) {
    if (tid == 0) O.ok = 0;
    return;
  }
  for (int q = tid; q < bank_rows * kMaxRatios; q += kFinalBlock) ratio[q] = inv_ratio[q];
  const int nc = J.n_cuts;
  if (given) {
    if (tid == 0) {
      const double c = given_cost[m];
      S.ok = c < DBL_MAX && isfinite(c);
      S.cx = given_c[2 * m];
      S.cy = given_c[2 * m + 1];
      S.min_res = (float)c;
      for (int r = 0; r < 9; ++r) sH[r] = given_H[9 * m + r];
      inverse3(sH, sHi);
    }
    if (tid < kMaxCuts) oob_at[tid] = 0;
    __syncthreads();
  } else {
    // the selection after the last iteration
    if (!searched) {
      PointRecord rec;
      load_records(J.n_iter, m, n_jobs, n_samples, grid_n, W, rec);
      state_at(J, J.n_iter, n_samples, grid_n, rec, S);
    } else {
      if (tid == 0) S = W.state[(size_t)(J.n_iter & 1) * n_jobs + m];
      __syncthreads();
    }
    if (S.ok && tid < 9) {
      const RefineHomDev& GH = W.hom[(size_t)m * G2MAX + S.best_g];
      sH[tid] = GH.H[tid];
      sHi[tid] = GH.Hi[tid];
    }
    __syncthreads();
  }
  if (!S.ok) {
    if (tid == 0) O.ok = 0;
    return;
  }
  const Img im{J.quad, J.iw, J.ih};
  const int nchunk = chunks_of(n_samples);
  for (int w = tid; w < nc * nchunk; w += kFinalBlock) {
    const int c = w / nc, k = w - c * nc, live = n_samples - c * kRefineChunk;
    float2 p, step;
    cut_walk_begin(sHi, J.stops[k], J.begin_sig, J.end_sig, ns, p, step);
    for (int q = 0; q < c * kRefineChunk; ++q) {
      p.x += step.x;
      p.y += step.y;
    }
    float val[kRefineChunk];
    if (sample_any<kRefineChunk, kRefineChunk>(im, sH, p, step, live, val) && given) atomicOr(&oob_at[k], 1);
#pragma unroll
    for (int t = 0; t < kRefineChunk; ++t)
      if (t < live) sig[k][c * kRefineChunk + t] = val[t] / 2;
  }
  __syncthreads();
  // The outputs live in host memory: they are stored after the last
  // barrier, which would otherwise wait for the stores to reach the host.
  if (given && tid < 64) {
    const uint32_t oob = (uint32_t)__ballot(tid < nc && oob_at[tid] != 0);
    if (tid == 0) S.sticky = oob;
  }
  __syncthreads();
  const uint32_t sticky = S.sticky;
  if (tid < 64) {
    const uint32_t valid = ~sticky & cut_bits(nc);
    if (tid < nc && ((valid >> tid) & 1u)) valid_cut[__popc(valid & ((1u << tid) - 1u))] = tid;
    if (tid == 0) n_valid = __popc(valid);
  }
  // orazioDistanceRobust statistics per valid cut (Identification.cpp:88-121)
  if (tid < nc && !((sticky >> tid) & 1u)) {
    // the signal is read kStatBatch samples at a time, so the reads are in
    // flight together, then consumed in order
    constexpr int kStatBatch = 10;
    const float* sg = sig[tid];
    MeanVar<false> mv;
    int i0 = 30;
    for (; i0 + kStatBatch <= n_samples; i0 += kStatBatch) {
      float v[kStatBatch];
#pragma unroll
      for (int j = 0; j < kStatBatch; ++j) v[j] = sg[i0 + j];
#pragma unroll
      for (int j = 0; j < kStatBatch; ++j) mv.add(v[j], i0 - 30 + j + 1);
    }
    for (; i0 < n_samples; ++i0) mv.add(sg[i0], i0 - 30 + 1);
    float s_mean = mv.mean, s_var = mv.var;
    if (mv.tiny()) {  // again, dividing
      MeanVar<true> me;
      for (int i = 30; i < n_samples; ++i) me.add(sg[i], i - 30 + 1);
      s_mean = me.mean;
      s_var = me.var;
    }
    float sumInf = 0, sumSup = 0;
    unsigned nInf = 0, nSup = 0;
    bool acc = false;
    for (int i0 = 0; i0 < n_samples; i0 += kStatBatch) {
      float v[kStatBatch];
#pragma unroll
      for (int j = 0; j < kStatBatch; ++j) v[j] = sg[min(i0 + j, n_samples - 1)];
      // without branches: the signal is non-negative, so adding +0 to a
      // sum leaves it unchanged
#pragma unroll
      for (int j = 0; j < kStatBatch; ++j) {
        const bool live = i0 + j < n_samples;
        const bool lo = live && v[j] < s_mean;
        acc = acc || lo;
        const bool take_lo = acc && lo, take_hi = live && acc && !lo;
        sumInf += take_lo ? v[j] : 0.f;
        nInf += take_lo;
        sumSup += take_hi ? v[j] : 0.f;
        nSup += take_hi;
      }
    }
    stat_var[tid] = s_var;
    stat_muw[tid] = sumSup / (float)nSup;
    stat_mub[tid] = sumInf / (float)nInf;
  } else if (tid == kFinalBlock - 64) {
    // sample positions x_i along the profile (another wavefront)
    const float stepX = (J.end_sig - J.begin_sig) / ((float)n_samples - 1.f);
    float x = J.begin_sig;
    for (int i = 0; i < n_samples; ++i) {
      xs[i] = x;
      x += stepX;
    }
  }
  __syncthreads();
  // the median profile over the valid cuts (Identification.cpp:920-934):
  // each value lands at its rank (ties broken by cut order), then the middle
  // order statistic, or the two middle ones summed in float and halved in
  // double, as the host's partial_sort_copy median does
  const int mv = n_valid;
  for (int q = tid; q < n_samples * mv; q += kFinalBlock) {
    const int i = q / mv, j = q - i * mv;
    const float v = sig[valid_cut[j]][i];
    int rank = 0;
    for (int l = 0; l < mv; ++l) {
      const float u = sig[valid_cut[l]][i];
      rank += (u < v) || (u == v && l < j);
    }
    ordered[i][rank] = v;
  }
  __syncthreads();
  for (int i = tid; i < n_samples; i += kFinalBlock) {
    float b = 0.f;
    if (mv % 2) {
      b = ordered[i][mv / 2];
    } else if (mv > 0) {
      const float sum = ordered[i][mv / 2] + ordered[i][mv / 2 - 1];
      b = (float)((double)sum / 2.0);
    }
    bar[i] = b;
  }
  __syncthreads();
  float bar_lo = FLT_MAX, bar_hi = -FLT_MAX;  // lane 0's are the block's
  if (tid < 64) {
    for (int i = tid; i < n_samples; i += 64) {
      bar_lo = fminf(bar_lo, bar[i]);
      bar_hi = fmaxf(bar_hi, bar[i]);
    }
    for (int o = 32; o > 0; o >>= 1) {
      bar_lo = fminf(bar_lo, __shfl_xor(bar_lo, o, 64));
      bar_hi = fmaxf(bar_hi, __shfl_xor(bar_hi, o, 64));
    }
  }
  // ring parity of every bank profile at every sample position, and each
  // sample's term under either parity (:124-160): the division is done once
  // per sample instead of once per sample and bank row
  for (int q = tid; q < bank_rows * n_samples; q += kFinalBlock) {
    const int i = q / bank_rows, idc = q - i * bank_rows;
    int ldum = 0;
    for (int j = 0; j < bank_cols; ++j)
      if (ratio[idc * kMaxRatios + j] <= xs[i]) ++ldum;
    parity[i][idc] = (uint8_t)(ldum & 1);
  }
  for (int q = tid; q < nc * n_samples; q += kFinalBlock) {
    const int k = q / n_samples, i = q - k * n_samples;
    if ((sticky >> k) & 1u) continue;
    const float v = sig[k][i], v2 = 2.0f * stat_var[k];
    const float tb = fmaxf(v - stat_mub[k], 0.f);
    const float tw = fminf(v - stat_muw[k], 0.f);
    term[1][k][i] = tb * tb / v2;
    term[0][k][i] = tw * tw / v2;
  }
  __syncthreads();
  // distance of each valid cut to each bank profile, summed in sample order
  for (int q = tid; q < nc * bank_rows; q += kFinalBlock) {
    const int k = q / bank_rows, idc = q - k * bank_rows;
    if ((sticky >> k) & 1u) continue;
    const float* t0 = term[0][k];
    const float* t1 = term[1][k];
    float distance = 0;
    constexpr int kSumBatch = 8;  // terms read together, then added in sample order
    for (int i0 = 0; i0 < n_samples; i0 += kSumBatch) {
      float v[kSumBatch];
#pragma unroll
      for (int j = 0; j < kSumBatch; ++j) {
        const int i = min(i0 + j, n_samples - 1);
        v[j] = parity[i][idc] ? t1[i] : t0[i];
      }
#pragma unroll
      for (int j = 0; j < kSumBatch; ++j)
        if (i0 + j < n_samples) distance += v[j];
    }
    dist[J.dist_offset + k * bank_rows + idc] = distance;
  }
  if (tid == 0) {
    O.ok = 1;
    O.cx = S.cx;
    O.cy = S.cy;
    for (int r = 0; r < 9; ++r) O.H[r] = sH[r];
    O.min_res = S.min_res;
    O.bar_min = bar_lo;
    O.bar_max = bar_hi;
  }
  if (tid < nc) O.oob[tid] = (uint8_t)((sticky >> tid) & 1u);
}

// A refinement job takes the stops of the selection it names (one block of
// 64 threads per job): its cut count is the selected count, and a job whose
// selection is empty gets no iteration.
__global__ __launch_bounds__(64) void k_take_stops(const RefineJobDev* __restrict__ src,
                                                   RefineJobDev* __restrict__ jobs,
                                                   const SelectOutDev* __restrict__ sel) {
  static_assert(sizeof(RefineJobDev) % 4 == 0, "jobs copied as words");
  constexpr int kWords = (int)(sizeof(RefineJobDev) / 4);
  const uint32_t* from = reinterpret_cast<const uint32_t*>(src + blockIdx.x);
  uint32_t* to = reinterpret_cast<uint32_t*>(jobs + blockIdx.x);
  for (int i = threadIdx.x; i < kWords; i += blockDim.x) to[i] = from[i];
  __syncthreads();
  RefineJobDev& J = jobs[blockIdx.x];
  const int s = J.sel_index;
  if (s < 0) return;
  const SelectOutDev& o = sel[s];
  const int ns = o.n_collected == 0 ? 0 : min(o.n_selected, kMaxCuts);
  if (threadIdx.x < ns) J.stops[threadIdx.x] = make_float2(o.stops[threadIdx.x].x, o.stops[threadIdx.x].y);
  if (threadIdx.x == 0) {
    J.n_cuts = ns;
    if (ns == 0) J.n_iter = 0;
  }
}

// The centre each marker has reached after at most `iters` launches of
// k_refine_iter, a wavefront per marker.
__global__ __launch_bounds__(64) void k_refine_centers(const RefineJobDev* __restrict__ jobs,
                                                       int iters, int n_samples, int grid_n,
                                                       RefineWork W, float2* __restrict__ centers,
                                                       int* __restrict__ found) {
  __shared__ RefineStateDev S;
  const int m = blockIdx.x;
  const RefineJobDev& J = jobs[m];
  const int it = min(J.n_iter, iters);
  PointRecord rec;
  load_records(it, m, gridDim.x, n_samples, grid_n, W, rec);
  state_at(J, it, n_samples, grid_n, rec, S);
  if (threadIdx.x == 0) put_center(J, it >= 1 && S.ok, S, m, centers, found);
}

Samples samples(int n) { return Samples{n, 1.0 / (double)(n - 1)}; }

// The launches of one search: a lane per cut and grid point, the chunks'
// sample buffers in dynamic LDS.
struct SearchShape {
  int per;      // chunks per block
  int block;
  size_t lds;
};
SearchShape search_shape(int max_cuts, int grid_n, int per) {
  const int cuts = std::min(std::max(max_cuts, 1), kMaxCuts), g2 = grid_n * grid_n;
  const int lanes = std::max(g2 * cuts, 2 * g2 * kRefineChunk);
  return SearchShape{per, (lanes + 63) / 64 * 64,
                     sizeof(float) * (per > 1 ? 2 : 1) * cuts * g2 * kRefineChunk};
}

void launch_iteration(const RefineJobDev* jobs, int n_jobs, int it, const SearchShape& sh,
                      int n_samples, int grid_n, const RefineWork& work, hipStream_t s) {
  const dim3 grid((chunks_of(n_samples) + sh.per - 1) / sh.per, n_jobs);
  k_refine_iter<<<grid, sh.block, sh.lds, s>>>(jobs, it, sh.per, samples(n_samples), grid_n, work);
}

// Markers from which k_refine_search takes over: where the two meet at the
// usual 22 cuts; they meet at about 105 markers of 8 cuts and 130 of 32.  100
// samples, 9 iterations and the centres, k_refine_iter against
// k_refine_search:
//    8 cuts  100 markers 118 / 123 us, 128 142 / 124, 150 164 / 125, 256 194 / 129
//   22 cuts  100 markers 183 / 259 us, 128 233 / 261, 150 277 / 266, 256 337 / 278
//   32 cuts  100 markers 284 / 361 us, 128 355 / 364, 150 418 / 367, 256 504 / 383
// The coarse step alone (with one descent step): 52 / 53 us at 128 markers of
// 8 cuts, 71 / 71 at 150 of 22, 80 / 83 at 128 of 32.
constexpr int kSearchMinJobs = 150;
// Chunks per block: as few as keep an iteration's blocks within two per CU
// (a third of nine wavefronts does not fit beside them; 100 markers 307 us
// with one chunk, 219 with two; 48 markers 158 / 166).
constexpr int kIterBlocks = 512;
int chunks_per_block(int n_jobs, int n_samples) {
  const int nchunk = chunks_of(n_samples);
  int per = 1;
  while (per < nchunk && (long long)n_jobs * ((nchunk + per - 1) / per) > kIterBlocks) ++per;
  return per;
}

constexpr int kSearchBlock = 512, kSearchBlockWide = 704;
static_assert(G2MAX * kMaxSumChunks <= kSearchBlockWide, "a lane per grid point and chunk");

void launch_search(const RefineJobDev* jobs, int n_jobs, int n_samples, int grid_n, int iters,
                   const RefineWork& work, float2* centers, int* found, hipStream_t s) {
  const Samples ns = samples(n_samples);
  if (grid_n * grid_n * sum_chunks_of(n_samples) <= kSearchBlock)
    k_refine_search<kSearchBlock><<<n_jobs, kSearchBlock, 0, s>>>(jobs, ns, grid_n, iters, work,
                                                                  centers, found);
  else
    k_refine_search<kSearchBlockWide><<<n_jobs, kSearchBlockWide, 0, s>>>(jobs, ns, grid_n, iters,
                                                                          work, centers, found);
}

void launch_iterations(const RefineJobDev* jobs, int n_jobs, int iters, int max_cuts, int n_samples,
                       int grid_n, const RefineWork& work, hipStream_t s) {
  const SearchShape sh = search_shape(max_cuts, grid_n, chunks_per_block(n_jobs, n_samples));
  for (int it = 0; it < iters; ++it)
    launch_iteration(jobs, n_jobs, it, sh, n_samples, grid_n, work, s);
}

}  // namespace

int launch_refine_centers(const RefineJobDev* jobs, int n_jobs, int iters, int max_cuts,
                          int n_samples, int grid_n, const RefineWork& work, float2* centers,
                          int* found, hipStream_t s) {
  if (n_jobs <= 0) return 0;
  if (n_jobs >= kSearchMinJobs) {
    launch_search(jobs, n_jobs, n_samples, grid_n, iters, work, centers, found, s);
  } else {
    launch_iterations(jobs, n_jobs, iters, max_cuts, n_samples, grid_n, work, s);
    k_refine_centers<<<n_jobs, 64, 0, s>>>(jobs, iters, n_samples, grid_n, work, centers, found);
  }
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_refine_readout(const RefineJobDev* jobs, int n_jobs, int n_samples, const float* H,
                          const float* centers, const double* cost, const float* inv_ratio,
                          int bank_rows, int bank_cols, const RefineWork& work, RefineOutDev* out,
                          float* dist, hipStream_t s) {
  if (n_jobs <= 0) return 0;
  k_refine_final<<<n_jobs, kFinalBlock, 0, s>>>(jobs, samples(n_samples), kMaxGrid, inv_ratio, bank_rows,
                                                 bank_cols, work, H, centers, cost, 0, out, dist);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_take_stops(const RefineJobDev* src, RefineJobDev* jobs, int n_jobs,
                      const SelectOutDev* sel, hipStream_t s) {
  if (n_jobs <= 0) return 0;
  k_take_stops<<<n_jobs, 64, 0, s>>>(src, jobs, sel);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_select_cuts(const SelectJobDev* jobs, int n_jobs, const float4* pts, float start_sig,
                       int n_samples, int n_ref, int select_max, SelectOutDev* out, hipStream_t s) {
  if (n_jobs <= 0) return 0;
  k_select_cuts<<<n_jobs, 256, 0, s>>>(jobs, pts, start_sig, n_samples, n_ref, select_max, out);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_refine(const RefineJobDev* jobs, int n_jobs, int max_iter, int max_cuts, int n_samples,
                  int grid_n, const float* inv_ratio, int bank_rows, int bank_cols, const RefineWork& work,
                  RefineOutDev* out, float* dist, hipStream_t s) {
  if (n_jobs <= 0) return 0;
  const int searched = n_jobs >= kSearchMinJobs;
  if (searched) launch_search(jobs, n_jobs, n_samples, grid_n, max_iter, work, nullptr, nullptr, s);
  else launch_iterations(jobs, n_jobs, max_iter, max_cuts, n_samples, grid_n, work, s);
  k_refine_final<<<n_jobs, kFinalBlock, 0, s>>>(jobs, samples(n_samples), grid_n, inv_ratio, bank_rows,
                                                 bank_cols, work, nullptr, nullptr, nullptr,
                                                 searched, out, dist);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace cctagx
