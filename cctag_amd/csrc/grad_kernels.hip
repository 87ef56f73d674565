// Differentiable identification refinement on gfx950.
//
// The grid search of refineConicFamilyGlob (Identification.cpp:813-1158)
// scores an imaged centre c by sampling every selected cut through the
// homography H(c) of the outer ellipse and the centre
// (computeHomographyFromEllipseAndImagedCenter, :739-798) and summing the
// squared differences between cuts.  Here that score is a differentiable
// function of H:
//
//   q_k  = pi(H^-1 p_k)                 marker-plane direction of stop p_k
//   y_ki = pi(H (t_i q_k, 1))           t_i = begin + i (end - begin)/(n - 1)
//   s_ki = bilinear(I, y_ki) / 2        Identification.hpp:197-222
//   C    = sum_i sum_{k<l valid} (s_ki - s_li)^2 / (m (m-1) / 2)
//
// (pi(w) = (w0/w2, w1/w2); a cut is valid when all its samples are inside
// the image).  One block runs the forward pass and the adjoint pass of a
// marker: dC/ds_ki = 2 (m s_ki - S_i) / pairs with S_i the sum over
// valid cuts, lambda = Jpi(w)^T dC/dy, and
//
//   dC/dH = sum_k [ sum_i lambda_ki u_ki^T  -  H^-T Jpi(v_k)^T (H_{:,01}^T L_k) v_k^T ]
//
// with v_k = H^-1 p_k and L_k = sum_i t_i lambda_ki (the second term is the
// dependence of the cut direction q_k on H).  What is asked for are
// derivatives along directions of H: its free entries, or dH/dc of the closed
// form (evaluated in forward mode with dual numbers) for the centre; each is
// contracted cut by cut, without forming dC/dH.  Interpolation runs in T (float
// in production, double for checking); lambda and every sum are in double.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>

#include "division.hpp"
#include "grad_device.hpp"
#include "host/rows.hpp"

namespace cctagx {
namespace {

// A dual number carrying one derivative (forward mode).
struct D1 {
  double v, d;
};
__device__ __forceinline__ D1 dc(double v) { return D1{v, 0.0}; }
__device__ __forceinline__ D1 operator+(D1 a, D1 b) { return D1{a.v + b.v, a.d + b.d}; }
__device__ __forceinline__ D1 operator-(D1 a, D1 b) { return D1{a.v - b.v, a.d - b.d}; }
__device__ __forceinline__ D1 operator-(D1 a) { return D1{-a.v, -a.d}; }
__device__ __forceinline__ D1 operator*(D1 a, D1 b) {
  return D1{a.v * b.v, a.d * b.v + a.v * b.d};
}
__device__ __forceinline__ D1 operator*(double a, D1 b) { return D1{a * b.v, a * b.d}; }
__device__ __forceinline__ D1 dsqrt(D1 a) {
  const double r = sqrt(a.v);
  return D1{r, a.d * (0.5 / r)};
}

__device__ __forceinline__ D1 pick(bool first, D1 a, D1 b) {
  return D1{first ? a.v : b.v, first ? a.d : b.d};
}

// Entry (row, col) of the closed-form homography of the ellipse's canonic
// form and an imaged centre (Identification.cpp:739-798), in double with the
// derivative along cx (along_y false) or cy, in image coordinates relative
// to (ox, oy).
__device__ D1 closed_form(const GradJobDev& J, double cx, double cy, int row, int col, bool along_y,
                          double ox, double oy) {
  const D1 x{cx, along_y ? 0.0 : 1.0}, y{cy, along_y ? 1.0 : 0.0};
  const float* T = J.t_can;
  const D1 u = (double)T[0] * x + (double)T[1] * y + dc(T[2]);
  const D1 v = (double)T[3] * x + (double)T[4] * y + dc(T[5]);
  const D1 w = (double)T[6] * x + (double)T[7] * y + dc(T[8]);
  const double iw = 1.0 / w.v;
  const D1 rw{iw, -w.d * iw * iw};
  const D1 xc = u * rw, yc = v * rw;
  const double Q11 = J.Q11, Q22 = J.Q22, Q33 = J.Q33;
  const D1 f = Q11 * xc * xc;
  // the entry's column of the canonic homography, scaled by its diagonal
  // (all three laid out and one picked: one square root, and no branch -- a
  // branch per column left the last entry of the third one unset)
  const D1 c0[3] = {dc(Q33), dc(0.0), -(Q11 * xc)};
  const D1 c1[3] = {Q22 * xc * yc, -f - dc(Q33), Q22 * yc};
  const D1 c2[3] = {-(Q33 * xc), -(Q33 * yc), dc(-Q33)};
  const D1 r0 = (Q22 * Q33 * (1.0 / Q11)) * (f + Q22 * yc * yc + dc(Q33));
  const D1 r2 = -(Q22 * (f + dc(Q33)));
  const D1 root = dsqrt(pick(col == 0, r0, r2));
  const D1 scale = pick(col == 1, dc(Q33), root);
  D1 h[3];
  for (int j = 0; j < 3; ++j) h[j] = pick(col == 0, c0[j], pick(col == 1, c1[j], c2[j]));
  const float* Ti = J.t_inv_can;
  const double o = row == 0 ? ox : row == 1 ? oy : 0.0;
  D1 e = dc(0.0);
  for (int j = 0; j < 3; ++j) e = e + ((double)Ti[row * 3 + j] - o * (double)Ti[6 + j]) * (h[j] * scale);
  return e;
}

// Entry (row, col) of the adjugate of a row-major 3x3 matrix.
__device__ __forceinline__ double adjugate(const double* m, int row, int col) {
  const int i1 = (col + 1) % 3, i2 = (col + 2) % 3, j1 = (row + 1) % 3, j2 = (row + 2) % 3;
  return m[i1 * 3 + j1] * m[i2 * 3 + j2] - m[i1 * 3 + j2] * m[i2 * 3 + j1];
}

constexpr int kLanesPerCut = 8;
constexpr int kMaxGradBlock = kMaxCuts * kLanesPerCut;
constexpr int kMaxGradWaves = kMaxGradBlock / 64;

// One marker's evaluation, by a block of kLanesPerCut lanes per cut.  Lane j
// of a cut takes its samples j, j + 8, ... (R of them) through both passes:
// the samples' image gradients stay in registers between the forward pass and
// the adjoint (in double), which needs only the sums L = sum_i t_i lambda_i
// and M = sum_i lambda_i per cut (u_ki = (t_i q_k, 1), so sum_i lambda_i u_i^T
// = [L q_k^T, M]).
//
// LOCAL (the refiner's calls): a sample's place t, its numerators and its
// denominator w(t) = t A_k + H_{:,2} (A_k = H_{:,01} q_k) are in double,
// relative to (ox, oy), the pixel of the centre; T holds the pixel and the
// offset into it (locate).  With all of it in float, positions in a 7360 px
// mosaic erred by ulps of the image (2.5e-4 px), and score and gradient of 2048
// markers by 2.8e-5 and 8.2e-4 against double sampling; relative to (ox, oy),
// still in float, by 3.0e-7 and 1.6e-5; so by 1.2e-8 and 1.8e-8.  20 descent
// steps of 4096 markers end within 1e-4 px of those with double sampling, not
// 4e-3.  (A float position of ulp precision, 1 / w in float and kept as a
// third value per sample between the passes, took as long for one evaluation
// and 1300 us for the 20 steps.)
// Otherwise (the identification): image coordinates, each float operation
// rounded on its own and the adjoint in double, which keeps the identified
// markers' qualities and homographies as they always were: a descent of 30
// steps ends where rounding sends it, 3e-4 apart in quality for positions
// that differ by 1e-4 px.
//
// Bound by instruction issue, at 4096 markers.  Before, the forward pass took
// two double divisions per sample, the adjoint sampled the image again and
// took three more, and the closed form, the inverse and the score's sum ran
// on one lane: 20 steps of 4096 markers 4270 us, now 1190; one evaluation of
// 2048 markers 124 us, now 36.
template <class T>
struct EvalShared {
  double H[9], Hi[9], det;        // relative to (ox, oy)
  double dir[2][9];               // dH / d(cx), dH / d(cy)
  double q[kMaxCuts][2], v[kMaxCuts][3];  // q = v / v2, v = H^-1 (p, 1)
  double A[kMaxCuts][3];          // H_{:,01} q
  double S[kMaxSamples];          // sum over the valid cuts of the doubled samples
  double sum[kMaxGradWaves][11];  // each wavefront's cost and derivatives
  uint32_t oob;
  uint32_t plain;                 // cuts whose denominators div2_rn takes
  int ox, oy;
};

// The image position (u / w, v / w): its pixel and the offsets into it.  In
// float (`plain`: w is in div2_rn's range) the pixel comes from a rounded
// quotient, the offset from what the pixel leaves of u, in double, so that it
// is off by an ulp of its own, not of the position, and a pixel that the
// rounding missed is put right.  A position within 2^-25 px of a pixel's
// border is on it (offset 0), whichever side the doubles' rounding left it.
__device__ __forceinline__ void locate(double u, double v, double w, bool plain, double& px, double& py,
                                       double& fx, double& fy) {
  const double x = u / w, y = v / w;
  px = floor(x);
  py = floor(y);
  fx = x - px;
  fy = y - py;
}
__device__ __forceinline__ void locate(double u, double v, double w, bool plain, float& px, float& py,
                                       float& fx, float& fy) {
  if (plain) {
    const float d = (float)w, r0 = __builtin_amdgcn_rcpf(d);
    const float r = __builtin_fmaf(__builtin_fmaf(-d, r0, 1.f), r0, r0);
    px = floorf((float)u * r);
    py = floorf((float)v * r);
    div2_rn((float)__builtin_fma(-(double)px, w, u), (float)__builtin_fma(-(double)py, w, v), d, fx, fy);
    const float ex = floorf(fx + 0x1p-25f), ey = floorf(fy + 0x1p-25f);
    px += ex;
    py += ey;
    fx -= ex;
    fy -= ey;
  } else {
    double x, y, ox, oy;
    locate(u, v, w, false, x, y, ox, oy);
    px = (float)x;
    py = (float)y;
    fx = (float)ox;
    fy = (float)oy;
  }
}
__device__ __forceinline__ float fused(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fused(double a, double b, double c) { return __builtin_fma(a, b, c); }

// Wavefront 0: the cuts' constants from the homography E.H (E.ox, E.oy set).
template <class T>
__device__ __forceinline__ void lay_out_cuts(const GradJobDev& J, EvalShared<T>& E) {
  const int k = threadIdx.x;
  double H[9], Hi[9];
  for (int e = 0; e < 9; ++e) H[e] = E.H[e];
  for (int r = 0; r < 3; ++r)
    for (int c = 0; c < 3; ++c) Hi[r * 3 + c] = adjugate(H, r, c);
  const double det = H[0] * Hi[0] + H[1] * Hi[3] + H[2] * Hi[6], id = 1.0 / det;
  for (int e = 0; e < 9; ++e) Hi[e] *= id;
  if (k == 0) {
    for (int e = 0; e < 9; ++e) E.Hi[e] = Hi[e];
    E.det = det;
    E.oob = 0;
  }
  bool plain = false;
  if (k < J.n_cuts) {
    const double px = (double)J.stops[k].x - E.ox, py = (double)J.stops[k].y - E.oy;
    double v[3];
    for (int r = 0; r < 3; ++r) v[r] = Hi[r * 3] * px + Hi[r * 3 + 1] * py + Hi[r * 3 + 2];
    const double qx = v[0] / v[2], qy = v[1] / v[2];
    E.q[k][0] = qx;
    E.q[k][1] = qy;
    for (int r = 0; r < 3; ++r) {
      E.v[k][r] = v[r];
      E.A[k][r] = H[r * 3] * qx + H[r * 3 + 1] * qy;
    }
    const double a = J.begin_sig * E.A[k][2] + H[8], b = J.end_sig * E.A[k][2] + H[8];
    plain = (a > 0.0) == (b > 0.0) && fmin(fabs(a), fabs(b)) > 0x1p-60 &&
            fmax(fabs(a), fabs(b)) < 0x1p60;
  }
  const uint32_t p = (uint32_t)__ballot(plain);
  if (k == 0) E.plain = p;
}

// Score and, per lane, the derivative sums of its cut at E.H (laid out, after
// a barrier).  Returns the valid cuts, none when there are fewer than two or
// H is singular; every lane of a valid cut holds the cut's L and M (scaled to
// dC/dw) and E.sum[wave][0] its wavefront's share of the score, to be read
// after a barrier.  sig: n_cuts x n_samples.
template <class T, int R, bool LOCAL>
__device__ __forceinline__ uint32_t eval_marker(const GradJobDev& J, int n_samples, EvalShared<T>& E, T* sig,
                                            double* L, double* M) {
  const int tid = threadIdx.x, nc = J.n_cuts;
  const int k = tid / kLanesPerCut, j = tid % kLanesPerCut;
  const bool on = k < nc;
  // the samples' places along the cut: in double, or (not LOCAL) as T rounds them
  const T b = (T)J.begin_sig, step = ((T)J.end_sig - (T)J.begin_sig) / (T)(n_samples - 1);
  const double db = J.begin_sig, dstep = ((double)J.end_sig - db) / (n_samples - 1);
  auto place = [&](int i) {
    return LOCAL ? __builtin_fma((double)i, dstep, db) : (double)(b + (T)i * step);
  };
  T gx[R], gy[R];  // per sample the doubled sample's derivatives along x and y
  if (on) {
    const T xlo = (T)(-E.ox), xhi = (T)(J.iw - 1 - E.ox), ylo = (T)(-E.oy), yhi = (T)(J.ih - 1 - E.oy);
    const int base = E.oy * J.iw + E.ox;
    const double A[3] = {E.A[k][0], E.A[k][1], E.A[k][2]};
    T H[9];
    for (int e = 0; e < 9; ++e) H[e] = (T)E.H[e];
    const T qx = (T)E.q[k][0], qy = (T)E.q[k][1];
    const bool plain = (E.plain >> k) & 1u;
    bool out = false;
    constexpr int kBatch = 7;  // samples whose image reads are in flight together
#pragma unroll
    for (int t0 = 0; t0 < R; t0 += kBatch) {
      T fx[kBatch], fy[kBatch];
      uint32_t q[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        if (t0 + u >= R) continue;
        const int i = j + (t0 + u) * kLanesPerCut;
        T px, py;  // the pixel
        bool in;
        if constexpr (LOCAL) {
          const double t = place(i);
          locate(__builtin_fma(t, A[0], E.H[2]), __builtin_fma(t, A[1], E.H[5]),
                 __builtin_fma(t, A[2], E.H[8]), plain, px, py, fx[u], fy[u]);
          in = px >= xlo && px < xhi && py >= ylo && py < yhi;
        } else {
          const T t = b + (T)i * step, ux = t * qx, uy = t * qy;
          const T w0 = H[0] * ux + H[1] * uy + H[2], w1 = H[3] * ux + H[4] * uy + H[5],
                  w2 = H[6] * ux + H[7] * uy + H[8];
          T x, y;
          if (plain) {
            div2_rn(w0, w1, w2, x, y);
          } else {
            x = w0 / w2;
            y = w1 / w2;
          }
          in = x >= xlo && x < xhi && y >= ylo && y < yhi;
          px = floor(x);
          py = floor(y);
          fx[u] = x - px;
          fy[u] = y - py;
        }
        out |= i < n_samples && !in;
        const int at = in && i < n_samples ? base + (int)py * J.iw + (int)px : 0;
        q[u] = J.quad[(uint32_t)at];
      }
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        if (t0 + u >= R) continue;
        const int i = j + (t0 + u) * kLanesPerCut;
        const T x = fx[u], y = fy[u];
        const T p00 = (T)(q[u] & 255u), p10 = (T)((q[u] >> 8) & 255u), p01 = (T)((q[u] >> 16) & 255u),
                p11 = (T)(q[u] >> 24);
        const T d0 = p10 - p00, d1 = p11 - p01;
        T val;
        if constexpr (LOCAL) {
          const T top = fused(x, d0, p00), dy = fused(x, d1, p01) - top;
          val = fused(y, dy, top);
          gx[t0 + u] = fused(y, d1 - d0, d0);
          gy[t0 + u] = dy;
        } else {
          const T x1 = (T)1 - x, y1 = (T)1 - y;
          val = p00 * x1 * y1 + p10 * x * y1 + p01 * x1 * y + p11 * x * y;
          gx[t0 + u] = d0 * y1 + d1 * y;
          gy[t0 + u] = (p01 - p00) * x1 + (p11 - p10) * x;
        }
        if (i < n_samples) sig[k * n_samples + i] = val;
      }
    }
    if (out) atomicOr(&E.oob, 1u << k);
  }
  __syncthreads();
  const uint32_t valid = ~E.oob & (nc >= 32 ? ~0u : (1u << nc) - 1u);
  const int m = __popc(valid);
  for (int i = tid; i < n_samples; i += blockDim.x) {
    double s = 0.0;
    constexpr int kRead = 8;  // reads in flight together
    for (int k0 = 0; k0 < nc; k0 += kRead) {
      T v[kRead];
#pragma unroll
      for (int u = 0; u < kRead; ++u) v[u] = sig[min(k0 + u, nc - 1) * n_samples + i];
#pragma unroll
      for (int u = 0; u < kRead; ++u)
        if (k0 + u < nc && ((valid >> (k0 + u)) & 1u)) s += (double)v[u];
    }
    E.S[i] = s;
  }
  __syncthreads();
  const double pairs = 0.5 * (double)m * (double)(m - 1);
  double cost = 0.0;  // sum over the cut of (m s - S)^2, s and S doubled
  for (int r = 0; r < 3; ++r) L[r] = M[r] = 0.0;
  if (on && ((valid >> k) & 1u)) {
    const double dm = (double)m, A[3] = {E.A[k][0], E.A[k][1], E.A[k][2]};
#pragma unroll
    for (int t = 0; t < R; ++t) {
      const int i = j + t * kLanesPerCut;
      if (i < n_samples) {
        const double d = dm * (double)sig[k * n_samples + i] - E.S[i];
        const double tt = place(i);
        cost = __builtin_fma(d, d, cost);
        const double rw = 1.0 / __builtin_fma(tt, A[2], E.H[8]);
        double g[3] = {(double)gx[t] * rw, (double)gy[t] * rw, 0.0};
        g[2] = -(g[0] * __builtin_fma(tt, A[0], E.H[2]) + g[1] * __builtin_fma(tt, A[1], E.H[5])) * rw;
#pragma unroll
        for (int r = 0; r < 3; ++r) {
          const double dg = d * g[r];
          M[r] += dg;
          L[r] = __builtin_fma(tt, dg, L[r]);
        }
      }
    }
  }
  // the cut's sums over its lanes, the score over the wavefront
  for (int o = 1; o < kLanesPerCut; o <<= 1)
    for (int r = 0; r < 3; ++r) {
      L[r] += __shfl_xor(L[r], o, 64);
      M[r] += __shfl_xor(M[r], o, 64);
    }
  for (int o = 1; o < 64; o <<= 1) cost += __shfl_xor(cost, o, 64);
  // sum_k (m s_k - S)^2 = m (m S2 - S^2); ds = dV / 2
  const double scale = 1.0 / (2.0 * pairs);
  for (int r = 0; r < 3; ++r) {
    L[r] *= scale;
    M[r] *= scale;
  }
  if ((tid & 63) == 0) E.sum[tid >> 6][0] = cost / (4.0 * (double)m * pairs);
  return m >= 2 && E.det != 0.0 && isfinite(E.det) ? valid : 0u;
}

// A valid cut's share of the score's derivative along dH = D (relative to the
// origin as E.H; a cut left out may have no finite direction, and 0 * inf is
// not 0): lambda . (D u) summed over its samples, and through the
// cut's direction q, dq = J_pi(v) dv, dv = -H^-1 D v.
template <class T>
__device__ __forceinline__ double along(const EvalShared<T>& E, int k, const double* D, const double* L,
                                        const double* M) {
  const double qx = E.q[k][0], qy = E.q[k][1];
  double acc = 0.0, e[3];
  for (int r = 0; r < 3; ++r) {
    acc += (D[r * 3] * qx + D[r * 3 + 1] * qy) * L[r] + D[r * 3 + 2] * M[r];
    e[r] = D[r * 3] * E.v[k][0] + D[r * 3 + 1] * E.v[k][1] + D[r * 3 + 2] * E.v[k][2];
  }
  double f[3];
  for (int r = 0; r < 3; ++r)
    f[r] = E.Hi[r * 3] * e[0] + E.Hi[r * 3 + 1] * e[1] + E.Hi[r * 3 + 2] * e[2];
  const double z0 = E.H[0] * L[0] + E.H[3] * L[1] + E.H[6] * L[2];
  const double z1 = E.H[1] * L[0] + E.H[4] * L[1] + E.H[7] * L[2];
  return acc - (z0 * (f[0] - qx * f[2]) + z1 * (f[1] - qy * f[2])) / E.v[k][2];
}

// Lane j of every cut adds its value over the wavefront's cuts (the same
// lane of each 8-lane group).
__device__ __forceinline__ double over_cuts(double v) {
  for (int o = kLanesPerCut; o < 64; o <<= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Score and gradient at given homographies, one block per marker.
template <class T, int R>
__global__ __launch_bounds__(kMaxGradBlock, sizeof(T) == 4 ? 4 : 1) void k_grad_eval(const GradJobDev* __restrict__ jobs,
                                                             const float* __restrict__ Hin, int n_samples,
                                                             double* __restrict__ cost,
                                                             double* __restrict__ grad) {
  extern __shared__ __attribute__((aligned(16))) unsigned char grad_lds[];
  T* sig = reinterpret_cast<T*>(grad_lds);
  __shared__ EvalShared<T> E;
  const int m = blockIdx.x, tid = threadIdx.x, waves = blockDim.x >> 6;
  const GradJobDev& J = jobs[m];
  const int nc = J.n_cuts;
  double L[3], M[3];
  // the origin: the pixel of the homography's centre, kept inside the image
  if (tid < 64) {
    const float* h = Hin + m * 9;
    const double w = h[8];
    const double cx = (double)h[2] / w, cy = (double)h[5] / w;
    const int ox = cx > 0.0 && cx < J.iw ? (int)cx : 0, oy = cy > 0.0 && cy < J.ih ? (int)cy : 0;
    if (tid < 9) {
      const double o = tid < 3 ? ox : tid < 6 ? oy : 0;
      E.H[tid] = (double)h[tid] - o * (double)h[6 + tid % 3];
    }
    if (tid == 0) {
      E.ox = ox;
      E.oy = oy;
    }
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  if (tid < 64) lay_out_cuts(J, E);
  __syncthreads();
  const uint32_t valid = eval_marker<T, R, true>(J, n_samples, E, sig, L, M);
  const bool ok = valid != 0;
  if (grad) {
    // directions 0..7: H's free entries (an entry of the last row moves the
    // relative rows above it too); 8, 9: the marker-plane shift of the centre
    // along x and y, H' = H [1 0 x; 0 1 y; 0 0 1]
    const int k = tid / kLanesPerCut, j = tid % kLanesPerCut;
    for (int d = j; d < 10; d += kLanesPerCut) {
      double D[9];
      for (int e = 0; e < 9; ++e) {
        const int r = e / 3, c = e % 3;
        if (d >= 8) D[e] = c == 2 ? E.H[r * 3 + d - 8] : 0.0;
        else if (c != d % 3) D[e] = 0.0;
        else if (d < 6) D[e] = e == d ? 1.0 : 0.0;
        else D[e] = r == 2 ? 1.0 : r == 0 ? -(double)E.ox : -(double)E.oy;
      }
      const double v = over_cuts((valid >> k) & 1u ? along(E, k, D, L, M) : 0.0);
      if ((tid & 63) < kLanesPerCut) E.sum[tid >> 6][1 + d] = v;
    }
  }
  __syncthreads();
  if (tid < (grad ? 11 : 1)) {
    double v = 0.0;
    for (int w = 0; w < waves; ++w) v += E.sum[w][tid];
    if (tid == 0) cost[m] = ok ? v : DBL_MAX;
    else grad[m * 10 + tid - 1] = ok ? v : 0.0;
  }
}

__global__ __launch_bounds__(256) void k_grad_homography(const GradJobDev* __restrict__ jobs, int n,
                                                         const float* __restrict__ centers,
                                                         float* __restrict__ H) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, m = i / 9, e = i - m * 9;
  if (m >= n) return;
  H[i] = (float)closed_form(jobs[m], centers[2 * m], centers[2 * m + 1], e / 3, e % 3, false, 0.0, 0.0).v;
}

// `steps` evaluations per marker, each one forward + adjoint pass at H(c):
// a step that lowers the score is kept and the step length grows by 1.5,
// otherwise the centre returns to the best one and the length halves; the
// next centre moves the best one by the length along -dC/dc.  Every lane of
// wavefront 0 keeps the descent's state; its lanes 0..17 take the closed
// form's entries and derivatives.
template <class T, int R, bool LOCAL>
__global__ __launch_bounds__(kMaxGradBlock, sizeof(T) == 4 ? 4 : 1) void k_grad_descend(const GradJobDev* __restrict__ jobs,
                                                                int steps, int n_samples,
                                                                const float* __restrict__ start,
                                                                float* __restrict__ centers,
                                                                double* __restrict__ cost) {
  extern __shared__ __attribute__((aligned(16))) unsigned char grad_lds[];
  T* sig = reinterpret_cast<T*>(grad_lds);
  __shared__ EvalShared<T> E;
  __shared__ int stop;
  const int m = blockIdx.x, tid = threadIdx.x, waves = blockDim.x >> 6;
  const GradJobDev& J = jobs[m];
  const int nc = J.n_cuts;
  double cx = start ? start[2 * m] : J.c0x, cy = start ? start[2 * m + 1] : J.c0y;
  double best_x = cx, best_y = cy, best_cost = DBL_MAX, gbx = 0.0, gby = 0.0, alpha = J.alpha0;
  double L[3], M[3];
  for (int it = 0; it < steps; ++it) {
    if (tid < 64) {
      const int ox = LOCAL && cx > 0.0 && cx < J.iw ? (int)cx : 0;
      const int oy = LOCAL && cy > 0.0 && cy < J.ih ? (int)cy : 0;
      const int e = min(tid >> 1, 8), s = tid & 1;
      const D1 h = closed_form(J, cx, cy, e / 3, e % 3, s, ox, oy);
      if (tid < 18) {
        if (s == 0) E.H[e] = h.v;
        E.dir[s][e] = h.d;
      }
      if (tid == 0) {
        E.ox = ox;
        E.oy = oy;
        stop = 0;
      }
    }
    __syncthreads();
    if (tid < 64) lay_out_cuts(J, E);
    __syncthreads();
    const uint32_t valid = eval_marker<T, R, LOCAL>(J, n_samples, E, sig, L, M);
    const bool ok = valid != 0;
    {
      const int k = tid / kLanesPerCut, s = tid & 1;
      const double v = over_cuts((valid >> k) & 1u ? along(E, k, E.dir[s], L, M) : 0.0);
      if ((tid & 63) < 2) E.sum[tid >> 6][1 + s] = v;
    }
    __syncthreads();
    if (tid < 64) {
      double sum[3] = {0.0, 0.0, 0.0};
      for (int w = 0; w < waves; ++w)
        for (int r = 0; r < 3; ++r) sum[r] += E.sum[w][r];
      if (ok && sum[0] < best_cost) {
        if (it > 0) alpha *= 1.5;
        best_x = cx;
        best_y = cy;
        best_cost = sum[0];
        gbx = sum[1];
        gby = sum[2];
      } else {
        alpha *= 0.5;
      }
      const double gn = sqrt(gbx * gbx + gby * gby);
      if (!(gn > 0.0) || !isfinite(gn) || best_cost == DBL_MAX) {
        if (tid == 0) stop = 1;
      } else {
        cx = best_x - alpha * gbx / gn;
        cy = best_y - alpha * gby / gn;
      }
    }
    __syncthreads();
    if (stop) break;
  }
  if (tid == 0) {
    centers[2 * m] = (float)best_x;
    centers[2 * m + 1] = (float)best_y;
    cost[m] = best_cost;
  }
}

// Per marker the descent's start: its coarse grid centre when it has one,
// else the job's c0.
__global__ __launch_bounds__(256) void k_grad_start(const GradJobDev* __restrict__ jobs, int n,
                                                    const int* __restrict__ coarse_of,
                                                    const float* __restrict__ coarse,
                                                    float* __restrict__ start) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= n) return;
  const int j = coarse_of[m];
  start[2 * m] = j >= 0 ? coarse[2 * j] : jobs[m].c0x;
  start[2 * m + 1] = j >= 0 ? coarse[2 * j + 1] : jobs[m].c0y;
}

// One word per pixel: its 2x2 neighbourhood, indices clamped to the image.
__global__ __launch_bounds__(256) void k_quads(const uint8_t* __restrict__ img, int w, int h,
                                               size_t pitch, uint32_t* __restrict__ quad) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= w * h) return;
  const int y = i / w, x = i - y * w;
  const uint8_t* r0 = img + (size_t)y * pitch + x;
  const uint8_t* r1 = y + 1 < h ? r0 + pitch : r0;
  const int dx = x + 1 < w ? 1 : 0;
  quad[i] = (uint32_t)r0[0] | (uint32_t)r0[dx] << 8 | (uint32_t)r1[0] << 16 | (uint32_t)r1[dx] << 24;
}

// A block's shape: kLanesPerCut lanes per cut; kSamplesPerLane samples of a
// lane are kept in registers (13 cover 104 samples, 16 kMaxSamples).
struct GradShape {
  int block;
  size_t lds;
};
template <class T>
GradShape grad_shape(int max_cuts, int n_samples) {
  const int cuts = std::min(std::max(max_cuts, 1), kMaxCuts);
  return GradShape{(cuts * kLanesPerCut + 63) / 64 * 64, sizeof(T) * cuts * n_samples};
}
constexpr int kFewSamples = 13, kAllSamples = 16;
static_assert(kAllSamples * kLanesPerCut >= kMaxSamples, "every sample has a lane");

template <class T>
void eval_launch(const GradJobDev* jobs, int n, const float* H, int max_cuts, int n_samples,
                 double* cost, double* grad, hipStream_t s) {
  const GradShape sh = grad_shape<T>(max_cuts, n_samples);
  if (n_samples <= kFewSamples * kLanesPerCut)
    k_grad_eval<T, kFewSamples><<<n, sh.block, sh.lds, s>>>(jobs, H, n_samples, cost, grad);
  else
    k_grad_eval<T, kAllSamples><<<n, sh.block, sh.lds, s>>>(jobs, H, n_samples, cost, grad);
}

template <class T, bool LOCAL>
void descend_launch(const GradJobDev* jobs, int n, int steps, int max_cuts, int n_samples,
                    const float* start, float* centers, double* cost, hipStream_t s) {
  const GradShape sh = grad_shape<T>(max_cuts, n_samples);
  if (n_samples <= kFewSamples * kLanesPerCut)
    k_grad_descend<T, kFewSamples, LOCAL><<<n, sh.block, sh.lds, s>>>(jobs, steps, n_samples, start,
                                                                      centers, cost);
  else
    k_grad_descend<T, kAllSamples, LOCAL><<<n, sh.block, sh.lds, s>>>(jobs, steps, n_samples, start,
                                                                      centers, cost);
}

}  // namespace

hipError_t upload_rows(uint8_t* dst, size_t capacity, const uint8_t* src, int width, int height,
                       size_t stride, hipStream_t s, size_t* pitch) {
  if (rows_fit(capacity, width, height, stride)) {
    *pitch = stride;
    return hipMemcpyAsync(dst, src, (size_t)(height - 1) * stride + width, hipMemcpyHostToDevice, s);
  }
  *pitch = width;
  return hipMemcpy2DAsync(dst, width, src, stride, width, height, hipMemcpyHostToDevice, s);
}

int launch_quads(const uint8_t* img, int w, int h, size_t pitch, uint32_t* quad, hipStream_t s) {
  if (w < 2 || h < 2) return -1;
  k_quads<<<(w * h + 255) / 256, 256, 0, s>>>(img, w, h, pitch, quad);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_grad_start(const GradJobDev* jobs, int n, const int* coarse_of, const float* coarse,
                      float* start, hipStream_t s) {
  if (n <= 0) return 0;
  k_grad_start<<<(n + 255) / 256, 256, 0, s>>>(jobs, n, coarse_of, coarse, start);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_grad_eval(const GradJobDev* jobs, int n, const float* H, int max_cuts, int n_samples,
                     bool fp64, double* cost, double* grad, hipStream_t s) {
  if (n <= 0) return 0;
  if (fp64) eval_launch<double>(jobs, n, H, max_cuts, n_samples, cost, grad, s);
  else eval_launch<float>(jobs, n, H, max_cuts, n_samples, cost, grad, s);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_grad_homography(const GradJobDev* jobs, int n, const float* centers, float* H,
                           hipStream_t s) {
  if (n <= 0) return 0;
  k_grad_homography<<<(9 * n + 255) / 256, 256, 0, s>>>(jobs, n, centers, H);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_grad_descend(const GradJobDev* jobs, int n, int steps, int max_cuts, int n_samples,
                        GradSampling sampling, const float* start, float* centers, double* cost,
                        hipStream_t s) {
  if (n <= 0) return 0;
  if (sampling == GradSampling::fp64)
    descend_launch<double, true>(jobs, n, steps, max_cuts, n_samples, start, centers, cost, s);
  else if (sampling == GradSampling::local)
    descend_launch<float, true>(jobs, n, steps, max_cuts, n_samples, start, centers, cost, s);
  else
    descend_launch<float, false>(jobs, n, steps, max_cuts, n_samples, start, centers, cost, s);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace cctagx
