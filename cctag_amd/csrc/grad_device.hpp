// Device-side job layout and launchers of the differentiable refinement.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "host/ident.hpp"

namespace cctagx {

struct GradJobDev {
  const uint32_t* quad;  // the marker's image (level 0) as quads (bytes (x, y), (x+1, y),
                         // (x, y+1), (x+1, y+1) of word (x, y)), row-major, width iw
  int iw, ih;
  float Q11, Q22, Q33;             // canonic form of the outer ellipse
  float t_can[9], t_inv_can[9];    // image <-> canonic frame
  float begin_sig, end_sig;
  float alpha0;                    // first step of the centre descent, px
  int n_cuts;
  float c0x, c0y;                  // initial imaged centre
  float2 stops[kMaxCuts];
};

// The rows of a host image to the device (room for `capacity` bytes, at least
// width * height): as they lie, one transfer, when they fit with their stride,
// else packed row by row (a 2-D copy from pageable memory takes about 9 us a
// row).  *pitch: the device rows' distance.
hipError_t upload_rows(uint8_t* dst, size_t capacity, const uint8_t* src, int width, int height,
                       size_t stride, hipStream_t s, size_t* pitch);
// The quads of a w x h image (w, h >= 2, rows `pitch` bytes apart) into quad
// (w * h words).
int launch_quads(const uint8_t* img, int w, int h, size_t pitch, uint32_t* quad, hipStream_t s);
// max_cuts: the most cuts of a job.
int launch_grad_eval(const GradJobDev* jobs, int n, const float* H, int max_cuts, int n_samples,
                     bool fp64, double* cost, double* grad, hipStream_t s);
int launch_grad_homography(const GradJobDev* jobs, int n, const float* centers, float* H,
                           hipStream_t s);
// start (2 per marker) = coarse[coarse_of[m]] when coarse_of[m] >= 0, else
// the job's c0.
int launch_grad_start(const GradJobDev* jobs, int n, const int* coarse_of, const float* coarse,
                      float* start, hipStream_t s);
// How the descent samples: in float at positions relative to the marker
// (local), in float at image positions (image: the identification's), or in
// double.
enum class GradSampling { local, image, fp64 };
// `steps` descent steps per marker from start (2 per marker) or, when start
// is null, from the job's c0.
int launch_grad_descend(const GradJobDev* jobs, int n, int steps, int max_cuts, int n_samples,
                        GradSampling sampling, const float* start, float* centers, double* cost,
                        hipStream_t s);

}  // namespace cctagx
