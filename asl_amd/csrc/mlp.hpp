// Launchers of the closure-network training kernels (mlp.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace aslhip {

constexpr int MLP_GRAD_BLOCK = 256;   // lanes of a gradient workgroup (4 wavefronts of 32 samples at a time)
constexpr int MLP_PSTRIDE = 1376;     // floats per workgroup partial: 1345 gradients + loss, whole 128-byte lines

struct MlpGradArgs {
  const float *x;        // n x 7 normalised inputs
  const float *t;        // n targets
  long long n;           // samples in the data set
  long long first;       // seed == 0: the batch is samples first .. first+count-1
  unsigned long long seed;  // else: sample k of the batch is mix64-hashed from (seed, k)
  int count;             // samples in the batch
  float inv_batch;       // 1 / count
  const float *p;        // parameters (FP32)
  float *partial;        // nblocks x MLP_PSTRIDE
};

struct AdamArgs {
  float lr, beta1, beta2, eps;
  float bc1, bc2;  // 1 - beta1^t, 1 - beta2^t
};

// Workgroups (partial sums) of a batch of count samples.
int mlp_grad_blocks(int count);
hipError_t launch_mlp_grad(const MlpGradArgs &a, hipStream_t s);
hipError_t launch_mlp_reduce(const float *partial, int nblocks, double inv_count, float *grad, double *loss,
                             hipStream_t s);
// The reduction followed by an Adam step of the parameters p (moments m, v).
hipError_t launch_mlp_reduce_adam(const float *partial, int nblocks, double inv_count, float *grad, double *loss,
                                  float *p, float *m, float *v, const AdamArgs &a, hipStream_t s);

}  // namespace aslhip
