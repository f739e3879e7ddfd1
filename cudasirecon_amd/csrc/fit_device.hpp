// Device helpers shared by the k0 search's kernels (stages_k0.hip) and the
// line searches on the device (stages_fit.hip).
#pragma once
#include "device_math.hpp"
#include "stages.hpp"

namespace simr {

__device__ __forceinline__ void better(float& v, int& i, float v2, int i2) {
  if (v2 > v || (v2 == v && i2 < i)) {
    v = v2;
    i = i2;
  }
}

__device__ __forceinline__ float intensity(float2 a) {
#pragma clang fp contract(off)
  return a.x * a.x + a.y * a.y;
}

// The fit's results into host memory, then the completion flag; by one
// workgroup, after a barrier behind its last writes of amps and corr.
__device__ __forceinline__ void fit_publish(const FitState* fs, const FitPub& pub, const float2* amps,
                                            const float* corr) {
  FitOut* out = pub.out;
  const int t = threadIdx.x;
  if (t < pub.ndirs) {
    const FitDir& f = fs->d[t];
    out->k0[t] = f.k0;
    out->kov[t] = f.kov;
    out->n_angle_evals[t] = f.n_angle_evals;
    out->n_mag_evals[t] = f.n_mag_evals;
    out->n_reductions[t] = f.n_reductions;
  }
  for (int i = t; i < pub.ndirs * pub.norders; i += blockDim.x) {
    out->amps[i] = amps[i];
    out->corr[i] = corr[i];
  }
  if (t == 0) {
    int ndone = 0, rounds = 0, over = 0;
    for (int d = 0; d < pub.ndirs; ++d) {
      ndone += fs->d[d].phase == kFitDone ? 1 : 0;
      rounds = max(rounds, fs->d[d].rounds);
      over |= fs->d[d].overflow;
    }
    out->ndone = ndone;
    out->rounds = rounds;
    out->overflow = over;
  }
  __threadfence_system();  // out is host memory
  __syncthreads();
  if (t == 0) __hip_atomic_store(pub.flag, pub.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace simr
