// Sampled Kullback-Leibler value and gradient around the batched evaluation.
#pragma once
#include "common.hpp"

namespace jubik {

// Two latent fields (the second NULL without a spectral index), n values each.
struct KlFields {
  const void* xbar[2];   // mean (n)
  const void* delta[2];  // sample offsets (S, n)
  void* pos[2];          // positions (S, n)
  const void* grad[2];   // gradients at the positions (S, n)
  void* out[2];          // mean gradient (n)
};

// pos[s] = xbar + delta[s]; prior[0] (host or device) = sum of all pos^2,
// through at most max_partial FP64 partials in ``work``, in a fixed order.
int kl_positions(int dtype, int S, int64_t n, const KlFields& f, double* work,
                 int64_t max_partial, double* prior, hipStream_t s);
// out = mean over s of (grad[s] + pos[s]), summed in FP64.
int kl_mean(int dtype, int S, int64_t n, const KlFields& f, hipStream_t s);

}  // namespace jubik
