// letkf_eig.h -- helpers shared by the transform kernels (letkf_eig.hip,
// letkf_sqrt.hip).
#pragma once
#include "letkf_device.h"
#include "letkf_kernels.h"

namespace dida {

// The analysis of workgroup (or lane) `slot`: a = global index, ai = index of
// the batch-local inputs (A, b, refl, tau, d, e), ar = index of the pass's own
// scratch (rot, hdr, nchase, lam).  False when the slot holds no analysis.
__device__ __forceinline__ bool eig_slot(const EigParams& p, long long slot, long long& a,
                                         long long& ai, long long& ar) {
  if (p.list) {
    const int n = min(*p.list_n, p.list_cap);
    if (slot >= n) return false;
    a = p.list[slot];
    ai = a - p.a0;
    ar = slot;
  } else {
    if (slot >= p.n_an) return false;
    a = p.a0 + slot;
    ai = slot;
    ar = slot;
  }
  return true;
}

// trans and overline_w of an analysis whose eigensolve failed on both passes
__device__ __forceinline__ void nan_transform(const EigParams& p, long long a) {
  const int k = p.k;
  const double nan = __longlong_as_double(0x7ff8000000000000LL);
  if (p.trans_out)
    for (int e = threadIdx.x; e < k * k; e += blockDim.x) p.trans_out[a * (long long)k * k + e] = nan;
  if (p.w_out)
    for (int e = threadIdx.x; e < k; e += blockDim.x) p.w_out[a * (long long)k + e] = nan;
}

// offset (in doubles) of tile (I, J) register r of lane l in a trans block
template <int KMAX>
__device__ __forceinline__ int tile_off(int I, int J, int r, int l) {
  return ((I * (KMAX / 16) + J) * 4 + r) * 64 + l;
}

}  // namespace dida
