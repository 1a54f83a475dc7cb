// letkf_eig.h -- helpers shared by the transform kernels (letkf_eig.hip,
// letkf_sqrt.hip).
#pragma once
#include "letkf_device.h"
#include "letkf_kernels.h"

namespace dida {

// Keeps x in registers here, in program order: the unrolled blocks of these
// kernels are long runs of pure arithmetic, which the compiler otherwise
// gathers far from their loads, and spills.
__device__ __forceinline__ void pin(double& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void pin(d4& x) { asm volatile("" : "+v"(x)); }

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

// trans and overline_w of a failed analysis
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

// Products with a vector that every lane needs all of, without reading it from
// LDS entry by entry: x holds x(16 t + i) in lane i of every row of 16 lanes,
// and row_newbcast takes entry n of it as an operand of the FMA.  (Broadcast
// reads cost a wavefront's full LDS bandwidth each; the four wavefronts of a
// CU's SIMDs share one LDS.)  The two wait states before the first DPP read
// cover a register copy the compiler may place right before the block.
#define DIDA_DPP_FMA(d, x, a, n) \
  "v_fmac_f64_dpp %" #d ", %" #x ", %" #a " row_newbcast:" #n " row_mask:0xf bank_mask:0xf\n\t"
// p_(c mod 4) += x(8 HI + c) a[c], c = 0..7
template <int HI>
__device__ __forceinline__ void bcast_dot8(double (&p)[4], double x, const double* a) {
  if constexpr (HI == 0) {
    asm("s_nop 1\n\t" DIDA_DPP_FMA(0, 4, 5, 0) DIDA_DPP_FMA(1, 4, 6, 1) DIDA_DPP_FMA(2, 4, 7, 2)
            DIDA_DPP_FMA(3, 4, 8, 3) DIDA_DPP_FMA(0, 4, 9, 4) DIDA_DPP_FMA(1, 4, 10, 5)
                DIDA_DPP_FMA(2, 4, 11, 6) DIDA_DPP_FMA(3, 4, 12, 7)
        : "+&v"(p[0]), "+&v"(p[1]), "+&v"(p[2]), "+&v"(p[3])
        : "v"(x), "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]),
          "v"(a[7]));
  } else {
    asm("s_nop 1\n\t" DIDA_DPP_FMA(0, 4, 5, 8) DIDA_DPP_FMA(1, 4, 6, 9) DIDA_DPP_FMA(2, 4, 7, 10)
            DIDA_DPP_FMA(3, 4, 8, 11) DIDA_DPP_FMA(0, 4, 9, 12) DIDA_DPP_FMA(1, 4, 10, 13)
                DIDA_DPP_FMA(2, 4, 11, 14) DIDA_DPP_FMA(3, 4, 12, 15)
        : "+&v"(p[0]), "+&v"(p[1]), "+&v"(p[2]), "+&v"(p[3])
        : "v"(x), "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]),
          "v"(a[7]));
  }
}
// a[c] += x(8 HI + c) f, c = 0..7
template <int HI>
__device__ __forceinline__ void bcast_axpy8(double* a, double x, double f) {
  if constexpr (HI == 0) {
    asm("s_nop 1\n\t" DIDA_DPP_FMA(0, 8, 9, 0) DIDA_DPP_FMA(1, 8, 9, 1) DIDA_DPP_FMA(2, 8, 9, 2)
            DIDA_DPP_FMA(3, 8, 9, 3) DIDA_DPP_FMA(4, 8, 9, 4) DIDA_DPP_FMA(5, 8, 9, 5)
                DIDA_DPP_FMA(6, 8, 9, 6) DIDA_DPP_FMA(7, 8, 9, 7)
        : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3]), "+&v"(a[4]), "+&v"(a[5]),
          "+&v"(a[6]), "+&v"(a[7])
        : "v"(x), "v"(f));
  } else {
    asm("s_nop 1\n\t" DIDA_DPP_FMA(0, 8, 9, 8) DIDA_DPP_FMA(1, 8, 9, 9) DIDA_DPP_FMA(2, 8, 9, 10)
            DIDA_DPP_FMA(3, 8, 9, 11) DIDA_DPP_FMA(4, 8, 9, 12) DIDA_DPP_FMA(5, 8, 9, 13)
                DIDA_DPP_FMA(6, 8, 9, 14) DIDA_DPP_FMA(7, 8, 9, 15)
        : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3]), "+&v"(a[4]), "+&v"(a[5]),
          "+&v"(a[6]), "+&v"(a[7])
        : "v"(x), "v"(f));
  }
}
#undef DIDA_DPP_FMA

}  // namespace dida
