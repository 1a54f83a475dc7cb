// letkf_eig.hip -- the transform of a batch of local analyses and the ensemble
// update: tridiagonalisation, the QL of indefinite matrices, the update, and the
// launches.
//
// The k x k matrices M = A + (k-1)/rho I of one batch are reduced to
// tridiagonal form, and trans and overline_w follow from that form:
//
//   k_tridiag   one wavefront per matrix (k <= 32: two), lane r keeps row r of A
//               in VGPRs; writes the reflectors, tau, and the tridiagonal (d, e)
//   k_vec       trans and overline_w from the inverse square root of the
//               tridiagonal form and its reflectors (letkf_sqrt.hip, with
//               k_lmin before it for the reduced precisions' guard)
//   k_update    the ensemble update xa = trans^T xb + axb, re-centred
//               (xb_2_xa, letkf_compute.F90:259-329, or the per-level update
//               of the vertical loop, letkf_compute.F90:501-552)
// k = 65..128 runs k_tridiag128 and k_update128 with half rows per thread
// (256 threads per matrix).
//
// A matrix whose M is finite but not positive definite goes to k_indef, which
// diagonalises it by implicit QL with Wilkinson shift (Golub & Van Loan Alg.
// 8.3.1, Sec. 8.3.5; Bowdler, Martin, Reinsch & Wilkinson 1968) from its
// tridiagonal form, before the update and with no host synchronisation.  An
// analysis whose QL does not converge, or whose M or overline_w is not finite,
// leaves xa = xb, axa = axb for its state and NaN in trans/overline_w; the
// caller gets the count.
//
// With the QL limits lowered from the environment (EigParams::ql_first) the
// first pass is the QL recurrence for every matrix, so that its flag paths can
// be tested; the matrices it flags go to a device-side list and a second,
// list pass with twice the limits:
//
//   k_ql_log    one LANE per matrix (64 matrices per wavefront): the scalar
//               QL recurrence, which is a serial chain per matrix; writes the
//               eigenvalues and a log of the Givens rotations of every chase
//   k_rot       one wavefront per matrix (k <= 64; k_rot128 above), lane r
//               keeps row r of Z in VGPRs: Q = H_0 ... H_{k-3} by forward
//               accumulation, the logged rotations applied in order (V = Q Z),
//               then overline_w = V diag(1/lambda) V^T b and
//               trans = V diag(sqrt((k-1)/lambda)) V^T + overline_w 1^T
//               (letkf_core.F90:129-225) on f64 MFMA
#include <algorithm>

#include "letkf_device.h"
#include "letkf_kernels.h"
#include "letkf_eig.h"

namespace dida {

__global__ void k_zero_ints(int* __restrict__ p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// State rows of one analysis: the columns of its cube and, on the vertical
// loop, the levels of its chunk (with the 2-D variables on the top chunk).
struct AnRows {
  int sj, ej, si, ei, sk, ek;
  long long lat_ext;
};
__device__ __forceinline__ AnRows an_rows(const EigParams& p, long long a) {
  AnRows r;
  const int ah = (int)(a / p.nzc), kc = (int)(a % p.nzc);
  const int ic = ah % p.g.nlat_c, jc = ah / p.g.nlat_c;
  cube_span(p.g, ic, p.g.nlat, &r.sj, &r.ej);
  cube_span(p.g, jc, p.g.nlon, &r.si, &r.ei);
  r.lat_ext = p.g.nlat + 2 * p.halo;
  r.sk = 1;
  r.ek = p.nz;
  if (p.vertical) {
    r.sk = kc * p.cube_nz + 1;
    r.ek = min(r.sk + p.cube_nz - 1, p.nz);
  }
  return r;
}

// ---------------------------------------------------------------------------
// k_tridiag
// ---------------------------------------------------------------------------
// arow[c] for a wavefront-uniform column c: a switch lowered to a short tree
// of scalar branches (no per-column selects or dynamic register indexing)
template <int N>
__device__ __forceinline__ double pick_column(const double (&arow)[N], int c) {
  double x = 0.0;
  switch (c) {
#define DIDA_COL_CASE(i) \
  case i:                \
    if constexpr (i < N) x = arow[i]; \
    break;
#define DIDA_COL_CASE8(b) \
  DIDA_COL_CASE(b) DIDA_COL_CASE(b + 1) DIDA_COL_CASE(b + 2) DIDA_COL_CASE(b + 3) \
  DIDA_COL_CASE(b + 4) DIDA_COL_CASE(b + 5) DIDA_COL_CASE(b + 6) DIDA_COL_CASE(b + 7)
    DIDA_COL_CASE8(0) DIDA_COL_CASE8(8) DIDA_COL_CASE8(16) DIDA_COL_CASE8(24)
    DIDA_COL_CASE8(32) DIDA_COL_CASE8(40) DIDA_COL_CASE8(48) DIDA_COL_CASE8(56)
#undef DIDA_COL_CASE8
#undef DIDA_COL_CASE
    default:
      break;
  }
  return x;
}

// Sum over the KMAX lanes of a matrix (all lanes active): rows of 16 on DPP,
// then the rows by shuffles.
template <int KMAX>
__device__ __forceinline__ double matrix_sum(double v) {
  v += dpp_d<0xB1>(v);     // quad_perm [1,0,3,2]
  v += dpp_d<0x4E>(v);     // quad_perm [2,3,0,1]
  v += dpp_d<0x141>(v);    // row_half_mirror
  v += dpp_d<0x140>(v);    // row_mirror
  v += __shfl_xor(v, 16, 64);
  return KMAX == 64 ? v + __shfl_xor(v, 32, 64) : v;
}

// k = 64: one matrix per wavefront; k <= 32: two, one per half (with one, half
// the lanes had no row).  Per step the products and the update take v and w
// as row broadcasts of the FMA (bcast_dot8, bcast_axpy8): w and v go through
// LDS once, and each lane reads the NT entries of them that its row of 16
// broadcasts.  Read entry by entry from LDS, the four SIMDs' 48 broadcast
// reads a step bound the kernel; now VALU issue does (14.8k instructions per
// wavefront, 6.1k of them FMAs).  64,800 matrices of k = 64: 3.25 -> 2.25 ms,
// the same bits; 2,073,600 of k = 32: 37.5 -> 11.9 ms.
template <int KMAX>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(KMAX == 64 ? 3 : 4)))
void k_tridiag(EigParams p) {
  constexpr int NT = KMAX / 16, MPW = 64 / KMAX;
  __shared__ double sv[64], sw[64];
  __shared__ double se_s[64], st_s[64];
  __shared__ double sxn[64];             // column j+1 after step j's update
  const int lane = threadIdx.x, r = lane & (KMAX - 1), m0 = lane - r;
  const long long nal = (long long)blockIdx.x * MPW + (m0 ? 1 : 0);
  // a wavefront's second matrix past the batch's end repeats the last one,
  // storing nothing
  const bool valid = MPW == 1 || nal < p.n_an;
  const long long al = valid ? nal : p.n_an - 1;
  const int k = p.k, kp = p.kp;
  const double* __restrict__ Ag = p.A + al * (long long)kp * kp;
  double* __restrict__ refl = p.refl + al * (long long)kp * kp;
  const bool in_r = r < k;
  const double* const svr = sv + m0 + (lane & 15);
  const double* const swr = sw + m0 + (lane & 15);

  double arow[KMAX];
  if (p.a_f32) {
    // FP32 in tile order (a_entry; kp = KMAX): one base address per lane and
    // a constant offset per column, every load unconditional and in bounds,
    // then a select
    const float* __restrict__ Af = reinterpret_cast<const float*>(Ag) + a_tile_pos(r, KMAX);
    float av[KMAX];
#pragma unroll
    for (int c = 0; c < KMAX; ++c) av[c] = Af[a_tile_pos(c, KMAX) * KMAX];
#pragma unroll
    for (int c = 0; c < KMAX; ++c) arow[c] = (in_r && c < k) ? (double)av[c] : 0.0;
  } else {
    // (kp = KMAX here too) the pins keep the loads out of the selects: a load
    // under the select's test waits for the one before it
#pragma unroll
    for (int c = 0; c < KMAX; ++c) arow[c] = Ag[(long long)c * KMAX + r];
#pragma unroll
    for (int c = 0; c < KMAX; ++c) pin(arow[c]);
#pragma unroll
    for (int c = 0; c < KMAX; ++c) arow[c] = (in_r && c < k) ? arow[c] : 0.0;
  }
  sxn[lane] = arow[0];
  se_s[lane] = st_s[lane] = 0.0;
  __syncthreads();

  for (int j = 0; j + 2 < k; ++j) {
    const bool act = in_r && r > j;
    const double xcol = sxn[lane], x0 = sxn[m0 + j + 1];
    const double x = act ? xcol : 0.0;
    const double rest = matrix_sum<KMAX>((act && r > j + 1) ? x * x : 0.0);
    __builtin_amdgcn_sched_barrier(0);
    // a column already in tridiagonal form (rest = 0) takes the same path with
    // v = 0 and tau = 0: the update is then exactly the identity
    const bool none = rest == 0.0;
    const double nrm = sqrt(rest + x0 * x0);
    const double alpha = (x0 >= 0.0) ? -nrm : nrm;
    const double v0 = x0 - alpha;
    const double tau = none ? 0.0 : 2.0 / (rest + v0 * v0);
    const double v = (act && !none) ? ((r == j + 1) ? v0 : x) : 0.0;
    sv[lane] = v;
    __syncthreads();
    double vt[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) vt[t] = svr[16 * t];
    // p = tau A v over the trailing columns (v is zero for c <= j); four
    // partial sums
    double pr4[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if (16 * t + 7 > j) bcast_dot8<0>(pr4, vt[t], arow + 16 * t);
      if (16 * t + 15 > j) bcast_dot8<1>(pr4, vt[t], arow + 16 * t + 8);
    }
    double pr = (pr4[0] + pr4[1]) + (pr4[2] + pr4[3]);
    pr = act ? pr * tau : 0.0;
    const double K = 0.5 * tau * matrix_sum<KMAX>(v * pr);
    __builtin_amdgcn_sched_barrier(0);
    const double wr = act ? pr - K * v : 0.0;
    sw[lane] = wr;
    if (valid) refl[(long long)j * kp + r] = v;
    if (r == 0) { se_s[m0 + j] = none ? x0 : alpha; st_s[m0 + j] = tau; }
    __syncthreads();
    // rank-2 update A -= v w^T + w v^T (v and w are zero for c <= j); column
    // j+1 goes through LDS after the whole update
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const double wt = swr[16 * t];
      if (16 * t + 7 > j) {
        bcast_axpy8<0>(arow + 16 * t, wt, -v);
        bcast_axpy8<0>(arow + 16 * t, vt[t], -wr);
      }
      if (16 * t + 15 > j) {
        bcast_axpy8<1>(arow + 16 * t + 8, wt, -v);
        bcast_axpy8<1>(arow + 16 * t + 8, vt[t], -wr);
      }
    }
    sxn[lane] = pick_column(arow, j + 1);
    __syncthreads();
  }
  // diagonal and the last subdiagonal entry
  double dr = 0.0, ek2 = 0.0;
#pragma unroll
  for (int c = 0; c < KMAX; ++c) {
    dr = (c == r) ? arow[c] : dr;
    ek2 = (c == k - 2) ? arow[c] : ek2;
  }
  sxn[lane] = ek2;
  __syncthreads();
  ek2 = sxn[m0 + k - 1];
  if (!valid) return;
  p.d[al * kp + r] = in_r ? dr : 0.0;
  p.e[al * kp + r] = r == k - 2 ? ek2 : se_s[lane];
  p.tau[al * kp + r] = st_s[lane];
}

// ---------------------------------------------------------------------------
// k_ql_log: one lane per matrix
// ---------------------------------------------------------------------------
// d and e of the 64 matrices live in LDS as [i][lane], behind one padding
// row (index -1) so that the sweep's prefetch of i - 1 stays in bounds at
// i = 0.
template <int KMAX>
__global__ __launch_bounds__(64) void k_ql_log(EigParams p) {
  __shared__ double sd_l[KMAX + 1][64];
  __shared__ double se_l[KMAX + 1][64];
  const int lane = threadIdx.x;
#define SD(i) sd_l[(i) + 1][lane]
#define SE(i) se_l[(i) + 1][lane]
  SD(-1) = 0.0;
  SE(-1) = 0.0;
  long long a = 0, ai = 0, ar = 0;
  const bool valid = eig_slot(p, (long long)blockIdx.x * 64 + lane, a, ai, ar);
  const int k = p.k, kp = p.kp;
  double tnorm = 0.0;
  for (int i = 0; i < KMAX; ++i) {
    double dv = 0.0, ev = 0.0;
    if (valid && i < k) {
      dv = p.d[ai * kp + i];
      ev = p.e[ai * kp + i];
    }
    SD(i) = dv;
    SE(i) = ev;
    tnorm = fmax(tnorm, fabs(dv) + fabs(ev));
  }
  if (!valid) return;
  const double eps = 2.220446049250313e-16;
  double2* __restrict__ rot = p.rot + ar * (long long)p.rot_cap;
  int4* __restrict__ hdr = p.hdr + ar * (long long)p.hdr_cap;
  int nrot = 0, nhdr = 0, status = 0;
  for (int l = 0; l < k && status == 0; ++l) {
    int iter = 0;
    for (;;) {
      // first m >= l with a negligible e[m] (a loop with one exit: no
      // per-iteration break bookkeeping)
      int m = l;
      double dm = SD(l);
      bool go = m < k - 1;
      while (go) {
        const double dm1 = SD(m + 1);
        const double em = fabs(SE(m));
        go = !(em <= eps * (fabs(dm) + fabs(dm1)) || em <= eps * tnorm);
        if (go) {
          ++m;
          dm = dm1;
          go = m < k - 1;
        }
      }
      if (m == l) break;
      if (++iter > p.max_iter) { status = l + 1; break; }
      if (nhdr >= p.hdr_cap || nrot + (m - l) + 14 > p.rot_cap) { status = kStatusLogFull; break; }
      double g = (SD(l + 1) - SD(l)) / (2.0 * SE(l));
      double r = hypot(g, 1.0);
      g = SD(m) - SD(l) + SE(l) / (g + (g >= 0.0 ? fabs(r) : -fabs(r)));
      double s = 1.0, c = 1.0, pp = 0.0;
      // the chase's log is block-aligned: positions m .. 8 ceil(m/8) - 1
      // (above it) and 8 floor(lo/8) .. lo - 1 (below) hold the identity, so
      // a reader takes whole blocks of 8 positions without masking
      const int off = nrot;
      for (int q = ((m + 7) & ~7) - 1; q >= m; --q) rot[nrot++] = make_double2(1.0, 0.0);
      int i = m - 1;
      bool underflow = false;
      int iu = l - 1;
      // d[i], e[i] of the next step are read before this step's stores.  The
      // body is straight-line: pointers walk down the lane's LDS column and
      // its log, and an underflow (r2 == 0, rare) is repaired after the
      // step's stores under a wavefront-uniform test, then ends the lane's
      // loop; so the lanes' divergence costs one exit test per step
      double ei = SE(i), di = SD(i), di1 = SD(i + 1);
      double* pd = &SD(i);
      double* pe = &SE(i);
      double2* pr = rot + nrot;
      for (; i >= l; --i, pd -= 64, pe -= 64, ++pr) {
        const double ein = pe[-64], din = pd[-64];
        const double f = s * ei, bb = c * ei;
        // one reciprocal square root instead of sqrt and a divide on the
        // serial chain: r = sqrt(f^2 + g^2), s = f / r, c = g / r
        const double r2 = fma(f, f, g * g);
        const double rinv = rsqrt(r2);
        const double sd_uz = di1 - pp;
        s = f * rinv;
        c = g * rinv;
        g = di1 - pp;
        r = (di - g) * s + 2.0 * c * bb;
        pp = s * r;
        pe[64] = r2 * rinv;
        pd[64] = g + pp;
        g = c * r - bb;
        *pr = make_double2(c, s);
        if (__builtin_amdgcn_ballot_w64(r2 == 0.0)) {
          if (r2 == 0.0) {
            // the chase stops at i: e[i+1] = 0, d[i+1] = d[i+1] - p, no
            // rotation logged for this step
            pe[64] = 0.0;
            pd[64] = sd_uz;
            underflow = true;
            iu = i;
            i = l;
            --pr;
          }
        }
        ei = ein;
        di1 = di;
        di = din;
      }
      nrot = (int)(pr - rot);
      if (underflow) SE(m) = 0.0;
      const int lo = underflow ? iu + 1 : l;
      for (int q = lo - 1; q >= (lo & ~7); --q) rot[nrot++] = make_double2(1.0, 0.0);
      if (m - lo > 0) hdr[nhdr++] = make_int4(lo, m, off, nrot - off);
      else nrot = off;
      if (underflow) continue;
      SD(l) -= pp;
      SE(l) = g;
      SE(m) = 0.0;
    }
  }
  for (int i = 0; i < k; ++i) p.lam[ar * kp + i] = SD(i);
  p.nchase[ar] = nhdr;
  p.status[a] = status;
  if (status != 0 && !p.list) {
    const int s = atomicAdd(p.flag_n, 1);
    if (s < p.flag_cap) p.flag_list[s] = (int)a;
    else p.status[a] = kStatusNotRedone;
    atomicAdd(p.flag_total, 1);
  }
}
#undef SD
#undef SE

// Sum over the NW wavefronts of a workgroup; every thread gets the same value
// (wave sums, then the partials in a fixed order).  `red` holds two slots of
// NW partials so that back-to-back calls need one barrier each.
template <int NW>
__device__ __forceinline__ double block_sum(double v, double* red, int& slot) {
  const double w = wave_sum_full(v);
  if constexpr (NW == 1) {
    return uniform(w);
  } else {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) red[NW * slot + wv] = w;
    __syncthreads();
    double r = red[NW * slot];
#pragma unroll
    for (int i = 1; i < NW; ++i) r += red[NW * slot + i];
    slot ^= 1;
    return uniform(r);
  }
}

// ---------------------------------------------------------------------------
// k_rot (ql_first): V (Q accumulation, logged rotations), overline_w and
// trans = T + overline_w 1^T with LDS staged in small chunks, trans written
// in the register layout of the update's MFMA B operand over the analysis'
// reflector block (consumed by then), as k_vec does.  k_update streams the
// state vectors of the analysis through that operand.
// ---------------------------------------------------------------------------
// The rotations of positions 8B .. 8B+7 of a chase: the log holds whole
// blocks of 8 positions (identity outside the chase), position i at ring
// entry base - i, so a block is eight consecutive entries read from one
// address (the ring keeps a copy of its first 8 entries past its end, so a
// run never wraps).  base is wavefront-uniform.
template <int RING>
__device__ __forceinline__ void ring_block(const double2* sring, int base, int B,
                                           double2 (&cs)[8]) {
  const double2* e = sring + ((base - 8 * B - 7) & (RING - 1));
#pragma unroll
  for (int t = 0; t < 8; ++t) cs[t] = e[7 - t];
}

// Read-only global memory addressed uniformly across the wavefront: loads
// through these pointer types go to the scalar unit (s_load).  Only for data
// that no kernel writes while the reader runs.
typedef const __attribute__((address_space(4))) int* uniform_int_cptr;
typedef const __attribute__((address_space(4))) double* uniform_dbl_cptr;
// a row of zeros in read-only global memory, for scalar reads past the last
// reflector
__device__ const double kZeroRow[128] = {};
__device__ __forceinline__ int4 load_uniform_int4(uniform_int_cptr q, int i) {
  return make_int4(q[4 * i], q[4 * i + 1], q[4 * i + 2], q[4 * i + 3]);
}

template <int KMAX>
struct VecLds {
  static constexpr int LDV = KMAX + 1;
  static constexpr int RING = 8 * KMAX;              // rotation ring (entries)
  static constexpr int REFILL = RING / 2;
  static constexpr int A = 16 * LDV;                 // 16 reflectors
  static constexpr int B = 2 * (RING + 8);          // rotation ring + its mirrored head
  static constexpr int C = 16 * LDV;                 // 16 columns of V
  static constexpr int N = (A > B ? (A > C ? A : C) : (B > C ? B : C));
};

template <int KMAX>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
void k_rot(EigParams p) {
  constexpr int NB = KMAX / 8;
  constexpr int TT = KMAX / 16;
  constexpr int IPP = TT < 2 ? TT : 2;               // tile rows per pass
  using L = VecLds<KMAX>;
  constexpr int LDV = L::LDV, RING = L::RING, REFILL = L::REFILL;
  static_assert(REFILL >= KMAX + 16 && REFILL % 64 == 0, "a refill covers any chase");
  __shared__ __align__(16) double sbuf[L::N];
  // stage C's vectors share one array with stage A's Gram matrices (16 x 16),
  // which are dead by then
  constexpr int NSC = 5 * KMAX > 256 ? 5 * KMAX : 256;
  __shared__ double ssc[NSC], stau[KMAX];
  double* const sf = ssc;
  double* const sg = ssc + KMAX;
  double* const sb = ssc + 2 * KMAX;
  double* const st = ssc + 3 * KMAX;
  double* const sw = ssc + 4 * KMAX;
  double* const sgram = ssc;
  const int lane = threadIdx.x;
  long long a, ai, ar;
  if (!eig_slot(p, blockIdx.x, a, ai, ar)) return;
  if (p.status[a] != 0) {                // redone by the list pass, or failed
    if (p.list || p.status[a] == kStatusNotRedone) nan_transform(p, a);
    return;
  }
  const int k = p.k, kp = p.kp;
  const bool in_r = lane < k;
  double* __restrict__ refl = p.refl + ai * (long long)kp * kp;
  const double* __restrict__ tg = p.tau + ai * kp;
  const int nref = k > 2 ? k - 2 : 0;

  // ---- A. Z <- Z H_j, reflectors staged 16 at a time ----
  // The next 16 reflectors are loaded into registers while the current 16
  // are applied, so their memory latency is hidden behind the work.
  if (lane < nref) stau[lane] = tg[lane];
  double z[KMAX];
#pragma unroll
  for (int c = 0; c < KMAX; ++c) z[c] = (c == lane) ? 1.0 : 0.0;
  double vnext[16];
#pragma unroll
  for (int t = 0; t < 16; ++t)
    vnext[t] = (t < nref && lane < KMAX) ? refl[(long long)t * kp + lane] : 0.0;
  // Reflectors apply in groups of four: the four dots from the same z, each
  // corrected by the earlier ones' scales times the pairwise products
  // v_s . v_t (the dot with z as the earlier reflectors of the group left
  // it), then one pass z -= sum_t alpha_t v_t.  A group is one dependent
  // step instead of four.  The products v_s . v_t of a staged block are its
  // Gram matrix V^T V, one f64 MFMA 16x16x4 per four columns.
  for (int j0 = 0; j0 < nref; j0 += 16) {
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 16; ++t)
      if (lane < KMAX) sbuf[t * LDV + lane] = vnext[t];
    __syncthreads();
    {
      const int i16 = lane & 15, q = lane >> 4;
      d4 g = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s4 = 0; s4 < KMAX / 4; ++s4) {
        const double v = sbuf[i16 * LDV + 4 * s4 + q];      // V[4 s4 + q][i16]
        g = __builtin_amdgcn_mfma_f64_16x16x4f64(v, v, g, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) sgram[(q + 4 * r) * 16 + i16] = g[r];
    }
#pragma unroll
    for (int t = 0; t < 16; ++t)
      vnext[t] = (j0 + 16 + t < nref && lane < KMAX) ? refl[(long long)(j0 + 16 + t) * kp + lane]
                                                     : 0.0;
    __syncthreads();
    const int j1 = min(j0 + 16, nref);
    for (int j = j0; j < j1; j += 4) {
      // past nref the staged columns are zero (tau 0), so a short last group
      // runs with zero reflectors
      const int t0 = j - j0;
      double tau[4], al[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) tau[u] = j + u < j1 ? uniform(stau[j + u]) : 0.0;
      // the group's reflector entries are the same for every lane: they are
      // read as scalars (s_load from the reflector block, rows past the last
      // reflector from a zero row) and enter the FMAs as scalar operands, so
      // the group's two passes take no LDS bandwidth
      uniform_dbl_cptr qr[4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        qr[u] = j + u < j1 ? (uniform_dbl_cptr)(refl + (long long)(j + u) * kp)
                           : (uniform_dbl_cptr)kZeroRow;
      double acc[4][2];
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[u][0] = acc[u][1] = 0.0;
#pragma unroll
      for (int B = 0; B < NB; ++B) {
        if (8 * B + 7 <= j) continue;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          const int c = 8 * B + t;
#pragma unroll
          for (int u = 0; u < 4; ++u) acc[u][t & 1] = fma(z[c], qr[u][c], acc[u][t & 1]);
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        double d = acc[u][0] + acc[u][1];
#pragma unroll
        for (int v = 0; v < u; ++v) d = fma(-al[v], uniform(sgram[(t0 + v) * 16 + t0 + u]), d);
        al[u] = d * tau[u];
      }
#pragma unroll
      for (int B = 0; B < NB; ++B) {
        if (8 * B + 7 <= j) continue;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          const int c = 8 * B + t;
          double zc = z[c];
#pragma unroll
          for (int u = 0; u < 4; ++u) zc = fma(-al[u], qr[u][c], zc);
          z[c] = zc;
        }
      }
    }
  }
  __syncthreads();

  // ---- B. logged QL rotations streamed through an LDS ring of REFILL-entry refills ----
  {
    double2* sring = reinterpret_cast<double2*>(sbuf);
    const double2* __restrict__ rot = p.rot + ar * (long long)p.rot_cap;
    // the chase headers are read as scalars (s_load), so waiting for one does
    // not wait for the vector loads of the next refill issued before it
    const uniform_int_cptr hdr =
        (uniform_int_cptr)(p.hdr + (long long)uniform((int)ar) * p.hdr_cap);
    const int nch = uniform(min(p.nchase[ar], p.hdr_cap));
    int nrot = 0;
    if (nch > 0) {
      const int4 hl = load_uniform_int4(hdr, nch - 1);
      nrot = uniform(hl.z + hl.w);
    }
    int committed = 0;
    int4 hn = nch > 0 ? load_uniform_int4(hdr, 0) : make_int4(0, 0, 0, 0);
    // the entries of the next refill, loaded one refill ahead so that the
    // log's memory latency is hidden behind the chases in between
    double2 vnext[REFILL / 64];
#pragma unroll
    for (int t = 0; t < REFILL / 64; ++t) {
      const int e = 64 * t + lane;
      vnext[t] = (e < nrot) ? rot[e] : make_double2(1.0, 0.0);
    }
    for (int ch = 0; ch < nch; ++ch) {
      int4 h = hn;
      h.x = uniform(h.x);
      h.y = uniform(h.y);
      h.z = uniform(h.z);
      h.w = uniform(h.w);
      if (ch + 1 < nch) hn = load_uniform_int4(hdr, ch + 1);
      const int lo = h.x, hi = h.y;
      if (h.z + h.w > committed) {
        __syncthreads();
#pragma unroll
        for (int t = 0; t < REFILL / 64; ++t) {
          const int slot = (committed + 64 * t + lane) & (RING - 1);
          sring[slot] = vnext[t];
          if (slot < 8) sring[RING + slot] = vnext[t];
        }
        committed += REFILL;
#pragma unroll
        for (int t = 0; t < REFILL / 64; ++t) {
          const int e = committed + 64 * t + lane;
          vnext[t] = (e < nrot) ? rot[e] : make_double2(1.0, 0.0);
        }
        __syncthreads();
      }
      const int bhi = (hi - 1) >> 3, blo = lo >> 3;
      const int base = h.z + ((hi + 7) & ~7) - 1;
      double carry = 0.0;
#pragma unroll
      for (int B = NB - 1; B >= 0; --B) {
        if (B > bhi || B < blo) continue;
        const int top = (8 * B + 7 < KMAX - 1) ? 8 * B + 7 : KMAX - 2;
        if (B == bhi) carry = z[top + 1];
        double2 cs[8];
        ring_block<RING>(sring, base, B, cs);
#pragma unroll
        for (int t = 7; t >= 0; --t) {
          const int i = 8 * B + t;
          if (i > KMAX - 2) continue;
          const double zi = z[i];
          // carry is the serial chain: one FMA per step
          z[i + 1] = fma(cs[t].x, carry, cs[t].y * zi);
          carry = fma(-cs[t].y, carry, cs[t].x * zi);
        }
        if (B == blo) z[8 * B] = carry;
      }
    }
  }

  // ---- C. eigenvalue functions (letkf_core.F90:107-113, guard for reduced modes) ----
  double lam = in_r ? p.lam[ar * kp + lane] : 0.0;
  if (p.guard) {
    const double mn = wave_min_full(in_r ? lam : 1e300);
    if (mn < 0.0) lam = lam - mn;
  }
  lam = lam * 1.0 + (double)(k - 1) / p.inflation;
  if (lane < KMAX) {
    sf[lane] = in_r ? sqrt((double)(k - 1) / lam) : 0.0;
    sg[lane] = in_r ? 1.0 / lam : 0.0;
    sb[lane] = in_r ? p.b[ai * kp + lane] : 0.0;
  }
  // T = V diag(f) V^T on f64 MFMA in IPP tile rows per pass; V is staged
  // 16 columns at a time ([column][row] in LDS).  The first pass also forms
  // st = diag(1/lambda) V^T b (letkf_core.F90:129-195 regrouped).
  const int i16 = lane & 15, q = lane >> 4;
  double* sVc = sbuf;
  double wbar = 0.0;
#pragma unroll
  for (int pass = 0; pass < TT / IPP; ++pass) {
    d4 acc[IPP][TT];
#pragma unroll
    for (int I = 0; I < IPP; ++I)
#pragma unroll
      for (int J = 0; J < TT; ++J) acc[I][J] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int c = 0; c < TT; ++c) {
      __syncthreads();
      if (lane < KMAX) {
#pragma unroll
        for (int t = 0; t < 16; ++t) sVc[t * LDV + lane] = z[16 * c + t];
      }
      __syncthreads();
      if (pass == 0 && lane < 16) {
        double tb = 0.0;
        for (int r = 0; r < KMAX; ++r) tb = fma(sVc[lane * LDV + r], sb[r], tb);
        st[16 * c + lane] = tb * sg[16 * c + lane];
      }
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        const int t = 4 * s4 + q;                      // column within the chunk
        const double fc = sf[16 * c + t];
        double fr[TT];
#pragma unroll
        for (int J = 0; J < TT; ++J) fr[J] = sVc[t * LDV + 16 * J + i16];
#pragma unroll
        for (int I = 0; I < IPP; ++I)
#pragma unroll
          for (int J = 0; J < TT; ++J)
            acc[I][J] = __builtin_amdgcn_mfma_f64_16x16x4f64(fr[pass * IPP + I], fc * fr[J],
                                                             acc[I][J], 0, 0, 0);
      }
    }
    if (pass == 0) {
      __syncthreads();
#pragma unroll
      for (int c = 0; c < KMAX; ++c) wbar = fma(z[c], st[c], wbar);
      if (lane < KMAX) sw[lane] = in_r ? wbar : 0.0;
      __syncthreads();
    }
    // trans(f, e) = T(f, e) + overline_w(f)  (letkf_core.F90:221-225)
#pragma unroll
    for (int I = 0; I < IPP; ++I)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double wf = sw[16 * (pass * IPP + I) + q + 4 * r];
#pragma unroll
        for (int J = 0; J < TT; ++J) acc[I][J][r] += wf;
      }
    if (p.trans_out) {
      double* tr = p.trans_out + a * (long long)k * k;
#pragma unroll
      for (int I = 0; I < IPP; ++I)
#pragma unroll
        for (int J = 0; J < TT; ++J)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int f = 16 * (pass * IPP + I) + q + 4 * r, e = 16 * J + i16;
            if (f < k && e < k) tr[(long long)e * k + f] = acc[I][J][r];
          }
    }
    if (p.xb || p.xb32) {
      // the B operand of the update, over the (consumed) reflector block; for
      // the FP32 state in FP32 (the update rounds it to FP32 anyway), half
      // the bytes to write here and to read there
      if (p.state_f32) {
        float* const rf = reinterpret_cast<float*>(refl);
#pragma unroll
        for (int I = 0; I < IPP; ++I)
#pragma unroll
          for (int J = 0; J < TT; ++J)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              rf[tile_off<KMAX>(pass * IPP + I, J, r, lane)] = (float)acc[I][J][r];
      } else {
#pragma unroll
        for (int I = 0; I < IPP; ++I)
#pragma unroll
          for (int J = 0; J < TT; ++J)
#pragma unroll
            for (int r = 0; r < 4; ++r) refl[tile_off<KMAX>(pass * IPP + I, J, r, lane)] = acc[I][J][r];
      }
    }
  }
  if (__builtin_amdgcn_ballot_w64(in_r && !__builtin_isfinite(wbar))) {
    __syncthreads();                               // the trans writes above are done
    if (lane == 0) p.status[a] = kStatusNonFinite;
    nan_transform(p, a);
    return;
  }
  if (p.w_out && in_r) p.w_out[a * (long long)k + lane] = wbar;
}

// ---------------------------------------------------------------------------
// k_indef: the matrices k_vec found finite but not positive definite
// (kStatusIndefinite: R^-1 < 0, or an M so ill conditioned that its smallest
// eigenvalue is rounding), by QL with Wilkinson shift from their tridiagonal
// form, as k_ql_log and k_rot, however many there are.
// ---------------------------------------------------------------------------
// A workgroup takes every gridDim-th matrix of the batch that carries the
// status: thread 0 runs the QL recurrence a chase at a time, thread r applies
// the chase's rotations to row r of Z in LDS.  Rare, so plain (a log of the
// rotations, which k_ql_log keeps per matrix, would be four times the matrix);
// a batch without such a matrix pays the launch and one read.  The bound is
// thread 0's chain, one matrix per workgroup that fits the LDS: 4,050 of k = 20
// 1.2 ms, of k = 64 4.7 ms, of k = 128 40 ms (the QL pass of a whole batch took
// 0.4, 2.0 and 4.5).  Runs before the update, which then takes every analysis
// in one pass.
template <int KMAX>
__global__ __launch_bounds__(KMAX < 64 ? 64 : KMAX) void k_indef(EigParams p) {
  if (*p.flag_n == 0) return;
  __shared__ double sZ[KMAX * KMAX];                 // column-major: Z(r, c) at c KMAX + r
  __shared__ double sd[KMAX], se[KMAX], sv[KMAX], sb[KMAX], sw[KMAX];
  __shared__ double2 srot[KMAX];                     // (c, s) of position i of the chase
  __shared__ int s_lo, s_hi, s_end;                  // the chase; s_end: no chase left
  const int r = threadIdx.x;
  const bool row = r < KMAX;
  const int k = p.k, kp = p.kp;
  const double eps = 2.220446049250313e-16;
  for (long long al = blockIdx.x; al < p.n_an; al += gridDim.x) {
    const long long a = p.a0 + al;
    if (p.status[a] != kStatusIndefinite) continue;
    double* refl = p.refl + al * (long long)kp * kp;
    if (row) {
      sd[r] = r < k ? p.d[al * kp + r] : 0.0;
      se[r] = r + 1 < k ? p.e[al * kp + r] : 0.0;
      sb[r] = r < k ? p.b[al * kp + r] : 0.0;
      for (int c = 0; c < KMAX; ++c) sZ[c * KMAX + r] = c == r ? 1.0 : 0.0;
    }
    // Z = Q = H_0 .. H_(k-3)
    for (int j = 0; j + 2 < k; ++j) {
      __syncthreads();
      if (row) sv[r] = refl[(long long)j * kp + r];
      __syncthreads();
      if (row) {
        double dot = 0.0;
        for (int c = j + 1; c < k; ++c) dot = fma(sZ[c * KMAX + r], sv[c], dot);
        dot *= p.tau[al * kp + j];
        for (int c = j + 1; c < k; ++c) sZ[c * KMAX + r] = fma(-dot, sv[c], sZ[c * KMAX + r]);
      }
    }
    __syncthreads();
    double tnorm = 0.0;
    for (int i = 0; i < k; ++i) tnorm = fmax(tnorm, fabs(sd[i]) + fabs(se[i]));
    int l = 0, iter = 0, status = 0;                 // thread 0's
    for (;;) {
      if (r == 0) {
        s_lo = s_hi = 0;
        s_end = 0;
        // the first l that is not an eigenvalue yet, and its block l .. m
        int m = l;
        for (; l < k; ++l, iter = 0) {
          for (m = l; m < k - 1; ++m) {
            const double em = fabs(se[m]);
            if (em <= eps * (fabs(sd[m]) + fabs(sd[m + 1])) || em <= eps * tnorm) break;
          }
          if (m > l) break;
        }
        if (l < k && ++iter > p.max_iter) status = l + 1;
        if (l >= k || status != 0) {
          s_end = 1;
        } else {
          double g = (sd[l + 1] - sd[l]) / (2.0 * se[l]);
          double t = hypot(g, 1.0);
          g = sd[m] - sd[l] + se[l] / (g + (g >= 0.0 ? fabs(t) : -fabs(t)));
          double s = 1.0, c = 1.0, pp = 0.0;
          int i = m - 1;
          for (; i >= l; --i) {
            const double f = s * se[i], bb = c * se[i];
            const double r2 = fma(f, f, g * g);
            const double rinv = rsqrt(r2);
            if (r2 == 0.0) {                         // underflow: the chase stops here
              se[i + 1] = 0.0;
              sd[i + 1] -= pp;
              break;
            }
            se[i + 1] = r2 * rinv;
            s = f * rinv;
            c = g * rinv;
            g = sd[i + 1] - pp;
            t = (sd[i] - g) * s + 2.0 * c * bb;
            pp = s * t;
            sd[i + 1] = g + pp;
            g = c * t - bb;
            srot[i] = make_double2(c, s);
          }
          s_lo = i + 1;
          s_hi = m;
          if (i < l) {
            sd[l] -= pp;
            se[l] = g;
          }
          se[m] = 0.0;
        }
      }
      __syncthreads();
      if (s_end) break;
      if (row) {
        const int lo = s_lo, hi = s_hi;
        double carry = sZ[hi * KMAX + r];
        for (int i = hi - 1; i >= lo; --i) {
          const double2 cs = srot[i];
          const double z = sZ[i * KMAX + r];
          sZ[(i + 1) * KMAX + r] = fma(cs.x, carry, cs.y * z);
          carry = fma(-cs.y, carry, cs.x * z);
        }
        sZ[lo * KMAX + r] = carry;
      }
      __syncthreads();
    }
    // functions of the eigenvalues (letkf_core.F90:107-113, the guard of the
    // reduced precisions): sv = sqrt((k-1)/lambda), sw = 1/lambda V^T b
    double lmin = 0.0;
    if (p.guard)
      for (int i = 0; i < k; ++i) lmin = fmin(lmin, sd[i]);
    if (row) {
      const double lam = r < k ? sd[r] - lmin + (double)(k - 1) / p.inflation : 1.0;
      double tb = 0.0;
      for (int i = 0; i < k; ++i) tb = fma(sZ[r * KMAX + i], sb[i], tb);
      sv[r] = r < k ? sqrt((double)(k - 1) / lam) : 0.0;
      sw[r] = r < k ? tb / lam : 0.0;
    }
    __syncthreads();
    double w = 0.0;
    if (r < k)
      for (int c = 0; c < k; ++c) w = fma(sZ[c * KMAX + r], sw[c], w);
    const bool bad = __syncthreads_or((r == 0 && status != 0) || !__builtin_isfinite(w));
    if (r == 0) p.status[a] = status != 0 ? status : bad ? kStatusNonFinite : 0;
    if (bad) {
      nan_transform(p, a);
    } else {
      if (p.w_out && r < k) p.w_out[a * (long long)k + r] = w;
      // trans(f, e) = T(f, e) + overline_w(f) (letkf_core.F90:221-225), f = r;
      // for the update in the layout k_vec leaves, zero past k
      float* const rf = reinterpret_cast<float*>(refl);
      if (row)
        for (int e = 0; e < KMAX; ++e) {
          double t = 0.0;
          if (r < k && e < k) {
            for (int c = 0; c < k; ++c) t = fma(sZ[c * KMAX + r] * sv[c], sZ[c * KMAX + e], t);
            t += w;
            if (p.trans_out) p.trans_out[a * (long long)k * k + (long long)e * k + r] = t;
          }
          if (p.xb || p.xb32) {
            const int o = tile_off<KMAX>(r >> 4, e >> 4, (r & 15) >> 2, 16 * (r & 3) + (e & 15));
            if (p.state_f32) rf[o] = (float)t;
            else refl[o] = t;
          }
        }
    }
    __syncthreads();
  }
}

// State precision of the update: FP64 (xb/xa) or FP32 (xb32/xa32) members on
// f64 or f32 MFMA 16x16x4 (the two share their operand layout).
template <class TS> struct StateT;
template <> struct StateT<double> {
  using acc = d4;
  static __device__ __forceinline__ const double* xb(const EigParams& p) { return p.xb; }
  static __device__ __forceinline__ double* xa(const EigParams& p) { return p.xa; }
  static __device__ __forceinline__ acc mma(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};
template <> struct StateT<float> {
  using acc = f4;
  static __device__ __forceinline__ const float* xb(const EigParams& p) { return p.xb32; }
  static __device__ __forceinline__ float* xa(const EigParams& p) { return p.xa32; }
  static __device__ __forceinline__ acc mma(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

// One state row o (k members at o*k) of a fused-epilogue column: the
// background mean ab, the analysis members xe (k of them, FP64) with mean aa;
// writes xa_out and the two spreads (module_da_parallel.F90:222-258).
__device__ __forceinline__ long long spread_index(const EigParams& p, int lo, int la, int v) {
  return ((long long)(lo - 1) * p.g.nlat + (la - 1)) * p.n + v;
}

// True when the update is the last word on an analysis with a nonzero status,
// so that its state rows keep the background; false when the list pass follows.
__device__ __forceinline__ bool keeps_background(const EigParams& p, int status) {
  return p.list || !p.ql_first || status == kStatusNotRedone || status == kStatusNonFinite;
}

// A failed analysis: xa = xb, axa = axb, or with the fused epilogue
// xa_out = xb + axb and spread_a = spread_b.
template <class TS, int EPI>
__device__ void copy_background_t(const EigParams& p, long long a) {
  const AnRows R = an_rows(p, a);
  const int k = p.k;
  const TS* __restrict__ xb = StateT<TS>::xb(p);
  for (int lo = R.si; lo <= R.ei; ++lo)
    for (int la = R.sj; la <= R.ej; ++la) {
      const long long off = ((long long)(lo - 1 + p.halo) * R.lat_ext + (la - 1 + p.halo)) * p.n;
      for (int vv = 0; vv < p.n_var; ++vv) {
        int l0, l1;
        const int start = p.var_start[vv] - 1;
        if (p.var_lev[vv] == 1) {
          if (p.vertical && R.ek != p.nz) continue;
          l0 = l1 = start;
        } else if (p.vertical) {
          l0 = start + R.sk - 1;
          l1 = start + R.ek - 1;
        } else {
          l0 = start;
          l1 = start + p.var_lev[vv] - 1;
        }
        for (int nk = l0 + (int)threadIdx.x; nk <= l1; nk += blockDim.x) {
          const long long o = off + nk;
          const double ab = p.axb[o];
          double sb = 0.0;
          for (int m = 0; m < k; ++m) {
            const double x = (double)xb[o * k + m];
            if (EPI) p.xa_out[o * k + m] = x + ab;
            else StateT<TS>::xa(p)[o * k + m] = xb[o * k + m];
            sb += x * x;
          }
          if (EPI) {
            const double sp = sqrt(sb / (double)(float)k);
            p.spread_b[spread_index(p, lo, la, nk)] = sp;
            p.spread_a[spread_index(p, lo, la, nk)] = sp;
          } else {
            p.axa[o] = ab;
          }
        }
      }
    }
}

// k_update: xa(:, v) = trans^T xb(:, v) + axb(v), then re-centred, for the
// variables v of one analysis (letkf_core.F90 ensemble update; the re-centring
// is the mean/perturbation split of letkf_run).  One block of four wavefronts
// per analysis: trans (k x k, from the B-operand tiles k_vec leaves in the
// reflector block) is staged once in LDS and wavefront w takes the
// (column, 16-variable group) items w, w + 4, ...  The MFMA reduction index
// is permuted -- at step s, lane quarter q carries member S q + s (S = KMAX/4)
// -- so that a lane's A operands for a group are one contiguous run of S
// members of one variable (16-byte loads); B takes the same permutation from
// LDS.  Registers stay near 100, so four blocks share a CU and the loads of
// one wavefront overlap the MFMAs of the others.
//
// TS is the storage precision of the perturbations (FP32: f32 MFMA with FP32
// accumulation; the means and the re-centring stay FP64).  EPI = 1 fuses the
// caller's epilogue into the output pass: full members gamma1 (axb + xb) +
// gamma2 (axa + xa) (the background where |lat| > polar_lat) and the spreads,
// written in place of xa/axa.
template <int KMAX, class TS, int EPI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
void k_update(EigParams p) {
  using ST = StateT<TS>;
  using acc_t = typename ST::acc;
  constexpr int TT = KMAX / 16;
  constexpr int S = KMAX / 4;
  constexpr int VEC = 16 / sizeof(TS);       // members per 16-byte load
  // S * LDT = 16 (mod 32) for FP64: the four lane quarters of a B read fall
  // on disjoint banks in each half-wavefront
  constexpr int LDT = KMAX == 64 ? KMAX + 1 : KMAX + 2;
  static_assert(KMAX == 32 || KMAX == 64, "k_update covers k <= 64");
  __shared__ TS sT[KMAX * LDT];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  long long a, ai, ar;
  if (!eig_slot(p, blockIdx.x, a, ai, ar)) return;
  if (p.status[a] != 0) {                // failed, or redone by the list pass
    if (keeps_background(p, p.status[a])) copy_background_t<TS, EPI>(p, a);
    return;
  }
  const int k = p.k;
  const int i16 = lane & 15, q = lane >> 4;
  // the row of a 16x16 MFMA result that register r of lane quarter q holds:
  // q + 4 r for f64 16x16x4, 4 q + r for f32 16x16x4
  constexpr bool F32 = sizeof(TS) == 4;
  auto out_row = [q](int r) { return F32 ? 4 * q + r : q + 4 * r; };
  const TS* __restrict__ xb = ST::xb(p);
  // trans tiles from k_vec: FP32 for the FP32 state, else FP64
  const double* __restrict__ tb = p.refl + ai * (long long)p.kp * p.kp;
  const TS* __restrict__ tbs = reinterpret_cast<const TS*>(tb);
  for (int idx = tid; idx < TT * TT * 4 * 64; idx += 256) {
    const int l = idx & 63, c = idx >> 6, r = c & 3, IJ = c >> 2;
    const int row = 16 * (IJ / TT) + 4 * r + (l >> 4), col = 16 * (IJ % TT) + (l & 15);
    sT[row * LDT + col] = (row < k && col < k) ? tbs[idx] : (TS)0;
  }

  const AnRows R = an_rows(p, a);
  const int sj = R.sj, ej = R.ej, si = R.si, ei = R.ei, sk = R.sk, ek = R.ek;
  const long long lat_ext = R.lat_ext;
  // the analysis's state rows: all n of the column, or (vertical loop) the
  // levels sk..ek of each 3-D variable and the 2-D variables on the top chunk;
  // sidx maps the v-th of them to its offset in the column
  auto run_len = [&](int vv) {
    return p.var_lev[vv] == 1 ? (ek == p.nz ? 1 : 0) : ek - sk + 1;
  };
  int nvec = p.n;
  if (p.vertical) {
    nvec = 0;
    for (int vv = 0; vv < p.n_var; ++vv) nvec += run_len(vv);
  }
  auto sidx = [&](int v) {
    if (v >= nvec) return -1;
    if (!p.vertical) return v;
    int rem = v;
    for (int vv = 0; vv < p.n_var; ++vv) {
      const int len = run_len(vv);
      if (rem < len) return p.var_start[vv] - 1 + (p.var_lev[vv] == 1 ? 0 : sk - 1) + rem;
      rem -= len;
    }
    return -1;
  };
  const int ngrp = (nvec + 15) / 16;
  const int ncl = ej - sj + 1;
  const int n_items = (ei - si + 1) * ncl * ngrp;
  const bool vec_ld = (k == KMAX) && ((reinterpret_cast<uintptr_t>(xb) & 15) == 0);
  auto item_off = [&](int it) {
    const int cl = it / ngrp;
    const int lo = si + cl / ncl, la = sj + cl % ncl;
    return ((long long)(lo - 1 + p.halo) * lat_ext + (la - 1 + p.halo)) * p.n;
  };
  // A operands of item it: variable 16 g + i16, members S q .. S q + S - 1
  auto load_a = [&](int it, TS (&af)[S]) {
    const long long off = item_off(it);
    const int s_a = sidx(16 * (it % ngrp) + i16);
    if (s_a >= 0 && vec_ld) {
      const uint4* xr = reinterpret_cast<const uint4*>(xb + (off + s_a) * k + S * q);
#pragma unroll
      for (int u = 0; u < S / VEC; ++u) {
        const uint4 t4 = xr[u];
        const TS* tv = reinterpret_cast<const TS*>(&t4);
#pragma unroll
        for (int x = 0; x < VEC; ++x) af[VEC * u + x] = tv[x];
      }
    } else {
      const TS* xr = xb + (off + (s_a >= 0 ? s_a : 0)) * k;
#pragma unroll
      for (int u = 0; u < S; ++u) {
        const int m = S * q + u;
        af[u] = (s_a >= 0 && m < k) ? xr[m] : (TS)0;
      }
    }
  };
  // the first item's A operands are read before the staging barrier, each
  // later item's as soon as the previous item's MFMAs have consumed theirs
  TS af[S];
  if (w < n_items) load_a(w, af);
  __syncthreads();
  for (int it = w; it < n_items; it += 4) {
    const long long off = item_off(it);
    const int v0 = 16 * (it % ngrp);
    double ab4[4];
    int st4[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      st4[r] = sidx(v0 + out_row(r));
      ab4[r] = (st4[r] >= 0) ? p.axb[off + st4[r]] : 0.0;
    }
    acc_t out[TT];
#pragma unroll
    for (int J = 0; J < TT; ++J) out[J] = acc_t{0, 0, 0, 0};
    // B of step s + 1 is read while the MFMAs of step s run; the scheduling
    // barriers keep the compiler from hoisting every B read (and its
    // registers) to the top of the loop
    const TS* bq = sT + S * q * LDT + i16;
    TS bn[TT];
#pragma unroll
    for (int J = 0; J < TT; ++J) bn[J] = bq[16 * J];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      TS b[TT];
#pragma unroll
      for (int J = 0; J < TT; ++J) b[J] = bn[J];
      if (s + 1 < S) {
#pragma unroll
        for (int J = 0; J < TT; ++J) bn[J] = bq[(s + 1) * LDT + 16 * J];
      }
#pragma unroll
      for (int J = 0; J < TT; ++J) out[J] = ST::mma(af[s], b[J], out[J]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (it + 4 < n_items) load_a(it + 4, af);
    // lane (i16, q) holds xa of variable v0 + out_row(r), member 16 J + i16
    int lo_c = 0, la_c = 0;
    bool polar = false;
    if (EPI) {
      const int cl = it / ngrp;
      lo_c = si + cl / ncl;
      la_c = sj + cl % ncl;
      polar = fabs((double)p.g.glat[la_c - 1]) > p.polar_lat;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      double sum = 0.0;
      double xe[TT];
#pragma unroll
      for (int J = 0; J < TT; ++J) {
        const int e = 16 * J + i16;
        xe[J] = (e < k) ? (double)out[J][r] + ab4[r] : 0.0;
        sum += xe[J];
      }
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) sum += __shfl_xor(sum, o, 64);
      const double mean = sum / k;
      if (!EPI) {
        if (st4[r] >= 0) {
          const long long o = off + st4[r];
          TS* __restrict__ xa = ST::xa(p);
#pragma unroll
          for (int J = 0; J < TT; ++J) {
            const int e = 16 * J + i16;
            if (e < k) xa[o * k + e] = (TS)(xe[J] - mean);
          }
          if (i16 == 0) p.axa[o] = mean;
        }
      } else {
        // the caller's epilogue (module_da_parallel.F90:219-261)
        const long long o = off + (st4[r] >= 0 ? st4[r] : 0);
        double sb = 0.0, sa = 0.0;
        double xo[TT];
#pragma unroll
        for (int J = 0; J < TT; ++J) {
          const int e = 16 * J + i16;
          const bool in = e < k && st4[r] >= 0;
          const double xbe = in ? (double)xb[o * k + e] : 0.0;
          const double xae = xe[J] - mean;
          double v;
          if (polar) {
            v = xbe + ab4[r];
            sa += xbe * xbe;
          } else {
            v = p.gamma1 * (ab4[r] + xbe) + p.gamma2 * (mean + xae);
            if (e < k) sa += (v - mean) * (v - mean);
          }
          xo[J] = v;
          sb += xbe * xbe;
        }
#pragma unroll
        for (int o2 = 1; o2 < 16; o2 <<= 1) {
          sb += __shfl_xor(sb, o2, 64);
          sa += __shfl_xor(sa, o2, 64);
        }
        if (st4[r] >= 0) {
#pragma unroll
          for (int J = 0; J < TT; ++J) {
            const int e = 16 * J + i16;
            if (e < k) p.xa_out[o * k + e] = xo[J];
          }
          if (i16 == 0) {
            const long long so = spread_index(p, lo_c, la_c, st4[r]);
            p.spread_b[so] = sqrt(sb / (double)(float)k);
            p.spread_a[so] = sqrt(sa / (double)(float)k);
          }
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// k_rot128 + k_update128: k = 65..128 with the rows of Z in registers.
// 256 threads per matrix: thread t keeps half h = t / 128 (columns
// 64h .. 64h+63) of row r = t % 128.  A chase that crosses the middle (lo < 64
// <= hi) runs on the upper half first; its carry goes to the lower half
// through LDS, and the lower half's step at position 63 returns the new
// column-64 entry the same way.  The lower part runs one chase late, beside
// the next chase's upper part, so both halves work through runs of crossing
// chases.
// ---------------------------------------------------------------------------

// Householder tridiagonalisation for k = 65..128 with half rows of A in
// registers (thread t: row t % 128, the columns of parity h = t / 128, one
// half per wavefront): the halves interleave, so both keep the same share of
// the shrinking trailing matrix, and blocks of columns <= j (where v and w
// are zero) are skipped.  v and w enter the FMAs as row broadcasts, as in
// k_tridiag (64,800 matrices of k = 128: 34.3 -> 23.9 ms).  A column already
// in tridiagonal form runs the same
// step with v = 0 and tau = 0 (an exact identity update), so the loop has one
// path and A stays in the same registers.  Three wavefronts per SIMD.  Same
// outputs as k_tridiag.  Three barriers per step:
//  - the pivot column j is in LDS (double-buffered by the parity of j) with
//    rows <= j zeroed; each wavefront writes v_{j+1} = x0 - alpha over its
//    entry j+1 before reading it (every wavefront writes the same value), so
//    v is read from the column directly; x0 and the sum of squares of the
//    column below it come from the previous step;
//  - the partial products of the two halves and the per-wavefront partials of
//    v.p share one barrier;
//  - w, then the update, the extraction of column j+1 (stores under
//    wavefront-uniform branches, read back for its squares) share the step's
//    last barrier.
// Partial sums are combined in a fixed order, so every thread holds the same
// values.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_tridiag128(EigParams p) {
  constexpr int KMAX = 128;
  __shared__ double sx[2][KMAX];          // pivot column, rows <= j zeroed
  __shared__ double sx0[2];               // A(j+1, j) of the pivot column
  __shared__ double sw[KMAX], spr[2][KMAX];
  __shared__ double se_s[KMAX + 1], st_s[KMAX + 1], sd[KMAX];
  __shared__ double rsq[2][4], rvp[4];    // per-wavefront partials
  const int tid = threadIdx.x;
  const int r = tid & 127, h = uniform(tid >> 7);   // the half is one per wavefront
  const int wv = tid >> 6, lane = tid & 63;
  const long long a = p.a0 + blockIdx.x;
  if (a >= p.a0 + p.n_an) return;
  const long long al = a - p.a0;
  const int k = p.k, kp = p.kp;
  const double* __restrict__ Ag = p.A + al * (long long)kp * kp;
  double* __restrict__ refl = p.refl + al * (long long)kp * kp;
  const bool in_r = r < k;
  double arow[64];
  // eight columns in flight at a time: the loads need one address each
#pragma unroll
  for (int B = 0; B < 8; ++B) {
#pragma unroll
    for (int c = 8 * B; c < 8 * B + 8; ++c) {
      // unconditional in-bounds load (r < kp), then a select: no branch
      // per column
      const int col = 2 * c + h;
      const double av = Ag[(long long)col * kp + r];
      arow[c] = (in_r && col < k) ? av : 0.0;
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // column 0 (held by half 0) and the squares of its rows > 1
  if (h == 0) {
    sx[0][r] = (r > 0) ? arow[0] : 0.0;
    if (r == 1) sx0[0] = arow[0];
  }
  {
    const double sq = wave_sum_full((h == 0 && r > 1) ? arow[0] * arow[0] : 0.0);
    if (lane == 0) rsq[0][wv] = sq;
  }
  __syncthreads();
  // column j+1 -> sx[nxt] (rows <= j+1 zeroed) and sx0[nxt]; partial squares
  // of its rows > j+2 -> rsq[nxt]
  auto pass_column = [&](int j, int nxt) {
    const int hj1 = (j + 1) & 1;
    if (h == hj1) {
      const double xc = pick_column(arow, (j + 1) >> 1);
      sx[nxt][r] = (r > j + 1) ? xc : 0.0;
      if (r == j + 2) sx0[nxt] = xc;
    }
    const double xn = (h == hj1 && r > j + 2) ? sx[nxt][r] : 0.0;
    const double sq = wave_sum_full(xn * xn);
    if (lane == 0) rsq[nxt][wv] = sq;
  };
  for (int j = 0; j + 2 < k; ++j) {
    const int cur = j & 1, nxt = cur ^ 1;
    double* col = sx[cur];
    const bool act = in_r && r > j;
    const double x0 = uniform(sx0[cur]);
    const double rest = (rsq[cur][0] + rsq[cur][1]) + (rsq[cur][2] + rsq[cur][3]);
    // a column already in tridiagonal form (rest = 0) takes the same path
    // with v = 0 and tau = 0: the update is then exactly the identity
    const bool none = rest == 0.0;
    const double nrm = sqrt(rest + x0 * x0);
    const double alpha = (x0 >= 0.0) ? -nrm : nrm;
    const double v0 = none ? 0.0 : x0 - alpha;
    const double tau = none ? 0.0 : 2.0 / (rest + v0 * v0);
    if (lane == 0) col[j + 1] = v0;
    const double vr = act ? col[r] : 0.0;
    // partial p over this half (v_c = 0 for c <= j; row broadcasts as in
    // k_tridiag, lane i of a row holding entry 2 (16 t + i) + h)
    double vt[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) vt[t] = col[2 * (16 * t + (lane & 15)) + h];
    double p4[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (32 * t + 14 + h > j) bcast_dot8<0>(p4, vt[t], arow + 16 * t);
      if (32 * t + 30 + h > j) bcast_dot8<1>(p4, vt[t], arow + 16 * t + 8);
    }
    const double ph = (p4[0] + p4[1]) + (p4[2] + p4[3]);
    if (in_r) spr[h][r] = ph;
    {
      const double vp = wave_sum_full(vr * ph);
      if (lane == 0) rvp[wv] = vp;
    }
    __syncthreads();
    const double pr = act ? (spr[0][r] + spr[1][r]) * tau : 0.0;
    const double K = 0.5 * tau * tau * ((rvp[0] + rvp[1]) + (rvp[2] + rvp[3]));
    const double wr = act ? pr - K * vr : 0.0;
    if (h == 0) sw[r] = wr;
    __syncthreads();
    // A -= v w^T + w v^T over this half (vr = wr = 0 in rows <= j)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const double wt = sw[2 * (16 * t + (lane & 15)) + h];
      if (32 * t + 14 + h > j) {
        bcast_axpy8<0>(arow + 16 * t, wt, -vr);
        bcast_axpy8<0>(arow + 16 * t, vt[t], -wr);
      }
      if (32 * t + 30 + h > j) {
        bcast_axpy8<1>(arow + 16 * t + 8, wt, -vr);
        bcast_axpy8<1>(arow + 16 * t + 8, vt[t], -wr);
      }
    }
    pass_column(j, nxt);
    if (h == 0) refl[(long long)j * kp + r] = vr;
    if (tid == 0) { se_s[j] = none ? x0 : alpha; st_s[j] = tau; }
    __syncthreads();
  }
  // diagonal (thread of the half holding column r) and e[k-2] = A[k-1][k-2]
#pragma unroll
  for (int c = 0; c < 64; ++c)
    if (2 * c + h == r) sd[r] = arow[c];
  if (r == k - 1) {
#pragma unroll
    for (int c = 0; c < 64; ++c)
      if (2 * c + h == k - 2) se_s[KMAX] = arow[c];
  }
  __syncthreads();
  if (h != 0) return;
  double* __restrict__ dg = p.d + al * kp;
  double* __restrict__ eg = p.e + al * kp;
  double* __restrict__ tg = p.tau + al * kp;
  dg[r] = in_r ? sd[r] : 0.0;
  double ev = 0.0, tv = 0.0;
  if (r + 2 < k) { ev = se_s[r]; tv = st_s[r]; }
  else if (r == k - 2) ev = se_s[KMAX];
  eg[r] = ev;
  tg[r] = tv;
}

// Applies the positions il in [lo_l, hi_l) of a chase to a half row
// z[0..63] (rotation of local position il at ring entry base_l - il, identity
// outside); z[64] is `ztop` (in/out).  The carry enters at the top block as
// z[top+1] and leaves as the return value; with `final_write`, z[lo_l] takes
// it (the chase ends in this half).
template <int RING>
__device__ __forceinline__ double chase_half(double (&z)[64], double& ztop, int lo_l, int hi_l,
                                             const double2* sring, int base_l, bool final_write,
                                             bool top_done) {
  const int bhi = (hi_l - 1) >> 3, blo = lo_l >> 3;
  double carry = 0.0;
#pragma unroll
  for (int B = 7; B >= 0; --B) {
    if (B > bhi || B < blo) continue;
    if (B == bhi) carry = (B == 7) ? ztop : z[8 * B + 8];
    double2 cs[8];
    ring_block<RING>(sring, base_l, B, cs);
    if (B == 7 && top_done) cs[7] = make_double2(1.0, 0.0);
#pragma unroll
    for (int t = 7; t >= 0; --t) {
      const int i = 8 * B + t;
      const double zi = z[i];
      const double up = fma(cs[t].x, carry, cs[t].y * zi);
      if (i == 63) ztop = up;
      else z[i + 1] = up;
      carry = fma(-cs[t].y, carry, cs[t].x * zi);
    }
    if (B == blo && final_write) z[8 * B] = carry;
  }
  return carry;
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_rot128(EigParams p) {
  constexpr int KMAX = 128, LDV = KMAX + 1, NT = 256;
  constexpr int RING = 1024, REFILL = 512;
  __shared__ __align__(16) double sbuf[16 * LDV > 2 * (RING + 8) ? 16 * LDV : 2 * (RING + 8)];
  __shared__ double sf[KMAX], sg[KMAX], sb[KMAX], st[KMAX], sw[KMAX], stau[KMAX];
  __shared__ double sx[2][2][KMAX];      // partial dots [parity][half][row]
  __shared__ double sc[KMAX], sz64[KMAX];
  __shared__ double red[8];
  const int tid = threadIdx.x;
  const int r = tid & 127, h = uniform(tid >> 7);   // the half is one per wavefront
  const int lane = tid & 63, wv = uniform(tid >> 6);
  long long a, ai, ar;
  if (!eig_slot(p, blockIdx.x, a, ai, ar)) return;
  if (p.status[a] != 0) {                // redone by the list pass, or failed
    if (p.list || p.status[a] == kStatusNotRedone) nan_transform(p, a);
    return;
  }
  const int k = p.k, kp = p.kp;
  const bool in_r = r < k;
  double* __restrict__ refl = p.refl + ai * (long long)kp * kp;
  const double* __restrict__ tg = p.tau + ai * kp;
  const int nref = k > 2 ? k - 2 : 0;

  // ---- A. Z <- Z H_j: half dots exchanged through LDS ----
  if (tid < nref) stau[tid] = tg[tid];
  double z[64];
#pragma unroll
  for (int c = 0; c < 64; ++c) z[c] = (64 * h + c == r) ? 1.0 : 0.0;
  for (int j0 = 0; j0 < nref; j0 += 16) {
    __syncthreads();
    for (int e = tid; e < 16 * KMAX; e += NT) {
      const int t = e / KMAX, c = e % KMAX;
      sbuf[t * LDV + c] = (j0 + t < nref) ? refl[(long long)(j0 + t) * kp + c] : 0.0;
    }
    __syncthreads();
    const int j1 = min(j0 + 16, nref);
    for (int j = j0; j < j1; ++j) {
      const double tau = uniform(stau[j]);
      const double* q = sbuf + (j - j0) * LDV + 64 * h;
      // the reflector is zero over columns <= j: blocks of 8 there are skipped
      double d0 = 0.0, d1 = 0.0;
#pragma unroll
      for (int B = 0; B < 8; ++B) {
        if (64 * h + 8 * B + 7 <= j) continue;
#pragma unroll
        for (int c = 8 * B; c < 8 * B + 8; c += 2) {
          d0 = fma(z[c], q[c], d0);
          d1 = fma(z[c + 1], q[c + 1], d1);
        }
      }
      sx[j & 1][h][r] = d0 + d1;
      __syncthreads();
      const double dot = (sx[j & 1][0][r] + sx[j & 1][1][r]) * tau;
#pragma unroll
      for (int B = 0; B < 8; ++B) {
        if (64 * h + 8 * B + 7 <= j) continue;
#pragma unroll
        for (int c = 8 * B; c < 8 * B + 8; ++c) z[c] = fma(-dot, q[c], z[c]);
      }
    }
  }
  __syncthreads();

  // ---- B. logged QL rotations ----
  {
    double2* sring = reinterpret_cast<double2*>(sbuf);
    const double2* __restrict__ rot = p.rot + ar * (long long)p.rot_cap;
    const int4* __restrict__ hdr = p.hdr + ar * (long long)p.hdr_cap;
    const int nch = uniform(min(p.nchase[ar], p.hdr_cap));
    int nrot = 0;
    if (nch > 0) {
      const int4 hl = hdr[nch - 1];
      nrot = uniform(hl.z + hl.w);
    }
    int committed = 0;
    double ztop = 0.0;
    // A crossing chase's lower part runs one chase late, beside the next
    // chase's upper part: its step at position 63 (which needs the upper
    // part's carry and gives column 64 back) runs alone between two barriers,
    // the rest of it together with the next chase's piece in the other half.
    bool pend = false;
    int plo = 0, pbase = 0;
    for (int ch = 0; ch <= nch; ++ch) {
      const bool have = ch < nch;       // ch == nch: the last pending lower part
      int lo = 0, hi = 0, base = 0;
      bool cross = false;
      if (have) {
        const int4 hh = hdr[ch];
        lo = uniform(hh.x);
        hi = uniform(hh.y);
        const int off = uniform(hh.z), len = uniform(hh.w);
        // refills are the only block-wide barriers besides the crossing
        // chases': the slots a refill overwrites may still be read by a chase
        // that started below the previous refill's entries, hence the leading
        // barrier (the pending chase is the previous one: a refill, needed
        // only when this chase ends past the ring's entries, never reaches it)
        if (off + len > committed) {
          __syncthreads();
          for (int e = tid; e < REFILL; e += NT) {
            const int g = committed + e;
            const double2 v = (g < nrot) ? rot[g] : make_double2(1.0, 0.0);
            const int slot = g & (RING - 1);
            sring[slot] = v;
            if (slot < 8) sring[RING + slot] = v;
          }
          committed += REFILL;
          __syncthreads();
        }
        base = off + ((hi + 7) & ~7) - 1;
        cross = lo < 64 && hi >= 64;
      }
      if (pend) {
        // position 63 of the pending chase: carry from the upper part (sc),
        // new column 64 to the upper half (sz64); z[63] keeps the carry on
        if (h == 0) {
          const double cin = sc[r];
          const double2 cs = sring[(pbase - 63) & (RING - 1)];
          const double z63 = z[63];
          sz64[r] = fma(cs.x, cin, cs.y * z63);
          z[63] = fma(-cs.y, cin, cs.x * z63);
        }
        __syncthreads();
        if (h == 1) z[0] = sz64[r];
      }
      // piece 0: the rest of the pending lower part (its position 63 is done);
      // piece 1: this chase's piece in this half (a crossing chase: the upper
      // part, whose carry goes to sc)
      for (int t = 0; t < 2; ++t) {
        bool act = false, fw = true;
        int lo_l = 0, hi_l = 0, bl = 0;
        if (t == 0) {
          act = pend && h == 0;
          lo_l = plo;
          hi_l = 64;
          bl = pbase;
        } else if (cross) {
          act = h == 1 && hi > 64;
          hi_l = hi - 64;
          bl = base - 64;
          fw = false;
        } else if (have) {
          act = (hi <= 63 && h == 0) || (lo >= 64 && h == 1);
          lo_l = lo - 64 * h;
          hi_l = hi - 64 * h;
          bl = base - 64 * h;
        }
        if (act) {
          ztop = 0.0;
          const double cy = chase_half<RING>(z, ztop, lo_l, hi_l, sring, bl, fw, t == 0);
          if (t == 1 && cross) sc[r] = cy;
        }
      }
      // hi == 64: no position in the upper half, the carry is column 64
      if (cross && h == 1 && hi == 64) sc[r] = z[0];
      pend = cross;
      if (pend) {
        plo = lo;
        pbase = base;
        __syncthreads();
      }
    }
  }
  __syncthreads();

  // ---- C. eigenvalue functions, T = V diag(f) V^T on MFMA, overline_w ----
  if (tid < KMAX) {
    double lam = tid < k ? p.lam[ar * kp + tid] : 0.0;
    sf[tid] = lam;
  }
  __syncthreads();
  if (p.guard) {
    double mn = 1e300;
    for (int i = 0; i < k; ++i) mn = fmin(mn, sf[i]);
    __syncthreads();
    if (tid < k && mn < 0.0) sf[tid] -= mn;
    __syncthreads();
  }
  if (tid < KMAX) {
    const bool ok = tid < k;
    const double lam = ok ? sf[tid] * 1.0 + (double)(k - 1) / p.inflation : 1.0;
    sg[tid] = ok ? 1.0 / lam : 0.0;
    sb[tid] = ok ? p.b[ai * kp + tid] : 0.0;
    sf[tid] = ok ? sqrt((double)(k - 1) / lam) : 0.0;
  }
  // st = diag(1/lambda) V^T b: column sums over rows, V staged 16 columns at
  // a time ([column][row]); T tiles: wave w computes J in {2w, 2w+1}, in two
  // passes over I (4 tile rows each)
  const int i16 = lane & 15, q = lane >> 4;
  double* sVc = sbuf;
  double wpart = 0.0;
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    d4 acc[4][2];
#pragma unroll
    for (int I = 0; I < 4; ++I)
#pragma unroll
      for (int J = 0; J < 2; ++J) acc[I][J] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int c = 0; c < 8; ++c) {                // chunk c: columns 16c .. 16c+15
      __syncthreads();
      if (h == (c >> 2)) {
#pragma unroll
        for (int t = 0; t < 16; ++t) sVc[t * LDV + r] = z[16 * (c & 3) + t];
      }
      __syncthreads();
      if (pass == 0 && tid < 16) {
        double tb = 0.0;
        for (int rr = 0; rr < KMAX; ++rr) tb = fma(sVc[tid * LDV + rr], sb[rr], tb);
        st[16 * c + tid] = tb * sg[16 * c + tid];
      }
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        const int t = 4 * s4 + q;
        const double fc = sf[16 * c + t];
        double fa[4], fb[2];
#pragma unroll
        for (int I = 0; I < 4; ++I) fa[I] = sVc[t * LDV + 16 * (4 * pass + I) + i16];
#pragma unroll
        for (int J = 0; J < 2; ++J) fb[J] = fc * sVc[t * LDV + 16 * (2 * wv + J) + i16];
#pragma unroll
        for (int I = 0; I < 4; ++I)
#pragma unroll
          for (int J = 0; J < 2; ++J)
            acc[I][J] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[I], fb[J], acc[I][J], 0, 0, 0);
      }
    }
    if (pass == 0) {
      __syncthreads();
      // overline_w(r) = sum_c V[r][c] st_c, halves summed through LDS
#pragma unroll
      for (int c = 0; c < 64; ++c) wpart = fma(z[c], st[64 * h + c], wpart);
      sx[0][h][r] = wpart;
      __syncthreads();
      if (tid < KMAX) sw[tid] = tid < k ? sx[0][0][tid] + sx[0][1][tid] : 0.0;
      __syncthreads();
    }
    // trans(f, e) = T(f, e) + overline_w(f)
#pragma unroll
    for (int I = 0; I < 4; ++I)
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const double wf = sw[16 * (4 * pass + I) + q + 4 * rr];
#pragma unroll
        for (int J = 0; J < 2; ++J) acc[I][J][rr] += wf;
      }
    if (p.trans_out) {
      double* tr = p.trans_out + a * (long long)k * k;
#pragma unroll
      for (int I = 0; I < 4; ++I)
#pragma unroll
        for (int J = 0; J < 2; ++J)
#pragma unroll
          for (int rr = 0; rr < 4; ++rr) {
            const int f = 16 * (4 * pass + I) + q + 4 * rr, e = 16 * (2 * wv + J) + i16;
            if (f < k && e < k) tr[(long long)e * k + f] = acc[I][J][rr];
          }
    }
    if (p.xb || p.xb32) {
      __syncthreads();                             // every read of the reflector block is done
#pragma unroll
      for (int I = 0; I < 4; ++I)
#pragma unroll
        for (int J = 0; J < 2; ++J)
#pragma unroll
          for (int rr = 0; rr < 4; ++rr) {
            // in the precision of the state, as k_vec leaves it
            const int o = tile_off<KMAX>(4 * pass + I, 2 * wv + J, rr, lane);
            if (p.state_f32) reinterpret_cast<float*>(refl)[o] = (float)acc[I][J][rr];
            else refl[o] = acc[I][J][rr];
          }
    }
  }
  // every thread scans overline_w in LDS, so the decision is uniform
  bool bad = false;
  for (int f = 0; f < k; ++f) bad = bad || !__builtin_isfinite(sw[f]);
  if (bad) {
    __syncthreads();                               // the trans writes above are done
    if (threadIdx.x == 0) p.status[a] = kStatusNonFinite;
    nan_transform(p, a);
    return;
  }
  if (p.w_out && h == 0 && in_r) p.w_out[a * (long long)k + r] = sw[r];
}

// Exchanges the upper 32 lanes of x with the lower 32 of y, and the odd rows of
// 16 lanes of x with the even rows of y: together, over four registers, the
// transposition between registers and lane quarters.
__device__ __forceinline__ void swap_halves(float& x, float& y) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  x = __uint_as_float(r[0]);
  y = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap_rows(float& x, float& y) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  x = __uint_as_float(r[0]);
  y = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap_halves(double&, double&) {}
__device__ __forceinline__ void swap_rows(double&, double&) {}

// Xa = Xb trans for k = 65..128: wave w produces members 32w .. 32w+31, its
// trans columns (128 x 32) in registers; all four take the same groups of 16
// state vectors.  TS and EPI as k_update.
//
// The bound is the state and trans in HBM (10.7 GB for the FP32 state of
// 64,800 columns of 97 vectors at k = 128) and the f32 MFMAs beside it.  A
// operands come straight from the state in 16-byte pieces, one load instruction
// covering 64 contiguous bytes of each of 16 vectors, the next group's as soon
// as the MFMAs have consumed this one's.  FP64 permutes the reduction index to
// the pieces (step s, lane quarter q carry member 8 (s / 2) + 2 q + s mod 2);
// FP32, whose sums would round differently, transposes four pieces between the
// lane quarters instead (v_permlane swaps) and keeps members 4 s + q.  LDS only
// carries the wavefronts' shares of the means, one barrier a group.  (Staged through LDS
// between two barriers a group, with no load in flight across them, and sums
// by shuffles, 10.7 ms there; now 6.1, cycle 63.3 ms; FP32 in the order of
// the pieces 4.3 and 61.0 ms.)  FP64 spills 32 registers, 72 with the epilogue:
// its trans fills half of them.
template <class TS, int EPI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void k_update128(EigParams p) {
  using ST = StateT<TS>;
  using acc_t = typename ST::acc;
  constexpr int KMAX = 128, S = KMAX / 4;
  constexpr int VEC = 16 / sizeof(TS);       // members per 16-byte load
  // shares of the sums of a group's 16 vectors: of the members (a buffer for
  // each of two groups in turn), and with EPI of the two spreads
  __shared__ double spart[2][4][16];
  __shared__ double sspr[EPI ? 2 : 1][4][16];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wv = tid >> 6;
  long long a, ai, ar;
  if (!eig_slot(p, blockIdx.x, a, ai, ar)) return;
  if (p.status[a] != 0) {                // failed, or redone by the list pass
    if (keeps_background(p, p.status[a])) copy_background_t<TS, EPI>(p, a);
    return;
  }
  const int k = p.k, kp = p.kp;
  const int i16 = lane & 15, q = lane >> 4;
  // the row of a 16x16 MFMA result that register rr of lane quarter q holds:
  // q + 4 rr for f64 16x16x4, 4 q + rr for f32 16x16x4
  constexpr bool F32 = sizeof(TS) == 4;
  auto out_row = [q](int rr) { return F32 ? 4 * q + rr : q + 4 * rr; };
  auto piece = [q](int s) { return 4 * VEC * (s / VEC) + VEC * q + s % VEC; };
  auto member = [q, piece](int s) { return F32 ? 4 * s + q : piece(s); };
  const TS* __restrict__ xb = ST::xb(p);
  // trans tiles from the transform, in the state's precision
  const TS* __restrict__ tb =
      reinterpret_cast<const TS*>(p.refl + ai * (long long)kp * kp);
  // tile_off of member(s)'s row, split in the lane's part and a constant
  const TS* __restrict__ tl =
      tb + tile_off<KMAX>(0, 2 * wv, F32 ? 0 : q >> 1, F32 ? lane : 32 * (q & 1) + i16);
  TS bop[S][2];
#pragma unroll
  for (int s = 0; s < S; ++s) {
#pragma unroll
    for (int J = 0; J < 2; ++J)
      bop[s][J] = tl[tile_off<KMAX>(s >> 2, J, F32 ? s & 3 : s & 2, F32 ? 0 : 16 * (s & 1))];
    if (s % 8 == 7) __builtin_amdgcn_sched_barrier(0);
  }

  const AnRows R = an_rows(p, a);
  const int sj = R.sj, ej = R.ej, si = R.si, ei = R.ei, sk = R.sk, ek = R.ek;
  const long long lat_ext = R.lat_ext;
  // the analysis's state rows, as in k_update
  auto run_len = [&](int vv) {
    return p.var_lev[vv] == 1 ? (ek == p.nz ? 1 : 0) : ek - sk + 1;
  };
  int nvec = p.n;
  if (p.vertical) {
    nvec = 0;
    for (int vv = 0; vv < p.n_var; ++vv) nvec += run_len(vv);
  }
  auto sidx = [&](int v) {
    if (v >= nvec) return -1;
    if (!p.vertical) return v;
    int rem = v;
    for (int vv = 0; vv < p.n_var; ++vv) {
      const int len = run_len(vv);
      if (rem < len) return p.var_start[vv] - 1 + (p.var_lev[vv] == 1 ? 0 : sk - 1) + rem;
      rem -= len;
    }
    return -1;
  };
  const int ngrp = (nvec + 15) / 16;
  const int ncl = ej - sj + 1;
  const int n_items = (ei - si + 1) * ncl * ngrp;
  // every vector starts at a 16-byte boundary and ends at a whole piece
  const bool vec_ld = k % VEC == 0 && (reinterpret_cast<uintptr_t>(xb) & 15) == 0;
  auto item_off = [&](int it) {
    const int cl = it / ngrp;
    const int lo = si + cl / ncl, la = sj + cl % ncl;
    return ((long long)(lo - 1 + p.halo) * lat_ext + (la - 1 + p.halo)) * p.n;
  };
  // steps s0 .. s0 + SA - 1 of item it; FP64's trans fills half of the
  // registers, so its operands come in two halves, each before its MFMAs
  constexpr int SA = F32 ? S : S / 2;
  TS af[SA];
  auto load_a = [&](int it, auto first) {
    constexpr int s0 = decltype(first)::value;
    const int s_a = sidx(16 * (it % ngrp) + i16);
    const TS* xr = xb + (item_off(it) + (s_a >= 0 ? s_a : 0)) * k;
    if (vec_ld) {
#pragma unroll
      for (int s = 0; s < SA; s += VEC) {
        // an in-row load and a select: no branch
        const int m = piece(s0 + s);
        const uint4 t4 = *reinterpret_cast<const uint4*>(xr + (m < k ? m : 0));
        const TS* tv = reinterpret_cast<const TS*>(&t4);
#pragma unroll
        for (int x = 0; x < VEC; ++x) af[s + x] = (s_a >= 0 && m < k) ? tv[x] : (TS)0;
        // register x of quarter q: member 16 (s / 4) + 4 q + x -> 4 x + q
        if constexpr (F32) {
          swap_halves(af[s], af[s + 2]);
          swap_halves(af[s + 1], af[s + 3]);
          swap_rows(af[s], af[s + 1]);
          swap_rows(af[s + 2], af[s + 3]);
        }
      }
    } else {
#pragma unroll
      for (int s = 0; s < SA; ++s) {
        const int m = member(s0 + s);
        const TS x = xr[m < k ? m : 0];
        af[s] = (s_a >= 0 && m < k) ? x : (TS)0;
        if (s % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // the sum over a row of 16 lanes, in every lane of it
  auto row_sum = [](double v) {
    v += dpp_d<0xB1>(v);    // quad_perm [1,0,3,2]
    v += dpp_d<0x4E>(v);    // quad_perm [2,3,0,1]
    v += dpp_d<0x141>(v);   // row_half_mirror
    return v + dpp_d<0x140>(v);   // row_mirror
  };
  auto four = [](const double (&x)[4][16], int v) { return (x[0][v] + x[1][v]) + (x[2][v] + x[3][v]); };
  using First = std::integral_constant<int, 0>;
  using Second = std::integral_constant<int, S - SA>;
  if (n_items > 0) load_a(0, First{});
  for (int it = 0; it < n_items; ++it) {
    const long long off = item_off(it);
    const int v0 = 16 * (it % ngrp);
    double ab4[4];
    int st4[4];
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      st4[rr] = sidx(v0 + out_row(rr));
      ab4[rr] = st4[rr] >= 0 ? p.axb[off + st4[rr]] : 0.0;
    }
    acc_t out[2];
#pragma unroll
    for (int J = 0; J < 2; ++J) out[J] = acc_t{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < SA; ++s)
#pragma unroll
      for (int J = 0; J < 2; ++J) out[J] = ST::mma(af[s], bop[s][J], out[J]);
    if constexpr (SA < S) {
      load_a(it, Second{});
#pragma unroll
      for (int s = 0; s < SA; ++s)
#pragma unroll
        for (int J = 0; J < 2; ++J) out[J] = ST::mma(af[s], bop[SA + s][J], out[J]);
    }
    if (it + 1 < n_items) load_a(it + 1, First{});
    // lane holds Xa[vector out_row(rr)][member 32w + 16J + i16]
    double xe[4][2];
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      double sum = 0.0;
#pragma unroll
      for (int J = 0; J < 2; ++J) {
        const int e = 32 * wv + 16 * J + i16;
        xe[rr][J] = (e < k) ? (double)out[J][rr] + ab4[rr] : 0.0;
        sum += xe[rr][J];
      }
      sum = row_sum(sum);
      if (i16 == 0) spart[it & 1][wv][out_row(rr)] = sum;
    }
    __syncthreads();
    if (!EPI) {
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        if (st4[rr] < 0) continue;
        const double mean = four(spart[it & 1], out_row(rr)) / k;
        const long long o = off + st4[rr];
        TS* __restrict__ xa = ST::xa(p);
#pragma unroll
        for (int J = 0; J < 2; ++J) {
          const int e = 32 * wv + 16 * J + i16;
          if (e < k) xa[o * k + e] = (TS)(xe[rr][J] - mean);
        }
        if (wv == 0 && i16 == 0) p.axa[o] = mean;
      }
    } else {
      // the caller's epilogue (module_da_parallel.F90:219-261); the spreads'
      // member sums go through LDS like the mean
      const int cl = it / ngrp, lo = si + cl / ncl, la = sj + cl % ncl;
      const bool polar = fabs((double)p.g.glat[la - 1]) > p.polar_lat;
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const int vi = out_row(rr);
        const double mean = four(spart[it & 1], vi) / k;
        const long long o = off + (st4[rr] >= 0 ? st4[rr] : 0);
        double sb = 0.0, sa = 0.0;
#pragma unroll
        for (int J = 0; J < 2; ++J) {
          const int e = 32 * wv + 16 * J + i16;
          const bool in = e < k && st4[rr] >= 0;
          const double xbe = in ? (double)xb[o * k + e] : 0.0;
          double vv;
          if (polar) {
            vv = xbe + ab4[rr];
            sa += xbe * xbe;
          } else {
            vv = p.gamma1 * (ab4[rr] + xbe) + p.gamma2 * (mean + (xe[rr][J] - mean));
            if (e < k) sa += (vv - mean) * (vv - mean);
          }
          sb += xbe * xbe;
          if (in) p.xa_out[o * k + e] = vv;
        }
        sb = row_sum(sb);
        sa = row_sum(sa);
        if (i16 == 0) {
          sspr[0][wv][vi] = sb;
          sspr[EPI ? 1 : 0][wv][vi] = sa;
        }
      }
      __syncthreads();
      if (wv == 0 && i16 == 0) {
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          if (st4[rr] < 0) continue;
          const int vi = out_row(rr);
          const long long so = spread_index(p, lo, la, st4[rr]);
          p.spread_b[so] = sqrt(four(sspr[0], vi) / (double)(float)k);
          p.spread_a[so] = sqrt(four(sspr[EPI ? 1 : 0], vi) / (double)(float)k);
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// k = 65..128: the matrix does not fit a wavefront's registers, so the two
// per-matrix phases keep it in LDS (one 128-thread workgroup per matrix,
// thread r owns row r); the QL recurrence is k_ql_log<128>.
// ---------------------------------------------------------------------------

// Householder tridiagonalisation with A in LDS, one thread per row (one
// workgroup of max(KMAX, 64) threads per matrix); same outputs as k_tridiag.
template <int KMAX>
__global__ __launch_bounds__(KMAX < 64 ? 64 : KMAX) void k_tridiag_lds(EigParams p) {
  constexpr int NT = KMAX < 64 ? 64 : KMAX;
  constexpr int NW = NT / 64;
  constexpr int LD = KMAX + 1;
  __shared__ double sA[KMAX * LD];
  __shared__ double sv[KMAX], sw[KMAX];
  __shared__ double se_s[KMAX + 1], st_s[KMAX + 1];
  __shared__ double red[2 * NW];
  const int r = threadIdx.x;
  const long long a = p.a0 + blockIdx.x;
  if (a >= p.a0 + p.n_an) return;
  const long long al = a - p.a0;
  const int k = p.k, kp = p.kp;
  const double* __restrict__ Ag = p.A + al * (long long)kp * kp;
  double* __restrict__ refl = p.refl + al * (long long)kp * kp;
  const bool row = r < KMAX;             // thread owns a row of the LDS matrix
  const bool in_r = r < k;
  if (row)
    for (int c = 0; c < KMAX; ++c)
      sA[c * LD + r] = (in_r && c < k) ? a_entry(Ag, p.a_f32, kp, r, c) : 0.0;
  int slot = 0;
  __syncthreads();
  for (int j = 0; j + 2 < k; ++j) {
    const bool act = in_r && r > j;
    const double x = act ? sA[j * LD + r] : 0.0;
    const double x0 = uniform(sA[j * LD + j + 1]);
    const double rest = block_sum<NW>((act && r > j + 1) ? x * x : 0.0, red, slot);
    if (rest == 0.0) {
      if (row) refl[(long long)j * kp + r] = 0.0;
      if (r == 0) { se_s[j] = x0; st_s[j] = 0.0; }
      continue;
    }
    const double nrm = sqrt(rest + x0 * x0);
    const double alpha = (x0 >= 0.0) ? -nrm : nrm;
    const double v0 = x0 - alpha;
    const double tau = 2.0 / (rest + v0 * v0);
    const double v = act ? ((r == j + 1) ? v0 : x) : 0.0;
    if (row) sv[r] = v;
    __syncthreads();
    double pr0 = 0.0, pr1 = 0.0;
    if (act) {
      int c = j + 1;
      for (; c + 1 < k; c += 2) {
        pr0 = fma(sA[c * LD + r], sv[c], pr0);
        pr1 = fma(sA[(c + 1) * LD + r], sv[c + 1], pr1);
      }
      if (c < k) pr0 = fma(sA[c * LD + r], sv[c], pr0);
    }
    const double pr = act ? (pr0 + pr1) * tau : 0.0;
    const double K = 0.5 * tau * block_sum<NW>(v * pr, red, slot);
    const double wr = act ? pr - K * v : 0.0;
    if (row) sw[r] = wr;
    __syncthreads();
    if (act)
      for (int c = j + 1; c < k; ++c) sA[c * LD + r] -= v * sw[c] + wr * sv[c];
    if (row) refl[(long long)j * kp + r] = v;
    if (r == 0) { se_s[j] = alpha; st_s[j] = tau; }
    __syncthreads();
  }
  __syncthreads();
  if (!row) return;
  double* __restrict__ dg = p.d + al * kp;
  double* __restrict__ eg = p.e + al * kp;
  double* __restrict__ tg = p.tau + al * kp;
  dg[r] = in_r ? sA[r * LD + r] : 0.0;
  double ev = 0.0, tv = 0.0;
  if (r + 2 < k) { ev = se_s[r]; tv = st_s[r]; }
  else if (r == k - 2) ev = sA[(k - 2) * LD + k - 1];
  eg[r] = ev;
  tg[r] = tv;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// true when the batch updates a state (not only transforms)
static bool has_state(const EigParams& p) { return p.xb || p.xb32; }

// the update kernel for the batch's width, state precision and output mode
template <int KMAX>
static void launch_update(hipStream_t st, const EigParams& p, unsigned nb) {
  if constexpr (KMAX == 128) {
    if (p.state_f32) {
      if (p.epi) hipLaunchKernelGGL((k_update128<float, 1>), dim3(nb), dim3(256), 0, st, p);
      else hipLaunchKernelGGL((k_update128<float, 0>), dim3(nb), dim3(256), 0, st, p);
    } else {
      if (p.epi) hipLaunchKernelGGL((k_update128<double, 1>), dim3(nb), dim3(256), 0, st, p);
      else hipLaunchKernelGGL((k_update128<double, 0>), dim3(nb), dim3(256), 0, st, p);
    }
  } else {
    if (p.state_f32) {
      if (p.epi) hipLaunchKernelGGL((k_update<KMAX, float, 1>), dim3(nb), dim3(256), 0, st, p);
      else hipLaunchKernelGGL((k_update<KMAX, float, 0>), dim3(nb), dim3(256), 0, st, p);
    } else {
      if (p.epi) hipLaunchKernelGGL((k_update<KMAX, double, 1>), dim3(nb), dim3(256), 0, st, p);
      else hipLaunchKernelGGL((k_update<KMAX, double, 0>), dim3(nb), dim3(256), 0, st, p);
    }
  }
}

// one of the four stages over the batch p: tridiagonalisation; the guard's
// smallest eigenvalue (reduced precision); trans and overline_w; update.  With
// ql_first stages 1 and 2 are the QL recurrence and its rotations.
template <int KMAX>
static hipError_t launch_eig_stage_k(hipStream_t st, const EigParams& p, int stage) {
  const unsigned nb = (unsigned)p.n_an;
  const unsigned nq = (unsigned)((p.n_an + 63) / 64);
  if (stage == 0) {
    if (p.tridiag_lds) hipLaunchKernelGGL(k_tridiag_lds<KMAX>, dim3(nb), dim3(KMAX < 64 ? 64 : KMAX), 0, st, p);
    else if constexpr (KMAX == 128) hipLaunchKernelGGL(k_tridiag128, dim3(nb), dim3(256), 0, st, p);
    else hipLaunchKernelGGL(k_tridiag<KMAX>, dim3(KMAX == 32 ? (nb + 1) / 2 : nb), dim3(64), 0, st, p);
  } else if (stage == 3) {
    if (has_state(p)) launch_update<KMAX>(st, p, nb);
  } else if (!p.ql_first) {
    const hipError_t e = launch_sqrt(st, p, stage == 1);
    if (e != hipSuccess) return e;
    if (stage == 2)
      hipLaunchKernelGGL(k_indef<KMAX>, dim3((unsigned)std::min(p.n_an, KMAX < 128 ? 1024LL : 256LL)),
                         dim3(KMAX < 64 ? 64 : KMAX), 0, st, p);
  } else if (stage == 1) {
    hipLaunchKernelGGL(k_ql_log<KMAX>, dim3(nq), dim3(64), 0, st, p);
  } else {
    if constexpr (KMAX == 128) hipLaunchKernelGGL(k_rot128, dim3(nb), dim3(256), 0, st, p);
    else hipLaunchKernelGGL(k_rot<KMAX>, dim3(nb), dim3(64), 0, st, p);
  }
  return hipGetLastError();
}

static hipError_t launch_eig_stage(hipStream_t st, const EigParams& p, int stage) {
  if (p.k <= 32) return launch_eig_stage_k<32>(st, p, stage);
  if (p.k <= 64) return launch_eig_stage_k<64>(st, p, stage);
  return launch_eig_stage_k<128>(st, p, stage);
}

hipError_t launch_eig(hipStream_t st, const EigParams& p, hipEvent_t* ev) {
  if (p.n_an <= 0) return hipSuccess;
  if (p.k > 128) return hipErrorInvalidValue;
  for (int stage = 0; stage < 4; ++stage) {
    hipError_t e = ev ? hipEventRecord(ev[stage], st) : hipSuccess;
    if (e == hipSuccess) e = launch_eig_stage(st, p, stage);
    if (e != hipSuccess) return e;
  }
  return ev ? hipEventRecord(ev[4], st) : hipSuccess;
}

hipError_t launch_zero_ints(hipStream_t st, int* p, int n) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_zero_ints, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, n);
  return hipGetLastError();
}

// The list pass: QL, eigenvectors + trans and update over the analyses the
// first pass flagged (p.list, *p.list_n of them, at most p.list_cap).  Grids
// are sized for list_cap; workgroups past the count exit at once, so the
// launch needs no count on the host.
hipError_t launch_eig_rerun(hipStream_t st, const EigParams& p) {
  if (!p.list || p.list_cap <= 0) return hipSuccess;
  const unsigned nb = (unsigned)p.list_cap;
  const unsigned nq = (unsigned)((p.list_cap + 63) / 64);
  for (int stage = 1; stage < 4; ++stage) {
    if (p.k <= 32) {
      if (stage == 1) hipLaunchKernelGGL(k_ql_log<32>, dim3(nq), dim3(64), 0, st, p);
      else if (stage == 2) hipLaunchKernelGGL(k_rot<32>, dim3(nb), dim3(64), 0, st, p);
      else if (has_state(p)) launch_update<32>(st, p, nb);
    } else if (p.k <= 64) {
      if (stage == 1) hipLaunchKernelGGL(k_ql_log<64>, dim3(nq), dim3(64), 0, st, p);
      else if (stage == 2) hipLaunchKernelGGL(k_rot<64>, dim3(nb), dim3(64), 0, st, p);
      else if (has_state(p)) launch_update<64>(st, p, nb);
    } else {
      if (stage == 1) hipLaunchKernelGGL(k_ql_log<128>, dim3(nq), dim3(64), 0, st, p);
      else if (stage == 2) hipLaunchKernelGGL(k_rot128, dim3(nb), dim3(256), 0, st, p);
      else if (has_state(p)) launch_update<128>(st, p, nb);
    }
  }
  return hipGetLastError();
}

}  // namespace dida
