// letkf_sqrt.hip -- trans and overline_w from the tridiagonal form, without
// eigenvectors.
//
// letkf_core needs (letkf_core.F90:107-225), with M = A + (k-1)/rho I,
//   T = sqrt(k-1) M^(-1/2)   and   overline_w = M^(-1) b,
// and trans = T + overline_w 1^T.  With A = Q D Q^T tridiagonalised
// (k_tridiag: reflectors and D), M^(-1/2) = Q (D + (k-1)/rho I)^(-1/2) Q^T:
//
//   1. The inverse square root of the tridiagonal matrix by the trapezoidal
//      rule on an elliptic contour (Hale, Higham & Trefethen, SIAM J. Numer.
//      Anal. 46, 2008, method 3): x^(-1/2) = sum_j c_j / (x + s_j) on
//      [m, M] to rounding with N = 1.86 ln(16 M/m) poles (15 at M/m = 100),
//      all c_j, s_j > 0, so nothing cancels.  m is known, (k-1)/rho.
//   2. Each resolvent G = (D + s_j)^(-1) is semiseparable: from the pivots
//      eta_l of the elimination that runs up from the last row,
//      G(i,l+1) = r_l G(i,l) for l >= i with r_l = -e_l / eta_(l+1), and
//      G(l+1,l+1) = 1/eta_(l+1) + r_l^2 G(l,l), G(0,0) = 1/eta_0 (sums of
//      positive terms).  Off-diagonal 16x16 tiles of sum_j c_j G_j are
//      products of 16 x N by N x 16 factors (MFMA); diagonal tiles follow the
//      recurrence along the row.
//   3. The two-sided product with Q in blocks of 16 reflectors (compact WY,
//      Schreiber & Van Loan 1989): S <- P S P^T, P = I - V W V^T, as the
//      symmetric rank-32 update S + V X^T + X V^T with
//      X = -S V W^T + 1/2 V (W V^T S V W^T), on f64 MFMA with S in registers.
//      A 16x16x4 f64 result tile (row q + 4r, column i) is the B operand of
//      its own tile and the A operand of the transposed tile, so S, the
//      products Y and X move through no LDS.
//   4. overline_w = T (T b) / (k-1).
//
// It replaces the QL recurrence and the product of its rotations (k_indef keeps
// them for M not positive definite), ~4,500 dependent Givens steps per matrix at k = 64
// and 6 k flops for each.  64,800 matrices: k = 64, 3.95 + 7.25 -> 0.22
// (k_lmin) + 2.5 ms; k = 128, 50 + 80 -> 0.43 + 20 ms; and a single matrix of
// k = 64 takes 50 us here against 1.3 ms.  Bound: the wavefront's own chain
// (per matrix of k = 64 some 150k cycles with two wavefronts on a SIMD, of
// which 47k are MFMA issue; the pivots 25k, W 20k, the last stores 15k).
#include "letkf_device.h"
#include "letkf_kernels.h"
#include "letkf_eig.h"

namespace dida {

// 1/x to rounding for normal x: the hardware estimate (24 bits) and one step
// of third order, r (1 + h + h^2) with h = 1 - x r: three dependent FMAs where
// two Newton steps take four
__device__ __forceinline__ double rcp_nr(double x) {
  const double r = __builtin_amdgcn_rcp(x);
  const double h = fma(-x, r, 1.0);
  return fma(r, fma(h, h, h), r);
}

// ---------------------------------------------------------------------------
// k_lmin (reduced-precision products): the smallest eigenvalue of the
// tridiagonal form where it is negative, else 0, for the guard
// (letkf_core_mpal.F90:113-118).
// ---------------------------------------------------------------------------
// Eight lanes per matrix.  All pivots of D - x are positive exactly when x is
// below every eigenvalue, so each pass tests eight points at once and keeps
// the ninth of the interval where the answer lies: first a logarithmic scale
// from the norm G down to 2^-56 G, then linear, to 2^-54 G.  One wavefront
// takes 8 matrices: the recurrence is a chain of k divisions, and eight lanes
// keep the passes (15) and the LDS (4 KB at k = 32, 16 KB at 128) small.
template <int KMAX>
__global__ __launch_bounds__(64) void k_lmin(EigParams p) {
  __shared__ double sa[KMAX][8], se2[KMAX][8];
  const int lane = threadIdx.x, t = lane & 7, mt = lane >> 3;
  const int k = p.k, kp = p.kp;
  const long long al0 = (long long)blockIdx.x * 8;
  for (int e = lane; e < 8 * KMAX; e += 64) {
    const int m = e / KMAX, i = e % KMAX;
    const bool in = al0 + m < p.n_an && i < k;
    sa[i][m] = in ? p.d[(al0 + m) * kp + i] : 1.0;
    const double ev = (in && i + 1 < k) ? p.e[(al0 + m) * kp + i] : 0.0;
    se2[i][m] = ev * ev;
  }
  __syncthreads();
  // G bounds every eigenvalue in absolute value
  double G = 0.0, prev = 0.0;
  for (int i = 0; i < k; ++i) {
    const double ev = sqrt(se2[i][mt]);
    G = fmax(G, fabs(sa[i][mt]) + prev + ev);
    prev = ev;
  }
  auto below = [&](double x) -> bool {     // x < lambda_min
    double eta = sa[0][mt] - x;
    bool pos = eta > 0.0;
    for (int i = 1; i < k; ++i) {
      eta = fma(-se2[i - 1][mt], rcp_nr(eta), sa[i][mt] - x);
      pos = pos && eta > 0.0;
    }
    return pos;
  };
  // points below the answer among the group's eight (they descend with t):
  // the first such t, 8 if none
  auto first_below = [&](double x) -> int {
    const unsigned long long b = __builtin_amdgcn_ballot_w64(below(x));
    const unsigned g = (unsigned)(b >> (8 * mt)) & 0xffu;
    return g ? __builtin_ctz(g) : 8;
  };
  double lo = 0.0, hi = 0.0;               // lambda_min in [lo, hi)
  {
    // 0, then -G 2^-56 .. -G 2^-8 by factors of 2^8
    const double x = t == 0 ? 0.0 : -G * exp2(-56.0 + 8.0 * (t - 1));
    const int f = first_below(x);
    if (f > 0) {
      lo = f == 8 ? -G * 1.0000001 : -G * exp2(-56.0 + 8.0 * (f - 1));
      hi = f == 1 ? 0.0 : -G * exp2(-56.0 + 8.0 * (f - 2));
    }
  }
  const double tol = G * 5.551115123125783e-17;
  // every lane of the wavefront runs the passes of the widest interval
  while (__builtin_amdgcn_ballot_w64(hi - lo > tol)) {
    const double w = (hi - lo) * (1.0 / 9.0);
    const int f = first_below(hi - w * (t + 1));
    const double nhi = f == 0 ? hi : hi - w * f;
    const double nlo = f == 8 ? lo : hi - w * (f + 1);
    if (!(nhi - nlo < hi - lo)) break;     // NaN, or the interval is one ulp
    if (hi - lo > tol) { lo = nlo; hi = nhi; }
  }
  if (t == 0 && al0 + mt < p.n_an) p.lam[(al0 + mt) * kp] = 0.5 * (lo + hi);
}

// ---------------------------------------------------------------------------
// k_vec
// ---------------------------------------------------------------------------
// The j-th pole and weight of x^(-1/2) on [1, kappa], of N, from theta series
// in the nome q = 1 / (16 kappa) (slightly below the nome of the modulus
// kappa^(-1/2), so the interval covered is slightly larger; kappa >= 4 keeps
// three terms enough).  The half of the contour past the quarter period uses
// the reflection sn(iK' - w) = 1 / (kmod sn w).
__device__ __forceinline__ void sqrt_pole(double q, double L, int N, int j, double& s2, double& c) {
  const bool refl = 2 * j + 1 > N;
  const double v = 0.5 * L * ((refl ? N - 1 - j : j) + 0.5) / N;
  const double E = exp(v), Ei = 1.0 / E;
  const double E2 = E * E, Ei2 = Ei * Ei, E3 = E2 * E, Ei3 = Ei2 * Ei;
  const double E4 = E2 * E2, Ei4 = Ei2 * Ei2, E6 = E3 * E3, Ei6 = Ei3 * Ei3;
  const double q2 = q * q, q4 = q2 * q2, q6 = q4 * q2, q9 = q4 * q4 * q;
  const double th3 = 1.0 + 2.0 * (q + q4 + q9), th4 = 1.0 - 2.0 * (q - q4 + q9);
  const double d2 = 1.0 + q2 + q6;
  const double C4 = 1.0 - q * (E2 + Ei2) + q4 * (E4 + Ei4) - q9 * (E6 + Ei6);
  const double C3 = 1.0 + q * (E2 + Ei2) + q4 * (E4 + Ei4) + q9 * (E6 + Ei6);
  const double S1 = 0.5 * ((E - Ei) - q2 * (E3 - Ei3) + q6 * (E4 * E - Ei4 * Ei));
  const double C2 = 0.5 * ((E + Ei) + q2 * (E3 + Ei3) + q6 * (E4 * E + Ei4 * Ei));
  double s = th3 * S1 / (d2 * C4);
  double D = th4 * th4 * C2 * C3 / (th3 * C4 * C4 * d2);
  if (refl) {
    const double kmod = 4.0 * sqrt(q) * d2 * d2 / (th3 * th3);
    const double ks = kmod * s;
    D = D / (ks * s);
    s = 1.0 / ks;
  }
  s2 = s * s;
  c = th3 * th3 * L / (3.14159265358979323846 * N) * D;
}

// NW wavefronts share a matrix, wavefront w owning the tile columns
// [w CPW, (w + 1) CPW) of S.  k <= 64: one wavefront (S is 128 registers at
// k = 64, two wavefronts per SIMD); k <= 128: four.
template <int KMAX, int NW>
struct SqrtLds {
  static constexpr int TT = KMAX / 16, NP = 16;
  static constexpr int LDP = NP + 1;               // r, g rows (one per state index)
  static constexpr int LDV = KMAX + 1, LDT = 17;
  // stages 1, 2: r, g, the tile products R, the tridiagonal matrix; then the
  // diagonal tiles; stage 3: the reflectors V, then Gram / Z^T in turn, W, and
  // for NW > 1 the partial products and the shared X tiles
  static constexpr int F = 2 * KMAX * LDP + TT * NP + 2 * KMAX;
  static constexpr int FD = TT * 16 * LDT;
  static constexpr int B = 2 * 16 * LDV + 16 * LDT + (NW > 1 ? NW * 256 + TT * 256 : 0);
  static constexpr int N = F > B ? (F > FD ? F : FD) : (B > FD ? B : FD);
};

// k <= 32: three wavefronts per SIMD hide more of each one's chain than the
// spills they cost (200 B a lane): 2,073,600 matrices 28 -> 25 ms, four
// wavefronts 31 ms.  k > 32 spills at two already (k = 64: 196 B, k = 128: 340).
template <int KMAX, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(KMAX == 32 ? 3 : 2)))
void k_vec(EigParams p) {
  using Lds = SqrtLds<KMAX, NW>;
  constexpr int TT = Lds::TT, NP = Lds::NP, LDP = Lds::LDP, LDV = Lds::LDV, LDT = Lds::LDT;
  constexpr int CPW = TT / NW;
  static_assert(TT % NW == 0, "tile columns split evenly");
  __shared__ __align__(16) double sbuf[Lds::N];
  __shared__ double sb[KMAX], sw[KMAX];
  __shared__ double sred[4];
  __shared__ int s_ok;                             // apart from sred: no barrier between them
  double* const sr = sbuf;                         // [KMAX][LDP]
  double* const sg = sr + KMAX * LDP;              // [KMAX][LDP], right after sr
  double* const sR = sg + KMAX * LDP;              // [TT][NP]
  double* const sd = sR + TT * NP;                 // diagonal and subdiagonal, shifted
  double* const se = sd + KMAX;
  const int tid = threadIdx.x, lane = tid & 63, w = NW > 1 ? uniform(tid >> 6) : 0;
  const int i16 = lane & 15, q = lane >> 4;
  const long long al = blockIdx.x, a = p.a0 + al;
  const int k = p.k, kp = p.kp;
  double* __restrict__ refl = p.refl + al * (long long)kp * kp;
  const double* __restrict__ tg = p.tau + al * kp;
  const double m0 = (double)(k - 1) / p.inflation;

  // ---- the shifted tridiagonal matrix, its norm and the poles ----
  double shift = m0;
  if (p.guard) {
    const double lm = p.lam[al * kp];
    if (lm < 0.0) shift -= lm;
  }
  double bound = 0.0;
  for (int i = tid; i < KMAX; i += 64 * NW) {
    const bool in = i < k;
    const double dv = in ? p.d[al * kp + i] + shift : m0;
    const double ev = (in && i + 1 < k) ? p.e[al * kp + i] : 0.0;
    const double el = (in && i > 0) ? p.e[al * kp + i - 1] : 0.0;
    sd[i] = dv;
    se[i] = ev;
    sb[i] = in ? p.b[al * kp + i] : 0.0;
    bound = fmax(bound, fabs(dv) + fabs(ev) + fabs(el));
  }
  bound = wave_reduce_full(bound, [](double x, double y) { return fmax(x, y); });
  if constexpr (NW > 1) {
    if (lane == 0) sred[w] = bound;
  }
  __syncthreads();
  if constexpr (NW > 1) bound = fmax(fmax(sred[0], sred[1]), fmax(sred[2], sred[3]));
  bound = uniform(bound);

  // Rows past k stay out of the recurrences: S is zero there.
  // m: a lower bound of the spectrum.  0.9 (k-1)/rho holds for every A whose
  // negative rounding is small; it is checked beside the first poles' pivots
  // (lane NP tests that D - m has positive pivots), and where it fails the
  // largest (0.9 / 2^t) (k-1)/rho that holds is taken, once.  None holding (or
  // (k-1)/rho = 0, an infinite rho): D is not positive definite, or has no such
  // bound, and k_indef takes the matrix, or it is not finite.
  double m = 0.9 * m0, L = 0.0, qn = 0.0;
  int N = 0;
  // pivots of the poles c0 .. c0 + NP - 1, one lane per pole (wavefront 0); a
  // lane past the last pole carries weight 0.  False when a pivot is not
  // positive.
  auto chain = [&](int c0) -> bool {
    bool ok = true;
    if (w == 0) {
      double s2 = 1.0, c = 0.0;
      const int j = c0 + lane;
      if (lane < NP && j < N) {
        sqrt_pole(qn, L, N, j, s2, c);
        c *= sqrt(m * (double)(k - 1));
      }
      const double sg_ = lane == NP ? -m : s2 * m;
      if (lane <= NP) {
        double eta = sd[k - 1] + sg_;
        bool pos = eta > 0.0;
        double ie = rcp_nr(eta);
        if (lane < NP) {
          for (int l = KMAX - 1; l >= k; --l) {
            sr[l * LDP + lane] = 0.0;
            sg[l * LDP + lane] = 0.0;
          }
          sg[(k - 1) * LDP + lane] = ie;
          sr[(k - 1) * LDP + lane] = 0.0;
        }
        // lanes that store nothing write a column of padding (NP); the loads
        // of eight steps go ahead of their chain
        const int col = lane < NP ? lane : NP;
        for (int l0 = (k - 2) & ~7; l0 >= 0; l0 -= 8) {
          double d8[8], e8[8];
#pragma unroll
          for (int t = 0; t < 8; ++t) {
            d8[t] = sd[l0 + t];
            e8[t] = se[l0 + t];
          }
#pragma unroll
          for (int t = 7; t >= 0; --t) {
            if (l0 + t > k - 2) continue;
            const double e = e8[t];
            eta = fma(-e * e, ie, d8[t] + sg_);
            pos = pos && eta > 0.0;
            sr[(l0 + t) * LDP + col] = -e * ie;
            ie = rcp_nr(eta);
            sg[(l0 + t) * LDP + col] = ie;
          }
        }
        // c_j times the diagonal of the resolvent
        double g = c * ie;
        sg[col] = g;
        for (int l0 = 0; l0 + 1 < k; l0 += 8) {
          double r8[8], i8[8];
#pragma unroll
          for (int t = 0; t < 8; ++t) {
            const int l = min(l0 + t, KMAX - 2);
            r8[t] = sr[l * LDP + col];
            i8[t] = c * sg[(l + 1) * LDP + col];
          }
#pragma unroll
          for (int t = 0; t < 8; ++t) {
            if (l0 + t + 1 >= k) continue;
            g = fma(r8[t] * r8[t], g, i8[t]);
            sg[(l0 + t + 1) * LDP + col] = g;
          }
        }
        ok = pos;
      }
      ok = !__builtin_amdgcn_ballot_w64(lane <= NP && !ok);
    }
    return ok;
  };
  for (bool again = false;; again = true) {
    const double kappa = fmax(bound / m, 4.0);
    qn = 1.0 / (16.0 * kappa);
    L = -log(qn);
    // sqrt_pole's terms stay finite up to 1e200 (862 poles)
    const bool in_range = kappa <= 1e200;
    N = in_range ? (int)(1.86 * L + 0.8) : 0;
    bool ok = chain(0) && in_range;
    if constexpr (NW > 1) {
      if (tid == 0) s_ok = ok;
      __syncthreads();
      ok = s_ok != 0;
      __syncthreads();
    }
    if (ok) break;
    // lane t: does D - 0.9 2^-(t+1) m0 have positive pivots?
    const double x = 0.9 * m0 * exp2(-1.0 - (double)lane);
    double eta = sd[k - 1] - x;
    bool pos = eta > 0.0;
    for (int l = k - 2; l >= 0; --l) {
      const double e = se[l];
      eta = fma(-e * e, rcp_nr(eta), sd[l] - x);
      pos = pos && eta > 0.0;
    }
    const unsigned long long bal = __builtin_amdgcn_ballot_w64(pos);
    const int f = bal ? __builtin_ctzll(bal) : 64;
    if (again || !(m0 > 0.0) || f > 50 || !(bound < 1e290)) {
      // k_indef takes a finite matrix; nothing comes of one that is not
      bool fin = true;
      for (int i = lane; i < k; i += 64)
        fin = fin && __builtin_isfinite(p.d[al * kp + i]) && __builtin_isfinite(p.e[al * kp + i]);
      fin = __builtin_amdgcn_ballot_w64(!fin) == 0;
      if (tid == 0) {
        p.status[a] = fin ? kStatusIndefinite : kStatusNonFinite;
        if (fin) atomicAdd(p.flag_n, 1);
        atomicAdd(p.flag_total, 1);
      }
      if (!fin) nan_transform(p, a);
      return;
    }
    m = 0.9 * m0 * exp2(-1.0 - (double)f);
  }
  d4 S[TT][CPW];
#pragma unroll
  for (int I = 0; I < TT; ++I)
#pragma unroll
    for (int J = 0; J < CPW; ++J) S[I][J] = d4{0.0, 0.0, 0.0, 0.0};
  // row i16 of a diagonal tile this wavefront owns (lane quarter q: its q-th;
  // k = 32 and 128 own two, so the upper lanes repeat the lower ones' work)
  const int dt = w * CPW + (q < CPW ? q : q % CPW);
  double fd[16];
#pragma unroll
  for (int o = 0; o < 16; ++o) fd[o] = 0.0;

  for (int c0 = 0;;) {
    __syncthreads();
    // diagonal tiles: lane (tile, i16) follows row i16 of its tile to the
    // right, all poles at once (entries past the tile's end are not used; the
    // last rows' reads past sr fall in sg)
    {
      double g[NP];
      const int row = 16 * dt + i16;
#pragma unroll
      for (int j = 0; j < NP; ++j) g[j] = sg[row * LDP + j];
#pragma unroll
      for (int o = 0; o < 16; ++o) {
        if (o > 0) {
#pragma unroll
          for (int j = 0; j < NP; ++j) g[j] *= sr[(row + o - 1) * LDP + j];
        }
        double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
#pragma unroll
        for (int j = 0; j < NP; j += 4) {
          s0 += g[j];
          s1 += g[j + 1];
          s2 += g[j + 2];
          s3 += g[j + 3];
        }
        fd[o] += (s0 + s1) + (s2 + s3);
        pin(fd[o]);
      }
    }
    __syncthreads();
    // per tile and pole: U = g times the product of r to the tile's end, P =
    // the product of r from the tile's start, R = the whole tile's product
    for (int e = tid; e < TT * NP; e += 64 * NW) {
      const int t16 = 16 * (e / NP), j = e % NP;
      double suf = 1.0;
#pragma unroll
      for (int l = 15; l >= 0; --l) {
        suf *= sr[(t16 + l) * LDP + j];
        sg[(t16 + l) * LDP + j] *= suf;
      }
      sR[e] = suf;
      double pre = 1.0;
#pragma unroll
      for (int l = 0; l < 16; ++l) {
        const double r = sr[(t16 + l) * LDP + j];
        sr[(t16 + l) * LDP + j] = pre;
        pre *= r;
      }
    }
    __syncthreads();
    // off-diagonal tiles: S(I, J) += U_I (prod R) P_J^T and its transpose
#pragma unroll
    for (int Jl = 0; Jl < CPW; ++Jl) {
      const int J = w * CPW + Jl;
      double pj[4], uj[4], f[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        pj[s] = sr[(16 * J + i16) * LDP + 4 * s + q];
        uj[s] = sg[(16 * J + i16) * LDP + 4 * s + q];
        f[s] = 1.0;
      }
#pragma unroll
      for (int d = 1; d < TT; ++d) {               // I = J - d
#pragma unroll
        for (int I = 0; I < TT; ++I)
          if (I == J - d) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
              S[I][Jl] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                  sg[(16 * I + i16) * LDP + 4 * s + q] * f[s], pj[s], S[I][Jl], 0, 0, 0);
            pin(S[I][Jl]);
          }
        if (J - d >= 0) {
#pragma unroll
          for (int s = 0; s < 4; ++s) f[s] *= sR[(J - d) * NP + 4 * s + q];
        }
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) f[s] = 1.0;
#pragma unroll
      for (int d = 1; d < TT; ++d) {               // I = J + d
#pragma unroll
        for (int I = 0; I < TT; ++I)
          if (I == J + d) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
              S[I][Jl] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                  sr[(16 * I + i16) * LDP + 4 * s + q], uj[s] * f[s], S[I][Jl], 0, 0, 0);
            pin(S[I][Jl]);
          }
        if (J + d < TT) {
#pragma unroll
          for (int s = 0; s < 4; ++s) f[s] *= sR[(J + d) * NP + 4 * s + q];
        }
      }
    }
    __syncthreads();
    c0 += NP;
    if (c0 >= N) break;
    (void)chain(c0);
  }
  // the diagonal tiles through LDS into the result layout
#pragma unroll
  for (int o = 0; o < 16; ++o)
    if (q < CPW && i16 + o < 16) {
      sbuf[(dt * 16 + i16) * LDT + i16 + o] = fd[o];
      sbuf[(dt * 16 + i16 + o) * LDT + i16] = fd[o];
    }
  __syncthreads();
#pragma unroll
  for (int Jl = 0; Jl < CPW; ++Jl) {
#pragma unroll
    for (int I = 0; I < TT; ++I)
      if (I == w * CPW + Jl) {
#pragma unroll
        for (int r = 0; r < 4; ++r) S[I][Jl][r] = sbuf[(I * 16 + q + 4 * r) * LDT + i16];
      }
  }

  // ---- S <- Q S Q^T, the last block of 16 reflectors first ----
  double* const sV = sbuf;                         // [16 reflectors][LDV]
  double* const sZ = sV + 16 * LDV;                // Z^T, [16][LDV]
  double* const sG = sZ;                           // Gram of the block, before Z
  double* const sT = sZ + 16 * LDV;                // -W of the block
  double* const sM = sT + 16 * LDT;                // NW > 1: partial V^T Z
  double* const sX = sM + NW * 256;                // NW > 1: X^T tiles
  const int nref = k > 2 ? k - 2 : 0;
  constexpr int RPW = 16 / NW;                     // reflectors a wavefront stages
  constexpr int CV = KMAX < 64 ? 1 : KMAX / 64;    // values per lane and reflector
  // rolled over the blocks (the code of all of them unrolled is larger than
  // the instruction cache), with uniform branches around the tile rows where
  // V is zero
#pragma unroll 1
  for (int b = (nref + 15) / 16 - 1; b >= 0; --b) {
    double vv[RPW * CV];
#pragma unroll
    for (int t = 0; t < RPW; ++t)
#pragma unroll
      for (int h = 0; h < CV; ++h) {
        // unconditional loads (the block has kp rows), then a select: a load
        // under a test waits for the one before it (18k cycles a block)
        const int j = 16 * b + w * RPW + t, c = KMAX < 64 ? i16 + 16 * (q & 1) : lane + 64 * h;
        vv[t * CV + h] = refl[(long long)j * kp + c];
      }
    const double tau = 16 * b + i16 < nref ? tg[16 * b + i16] : 0.0;
    __syncthreads();
#pragma unroll
    for (int t = 0; t < RPW; ++t)
#pragma unroll
      for (int h = 0; h < CV; ++h) {
        const int j = 16 * b + w * RPW + t, c = KMAX < 64 ? i16 + 16 * (q & 1) : lane + 64 * h;
        sV[(w * RPW + t) * LDV + c] = j < nref ? vv[t * CV + h] : 0.0;
      }
    __syncthreads();
    // W of P = I - V W V^T (upper triangular), row i16 in every lane quarter;
    // its negative goes to LDS
    {
      d4 g = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int I = 0; I < TT; ++I)
        if (I >= b)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const double v = sV[i16 * LDV + 16 * I + 4 * s + q];
          g = __builtin_amdgcn_mfma_f64_16x16x4f64(v, v, g, 0, 0, 0);
        }
      pin(g);
#pragma unroll
      for (int r = 0; r < 4; ++r) sG[(q + 4 * r) * LDT + i16] = g[r];
      __syncthreads();
      // row i16 of W, column by column: W(:, j) = tau_j (e_j - sum_(l<j)
      // W(:, l) G(l, j)), each finished column taken out of all later ones at
      // once, so the chain is two operations a column
      double wr[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) wr[j] = i16 == j ? 1.0 : 0.0;
#pragma unroll
      for (int l = 0; l < 16; ++l) {
        wr[l] *= readlane_d(tau, l);
#pragma unroll
        for (int j = l + 1; j < 16; ++j) wr[j] = fma(-wr[l], sG[l * LDT + j], wr[j]);
        if ((l & 3) == 3) {
#pragma unroll
          for (int j = 0; j < 16; ++j) pin(wr[j]);
        }
      }
#pragma unroll
      for (int j = 0; j < 16; ++j)
        if ((j & 3) == q) sT[i16 * LDT + j] = -wr[j];
    }
    __syncthreads();
    double wt[4];                                  // -W, A operand (also the B operand of -W^T)
#pragma unroll
    for (int s = 0; s < 4; ++s) wt[s] = sT[i16 * LDT + 4 * s + q];
    // Z^T = -W (V^T S), tile columns of this wavefront
    d4 Z[CPW];
    {
      d4 Y[CPW];
#pragma unroll
      for (int J = 0; J < CPW; ++J) Y[J] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int I = 0; I < TT; ++I)
        if (I >= b)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const double v = sV[i16 * LDV + 16 * I + 4 * s + q];
#pragma unroll
          for (int J = 0; J < CPW; ++J)
            Y[J] = __builtin_amdgcn_mfma_f64_16x16x4f64(v, S[I][J][s], Y[J], 0, 0, 0);
          if (s == 3) {
#pragma unroll
            for (int J = 0; J < CPW; ++J) pin(Y[J]);
          }
        }
#pragma unroll
      for (int J = 0; J < CPW; ++J) {
        Z[J] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 4; ++s)
          Z[J] = __builtin_amdgcn_mfma_f64_16x16x4f64(wt[s], Y[J][s], Z[J], 0, 0, 0);
      }
    }
    // K = W V^T S V W^T: first V^T Z = -(V^T S V) W^T over the rows of this
    // wavefront's tile columns (Z through LDS: its transposed operand)
#pragma unroll
    for (int J = 0; J < CPW; ++J)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sZ[(q + 4 * r) * LDV + 16 * (w * CPW + J) + i16] = Z[J][r];
    __syncthreads();
    d4 M1 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int J = 0; J < CPW; ++J) {
      if (w * CPW + J < b) continue;               // V is zero there
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int c = 16 * (w * CPW + J) + 4 * s + q;
        M1 = __builtin_amdgcn_mfma_f64_16x16x4f64(sV[i16 * LDV + c], sZ[i16 * LDV + c], M1, 0, 0, 0);
      }
    }
    if constexpr (NW > 1) {
#pragma unroll
      for (int r = 0; r < 4; ++r) sM[(w * 4 + r) * 64 + lane] = M1[r];
      __syncthreads();
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        double s = sM[r * 64 + lane];
#pragma unroll
        for (int u = 1; u < NW; ++u) s += sM[(u * 4 + r) * 64 + lane];
        M1[r] = s;
      }
    }
    d4 K = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < 4; ++s)
      K = __builtin_amdgcn_mfma_f64_16x16x4f64(M1[s], wt[s], K, 0, 0, 0);
    // X^T = Z^T + 1/2 K V^T
#pragma unroll
    for (int J = 0; J < CPW; ++J) {
      if (w * CPW + J >= b) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
          Z[J] = __builtin_amdgcn_mfma_f64_16x16x4f64(
              0.5 * K[s], sV[(4 * s + q) * LDV + 16 * (w * CPW + J) + i16], Z[J], 0, 0, 0);
      }
      if constexpr (NW > 1) {
#pragma unroll
        for (int r = 0; r < 4; ++r) sX[((w * CPW + J) * 4 + r) * 64 + lane] = Z[J][r];
      }
    }
    if constexpr (NW > 1) __syncthreads();
    // S(I, J) += V_I X_J^T (I >= b) + X_I V_J^T (J >= b)
#pragma unroll
    for (int I = 0; I < TT; ++I)
      if (I >= b) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const double v = sV[(4 * s + q) * LDV + 16 * I + i16];
#pragma unroll
          for (int J = 0; J < CPW; ++J)
            S[I][J] = __builtin_amdgcn_mfma_f64_16x16x4f64(v, Z[J][s], S[I][J], 0, 0, 0);
        }
#pragma unroll
        for (int J = 0; J < CPW; ++J) pin(S[I][J]);
      }
#pragma unroll
    for (int J = 0; J < CPW; ++J)
      if (w * CPW + J >= b) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const double v = sV[(4 * s + q) * LDV + 16 * (w * CPW + J) + i16];
#pragma unroll
          for (int I = 0; I < TT; ++I) {
            double x;
            if constexpr (NW > 1) x = sX[(I * 4 + s) * 64 + lane];
            else x = Z[I < CPW ? I : 0][s];
            S[I][J] = __builtin_amdgcn_mfma_f64_16x16x4f64(x, v, S[I][J], 0, 0, 0);
          }
        }
#pragma unroll
        for (int I = 0; I < TT; ++I) pin(S[I][J]);
      }
  }

  // ---- overline_w = S (S b) / (k-1); S is symmetric, so each lane sums the
  // rows it holds of its columns and the four lane quarters are added ----
  auto matvec = [&](const double* x, double (&y)[CPW]) {
#pragma unroll
    for (int J = 0; J < CPW; ++J) {
      double s0 = 0.0, s1 = 0.0;
#pragma unroll
      for (int I = 0; I < TT; ++I) {
        s0 = fma(S[I][J][0], x[16 * I + q], s0);
        s1 = fma(S[I][J][1], x[16 * I + q + 4], s1);
        s0 = fma(S[I][J][2], x[16 * I + q + 8], s0);
        s1 = fma(S[I][J][3], x[16 * I + q + 12], s1);
      }
      double s = s0 + s1;
      s += __shfl_xor(s, 16, 64);
      y[J] = s + __shfl_xor(s, 32, 64);
    }
  };
  double y[CPW];
  matvec(sb, y);
  if (q == 0) {
#pragma unroll
    for (int J = 0; J < CPW; ++J) sw[16 * (w * CPW + J) + i16] = y[J];
  }
  __syncthreads();
  matvec(sw, y);
  __syncthreads();
  bool bad = false;
#pragma unroll
  for (int J = 0; J < CPW; ++J) {
    const int f = 16 * (w * CPW + J) + i16;
    y[J] = f < k ? y[J] / (double)(k - 1) : 0.0;
    bad = bad || !__builtin_isfinite(y[J]);
    if (q == 0) sw[f] = y[J];
  }
  bad = __builtin_amdgcn_ballot_w64(bad) != 0;
  if constexpr (NW > 1) {
    if (lane == 0) sred[w] = bad ? 1.0 : 0.0;
  }
  __syncthreads();
  if constexpr (NW > 1) bad = sred[0] + sred[1] + sred[2] + sred[3] != 0.0;
  if (bad) {
    if (tid == 0) p.status[a] = kStatusNonFinite;
    nan_transform(p, a);
    return;
  }
  if (tid == 0) p.status[a] = 0;
  if (p.w_out)
    for (int f = tid; f < k; f += 64 * NW) p.w_out[a * (long long)k + f] = sw[f];
  if (p.trans_out) {
    // trans(f, e) = S(e, f) + overline_w(f): f along the lanes
    double* tr = p.trans_out + a * (long long)k * k;
#pragma unroll
    for (int J = 0; J < CPW; ++J) {
      const int f = 16 * (w * CPW + J) + i16;
#pragma unroll
      for (int I = 0; I < TT; ++I)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int e = 16 * I + q + 4 * r;
          if (f < k && e < k) tr[(long long)e * k + f] = S[I][J][r] + y[J];
        }
    }
  }
  if (p.xb || p.xb32) {
    // the B operand of the update over the reflector block (consumed by now;
    // the last block's reflectors were staged before the barriers above); for
    // the FP32 state in FP32 (the update rounds it to FP32 anyway)
    float* const rf = reinterpret_cast<float*>(refl);
#pragma unroll
    for (int I = 0; I < TT; ++I)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double wf = sw[16 * I + q + 4 * r];
#pragma unroll
        for (int J = 0; J < CPW; ++J) {
          const double v = S[I][J][r] + wf;
          const int o = tile_off<KMAX>(I, w * CPW + J, r, lane);
          if (p.state_f32) rf[o] = (float)v;
          else refl[o] = v;
        }
      }
  }
}

hipError_t launch_sqrt(hipStream_t st, const EigParams& p, bool guard_pass) {
  const unsigned nb = (unsigned)p.n_an;
  if (guard_pass) {
    if (!p.guard) return hipSuccess;
    const unsigned n8 = (unsigned)((p.n_an + 7) / 8);
    if (p.k <= 32) hipLaunchKernelGGL(k_lmin<32>, dim3(n8), dim3(64), 0, st, p);
    else if (p.k <= 64) hipLaunchKernelGGL(k_lmin<64>, dim3(n8), dim3(64), 0, st, p);
    else hipLaunchKernelGGL(k_lmin<128>, dim3(n8), dim3(64), 0, st, p);
  } else {
    if (p.k <= 32) hipLaunchKernelGGL((k_vec<32, 1>), dim3(nb), dim3(64), 0, st, p);
    else if (p.k <= 64) hipLaunchKernelGGL((k_vec<64, 1>), dim3(nb), dim3(64), 0, st, p);
    else hipLaunchKernelGGL((k_vec<128, 4>), dim3(nb), dim3(256), 0, st, p);
  }
  return hipGetLastError();
}

}  // namespace dida
