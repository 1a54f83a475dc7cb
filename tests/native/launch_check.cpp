// The transform's launchers report a failed launch.  The launch calls and
// hipGetLastError are replaced here, so no kernel runs and no GPU is needed:
// each launch of a call fails in turn, and the call has to return its error.
#include <cstdio>

#include "letkf_kernels.h"

static int g_launch, g_fail;
static hipError_t g_last;

extern "C" hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) {
  return hipSuccess;
}
extern "C" hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds,
                                                hipStream_t* st) {
  *grid = *block = dim3(1);
  *lds = 0;
  *st = nullptr;
  return hipSuccess;
}
extern "C" hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
  if (++g_launch != g_fail) return hipSuccess;
  return g_last = hipErrorLaunchFailure;
}
extern "C" hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}

static hipError_t call(const dida::EigParams& p, bool rerun, int fail) {
  g_launch = 0;
  g_fail = fail;
  g_last = hipSuccess;
  return rerun ? dida::launch_eig_rerun(nullptr, p) : dida::launch_eig(nullptr, p, nullptr);
}

int main() {
  int bad = 0, calls = 0;
  const double x = 0.0;
  const int list = 0;
  for (int k : {20, 40, 100})
    for (int guard : {0, 1})
      for (int ql : {0, 1})
        for (int state : {0, 1})
          for (int rerun = 0; rerun <= ql; ++rerun) {
            dida::EigParams p{};
            p.k = k;
            p.kp = k <= 32 ? 32 : k <= 64 ? 64 : 128;
            p.n_an = 3;
            p.inflation = 1.0;
            p.guard = guard;
            p.ql_first = ql;
            p.xb = state ? &x : nullptr;
            p.list = rerun ? &list : nullptr;
            p.list_cap = rerun;
            const hipError_t e = call(p, rerun, 0);
            const int n = g_launch;
            if (e != hipSuccess || n < 2) {
              std::printf("k %d: %d launches, %s\n", k, n, hipGetErrorString(e));
              return 1;
            }
            for (int fail = 1; fail <= n; ++fail, ++calls)
              if (call(p, rerun, fail) != hipErrorLaunchFailure) {
                std::printf("k %d guard %d ql_first %d state %d rerun %d: launch %d of %d failed, "
                            "the call did not\n", k, guard, ql, state, rerun, fail, n);
                ++bad;
              }
          }
  std::printf(bad ? "%d of %d calls lost an error\n" : "launch_check ok\n", bad, calls);
  return bad != 0;
}
