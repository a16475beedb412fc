// Test-only entry point (not part of the C ABI): the direct gather GEMM of
// the FP64 form (M2M, L2L, solves), as the library launches it.
#include <hip/hip_runtime.h>

#include <vector>

#include "nnk_gemm.hpp"
#include "nnk_handles.hpp"

using namespace nnk;

// njobs jobs of N[j] columns over the same nb operators (at[nb][Kpad][Mpad]);
// gidx: the jobs' nb x N[j] tables one after the other, cidx likewise (null:
// none)
extern "C" int nnk_selftest_gemm_direct(int M, int K, int Mpad, int Kpad, const double *at, int nb, const double *x,
                                        int nx, int ldx, const int *gidx, const int *cidx, const int *N, int njobs,
                                        double *c, int nc, int ldc, int beta, int ordered) {
  try {
    const size_t mat = (size_t)Kpad * Mpad;
    DBuf dA, dX, dC, dP, dJ;
    dA.upload(std::vector<double>(at, at + mat * nb));
    dX.upload(std::vector<double>(x, x + (size_t)nx * ldx));
    dC.upload(std::vector<double>(c, c + (size_t)nc * ldc));
    std::vector<const double *> ptrs(nb);
    for (int b = 0; b < nb; b++) ptrs[b] = dA.as<double>() + b * mat;
    dP.upload(ptrs);
    std::vector<DBuf> own(2 * njobs);
    std::vector<GemmJob> jobs(njobs);
    int maxN = 0;
    for (int j = 0; j < njobs; j++) {
      GemmJob &J = jobs[j];
      J.A = dP.as<const double *>();
      J.gidx = J.cidx = nullptr;
      if (gidx) {
        own[2 * j].upload(std::vector<int>(gidx, gidx + (size_t)nb * N[j]));
        J.gidx = own[2 * j].as<int32_t>();
        gidx += (size_t)nb * N[j];
      }
      if (cidx) {
        own[2 * j + 1].upload(std::vector<int>(cidx, cidx + N[j]));
        J.cidx = own[2 * j + 1].as<int32_t>();
        cidx += N[j];
      }
      J.nb = nb;
      J.N = N[j];
      maxN = std::max(maxN, N[j]);
    }
    dJ.upload(jobs);
    if (!ordered)
      launch_gemm_direct(M, K, Mpad, Kpad, dX.as<double>(), ldx, dC.as<double>(), ldc, beta, dJ.as<GemmJob>(), njobs,
                         maxN, 0);
    else if (ordered == 1) {
      if (!launch_gemm_ordered(M, K, Mpad, Kpad, dX.as<double>(), ldx, dC.as<double>(), ldc, beta, dJ.as<GemmJob>(),
                               njobs, maxN, 0))
        return 2;
    } else   // the kernel whose order it has
      hipLaunchKernelGGL((k_gemm_gather<GBM, GBN0, GBK, 0>), dim3(njobs * (Mpad / GBM) * ((maxN + GBN0 - 1) / GBN0)),
                         dim3(256), 0, 0, M, K, Mpad, Kpad, dX.as<double>(), ldx, dC.as<double>(), ldc, beta,
                         dJ.as<GemmJob>(), njobs, Mpad / GBM, 1, nullptr, maxN);
    NNK_HIP(hipDeviceSynchronize());
    NNK_HIP(hipMemcpy(c, dC.p, sizeof(double) * (size_t)nc * ldc, hipMemcpyDeviceToHost));
    return 0;
  } catch (...) {
    return 1;
  }
}
