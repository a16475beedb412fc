// Test-only entry points (not part of the C ABI): what the planner shared
// among workgroups, and one step of the GMRES orthogonalisation.
#include <hip/hip_runtime.h>

#include <vector>

#include "nnk_handles.hpp"
#include "nnk_mobility.hpp"

using namespace nnk;

extern "C" void nnk_selftest_shared(nnk_fmm *h, int *leaves, int *x_lists) {
  *leaves = h->f->shared_leaves();
  *x_lists = h->f->shared_x_lists();
}

// w (n) against the k vectors of V (n each): w and y in place, hc the 2 m1 + 1
// coefficients and norm
extern "C" int nnk_selftest_cgs2(int64_t n, int k, int m1, const double *V, double *w, double *y, double *hc) {
  try {
    DBuf dV, dw, dy, dh, part;
    dV.upload(std::vector<double>(V, V + (size_t)n * k));
    dw.upload(std::vector<double>(w, w + n));
    dy.upload(std::vector<double>(y, y + n));
    dh.upload(std::vector<double>(hc, hc + 2 * (size_t)m1 + 1));
    part.alloc(sizeof(double) * Mobility::cgs2_part(m1));
    Mobility::cgs2(n, dV.as<double>(), k, dw.as<double>(), dy.as<double>(), dh.as<double>(), m1, part.as<double>(), 0);
    NNK_HIP(hipDeviceSynchronize());
    NNK_HIP(hipMemcpy(w, dw.p, sizeof(double) * n, hipMemcpyDeviceToHost));
    NNK_HIP(hipMemcpy(y, dy.p, sizeof(double) * n, hipMemcpyDeviceToHost));
    NNK_HIP(hipMemcpy(hc, dh.p, sizeof(double) * (2 * (size_t)m1 + 1), hipMemcpyDeviceToHost));
    return 0;
  } catch (...) {
    return 1;
  }
}
