// Test-only entry points of the frequency-space M2L (part of
// libnnk_selftest.so): its host planner on given gather tables (no GPU
// call) and the transforms and products on given densities.
#include <hip/hip_runtime.h>

#include <cstring>
#include <vector>

#include "nnk_fmm.hpp"

using namespace nnk;

namespace {

SpecLevel plan(const int32_t *ncls, const int32_t *cls, const int32_t *gv, int32_t count, const int32_t *parent,
               const int32_t *child0, const uint8_t *has_src) {
  std::vector<int32_t> c[8], g[8];
  for (int a = 0; a < 8; a++) {
    c[a].assign(cls, cls + ncls[a]);
    cls += ncls[a];
    g[a].assign(gv, gv + 189 * (size_t)ncls[a]);
    gv += 189 * (size_t)ncls[a];
  }
  SpecLevel L;
  plan_spectral_level(c, g, std::vector<int32_t>(parent, parent + count), std::vector<int32_t>(child0, child0 + count),
                      std::vector<uint8_t>(has_src, has_src + count + 1), L);
  return L;
}

}  // namespace

// sizes: ok, target parents, source parents; pairs; and the tables (sized
// by the caller for count parents)
extern "C" int nnk_selftest_spectral_plan(const int32_t *ncls, const int32_t *cls, const int32_t *gv, int32_t count,
                                          const int32_t *parent, const int32_t *child0, const uint8_t *has_src,
                                          int32_t *sizes, int64_t *pairs, int32_t *tgt0, int32_t *tmask, int32_t *src0,
                                          int32_t *smask, int32_t *nb) {
  try {
    const SpecLevel L = plan(ncls, cls, gv, count, parent, child0, has_src);
    sizes[0] = L.ok;
    sizes[1] = (int32_t)L.tgt0.size();
    sizes[2] = (int32_t)L.src0.size();
    pairs[0] = L.pairs;
    pairs[1] = L.tile_dirs;
    if (!L.ok) return 0;
    std::copy(L.tgt0.begin(), L.tgt0.end(), tgt0);
    std::copy(L.tmask.begin(), L.tmask.end(), tmask);
    std::copy(L.src0.begin(), L.src0.end(), src0);
    std::copy(L.smask.begin(), L.smask.end(), smask);
    std::copy(L.nb.begin(), L.nb.end(), nb);
    return 0;
  } catch (...) {
    return 1;
  }
}

// chk (count x K, in: untouched rows keep their values) from up (count x K);
// the level is entered twice (levels = 2: the second copy on other operators
// of box width 2 w, whose rows follow the first's at count * K)
extern "C" int nnk_selftest_spectral_run(const int32_t *ncls, const int32_t *cls, const int32_t *gv, int32_t count,
                                         const int32_t *parent, const int32_t *child0, const uint8_t *has_src, int res,
                                         const int32_t *codes, int nq, double w, double eps, double mu, int levels,
                                         int64_t buf_bytes, const double *up, double *chk) {
  try {
    SpecLevel L = plan(ncls, cls, gv, count, parent, child0, has_src);
    if (!L.ok) return 2;
    SpectralM2L M(res, std::vector<int32_t>(codes, codes + nq), 3 * nq);
    for (int l = 0; l < levels; l++) {
      auto ops = std::make_shared<SpecOps>();
      spectral_ops(res, (l + 1) * w, eps, mu, *ops);
      M.add(L, ops);
      for (auto &v : L.tgt0) v += count;
      for (auto &v : L.src0) v += count;
    }
    M.finish((size_t)buf_bytes);
    const size_t n = (size_t)levels * count * 3 * nq;
    DBuf u, c;
    u.upload(std::vector<double>(up, up + n));
    c.upload(std::vector<double>(chk, chk + n));
    M.run(u.as<double>(), c.as<double>(), 0);
    NNK_HIP(hipDeviceSynchronize());
    NNK_HIP(hipMemcpy(chk, c.p, sizeof(double) * n, hipMemcpyDeviceToHost));
    return 0;
  } catch (...) {
    return 1;
  }
}
