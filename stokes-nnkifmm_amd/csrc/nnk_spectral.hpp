// M2L of the FP64 forms in frequency space (csrc/nnk_spectral.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <memory>
#include <vector>

#include "nnk_common.hpp"

namespace nnk {

// surface resolutions (points per edge) with compiled transforms; others
// keep the dense translations
constexpr int kSpecMinRes = 3, kSpecMaxRes = 10;
inline bool spectral_res(int res) { return res >= kSpecMinRes && res <= kSpecMaxRes; }
// unique frequencies of the real (2 res - 1)^3 transform
inline int spectral_freqs(int res) { return ((2 * res - 1) * (2 * res - 1) * (2 * res - 1) + 1) / 2; }

// One level's V-list interactions by parent: children of target parent t
// (node slots tgt0[t] .. +7, those in tmask[t] wanted) see the children of
// the source parents nb[d * nt + t] (-1 none; d counts the 26 neighbour
// directions in (dx, dy, dz) order, z fastest, without the parent itself).
// src0/smask: first child slot of each source parent and the children that
// carry an up density.
struct SpecLevel {
  int level = 0;
  bool ok = false;           // the V lists are exactly the parents' product sets
  std::vector<int32_t> tgt0, tmask, src0, smask;
  std::vector<int32_t> nb;   // 26 x nt, source parent index or -1
  int64_t pairs = 0;         // V-list pairs covered
  int64_t tile_dirs = 0;     // (16-parent tile, active direction) products
};

// Regroups a level's V lists by parent: cls[a] (slots of the level's target
// nodes of child class a), gv[a] (189 x |cls[a]| source slots, -1 none, in
// class_offset_slots order), parent[] (1-based ids by slot), child0[] (first
// child slot by parent slot).  ok = false where the lists are not what the
// parents' neighbourhoods imply (then the dense translations stay).
void plan_spectral_level(const std::vector<int32_t> *cls, const std::vector<int32_t> *gv,
                         const std::vector<int32_t> &parent, const std::vector<int32_t> &child0,
                         const std::vector<uint8_t> &has_src, SpecLevel &out);

// the translation operators of one level in frequency space:
// [frequency][7^3 offset slot][xx xy xz yy yz zz][re im]; read-only once
// built (shared through the operator cache)
struct SpecOps {
  DBuf tab;
  size_t bytes() const { return tab.bytes; }
};
void spectral_ops(int res, double w, double eps, double mu, SpecOps &out);

// All spectral levels of one tree: forward transforms of the source nodes'
// up densities, one complex product per frequency, inverse transforms into
// the target nodes' check potentials.
class SpectralM2L {
 public:
  // surface codes ix | iy << 8 | iz << 16 of the nq surface points
  SpectralM2L(int res, const std::vector<int32_t> &codes, int K);
  void add(const SpecLevel &L, std::shared_ptr<const SpecOps> ops);
  // uploads the tables and reserves the workspace, at most buf_bytes (or
  // one kx plane of the transforms, if that is more)
  void finish(size_t buf_bytes = (size_t)4 << 30);
  bool empty() const { return nt_ == 0; }
  // chk[target node] = sum over its V list of T uppot[source node]
  void run(const double *uppot, double *chk, hipStream_t s) const;

 private:
  int res_, K_;
  int nt_ = 0, ns_ = 0;
  std::vector<std::shared_ptr<const SpecOps>> ops_;
  std::vector<int32_t> h_tgt0_, h_tmask_, h_src0_, h_smask_;
  std::vector<std::vector<int32_t>> h_nb_;   // per level
  std::vector<int> lev_t0_, lev_nt_, lev_s0_;
  std::vector<int32_t> h_qmap_;
  DBuf qmap_, tw_, tgt0_, tmask_, src0_, smask_, nb_, tiles_, tab_;
  DBuf X_, Y_;
  int ntiles_ = 0, kx_step_ = 0;
  bool split_ = false;       // the four wavefronts of a tile split its directions
};

}  // namespace nnk
