// fr_ctx.h -- the library context behind the opaque fr_ctx handle.
#pragma once
#include <map>
#include <tuple>
#include <utility>
#include <vector>

#include "fr_ccp.h"
#include "fr_common.h"
#include "fr_kernels.h"

struct fr_ctx : public fr::Ctx {
  std::vector<fr::InsertTask> host_tasks;
  static constexpr int kSlots = 36;
  void* slots[kSlots] = {};
  size_t slot_bytes[kSlots] = {};
  void* slot(int k, size_t bytes, int* err);
  // grow-only pinned host staging (one buffer), for the small per-round
  // transfers of the lock-stepped minimisations
  void* hpin = nullptr;
  size_t hpin_bytes = 0;
  void* host_pinned(size_t bytes, int* err);
  // the index checks' results, one record per workgroup, in host memory
  static constexpr int kRangeBlocks = 64;
  int4* hrange = nullptr;
  int index_range(long long n, const int* d_idx, const float* d_amag, int* lo, int* hi,
                  fr::AmagMix* mix);
  // search annulus and shift-phase tables, cached per (NSAM, MAXR1, MAXR2)
  int skey[3] = {0, 0, 0};
  int kc = 0, kpad = 0, nsamr = 0;
  int* d_kidx = nullptr;
  float* d_shx = nullptr;
  float* d_shy = nullptr;
  // constant tables of the fused CC3M, built on first use and kept until the
  // context is destroyed (captured graphs hold their addresses)
  std::map<int, float*> dft_tabs;                        // per NSAM
  std::map<std::pair<int, int>, int*> pts_tabs;          // per (MAXR1^2, MAXR2^2)
  struct RingTab {
    float* d = nullptr;
    int cnt = 0;
  };
  std::map<std::tuple<int, float, float>, RingTab> ring_tabs;  // per (NSAM, RI2, RI3)
  int cc3m_tables(const fr::Cc3mArgs& a, fr::Cc3mTables* t);
  std::map<std::pair<int, int>, float*> band_dft_tabs;         // per (M, frequencies held)
  std::map<std::pair<int, int>, int*> band_pair_tabs;          // per (MAXR1^2, MAXR2^2)
  // per (NSAM, M, RI2, RI3, RIH, HALFW)
  std::map<std::tuple<int, int, float, float, float, float>, float*> band_wmap_tabs;
  struct RingHat {
    void* buf;
    fr::Cc3mRing ring;
  };
  std::map<std::tuple<int, int, float, float>, RingHat> ring_hats;  // per (NSAM, MAXR2, RI2, RI3)
  int cc3m_ring(int nsam, int maxr2, float ri2, float ri3, fr::Cc3mRing* t);
  int cc3m_band_tables(const fr::Cc3mArgs& a, fr::Cc3mBandTables* t);
  // a second stream, for the part of a batch that other kernels take than the rest.
  // side_open orders it after what the context's stream holds; who uses it waits for
  // it on the host before returning.
  hipStream_t side = nullptr;
  hipEvent_t side_fork = nullptr;
  int side_open();
  // launch choices per box size (set by fr_autotune_cc3m)
  struct Tune {
    int cc3m_fused = 1;   // band-pruned fused CC3M where it applies
    int cc3m_blocks = -1;  // persistent workgroups (0: one per item; -1: one full wave)
  };
  std::map<int, Tune> tune;
  Tune tune_for(int nsam) const;
  // constant tables of the exact CCP search, per (NSAM, MAXR2), kept until
  // the context is destroyed
  std::map<std::pair<int, int>, fr::CcpTablesDev> ccp_tabs;
  int ccp_tables(int nsam, int maxr2, fr::CcpTablesDev* t);
};

namespace fr {
// fr_cc3m_batch (cc3 = 0) and fr_cc3_batch (cc3 = 1).  mix: what the caller knows of
// the items' AMAG (it saves launches; an item's path does not depend on it)
int cc3m_batch(fr_ctx* c, int nsam, int n, const float* d_a3df, const float* d_spec,
               const float* d_ctff, const int* d_pidx, const float* d_dm, const float* d_shift,
               const float* d_amag, int maxr1, int maxr2, float rbfact, const float* d_fsct,
               const float* ring, float* d_score, int cc3, fr::AmagMix mix = {});
// fr_refine_batch with the symmetry matrix SM applied to every DM (null: identity)
int refine_items(fr_ctx* c, int nsam, int n, const float* d_a3df, const float* d_spec,
                 const float* d_ctff, const int* pidx, const float* amag, float* par,
                 const int* mask, int maxr1, int maxr2, float rbfact, const float* d_fsct,
                 const float* ring, const float* prior, int maxit, const float* sm,
                 int* nevals);
}  // namespace fr
