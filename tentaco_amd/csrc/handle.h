// Device-resident CSF handle (the opaque tentaco_csf of the C ABI).
#pragma once

#include <mutex>
#include <vector>

#include "internal.h"
#include "kept.h"
#include "tuning.h"

namespace tt {
// The edge walk's wave starts of a handle, one table per run length (a power
// of two from 16 to 1024 nonzeros): they depend on the CSF alone. A table is
// complete when it is entered and stays until the handle is freed, so calls
// on any stream or thread, and captured graphs, may read it. Writing the
// brackets on every call took 11-16 us of serial searches and left each wave
// a search of its own (1.5M nonzeros, 5-mode, rank 16: 67 us a call, 47 us
// with the table).
struct WalkStarts {
  // The shared rows of edge-parallel tiles of nb nonzeros per workgroup at one
  // rank. A call adds to them, so each waits for the one before on whatever
  // stream (`used`, recorded behind every call, both under mu); a call under
  // capture, whose replays no one orders, does without them.
  struct Tile {
    int64_t nb = 0;
    int rank = 0;
    bool operator==(const Tile& o) const { return nb == o.nb && rank == o.rank; }
  };
  struct Shared {
    void* mem = nullptr;
    hipEvent_t used = nullptr;
    WalkTables t;
  };
  std::mutex mu;
  Kept<int64_t, int32_t*> starts{8};  // (there are 7 run lengths: none goes while in use)
  Kept<Tile, Shared> shared{8};       // (no graph holds them)
  uint32_t* bits = nullptr;
};
}  // namespace tt

struct tentaco_csf {
  int order = 0;
  int32_t dims[tt::kMaxOrder] = {};
  int32_t nodes[tt::kMaxOrder] = {};
  int32_t max_crd[tt::kMaxOrder] = {};  // largest coordinate per level, -1 if none
  bool dense_root = false;
  int32_t* d_crd0 = nullptr;
  int32_t* d_pos[tt::kMaxOrder] = {};
  int32_t* d_crd[tt::kMaxOrder] = {};
  float* d_vals = nullptr;
  void* ws = nullptr;
  size_t ws_bytes = 0;
  // workspaces replaced by a larger one; a graph captured earlier may still
  // use them, so they are freed with the handle, never before
  std::vector<void*> ws_retired;
  tt::WalkStarts starts;
  // workspace reserved by the caller (or for one host call): later calls
  // allocate nothing, so they write brackets where no start table exists
  bool reserved = false;
  tt::TuneTable tune;  // per-rank best variant found by the autotuner
  tt::CsfStats stats;
  // device buffers of the stream-ordered host-pointer path (factors of
  // levels 1..order-1 and the output), grown on demand
  float* stage_f[tt::kMaxOrder] = {};
  size_t stage_f_cap[tt::kMaxOrder] = {};
  float* stage_a = nullptr;
  size_t stage_a_cap = 0;
  // 3-mode expansion for the short-fibre slice path (built on first use)
  int32_t* d_crd1_of_nnz = nullptr;
  int32_t* d_nnz_of_root = nullptr;
  uint2* d_pad = nullptr;  // padded slice layout (short-fibre 3-mode tensors)
  int32_t pad_width = 0;
  uint2* d_pair = nullptr;     // paired slice layout (slices of at most 256 nonzeros)
  int4* d_pair_info = nullptr;
  int32_t npairs = 0;
  std::vector<int32_t> host_pairs;  // the pairing from host validation (2 per pair)
  // fibre-start bitmap and unit table of the TTV unit kernel (built on the
  // first TTV call outside stream capture)
  tt::TtvPlan ttv;
  int ttv_bands = 0;  // banded TTV layout: 0 picks, 1 one window, n >= 2 n bands
  // transposed index per level 1..order-1 (built on the first MTTKRP of
  // that level outside stream capture, or by tentaco_csf_reserve_level)
  tt::LevelIndex lvl[tt::kMaxOrder];
  tentaco_mlp* selector = nullptr;  // learned selector for AUTO (not owned)
  float min_margin = 0.03f;         // below it AUTO times candidates instead
  int fallback_k = 4;               // time the k best-predicted variants; 0: the full sweep

  tt::CsfDev view() const {
    tt::CsfDev v;
    v.order = order;
    v.nnz = nodes[order - 1];
    for (int m = 0; m < order; ++m) v.nodes[m] = nodes[m];
    v.crd0 = d_crd0;
    for (int m = 1; m < order; ++m) {
      v.pos[m] = d_pos[m];
      v.crd[m] = d_crd[m];
    }
    v.vals = d_vals;
    v.crd1_of_nnz = d_crd1_of_nnz;
    v.nnz_of_root = d_nnz_of_root;
    v.pad = d_pad;
    v.pad_width = pad_width;
    v.pair = d_pair;
    v.pair_info = d_pair_info;
    v.npairs = npairs;
    return v;
  }
};

namespace tt {
// The 24 selector features of a handle at rank R.
int csf_features(const tentaco_csf* h, int R, float* features);
// The selector's pick for an order-`order` tensor at rank R (variants that do
// not fit are skipped); margin = predicted time of the runner-up / best - 1.
int mlp_select(tentaco_mlp* m, int order, int R, const float* features, int* variant,
               float* margin, float* pred_ms);
}  // namespace tt
