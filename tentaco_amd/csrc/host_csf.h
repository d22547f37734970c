// Owned host-side CSF (builder / generator output) with a taco_tensor_t view.
#pragma once

#include <cstdint>
#include <functional>
#include <vector>

#include "../../include/taco_tensor_t.h"
#include "tuning.h"

namespace tt {

// What validation learns about a host CSF: dimensions, node count and
// largest coordinate per level (-1 for an empty level), whether the root is
// dense (crd0 = 0..dims0-1), and the selector's structure statistics.
struct CsfCheck {
  int32_t dims[kMaxOrder] = {};
  int32_t nodes[kMaxOrder] = {};
  int32_t max_crd[kMaxOrder] = {};
  bool dense_root = false;
  CsfStats stats;
  // 3-mode CSFs whose root nodes hold at most kPairCap nonzeros: root nodes
  // in pairs for the paired slice layout (first, second or -1), the largest
  // with the smallest that fits kPairCap slots together, else alone
  std::vector<int32_t> pairs;
};
constexpr int64_t kPairCap = 256;
// The pairing above from the nonzero count of every root node.
void pair_slices(const std::vector<int32_t>& counts, int64_t cap, std::vector<int32_t>* pairs);
// Validate B as an order-`order` CSF (the device API's operand contract);
// TENTACO_OK or an error code with tentaco_last_error() set. `put(m, parents,
// nodes)`, if given, is called for each level m >= 1 once its arrays may be
// read (pos checked, crd present) and may copy them while the check of a long
// crd array still runs on other threads; an error of its own is returned only
// for a B without faults.
using LevelFn = std::function<int(int, int64_t, int64_t)>;
int validate_csf(const taco_tensor_t* B, int order, CsfCheck* out, const LevelFn& put = {});

struct HostCsf {
  int order = 0;
  std::vector<int32_t> dims;
  std::vector<std::vector<int32_t>> pos, crd;  // level 0 = {0, dims0} / 0..dims0-1
  std::vector<float> vals;

  taco_tensor_t view{};
  std::vector<int32_t> dims_i32;
  std::vector<int32_t*> idx_ptrs;
  std::vector<int32_t**> lvl_ptrs;
  void make_view();
};

// Lexicographic COO -> CSF (dense root); coords mode-major, duplicates summed
// in input order. Inputs must already be validated (coords inside dims).
int build_csf_from_coo(int order, const int32_t* dims, int64_t n, const int32_t* coords,
                       const float* vals, HostCsf* out);

}  // namespace tt

struct tentaco_host_csf {
  tt::HostCsf h;
};
