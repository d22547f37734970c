// Batched MTTKRP over many (tensor, mode) tasks in one persistent launch, its
// hipGraph capture and its tile autotuner. The per-task alternative is one
// tentaco_mttkrp_dev call per task.

#include <algorithm>
#include <cstring>
#include <vector>

#include "handle.h"
#include "internal.h"

struct tentaco_batch {
  int ntasks = 0;
  int R = 0;
  std::vector<tentaco_csf*> tasks;  // sorted by order (stable)
  std::vector<int> perm;            // sorted position -> the caller's task index
  std::vector<tt::BatchTaskDev> host_tasks;  // sorted positions
  bool have_operands = false;
  // device tables
  tt::BatchTaskDev* d_tasks = nullptr;
  int64_t* d_fill_off = nullptr;
  int64_t* d_bnd_off = nullptr;
  int64_t* d_item_off = nullptr;
  uint32_t* d_rowbits = nullptr;  // per task, one bit per output row
  int32_t* d_counter = nullptr;
  int32_t* d_starts = nullptr;
  float4** d_bnd_rows = nullptr;  // the rows of slices that items share
  double* d_bnd_w = nullptr;      // and their sums
  int2* d_slots = nullptr;
  tt::BatchLaunch L;
  std::vector<int64_t> h_fill, h_bnd;  // host prefix tables (ntasks + 1)
  // streams and events of the concurrent order launches
  hipStream_t conc[tt::kMaxOrder + 1] = {};
  hipEvent_t cev[tt::kMaxOrder + 1] = {};
  // graph
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
};

namespace tt {
namespace {

template <class T>
int dev_alloc(T** p, size_t n) {
  *p = nullptr;
  if (hipMalloc(reinterpret_cast<void**>(p), std::max<size_t>(n, 1) * sizeof(T)) != hipSuccess) {
    *p = nullptr;
    return fail(TENTACO_ENOMEM, "batch table allocation failed");
  }
  return TENTACO_OK;
}

void drop_graph(tentaco_batch* b) {
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  b->exec = nullptr;
  b->graph = nullptr;
}

void free_tables(tentaco_batch* b) {
  (void)hipFree(b->d_tasks);
  (void)hipFree(b->d_bnd_off);
  (void)hipFree(b->d_item_off);
  (void)hipFree(b->d_starts);
  (void)hipFree(b->d_bnd_rows);
  (void)hipFree(b->d_bnd_w);
  (void)hipFree(b->d_slots);
  b->d_tasks = nullptr;
  b->d_bnd_off = b->d_item_off = nullptr;
  b->d_starts = nullptr;
  b->d_bnd_rows = nullptr;
  b->d_bnd_w = nullptr;
  b->d_slots = nullptr;
}

// The batch runs the edge-parallel walk only: its block-level combine keeps
// the FP32 atomics per output row few. The edge-serial walk adds one atomic
// per lane group, and on giant slices that exceeded 1e-5 relative L2.
int check_tile(int family, int block, int group) {
  if (family == kEdgeSerial)
    return fail(TENTACO_EUNSUPPORTED,
                "the batch runs the edge-parallel walk only (family 1); edge-serial tiles are "
                "per-tensor (tentaco_mttkrp_dev), where rows accumulate in FP64");
  if (family != kEdgeParallel) return fail(TENTACO_EINVAL, "batch family must be 1 (edge-parallel)");
  if (block != 128 && block != 256 && block != 512)
    return fail(TENTACO_EINVAL, "batch block %d not in {128,256,512}", block);
  if (group < 1 || group > 1024) return fail(TENTACO_EINVAL, "batch group %d", group);
  return TENTACO_OK;
}

// Rebuild the item/boundary/fill tables and the bracket workspace for the
// per-order tiles in b->L (a task's items use its order's nonzeros per item),
// and upload the task table.
int configure_tables(tentaco_batch* b) {
  if (!b->have_operands) return fail(TENTACO_EINVAL, "set operands before configuring");
  drop_graph(b);
  BatchLaunch& L = b->L;
  const int lpr = lanes_per_row(b->R);
  for (int N = 0; N <= kMaxOrder; ++N) L.nb[N] = int32_t((L.blk[N] / lpr) * L.grp[N]);
  std::vector<int64_t> bnd(b->ntasks + 1, 0), item(b->ntasks + 1, 0), start_off(b->ntasks + 1, 0);
  for (int t = 0; t < b->ntasks; ++t) {
    const tentaco_csf* h = b->tasks[t];
    const int64_t nnz = h->nodes[h->order - 1];
    const int64_t NB = L.nb[h->order];
    const int64_t nblk = (nnz + NB - 1) / NB;
    item[t + 1] = item[t] + nblk;
    bnd[t + 1] = bnd[t] + nblk + 1;
    start_off[t + 1] = start_off[t] + (nblk + 1) * (L.blk[h->order] / 64) * (h->order - 1);
  }
  if (item[b->ntasks] >= (int64_t(1) << 31))
    return fail(TENTACO_EUNSUPPORTED, "batch has too many work items");
  free_tables(b);
  int rc = dev_alloc(&b->d_tasks, size_t(b->ntasks));
  if (!rc) rc = dev_alloc(&b->d_bnd_off, size_t(b->ntasks));
  if (!rc) rc = dev_alloc(&b->d_item_off, size_t(b->ntasks) + 1);  // + the total
  if (!rc) rc = dev_alloc(&b->d_starts, size_t(start_off[b->ntasks]));
  if (!rc) rc = dev_alloc(&b->d_bnd_rows, size_t(bnd[b->ntasks]) * 2);
  const size_t wlen = size_t(bnd[b->ntasks]) * 2 * size_t(b->R);
  if (!rc) rc = dev_alloc(&b->d_bnd_w, wlen);
  if (!rc) rc = dev_alloc(&b->d_slots, size_t(item[b->ntasks]));
  if (rc) return rc;
  TT_HIP_CHECK(hipMemset(b->d_bnd_w, 0, sizeof(double) * wlen));
  for (int t = 0; t < b->ntasks; ++t) {
    BatchTaskDev& T = b->host_tasks[t];
    T.starts = b->d_starts + start_off[t];
    T.W = b->d_bnd_w + bnd[t] * 2 * b->R;
    T.slots = b->d_slots + item[t];
  }
  TT_HIP_CHECK(hipMemcpy(b->d_tasks, b->host_tasks.data(), sizeof(BatchTaskDev) * b->ntasks,
                         hipMemcpyHostToDevice));
  TT_HIP_CHECK(hipMemcpy(b->d_bnd_off, bnd.data(), sizeof(int64_t) * b->ntasks,
                         hipMemcpyHostToDevice));
  TT_HIP_CHECK(hipMemcpy(b->d_item_off, item.data(), sizeof(int64_t) * (b->ntasks + 1),
                         hipMemcpyHostToDevice));
  b->h_bnd = bnd;
  L.h_bnd_off = b->h_bnd.data();
  L.h_fill_off = b->h_fill.data();
  L.tasks = b->d_tasks;
  L.ntasks = b->ntasks;
  L.bnd_off = b->d_bnd_off;
  L.total_bnd = bnd[b->ntasks];
  L.bnd_rows = b->d_bnd_rows;
  L.bnd_w = b->d_bnd_w;
  L.item_off = b->d_item_off;
  L.total_items = int32_t(item[b->ntasks]);
  L.counter = b->d_counter;
  L.R = b->R;
  int dev = 0;
  TT_HIP_CHECK(hipGetDevice(&dev));
  hipDeviceProp_t prop;
  TT_HIP_CHECK(hipGetDeviceProperties(&prop, dev));
  // order groups of the sorted task table and a persistent grid per order
  L.grid = 0;
  for (int N = 0; N <= kMaxOrder + 1; ++N) {
    int s = 0;
    while (s < b->ntasks && b->tasks[s]->order < N) ++s;
    L.grp_task[N] = s;
    L.grp_item[N] = int32_t(item[s]);
  }
  for (int N = 2; N <= kMaxOrder; ++N) {
    L.grp_grid[N] = 0;
    if (L.grp_item[N + 1] <= L.grp_item[N]) continue;
    int per_cu = 1;
    rc = batch_occupancy(L.fam[N], L.blk[N], b->R, L.nb[N], N, &per_cu);
    if (rc) return rc;
    L.grp_grid[N] = std::max(1, per_cu) * prop.multiProcessorCount;
    L.grid = std::max(L.grid, L.grp_grid[N]);
  }
  int orders = 0, block = 0;
  bool one_block = true;
  for (int N = 2; N <= kMaxOrder; ++N) {
    if (L.grp_task[N + 1] <= L.grp_task[N]) continue;
    one_block = one_block && (orders == 0 || L.blk[N] == block);
    block = L.blk[N];
    ++orders;
  }
  L.all_grid = 0;
  if (orders > 1 && one_block && L.total_items > 0) {
    int per_cu = 1;
    rc = batch_all_occupancy(block, b->R, &per_cu);
    if (rc) return rc;
    L.all_grid = std::max(1, per_cu) * prop.multiProcessorCount;
    L.grid = L.all_grid;
  }
  // the brackets depend on the CSFs and the tiles only: written once here,
  // read by every launch
  rc = launch_batch_brackets(L, nullptr);
  if (rc) return rc;
  TT_HIP_CHECK(hipDeviceSynchronize());
  return TENTACO_OK;
}

// The one-time fill of the retained output mode (synchronous).
int zero_retained_outputs(tentaco_batch* b) {
  if (!b->have_operands || !b->L.retain) return TENTACO_OK;
  int rc = launch_batch_zero_outputs(b->L, nullptr);
  if (rc) return rc;
  TT_HIP_CHECK(hipDeviceSynchronize());
  return TENTACO_OK;
}

void set_tile(tentaco_batch* b, int order, int family, int block, int group) {
  b->L.fam[order] = family;
  b->L.blk[order] = block;
  b->L.grp[order] = group;
}

// The order group with the most items (the one whose settings the
// single-valued queries report).
int main_order(const BatchLaunch& L) {
  int best = kMaxOrder, most = -1;
  for (int N = 2; N <= kMaxOrder; ++N) {
    const int32_t n = L.grp_item[N + 1] - L.grp_item[N];
    if (n > most) {
      most = n;
      best = N;
    }
  }
  return best;
}

}  // namespace
}  // namespace tt

using namespace tt;

extern "C" {

int tentaco_batch_create(tentaco_csf* const* tasks, int ntasks, int R, tentaco_batch** out) {
  clear_error();
  if (!out || !tasks || ntasks <= 0) return fail(TENTACO_EINVAL, "empty batch");
  *out = nullptr;
  if (R != 16 && R != 32 && R != 64)
    return fail(TENTACO_EUNSUPPORTED, "batched launch supports R in {16,32,64}");
  for (int t = 0; t < ntasks; ++t)
    if (!tasks[t]) return fail(TENTACO_EINVAL, "task %d handle is NULL", t);
  auto* b = new tentaco_batch;
  b->ntasks = ntasks;
  b->R = R;
  b->perm.resize(size_t(ntasks));
  for (int t = 0; t < ntasks; ++t) b->perm[size_t(t)] = t;
  std::stable_sort(b->perm.begin(), b->perm.end(),
                   [&](int x, int y) { return tasks[x]->order < tasks[y]->order; });
  for (int t = 0; t < ntasks; ++t) b->tasks.push_back(tasks[b->perm[size_t(t)]]);
  b->host_tasks.resize(size_t(ntasks));
  if (hipMalloc(&b->d_counter, sizeof(int32_t) * (kMaxOrder + 1)) != hipSuccess) {
    delete b;
    return fail(TENTACO_ENOMEM, "counter allocation failed");
  }
  // the streams of the concurrent order launches (default priority), where
  // there are several; without them the orders run one after another
  bool ok = b->tasks.front()->order != b->tasks.back()->order;
  for (int k = 0; k <= kMaxOrder && ok; ++k)
    ok = hipStreamCreateWithFlags(&b->conc[k], hipStreamNonBlocking) == hipSuccess &&
         hipEventCreateWithFlags(&b->cev[k], hipEventDisableTiming) == hipSuccess;
  for (int k = 0; k <= kMaxOrder && ok; ++k) {
    b->L.conc[k] = b->conc[k];
    b->L.cev[k] = b->cev[k];
  }
  *out = b;
  return TENTACO_OK;
}

int tentaco_batch_set_operands(tentaco_batch* b, const float* const* factors_dev,
                               float* const* outs_dev, const int32_t* out_rows) {
  clear_error();
  if (!b || !factors_dev || !outs_dev || !out_rows) return fail(TENTACO_EINVAL, "NULL argument");
  std::vector<int64_t> fill(b->ntasks + 1, 0);
  for (int s = 0; s < b->ntasks; ++s) {
    const int t = b->perm[size_t(s)];  // the caller's index of sorted position s
    const tentaco_csf* h = b->tasks[s];
    if (out_rows[t] <= h->max_crd[0])
      return fail(TENTACO_EINVAL, "task %d output has %d rows, root coordinates reach %d", t,
                  out_rows[t], h->max_crd[0]);
    if (!outs_dev[t]) return fail(TENTACO_EINVAL, "task %d output is NULL", t);
    if (reinterpret_cast<uintptr_t>(outs_dev[t]) & 15)
      return fail(TENTACO_EINVAL, "task %d output is not 16-byte aligned", t);
    BatchTaskDev& T = b->host_tasks[size_t(s)];
    T.B = h->view();
    for (int m = 1; m < h->order; ++m) {
      const float* f = factors_dev[size_t(t) * (kMaxOrder - 1) + (m - 1)];
      if (!f) return fail(TENTACO_EINVAL, "task %d factor of level %d is NULL", t, m);
      T.F.M[m] = f;
    }
    T.A = outs_dev[t];
    T.rows = out_rows[t];
    fill[s + 1] = fill[s] + int64_t(out_rows[t]) * b->R;
  }
  (void)hipFree(b->d_fill_off);
  b->d_fill_off = nullptr;
  (void)hipFree(b->d_rowbits);
  b->d_rowbits = nullptr;
  // the row bitmaps of every task (one 32-bit word per 32 rows), built once
  std::vector<int64_t> woff(b->ntasks + 1, 0);
  for (int s = 0; s < b->ntasks; ++s) woff[s + 1] = woff[s] + (b->host_tasks[s].rows + 31) / 32;
  int rc = dev_alloc(&b->d_fill_off, size_t(b->ntasks));
  if (!rc) rc = dev_alloc(&b->d_rowbits, size_t(woff[b->ntasks]));
  if (rc) return rc;
  TT_HIP_CHECK(hipMemset(b->d_rowbits, 0, sizeof(uint32_t) * std::max<int64_t>(woff[b->ntasks], 1)));
  for (int s = 0; s < b->ntasks; ++s) {
    b->host_tasks[s].rowbits = b->d_rowbits + woff[s];
    rc = launch_batch_rowbits(b->host_tasks[s].B, b->d_rowbits + woff[s], nullptr);
    if (rc) return rc;
  }
  TT_HIP_CHECK(hipDeviceSynchronize());
  TT_HIP_CHECK(hipMemcpy(b->d_fill_off, fill.data(), sizeof(int64_t) * b->ntasks,
                         hipMemcpyHostToDevice));
  b->L.fill_off = b->d_fill_off;
  b->L.total_fill = fill[b->ntasks];
  b->h_fill = fill;
  b->L.h_fill_off = b->h_fill.data();
  b->have_operands = true;
  if (b->L.blk[kMaxOrder] == 0) {  // never configured
    int64_t nnz = 0;
    for (const tentaco_csf* h : b->tasks) nnz += h->nodes[h->order - 1];
    const int group = batch_group(nnz, b->R);
    for (int N = 0; N <= kMaxOrder; ++N) set_tile(b, N, kEdgeParallel, 256, group);
  }
  rc = configure_tables(b);
  if (rc) return rc;
  return zero_retained_outputs(b);
}

int tentaco_batch_set_output_mode(tentaco_batch* b, int mode) {
  clear_error();
  if (!b) return fail(TENTACO_EINVAL, "batch is NULL");
  if (mode != TENTACO_BATCH_OUTPUTS_WRITTEN && mode != TENTACO_BATCH_OUTPUTS_RETAINED)
    return fail(TENTACO_EINVAL, "output mode %d", mode);
  drop_graph(b);
  b->L.retain = mode == TENTACO_BATCH_OUTPUTS_RETAINED ? 1 : 0;
  return zero_retained_outputs(b);
}

int tentaco_batch_get_output_mode(const tentaco_batch* b, int* mode) {
  if (!b || !mode) return fail(TENTACO_EINVAL, "NULL argument");
  *mode = b->L.retain ? TENTACO_BATCH_OUTPUTS_RETAINED : TENTACO_BATCH_OUTPUTS_WRITTEN;
  return TENTACO_OK;
}

int tentaco_batch_configure(tentaco_batch* b, int family, int block, int group) {
  clear_error();
  if (!b) return fail(TENTACO_EINVAL, "batch is NULL");
  int rc = check_tile(family, block, group);
  if (rc) return rc;
  if (!b->have_operands) return fail(TENTACO_EINVAL, "set operands before configuring");
  for (int N = 0; N <= kMaxOrder; ++N) set_tile(b, N, family, block, group);
  return configure_tables(b);
}

int tentaco_batch_configure_order(tentaco_batch* b, int order, int family, int block, int group,
                                  int schedule) {
  clear_error();
  if (!b) return fail(TENTACO_EINVAL, "batch is NULL");
  if (order < 2 || order > kMaxOrder)
    return fail(TENTACO_EINVAL, "order %d outside 2..%d", order, kMaxOrder);
  int rc = check_tile(family, block, group);
  if (rc) return rc;
  if (schedule != 0 && schedule != 1) return fail(TENTACO_EINVAL, "schedule must be 0 or 1");
  if (!b->have_operands) return fail(TENTACO_EINVAL, "set operands before configuring");
  set_tile(b, order, family, block, group);
  b->L.sch[order] = schedule;
  return configure_tables(b);
}

int tentaco_batch_get_config(const tentaco_batch* b, int order, int* family, int* block,
                             int* group, int* schedule) {
  if (!b) return fail(TENTACO_EINVAL, "batch is NULL");
  if (order < 2 || order > kMaxOrder)
    return fail(TENTACO_EINVAL, "order %d outside 2..%d", order, kMaxOrder);
  if (family) *family = b->L.fam[order];
  if (block) *block = b->L.blk[order];
  if (group) *group = b->L.grp[order];
  if (schedule) *schedule = b->L.sch[order];
  return TENTACO_OK;
}

int tentaco_batch_set_schedule(tentaco_batch* b, int schedule) {
  clear_error();
  if (!b) return fail(TENTACO_EINVAL, "batch is NULL");
  if (schedule != 0 && schedule != 1) return fail(TENTACO_EINVAL, "schedule must be 0 or 1");
  for (int N = 0; N <= kMaxOrder; ++N) {
    if (b->L.sch[N] != schedule) drop_graph(b);
    b->L.sch[N] = schedule;
  }
  return TENTACO_OK;
}

int tentaco_batch_get_schedule(const tentaco_batch* b, int* schedule) {
  if (!b || !schedule) return fail(TENTACO_EINVAL, "NULL argument");
  *schedule = b->L.sch[main_order(b->L)];
  return TENTACO_OK;
}

int tentaco_batch_run(tentaco_batch* b, void* stream) {
  if (!b || !b->have_operands) return fail(TENTACO_EINVAL, "batch has no operands");
  return launch_batch(b->L, static_cast<hipStream_t>(stream));
}

int tentaco_batch_capture(tentaco_batch* b, void* stream) {
  clear_error();
  if (!b || !b->have_operands) return fail(TENTACO_EINVAL, "batch has no operands");
  drop_graph(b);
  hipStream_t st = static_cast<hipStream_t>(stream);
  bool own = false;
  if (!st) {
    TT_HIP_CHECK(hipStreamCreate(&st));  // capture needs a non-default stream
    own = true;
  }
  TT_HIP_CHECK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
  int rc = launch_batch(b->L, st);
  hipGraph_t g = nullptr;
  const hipError_t e = hipStreamEndCapture(st, &g);
  if (own) (void)hipStreamDestroy(st);
  if (rc) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  if (e != hipSuccess) return fail(TENTACO_EHIP, "graph capture failed: %s", hipGetErrorString(e));
  b->graph = g;
  TT_HIP_CHECK(hipGraphInstantiate(&b->exec, g, nullptr, nullptr, 0));
  return TENTACO_OK;
}

int tentaco_batch_launch(tentaco_batch* b, void* stream) {
  if (!b || !b->exec) return fail(TENTACO_EINVAL, "batch graph not captured");
  TT_HIP_CHECK(hipGraphLaunch(b->exec, static_cast<hipStream_t>(stream)));
  return TENTACO_OK;
}

int tentaco_batch_items(const tentaco_batch* b, int32_t* items, int32_t* grid, int32_t* nb) {
  if (!b) return fail(TENTACO_EINVAL, "batch is NULL");
  if (items) *items = b->L.total_items;
  if (grid) *grid = b->L.grid;
  if (nb) *nb = b->L.nb[main_order(b->L)];
  return TENTACO_OK;
}

int tentaco_batch_autotune(tentaco_batch* b, int reps, void* stream, int* best_family,
                           int* best_block, int* best_group, float* best_ms) {
  clear_error();
  if (!b || !b->have_operands) return fail(TENTACO_EINVAL, "batch has no operands");
  if (reps < 1) reps = 1;
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipEvent_t e0, e1;
  TT_HIP_CHECK(hipEventCreate(&e0));
  TT_HIP_CHECK(hipEventCreate(&e1));
  struct Ev {
    hipEvent_t a, b;
    ~Ev() {
      (void)hipEventDestroy(a);
      (void)hipEventDestroy(b);
    }
  } ev{e0, e1};
  std::vector<float> t(static_cast<size_t>(reps));
  // median of `reps` timed runs after a warm-up of the current configuration
  auto timed = [&](float* med) -> int {
    int rc = tentaco_batch_run(b, stream);
    for (int r = 0; r < reps && !rc; ++r) {
      (void)hipEventRecord(e0, st);
      rc = tentaco_batch_run(b, stream);
      (void)hipEventRecord(e1, st);
      (void)hipEventSynchronize(e1);
      (void)hipEventElapsedTime(&t[size_t(r)], e0, e1);
    }
    if (rc) return rc;
    std::sort(t.begin(), t.end());
    *med = t[t.size() / 2];
    return TENTACO_OK;
  };
  // 1. one tile for every order, with either schedule
  float bm = -1.f;
  int bf = -1, bb = 0, bg = 0, bs = 0;
  for (int sched = 0; sched < 2; ++sched)
    for (int fam = kEdgeParallel; fam <= kEdgeParallel; ++fam)
      for (int blk : {128, 256, 512})
        for (int grp : {4, 8, 16, 32, 64}) {
          float med = 0.f;
          int rc = tentaco_batch_configure(b, fam, blk, grp);
          if (!rc) rc = tentaco_batch_set_schedule(b, sched);
          if (!rc) rc = timed(&med);
          if (rc == TENTACO_EUNSUPPORTED) {
            clear_error();
            continue;
          }
          if (rc) return rc;
          if (bf < 0 || med < bm) {
            bm = med;
            bf = fam;
            bb = blk;
            bg = grp;
            bs = sched;
          }
        }
  if (bf < 0) return fail(TENTACO_EUNSUPPORTED, "no batch configuration ran");
  int rc = tentaco_batch_configure(b, bf, bb, bg);
  if (!rc) rc = tentaco_batch_set_schedule(b, bs);
  if (rc) return rc;
  // 2. each order group's own tile, the others held at their best, timed as
  // whole runs in the batch's output mode (the orders run together, so a
  // group's best tile depends on the others' work beside it)
  for (int N = 2; N <= kMaxOrder; ++N) {
    if (b->L.grp_task[N + 1] <= b->L.grp_task[N]) continue;
    int of = b->L.fam[N], ob = b->L.blk[N], og = b->L.grp[N], os = b->L.sch[N];
    const int f0 = of, b0 = ob, g0 = og, s0 = os;
    for (int sched = 0; sched < 2; ++sched)
    for (int fam = kEdgeParallel; fam <= kEdgeParallel; ++fam)
      for (int blk : {128, 256, 512})
        for (int grp : {4, 8, 16, 32, 64}) {
          if (fam == f0 && blk == b0 && grp == g0 && sched == s0) continue;
          float med = 0.f;
          rc = tentaco_batch_configure_order(b, N, fam, blk, grp, sched);
          if (!rc) rc = timed(&med);
          if (rc == TENTACO_EUNSUPPORTED) {
            clear_error();
            continue;
          }
          if (rc) return rc;
          if (med < bm) {
            bm = med;
            of = fam;
            ob = blk;
            og = grp;
            os = sched;
          }
        }
    rc = tentaco_batch_configure_order(b, N, of, ob, og, os);
    if (rc) return rc;
  }
  if (best_family) *best_family = bf;
  if (best_block) *best_block = bb;
  if (best_group) *best_group = bg;
  if (best_ms) *best_ms = bm;
  return TENTACO_OK;
}

int tentaco_batch_free(tentaco_batch* b) {
  if (!b) return TENTACO_OK;
  drop_graph(b);
  free_tables(b);
  (void)hipFree(b->d_counter);
  (void)hipFree(b->d_fill_off);
  (void)hipFree(b->d_rowbits);
  for (int k = 0; k <= kMaxOrder; ++k) {
    if (b->cev[k]) (void)hipEventDestroy(b->cev[k]);
    if (b->conc[k]) (void)hipStreamDestroy(b->conc[k]);
  }
  delete b;
  return TENTACO_OK;
}

}  // extern "C"
