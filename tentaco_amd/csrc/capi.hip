// C ABI of the tentaco library: validation, device-resident CSF handles,
// per-call staging for the host-pointer entry points, hipEvent timing and the
// reference's symbol names. Kernels live in mttkrp.hip / ttv.hip.

#include <algorithm>
#include <cmath>
#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "host_csf.h"
#include "internal.h"
#include "tuning.h"

using tt::fail;

#include "handle.h"

namespace tt {
namespace {

// Host-side structural validation (host_csf.cpp), copied into the handle.
int validate_csf(const taco_tensor_t* B, int order, tentaco_csf* h, const LevelFn& put = {}) {
  CsfCheck ck;
  const int rc = validate_csf(B, order, &ck, put);
  if (rc) return rc;
  for (int m = 0; m < kMaxOrder; ++m) {
    h->dims[m] = ck.dims[m];
    h->nodes[m] = ck.nodes[m];
    h->max_crd[m] = ck.max_crd[m];
  }
  h->dense_root = ck.dense_root;
  h->stats = ck.stats;
  h->host_pairs = std::move(ck.pairs);
  return TENTACO_OK;
}

template <class T>
int upload_array(T** dst, const T* src, int64_t n) {
  *dst = nullptr;
  const size_t bytes = size_t(std::max<int64_t>(n, 1)) * sizeof(T);
  if (hipMalloc(reinterpret_cast<void**>(dst), bytes) != hipSuccess) {
    *dst = nullptr;
    return fail(TENTACO_ENOMEM, "hipMalloc of %zu bytes failed", bytes);
  }
  if (n > 0) TT_HIP_CHECK(hipMemcpy(*dst, src, size_t(n) * sizeof(T), hipMemcpyHostToDevice));
  return TENTACO_OK;
}

void free_starts(int32_t* p) { (void)hipFree(p); }

void free_shared(const WalkStarts::Shared& x) {
  if (x.used) {
    (void)hipEventSynchronize(x.used);  // the last call that adds to them
    (void)hipEventDestroy(x.used);
  }
  (void)hipFree(x.mem);
}

void free_handle(tentaco_csf* h) {
  if (!h) return;
  (void)hipFree(h->d_crd0);
  for (int m = 0; m < kMaxOrder; ++m) {
    (void)hipFree(h->d_pos[m]);
    (void)hipFree(h->d_crd[m]);
  }
  (void)hipFree(h->d_vals);
  (void)hipFree(h->ws);
  for (void* w : h->ws_retired) (void)hipFree(w);
  h->starts.starts.clear(free_starts);
  h->starts.shared.clear(free_shared);
  (void)hipFree(h->starts.bits);
  for (int m = 0; m < kMaxOrder; ++m) (void)hipFree(h->stage_f[m]);
  (void)hipFree(h->stage_a);
  (void)hipFree(h->d_crd1_of_nnz);
  (void)hipFree(h->d_nnz_of_root);
  (void)hipFree(h->d_pad);
  (void)hipFree(h->d_pair);  // the pair layout's one allocation
  free_ttv_plan(&h->ttv);
  for (int m = 0; m < kMaxOrder; ++m) free_level_index(&h->lvl[m]);
  delete h;
}

// Whether the paired slice layout is built for this handle: 3-mode short
// fibres, packable coordinates, slices that pair within the slots, at most
// twice the nonzeros in slots.
bool pairs_apply(const tentaco_csf* h) {
  if (h->order != 3) return false;
  const int64_t nnz = h->nodes[2], np = int64_t(h->host_pairs.size() / 2);
  return nnz * 4 <= int64_t(h->nodes[1]) * 5 && h->max_crd[1] < 65535 && h->max_crd[2] < 65535 &&
         h->stats.max_slice_nnz <= kPairSlots && np > 0 && np * kPairSlots <= 2 * nnz;
}

// The 3-mode expansion (level-1 coordinate per nonzero, first nonzero per
// root node) that the slice-row kernel's short-fibre path reads; built once,
// on `st`.
// Under stream capture nothing is built (the kernels that fill it would run
// only at replay): the slice-row launch then takes the kernel that needs no
// expansion.
int ensure_expand3(tentaco_csf* h, hipStream_t st) {
  if (h->order != 3 || h->d_crd1_of_nnz) return TENTACO_OK;
  const int64_t nnz = h->nodes[2];
  if (nnz <= 0) return TENTACO_OK;
  {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    TT_HIP_CHECK(hipStreamIsCapturing(st, &cs));
    if (cs != hipStreamCaptureStatusNone) return TENTACO_OK;
  }
  int32_t *kq = nullptr, *nzr = nullptr;
  if (hipMalloc(reinterpret_cast<void**>(&kq), size_t(nnz) * sizeof(int32_t)) != hipSuccess)
    return fail(TENTACO_ENOMEM, "expansion: hipMalloc of %lld ints failed", (long long)nnz);
  if (hipMalloc(reinterpret_cast<void**>(&nzr), (size_t(h->nodes[0]) + 1) * sizeof(int32_t)) !=
      hipSuccess) {
    (void)hipFree(kq);
    return fail(TENTACO_ENOMEM, "expansion: hipMalloc failed");
  }
  int rc = launch_expand3(h->view(), kq, nzr, st);
  if (rc) {
    (void)hipStreamSynchronize(st);
    (void)hipFree(kq);
    (void)hipFree(nzr);
    return rc;
  }
  h->d_crd1_of_nnz = kq;
  h->d_nnz_of_root = nzr;
  // the padded slice layout: short fibres, packable coordinates, slices of at
  // most 512 nonzeros and at most twice the nonzeros in slots; optional
  const int64_t width = std::max<int64_t>(64, (h->stats.max_slice_nnz + 63) / 64 * 64);
  const bool short_fibres = nnz * 4 <= int64_t(h->nodes[1]) * 5;
  if (short_fibres && h->max_crd[1] < 65535 && h->max_crd[2] < 65535 && width <= 512 &&
      int64_t(h->nodes[0]) * width <= 2 * nnz) {
    uint2* pad = nullptr;
    if (hipMalloc(reinterpret_cast<void**>(&pad), size_t(h->nodes[0]) * size_t(width) * sizeof(uint2)) ==
        hipSuccess) {
      if (launch_pad3(h->view(), nzr, int32_t(width), pad, st) == TENTACO_OK) {
        h->d_pad = pad;
        h->pad_width = int32_t(width);
      } else {
        (void)hipStreamSynchronize(st);
        (void)hipFree(pad);
        clear_error();
      }
    }
  }
  // the paired slice layout: the same conditions, slices of at most
  // kPairSlots nonzeros, pairs from host validation (largest with smallest
  // that fits), and at most twice the nonzeros in slots; optional
  static_assert(kPairCap == kPairSlots, "pairing capacity");
  const int32_t np = int32_t(h->host_pairs.size() / 2);
  if (pairs_apply(h)) {
    // one allocation: slots, per-pair info, the pairs (kept with it)
    const size_t b_slots = size_t(np) * kPairSlots * sizeof(uint2);
    const size_t b_info = (size_t(np) * sizeof(int4) + 255) & ~size_t(255);
    char* mem = nullptr;
    bool ok = hipMalloc(reinterpret_cast<void**>(&mem), b_slots + b_info + size_t(np) * sizeof(int2)) ==
              hipSuccess;
    uint2* slots = reinterpret_cast<uint2*>(mem);
    int4* info = reinterpret_cast<int4*>(mem + b_slots);
    int2* dpairs = reinterpret_cast<int2*>(mem + b_slots + b_info);
    ok = ok && hipMemcpyAsync(dpairs, h->host_pairs.data(), size_t(np) * sizeof(int2),
                              hipMemcpyHostToDevice, st) == hipSuccess;
    ok = ok && launch_pair3(h->view(), nzr, dpairs, np, slots, info, st) == TENTACO_OK;
    ok = ok && hipStreamSynchronize(st) == hipSuccess;
    if (ok) {
      h->d_pair = slots;
      h->d_pair_info = info;
      h->npairs = np;
    } else {
      (void)hipStreamSynchronize(st);
      (void)hipFree(mem);
      clear_error();
    }
  }
  return TENTACO_OK;
}

// The TTV unit kernel's plan, built once per handle on `st` (synchronizes).
// Under stream capture nothing is built and the bracket kernel runs instead.
// c is read up to the largest leaf coordinate, never beyond.
int ensure_ttv_plan(tentaco_csf* h, hipStream_t st) {
  if (h->ttv.built) return TENTACO_OK;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  TT_HIP_CHECK(hipStreamIsCapturing(st, &cs));
  if (cs != hipStreamCaptureStatusNone) return TENTACO_OK;
  return build_ttv_plan(h->view(), h->max_crd[h->order - 1] + 1, h->ttv_bands,
                        int64_t(h->stats.child_max[h->order - 1]), &h->ttv, st);
}

// Grow a device buffer to at least `bytes` (contents are not kept).
int grow(float** p, size_t* cap, size_t bytes) {
  if (bytes <= *cap && *p) return TENTACO_OK;
  (void)hipFree(*p);
  *p = nullptr;
  *cap = 0;
  if (hipMalloc(reinterpret_cast<void**>(p), std::max<size_t>(bytes, 4)) != hipSuccess) {
    *p = nullptr;
    return fail(TENTACO_ENOMEM, "hipMalloc of %zu bytes failed", bytes);
  }
  *cap = bytes;
  return TENTACO_OK;
}

// Grow the handle's workspace to at least `bytes`. A call enqueued on a
// capturing stream may not grow it (the graph would keep a buffer that a
// later eager call could replace): it fails and names the reserve call that
// avoids this. A replaced workspace is kept until the handle is freed, since
// a graph captured earlier may still read it.
int reserve_ws(tentaco_csf* h, size_t bytes, hipStream_t st) {
  if (bytes <= h->ws_bytes) return TENTACO_OK;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  TT_HIP_CHECK(hipStreamIsCapturing(st, &cs));
  if (cs != hipStreamCaptureStatusNone)
    return fail(TENTACO_EINVAL,
                "call under stream capture needs %zu bytes of workspace, %zu reserved: "
                "call tentaco_csf_reserve_rows with this rank, variant and output rows "
                "before capturing",
                bytes, h->ws_bytes);
  void* p = nullptr;
  if (hipMalloc(&p, bytes) != hipSuccess)
    return fail(TENTACO_ENOMEM, "workspace hipMalloc of %zu bytes failed", bytes);
  if (h->ws) h->ws_retired.push_back(h->ws);
  h->ws = p;
  h->ws_bytes = bytes;
  return TENTACO_OK;
}

// The wave starts of runs of wn nonzeros, complete for every stream; whether they
// could be built.
bool build_starts(const CsfDev& B, int64_t wn, hipStream_t st, int32_t** out) {
  int32_t* p = nullptr;
  if (hipMalloc(reinterpret_cast<void**>(&p), edge_brk_bytes(B, wn)) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  const int rc = launch_walk_starts(B, wn, p, st);
  if (hipStreamSynchronize(st) != hipSuccess || rc) {
    (void)hipGetLastError();
    clear_error();
    (void)hipFree(p);
    return false;
  }
  *out = p;
  return true;
}

// The shared rows of edge-parallel tiles of NB nonzeros at rank R, complete for
// every stream; whether they could be built. (under h->starts.mu, which guards
// bits)
bool build_shared_rows(tentaco_csf* h, int64_t NB, int R, hipStream_t st, WalkStarts::Shared* out) {
  const CsfDev B = h->view();
  WalkStarts& s = h->starts;
  WalkStarts::Shared x;
  const int64_t nblk = (int64_t(B.nnz) + NB - 1) / NB;
  const size_t o_rows = (size_t(nblk) * sizeof(int2) + 255) / 256 * 256;
  const size_t o_w = o_rows + (size_t(nblk) * 2 * sizeof(int32_t) + 255) / 256 * 256;
  const size_t wbytes = size_t(nblk) * 2 * size_t(R) * sizeof(double);
  const int32_t nbits = h->max_crd[0] + 1;
  const size_t bbytes = (size_t(nbits) + 31) / 32 * sizeof(uint32_t);
  uint32_t* bits = s.bits;
  bool ok = hipMalloc(&x.mem, o_w + wbytes) == hipSuccess;
  if (!ok) x.mem = nullptr;
  ok = ok && hipEventCreateWithFlags(&x.used, hipEventDisableTiming | hipEventDisableSystemFence) ==
                 hipSuccess;
  if (ok && !bits) {
    ok = hipMalloc(reinterpret_cast<void**>(&bits), bbytes) == hipSuccess;
    if (!ok) bits = nullptr;
    ok = ok && hipMemsetAsync(bits, 0, bbytes, st) == hipSuccess &&
         launch_batch_rowbits(B, bits, st) == TENTACO_OK;
  }
  char* base = static_cast<char*>(x.mem);
  int2* slots = reinterpret_cast<int2*>(base);
  int32_t* rows = reinterpret_cast<int32_t*>(base + o_rows);
  double* W = reinterpret_cast<double*>(base + o_w);
  ok = ok && hipMemsetAsync(W, 0, wbytes, st) == hipSuccess &&
       launch_shared_rows(B, int32_t(NB), slots, rows, st) == TENTACO_OK;
  ok = hipStreamSynchronize(st) == hipSuccess && ok;
  if (!ok) {
    (void)hipGetLastError();
    clear_error();
    (void)hipFree(x.mem);
    if (x.used) (void)hipEventDestroy(x.used);
    if (!s.bits) (void)hipFree(bits);
    return false;
  }
  s.bits = bits;
  x.t.slots = slots;
  x.t.rows = rows;
  x.t.bits = bits;
  x.t.nbits = nbits;
  x.t.W = W;
  *out = x;
  return true;
}

// Workgroups from which an edge-parallel variant's calls share rows in FP64 (AUTO's
// sized tile: auto_needs_rows). A long slice's row takes an FP32 addition from every
// workgroup, so its error grows with the root of their number: 100M nonzeros in
// 48,828 workgroups 4.6e-7 against FP64, 1.2e-7 with FP64 rows, 30M (5-mode) 5.8e-7
// and 1.2e-7. The rows' kernel and the event between calls cost 4 us more than the
// fill (1.5M nonzeros 28.9 and 33.1), a few in 100 of a call of that many workgroups.
constexpr int64_t kSharedBlocks = 2048;

// What walk_tables may build: nothing, what was not tried yet, or anything.
enum class Build { kNo, kYes, kAgain };

// What the handle keeps for variant vr at rank R (edge families), or nulls.
// With `build`, a missing table is built on st and waited for, so that it is
// complete for every stream; not under capture. One that cannot be built leaves
// the calls on the brackets they write themselves and on FP32 atomics, and only
// reserve tries again. rows: shared rows however few the workgroups. used: the
// event of the shared rows. (under h->starts.mu, which the caller holds until a
// call with shared rows is enqueued)
WalkTables walk_tables(tentaco_csf* h, const Variant& vr, int R, bool rows, Build build, hipStream_t st,
                       hipEvent_t* used = nullptr) {
  const CsfDev B = h->view();
  WalkTables t;
  if (vr.family == kSliceRow || vr.family < 0 || B.nnz <= 0) return t;
  const int64_t wn = nnz_per_wave(vr, R), NB = nnz_per_block(vr, R);
  WalkStarts& s = h->starts;
  const bool ep = vr.family == kEdgeParallel && (rows || B.nnz >= kSharedBlocks * NB);
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  const bool capturing =
      (ep || build != Build::kNo) &&
      (hipStreamIsCapturing(st, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone);
  const bool make = build != Build::kNo && !capturing, again = build == Build::kAgain;
  int32_t** starts = s.starts.get(
      wn, make, again, [&](int32_t** p) { return build_starts(B, wn, st, p); }, free_starts);
  if (!starts) return t;
  if (ep && !capturing) {
    const WalkStarts::Shared* x = s.shared.get(
        {NB, R}, make, again, [&](WalkStarts::Shared* y) { return build_shared_rows(h, NB, R, st, y); },
        free_shared);
    if (x) {
      t = x->t;
      if (used) *used = x->used;
    }
  }
  t.starts = *starts;
  return t;
}

// The tables that a sweep needs for one variant, held while it is timed: those
// the handle did not keep before are dropped again. (Kept for all the variants of
// a sweep, 100M nonzeros at rank 64 held 6 GB, and the rows of a later rank's
// choice found no place.)
class SweepTables {
 public:
  SweepTables(tentaco_csf* h, int v, int R, hipStream_t st) : h_(h) {
    std::lock_guard<std::mutex> lk(h->starts.mu);
    starts_ = h->starts.starts.mark();
    shared_ = h->starts.shared.mark();
    if (variant_fits(h->order, R, v)) (void)walk_tables(h, variant_of(v), R, false, Build::kYes, st);
  }
  ~SweepTables() {
    std::lock_guard<std::mutex> lk(h_->starts.mu);
    h_->starts.shared.back_to(shared_, free_shared);
    h_->starts.starts.back_to(starts_, free_starts);
  }
  SweepTables(const SweepTables&) = delete;
  SweepTables& operator=(const SweepTables&) = delete;

 private:
  tentaco_csf* h_;
  decltype(WalkStarts::starts)::Mark starts_;
  decltype(WalkStarts::shared)::Mark shared_;
};

int resolve_variant(const tentaco_csf* h, int R, int variant) {
  if (variant == TENTACO_VARIANT_DEFAULT) return default_variant();
  if (variant == TENTACO_VARIANT_AUTO) {
    const int tuned = h->tune.lookup(R);
    if (tuned >= 0) return tuned;
    return auto_variant(h->stats, h->order, R);
  }
  return variant;
}

// What a call with `variant` that resolved to v runs: AUTO's structural choice
// is resized to the tensor, anything else is the variant's own tile.
Variant tile_of(const tentaco_csf* h, int R, int variant, int v) {
  if (variant == TENTACO_VARIANT_AUTO && h->tune.lookup(R) < 0)
    return auto_tile(h->stats, h->order, R, pairs_apply(h));
  return variant_of(v);
}

// Whether that tile is only run with FP64 rows (see auto_needs_rows).
bool needs_rows(const tentaco_csf* h, int R, int variant, int v, const Variant& tile) {
  return variant == TENTACO_VARIANT_AUTO && h->tune.lookup(R) < 0 &&
         auto_needs_rows(h->stats, R, tile, variant_of(v));
}

// What such a call runs where FP64 rows are not to be had: for calls without
// kept state.
Variant plain_tile(const tentaco_csf* h, int R, int variant, int v) {
  const Variant tile = tile_of(h, R, variant, v);
  return needs_rows(h, R, variant, v, tile) ? variant_of(v) : tile;
}

// Load the code objects of MTTKRPs of this order and of TTV on the current device
// once, before the first timed region (the first launch from a code object loads
// it, which would otherwise land inside get_gpu_timer_result's region: 3.8 ms for
// an order's kernels).
int warm_device(int order) {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static bool done[kMaxDevices][kMaxOrder + 1] = {};
  int dev = 0;
  TT_HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return TENTACO_OK;
  std::lock_guard<std::mutex> lk(mu);
  if (done[dev][order]) return TENTACO_OK;
  int rc = warm_mttkrp_module(order, nullptr);
  if (!rc) rc = warm_ttv_module(nullptr);
  if (rc) return rc;
  TT_HIP_CHECK(hipStreamSynchronize(nullptr));
  done[dev][order] = true;
  return TENTACO_OK;
}

// ---- hot-region timer (GPUTimer, gpu_library.h:949-988) -------------------
std::atomic<float> g_last_ms{-1.f};
std::mutex g_timer_mu;
hipEvent_t g_ev0 = nullptr, g_ev1 = nullptr;

int ensure_events() {
  if (!g_ev0) TT_HIP_CHECK(hipEventCreate(&g_ev0));
  if (!g_ev1) TT_HIP_CHECK(hipEventCreate(&g_ev1));
  return TENTACO_OK;
}

// A handle with B's arrays on the device. A level's arrays are copied while its
// coordinates are still being checked (2M nonzeros: of 0.4 ms of checks 0.15
// are left in the way). Copying through pinned slabs of the call's own instead
// gained as much as allocating them takes, and allocating them took several ms
// now and then.
int upload_csf(const taco_tensor_t* B, int order, tentaco_csf** out) {
  tentaco_csf* h = new tentaco_csf;
  h->order = order;
  bool warm = false;
  int rc = validate_csf(B, order, h, [&](int m, int64_t parents, int64_t nodes) {
    int r = warm ? TENTACO_OK : warm_device(order);
    warm = true;
    if (!r) r = upload_array(&h->d_pos[m], B->indices[m][0], parents + 1);
    if (!r) r = upload_array(&h->d_crd[m], B->indices[m][1], nodes);
    return r;
  });
  if (!rc) rc = upload_array(&h->d_crd0, B->indices[0][1], h->nodes[0]);
  if (!rc) rc = upload_array(&h->d_vals, B->vals, h->nodes[order - 1]);
  if (rc) {
    free_handle(h);
    return rc;
  }
  *out = h;
  return TENTACO_OK;
}

// ---- per-call staging for the host-pointer entry points ------------------
struct DevBuf {
  void* p = nullptr;
  ~DevBuf() { (void)hipFree(p); }
};

int check_factor(const taco_tensor_t* F, int level, const tentaco_csf* h, int R) {
  if (!F || !F->dimensions || !F->vals)
    return fail(TENTACO_EINVAL, "factor of level %d is NULL/incomplete", level);
  if (F->dimensions[1] != R)
    return fail(TENTACO_EINVAL, "factor of level %d has %d columns, expected R=%d", level,
                F->dimensions[1], R);
  if (F->dimensions[0] <= h->max_crd[level])
    return fail(TENTACO_EINVAL, "factor of level %d has %d rows but coordinates reach %d",
                level, F->dimensions[0], h->max_crd[level]);
  return TENTACO_OK;
}

int host_mttkrp(int order, taco_tensor_t* A, taco_tensor_t* B,
                taco_tensor_t* const* factors, int variant) {
  clear_error();
  if (!A || !A->dimensions || !A->vals) return fail(TENTACO_EINVAL, "A is NULL/incomplete");
  if (!factors) return fail(TENTACO_EINVAL, "factors is NULL");
  DevBuf fb[kMaxOrder], abuf;
  tentaco_csf* h = nullptr;
  int rc = upload_csf(B, order, &h);
  if (rc) return rc;
  struct Guard {
    tentaco_csf* h;
    ~Guard() { free_handle(h); }
  } guard{h};
  const int R = A->dimensions[1];
  const int32_t a_rows = A->dimensions[0];
  if (R <= 0) return fail(TENTACO_EINVAL, "A has %d columns", R);
  if (a_rows <= h->max_crd[0])
    return fail(TENTACO_EINVAL, "A has %d rows but root coordinates reach %d", a_rows,
                h->max_crd[0]);
  const float* fdev[kMaxOrder] = {};
  for (int m = 1; m < order; ++m) {
    rc = check_factor(factors[m - 1], m, h, R);
    if (rc) return rc;
    float* d = nullptr;
    rc = upload_array(&d, factors[m - 1]->vals, int64_t(factors[m - 1]->dimensions[0]) * R);
    fb[m].p = d;
    if (rc) return rc;
    fdev[m - 1] = d;
  }
  const size_t abytes = size_t(a_rows) * size_t(R) * sizeof(float);
  if (hipMalloc(&abuf.p, std::max<size_t>(abytes, 4)) != hipSuccess)
    return fail(TENTACO_ENOMEM, "hipMalloc of A (%zu bytes) failed", abytes);
  const int v = resolve_variant(h, R, variant);
  const Variant vr = plain_tile(h, R, variant, v);
  if (vr.family < 0) return fail(TENTACO_EINVAL, "variant %d out of range", variant);
  rc = reserve_ws(h, mttkrp_workspace_bytes(h->view(), R, vr, a_rows), nullptr);
  if (rc) return rc;
  h->reserved = true;  // a handle for one call: its start table would be used once
  if (vr.family == kSliceRow) {
    rc = ensure_expand3(h, nullptr);  // per-handle structure, outside the timed region
    if (rc) return rc;
  }
  rc = warm_device(order);
  if (rc) return rc;
  TT_HIP_CHECK(hipDeviceSynchronize());
  {
    std::lock_guard<std::mutex> lk(g_timer_mu);
    rc = ensure_events();
    if (rc) return rc;
    TT_HIP_CHECK(hipEventRecord(g_ev0, nullptr));
    rc = tentaco_mttkrp_dev(h, R, fdev, static_cast<float*>(abuf.p), a_rows, variant, nullptr);
    if (rc) return rc;
    TT_HIP_CHECK(hipEventRecord(g_ev1, nullptr));
    TT_HIP_CHECK(hipEventSynchronize(g_ev1));
    float ms = -1.f;
    TT_HIP_CHECK(hipEventElapsedTime(&ms, g_ev0, g_ev1));
    g_last_ms.store(ms);
  }
  TT_HIP_CHECK(hipMemcpy(A->vals, abuf.p, abytes, hipMemcpyDeviceToHost));
  return TENTACO_OK;
}

int host_ttv(int order, taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* c) {
  clear_error();
  if (!A || !A->vals) return fail(TENTACO_EINVAL, "A is NULL/incomplete");
  if (!c || !c->dimensions || !c->vals) return fail(TENTACO_EINVAL, "c is NULL/incomplete");
  DevBuf cbuf, ybuf;
  tentaco_csf* h = nullptr;
  int rc = upload_csf(B, order, &h);
  if (rc) return rc;
  struct Guard {
    tentaco_csf* h;
    ~Guard() { free_handle(h); }
  } guard{h};
  // a handle for one call: the banded layout's build would cost more than
  // it saves
  h->ttv_bands = 1;
  if (c->dimensions[0] <= h->max_crd[order - 1])
    return fail(TENTACO_EINVAL, "c has %d entries but coordinates reach %d", c->dimensions[0],
                h->max_crd[order - 1]);
  const int32_t nf = h->nodes[order - 2];
  if (A->dimensions && A->dimensions[0] < nf)
    return fail(TENTACO_EINVAL, "A has %d entries, B has %d fibers", A->dimensions[0], nf);
  float* cd = nullptr;
  rc = upload_array(&cd, c->vals, c->dimensions[0]);
  cbuf.p = cd;
  if (rc) return rc;
  if (hipMalloc(&ybuf.p, std::max<size_t>(size_t(nf) * 4, 4)) != hipSuccess)
    return fail(TENTACO_ENOMEM, "hipMalloc of y failed");
  rc = ensure_ttv_plan(h, nullptr);  // outside the timed region
  if (rc) return rc;
  rc = warm_device(order);
  if (rc) return rc;
  TT_HIP_CHECK(hipDeviceSynchronize());
  {
    std::lock_guard<std::mutex> lk(g_timer_mu);
    rc = ensure_events();
    if (rc) return rc;
    TT_HIP_CHECK(hipEventRecord(g_ev0, nullptr));
    rc = tentaco_ttv_dev(h, cd, static_cast<float*>(ybuf.p), nullptr);
    if (rc) return rc;
    TT_HIP_CHECK(hipEventRecord(g_ev1, nullptr));
    TT_HIP_CHECK(hipEventSynchronize(g_ev1));
    float ms = -1.f;
    TT_HIP_CHECK(hipEventElapsedTime(&ms, g_ev0, g_ev1));
    g_last_ms.store(ms);
  }
  if (nf > 0) TT_HIP_CHECK(hipMemcpy(A->vals, ybuf.p, size_t(nf) * 4, hipMemcpyDeviceToHost));
  return TENTACO_OK;
}

// Legacy void entry points report failures on stderr (as gpuErrchk does,
// gpu_library.h:22-30) and through tentaco_last_error(), without exiting.
void legacy_report(const char* fn, int rc) {
  if (rc) std::fprintf(stderr, "tentaco %s failed (%d): %s\n", fn, rc, last_error_text());
}

int variant_index(int family, int block, int group) {
  int bi = -1, gi = -1;
  for (int i = 0; i < kNumGridBlocks; ++i)
    if (kGridBlocks[i] == block) bi = i;
  for (int i = 0; i < kNumGridGroups; ++i)
    if (kGridGroups[i] == group) gi = i;
  if (bi < 0 || gi < 0) return default_variant();
  return family * kNumGridBlocks * kNumGridGroups + bi * kNumGridGroups + gi;
}

// The variant a reference tuning name runs (its parameters as in
// legacy_names.inc): family < 0 is the fixed default; family 0 (eb_sr) is
// the edge-serial tile (block, run length p); family 1 (eb_pr) is the
// edge-parallel tile whose nonzeros per workgroup, at rank R, are nearest
// to the reference's Nnz = p on a log scale, ties going to the reference's
// block size and then to the smaller tile. Tiles that exceed the LDS limit
// at this order and rank are skipped.
int legacy_variant(int family, int block, int p, int R, int order) {
  if (family < 0) return default_variant();
  if (family == 0) return variant_index(0, block, p);
  int best = -1;
  double best_d = 0.0;
  int best_tie = 0;
  int64_t best_nb = 0;
  for (int bi = 0; bi < kNumGridBlocks; ++bi) {
    for (int gi = 0; gi < kNumGridGroups; ++gi) {
      const int v = variant_index(1, kGridBlocks[bi], kGridGroups[gi]);
      if (!variant_fits(order, R, v)) continue;
      const int64_t nb = nnz_per_block(variant_of(v), R);
      const double d = std::fabs(std::log2(double(nb) / double(std::max(p, 1))));
      const int tie = kGridBlocks[bi] == block ? 0 : 1;
      const bool better = best < 0 || d < best_d - 1e-9 ||
                          (std::fabs(d - best_d) <= 1e-9 &&
                           (tie < best_tie || (tie == best_tie && nb < best_nb)));
      if (better) {
        best = v;
        best_d = d;
        best_tie = tie;
        best_nb = nb;
      }
    }
  }
  return best >= 0 ? best : default_variant();
}

struct LegacyName {
  const char* name;
  int family, block, p;
};
const LegacyName kLegacyNames[] = {
    {"mttkrp_gpu_taco", -1, 0, 0},
#define TT_V(name, fam, tb, p) {#name, fam, tb, p},
#include "legacy_names.inc"
#undef TT_V
};

}  // namespace
}  // namespace tt

// ---- MTTKRP without allocation --------------------------------------------
// The scratch of tentaco_mttkrp_dev_noalloc: the partition brackets and, for
// the edge-serial family, the FP64 rows of one call. One copy per device,
// held until the process ends. In host code `scratch` names a host-side
// stand-in: kernels get the device address from hipGetSymbolAddress.
constexpr size_t kScratchBytes = size_t(32) << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace tt {
namespace {
constexpr int kScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kScratchDevices] = {};

// The current device's scratch address, looked up once per device.
int scratch_address(void** out) {
  int dev = 0;
  TT_HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kScratchDevices)
    return fail(TENTACO_EUNSUPPORTED, "device %d beyond the %d the scratch table holds", dev,
                kScratchDevices);
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(TENTACO_EHIP, "hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return TENTACO_OK;
}
}  // namespace
}  // namespace tt


using namespace tt;

extern "C" {

int tentaco_version(void) { return 10000; }

int tentaco_device_check(void) {
  clear_error();
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n <= 0)
    return fail(TENTACO_ENOGPU, "no HIP device visible");
  int dev = 0;
  TT_HIP_CHECK(hipGetDevice(&dev));
  hipDeviceProp_t prop;
  TT_HIP_CHECK(hipGetDeviceProperties(&prop, dev));
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return fail(TENTACO_ENOGPU, "device %d is %s, this build targets gfx950", dev,
                prop.gcnArchName);
  return TENTACO_OK;
}

int tentaco_csf_upload(const taco_tensor_t* B, int order, tentaco_csf** out) {
  clear_error();
  if (!out) return fail(TENTACO_EINVAL, "out is NULL");
  *out = nullptr;
  return upload_csf(B, order, out);
}

int tentaco_csf_upload_async(const taco_tensor_t* B, int order, void* stream, tentaco_csf** out) {
  clear_error();
  if (!out) return fail(TENTACO_EINVAL, "out is NULL");
  *out = nullptr;
  hipStream_t st = static_cast<hipStream_t>(stream);
  tentaco_csf* h = new tentaco_csf;
  h->order = order;
  int rc = validate_csf(B, order, h);
  if (rc) {
    delete h;
    return rc;
  }
  auto put = [&](int32_t** dst, const int32_t* src, int64_t n) -> int {
    const size_t bytes = size_t(std::max<int64_t>(n, 1)) * sizeof(int32_t);
    if (hipMalloc(reinterpret_cast<void**>(dst), bytes) != hipSuccess) {
      *dst = nullptr;
      return fail(TENTACO_ENOMEM, "hipMalloc of %zu bytes failed", bytes);
    }
    if (n > 0) TT_HIP_CHECK(hipMemcpyAsync(*dst, src, size_t(n) * sizeof(int32_t), hipMemcpyHostToDevice, st));
    return TENTACO_OK;
  };
  rc = put(&h->d_crd0, B->indices[0][1], h->nodes[0]);
  for (int m = 1; m < order && !rc; ++m) {
    rc = put(&h->d_pos[m], B->indices[m][0], int64_t(h->nodes[m - 1]) + 1);
    if (!rc) rc = put(&h->d_crd[m], B->indices[m][1], h->nodes[m]);
  }
  if (!rc) {
    const int64_t nnz = h->nodes[order - 1];
    const size_t bytes = size_t(std::max<int64_t>(nnz, 1)) * sizeof(float);
    if (hipMalloc(reinterpret_cast<void**>(&h->d_vals), bytes) != hipSuccess) {
      h->d_vals = nullptr;
      rc = fail(TENTACO_ENOMEM, "hipMalloc of %zu bytes failed", bytes);
    } else if (nnz > 0 && hipMemcpyAsync(h->d_vals, B->vals, size_t(nnz) * sizeof(float),
                                         hipMemcpyHostToDevice, st) != hipSuccess) {
      rc = fail(TENTACO_EHIP, "value upload failed");
    }
  }
  if (rc) {
    (void)hipStreamSynchronize(st);
    free_handle(h);
    return rc;
  }
  *out = h;
  return TENTACO_OK;
}

int tentaco_mttkrp_host_async(tentaco_csf* h, int R, taco_tensor_t* const* factors,
                              taco_tensor_t* A, int variant, void* stream) {
  clear_error();
  if (!h) return fail(TENTACO_EINVAL, "handle is NULL");
  if (!A || !A->dimensions || !A->vals) return fail(TENTACO_EINVAL, "A is NULL/incomplete");
  if (!factors) return fail(TENTACO_EINVAL, "factors is NULL");
  if (R <= 0 || A->dimensions[1] != R)
    return fail(TENTACO_EINVAL, "A has %d columns, expected R=%d", A->dimensions[1], R);
  const int32_t a_rows = A->dimensions[0];
  if (a_rows <= h->max_crd[0])
    return fail(TENTACO_EINVAL, "A has %d rows but root coordinates reach %d", a_rows,
                h->max_crd[0]);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const float* fdev[kMaxOrder] = {};
  for (int m = 1; m < h->order; ++m) {
    int rc = check_factor(factors[m - 1], m, h, R);
    if (rc) return rc;
    const size_t bytes = size_t(factors[m - 1]->dimensions[0]) * size_t(R) * sizeof(float);
    rc = grow(&h->stage_f[m], &h->stage_f_cap[m], bytes);
    if (rc) return rc;
    TT_HIP_CHECK(hipMemcpyAsync(h->stage_f[m], factors[m - 1]->vals, bytes, hipMemcpyHostToDevice, st));
    fdev[m - 1] = h->stage_f[m];
  }
  const size_t abytes = size_t(a_rows) * size_t(R) * sizeof(float);
  int rc = grow(&h->stage_a, &h->stage_a_cap, abytes);
  if (rc) return rc;
  rc = tentaco_mttkrp_dev(h, R, fdev, h->stage_a, a_rows, variant, stream);
  if (rc) return rc;
  TT_HIP_CHECK(hipMemcpyAsync(A->vals, h->stage_a, abytes, hipMemcpyDeviceToHost, st));
  return TENTACO_OK;
}

int tentaco_host_alloc(void** ptr, size_t bytes) {
  clear_error();
  if (!ptr) return fail(TENTACO_EINVAL, "ptr is NULL");
  *ptr = nullptr;
  if (hipHostMalloc(ptr, std::max<size_t>(bytes, 4), hipHostMallocDefault) != hipSuccess) {
    *ptr = nullptr;
    return fail(TENTACO_ENOMEM, "hipHostMalloc of %zu bytes failed", bytes);
  }
  return TENTACO_OK;
}

int tentaco_host_free(void* ptr) {
  if (ptr) TT_HIP_CHECK(hipHostFree(ptr));
  return TENTACO_OK;
}

int tentaco_stream_create(void** stream) {
  clear_error();
  if (!stream) return fail(TENTACO_EINVAL, "stream is NULL");
  hipStream_t s = nullptr;
  TT_HIP_CHECK(hipStreamCreate(&s));  // default priority
  *stream = s;
  return TENTACO_OK;
}

int tentaco_stream_destroy(void* stream) {
  if (stream) TT_HIP_CHECK(hipStreamDestroy(static_cast<hipStream_t>(stream)));
  return TENTACO_OK;
}

int tentaco_stream_synchronize(void* stream) {
  TT_HIP_CHECK(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
  return TENTACO_OK;
}

int tentaco_csf_free(tentaco_csf* h) {
  free_handle(h);
  return TENTACO_OK;
}

int tentaco_csf_info(const tentaco_csf* h, int* order, int64_t* nnz, int32_t* nodes) {
  if (!h) return fail(TENTACO_EINVAL, "handle is NULL");
  if (order) *order = h->order;
  if (nnz) *nnz = h->nodes[h->order - 1];
  if (nodes)
    for (int m = 0; m < kMaxOrder; ++m) nodes[m] = m < h->order ? h->nodes[m] : 0;
  return TENTACO_OK;
}

int tentaco_csf_reserve_rows(tentaco_csf* h, int R, int variant, int32_t a_rows) {
  clear_error();
  if (!h) return fail(TENTACO_EINVAL, "handle is NULL");
  if (a_rows <= h->max_crd[0])
    return fail(TENTACO_EINVAL, "A has %d rows but root coordinates reach %d", a_rows,
                h->max_crd[0]);
  size_t need = ttv_workspace_bytes(h->view());
  if (variant == TENTACO_VARIANT_AUTO && h->tune.lookup(R) < 0) {
    // AUTO may pick any variant later: reserve for the largest need
    for (int v = 0; v < kNumVariants; ++v)
      need = std::max(need, mttkrp_workspace_bytes(h->view(), R, variant_of(v), a_rows));
  } else {
    const Variant vr = variant_of(resolve_variant(h, R, variant));
    if (vr.family < 0) return fail(TENTACO_EINVAL, "variant %d out of range", variant);
    need = std::max(need, mttkrp_workspace_bytes(h->view(), R, vr, a_rows));
  }
  // the slice-row kernel's 3-mode expansion, so that no later call allocates
  int rc = ensure_expand3(h, nullptr);
  if (!rc) rc = (hipDeviceSynchronize() == hipSuccess) ? TENTACO_OK
                                                       : fail(TENTACO_EHIP, "synchronize failed");
  if (rc) return rc;
  rc = reserve_ws(h, need, nullptr);
  if (rc) return rc;
  // the tables of the tile that calls with this argument run, and of the one
  // that calls under capture run in its place
  const int v = resolve_variant(h, R, variant);
  const Variant tile = tile_of(h, R, variant, v);
  const bool rows = needs_rows(h, R, variant, v, tile);
  std::lock_guard<std::mutex> lk(h->starts.mu);
  (void)walk_tables(h, tile, R, rows, Build::kAgain, nullptr);
  if (rows) (void)walk_tables(h, variant_of(v), R, false, Build::kAgain, nullptr);
  h->reserved = true;
  return TENTACO_OK;
}

int tentaco_csf_reserve(tentaco_csf* h, int R, int variant) {
  if (!h) return fail(TENTACO_EINVAL, "handle is NULL");
  return tentaco_csf_reserve_rows(h, R, variant, h->dims[0]);
}

// AUTO on a rank with no tuned entry and a selector attached: take the
// selector's pick when its predicted margin is at least min_margin (and keep
// it for this rank), else run the sweep, which records the measured best.
// Under stream capture neither may run (both synchronise), so the structural
// heuristic answers instead.
static int sweep_impl(tentaco_csf* h, int R, const float* const* factors_dev, float* A_dev,
                      int32_t a_rows, int reps, float cut, void* stream, const bool* use,
                      float* times_ms);

// Records v for AUTO at rank R, with its tables: calls on a reserved handle build
// none, and this one may (it was chosen by measuring or by the selector, which
// allocate too). Not under capture.
static void choose(tentaco_csf* h, int R, int v, int source, hipStream_t st) {
  h->tune.set(R, v, source);
  std::lock_guard<std::mutex> lk(h->starts.mu);
  (void)walk_tables(h, variant_of(v), R, false, Build::kYes, st);
}

static int auto_with_selector(tentaco_csf* h, int R, const float* const* factors_dev,
                              float* A_dev, int32_t a_rows, hipStream_t st, int* out) {
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  TT_HIP_CHECK(hipStreamIsCapturing(st, &cs));
  if (cs != hipStreamCaptureStatusNone) {
    *out = auto_variant(h->stats, h->order, R);
    return TENTACO_OK;
  }
  float f[TENTACO_NUM_FEATURES];
  int rc = csf_features(h, R, f);
  if (rc) return rc;
  int pick = -1;
  float margin = 0.f;
  float pred[kNumVariants];
  rc = mlp_select(h->selector, h->order, R, f, &pick, &margin, pred);
  if (rc) return rc;
  if (margin >= h->min_margin) {
    choose(h, R, pick, TENTACO_TUNED_SELECTOR, st);
    *out = pick;
    return TENTACO_OK;
  }
  if (h->fallback_k > 0) {
    // time only the k best-predicted variants that fit
    int order_v[kNumVariants];
    int n = 0;
    for (int v = 0; v < kNumVariants; ++v)
      if (variant_fits(h->order, R, v)) order_v[n++] = v;
    std::stable_sort(order_v, order_v + n, [&](int a, int b) { return pred[a] < pred[b]; });
    bool use[kNumVariants] = {};
    for (int i = 0; i < std::min(n, h->fallback_k); ++i) use[order_v[i]] = true;
    float t[kNumVariants];
    rc = sweep_impl(h, R, factors_dev, A_dev, a_rows, 3, 0.f, st, use, t);
    if (rc) return rc;
    int best = -1;
    for (int v = 0; v < kNumVariants; ++v)
      if (t[v] >= 0.f && (best < 0 || t[v] < t[best])) best = v;
    if (best < 0) best = pick;
    choose(h, R, best, TENTACO_TUNED_SELECTOR_TIMED, st);
    *out = best;
    return TENTACO_OK;
  }
  int best = -1;
  rc = tentaco_csf_autotune(h, R, factors_dev, A_dev, a_rows, 3, st, &best, nullptr);
  if (rc) return rc;
  *out = best;
  return TENTACO_OK;
}

int tentaco_mttkrp_dev(tentaco_csf* h, int R, const float* const* factors_dev, float* A_dev,
                       int32_t a_rows, int variant, void* stream) {
  if (!h) return fail(TENTACO_EINVAL, "handle is NULL");
  if (!A_dev || !factors_dev) return fail(TENTACO_EINVAL, "NULL device buffer");
  if (R <= 0) return fail(TENTACO_EINVAL, "R=%d", R);
  if (a_rows <= h->max_crd[0])
    return fail(TENTACO_EINVAL, "A has %d rows but root coordinates reach %d", a_rows,
                h->max_crd[0]);
  FactorsDev F;
  for (int m = 1; m < h->order; ++m) {
    if (!factors_dev[m - 1]) return fail(TENTACO_EINVAL, "factor of level %d is NULL", m);
    F.M[m] = factors_dev[m - 1];
  }
  int v = -1;
  int rc = TENTACO_OK;
  if (variant == TENTACO_VARIANT_AUTO && h->tune.lookup(R) < 0 && h->selector) {
    rc = auto_with_selector(h, R, factors_dev, A_dev, a_rows, static_cast<hipStream_t>(stream), &v);
    if (rc) return rc;
  } else {
    v = resolve_variant(h, R, variant);
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  Variant vr = tile_of(h, R, variant, v);
  if (vr.family < 0) return fail(TENTACO_EINVAL, "variant %d out of range", variant);
  if (vr.family == kSliceRow) {
    rc = ensure_expand3(h, st);
    if (rc) return rc;
  }
  const CsfDev B = h->view();
  const bool rows = needs_rows(h, R, variant, v, vr);
  std::unique_lock<std::mutex> lk(h->starts.mu);
  const Build build = h->reserved ? Build::kNo : Build::kYes;
  hipEvent_t used = nullptr;
  WalkTables tables = walk_tables(h, vr, R, rows, build, st, &used);
  if (rows && !tables.slots) {  // no FP64 rows here: the variant's own tile
    vr = variant_of(v);
    tables = walk_tables(h, vr, R, false, build, st, &used);
  }
  rc = reserve_ws(h, mttkrp_workspace_bytes(B, R, vr, a_rows), st);
  if (rc) return rc;
  const bool dense = h->dense_root && a_rows == h->nodes[0];
  if (!tables.slots) {
    lk.unlock();
    return launch_mttkrp(B, F, R, A_dev, a_rows, dense, vr, h->ws, tables, st);
  }
  TT_HIP_CHECK(hipStreamWaitEvent(st, used, 0));
  rc = launch_mttkrp(B, F, R, A_dev, a_rows, dense, vr, h->ws, tables, st);
  TT_HIP_CHECK(hipEventRecord(used, st));
  return rc;
}

int tentaco_mttkrp_dev_noalloc(tentaco_csf* h, int R, const float* const* factors_dev,
                               float* A_dev, int32_t a_rows, int variant, void* stream) {
  if (!h) return fail(TENTACO_EINVAL, "handle is NULL");
  if (!A_dev || !factors_dev) return fail(TENTACO_EINVAL, "NULL device buffer");
  if (R <= 0) return fail(TENTACO_EINVAL, "R=%d", R);
  if (a_rows <= h->max_crd[0])
    return fail(TENTACO_EINVAL, "A has %d rows but root coordinates reach %d", a_rows,
                h->max_crd[0]);
  FactorsDev F;
  for (int m = 1; m < h->order; ++m) {
    if (!factors_dev[m - 1]) return fail(TENTACO_EINVAL, "factor of level %d is NULL", m);
    F.M[m] = factors_dev[m - 1];
  }
  // AUTO: the recorded choice or the structural heuristic (the selector and
  // the sweep allocate and synchronise)
  const int v = resolve_variant(h, R, variant);
  const Variant vr = plain_tile(h, R, variant, v);
  if (vr.family < 0) return fail(TENTACO_EINVAL, "variant %d out of range", variant);
  const CsfDev B = h->view();
  const size_t need = mttkrp_workspace_bytes(B, R, vr, a_rows);
  if (need > kScratchBytes)
    return fail(TENTACO_EUNSUPPORTED,
                "variant %s at R=%d with %d output rows needs %zu bytes of scratch; the "
                "allocation-free entry point holds %zu",
                tentaco_variant_name(v), R, a_rows, need, kScratchBytes);
  void* ws = nullptr;
  if (need > 0) {
    const int rc = scratch_address(&ws);
    if (rc) return rc;
  }
  // slice-row: the 3-mode expansion and padded layout are used when a
  // reserve call built them, never built here
  const bool dense = h->dense_root && a_rows == h->nodes[0];
  return launch_mttkrp(B, F, R, A_dev, a_rows, dense, vr, ws, WalkTables{},
                       static_cast<hipStream_t>(stream));
}

// The sweep over the variants with use[v] set (all when use is NULL);
// times_ms[v] = -1 for the others.
static int sweep_impl(tentaco_csf* h, int R, const float* const* factors_dev, float* A_dev,
                      int32_t a_rows, int reps, float cut, void* stream, const bool* use,
                      float* times_ms) {
  if (reps < 1) reps = 1;
  hipStream_t st = static_cast<hipStream_t>(stream);
  // reserve the largest tile's workspace first: no timed call allocates
  {
    size_t need = 0;
    for (int v = 0; v < kNumVariants; ++v)
      need = std::max(need, mttkrp_workspace_bytes(h->view(), R, variant_of(v), a_rows));
    int rc = reserve_ws(h, need, st);
    if (rc) return rc;
  }
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
  // time `calls` back-to-back calls of variant v between one event pair
  auto timed = [&](int v, int calls, float* ms) -> int {
    TT_HIP_CHECK(hipEventRecord(e0, st));
    for (int c = 0; c < calls; ++c) {
      int rc = tentaco_mttkrp_dev(h, R, factors_dev, A_dev, a_rows, v, stream);
      if (rc) return rc;
    }
    TT_HIP_CHECK(hipEventRecord(e1, st));
    TT_HIP_CHECK(hipEventSynchronize(e1));
    float t = 0.f;
    TT_HIP_CHECK(hipEventElapsedTime(&t, e0, e1));
    *ms = t / float(calls);
    return TENTACO_OK;
  };
  // phase 1: a timed warm-up per variant; when it is short (< 2 ms, where
  // first-launch costs would show) a second call is the probe
  float best_probe = -1.f;
  for (int v = 0; v < kNumVariants; ++v) {
    times_ms[v] = -1.f;
    if (use && !use[v]) continue;
    float p = 0.f;
    SweepTables tables(h, v, R, st);
    int rc = timed(v, 1, &p);
    if (rc == TENTACO_EUNSUPPORTED) {
      clear_error();
      continue;
    }
    if (rc) return rc;
    if (p < 2.f) {
      rc = timed(v, 1, &p);
      if (rc) return rc;
    }
    times_ms[v] = p;
    if (best_probe < 0.f || p < best_probe) best_probe = p;
  }
  if (best_probe < 0.f) return fail(TENTACO_EUNSUPPORTED, "no variant ran");
  // phase 2: the median of `reps` repetitions for every variant within the
  // cut; a repetition spans about 100 us (up to 32 calls) so that launch
  // latency does not dominate small tensors
  std::vector<float> t(static_cast<size_t>(reps));
  for (int v = 0; v < kNumVariants; ++v) {
    const float p = times_ms[v];
    if (p < 0.f) continue;
    if (cut > 0.f && p > cut * best_probe) continue;
    SweepTables tables(h, v, R, st);
    int calls = int(std::ceil(0.1f / std::max(p, 1e-4f)));
    calls = std::min(32, std::max(1, calls));
    for (int r = 0; r < reps; ++r) {
      int rc = timed(v, calls, &t[size_t(r)]);
      if (rc) return rc;
    }
    std::sort(t.begin(), t.end());
    times_ms[v] = t[t.size() / 2];
  }
  return TENTACO_OK;
}

int tentaco_mttkrp_dev_repeat(tentaco_csf* h, int R, const float* const* factors_dev,
                              float* A_dev, int32_t a_rows, int variant, void* stream,
                              int count) {
  if (count < 0) return fail(TENTACO_EINVAL, "count = %d", count);
  for (int i = 0; i < count; ++i) {
    int rc = tentaco_mttkrp_dev(h, R, factors_dev, A_dev, a_rows, variant, stream);
    if (rc) return rc;
  }
  return TENTACO_OK;
}

int tentaco_mttkrp_level_dev(tentaco_csf* h, int level, int R, const float* const* factors_dev,
                             float* A_dev, int32_t a_rows, void* stream) {
  clear_error();
  if (!h) return fail(TENTACO_EINVAL, "handle is NULL");
  if (!A_dev || !factors_dev) return fail(TENTACO_EINVAL, "NULL device buffer");
  if (R <= 0) return fail(TENTACO_EINVAL, "R=%d", R);
  if (level < 1 || level >= h->order)
    return fail(TENTACO_EINVAL, "level %d outside 1..%d", level, h->order - 1);
  if (a_rows <= h->max_crd[level])
    return fail(TENTACO_EINVAL, "A has %d rows but level-%d coordinates reach %d", a_rows, level,
                h->max_crd[level]);
  FactorsDev F;
  for (int l = 0; l < h->order; ++l) {
    if (l == level) continue;
    if (!factors_dev[l]) return fail(TENTACO_EINVAL, "factor of level %d is NULL", l);
    F.M[l] = factors_dev[l];
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  // through the level's transposed index, built on first use outside
  // capture (under capture without it: the atomic level kernel)
  LevelIndex& X = h->lvl[level];
  if (!X.built) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    TT_HIP_CHECK(hipStreamIsCapturing(st, &cs));
    if (cs == hipStreamCaptureStatusNone) {
      const int rc = build_level_index(h->view(), level, h->dims[level], &X, st);
      if (rc) return rc;
    }
  }
  if (X.built) {
    if (level == h->order - 1) return launch_mttkrp_leaf(h->view(), X, F, R, A_dev, a_rows, st);
    return launch_mttkrp_inner(h->view(), X, F, level, R, A_dev, a_rows, st);
  }
  return launch_mttkrp_level(h->view(), F, level, R, A_dev, a_rows, st);
}

int tentaco_csf_reserve_level(tentaco_csf* h, int level) {
  clear_error();
  if (!h) return fail(TENTACO_EINVAL, "handle is NULL");
  if (level < 1 || level >= h->order)
    return fail(TENTACO_EINVAL, "level %d outside 1..%d", level, h->order - 1);
  if (h->lvl[level].built) return TENTACO_OK;
  return build_level_index(h->view(), level, h->dims[level], &h->lvl[level], nullptr);
}

int tentaco_csf_sweep(tentaco_csf* h, int R, const float* const* factors_dev, float* A_dev,
                      int32_t a_rows, int reps, float cut, void* stream, float* times_ms) {
  clear_error();
  if (!h) return fail(TENTACO_EINVAL, "handle is NULL");
  if (!times_ms) return fail(TENTACO_EINVAL, "times_ms is NULL");
  return sweep_impl(h, R, factors_dev, A_dev, a_rows, reps, cut, stream, nullptr, times_ms);
}

int tentaco_csf_autotune(tentaco_csf* h, int R, const float* const* factors_dev, float* A_dev,
                         int32_t a_rows, int reps, void* stream, int* best, float* times_ms) {
  std::vector<float> t(static_cast<size_t>(kNumVariants), -1.f);
  int rc = tentaco_csf_sweep(h, R, factors_dev, A_dev, a_rows, reps, 4.0f, stream, t.data());
  if (rc) return rc;
  int best_v = -1;
  for (int v = 0; v < kNumVariants; ++v)
    if (t[size_t(v)] >= 0.f && (best_v < 0 || t[size_t(v)] < t[size_t(best_v)])) best_v = v;
  if (best_v < 0) return fail(TENTACO_EUNSUPPORTED, "no variant ran");
  choose(h, R, best_v, TENTACO_TUNED_SWEEP, static_cast<hipStream_t>(stream));
  if (best) *best = best_v;
  if (times_ms) std::copy(t.begin(), t.end(), times_ms);
  return TENTACO_OK;
}

int tentaco_csf_set_tuned(tentaco_csf* h, int R, int variant) {
  if (!h) return fail(TENTACO_EINVAL, "handle is NULL");
  if (variant_of(variant).family < 0) return fail(TENTACO_EINVAL, "variant %d out of range", variant);
  h->tune.set(R, variant, TENTACO_TUNED_SET);
  return TENTACO_OK;
}

int tentaco_csf_tuned(const tentaco_csf* h, int R, int* variant, int* source) {
  if (!h) return fail(TENTACO_EINVAL, "handle is NULL");
  int src = 0;
  const int v = h->tune.lookup(R, &src);
  if (variant) *variant = v;
  if (source) *source = v < 0 ? 0 : src;
  return TENTACO_OK;
}

int tentaco_csf_set_selector_fallback(tentaco_csf* h, int top_k) {
  if (!h) return fail(TENTACO_EINVAL, "handle is NULL");
  if (top_k < 0) return fail(TENTACO_EINVAL, "top_k must be >= 0");
  h->fallback_k = top_k;
  return TENTACO_OK;
}

int tentaco_csf_set_selector(tentaco_csf* h, tentaco_mlp* m, float min_margin) {
  if (!h) return fail(TENTACO_EINVAL, "handle is NULL");
  if (m && tentaco_mlp_num_params(kNumVariants) <= 0)
    return fail(TENTACO_EINVAL, "selector is malformed");
  if (!(min_margin >= 0.f)) return fail(TENTACO_EINVAL, "min_margin must be >= 0");
  h->selector = m;
  h->min_margin = min_margin;
  return TENTACO_OK;
}

int tentaco_csf_set_ttv_bands(tentaco_csf* h, int bands) {
  clear_error();
  if (!h) return fail(TENTACO_EINVAL, "handle is NULL");
  if (bands < 0 || bands > kMaxBands)
    return fail(TENTACO_EINVAL, "bands must be 0 (pick), 1 (one window) or 2..%d", kMaxBands);
  if (bands == h->ttv_bands) return TENTACO_OK;
  h->ttv_bands = bands;
  if (h->ttv.built) {
    // the plan is rebuilt at the next TTV outside capture; a graph captured
    // earlier may still read the old one, so its memory lives until the
    // handle is freed
    for (void* m : {h->ttv.mem, h->ttv.mem2, h->ttv.bmem, h->ttv.bmem2})
      if (m) h->ws_retired.push_back(m);
    h->ttv = TtvPlan{};
  }
  return TENTACO_OK;
}

int tentaco_csf_ttv_layout(const tentaco_csf* h, int* bands, int64_t* device_bytes) {
  clear_error();
  if (!h) return fail(TENTACO_EINVAL, "handle is NULL");
  const TtvPlan& P = h->ttv;
  if (bands) *bands = !P.built || !P.ok ? 0 : P.nbands >= 2 ? P.nbands : 1;
  if (device_bytes) {
    int64_t b = 0;
    if (P.ok && P.nbands >= 2)
      b = int64_t(P.b_len) * 8 + int64_t(P.b_len) / 8 + int64_t(P.b_nseg) * 4 +
          int64_t(P.nbands) * P.b_fwords * 8;
    *device_bytes = b;
  }
  return TENTACO_OK;
}

int tentaco_ttv_dev(tentaco_csf* h, const float* c_dev, float* A_dev, void* stream) {
  if (!h) return fail(TENTACO_EINVAL, "handle is NULL");
  if (!c_dev || !A_dev) return fail(TENTACO_EINVAL, "NULL device buffer");
  const CsfDev B = h->view();
  hipStream_t st = static_cast<hipStream_t>(stream);
  int rc = ensure_ttv_plan(h, st);
  if (rc) return rc;
  if (h->ttv.ok) return launch_ttv_units(B, h->ttv, c_dev, A_dev, st);
  rc = reserve_ws(h, ttv_workspace_bytes(B), st);
  if (rc) return rc;
  return launch_ttv(B, c_dev, A_dev, h->ws, st);
}

int tentaco_mttkrp3(taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* C, taco_tensor_t* D) {
  taco_tensor_t* f[2] = {C, D};
  return host_mttkrp(3, A, B, f, TENTACO_VARIANT_AUTO);
}

int tentaco_mttkrp4(taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* C, taco_tensor_t* D,
                    taco_tensor_t* E) {
  taco_tensor_t* f[3] = {C, D, E};
  return host_mttkrp(4, A, B, f, TENTACO_VARIANT_AUTO);
}

int tentaco_mttkrp5(taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* C, taco_tensor_t* D,
                    taco_tensor_t* E, taco_tensor_t* F) {
  taco_tensor_t* f[4] = {C, D, E, F};
  return host_mttkrp(5, A, B, f, TENTACO_VARIANT_AUTO);
}

int tentaco_mttkrp(int order, taco_tensor_t* A, taco_tensor_t* B,
                   taco_tensor_t* const* factors, int variant) {
  return host_mttkrp(order, A, B, factors, variant);
}

int tentaco_ttv(taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* c) {
  return host_ttv(3, A, B, c);
}

int tentaco_ttv_n(int order, taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* c) {
  return host_ttv(order, A, B, c);
}

float get_gpu_timer_result(void) { return g_last_ms.load(); }

float tentaco_legacy_timer_ms(void) { return g_last_ms.load(); }

void tentaco_legacy_mttkrp3(int family, int block, int p, const char* name, taco_tensor_t* A,
                            taco_tensor_t* B, taco_tensor_t* C, taco_tensor_t* D) {
  taco_tensor_t* f[2] = {C, D};
  int v = TENTACO_VARIANT_DEFAULT;
  if (family >= 0) {
    // the rank comes from A (checked again by the call itself)
    const int R = (A && A->dimensions) ? A->dimensions[1] : 0;
    v = legacy_variant(family, block, p, R > 0 ? R : 32, 3);
  }
  legacy_report(name ? name : "mttkrp", host_mttkrp(3, A, B, f, v));
}

int tentaco_legacy_variant(const char* name, int R, int order, int* variant) {
  clear_error();
  if (!name || !variant) return fail(TENTACO_EINVAL, "NULL argument");
  if (R <= 0 || order < 2 || order > kMaxOrder)
    return fail(TENTACO_EINVAL, "R=%d, order=%d", R, order);
  for (const LegacyName& n : kLegacyNames) {
    if (std::strcmp(n.name, name) == 0) {
      *variant = legacy_variant(n.family, n.block, n.p, R, order);
      return TENTACO_OK;
    }
  }
  return fail(TENTACO_EINVAL, "%s is not one of the reference's MTTKRP names", name);
}

void tentaco_legacy_ttv3(const char* name, taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* C) {
  legacy_report(name ? name : "ttv", host_ttv(3, A, B, C));
}

void mttkrp_gpu_taco(taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* C, taco_tensor_t* D) {
  tentaco_legacy_mttkrp3(-1, 0, 0, "mttkrp_gpu_taco", A, B, C, D);
}

void ttv_csf_gpu_taco(taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* C) {
  tentaco_legacy_ttv3("ttv_csf_gpu_taco", A, B, C);
}

#define TT_V(name, fam, tb, p)                                                       \
  void name(taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* C, taco_tensor_t* D) { \
    tentaco_legacy_mttkrp3(fam, tb, p, #name, A, B, C, D);                           \
  }
#include "legacy_names.inc"
#undef TT_V

int tentaco_num_variants(void) { return kNumVariants; }

const char* tentaco_variant_name(int v) {
  static std::vector<std::string> names = [] {
    std::vector<std::string> n;
    for (int i = 0; i < kNumVariants; ++i) {
      const Variant vr = variant_of(i);
      char buf[64];
      if (vr.family == kSliceRow) std::snprintf(buf, sizeof buf, "sr_b%d", vr.block);
      else
        std::snprintf(buf, sizeof buf, "%s_b%d_g%d", vr.family == kEdgeSerial ? "es" : "ep",
                      vr.block, vr.group);
      n.emplace_back(buf);
    }
    return n;
  }();
  if (v < 0 || v >= kNumVariants) return nullptr;
  return names[v].c_str();
}

int tentaco_variant_params(int v, int* family, int* block, int* group) {
  const Variant vr = variant_of(v);
  if (vr.family < 0) return fail(TENTACO_EINVAL, "variant %d out of range", v);
  if (family) *family = vr.family;
  if (block) *block = vr.block;
  if (group) *group = vr.group;
  return TENTACO_OK;
}

int tentaco_default_variant(void) { return default_variant(); }

int tentaco_variant_fits(int order, int R, int v) { return variant_fits(order, R, v) ? 1 : 0; }

int tentaco_csf_resolve_variant(const tentaco_csf* h, int R, int variant, int* out) {
  clear_error();
  if (!h || !out) return fail(TENTACO_EINVAL, "NULL argument");
  if (R <= 0) return fail(TENTACO_EINVAL, "R=%d", R);
  const int v = resolve_variant(h, R, variant);
  if (variant_of(v).family < 0) return fail(TENTACO_EINVAL, "variant %d out of range", variant);
  *out = v;
  return TENTACO_OK;
}

int tentaco_dev_malloc(void** ptr, size_t bytes) {
  if (!ptr) return fail(TENTACO_EINVAL, "ptr is NULL");
  if (hipMalloc(ptr, std::max<size_t>(bytes, 4)) != hipSuccess) {
    *ptr = nullptr;
    return fail(TENTACO_ENOMEM, "hipMalloc of %zu bytes failed", bytes);
  }
  return TENTACO_OK;
}

int tentaco_dev_free(void* ptr) {
  TT_HIP_CHECK(hipFree(ptr));
  return TENTACO_OK;
}

int tentaco_memcpy_h2d(void* dst, const void* src, size_t bytes) {
  TT_HIP_CHECK(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
  return TENTACO_OK;
}

int tentaco_memcpy_d2h(void* dst, const void* src, size_t bytes) {
  TT_HIP_CHECK(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
  return TENTACO_OK;
}

int tentaco_dev_synchronize(void) {
  TT_HIP_CHECK(hipDeviceSynchronize());
  return TENTACO_OK;
}

int tentaco_flush_cache(void* stream) {
  // Reads a 512 MiB buffer (twice the 256 MB Infinity Cache) so that the
  // next kernel starts with cold L2/MALL holding only clean lines: the
  // analog of Timer::clear_cache (timers.h:62-75), which reads a large
  // array, for the GPU timing protocol. The buffer is filled once, when it
  // is allocated.
  static void* buf = nullptr;
  static std::mutex mu;
  constexpr size_t kBytes = size_t(512) << 20;
  {
    std::lock_guard<std::mutex> lk(mu);
    if (!buf) {
      if (hipMalloc(&buf, kBytes + 256) != hipSuccess) {
        buf = nullptr;
        return fail(TENTACO_ENOMEM, "flush buffer allocation failed");
      }
      int rc = launch_fill(static_cast<float*>(buf), int64_t((kBytes + 256) / sizeof(float)), 1.0f,
                           static_cast<hipStream_t>(stream));
      if (rc) return rc;
    }
  }
  float* b = static_cast<float*>(buf);
  return launch_flush_read(b, int64_t(kBytes / sizeof(float)), b + kBytes / sizeof(float),
                           static_cast<hipStream_t>(stream));
}

int tentaco_timer_start(void* stream) {
  std::lock_guard<std::mutex> lk(g_timer_mu);
  int rc = ensure_events();
  if (rc) return rc;
  TT_HIP_CHECK(hipEventRecord(g_ev0, static_cast<hipStream_t>(stream)));
  return TENTACO_OK;
}

int tentaco_timer_stop(void* stream, float* ms) {
  std::lock_guard<std::mutex> lk(g_timer_mu);
  int rc = ensure_events();
  if (rc) return rc;
  TT_HIP_CHECK(hipEventRecord(g_ev1, static_cast<hipStream_t>(stream)));
  TT_HIP_CHECK(hipEventSynchronize(g_ev1));
  float t = -1.f;
  TT_HIP_CHECK(hipEventElapsedTime(&t, g_ev0, g_ev1));
  if (ms) *ms = t;
  return TENTACO_OK;
}

}  // extern "C"
