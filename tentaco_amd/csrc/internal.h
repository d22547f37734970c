// Internal declarations shared by the tentaco HIP sources (not installed).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>

#include "../../include/taco_tensor_t.h"
#include "../../include/tentaco.h"

namespace tt {

constexpr int kMaxOrder = 5;

// Device view of a CSF tensor. Level 0 is the root (n0 nodes, output row of
// node x is crd0[x]); level m >= 1 has nodes[m] nodes whose parent ranges are
// pos[m][x]..pos[m][x+1] for parent x at level m-1; level order-1 holds the
// nonzeros (nodes[order-1] == nnz) with their values in vals.
struct CsfDev {
  int order = 0;
  int32_t nnz = 0;
  int32_t nodes[kMaxOrder] = {};
  const int32_t* crd0 = nullptr;
  const int32_t* pos[kMaxOrder] = {};
  const int32_t* crd[kMaxOrder] = {};
  const float* vals = nullptr;
  // optional, 3-mode only (built once per handle): the level-1 coordinate of
  // every nonzero and the first nonzero of every root node (n0 + 1 entries)
  const int32_t* crd1_of_nnz = nullptr;
  const int32_t* nnz_of_root = nullptr;
  // optional, 3-mode short fibres (built once per handle): every root node's
  // nonzeros at the fixed slots [x * pad_width, x * pad_width + count) as
  // ((level-1 coordinate << 16) | leaf coordinate, value bits); unused slots
  // hold kPadEmpty
  const uint2* pad = nullptr;
  int32_t pad_width = 0;
  // optional, 3-mode short fibres with slices of at most kPairSlots
  // nonzeros (built once per handle): root nodes in pairs, each pair's
  // nonzeros at the fixed slots [g * kPairSlots, (g + 1) * kPairSlots) in the
  // pad encoding (the first slice's, then the second's), and per pair
  // (output row of the first, of the second or -1, first slice's count, 0)
  const uint2* pair = nullptr;
  const int4* pair_info = nullptr;
  int32_t npairs = 0;
};
constexpr uint32_t kPadEmpty = 0xFFFFFFFFu;
constexpr int32_t kPairSlots = 256;

// Factor matrices by level: M[m] for m = 1..order-1, row-major rows x R.
struct FactorsDev {
  const float* M[kMaxOrder] = {};
};

// Kernel families of the MTTKRP variant table.
enum Family { kEdgeSerial = 0, kEdgeParallel = 1, kSliceRow = 2 };

struct Variant {
  int family;
  int block;  // threads per workgroup
  int group;  // nonzeros per lane group (edge families); slice-row: 0, or the
              // nonzeros a wave's slices start among (slice_group_kernel)
};

constexpr int kNumGridBlocks = 3;
constexpr int kNumGridGroups = 5;
constexpr int kGridBlocks[kNumGridBlocks] = {128, 256, 512};
constexpr int kGridGroups[kNumGridGroups] = {4, 8, 16, 32, 64};
// 2 edge families x 3 blocks x 5 groups, then 3 slice-row block sizes.
constexpr int kNumVariants = 2 * kNumGridBlocks * kNumGridGroups + kNumGridBlocks;

Variant variant_of(int v);
int default_variant();

// Lanes that share one factor row for rank R: 4, 8 or 16, a float4 each and from
// rank 65 on several (ranks 1 to 3: 4, a column each).
int lanes_per_row(int R);
// Nonzeros per lane group of a batch tile of 256 threads that nobody chose,
// for tasks of nnz nonzeros in all.
int batch_group(int64_t nnz, int R);
// Nonzeros one workgroup covers for an edge-family variant at rank R.
int64_t nnz_per_block(const Variant& vr, int R);
// Workspace bytes an MTTKRP call with a_rows output rows needs (0 for the
// slice-row family): the
// brackets (256-byte padded) for the edge families, then for the
// edge-serial family the FP64 accumulation rows (a_rows x R doubles).
size_t mttkrp_workspace_bytes(const CsfDev& B, int R, const Variant& vr, int32_t a_rows);
size_t edge_brk_bytes(const CsfDev& B, int64_t NB);
size_t ttv_workspace_bytes(const CsfDev& B);

// What a handle keeps for a tile, or nulls.
struct WalkTables {
  // the walk's wave starts for nnz_per_wave(vr, R) (edge families; see
  // launch_walk_starts); null: the call writes the brackets into ws
  const int32_t* starts = nullptr;
  // edge-parallel tiles (see launch_shared_rows): the FP64 rows that workgroups
  // sharing a slice add to, zero between calls, two per workgroup; each
  // workgroup's two; their output rows (-1: another's); and one bit per output
  // row that a root node with nonzeros writes. slots null: FP32 atomics
  const int2* slots = nullptr;
  const int32_t* rows = nullptr;
  const uint32_t* bits = nullptr;
  int32_t nbits = 0;
  double* W = nullptr;
};
// Enqueue one MTTKRP on `stream`. A (a_rows x R) is fully overwritten;
// `dense_root` says crd0 == 0..n0-1 with n0 == a_rows (no zero fill needed
// for the slice-row family). ws must hold mttkrp_workspace_bytes bytes.
// tables: what the handle keeps for the tile.
int launch_mttkrp(const CsfDev& B, const FactorsDev& F, int R, float* A,
                  int32_t a_rows, bool dense_root, const Variant& vr,
                  void* ws, const WalkTables& tables, hipStream_t stream);
// Write the slots and rows of an edge-parallel tile of NB nonzeros.
int launch_shared_rows(const CsfDev& B, int32_t NB, int2* slots, int32_t* rows, hipStream_t stream);
// Nonzeros one wave of an edge-family variant walks at rank R.
int64_t nnz_per_wave(const Variant& vr, int R);
// Write the node at every level 0..N-2 that holds the first nonzero of each
// run of wn nonzeros (edge_brk_bytes(B, wn) bytes) on `stream`.
int launch_walk_starts(const CsfDev& B, int64_t wn, int32_t* starts, hipStream_t stream);
// Fill the 3-mode expansion arrays of CsfDev (crd1_of_nnz: nnz entries,
// nnz_of_root: n0 + 1 entries) from the CSF's own pos/crd on `stream`.
int launch_expand3(const CsfDev& B, int32_t* crd1_of_nnz, int32_t* nnz_of_root,
                   hipStream_t stream);
// Fill the padded slice layout (n0 x width slots) of a 3-mode CSF whose
// level-1 and leaf coordinates are below 65535 and whose root nodes hold at
// most `width` nonzeros; nnz_of_root from launch_expand3 (same stream).
int launch_pad3(const CsfDev& B, const int32_t* nnz_of_root, int32_t width, uint2* pad,
                hipStream_t stream);
// The paired slice layout (same coordinate limits, root nodes of at most
// kPairSlots nonzeros) from the pairs (first root node, second or -1) with
// at most kPairSlots nonzeros together: npairs * kPairSlots slots and the
// per-pair info the kernel reads (same stream).
int launch_pair3(const CsfDev& B, const int32_t* nnz_of_root, const int2* pairs, int32_t npairs,
                 uint2* slots, int4* info, hipStream_t stream);

// Enqueue the MTTKRP of the mode held at CSF level `level` (1..order-1) on
// the same CSF: F.M[l] is the factor of level l for every l != level
// (including the root, l = 0); A (a_rows x R) is zero-filled, then
// accumulated atomically.
int launch_mttkrp_level(const CsfDev& B, const FactorsDev& F, int level, int R, float* A,
                        int32_t a_rows, hipStream_t stream);
// Per-handle transposed index of one level L >= 1 of a CSF, for the
// MTTKRP of that level's mode on a CSF rooted elsewhere (one allocation):
// tpos has dim + 1 entry offsets (entries sorted by level-L coordinate,
// ties in CSF order). The leaf level (L = N-1) keeps per entry (ent) its
// coordinates at levels 0..N-2 and value up to order 3, else its level N-2
// node and value bits, and per level N-2 node the coordinates at levels
// 0..N-2 (anc, N-1 per node). An inner level's entries are the level N-2
// nodes by their ancestor's coordinate, each with its range of nonzeros
// (node: the starts, then the ends) and its coordinates at the other levels
// 0..N-2 (anc, level by level).
struct LevelIndex {
  bool built = false;
  int level = 0;
  int32_t dim = 0;
  void* mem = nullptr;
  int32_t* tpos = nullptr;
  void* ent = nullptr;
  int32_t* node = nullptr;
  int32_t* anc = nullptr;
};
// Build the index of `level` over coordinates 0..dim-1 on `stream` and
// wait for it (allocates; not for capture).
int build_level_index(const CsfDev& B, int level, int32_t dim, LevelIndex* X, hipStream_t stream);
void free_level_index(LevelIndex* X);
// Enqueue the level's MTTKRP through its index: F.M[m] is the factor of
// level m for every m != level; every one of A's a_rows rows is written
// once, without atomics.
int launch_mttkrp_leaf(const CsfDev& B, const LevelIndex& X, const FactorsDev& F, int R, float* A,
                       int32_t a_rows, hipStream_t stream);
int launch_mttkrp_inner(const CsfDev& B, const LevelIndex& X, const FactorsDev& F, int level,
                        int R, float* A, int32_t a_rows, hipStream_t stream);

// Enqueue one TTV: y has nodes[order-2] floats, c the last mode's extent.
int launch_ttv(const CsfDev& B, const float* c, float* y, void* ws,
               hipStream_t stream);

// Per-handle structure of the unit TTV kernel, built once from the CSF:
// a bitmap with one bit per nonzero that marks the first nonzero of every
// level N-2 node (fibre), the fibre holding the first nonzero of every
// 512-nonzero unit, the table where waves leave the pieces of fibres that
// cross their ranges, and the window of c cached in LDS.
constexpr int kMaxBands = 8;
struct TtvPlan {
  bool built = false;
  bool ok = false;             // the unit kernel applies
  bool whole = false;          // few units, no long or empty fibre: whole fibres by the wave
  void* mem = nullptr;         // one allocation holding the arrays below
  // with empty fibres, the bitmap and unit table index the non-empty fibres
  // only: ne_fid maps them to output positions and empty_ids lists the
  // fibres written as zero (both NULL without empty fibres; in mem2)
  void* mem2 = nullptr;
  int32_t* ne_fid = nullptr;
  int32_t* empty_ids = nullptr;
  int32_t n_empty = 0;
  uint32_t* flags = nullptr;   // nunits * 16 words
  int32_t* unit_fid = nullptr; // nunits entries
  int32_t* bnd_fid = nullptr;  // 2 per wave (max_waves)
  float* bnd_val = nullptr;
  int32_t nunits = 0;
  int32_t max_waves = 0;
  int32_t cdim = 0;            // entries of c read (largest leaf coordinate + 1)
  int32_t k0 = 0;              // c[k0 .. k0 + lc) is staged in LDS
  int32_t lc = 0;
  int lds_floats = 0;          // LDS instance (floats of c per workgroup)
  int grid = 0;                // workgroups per launch
  // Banded layout, when c does not fit one window: the nonzeros of each
  // band of band_w consecutive leaf coordinates, in CSF order, each band
  // padded to whole units (padding: coordinate -1, value 0). A band's
  // workgroups stage the band's part of c in LDS, so every gather is an LDS
  // read; the pieces of a fibre in the bands ("segments", numbered band by
  // band in fibre order) are summed into y by a last pass.
  int nbands = 0;              // 0: one window (the arrays above)
  int32_t band_w = 0;
  void* bmem = nullptr;        // one allocation holding the arrays below
  void* bmem2 = nullptr;       // b_seg (sized once the segments are counted)
  uint16_t* b_crd = nullptr;   // b_len window indexes (leaf coordinate - band start)
  float* b_vals = nullptr;
  uint32_t* b_flags = nullptr; // segment starts, b_len / 32 words
  int32_t* b_unit_fid = nullptr;  // segment at each unit's first position
  int32_t* b_bnd_fid = nullptr;   // crossing table, 2 per wave
  float* b_bnd_val = nullptr;
  float* b_seg = nullptr;         // segment sums
  uint32_t* b_present = nullptr;  // nbands x b_fwords: fibre f has a segment in band b
  int32_t* b_prefix = nullptr;    // segments before word w of b_present (band-major)
  int32_t b_fwords = 0;
  int32_t b_len = 0;
  int32_t b_nseg = 0;
  int b_grid = 0;
  // pieces that cross a range start: (first slot, last slot, piece, 0) of
  // their parts in the crossing table; their sum slots hold markers
  int4* b_crossing = nullptr;
  int32_t b_cross = 0;
  int32_t b_unit0[kMaxBands + 1] = {};  // first unit of band b
  int32_t b_wg0[kMaxBands + 1] = {};    // first workgroup of band b
};
// Build the plan on `stream` and wait for it (allocates; not for capture).
// cdim is how many entries of c the kernel may read (largest leaf
// coordinate + 1); beyond 2^30 - 8 the plan does not apply. bands: 0 picks
// (the banded layout when the best window of c would serve under 3/4 of the
// gathers), 1 keeps one window, 2..kMaxBands forces that many bands.
// max_fibre: the most nonzeros of a level N-2 node.
int build_ttv_plan(const CsfDev& B, int32_t cdim, int bands, int64_t max_fibre, TtvPlan* plan,
                   hipStream_t stream);
void free_ttv_plan(TtvPlan* plan);
// Enqueue one TTV through the unit kernel (plan.ok must hold): every entry of
// y is written exactly once, with no atomics on y, so results are bitwise
// reproducible.
int launch_ttv_units(const CsfDev& B, const TtvPlan& plan, const float* c, float* y,
                     hipStream_t stream);

// One task of a batched persistent launch (a CSF with its factors, output
// and the walk's wave starts).
struct BatchTaskDev {
  CsfDev B;
  FactorsDev F;
  float* A = nullptr;
  int32_t* starts = nullptr;  // per item and wave, the nodes of its first nonzero
  // FP64 rows that the items sharing a slice add to, and per item those of its
  // first and last slice; row 2 i is of the slice that starts with item i, row
  // 2 i + 1 of the one that starts inside item i and reaches its end
  double* W = nullptr;
  int2* slots = nullptr;
  // output rows, and one bit per row, set where a root node with at least
  // one nonzero writes the row
  int32_t rows = 0;
  const uint32_t* rowbits = nullptr;
};

struct BatchLaunch {
  const BatchTaskDev* tasks = nullptr;  // device
  int32_t ntasks = 0;
  const int64_t* fill_off = nullptr;    // device, prefix of output sizes (floats)
  int64_t total_fill = 0;
  const int64_t* bnd_off = nullptr;     // device, prefix of (items+1) per task
  int64_t total_bnd = 0;
  float4** bnd_rows = nullptr;          // device, output row (or null) of every FP64 row
  double* bnd_w = nullptr;              // device, the tasks' FP64 rows (2 per boundary), zero between runs
  const int64_t* item_off = nullptr;    // device, prefix of items per task (ntasks + 1)
  int32_t total_items = 0;
  int32_t* counter = nullptr;           // device work counter
  // Tile per order (index = order): family (edge-parallel only), block,
  // group and nonzeros per item (nb = block / lanes-per-row * group). The
  // prep skips the output rows that root nodes with nonzeros store (their
  // bits in the tasks' rowbits), except the rows of the slices holding an
  // item's first or last nonzero, which take atomics.
  // sch[N] is how the order's persistent workgroups take items: 0 from a
  // device work counter, 1 static cyclic.
  int fam[kMaxOrder + 1] = {}, blk[kMaxOrder + 1] = {}, grp[kMaxOrder + 1] = {};
  int sch[kMaxOrder + 1] = {};
  int32_t nb[kMaxOrder + 1] = {};
  int R = 32;
  int grid = 0;  // the largest per-order grid
  // the device task table is sorted by order: tasks [grp_task[N],
  // grp_task[N+1]) of order N hold items [grp_item[N], grp_item[N+1]) and run
  // in their own persistent launch of grp_grid[N] workgroups; counter holds
  // kMaxOrder + 1 work counters, one per order
  int32_t grp_task[kMaxOrder + 2] = {};
  int32_t grp_item[kMaxOrder + 2] = {};
  int grp_grid[kMaxOrder + 1] = {};
  // batches of several orders with one block size: the workgroups of the one
  // launch that holds them all (0: launches per order)
  int all_grid = 0;
  // host copies of fill_off and bnd_off with ntasks + 1 entries (the group
  // ranges of the per-order preps)
  const int64_t* h_fill_off = nullptr;
  const int64_t* h_bnd_off = nullptr;
  // output rows no root node stores: 0 = zeroed by every launch; 1 =
  // retained (zeroed once by launch_batch_zero_outputs, then left alone, so
  // a launch writes only the rows the walk stores and, behind it from their FP64
  // sums, the rows of slices that items share)
  int retain = 0;
  // launches per order run concurrently: each group after the largest on its
  // own stream conc[N] (default priority), forked from and joined back to the
  // launch stream through events cev[0] (fork) and cev[N] (group N done);
  // conc[0] == nullptr runs them in order
  hipStream_t conc[kMaxOrder + 1] = {};
  hipEvent_t cev[kMaxOrder + 1] = {};
};

// One launch of the batch. The waves' starts must have been written by
// launch_batch_brackets for the current tiles.
int launch_batch(const BatchLaunch& L, hipStream_t stream);
// Write every task's wave starts for the current tiles (they depend
// on the CSFs and the tiles only).
int launch_batch_brackets(const BatchLaunch& L, hipStream_t stream);
// Zero every output row that no launch stores (and the boundary rows): the
// one-time fill of the retained mode.
int launch_batch_zero_outputs(const BatchLaunch& L, hipStream_t stream);
// Set, in bits (pre-cleared, one bit per output row), the row of every root
// node of B that holds at least one nonzero.
int launch_batch_rowbits(const CsfDev& B, uint32_t* bits, hipStream_t stream);
int batch_occupancy(int family, int block, int R, int32_t NB, int order, int* per_cu);
int batch_all_occupancy(int block, int R, int* per_cu);

// Launch one empty kernel of each code object that an MTTKRP of this order / a
// TTV uses on `stream`, so that loading them falls outside any later timed region.
int warm_mttkrp_module(int order, hipStream_t stream);
int warm_ttv_module(hipStream_t stream);

// Read n floats of buf (16-byte aligned) through the caches on `stream`;
// out (4 bytes) is written only in a case that cannot occur.
int launch_flush_read(const float* buf, int64_t n, float* out, hipStream_t stream);

// Fill n floats with value on `stream` (kernel, not hipMemsetAsync, so it is
// safe inside captured graphs).
int launch_fill(float* p, int64_t n, float value, hipStream_t stream);

// Whether variant v's tile fits the LDS limit at this order and rank (the
// launch refuses it with TENTACO_EUNSUPPORTED otherwise).
bool variant_fits(int order, int R, int v);

// Event timing of the main kernel of a call (no-op unless the kernel timer
// is on): begin before the launch, end after it, on the launch stream.
void ktimer_begin(hipStream_t stream);
void ktimer_end(hipStream_t stream, const char* kernel);

// Error plumbing: record a message for tentaco_last_error() and return code.
int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
void clear_error();
const char* last_error_text();

}  // namespace tt

#define TT_HIP_CHECK(expr)                                                  \
  do {                                                                      \
    hipError_t tt_e_ = (expr);                                              \
    if (tt_e_ != hipSuccess)                                                \
      return ::tt::fail(TENTACO_EHIP, "%s failed: %s (%s:%d)", #expr,       \
                        hipGetErrorString(tt_e_), __FILE__, __LINE__);      \
  } while (0)
