// CSF MTTKRP kernels for gfx950 (wave64), orders 2..5.
//
//   A(i,:) = sum over the subtree of root node i of
//            B(i,k,l,...) * C(k,:) (.) D(l,:) (.) ...
//
// computed in factorised form: the upper levels' row product of a fibre is
// formed once, and multiplies the leaf rows of its nonzeros (the workspace
// kernels of tensor_kernels/mttkrp{3,4}_csf_cpu_taco_workspace.h and
// mttkrp5_csf_cpu_taco.h sum a fibre first). Factor rows are gathered as float4
// fragments over a row group of lanes (rowops.h).
//
// Three kernel families form the variant table:
//  * edge-serial (ES) and edge-parallel (EP): the nonzeros are cut into equal
//    runs, one per wave, of as many consecutive positions as the wave's row
//    groups would walk at G each (the reference's eb_sr work split,
//    mttkrp3_csf_ebsr.h:4-77, gives a run to a lane group). A slice that starts
//    and ends inside one run is stored; the first and last slices of a
//    workgroup's runs are summed in FP64 in LDS (the role of segReduceGroup,
//    gpu_library.h:295-321), and only the workgroup's first and last slice can
//    be another's too. ES adds them to FP64 rows of the whole output, EP to the
//    pre-zeroed output with FP32 atomics or, from 2048 workgroups on and under
//    AUTO from 300k nonzeros on, to FP64 rows of the shared slices
//    (edge_rows_kernel).
//  * slice-row (SR): one workgroup per root node, its level-1 children
//    spread over the workgroup's row groups, rows reduced with xor shuffles
//    and LDS and stored once; for 3-mode short fibres two slices to a workgroup
//    (slice_pair_kernel) or, for short slices under AUTO, whole slices by the wave
//    (slice_group_kernel). No atomics, no zero fill for a dense root,
//    deterministic; balanced only when slices are.
//
// Where a wave's run starts (its node at every level) is a table that the
// handle or batch keeps for a run length, or comes from brackets that the call
// itself writes, with the zero fill of A, in one prep launch (the reference's
// two partition-search launches plus cudaMemset, mttkrp3_csf_gpu_taco.h:88-94).

#include <algorithm>
#include <climits>

#include "internal.h"
#include "mttkrp_dispatch.h"
#include "rowops.h"
#include "tuning.h"

namespace tt {
namespace {

// ---------------------------------------------------------------------------
// prep: zero A and compute, for every workgroup boundary b (0..nblk), the
// node at each level that contains nonzero position min(b*NB, nnz-1).
// brk has (nblk+1) x (N-1) entries, level-major per boundary.
__global__ __launch_bounds__(256) void edge_prep_kernel(CsfDev B, float* A,
                                                        int64_t a_elems,
                                                        int32_t* brk,
                                                        int32_t nblk,
                                                        int32_t NB) {
  const int64_t tid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  // zero fill, float4 body + scalar tail
  const int64_t n4 = a_elems >> 2;
  float4* A4 = reinterpret_cast<float4*>(A);
  for (int64_t i = tid; i < n4; i += nthr) A4[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int64_t i = (n4 << 2) + tid; i < a_elems; i += nthr) A[i] = 0.f;
  if (B.nnz <= 0) return;
  const int N = B.order;
  for (int64_t b = tid; b <= nblk; b += nthr) {
    int64_t p = b * int64_t(NB);
    if (p > B.nnz - 1) p = B.nnz - 1;
    int32_t key = int32_t(p);
    for (int m = N - 2; m >= 0; --m) {
      const int32_t x = search_le(B.pos[m + 1], 0, B.nodes[m] - 1, key);
      brk[b * (N - 1) + m] = x;
      key = x;
    }
  }
}

// A = FP32(W) over n elements (the edge-serial family's FP64 rows).
__global__ __launch_bounds__(256) void narrow_kernel(const double* __restrict__ W,
                                                     float* __restrict__ A, int64_t n) {
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  const int64_t n2 = n >> 1;
  const double2* W2 = reinterpret_cast<const double2*>(W);
  float2* A2 = reinterpret_cast<float2*>(A);
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n2; i += nthr) {
    const double2 w = W2[i];
    A2[i] = make_float2(float(w.x), float(w.y));
  }
  if (blockIdx.x == 0 && threadIdx.x == 0 && (n & 1)) A[n - 1] = float(W[n - 1]);
}

__global__ __launch_bounds__(256) void expand3_kernel(const int32_t* __restrict__ pos1,
                                                      const int32_t* __restrict__ pos2,
                                                      const int32_t* __restrict__ crd1,
                                                      int32_t n0, int32_t nf,
                                                      int32_t* __restrict__ kq,
                                                      int32_t* __restrict__ nzr) {
  const int64_t tid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t f = tid; f < nf; f += nthr) {
    const int32_t k = crd1[f];
    for (int32_t q = pos2[f]; q < pos2[f + 1]; ++q) kq[q] = k;
  }
  for (int64_t x = tid; x <= n0; x += nthr) nzr[x] = pos2[pos1[x]];
}

__global__ __launch_bounds__(256) void pad3_fill_kernel(uint2* __restrict__ pad, int64_t n) {
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += nthr)
    pad[i] = make_uint2(kPadEmpty, 0u);
}

__global__ __launch_bounds__(256) void pad3_build_kernel(CsfDev B, const int32_t* __restrict__ nzr,
                                                         int32_t width, uint2* __restrict__ pad) {
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  const int32_t nf = B.nodes[1];
  for (int64_t f = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; f < nf; f += nthr) {
    const int32_t x = search_le(B.pos[1], 0, B.nodes[0] - 1, int32_t(f));
    const uint32_t hi = uint32_t(B.crd[1][f]) << 16;
    uint2* slot = pad + int64_t(x) * width - nzr[x];
    for (int32_t q = B.pos[2][f]; q < B.pos[2][f + 1]; ++q)
      slot[q] = make_uint2(hi | uint32_t(B.crd[2][q]), __float_as_uint(B.vals[q]));
  }
}

// Pair g's slots: the first root node's nonzeros, then the second's, then
// kPadEmpty; info[g] = (row of the first, row of the second or -1, count of
// the first, 0).
__global__ __launch_bounds__(256) void pair3_build_kernel(CsfDev B, const int32_t* __restrict__ nzr,
                                                          const int2* __restrict__ pairs,
                                                          int32_t npairs, uint2* __restrict__ slots,
                                                          int4* __restrict__ info) {
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  const int64_t n = int64_t(npairs) * kPairSlots;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += nthr) {
    const int32_t g = int32_t(i / kPairSlots);
    const int32_t t = int32_t(i % kPairSlots);
    const int2 pr = pairs[g];
    const int32_t na = nzr[pr.x + 1] - nzr[pr.x];
    const int32_t nb = pr.y >= 0 ? nzr[pr.y + 1] - nzr[pr.y] : 0;
    int32_t q = -1;
    if (t < na) q = nzr[pr.x] + t;
    else if (t < na + nb) q = nzr[pr.y] + (t - na);
    slots[i] = q >= 0 ? make_uint2((uint32_t(B.crd1_of_nnz[q]) << 16) | uint32_t(B.crd[2][q]),
                                   __float_as_uint(B.vals[q]))
                      : make_uint2(kPadEmpty, 0u);
    if (t == 0) info[g] = make_int4(B.crd0[pr.x], pr.y >= 0 ? B.crd0[pr.y] : -1, na, 0);
  }
}

__global__ __launch_bounds__(256) void fill_kernel(float* A, int64_t n, float value) {
  const int64_t tid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  const int64_t n4 = n >> 2;
  float4* A4 = reinterpret_cast<float4*>(A);
  const float4 v4 = make_float4(value, value, value, value);
  for (int64_t i = tid; i < n4; i += nthr) A4[i] = v4;
  for (int64_t i = (n4 << 2) + tid; i < n; i += nthr) A[i] = value;
}

// ---------------------------------------------------------------------------
// batched persistent launch: every (tensor, mode) task's nonzeros are cut into
// the same NB-sized items; persistent workgroups pull items from a device
// counter (left at zero by batch_rows_kernel) until the queue is empty, and run
// the edge walk of the item's task. Every workgroup leaves the loop when the
// counter passes the item count.
// Root node of CSF B that holds nonzero position p (the largest node at each
// level whose range starts at or before the key, so empty nodes are skipped).
__device__ __forceinline__ int32_t root_of_position(const CsfDev& B, int32_t p) {
  int32_t key = p;
  for (int m = B.order - 2; m >= 0; --m) key = search_le(B.pos[m + 1], 0, B.nodes[m] - 1, key);
  return key;
}

// Which FP64 row the slice of root node x adds to: 2 i if it starts with item
// (or workgroup) i of NB nonzeros, 2 i + 1 if inside it.
__device__ __forceinline__ int32_t slot_of_root(const CsfDev& B, int32_t x, int32_t NB) {
  for (int m = 1; m < B.order; ++m) x = B.pos[m][x];
  return 2 * (x / NB) + (x % NB ? 1 : 0);
}

// What a batch_rows_kernel launch does (bits): zero the output rows no root
// node stores, write the waves' starts and the shared rows' list, write the
// rows of the slices that items share.
constexpr int kRowsFill = 1, kRowsList = 2, kRowsShared = 4;

// Nonzeros per work item and waves per workgroup of each order group (kernel
// argument, by value).
struct BatchNB {
  int32_t nb[kMaxOrder + 1];
  int32_t nw[kMaxOrder + 1];
};

// The tasks' rows that the walk does not store, after it: with kRowsFill zero the
// outputs (quads [0, q_hi)), skipping a row
// whose bit is set in the task's rowbits, because a root node with nonzeros
// stores it; with kRowsShared write the rows of the slices that hold an item's
// first or last nonzero. Several items may share those, so the walk adds to FP64
// rows for them, which are left zero for the next run, as the work counters are
// (hundreds of FP32 additions to a long slice's row, in whichever order, were
// most of a batch's error: a sweep's worst factor against FP64, 30 seeds, had
// 7.5e-7 on average and 4.5e-6 at most, now 4.5e-7 and 8.1e-7). With kRowsList (once per configuration) write where the waves of
// each item start, its slots of FP64 rows, and the list of their output rows
// (entries [0, b_hi), two per item, null where an earlier item has the
// slice's). The list depends on the CSFs, outputs and tiles only; finding the
// rows on every run took 17 us a launch in a CP-ALS sweep over three tensors.
__global__ __launch_bounds__(256) void batch_rows_kernel(const BatchTaskDev* __restrict__ tasks,
                                                         int32_t nt,
                                                         const int64_t* __restrict__ fill_off,
                                                         int64_t q_hi,
                                                         const int64_t* __restrict__ bnd_off,
                                                         int64_t b_hi,
                                                         int32_t* __restrict__ counter,
                                                         BatchNB nbs, int R,
                                                         int qshift, int mode,
                                                         float4** __restrict__ bnd_rows,
                                                         double* __restrict__ bnd_w) {
  const int64_t tid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  // the work counters of the orders
  if (tid >= 2 && tid <= kMaxOrder) counter[tid] = 0;
  if (!(mode & kRowsFill)) q_hi = 0;
  // Zero the outputs as float4 quads (every output holds rows x R floats
  // with R a multiple of 4 and starts 16-byte aligned, which the host
  // checks). Each workgroup takes one contiguous range of quads, finds the
  // task of its first quad with one search and walks forward across task
  // boundaries (empty tasks included).
  // (quad e of a task is in row e >> qshift, with R / 4 == 1 << qshift)
  const int64_t per = (q_hi + gridDim.x - 1) / gridDim.x;
  const int64_t q0 = int64_t(blockIdx.x) * per;
  const int64_t q1 = q0 + per < q_hi ? q0 + per : q_hi;
  if (q0 < q1) {
    int32_t t = upper_index(fill_off, nt, q0 << 2);
    int64_t base = fill_off[t] >> 2;
    int64_t next = t + 1 < nt ? fill_off[t + 1] >> 2 : q_hi;
    float4* A4 = reinterpret_cast<float4*>(tasks[t].A);
    const uint32_t* bits = tasks[t].rowbits;
    // four quads per thread and pass, their bitmap words loaded before any
    // of their stores
    constexpr int U = 4;
    const int64_t stride = blockDim.x;
    for (int64_t q = q0 + threadIdx.x; q < q1; q += U * stride) {
      float4* dst[U];
      const uint32_t* wp[U];
      int sh[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t qq = q + u * stride;
        dst[u] = nullptr;
        if (qq >= q1) continue;
        if (qq >= next) {
          do {
            ++t;
            next = t + 1 < nt ? fill_off[t + 1] >> 2 : q_hi;
          } while (qq >= next);
          base = fill_off[t] >> 2;
          A4 = reinterpret_cast<float4*>(tasks[t].A);
          bits = tasks[t].rowbits;
        }
        const int64_t e = qq - base;
        const int64_t r = e >> qshift;
        dst[u] = A4 + e;
        wp[u] = bits + (r >> 5);
        sh[u] = int(r & 31);
      }
      uint32_t w[U];
#pragma unroll
      for (int u = 0; u < U; ++u) w[u] = dst[u] ? *wp[u] : 0u;
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (dst[u] && !((w[u] >> sh[u]) & 1u)) *dst[u] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  if (mode & kRowsShared) {
    const int64_t n = b_hi << (qshift + 1);
    for (int64_t i = tid; i < n; i += nthr) {
      float4* row = bnd_rows[i >> qshift];
      if (!row) continue;
      double2* w = reinterpret_cast<double2*>(bnd_w) + 2 * i;
      const double2 x = w[0], y = w[1];
      w[0] = w[1] = make_double2(0.0, 0.0);
      row[i & ((1 << qshift) - 1)] = make_float4(float(x.x), float(x.y), float(y.x), float(y.y));
    }
  }
  if (!(mode & kRowsList)) return;
  for (int64_t i = tid; i < b_hi; i += nthr) {
    const int32_t t = upper_index(bnd_off, nt, i);
    const BatchTaskDev& T = tasks[t];
    bnd_rows[2 * i] = bnd_rows[2 * i + 1] = nullptr;
    if (T.B.nnz <= 0) continue;
    const int64_t bi = i - bnd_off[t];
    const int N = T.B.order;
    const int32_t NB = nbs.nb[N];
    const int32_t nw = nbs.nw[N];
    // the starts of the item's waves
    for (int w = 0; w < nw; ++w) {
      int32_t key = int32_t(min(bi * int64_t(NB) + w * (NB / nw), int64_t(T.B.nnz) - 1));
      for (int m = N - 2; m >= 0; --m) {
        const int32_t x = search_le(T.B.pos[m + 1], 0, T.B.nodes[m] - 1, key);
        T.starts[(bi * nw + w) * (N - 1) + m] = x;
        key = x;
      }
    }
    // the item's first and last slice
    const int64_t p = bi * int64_t(NB);
    if (p >= T.B.nnz) continue;  // the boundary behind the last item
    const int32_t here = T.starts[bi * nw * (N - 1)];
    const int32_t back = root_of_position(T.B, int32_t(min(p + NB, int64_t(T.B.nnz)) - 1));
    auto row_of = [&](int32_t x) {
      return reinterpret_cast<float4*>(T.A + int64_t(T.B.crd0[x]) * R);
    };
    const int2 s = make_int2(slot_of_root(T.B, here, NB), slot_of_root(T.B, back, NB));
    T.slots[bi] = s;
    if (s.x == 2 * bi) bnd_rows[2 * i] = row_of(here);
    if (s.y == 2 * bi + 1) bnd_rows[2 * i + 1] = row_of(back);
  }
}

__global__ __launch_bounds__(256) void batch_rowbits_kernel(CsfDev B, uint32_t* __restrict__ bits) {
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t x = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; x < B.nodes[0]; x += nthr) {
    int32_t lo = int32_t(x), hi = int32_t(x) + 1;
    for (int m = 1; m < B.order; ++m) {
      lo = B.pos[m][lo];
      hi = B.pos[m][hi];
    }
    if (hi > lo) {
      const int32_t r = B.crd0[x];
      atomicOr(bits + (r >> 5), 1u << (r & 31));
    }
  }
}

// slots[b], rows[2 b], rows[2 b + 1] of the workgroups of one CSF, as
// batch_rows_kernel lists an item's (rows: output row, or -1).
__global__ __launch_bounds__(256) void shared_rows_kernel(CsfDev B, int32_t NB, int32_t nblk,
                                                          int2* __restrict__ slots,
                                                          int32_t* __restrict__ rows) {
  const int32_t b = int32_t(blockIdx.x * 256 + threadIdx.x);
  if (b >= nblk) return;
  const int64_t p = int64_t(b) * NB;
  const int32_t here = root_of_position(B, int32_t(p));
  const int32_t back = root_of_position(B, int32_t(min(p + NB, int64_t(B.nnz)) - 1));
  const int2 s = make_int2(slot_of_root(B, here, NB), slot_of_root(B, back, NB));
  slots[b] = s;
  rows[2 * b] = s.x == 2 * b ? B.crd0[here] : -1;
  rows[2 * b + 1] = s.y == 2 * b + 1 ? B.crd0[back] : -1;
}

// After an edge-parallel walk: a wave per 32 output rows zeroes those whose bit
// is clear (the walk stores the others), and waves write the shared rows, each
// row's columns on the smallest power of two of lanes, and zero them for the
// next call. In place of the fill of all of A before the walk.
__global__ __launch_bounds__(256) void edge_rows_kernel(const int32_t* __restrict__ rows, int32_t nrows,
                                                        double* __restrict__ W,
                                                        const uint32_t* __restrict__ bits, int32_t nbits,
                                                        float* __restrict__ A, int32_t a_rows, int R,
                                                        int lshift) {
  const int lane = int(threadIdx.x) & 63;
  const int32_t wave = int32_t(blockIdx.x * 4 + (threadIdx.x >> 6)), nwave = int32_t(gridDim.x * 4);
  const int32_t words = int32_t((int64_t(a_rows) + 31) / 32);
  const int per = 64 >> lshift, sub = lane >> lshift, c0 = lane & ((1 << lshift) - 1);
  // every load of a wave's first word, row number and column is in flight
  // before the first of them is waited for
  auto clear = [&](int32_t i) {  // the word's rows without a root node
    const int32_t left = a_rows - 32 * i;
    const uint32_t all = left >= 32 ? ~0u : (1u << left) - 1u;
    const int32_t known = nbits - 32 * i;  // rows from nbits on have none
    return known > 0 ? all & ~(known >= 32 ? bits[i] : bits[i] & ((1u << known) - 1u)) : all;
  };
  int64_t j = int64_t(wave) * per + sub;
  uint32_t none = wave < words ? clear(wave) : 0u;
  int32_t r = j < nrows ? rows[j] : -1;
  double w = j < nrows && c0 < R ? W[j * R + c0] : 0.0;
  for (int32_t i = wave; i < words;) {
    for (; none; none &= none - 1u) {
      float* row = A + (int64_t(32) * i + (__ffs(none) - 1)) * R;
      for (int c = lane; c < R; c += 64) row[c] = 0.f;
    }
    i += nwave;
    if (i < words) none = clear(i);
  }
  while (j < nrows) {
    if (r >= 0 && c0 < R) {
      for (int c = c0;;) {
        A[int64_t(r) * R + c] = float(w);
        W[j * R + c] = 0.0;
        c += 1 << lshift;
        if (c >= R) break;
        w = W[j * R + c];
      }
    }
    j += int64_t(nwave) * per;
    if (j < nrows) {
      r = rows[j];
      w = c0 < R ? W[j * R + c0] : 0.0;
    }
  }
}

// batch_rows_kernel over every task with one mode (bits), one launch.
int launch_batch_rows(const BatchLaunch& L, hipStream_t st, int mode) {
  if (L.ntasks <= 0) return TENTACO_OK;
  // the host prefix tables hold ntasks + 1 entries (the last is the total)
  const int64_t fill = L.h_fill_off[L.ntasks], bnd = L.h_bnd_off[L.ntasks];
  const int64_t fill_quads = (mode & kRowsFill) ? fill >> 2 : 0;
  const int qshift = L.R == 16 ? 2 : L.R == 32 ? 3 : 4;  // log2(R / 4), R in {16, 32, 64}
  const int64_t work = std::max<int64_t>(fill_quads, (mode & kRowsShared) ? bnd << (qshift + 1) : bnd);
  BatchNB nbs{};
  for (int N = 0; N <= kMaxOrder; ++N) {
    nbs.nb[N] = L.nb[N];
    nbs.nw[N] = std::max(1, L.blk[N] / 64);
  }
  batch_rows_kernel<<<grid_for(work, 256, 16384), 256, 0, st>>>(L.tasks, L.ntasks, L.fill_off, fill >> 2,
                                                                L.bnd_off, bnd, L.counter, nbs, L.R, qshift,
                                                                mode, L.bnd_rows, L.bnd_w);
  TT_HIP_CHECK(hipGetLastError());
  return TENTACO_OK;
}

// One launch for all orders up to kAllItems items a workgroup of it, and one
// per order beyond, on queues of their own: long batches keep every queue's
// workgroups busy, and there the orders' own register footprints count. us of a
// replay (retained outputs), 8 uneven tensors of 2 to 5 modes: R=32, 1 item a
// workgroup 120 and 149, 2 80 and 86, 7 347 and 377, 12 571 and 533, 32 1384
// and 1252; R=64: 10 473 and 490, 19 850 and 847, 48 2153 and 2050; R=16: 9 394
// and 437, 24 933 and 953.
constexpr int64_t kAllItems = 10;

int launch_batch_orders(const BatchLaunch& L, hipStream_t st) {
  int first = -1;
  bool one_schedule = true;
  for (int N = 2; N <= kMaxOrder; ++N) {
    if (L.grp_task[N + 1] <= L.grp_task[N]) continue;
    if (first < 0) first = N;
    one_schedule = one_schedule && L.sch[N] == L.sch[first];
  }
  if (first < 0) return TENTACO_OK;
  // the shared rows and (written outputs) the rows no launch stores
  auto rows = [&]() {
    return launch_batch_rows(L, st, L.retain ? kRowsShared : kRowsFill | kRowsShared);
  };
  int rc = TENTACO_OK;
  if (L.all_grid > 0 && one_schedule && L.total_items <= kAllItems * L.all_grid) {
    ktimer_begin(st);
    rc = all_orders_batch(L, L.blk[first], L.sch[first], st);
    if (rc) return rc;
    ktimer_end(st, "batch_kernel");
    return rows();
  }
  auto launch_order = [&](int N, hipStream_t s) -> int {
    switch (N) {
      case 2: return order_batch<2>(L, s);
      case 3: return order_batch<3>(L, s);
      case 4: return order_batch<4>(L, s);
      default: return order_batch<5>(L, s);
    }
  };
  // every order group's persistent launch at once, the group with the most
  // items on the launch stream and each other on its own stream (one after
  // another without those), so a group's tail overlaps the others' work
  int big = first;
  for (int N = first; N <= kMaxOrder; ++N)
    if (L.grp_item[N + 1] - L.grp_item[N] > L.grp_item[big + 1] - L.grp_item[big]) big = N;
  const bool conc = L.conc[0] != nullptr;
  auto beside = [&](int N) { return N != big && L.grp_task[N + 1] > L.grp_task[N]; };
  if (conc) TT_HIP_CHECK(hipEventRecord(L.cev[0], st));
  ktimer_begin(st);
  rc = launch_order(big, st);
  if (rc) return rc;
  for (int N = first; N <= kMaxOrder; ++N) {
    if (!beside(N)) continue;
    if (conc) TT_HIP_CHECK(hipStreamWaitEvent(L.conc[N], L.cev[0], 0));
    rc = launch_order(N, conc ? L.conc[N] : st);
    if (rc) return rc;
    if (conc) TT_HIP_CHECK(hipEventRecord(L.cev[N], L.conc[N]));
  }
  for (int N = first; conc && N <= kMaxOrder; ++N)
    if (beside(N)) TT_HIP_CHECK(hipStreamWaitEvent(st, L.cev[N], 0));
  ktimer_end(st, "batch_kernel");
  return rows();
}

}  // namespace

int launch_edge_prep(const CsfDev& B, float* Z, int64_t z_elems, int32_t* brk, int32_t nblk,
                     int32_t NB, hipStream_t st) {
  const int64_t work = std::max<int64_t>(z_elems / 4, int64_t(nblk) + 1);
  edge_prep_kernel<<<grid_for(work, 256, 16384), 256, 0, st>>>(B, Z, z_elems, brk, nblk, NB);
  TT_HIP_CHECK(hipGetLastError());
  return TENTACO_OK;
}

int launch_shared_rows(const CsfDev& B, int32_t NB, int2* slots, int32_t* rows, hipStream_t st) {
  const int32_t nblk = int32_t((int64_t(B.nnz) + NB - 1) / NB);
  shared_rows_kernel<<<(nblk + 255) / 256, 256, 0, st>>>(B, NB, nblk, slots, rows);
  TT_HIP_CHECK(hipGetLastError());
  return TENTACO_OK;
}

int launch_edge_rows(const WalkTables& wt, int32_t nblk, float* A, int32_t a_rows, int R, hipStream_t st) {
  int lshift = 0;
  while (lshift < 6 && (1 << lshift) < R) ++lshift;
  const int64_t waves = std::max<int64_t>((int64_t(a_rows) + 31) / 32, (2 * int64_t(nblk)) >> (6 - lshift));
  edge_rows_kernel<<<grid_for(waves, 4, 8192), 256, 0, st>>>(wt.rows, 2 * nblk, wt.W, wt.bits, wt.nbits, A,
                                                             a_rows, R, lshift);
  TT_HIP_CHECK(hipGetLastError());
  return TENTACO_OK;
}

int launch_narrow(const double* W, float* A, int64_t n, hipStream_t st) {
  narrow_kernel<<<grid_for(n / 2 + 1, 256, 16384), 256, 0, st>>>(W, A, n);
  TT_HIP_CHECK(hipGetLastError());
  return TENTACO_OK;
}

int launch_expand3(const CsfDev& B, int32_t* kq, int32_t* nzr, hipStream_t st) {
  if (B.order != 3) return fail(TENTACO_EINVAL, "expansion is for 3-mode tensors");
  const int64_t work = std::max<int64_t>(B.nodes[1], int64_t(B.nodes[0]) + 1);
  expand3_kernel<<<grid_for(work, 256, 16384), 256, 0, st>>>(B.pos[1], B.pos[2], B.crd[1],
                                                             B.nodes[0], B.nodes[1], kq, nzr);
  TT_HIP_CHECK(hipGetLastError());
  return TENTACO_OK;
}

int launch_pad3(const CsfDev& B, const int32_t* nzr, int32_t width, uint2* pad, hipStream_t st) {
  if (B.order != 3) return fail(TENTACO_EINVAL, "padded layout is for 3-mode tensors");
  const int64_t n = int64_t(B.nodes[0]) * width;
  pad3_fill_kernel<<<grid_for(n, 256, 16384), 256, 0, st>>>(pad, n);
  TT_HIP_CHECK(hipGetLastError());
  if (B.nodes[1] > 0) {
    pad3_build_kernel<<<grid_for(B.nodes[1], 256, 16384), 256, 0, st>>>(B, nzr, width, pad);
    TT_HIP_CHECK(hipGetLastError());
  }
  return TENTACO_OK;
}

int launch_pair3(const CsfDev& B, const int32_t* nzr, const int2* pairs, int32_t npairs,
                 uint2* slots, int4* info, hipStream_t st) {
  if (B.order != 3) return fail(TENTACO_EINVAL, "paired layout is for 3-mode tensors");
  if (npairs <= 0) return TENTACO_OK;
  const int64_t n = int64_t(npairs) * kPairSlots;
  pair3_build_kernel<<<grid_for(n, 256, 16384), 256, 0, st>>>(B, nzr, pairs, npairs, slots, info);
  TT_HIP_CHECK(hipGetLastError());
  return TENTACO_OK;
}

int warm_mttkrp_module(int order, hipStream_t st) {
  // no elements: the launches write nothing, they only load the code objects
  fill_kernel<<<1, 256, 0, st>>>(nullptr, 0, 0.f);
  TT_HIP_CHECK(hipGetLastError());
  switch (order) {
    case 2: return order_warm<2>(st);
    case 3: return order_warm<3>(st);
    case 4: return order_warm<4>(st);
    default: return order_warm<5>(st);
  }
}

int launch_fill(float* p, int64_t n, float value, hipStream_t st) {
  if (n <= 0) return TENTACO_OK;
  fill_kernel<<<grid_for(n / 4 + 1, 256, 16384), 256, 0, st>>>(p, n, value);
  TT_HIP_CHECK(hipGetLastError());
  return TENTACO_OK;
}

int launch_batch_rowbits(const CsfDev& B, uint32_t* bits, hipStream_t st) {
  if (B.nodes[0] <= 0) return TENTACO_OK;
  batch_rowbits_kernel<<<grid_for(B.nodes[0], 256, 8192), 256, 0, st>>>(B, bits);
  TT_HIP_CHECK(hipGetLastError());
  return TENTACO_OK;
}

int launch_batch_brackets(const BatchLaunch& L, hipStream_t st) {
  return launch_batch_rows(L, st, kRowsList);
}

int launch_batch_zero_outputs(const BatchLaunch& L, hipStream_t st) {
  return launch_batch_rows(L, st, kRowsFill | kRowsShared);
}

int launch_batch(const BatchLaunch& L, hipStream_t st) {
  if (L.R != 16 && L.R != 32 && L.R != 64)
    return fail(TENTACO_EUNSUPPORTED, "batched launch supports R in {16,32,64}");
  return launch_batch_orders(L, st);
}

int batch_all_occupancy(int block, int R, int* per_cu) { return all_orders_batch_occupancy(block, R, per_cu); }

int batch_occupancy(int family, int block, int R, int32_t NB, int order, int* per_cu) {
  if (R != 16 && R != 32 && R != 64)
    return fail(TENTACO_EUNSUPPORTED, "batched launch supports R in {16,32,64}");
  switch (order) {
    case 2: return order_batch_occupancy<2>(family, block, R, NB, per_cu);
    case 3: return order_batch_occupancy<3>(family, block, R, NB, per_cu);
    case 4: return order_batch_occupancy<4>(family, block, R, NB, per_cu);
    default: return order_batch_occupancy<5>(family, block, R, NB, per_cu);
  }
}

Variant variant_of(int v) {
  constexpr int per_family = kNumGridBlocks * kNumGridGroups;
  if (v < 0 || v >= kNumVariants) return Variant{-1, 0, 0};
  if (v < 2 * per_family) {
    const int fam = v / per_family;
    const int r = v % per_family;
    return Variant{fam, kGridBlocks[r / kNumGridGroups], kGridGroups[r % kNumGridGroups]};
  }
  return Variant{kSliceRow, kGridBlocks[v - 2 * per_family], 0};
}

int default_variant() {
  // eb_sr at block 512, 4 nonzeros per group: the TACO schedule of
  // mttkrp3_csf_gpu_taco.h:179-207
  return 0 * (kNumGridBlocks * kNumGridGroups) + 2 * kNumGridGroups + 0;
}

int auto_variant(const CsfStats& s, int order, int R) {
  constexpr int per_family = kNumGridBlocks * kNumGridGroups;
  auto edge = [&](int family, int bi, int gi) {
    return family * per_family + bi * kNumGridGroups + gi;
  };
  // slice-row pays off when there are enough non-empty slices to fill the
  // chip and no slice dominates (the longest is within 8x of the mean)
  if (s.nonempty_slices >= 2048 && s.nnz > 0) {
    const double mean = double(s.nnz) / s.nonempty_slices;
    if (double(s.max_slice_nnz) <= 8.0 * mean) return 2 * per_family + 1;  // sr_b256
  }
  // Otherwise edge-parallel, 256 threads x group 16 below 300k nonzeros and
  // 512 x 64 from there: over the 2,600 swept tensors of the selector's
  // training set this split is 1.31x the sweep's best (geometric mean),
  // against 10.9x for edge-serial 256 x 16. Tiles over the LDS limit at this
  // order and rank step down.
  const int picks[3] = {s.nnz < 300000 ? edge(1, 1, 2) : edge(1, 2, 4),  // ep_b256_g16 / ep_b512_g64
                        edge(1, 1, 2),                                    // ep_b256_g16
                        edge(0, 1, 2)};                                   // es_b256_g16
  for (int v : picks)
    if (variant_fits(order, R, v)) return v;
  return 2 * per_family + 1;  // sr_b256 (always fits)
}

Variant auto_tile(const CsfStats& s, int order, int R, bool paired) {
  const Variant vr = variant_of(auto_variant(s, order, R));
  if (vr.family == kSliceRow) {
    // 3-mode short fibres (the kernels over the expansion): the paired layout
    // where it exists; else whole slices by the wave below 12 nonzeros a
    // slice, one wave a slice up to 48 and two from there. Against the
    // variant's 256 threads, us at rank 32 / 50: mean 8 nonzeros 49 -> 13 /
    // 80 -> 21, mean 30 27 -> 15 / 46 -> 26, mean 60 15 -> 12 / 28 -> 21
    if (order != 3 || s.nnz <= 0 || s.child_mean[2] > 1.25) return vr;
    if (paired && (R == 16 || R == 32 || R == 64)) return vr;
    const double mean = double(s.nnz) / std::max(s.nonempty_slices, 1);
    if (mean < 12.0) return Variant{kSliceRow, vr.block, s.nnz < 500000 ? 64 : 128};
    return Variant{kSliceRow, mean <= 48.0 ? 64 : 128, 0};
  }
  if (vr.family != kEdgeParallel) return vr;
  // A wave's run of nonzeros is a serial chain, so up to about 3000 runs in
  // all (12 waves per CU) shorter runs are faster; beyond that more runs only
  // add each one's start and end. Runs hold 32 to 512 nonzeros, in 512-thread
  // workgroups below 300k nonzeros (fewer workgroups to combine) and 256 from
  // there. From 30M nonzeros on 512 threads and runs of 256 are 3-6% faster than
  // 256 and 512 (3-mode, rank 32, us of both: 30M 584 and 601, 45M 899 and 946, 60M
  // 1246 and 1327; 4-mode 30M, rank 64 1216 and 1250; 40M, rank 16 672 and 705), at
  // 20M 1 to 3% (403 and 415; rank 64 831 and 843), at 13M the same (244). Over
  // 60 tensors drawn from 10k to 12.6M nonzeros, orders 3-5, ranks 7-128, the
  // sizes are 1.08x the sweep's best edge-parallel tile (geometric mean); the
  // variants' own (256 x 16 and 512 x 64) are 1.33x.
  const int groups = 64 / lanes_per_row(R);
  const bool large = s.nnz >= 30000000;
  const int64_t want = std::max<int64_t>(32, std::min<int64_t>(large ? 256 : 512, s.nnz / 3000));
  Variant t{kEdgeParallel, s.nnz < 300000 || large ? 512 : 256, 4};
  while (t.group < 64 && int64_t(groups) * t.group * 3 / 2 <= want) t.group *= 2;
  return edge_tile_fits(order, R, t) ? t : vr;
}

bool auto_needs_rows(const CsfStats& s, int R, const Variant& tile, const Variant& v) {
  // From 300k nonzeros on the sized tile has 2 to 8 times the variant's
  // workgroups, whose FP32 additions to a long slice's row had 1.3 to 1.6 times
  // the error of the variant's tile before the walk (400k nonzeros 2.0 and
  // 1.4e-7 against FP64, 1.5M 5-mode 2.3 and 1.5, at rank 64 3.6 and 2.5; with
  // FP64 rows 1.0, 1.2 and 1.5). Below, it has no more error than that tile
  // had but for a tenth in one of seven (12 seeds each: 1.12 and 1.17e-7 at 10k,
  // 1.25 and 1.15 at 120k, 4-mode, 1.97 and 2.03 at 200k, 5-mode, 1.02 and 1.20 at
  // 290k), and the rows' kernel would be 4 of 11 us.
  return tile.family == kEdgeParallel && v.family == kEdgeParallel && s.nnz >= 300000 &&
         nnz_per_block(tile, R) < nnz_per_block(v, R);
}

int batch_group(int64_t nnz, int R) {
  // runs of 512 nonzeros a wave from 4M nonzeros in all, 256 below: at 256
  // threads, 19.6M nonzeros, rank 32: group 64 547 us a replay, 16 669; 1.26M:
  // 32 88, 64 103, 16 91; 19.6M, rank 16: 32 445, 64 542, 16 488
  const int groups = 64 / lanes_per_row(R);
  return std::min(64, (nnz >= 4000000 ? 512 : 256) / groups);
}

int lanes_per_row(int R) {
  return with_rank_layout(R, [](auto r) { return Lay<r()>::LPR; });
}

int64_t nnz_per_block(const Variant& vr, int R) {
  return int64_t(vr.block / lanes_per_row(R)) * vr.group;
}

bool edge_tile_fits(int order, int R, const Variant& vr) {
  constexpr int kUpperNodes = 256, kLeafNodes = 1024;
  const int64_t leaf = std::min<int64_t>(nnz_per_block(vr, R) + 1, kLeafNodes);
  const int64_t brackets = 4 * (2 * leaf + 1 + int64_t(order - 2) * (2 * kUpperNodes + 1));
  const int64_t rows = 2 * (vr.block / lanes_per_row(R));
  return brackets + (vr.family == kEdgeParallel ? rows * 4 * (R + 1) : 0) <= 65536;
}

bool variant_fits(int order, int R, int v) {
  const Variant vr = variant_of(v);
  if (vr.family < 0 || R <= 0) return false;
  return vr.family == kSliceRow || edge_tile_fits(order, R, vr);
}

int64_t nnz_per_wave(const Variant& vr, int R) {
  return int64_t(64 / lanes_per_row(R)) * vr.group;
}

int launch_walk_starts(const CsfDev& B, int64_t wn, int32_t* starts, hipStream_t st) {
  // the brackets of runs of wn nonzeros (one entry past the last run too)
  const int64_t runs = (int64_t(B.nnz) + wn - 1) / wn;
  return launch_edge_prep(B, nullptr, 0, starts, int32_t(runs), int32_t(wn), st);
}

size_t edge_brk_bytes(const CsfDev& B, int64_t NB) {
  const int64_t nblk = (int64_t(B.nnz) + NB - 1) / NB;
  const size_t bytes = size_t(nblk + 1) * size_t(B.order - 1) * sizeof(int32_t);
  return (bytes + 255) / 256 * 256;
}

size_t mttkrp_workspace_bytes(const CsfDev& B, int R, const Variant& vr, int32_t a_rows) {
  if (vr.family == kSliceRow || vr.family < 0) return 0;
  const size_t brk = edge_brk_bytes(B, nnz_per_block(vr, R));
  if (vr.family != kEdgeSerial) return brk;
  return brk + size_t(std::max<int32_t>(a_rows, 0)) * size_t(R) * sizeof(double);
}

int launch_mttkrp_level(const CsfDev& B, const FactorsDev& F, int level, int R, float* A,
                        int32_t a_rows, hipStream_t st) {
  if (R <= 0 || R > kMaxRankAny)
    return fail(TENTACO_EUNSUPPORTED, "rank R=%d outside 1..%d", R, kMaxRankAny);
  switch (B.order) {
    case 2: return order_level<2>(B, F, level, R, A, a_rows, st);
    case 3: return order_level<3>(B, F, level, R, A, a_rows, st);
    case 4: return order_level<4>(B, F, level, R, A, a_rows, st);
    case 5: return order_level<5>(B, F, level, R, A, a_rows, st);
    default: return fail(TENTACO_EUNSUPPORTED, "order %d outside 2..5", B.order);
  }
}

int launch_mttkrp(const CsfDev& B, const FactorsDev& F, int R, float* A,
                  int32_t a_rows, bool dense_root, const Variant& vr, void* ws,
                  const WalkTables& tables, hipStream_t st) {
  if (R <= 0 || R > kMaxRankAny)
    return fail(TENTACO_EUNSUPPORTED, "rank R=%d outside 1..%d", R, kMaxRankAny);
  if (vr.family < 0) return fail(TENTACO_EINVAL, "invalid variant");
  switch (B.order) {
    case 2: return order_mttkrp<2>(B, F, R, A, a_rows, dense_root, vr, ws, tables, st);
    case 3: return order_mttkrp<3>(B, F, R, A, a_rows, dense_root, vr, ws, tables, st);
    case 4: return order_mttkrp<4>(B, F, R, A, a_rows, dense_root, vr, ws, tables, st);
    case 5: return order_mttkrp<5>(B, F, R, A, a_rows, dense_root, vr, ws, tables, st);
    default: return fail(TENTACO_EUNSUPPORTED, "order %d outside 2..5", B.order);
  }
}

}  // namespace tt
