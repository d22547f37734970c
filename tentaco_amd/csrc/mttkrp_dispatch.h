// What the MTTKRP host code (mttkrp.hip) and the per-order kernel sources
// (mttkrp_order.h, mttkrp_o<N>.hip) call of each other.
#pragma once

#include "internal.h"

namespace tt {

inline int grid_for(int64_t work, int block, int cap) {
  int64_t g = (work + block - 1) / block;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return int(g);
}

// Whether the variant table offers an edge tile at this order and rank: the
// table's limit is 64 KB of node brackets and, for the edge-parallel family,
// of two rows per row group (what a tile of that size once staged in LDS).
// The walk itself needs less and takes every tile.
bool edge_tile_fits(int order, int R, const Variant& vr);

__device__ __forceinline__ int32_t upper_index(const int64_t* __restrict__ off, int32_t n,
                                               int64_t key) {
  // largest t in [0, n) with off[t] <= key
  int32_t lo = 0, hi = n - 1;
  while (lo < hi) {
    const int32_t mid = lo + ((hi - lo + 1) >> 1);
    if (off[mid] <= key) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Defined per order N in mttkrp_o<N>.hip; the public launches of internal.h
// pick the order. (order_warm: an empty launch, which loads the code object.)
template <int N>
int order_warm(hipStream_t st);
template <int N>
int order_mttkrp(const CsfDev& B, const FactorsDev& F, int R, float* A, int32_t a_rows,
                 bool dense_root, const Variant& vr, void* ws, const WalkTables& wt,
                 hipStream_t st);
template <int N>
int order_level(const CsfDev& B, const FactorsDev& F, int level, int R, float* A, int32_t a_rows,
                hipStream_t st);
template <int N>
int order_batch(const BatchLaunch& L, hipStream_t st);
template <int N>
int order_batch_occupancy(int family, int block, int R, int32_t NB, int* per_cu);
// Every order's items in one launch (mttkrp_batch.hip); all orders run blocks
// of one size with one schedule.
int all_orders_batch(const BatchLaunch& L, int block, int schedule, hipStream_t st);
int all_orders_batch_occupancy(int block, int R, int* per_cu);

// Defined in mttkrp.hip: zero z_elems floats of Z and write the brackets of
// nblk blocks of NB nonzeros; A = FP32(W) over n elements.
int launch_edge_prep(const CsfDev& B, float* Z, int64_t z_elems, int32_t* brk, int32_t nblk,
                     int32_t NB, hipStream_t st);
int launch_narrow(const double* W, float* A, int64_t n, hipStream_t st);
// After an edge-parallel walk over nblk workgroups with shared rows: write them
// (and zero them for the next call) and zero the rows that no root node writes.
int launch_edge_rows(const WalkTables& wt, int32_t nblk, float* A, int32_t a_rows, int R, hipStream_t st);

}  // namespace tt
