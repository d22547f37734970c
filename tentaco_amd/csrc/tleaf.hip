// Per-handle transposed indexes of the levels of a CSF, for the MTTKRP of a
// non-root mode on a CSF rooted at another mode without atomics, and the
// leaf-level kernel.
//
//   A_L(j,:) = sum over nonzeros with level-L coordinate j of
//              val * prod_{m != L} M_m(coordinate at level m, :)
//
// The index of level L, built once from B alone by a stable radix sort of
// the level's coordinates: tpos[j] is the first entry of coordinate j
// (dims[L] + 1 entries), entries in CSF order within a coordinate.
//  * Leaf level (L = N-1): entry t is (its level N-2 node, its value bits),
//    and anc[p] holds the coordinates at levels 0..N-2 of level N-2 node p:
//    8 bytes per nonzero plus 4 (N-1) bytes per level N-2 node.
//  * Inner level: entry t is a level-L node, and anc[y] holds the
//    coordinates at levels 0..L-1 of node y: 4 (L+1) bytes per level-L
//    node. Its kernel (inner_kernel, with the other subtree walks) adds, per
//    node, its ancestors' row product times the sum of its subtree.
// Leaf kernel: one workgroup of 1-4 waves computes one output row: lanes
// load 64 entries at a time, row groups take them by shuffles and gather
// the N-1 ancestor rows of each, and the row is reduced over the wave and
// the workgroup and stored once. Every output row is written exactly once
// (rows without nonzeros as zero), with no atomics, so results are bitwise
// reproducible.

#include <algorithm>
#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>

#include "internal.h"
#include "rowops.h"

namespace tt {
namespace {

// fib[q] = the level N-2 node holding nonzero q
__global__ __launch_bounds__(256) void tl_fib_kernel(const int32_t* __restrict__ pos, int32_t nf,
                                                     int32_t* __restrict__ fib) {
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; p < nf; p += nthr)
    for (int32_t q = pos[p]; q < pos[p + 1]; ++q) fib[q] = int32_t(p);
}

// anc[p * cnt + m] = coordinate at level m (m < cnt) of the ancestor of node
// p at level `lev` (the node itself at m == lev, when cnt > lev)
__global__ __launch_bounds__(256) void tl_anc_kernel(CsfDev B, int lev, int cnt,
                                                     int32_t* __restrict__ anc) {
  const int32_t n = B.nodes[lev];
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; p < n; p += nthr) {
    int32_t x = int32_t(p);
    for (int m = lev; m >= 1; --m) {
      if (m < cnt) anc[p * cnt + m] = B.crd[m][x];
      x = search_le(B.pos[m], 0, B.nodes[m - 1] - 1, x);
    }
    anc[p * cnt] = B.crd0[x];
  }
}

__global__ __launch_bounds__(256) void tl_iota_kernel(int32_t* __restrict__ v, int32_t n) {
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += nthr)
    v[i] = int32_t(i);
}

// tpos[j] = first t with key[t] >= j, j = 0..dim
__global__ __launch_bounds__(256) void tl_tpos_kernel(const int32_t* __restrict__ key, int32_t n,
                                                      int32_t dim, int32_t* __restrict__ tpos) {
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t j = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; j <= dim; j += nthr) {
    int32_t lo = 0, hi = n;
    while (lo < hi) {
      const int32_t mid = lo + ((hi - lo) >> 1);
      if (key[mid] < j) lo = mid + 1;
      else hi = mid;
    }
    tpos[j] = lo;
  }
}

__global__ __launch_bounds__(256) void tl_ent_kernel(const int32_t* __restrict__ order,
                                                     const int32_t* __restrict__ fib,
                                                     const float* __restrict__ vals, int32_t n,
                                                     uint2* __restrict__ ent) {
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; t < n; t += nthr) {
    const int32_t q = order[t];
    ent[t] = make_uint2(uint32_t(fib[q]), __float_as_uint(vals[q]));
  }
}

// Entries whose ancestor rows are in flight at once per row group: about 64
// VGPRs of rows, a power of two so that the batches tile the group's
// 64 / (64 / LPR) entries of a chunk exactly.
template <int N, int R>
constexpr int tl_batch() {
  constexpr int per = (N - 1) * Row<R>::NV * (R == 0 ? 1 : 4);
  constexpr int nt = 64 / (64 / Row<R>::LPR);
  int b = 1;
  while (2 * b * per <= 64 && 2 * b <= nt) b *= 2;
  return b;
}

template <int N, int R>
__global__ __launch_bounds__(256) void tleaf_kernel(const int32_t* __restrict__ tpos, int32_t tdim,
                                                    const uint2* __restrict__ ent,
                                                    const int32_t* __restrict__ anc, FactorsDev F,
                                                    float* __restrict__ A, int Rr) {
  using RO = Row<R>;
  using V = typename RO::V;
  constexpr int NV = RO::NV;
  constexpr int LPR = RO::LPR;
  constexpr int NG = 64 / LPR;
  constexpr int NT = 64 / NG;
  constexpr int TB = tl_batch<N, R>();
  static_assert(NT % TB == 0, "batches tile a chunk");
  __shared__ __align__(16) float red[4][Lay<R>::kMaxRank];
  const int32_t j = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  const int nwv = blockDim.x >> 6;
  const int gi = lane / LPR;
  const int c = lane % LPR;
  V acc[NV];
  RO::zero(acc);
  if (j < tdim) {
    const int32_t t0 = tpos[j];
    const int32_t t1 = tpos[j + 1];
    for (int32_t base = t0 + 64 * wv; base < t1; base += 64 * nwv) {
      const int32_t t = base + lane;
      const uint2 e = t < t1 ? ent[t] : make_uint2(0u, 0u);
#pragma unroll
      for (int u0 = 0; u0 < NT; u0 += TB) {
        V rows[TB][N - 1][NV];
        float vt[TB];
#pragma unroll
        for (int u = 0; u < TB; ++u) {
          // every lane runs both shuffles (a shuffle inside a branch would
          // read inactive source lanes as zero)
          const int src = (u0 + u) * NG + gi;
          const uint32_t p = __shfl(e.x, src);
          const float v = __uint_as_float(__shfl(e.y, src));
          const bool ok = base + src < t1;
          vt[u] = ok ? v : 0.f;
          const int32_t* a = anc + int64_t(ok ? p : 0u) * (N - 1);
#pragma unroll
          for (int m = 0; m < N - 1; ++m) RO::load(rows[u][m], F.M[m], a[m], c, Rr);
        }
#pragma unroll
        for (int u = 0; u < TB; ++u) {
#pragma unroll
          for (int m = 1; m < N - 1; ++m) RO::hmul(rows[u][0], rows[u][m]);
          RO::axpy(acc, vt[u], rows[u][0]);
        }
      }
    }
  }
  RO::wave_sum(acc);
  if (nwv == 1) {
    if (gi == 0) RO::store(A, j, c, Rr, acc);
    return;
  }
  if (gi == 0) {
    RO::put(red[wv], c, acc);
  }
  __syncthreads();
  if (wv == 0 && gi == 0) {
    for (int w = 1; w < nwv; ++w) {
      V o[NV];
      RO::get(red[w], c, o);
      RO::add(acc, o);
    }
    RO::store(A, j, c, Rr, acc);
  }
}

int grid_of(int64_t work) {
  int64_t g = (work + 255) / 256;
  return int(std::max<int64_t>(1, std::min<int64_t>(g, 16384)));
}

template <int N, int R>
int launch_tleaf_typed(const CsfDev& B, const LevelIndex& X, const FactorsDev& F, int Rr, float* A,
                       int32_t a_rows, hipStream_t st) {
  if (a_rows <= 0) return TENTACO_OK;
  // 1-4 waves per row, from the mean entries per row
  const int64_t mean = (int64_t(B.nnz) + X.dim - 1) / std::max<int32_t>(X.dim, 1);
  const int nwv = int(std::max<int64_t>(1, std::min<int64_t>(4, (mean + 255) / 256)));
  ktimer_begin(st);
  tleaf_kernel<N, R><<<a_rows, 64 * nwv, 0, st>>>(X.tpos, X.dim, X.ent, X.anc, F, A, Rr);
  TT_HIP_CHECK(hipGetLastError());
  ktimer_end(st, "tleaf_kernel");
  return TENTACO_OK;
}

template <int R>
int launch_tleaf_rank(const CsfDev& B, const LevelIndex& X, const FactorsDev& F, int Rr, float* A,
                      int32_t a_rows, hipStream_t st) {
  switch (B.order) {
    case 2: return launch_tleaf_typed<2, R>(B, X, F, Rr, A, a_rows, st);
    case 3: return launch_tleaf_typed<3, R>(B, X, F, Rr, A, a_rows, st);
    case 4: return launch_tleaf_typed<4, R>(B, X, F, Rr, A, a_rows, st);
    case 5: return launch_tleaf_typed<5, R>(B, X, F, Rr, A, a_rows, st);
    default: return fail(TENTACO_EUNSUPPORTED, "order %d outside 2..5", B.order);
  }
}

}  // namespace

void free_level_index(LevelIndex* X) {
  (void)hipFree(X->mem);
  *X = LevelIndex{};
}

int build_level_index(const CsfDev& B, int level, int32_t dim, LevelIndex* X, hipStream_t st) {
  free_level_index(X);
  const int N = B.order;
  if (level < 1 || level >= N) return fail(TENTACO_EINVAL, "level index: level %d", level);
  if (dim <= 0) return fail(TENTACO_EINVAL, "level index: dimension %d", dim);
  const bool leaf = level == N - 1;
  const int32_t n = B.nodes[level];                  // entries: the level's nodes
  const int anc_lev = leaf ? N - 2 : level;          // nodes the ancestor table is over
  const int cnt = leaf ? N - 1 : level;              // coordinates per such node
  const int32_t na = B.nodes[anc_lev];
  auto al = [](size_t x) { return (x + 255) & ~size_t(255); };
  const size_t b_tpos = al(sizeof(int32_t) * (size_t(dim) + 1));
  const size_t b_ent = al((leaf ? sizeof(uint2) : sizeof(int32_t)) * std::max<size_t>(n, 1));
  const size_t b_anc = al(sizeof(int32_t) * std::max<size_t>(size_t(na) * cnt, 1));
  void* mem = nullptr;
  if (hipMalloc(&mem, b_tpos + b_ent + b_anc) != hipSuccess)
    return fail(TENTACO_ENOMEM, "level index: hipMalloc of %zu bytes failed", b_tpos + b_ent + b_anc);
  X->mem = mem;
  X->level = level;
  X->tpos = static_cast<int32_t*>(mem);
  if (leaf) X->ent = reinterpret_cast<uint2*>(static_cast<char*>(mem) + b_tpos);
  else X->node = reinterpret_cast<int32_t*>(static_cast<char*>(mem) + b_tpos);
  X->anc = reinterpret_cast<int32_t*>(static_cast<char*>(mem) + b_tpos + b_ent);
  X->dim = dim;
  // temporaries: (leaf) the level N-2 node of every nonzero, the sort's
  // values in and out, its keys out, and its workspace
  const size_t b_n = al(sizeof(int32_t) * std::max<size_t>(n, 1));
  int end_bit = 1;
  while (end_bit < 31 && (int64_t(1) << end_bit) < int64_t(dim)) ++end_bit;
  size_t sort_bytes = 0;
  if (n > 0 &&
      rocprim::radix_sort_pairs(nullptr, sort_bytes, static_cast<const int32_t*>(nullptr),
                                static_cast<int32_t*>(nullptr), static_cast<const int32_t*>(nullptr),
                                static_cast<int32_t*>(nullptr), size_t(n), 0, end_bit, st) !=
          hipSuccess) {
    free_level_index(X);
    return fail(TENTACO_EHIP, "level index: sort size query failed");
  }
  void* tmp = nullptr;
  if (hipMalloc(&tmp, 4 * b_n + al(std::max<size_t>(sort_bytes, 1))) != hipSuccess) {
    free_level_index(X);
    return fail(TENTACO_ENOMEM, "level index: temporary allocation failed");
  }
  int32_t* fib = static_cast<int32_t*>(tmp);
  int32_t* ord_in = reinterpret_cast<int32_t*>(static_cast<char*>(tmp) + b_n);
  int32_t* ord = leaf ? reinterpret_cast<int32_t*>(static_cast<char*>(tmp) + 2 * b_n) : X->node;
  int32_t* key = reinterpret_cast<int32_t*>(static_cast<char*>(tmp) + 3 * b_n);
  void* sort_tmp = static_cast<char*>(tmp) + 4 * b_n;
  int rc = TENTACO_OK;
  if (na > 0) {
    tl_anc_kernel<<<grid_of(na), 256, 0, st>>>(B, anc_lev, cnt, X->anc);
    if (hipGetLastError() != hipSuccess) rc = fail(TENTACO_EHIP, "level index: anc launch failed");
  }
  if (!rc && n > 0) {
    if (leaf) tl_fib_kernel<<<grid_of(na), 256, 0, st>>>(B.pos[N - 1], na, fib);
    tl_iota_kernel<<<grid_of(n), 256, 0, st>>>(ord_in, n);
    if (hipGetLastError() != hipSuccess) rc = fail(TENTACO_EHIP, "level index: launch failed");
    // stable: equal coordinates keep CSF order
    if (!rc && rocprim::radix_sort_pairs(sort_tmp, sort_bytes, B.crd[level], key,
                                         static_cast<const int32_t*>(ord_in), ord, size_t(n), 0,
                                         end_bit, st) != hipSuccess)
      rc = fail(TENTACO_EHIP, "level index: sort failed");
    if (!rc && leaf) {
      tl_ent_kernel<<<grid_of(n), 256, 0, st>>>(ord, fib, B.vals, n, X->ent);
      if (hipGetLastError() != hipSuccess) rc = fail(TENTACO_EHIP, "level index: launch failed");
    }
  }
  if (!rc) {
    tl_tpos_kernel<<<grid_of(int64_t(dim) + 1), 256, 0, st>>>(key, n, dim, X->tpos);
    if (hipGetLastError() != hipSuccess) rc = fail(TENTACO_EHIP, "level index: launch failed");
  }
  const hipError_t e = hipStreamSynchronize(st);
  (void)hipFree(tmp);
  if (!rc && e != hipSuccess) rc = fail(TENTACO_EHIP, "level index build: %s", hipGetErrorString(e));
  if (rc) {
    free_level_index(X);
    return rc;
  }
  X->built = true;
  return TENTACO_OK;
}

int launch_mttkrp_leaf(const CsfDev& B, const LevelIndex& X, const FactorsDev& F, int R, float* A,
                       int32_t a_rows, hipStream_t st) {
  if (!X.built || X.level != B.order - 1 || !X.ent)
    return fail(TENTACO_EINVAL, "leaf index not built");
  if (R <= 0 || R > kMaxRankAny)
    return fail(TENTACO_EUNSUPPORTED, "rank R=%d outside 1..%d", R, kMaxRankAny);
  return with_rank_layout(
      R, [&](auto r) { return launch_tleaf_rank<r()>(B, X, F, R, A, a_rows, st); });
}

}  // namespace tt
