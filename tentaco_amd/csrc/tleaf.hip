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
//  * Leaf level (L = N-1): up to order 3 entry t is the nonzero's coordinates
//    at levels 0..N-2 and its value: 4 N bytes per nonzero. From order 4 it is
//    (its level N-2 node, its value bits), and anc[p] holds the coordinates
//    at levels 0..N-2 of level N-2 node p: 8 bytes per nonzero plus 4 (N-1)
//    bytes per level N-2 node. (The node costs a random line per entry; at
//    order 3 that was a third of the lines, and the coordinates cost 4 bytes
//    more than the node. 20M nonzeros, rank 32: 604 us against 275.)
//  * Inner level: the entries are the level N-2 nodes (the nonzeros' parents)
//    by the coordinate of their ancestor at level L: each the node's range of
//    nonzeros and its coordinates at the other levels 0..N-2: 4 N bytes per
//    level N-2 node. Its kernel walks the row's nonzeros as one list
//    (inner_leaf_kernel).
// Leaf kernel: one workgroup of 1-8 waves computes one output row: lanes
// load 64 entries at a time, row groups take them by shuffles and gather
// the N-1 ancestor rows of each, and the row is reduced over the wave and
// the workgroup and stored once. Every output row is written exactly once
// (rows without nonzeros as zero), with no atomics, so results are bitwise
// reproducible.

#include <algorithm>
#include <cfloat>
#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>

#include "index_range.h"
#include "internal.h"
#include "rowops.h"

namespace tt {
namespace {

// LDS per wave of inner_leaf_kernel: a record per nonzero of the chunk, the
// histogram, the ancestor products.
constexpr size_t kInnerLeafLds = 64 * 16 + 64 * 4 + 4096;

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

// A leaf entry up to order 3.
template <int N>
struct LeafEnt {
  int32_t c[N - 1];
  float v;
};

template <int N>
__global__ __launch_bounds__(256) void tl_coord_kernel(const int32_t* __restrict__ order,
                                                       const int32_t* __restrict__ fib,
                                                       const int32_t* __restrict__ anc,
                                                       const float* __restrict__ vals, int32_t n,
                                                       LeafEnt<N>* __restrict__ ent) {
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; t < n; t += nthr) {
    const int32_t q = order[t];
    const int64_t p = fib[q];
    LeafEnt<N> e;
#pragma unroll
    for (int m = 0; m < N - 1; ++m) e.c[m] = anc[p * (N - 1) + m];
    e.v = vals[q];
    ent[t] = e;
  }
}

// key[p] = coordinate at `level` above level N-2 node p (w = N-1 per node in anc)
__global__ __launch_bounds__(256) void tl_key_kernel(const int32_t* __restrict__ anc, int w,
                                                     int level, int32_t n,
                                                     int32_t* __restrict__ key) {
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; p < n; p += nthr)
    key[p] = anc[p * w + level];
}

// Entry t of an inner level: the node's nonzeros [range[t], range[n + t]) and
// its coordinates at the other levels, cor[i * n + t] for the i-th of them.
__global__ __launch_bounds__(256) void tl_range_kernel(const int32_t* __restrict__ order,
                                                       const int32_t* __restrict__ pos,
                                                       const int32_t* __restrict__ anc, int w,
                                                       int level, int32_t n,
                                                       int32_t* __restrict__ range,
                                                       int32_t* __restrict__ cor) {
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; t < n; t += nthr) {
    const int64_t p = order[t];
    range[t] = pos[p];
    range[index_end(n, int32_t(t))] = pos[p + 1];
    for (int m = 0, i = 0; m < w; ++m)
      if (m != level) cor[int64_t(i++) * n + t] = anc[p * w + m];
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
__global__ __launch_bounds__(512) void tleaf_kernel(const int32_t* __restrict__ tpos, int32_t tdim,
                                                    const void* __restrict__ entries,
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
  constexpr bool kCoords = N <= 3;
  __shared__ __align__(16) float red[8][Lay<R>::kMaxRank];
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
    const uint32_t step = 64 * nwv;
    const uint32_t end = uint32_t(t1);  // (unsigned: the bases below may pass 2^31 - 1)
    // An entry's coordinates and value arrive one chunk ahead, a lane each;
    // where they are its level N-2 node's, the node two chunks ahead.
    uint2 raw = make_uint2(0u, 0u);
    auto node_of = [&](uint32_t base) {
      if constexpr (!kCoords) {
        const int32_t t = index_ahead(int32_t(base), lane, t1 - 1);
        raw = static_cast<const uint2*>(entries)[t];
      }
    };
    auto coords_of = [&](uint32_t base) {
      LeafEnt<N> e;
      if constexpr (kCoords) {
        e = static_cast<const LeafEnt<N>*>(entries)[index_ahead(int32_t(base), lane, t1 - 1)];
      } else {
        const int32_t* a = anc + int64_t(raw.x) * (N - 1);
#pragma unroll
        for (int m = 0; m < N - 1; ++m) e.c[m] = a[m];
        e.v = __uint_as_float(raw.y);
      }
      return e;
    };
    const uint32_t b0 = uint32_t(t0) + 64 * wv;
    LeafEnt<N> e{}, next{};
    if (b0 < end) {
      node_of(b0);
      next = coords_of(b0);
      if (b0 + step < end) node_of(b0 + step);
    }
    for (uint32_t base = b0; base < end; base += step) {
      e = next;
      if (base + step < end) {
        next = coords_of(base + step);
        if (base + 2 * step < end) node_of(base + 2 * step);
      }
#pragma unroll
      for (int u0 = 0; u0 < NT; u0 += TB) {
        if (base + u0 * NG >= end) break;
        V rows[TB][N - 1][NV];
        float vt[TB];
#pragma unroll
        for (int u = 0; u < TB; ++u) {
          // every lane runs the shuffles (a shuffle inside a branch would
          // read inactive source lanes as zero)
          const int src = (u0 + u) * NG + gi;
          vt[u] = __shfl(e.v, src);
#pragma unroll
          for (int m = 0; m < N - 1; ++m)
            RO::load(rows[u][m], F.M[m], __shfl(e.c[m], src), c, Rr);
        }
#pragma unroll
        for (int u = 0; u < TB; ++u) {
#pragma unroll
          for (int m = 1; m < N - 1; ++m) RO::hmul(rows[u][0], rows[u][m]);
          // (a lane past the entries repeats the last one)
          RO::axpy_if(base + (u0 + u) * NG + gi < end, acc, vt[u], rows[u][0]);
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

// MTTKRP of an inner level through its index: A(j,:) sums, over the row's
// entries (level N-2 nodes below coordinate j), the product of the node's
// rows at the other levels times the sum of value x leaf row over its
// nonzeros. F.M[0..N-3] are the factors of the other levels 0..N-2 in order.
// One workgroup of 1-8 waves per output row. A wave takes 64 entries at a time
// and walks their nonzeros as one list, 64 to a chunk, a lane each: a
// histogram of the nodes' ends over the chunk and a lane scan give every
// lane its node, hence its nonzero. The products are formed once per node (PF
// at a time, in LDS) and the row groups take the nonzeros in turn. The next
// chunk's coordinates and values are loaded behind this one's rows. No
// atomics, no zero fill, bitwise reproducible.
//
// Taking the level's nodes in turn, a row group each with its subtree, left a
// chain of five dependent loads with four rows in flight and the waves to the
// subtrees' sizes: 20M nonzeros, 3-mode, rank 32: 596 us against 371; 8M,
// 4-mode, rank 32: 590 and 270 us at levels 1 and 2 against 111 and 96.
template <int N, int R>
__global__ __launch_bounds__(512) void inner_leaf_kernel(const int32_t* __restrict__ tpos,
                                                         int32_t tdim, int32_t nent,
                                                         const int32_t* __restrict__ range,
                                                         const int32_t* __restrict__ cor,
                                                         const int32_t* __restrict__ crd,
                                                         const float* __restrict__ vals,
                                                         FactorsDev F, float* __restrict__ A,
                                                         int Rr) {
  using RO = Row<R>;
  using V = typename RO::V;
  constexpr int NV = RO::NV;
  constexpr int LPR = RO::LPR;
  constexpr int L = N - 2;  // the other levels above the nonzeros
  constexpr int KR = Lay<R>::kMaxRank;
  constexpr int NGW = 64 / LPR;
  constexpr int PF0 = 4096 / (KR * 4);
  constexpr int PF = PF0 < 64 ? PF0 : 64;
  constexpr int SB = NV >= 4 ? 2 : NV == 2 ? 4 : LPR < 8 ? LPR : 8;
  extern __shared__ __align__(16) unsigned char smem[];
  const int32_t j = blockIdx.x;
  const int lane = int(threadIdx.x) & 63;
  const int wv = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int nwv = int(blockDim.x) >> 6;
  const int gi = lane / LPR;
  const int c = lane % LPR;
  unsigned char* mine = smem + size_t(wv) * kInnerLeafLds;
  int4* rec = reinterpret_cast<int4*>(mine);
  int32_t* hist = reinterpret_cast<int32_t*>(mine + 1024);
  float* P = reinterpret_cast<float*>(mine + 1280);
  const float* __restrict__ Ml = F.M[N - 1];
  // a chunk's nonzeros are summed apart from the row's earlier ones: one chain
  // of FP32 sums over a row had up to 29% more error at orders 4 and 5
  V acc[NV], sum[NV];
  RO::zero(acc);
  RO::zero(sum);
  if (j < tdim) {
    const int32_t t1 = tpos[j + 1];
    const int32_t step = 64 * nwv;
    // (unsigned: a base past the last entry may pass 2^31 - 1)
    for (uint32_t base = uint32_t(tpos[j]) + 64 * wv; base < uint32_t(t1); base += step) {
      // the window's nodes: lane i holds entry base + i
      const int32_t t = index_ahead(int32_t(base), lane, t1 - 1);
      const int32_t first = range[t];
      const int32_t len = base + lane < uint32_t(t1) ? range[index_end(nent, t)] - first : 0;
      int32_t co[L];
#pragma unroll
      for (int m = 0; m < L; ++m) co[m] = cor[int64_t(m) * nent + t];
      const int32_t end = wave_scan_add(len);  // of the node in the list
      const int32_t begin = end - len;
      const int32_t total = __builtin_amdgcn_readlane(end, 63);
      // list position p of the wave: its node, coordinate and value
      auto fetch = [&](uint32_t f0, int32_t& node, int32_t& l, float& v) {
        const uint32_t s = uint32_t(end) - f0;
        hist[lane] = 0;
        wave_lds_sync();
        if (s - 1u < 63u) atomicAdd(&hist[s], 1);
        wave_lds_sync();
        const int32_t h = hist[lane];
        wave_lds_sync();
        node = min(__popcll(__ballot(uint32_t(end) <= f0)) + wave_scan_add(h), 63);
        const int32_t q = __shfl(first - begin, node) + index_ahead(int32_t(f0), lane, total - 1);
        const bool ok = f0 + lane < uint32_t(total);
        l = ok ? crd[q] : 0;
        v = ok ? vals[q] : 0.f;
      };
      int32_t node, l, node_n = 0, l_n = 0;
      float v, v_n = 0.f;
      if (total > 0) fetch(0, node, l, v);
      for (uint32_t f0 = 0; f0 < uint32_t(total); f0 += 64) {
        const int32_t n = min(64, total - int32_t(f0));
        rec[lane] = make_int4(l, __float_as_int(v), node, 0);
        wave_lds_sync();
        const int32_t a0 = __builtin_amdgcn_readlane(node, 0);
        const int32_t a1 = __builtin_amdgcn_readlane(node, n - 1);
        if (f0 + 64 < uint32_t(total)) fetch(f0 + 64, node_n, l_n, v_n);
        // (cold) whether a row that multiplies a product of others is above 1
        auto raised = [&](int32_t f, int32_t fe) {
          float peak = 0.f;
          for (; L > 2 && f < fe; f += NGW) {
            V r[NV];
            RO::load(r, F.M[L - 1], __shfl(co[L - 1], min(f + gi, fe - 1)), c, Rr);
            peak = RO::peak(r, peak);
          }
          return __ballot(!(peak <= 1.f)) != 0;
        };
        // (cold) whether a product of the nodes' rows left the normal numbers where
        // no row has a 0
        auto product_lost = [&](int32_t f, int32_t fe) {
          bool lost = false;
          for (; f < fe; f += NGW) {
            const int32_t x = min(f + gi, fe - 1);
            V p[NV];
            RO::load(p, F.M[0], __shfl(co[0], x), c, Rr);
#pragma unroll
            for (int m = 1; m < L; ++m) {
              V r[NV];
              RO::load(r, F.M[m], __shfl(co[m], x), c, Rr);
              lost = RO::hmul_lost(p, r) || lost;
            }
          }
          return __ballot(lost) != 0;
        };
        // (cold) nonzeros [t, e) with P, whose first node is fa; the largest value
        // times leaf row
        auto add_p = [&](int32_t fa, int32_t t, int32_t e) {
          float peak = 0.f;
          for (; t < e; t += 2 * NGW) {
            V d[2][NV];
            int4 x[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              x[u] = rec[min(t + u * NGW + gi, e - 1)];
              RO::load(d[u], Ml, x[u].x, c, Rr);
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              V p[NV];
              RO::get(P + (x[u].z - fa) * KR, c, p);
              RO::scale(d[u], __int_as_float(x[u].y));
              peak = RO::peak(d[u], peak);
              RO::hfma_if(t + u * NGW + gi < e, acc, d[u], p);
            }
          }
          return peak;
        };
        // (cold) the same unless that is above kSafe: whether they are added
        auto with_p = [&](int32_t fa, int32_t t, int32_t e) {
          V before[NV];
#pragma unroll
          for (int i = 0; i < NV; ++i) before[i] = acc[i];
          if (!__ballot(!(add_p(fa, t, e) <= kSafe))) return true;
#pragma unroll
          for (int i = 0; i < NV; ++i) acc[i] = before[i];
          return false;
        };
        // (cold) nonzeros [t, e) without P
        auto rows_apart = [&](int32_t t, int32_t e) {
          for (; t < e; t += NGW) {
            const int4 x = rec[min(t + gi, e - 1)];
            V s[NV];
            RO::load(s, Ml, x.x, c, Rr);
            RO::scale(s, __int_as_float(x.y));
#pragma unroll
            for (int m = L - 1; m >= 0; --m) {
              V r[NV];
              RO::load(r, F.M[m], __shfl(co[m], x.z), c, Rr);
              RO::hmul(s, r);
            }
            if (t + gi < e) RO::add(acc, s);
          }
        };
        // nodes [fa, fe) of the chunk hold its nonzeros [a, e)
        for (int32_t fa = a0, a = 0; a < n;) {
          const int32_t fe = min(fa + PF, a1 + 1);
          const int32_t e = fe > a1 ? n : __builtin_amdgcn_readlane(begin, fe) - int32_t(f0);
          float least = FLT_MAX, most = 0.f;
          for (int32_t g0 = fa; g0 < fe; g0 += 2 * NGW) {
            V p[2][NV];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              const int32_t f = min(g0 + u * NGW + gi, fe - 1);
              RO::load(p[u], F.M[0], __shfl(co[0], f), c, Rr);
#pragma unroll
              for (int m = 1; m < L; ++m) {
                V r[NV];
                RO::load(r, F.M[m], __shfl(co[m], f), c, Rr);
                RO::hmul(p[u], r);
                RO::extent(p[u], c, Rr, least, most);
              }
            }
#pragma unroll
            for (int u = 0; u < 2; ++u)
              if (g0 + u * NGW + gi < fe) RO::put(P + (g0 + u * NGW + gi - fa) * KR, c, p[u]);
          }
          if constexpr (L > 1) {
            // as in the edge walk: products that are no normal numbers, and the
            // nonzeros take the rows apart where that matters
            if (__builtin_expect(__ballot(!(least >= FLT_MIN && most <= FLT_MAX)) != 0, 0)) {
              wave_lds_sync();
              if (__ballot(!(most <= FLT_MAX)) != 0 || raised(fa, fe) || !with_p(fa, a, e)) {
                if (product_lost(fa, fe)) rows_apart(a, e);
                else add_p(fa, a, e);
              }
              wave_lds_sync();
              a = e;
              fa = fe;
              continue;
            }
          }
          // (`whole`: no step is past the nonzeros, as most are not)
          auto steps = [&](auto S, auto whole, int32_t s0) {
            V d[S()][NV];
            auto record = [&](int u) {
              return rec[whole() ? s0 + u * NGW + gi : min(s0 + u * NGW + gi, e - 1)];
            };
#pragma unroll
            for (int u = 0; u < S(); ++u) RO::load(d[u], Ml, record(u).x, c, Rr);
            wave_lds_sync();
#pragma unroll
            for (int u = 0; u < S(); ++u) {
              const int4 x = record(u);
              V p[NV];
              RO::get(P + (x.z - fa) * KR, c, p);
              RO::scale(d[u], __int_as_float(x.y));
              // a step past the nonzeros adds nothing (not its weight 0: the
              // row it repeats may hold infinities)
              if constexpr (whole()) RO::hfma(acc, d[u], p);
              else RO::hfma_if(s0 + u * NGW + gi < e, acc, d[u], p);
            }
          };
          for (int32_t s0 = a; s0 < e;) {
            if (SB > 2 && e - s0 >= SB * NGW) {
              steps(std::integral_constant<int, SB>(), std::true_type(), s0);
              s0 += SB * NGW;
            } else if (SB > 2 && e - s0 > 2 * NGW) {
              steps(std::integral_constant<int, SB>(), std::false_type(), s0);
              s0 += SB * NGW;
            } else {
              steps(std::integral_constant<int, 2>(), std::false_type(), s0);
              s0 += 2 * NGW;
            }
          }
          wave_lds_sync();
          a = e;
          fa = fe;
        }
        node = node_n;
        l = l_n;
        v = v_n;
        RO::add(sum, acc);
        RO::zero(acc);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) acc[i] = sum[i];
  RO::wave_sum(acc);
  if (nwv == 1) {
    if (gi == 0) RO::store(A, j, c, Rr, acc);
    return;
  }
  if (gi == 0) RO::put(P, c, acc);
  __syncthreads();
  if (wv == 0 && gi == 0) {
    for (int w = 1; w < nwv; ++w) {
      V o[NV];
      RO::get(reinterpret_cast<const float*>(smem + size_t(w) * kInnerLeafLds + 1280), c, o);
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
  // 1-8 waves per row, from the mean entries per row
  const int64_t mean = (int64_t(B.nnz) + X.dim - 1) / std::max<int32_t>(X.dim, 1);
  const int nwv = int(std::max<int64_t>(1, std::min<int64_t>(8, (mean + 255) / 256)));
  ktimer_begin(st);
  tleaf_kernel<N, R><<<a_rows, 64 * nwv, 0, st>>>(X.tpos, X.dim, X.ent, X.anc, F, A, Rr);
  TT_HIP_CHECK(hipGetLastError());
  ktimer_end(st, "tleaf_kernel");
  return TENTACO_OK;
}

template <int N, int R>
int launch_inner_leaf_typed(const CsfDev& B, const LevelIndex& X, const FactorsDev& F0, int Rr,
                            float* A, int32_t a_rows, hipStream_t st) {
  if (a_rows <= 0) return TENTACO_OK;
  FactorsDev F;
  F.M[N - 1] = F0.M[N - 1];
  for (int m = 0, i = 0; m < N - 1; ++m)
    if (m != X.level) F.M[i++] = F0.M[m];
  // 1-8 waves per row, from the mean nodes and nonzeros per row
  const int32_t n = B.nodes[N - 2];
  const int64_t mean = std::max((int64_t(n) + X.dim - 1) / std::max<int32_t>(X.dim, 1),
                                (int64_t(B.nnz) / 8 + X.dim - 1) / std::max<int32_t>(X.dim, 1));
  const int nwv = int(std::max<int64_t>(1, std::min<int64_t>(8, (mean + 63) / 64)));
  ktimer_begin(st);
  inner_leaf_kernel<N, R><<<a_rows, 64 * nwv, nwv * kInnerLeafLds, st>>>(
      X.tpos, X.dim, n, X.node, X.anc, B.crd[N - 1], B.vals, F, A, Rr);
  TT_HIP_CHECK(hipGetLastError());
  ktimer_end(st, "inner_leaf_kernel");
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
  const int32_t na = B.nodes[N - 2];                 // the nonzeros' parents
  const int cnt = N - 1;                             // coordinates per parent
  const int32_t n = leaf ? B.nodes[N - 1] : na;      // entries
  auto al = [](size_t x) { return (x + 255) & ~size_t(255); };
  const size_t b_tpos = al(sizeof(int32_t) * (size_t(dim) + 1));
  const bool coords = leaf && N <= 3;                // entries hold coordinates
  const size_t b_ent = al((coords ? 4 * size_t(N) : 8) * std::max<size_t>(n, 1));
  // ancestors by node (kept for the leaf level from order 4, else a
  // temporary), or an inner level's coordinates by entry
  const size_t b_anc = al(sizeof(int32_t) * std::max<size_t>(size_t(na) * cnt, 1));
  const size_t b_keep =
      coords ? 0 : leaf ? b_anc : al(sizeof(int32_t) * std::max<size_t>(size_t(na) * (N - 2), 1));
  void* mem = nullptr;
  if (hipMalloc(&mem, b_tpos + b_ent + b_keep) != hipSuccess)
    return fail(TENTACO_ENOMEM, "level index: hipMalloc of %zu bytes failed",
                b_tpos + b_ent + b_keep);
  X->mem = mem;
  X->level = level;
  X->tpos = static_cast<int32_t*>(mem);
  if (leaf) X->ent = static_cast<char*>(mem) + b_tpos;
  else X->node = reinterpret_cast<int32_t*>(static_cast<char*>(mem) + b_tpos);
  if (!coords) X->anc = reinterpret_cast<int32_t*>(static_cast<char*>(mem) + b_tpos + b_ent);
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
  const size_t b_sort = al(std::max<size_t>(sort_bytes, 1));
  const size_t b_tanc = coords || !leaf ? b_anc : 0;
  if (hipMalloc(&tmp, 4 * b_n + b_sort + b_tanc) != hipSuccess) {
    free_level_index(X);
    return fail(TENTACO_ENOMEM, "level index: temporary allocation failed");
  }
  int32_t* fib = static_cast<int32_t*>(tmp);  // (an inner level's sort keys)
  int32_t* ord_in = reinterpret_cast<int32_t*>(static_cast<char*>(tmp) + b_n);
  int32_t* ord = reinterpret_cast<int32_t*>(static_cast<char*>(tmp) + 2 * b_n);
  int32_t* key = reinterpret_cast<int32_t*>(static_cast<char*>(tmp) + 3 * b_n);
  void* sort_tmp = static_cast<char*>(tmp) + 4 * b_n;
  int32_t* anc = b_tanc ? reinterpret_cast<int32_t*>(static_cast<char*>(tmp) + 4 * b_n + b_sort)
                        : X->anc;
  int rc = TENTACO_OK;
  if (na > 0) {
    tl_anc_kernel<<<grid_of(na), 256, 0, st>>>(B, N - 2, cnt, anc);
    if (hipGetLastError() != hipSuccess) rc = fail(TENTACO_EHIP, "level index: anc launch failed");
  }
  if (!rc && n > 0) {
    if (leaf) tl_fib_kernel<<<grid_of(na), 256, 0, st>>>(B.pos[N - 1], na, fib);
    else tl_key_kernel<<<grid_of(n), 256, 0, st>>>(anc, cnt, level, n, fib);
    tl_iota_kernel<<<grid_of(n), 256, 0, st>>>(ord_in, n);
    if (hipGetLastError() != hipSuccess) rc = fail(TENTACO_EHIP, "level index: launch failed");
    // stable: equal coordinates keep CSF order
    if (!rc && rocprim::radix_sort_pairs(sort_tmp, sort_bytes,
                                         leaf ? B.crd[level] : static_cast<const int32_t*>(fib), key,
                                         static_cast<const int32_t*>(ord_in), ord, size_t(n), 0,
                                         end_bit, st) != hipSuccess)
      rc = fail(TENTACO_EHIP, "level index: sort failed");
    if (!rc) {
      if (!leaf)
        tl_range_kernel<<<grid_of(n), 256, 0, st>>>(ord, B.pos[N - 1], anc, cnt, level, n, X->node,
                                                    X->anc);
      else if (N == 2)
        tl_coord_kernel<2><<<grid_of(n), 256, 0, st>>>(ord, fib, anc, B.vals, n,
                                                       static_cast<LeafEnt<2>*>(X->ent));
      else if (N == 3)
        tl_coord_kernel<3><<<grid_of(n), 256, 0, st>>>(ord, fib, anc, B.vals, n,
                                                       static_cast<LeafEnt<3>*>(X->ent));
      else
        tl_ent_kernel<<<grid_of(n), 256, 0, st>>>(ord, fib, B.vals, n, static_cast<uint2*>(X->ent));
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

int launch_mttkrp_inner(const CsfDev& B, const LevelIndex& X, const FactorsDev& F, int level,
                        int R, float* A, int32_t a_rows, hipStream_t st) {
  if (!X.built || X.level != level || level < 1 || level > B.order - 2 || !X.node)
    return fail(TENTACO_EINVAL, "level %d index not built", level);
  if (R <= 0 || R > kMaxRankAny)
    return fail(TENTACO_EUNSUPPORTED, "rank R=%d outside 1..%d", R, kMaxRankAny);
  return with_rank_layout(R, [&](auto r) {
    switch (B.order) {
      case 3: return launch_inner_leaf_typed<3, r()>(B, X, F, R, A, a_rows, st);
      case 4: return launch_inner_leaf_typed<4, r()>(B, X, F, R, A, a_rows, st);
      default: return launch_inner_leaf_typed<5, r()>(B, X, F, R, A, a_rows, st);
    }
  });
}

}  // namespace tt
