// The MTTKRP kernels templated on tensor order and rank layout, with their
// launches (the kernels' overview is in mttkrp.hip). Each order N is
// instantiated in its own source, mttkrp_o<N>.hip, so that the orders compile
// in parallel.
#pragma once

#include <algorithm>
#include <climits>

#include "internal.h"
#include "mttkrp_dispatch.h"
#include "rowops.h"

namespace tt {
namespace {

// ---------------------------------------------------------------------------
// edge-serial / edge-parallel work for workgroup-sized block b of one CSF
// (nonzeros [b*NB, (b+1)*NB)); shared by the per-tensor kernel and the
// persistent batch kernel.
//
// LDS layout (dynamic, `smem`): the EP reduction area (edge_ep_bytes), then
// for each walk level k = 0..N-2 the node bounds pos[k+1][lo..hi+1] and the
// node coordinates crd[k][lo..hi] of the workgroup's bracket [lo, hi]. The
// level above the nonzeros (k = N-2) gets room for min(NB+1, kLeafCap)
// nodes (NB+1 is the most a CSF built from coordinates can have there); the
// upper levels get kUpperCap. A level whose bracket does not fit is read
// from global memory instead, so large brackets and runs of empty nodes cost
// time, never correctness.
// The edge-serial family (EP false) needs W (the edge-parallel family
// ignores it): every row output goes to the FP64 buffer W instead of A.
// Slices complete inside a group are stored; the
// groups' first and last slices are combined across the wave's groups by a
// segmented suffix scan over shuffles, and each slice's sum per wave is
// added with one FP64 atomic. A giant slice then takes one atomic per wave,
// without FP32 rounding at each add.
// A device pointer the kernel knows to be global memory (loads through it
// are global loads, never flat ones).
__device__ __forceinline__ const __attribute__((address_space(1))) int32_t* as_global(
    const int32_t* p) {
  return reinterpret_cast<const __attribute__((address_space(1))) int32_t*>(
      reinterpret_cast<uintptr_t>(p));
}

template <int N, int R, bool EP>
__device__ __forceinline__ void edge_block(const CsfDev& B, const FactorsDev& F,
                                           float* __restrict__ A, int Rr,
                                           const int32_t* __restrict__ brk, int32_t b,
                                           int32_t G, int32_t NB, unsigned char* smem,
                                           double* __restrict__ W) {
  using RO = Row<R>;
  using V = typename RO::V;
  constexpr int NV = RO::NV;
  constexpr int LPR = RO::LPR;
  constexpr int NL = N - 1;  // levels 0..N-2 carry walk state

  const int gi = threadIdx.x / LPR;
  const int c = threadIdx.x % LPR;
  const int32_t nnz = B.nnz;
  const int32_t blk0 = b * NB;
  const int32_t blk1 = min(blk0 + NB, nnz);
  const int32_t p0 = blk0 + gi * G;
  const int32_t p1 = min(p0 + G, blk1);
  const bool active = p0 < p1;
  const int Rc = (R <= 0) ? Rr : R;

  // ---- stage the node brackets in LDS
  int32_t lo[NL], hib[NL];
  bool staged[NL];
  int32_t* spos[NL];
  int32_t* scrd[NL];
  {
    int32_t* base = reinterpret_cast<int32_t*>(
        smem + (EP ? edge_ep_bytes(blockDim.x, LPR, Rc) : size_t(0)));
#pragma unroll
    for (int k = NL - 1; k >= 0; --k) {
      const int32_t cap = (k == NL - 1) ? edge_leaf_cap(NB) : kUpperCap;
      lo[k] = brk[b * NL + k];
      hib[k] = brk[(b + 1) * NL + k];
      staged[k] = hib[k] - lo[k] + 1 <= cap;
      spos[k] = base;
      scrd[k] = base + cap + 1;
      base += 2 * cap + 1;
      if (staged[k]) {
        const int32_t* pk = B.pos[k + 1];
        const int32_t* ck = (k == 0) ? B.crd0 : B.crd[k];
        const int32_t n = hib[k] - lo[k] + 1;
        for (int32_t j = threadIdx.x; j <= n; j += blockDim.x) {
          spos[k][j] = pk[lo[k] + j];
          if (j < n) scrd[k][j] = ck[lo[k] + j];
        }
      }
    }
  }
  __syncthreads();
  // An LDS read when the level's brackets are staged, a global read
  // otherwise, as two loads of their own: one load through a pointer that
  // may be either would be a flat load, whose wait also drains every global
  // load in flight (the walk's row gathers). The global read is waited for
  // on its own path (the empty asm uses its value), so a use after the two
  // paths join waits only for the LDS read, not for the rows in flight.
  auto POS = [&](int k, int32_t x) -> int32_t {
    if (staged[k]) return spos[k][x - lo[k]];
    const int32_t v = as_global(B.pos[k + 1])[x];
    asm volatile("" ::"v"(v));
    return v;
  };
  auto CRD = [&](int k, int32_t x) -> int32_t {
    if (staged[k]) return scrd[k][x - lo[k]];
    const int32_t v = as_global((k == 0) ? B.crd0 : B.crd[k])[x];
    asm volatile("" ::"v"(v));
    return v;
  };
  auto SEARCH = [&](int k, int32_t a, int32_t z, int32_t key) {
    // largest x in [a, z] with POS(k, x) <= key (requires POS(k, a) <= key)
    while (a < z) {
      const int32_t mid = a + ((z - a + 1) >> 1);
      if (POS(k, mid) <= key) a = mid;
      else z = mid - 1;
    }
    return a;
  };

  int32_t cur[NL], cend[NL];
  V acc[NL][NV];
  V rowc[NL][NV];
#pragma unroll
  for (int k = 0; k < NL; ++k) {
    RO::zero(acc[k]);
    RO::zero(rowc[k]);
    cur[k] = 0;
    cend[k] = 0;
  }
  int32_t head = INT_MAX;
  int32_t head_row = 0;
  bool head_closed = false;
  V head_acc[NV];
  RO::zero(head_acc);

  if (active) {
    int32_t key = p0;
#pragma unroll
    for (int k = NL - 1; k >= 0; --k) {
      cur[k] = SEARCH(k, lo[k], hib[k], key);
      key = cur[k];
    }
#pragma unroll
    for (int k = 0; k < NL; ++k) {
      cend[k] = POS(k, cur[k] + 1);
      if (k >= 1) RO::load(rowc[k], F.M[k], CRD(k, cur[k]), c, Rr);
    }
    head = cur[0];
    head_row = CRD(0, cur[0]);

    const int32_t* __restrict__ lcrd = B.crd[N - 1];
    const float* __restrict__ vals = B.vals;
    const float* __restrict__ Mleaf = F.M[N - 1];
    // Leaf (coordinate, value) pairs arrive U at a time: lane c < U of a row
    // group loads pair t0 + c (one coalesced load per group and batch) and
    // the group's lanes exchange them with shuffles. Pairs are fetched two
    // batches ahead and leaf rows one batch ahead of their use.
    constexpr int U = LPR < 4 ? LPR : 4;
    const int gbase = (threadIdx.x & 63) - c;  // lane of this group's lane 0
    // (loads of an in-range position for every lane, masked afterwards: a
    // load behind a branch makes the compiler wait for it at the join)
    auto load_pairs = [&](int32_t t0, int32_t& lq, float& vq) {
      const int32_t t = t0 + c;
      const bool ok = c < U && t < p1;
      const int32_t tc = min(t, p1 - 1);
      const int32_t l = lcrd[tc];
      const float w = vals[tc];
      lq = ok ? l : 0;
      vq = ok ? w : 0.f;
    };
    auto issue = [&](int32_t lq, float vq, V (&d)[U][NV], float (&v)[U]) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int32_t l = __shfl(lq, gbase + u);
        v[u] = __shfl(vq, gbase + u);
        RO::load(d[u], Mleaf, l, c, Rr);
      }
    };
    auto consume = [&](int32_t t0, const V (&d)[U][NV], const float (&v)[U]) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int32_t t = t0 + u;
        if (t >= p1) break;
        if (t >= cend[NL - 1]) {
          // close the fiber at level N-2 and every ancestor that ends here
          bool closing = true;
          int32_t ckey = t;
#pragma unroll
          for (int k = NL - 1; k >= 0; --k) {
            if (closing) {
              const int32_t old = cur[k];
              if (k >= 1) {
                RO::hfma(acc[k - 1], acc[k], rowc[k]);
              } else {
                const int64_t row = CRD(0, old);
                if (old == head && !head_closed) {
                  head_closed = true;
#pragma unroll
                  for (int j = 0; j < NV; ++j) head_acc[j] = acc[0][j];
                } else {
                  if constexpr (EP) RO::store(A, row, c, Rr, acc[0]);
                  else RO::store_f64(W, row, c, Rr, acc[0]);
                }
              }
              RO::zero(acc[k]);
              int32_t x = old + 1;
              int32_t e = POS(k, x + 1);
              if (e <= ckey) {
                x = SEARCH(k, x + 1, hib[k], ckey);
                e = POS(k, x + 1);
              }
              cur[k] = x;
              cend[k] = e;
              if (k >= 1) {
                RO::load(rowc[k], F.M[k], CRD(k, x), c, Rr);
                closing = x >= cend[k - 1];
                ckey = x;
              }
            }
          }
        }
        RO::axpy(acc[NL - 1], v[u], d[u]);
      }
    };
    V dA[U][NV], dB[U][NV];
    float vA[U], vB[U];
    int32_t lA, lB;
    float wA, wB;
    load_pairs(p0, lA, wA);
    load_pairs(p0 + U, lB, wB);
    issue(lA, wA, dA, vA);
    for (int32_t t0 = p0; t0 < p1; t0 += 2 * U) {
      // invariant: rows of batch t0 in dA; pairs of batch t0+U in (lB, wB)
      if (t0 + U < p1) {
        load_pairs(t0 + 2 * U, lA, wA);
        issue(lB, wB, dB, vB);
      }
      consume(t0, dA, vA);
      if (t0 + U >= p1) break;
      if (t0 + 2 * U < p1) {
        load_pairs(t0 + 3 * U, lB, wB);
        issue(lA, wA, dA, vA);
      }
      consume(t0 + U, dB, vB);
    }
    // fold the open nodes into the open slice
#pragma unroll
    for (int k = NL - 1; k >= 1; --k) RO::hfma(acc[k - 1], acc[k], rowc[k]);
  }

  if constexpr (!EP) {
    // Entries e = 2 * gw + q of the wave's NGW groups: q = 0 is the group's
    // first slice (its partial if it closed inside the run, else 0), q = 1
    // the slice open at the run's end. Keys do not decrease with e; idle
    // groups (trailing) hold INT_MAX. Suffix scan: at stride s, entry e adds
    // entry e + s when both have the same key, so each key's first entry ends
    // with the key's sum over the wave. Stride 1 pairs (gw, 0) with (gw, 1)
    // and (gw, 1) with (gw + 1, 0); an even stride pairs (gw, q) with
    // (gw + s / 2, q). Every lane runs every shuffle.
    constexpr int NGW = 64 / LPR;
    const int lane = int(threadIdx.x) & 63;
    const int gw = lane / LPR;
    const int32_t k0 = active ? head : INT_MAX;
    const int32_t k1 = active ? cur[0] : INT_MAX;
    V v0[NV], v1[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      v0[j] = head_acc[j];
      v1[j] = acc[0][j];
    }
    auto shfl_v = [&](const V (&x)[NV], int src, V (&out)[NV]) {
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        if constexpr (R == 0) {
          out[j] = __shfl(x[j], src);
        } else {
          out[j].x = __shfl(x[j].x, src);
          out[j].y = __shfl(x[j].y, src);
          out[j].z = __shfl(x[j].z, src);
          out[j].w = __shfl(x[j].w, src);
        }
      }
    };
#pragma unroll
    for (int st = 1; st < 2 * NGW; st <<= 1) {
      const int dg = st == 1 ? 1 : st / 2;  // groups ahead of the source
      const int src = (lane + dg * LPR) & 63;
      const bool in_wave = gw + dg < NGW;
      V a0[NV], a1[NV], b0[NV], b1[NV];
      shfl_v(v0, src, b0);
      shfl_v(v1, src, b1);
      const int32_t n0 = __shfl(k0, src);
      const int32_t n1 = __shfl(k1, src);
      int32_t t0, t1;
      bool ok0, ok1;
      if (st == 1) {
        // (gw, 0) + (gw, 1) in this lane; (gw, 1) + (gw + 1, 0)
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          a0[j] = v1[j];
          a1[j] = b0[j];
        }
        t0 = k1;
        t1 = n0;
        ok0 = true;
        ok1 = in_wave;
      } else {
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          a0[j] = b0[j];
          a1[j] = b1[j];
        }
        t0 = n0;
        t1 = n1;
        ok0 = in_wave;
        ok1 = in_wave;
      }
      if (ok0 && k0 != INT_MAX && t0 == k0) RO::add(v0, a0);
      if (ok1 && k1 != INT_MAX && t1 == k1) RO::add(v1, a1);
    }
    // a key's first entry in the wave adds the sum
    const int32_t kprev = __shfl(k1, (lane - LPR) & 63);  // (gw - 1, 1)
    if (k0 != INT_MAX && (gw == 0 || kprev != k0))
      RO::atomic_add_f64(W, CRD(0, k0), c, Rr, v0);
    if (k1 != INT_MAX && k1 != k0) RO::atomic_add_f64(W, CRD(0, k1), c, Rr, v1);
  }

  if constexpr (EP) {
    // Segmented suffix scan over the 2 entries per row group (first slice,
    // last slice) of the workgroup; keys are nondecreasing, idle groups use
    // INT_MAX. Entry 2g = (head slice, its closed partial or 0), entry
    // 2g+1 = (open slice at run end, its partial).
    const int NGB = blockDim.x / LPR;
    const int E = 2 * NGB;
    int32_t* keys = reinterpret_cast<int32_t*>(smem);
    float* ev = reinterpret_cast<float*>(smem + size_t(E) * sizeof(int32_t));
    V val[2][NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      val[0][j] = head_acc[j];
      val[1][j] = acc[0][j];
    }
    const int32_t key0 = active ? head : INT_MAX;
    const int32_t key1 = active ? cur[0] : INT_MAX;
    if (c == 0) {
      keys[2 * gi] = key0;
      keys[2 * gi + 1] = key1;
    }
    auto put = [&](int e, const V (&x)[NV]) {
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const int k = RO::col(j, c, Rr);
        if constexpr (R == 0) {
          if (k < Rc) ev[size_t(e) * Rc + k] = x[j];
        } else if constexpr (R < 0) {
          store4(ev + size_t(e) * Rc + k, x[j]);
        } else {
          *reinterpret_cast<float4*>(ev + size_t(e) * Rc + k) = x[j];
        }
      }
    };
    auto get = [&](int e, V (&x)[NV]) {
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const int k = RO::col(j, c, Rr);
        if constexpr (R == 0) {
          x[j] = (k < Rc) ? ev[size_t(e) * Rc + k] : 0.f;
        } else if constexpr (R < 0) {
          x[j] = load4(ev + size_t(e) * Rc + k);
        } else {
          x[j] = *reinterpret_cast<const float4*>(ev + size_t(e) * Rc + k);
        }
      }
    };
    put(2 * gi, val[0]);
    put(2 * gi + 1, val[1]);
    __syncthreads();
    for (int s = 1; s < E; s <<= 1) {
      V add[2][NV];
      bool take[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int e = 2 * gi + q;
        take[q] = (e + s < E) && keys[e] != INT_MAX && keys[e + s] == keys[e];
        if (take[q]) get(e + s, add[q]);
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        if (take[q]) {
          RO::add(val[q], add[q]);
          put(2 * gi + q, val[q]);
        }
      }
      __syncthreads();
    }
    // segment heads write their totals; only the workgroup's first and last
    // slice can be shared with another workgroup
    const int32_t g_last = (blk1 - 1 - blk0) / G;
    const int32_t first_key = keys[0];
    const int32_t last_key = keys[2 * g_last + 1];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int e = 2 * gi + q;
      const int32_t k = keys[e];
      if (k == INT_MAX) continue;
      if (e > 0 && keys[e - 1] == k) continue;
      const int64_t row = CRD(0, k);
      if (k == first_key || k == last_key) RO::atomic_add(A, row, c, Rr, val[q]);
      else RO::store(A, row, c, Rr, val[q]);
    }
  }
  (void)head_row;
}

template <int N, int R, bool EP>
__global__ __launch_bounds__(512) void edge_kernel(CsfDev B, FactorsDev F,
                                                   float* __restrict__ A, int Rr,
                                                   const int32_t* __restrict__ brk,
                                                   int32_t G, int32_t NB,
                                                   double* __restrict__ W) {
  extern __shared__ __align__(16) unsigned char smem[];
  edge_block<N, R, EP>(B, F, A, Rr, brk, blockIdx.x, G, NB, smem, W);
}


// ---------------------------------------------------------------------------
// slice-row kernel: subtree sums, depth first.
template <int N, int M, int R>
__device__ __forceinline__ void subtree(const CsfDev& B, const FactorsDev& F,
                                        int32_t y, int c, int Rr,
                                        typename Row<R>::V (&out)[Row<R>::NV]);

// Sum of the subtrees of the children of node y at level M < N-1 (y's own
// factor row not applied); the nonzeros of a level N-2 node are read U at a
// time with all their leaf rows in flight.
template <int N, int M, int R>
__device__ __forceinline__ void children_sum(const CsfDev& B, const FactorsDev& F, int32_t y,
                                             int c, int Rr,
                                             typename Row<R>::V (&out)[Row<R>::NV]) {
  using RO = Row<R>;
  using V = typename RO::V;
  constexpr int NV = RO::NV;
  RO::zero(out);
  const int32_t a = B.pos[M + 1][y];
  const int32_t e = B.pos[M + 1][y + 1];
  if constexpr (M + 1 == N - 1) {
    const int32_t* __restrict__ lcrd = B.crd[N - 1];
    const float* __restrict__ vals = B.vals;
    const float* __restrict__ Ml = F.M[N - 1];
    constexpr int U = 4;
    for (int32_t q0 = a; q0 < e; q0 += U) {
      int32_t l[U];
      float v[U];
      V d[U][NV];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool ok = q0 + u < e;
        l[u] = ok ? lcrd[q0 + u] : 0;
        v[u] = ok ? vals[q0 + u] : 0.f;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) RO::load(d[u], Ml, l[u], c, Rr);
#pragma unroll
      for (int u = 0; u < U; ++u) RO::axpy(out, v[u], d[u]);
    }
  } else {
    for (int32_t ch = a; ch < e; ++ch) {
      V s[NV];
      subtree<N, M + 1, R>(B, F, ch, c, Rr, s);
      RO::add(out, s);
    }
  }
}

// The factorised value of node y at level M: its own factor row times the
// sum of its children's subtrees (val times the leaf row for a nonzero).
template <int N, int M, int R>
__device__ __forceinline__ void subtree(const CsfDev& B, const FactorsDev& F,
                                        int32_t y, int c, int Rr,
                                        typename Row<R>::V (&out)[Row<R>::NV]) {
  using RO = Row<R>;
  using V = typename RO::V;
  constexpr int NV = RO::NV;
  if constexpr (M == N - 1) {
    // a lone nonzero (order-2 tensors only reach this at level 1)
    V d[NV];
    RO::load(d, F.M[M], B.crd[M][y], c, Rr);
    RO::zero(out);
    RO::axpy(out, B.vals[y], d);
  } else {
    V own[NV];
    RO::load(own, F.M[M], B.crd[M][y], c, Rr);
    children_sum<N, M, R>(B, F, y, c, Rr, out);
    RO::hmul(out, own);
  }
}

// MTTKRP for the mode held at level L >= 1 of the CSF, without a CSF rooted
// at that mode:
//   A_L(j,:) = sum over nonzeros with level-L coordinate j of
//              val * prod_{l != L} M_l(coordinate at level l, :),
// with M_0 the root mode's factor. Every level-L node y contributes
//   (prod_{l < L} M_l(row of y's level-l ancestor)) * (factorised sum of y's
//   subtree below L; its value for a nonzero),
// added atomically into row crd_L[y] of the zero-filled A (nodes of
// different parents can share a coordinate). Row group g takes chunk g of
// CH consecutive level-L nodes (grid-stride), so work follows the level-L
// subtrees rather than the level-(L-1) parents, whose sizes can be Zipf
// skewed. The ancestors of a chunk's first node are found by upper-bound
// searches once; after that they advance with the node (nodes are in
// order), and the ancestor product is recomputed only when one changes.
template <int N, int L, int R>
__global__ __launch_bounds__(256) void level_kernel(CsfDev B, FactorsDev F, float* __restrict__ A,
                                                    int Rr, int32_t CH) {
  using RO = Row<R>;
  using V = typename RO::V;
  constexpr int NV = RO::NV;
  constexpr int LPR = RO::LPR;
  const int c = int(threadIdx.x) % LPR;
  const int64_t g0 = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) / LPR;
  const int64_t ng = int64_t(gridDim.x) * blockDim.x / LPR;
  const int32_t ny = B.nodes[L];
  for (int64_t chunk = g0; chunk * CH < ny; chunk += ng) {
    const int32_t y0 = int32_t(chunk * CH);
    const int32_t y1 = int32_t(min(int64_t(ny), chunk * CH + CH));
    // anc[l]: the level-l ancestor of the current node, l < L
    int32_t anc[L];
    {
      int32_t x = y0;
#pragma unroll
      for (int l = L - 1; l >= 0; --l) {
        x = search_le(B.pos[l + 1], 0, B.nodes[l] - 1, x);
        anc[l] = x;
      }
    }
    V above[NV];
    auto ancestors_product = [&]() {
      RO::load(above, F.M[0], B.crd0[anc[0]], c, Rr);
#pragma unroll
      for (int l = 1; l < L; ++l) {
        V r[NV];
        RO::load(r, F.M[l], B.crd[l][anc[l]], c, Rr);
        RO::hmul(above, r);
      }
    };
    ancestors_product();
    for (int32_t y = y0; y < y1; ++y) {
      // advance the ancestors so that pos[l+1][anc[l]] <= child < pos[l+1][anc[l]+1]
      bool moved = false;
      int32_t x = y;
#pragma unroll
      for (int l = L - 1; l >= 0; --l) {
        if (x >= B.pos[l + 1][anc[l] + 1]) {
          do {
            ++anc[l];
          } while (x >= B.pos[l + 1][anc[l] + 1]);
          moved = true;
        }
        x = anc[l];
      }
      if (moved) ancestors_product();
      V out[NV];
      if constexpr (L == N - 1) {
        RO::zero(out);
        RO::axpy(out, B.vals[y], above);
      } else {
        V below[NV];
        RO::zero(below);
        for (int32_t ch = B.pos[L + 1][y]; ch < B.pos[L + 1][y + 1]; ++ch) {
          V s2[NV];
          subtree<N, L + 1, R>(B, F, ch, c, Rr, s2);
          RO::add(below, s2);
        }
        RO::zero(out);
        RO::hfma(out, above, below);
      }
      RO::atomic_add(A, B.crd[L][y], c, Rr, out);
    }
  }
}

// MTTKRP for the mode held at inner level L (1 <= L <= N-2) through the
// per-handle transposed index of that level: the level-L nodes sorted by
// coordinate (node[t], rows tpos[j]..tpos[j+1]) and, per node, the
// coordinates of its ancestors at levels 0..L-1 (anc[y * L + m]). One
// workgroup of 1-4 waves computes output row j: its row groups take the
// row's nodes in turn, each adding (product of the node's ancestor rows) x
// (sum of the node's children's subtrees), and the row is reduced over the
// wave and the workgroup and stored once: no atomics, no zero fill,
// bitwise reproducible.
template <int N, int L, int R>
__global__ __launch_bounds__(256) void inner_kernel(const int32_t* __restrict__ tpos, int32_t tdim,
                                                    const int32_t* __restrict__ node,
                                                    const int32_t* __restrict__ anc, CsfDev B,
                                                    FactorsDev F, float* __restrict__ A, int Rr) {
  using RO = Row<R>;
  using V = typename RO::V;
  constexpr int NV = RO::NV;
  constexpr int LPR = RO::LPR;
  constexpr int NG = 64 / LPR;
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
    const int32_t t1 = tpos[j + 1];
    for (int32_t t = tpos[j] + wv * NG + gi; t < t1; t += NG * nwv) {
      const int32_t y = node[t];
      const int32_t* a = anc + int64_t(y) * L;
      V above[NV];
      RO::load(above, F.M[0], a[0], c, Rr);
#pragma unroll
      for (int m = 1; m < L; ++m) {
        V r[NV];
        RO::load(r, F.M[m], a[m], c, Rr);
        RO::hmul(above, r);
      }
      V below[NV];
      children_sum<N, L, R>(B, F, y, c, Rr, below);
      RO::hfma(acc, above, below);
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

// Order-3 slice: the wavefront walks the slice's level-1 fibers 64 at a time.
// Lane L loads fiber (base+L)'s bounds, coordinate and first nonzero with
// coalesced loads; row group g then takes fibers base + t*NG + g through
// lane shuffles and issues all its C and D row gathers for the chunk before
// using any of them. The next chunk's fiber metadata is loaded while the
// current chunk's rows are in flight.
template <int R>
__device__ __forceinline__ void slice3_accumulate(const CsfDev& B, const FactorsDev& F,
                                                  int32_t x, int lane, int gi, int c, int Rr,
                                                  int wv, int nwv,
                                                  typename Row<R>::V (&acc)[Row<R>::NV]) {
  using RO = Row<R>;
  using V = typename RO::V;
  constexpr int NV = RO::NV;
  constexpr int NG = 64 / RO::LPR;
  constexpr int NT = 64 / NG;                 // fibers per row group per chunk
  constexpr int TB = NT < 8 ? NT : 8;         // fibers whose rows are in flight per batch
  const int32_t* __restrict__ p2 = B.pos[2];
  const int32_t* __restrict__ c1 = B.crd[1];
  const int32_t* __restrict__ c2 = B.crd[2];
  const float* __restrict__ vals = B.vals;
  const float* __restrict__ Cm = F.M[1];
  const float* __restrict__ Dm = F.M[2];
  const int32_t f0 = B.pos[1][x];
  const int32_t f1 = B.pos[1][x + 1];
  auto meta = [&](int32_t base, int32_t& s, int32_t& e, int32_t& k, int32_t& l0, float& v0) {
    const int32_t f = base + lane;
    s = e = k = l0 = 0;
    v0 = 0.f;
    if (f < f1) {
      s = p2[f];
      e = p2[f + 1];
      k = c1[f];
      if (e > s) {
        l0 = c2[s];
        v0 = vals[s];
      }
    }
  };
  const int32_t step = 64 * nwv;
  int32_t ns, ne, nk, nl;
  float nv;
  if (f0 + 64 * wv < f1) meta(f0 + 64 * wv, ns, ne, nk, nl, nv);
  for (int32_t base = f0 + 64 * wv; base < f1; base += step) {
    const int32_t s = ns, e = ne, k = nk, l0 = nl;
    const float v0 = nv;
    if (base + step < f1) meta(base + step, ns, ne, nk, nl, nv);
#pragma unroll
    for (int t0 = 0; t0 < NT; t0 += TB) {
      V cr[TB][NV], dr[TB][NV];
      int32_t st[TB], et[TB];
      float vt[TB];
      bool ok[TB];
#pragma unroll
      for (int u = 0; u < TB; ++u) {
        const int src = (t0 + u) * NG + gi;
        const int32_t kt = __shfl(k, src);
        const int32_t lt = __shfl(l0, src);
        vt[u] = __shfl(v0, src);
        st[u] = __shfl(s, src);
        et[u] = __shfl(e, src);
        ok[u] = base + src < f1;
        RO::load(cr[u], Cm, ok[u] ? kt : 0, c, Rr);
        RO::load(dr[u], Dm, ok[u] ? lt : 0, c, Rr);
      }
#pragma unroll
      for (int u = 0; u < TB; ++u) {
        if (!ok[u]) continue;
        V w[NV];
        RO::zero(w);
        RO::axpy(w, vt[u], dr[u]);
        for (int32_t q = st[u] + 1; q < et[u]; ++q) {  // fibers longer than one nonzero
          V d[NV];
          RO::load(d, Dm, c2[q], c, Rr);
          RO::axpy(w, vals[q], d);
        }
        RO::hfma(acc, w, cr[u]);
      }
    }
  }
}

// Order-3 slice with short fibres (at most 1.25 nonzeros per fibre): lanes
// take the slice's nonzeros 64 at a time, each with its level-1 coordinate
// from the per-handle expansion, so the row gathers depend on one coalesced
// index load instead of the pos -> crd chain of the factorised walk;
// contribution = val * C(k,:) (.) D(l,:) per nonzero. Row group g takes
// nonzeros base + t*NG + g through lane shuffles, all row gathers of a
// chunk in flight at once.
template <int R>
__device__ __forceinline__ void slice3_short(const CsfDev& B, const FactorsDev& F, int32_t q0,
                                             int32_t q1, int lane, int gi, int c, int Rr, int wv,
                                             int nwv, typename Row<R>::V (&acc)[Row<R>::NV]) {
  using RO = Row<R>;
  using V = typename RO::V;
  constexpr int NV = RO::NV;
  constexpr int NG = 64 / RO::LPR;
  constexpr int NT = 64 / NG;
  const int32_t* __restrict__ kq = B.crd1_of_nnz;
  const int32_t* __restrict__ lq = B.crd[2];
  const float* __restrict__ vq = B.vals;
  const float* __restrict__ Cm = F.M[1];
  const float* __restrict__ Dm = F.M[2];
  for (int32_t base = q0 + 64 * wv; base < q1; base += 64 * nwv) {
    const int32_t q = base + lane;
    const bool okq = q < q1;
    const int32_t k = okq ? kq[q] : 0;
    const int32_t l = okq ? lq[q] : 0;
    const float v = okq ? vq[q] : 0.f;
    V cr[NT][NV], dr[NT][NV];
    float vt[NT];
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const int src = u * NG + gi;
      vt[u] = __shfl(v, src);
      RO::load(cr[u], Cm, __shfl(k, src), c, Rr);
      RO::load(dr[u], Dm, __shfl(l, src), c, Rr);
    }
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      V w[NV];
      RO::zero(w);
      RO::axpy(w, vt[u], dr[u]);
      RO::hfma(acc, w, cr[u]);
    }
  }
}

// One workgroup per root node; its blockDim/64 wavefronts split the slice
// (64-child chunks round-robin), reduce their rows with xor shuffles, then
// across wavefronts through LDS; one store per row, no atomics.
template <int N, int R>
__global__ __launch_bounds__(512) void slice_kernel(CsfDev B, FactorsDev F,
                                                    float* __restrict__ A,
                                                    int Rr) {
  using RO = Row<R>;
  using V = typename RO::V;
  constexpr int NV = RO::NV;
  constexpr int LPR = RO::LPR;
  constexpr int NG = 64 / LPR;
  __shared__ __align__(16) float red[8][Lay<R>::kMaxRank];
  const int32_t x = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  const int nwv = blockDim.x >> 6;
  const int gi = lane / LPR;
  const int c = lane % LPR;
  V acc[NV];
  RO::zero(acc);
  const int32_t a = B.pos[1][x];
  const int32_t e = B.pos[1][x + 1];
  if constexpr (N == 2) {
    // children are nonzeros: lanes load 64 at a time, row groups take them
    // through shuffles with every gather of a chunk in flight at once
    constexpr int NT = 64 / NG;
    for (int32_t base = a + 64 * wv; base < e; base += 64 * nwv) {
      const int32_t q = base + lane;
      const int32_t lq = q < e ? B.crd[1][q] : 0;
      const float vq = q < e ? B.vals[q] : 0.f;
      V d[NT][NV];
      float vt[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int src = t * NG + gi;
        vt[t] = __shfl(vq, src);
        RO::load(d[t], F.M[1], __shfl(lq, src), c, Rr);
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) RO::axpy(acc, vt[t], d[t]);
    }
  } else if constexpr (N == 3) {
    slice3_accumulate<R>(B, F, x, lane, gi, c, Rr, wv, nwv, acc);
  } else {
    for (int32_t y = a + wv * NG + gi; y < e; y += NG * nwv) {
      V s[NV];
      subtree<N, 1, R>(B, F, y, c, Rr, s);
      RO::add(acc, s);
    }
  }
  RO::wave_sum(acc);
  if (nwv == 1) {
    if (gi == 0) RO::store(A, B.crd0[x], c, Rr, acc);
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
    RO::store(A, B.crd0[x], c, Rr, acc);
  }
}

// Slice-row kernel for 3-mode tensors whose fibres are short (nnz at most
// 1.25 x fibres): the slice's nonzeros come straight from the per-handle
// expansion (slice3_short), then the same wave and LDS reduction and one
// store per row as slice_kernel.
template <int R>
__global__ __launch_bounds__(512) void slice_short_kernel(CsfDev B, FactorsDev F,
                                                          float* __restrict__ A, int Rr) {
  using RO = Row<R>;
  using V = typename RO::V;
  constexpr int NV = RO::NV;
  constexpr int LPR = RO::LPR;
  __shared__ __align__(16) float red[8][Lay<R>::kMaxRank];
  const int32_t x = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  const int nwv = blockDim.x >> 6;
  const int gi = lane / LPR;
  const int c = lane % LPR;
  V acc[NV];
  RO::zero(acc);
  slice3_short<R>(B, F, B.nnz_of_root[x], B.nnz_of_root[x + 1], lane, gi, c, Rr, wv, nwv, acc);
  RO::wave_sum(acc);
  if (nwv == 1) {
    if (gi == 0) RO::store(A, B.crd0[x], c, Rr, acc);
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
    RO::store(A, B.crd0[x], c, Rr, acc);
  }
}

// Slice-row kernel over the padded layout: one workgroup of pad_width
// threads per root node, each thread holding one slot, so the slice's
// nonzeros are read at addresses fixed at launch (no offset load first).
// Row groups take the wave's slots by shuffles as in slice_short_kernel,
// empty slots issue no gathers, and the same wave and LDS reduction ends in
// one store per row.
//
// Up to R = 32 the rows are global loads behind a branch per slot (empty
// slots skip them); from R = 64 they are buffer loads at 32-bit offsets, an
// empty slot passing an offset past the end, which reads zeros. The global
// form needs 155 (R = 64) to 256 (R = 128) VGPRs there, the buffer form 64;
// on the 4096^3 / 500k tensor the forms take 7.3 / 7.9 us at R = 32 and
// 13.5 / 13.0 us at R = 64.
//
// NW = pad width / 64 waves per workgroup (launch bounds and the LDS
// reduction sized to it); with an identity root (crd0[x] == x and one output
// row per slice) the row is the workgroup index, with no load.
template <int R, int NW>
__global__ __launch_bounds__(64 * NW) void slice_pad_kernel(CsfDev B, FactorsDev F,
                                                            float* __restrict__ A, int Rr,
                                                            int ident_root) {
  constexpr bool kBuffer = R >= 64;
  using RO = Row<R>;
  using V = typename RO::V;
  constexpr int NV = RO::NV;
  constexpr int LPR = RO::LPR;
  constexpr int NG = 64 / LPR;
  constexpr int NT = 64 / NG;
  constexpr int nwv = NW;
  __shared__ __align__(16) float red[NW][Lay<R>::kMaxRank];
  const int32_t x = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  const int gi = lane / LPR;
  const int c = lane % LPR;
  const uint2 e = B.pad[int64_t(x) * (64 * NW) + threadIdx.x];
  const int32_t row = ident_root ? x : B.crd0[x];
  const float* __restrict__ Cm = F.M[1];
  const float* __restrict__ Dm = F.M[2];
  const int32_t nrec = int32_t(65535u * uint32_t(R) * 4u);
  const __amdgpu_buffer_rsrc_t crs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(Cm), int16_t(0), nrec, 0x00020000);
  const __amdgpu_buffer_rsrc_t drs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(Dm), int16_t(0), nrec, 0x00020000);
  V cr[NT][NV], dr[NT][NV];
  float vt[NT];
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    const int src = u * NG + gi;
    const uint32_t kl0 = __shfl(e.x, src);
    const float v0 = __uint_as_float(__shfl(e.y, src));
    if constexpr (kBuffer) {
      // coordinates below 65535, so byte offsets fit 32 bits
      const bool real = kl0 != kPadEmpty;
      vt[u] = real ? v0 : 0.f;
      const uint32_t oc = real ? (kl0 >> 16) * uint32_t(R * 4) : 0x80000000u;
      const uint32_t od = real ? (kl0 & 0xFFFFu) * uint32_t(R * 4) : 0x80000000u;
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const uint32_t cj = uint32_t(RO::slot(j, c) * 4);
        cr[u][j] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(crs, oc + cj, 0, 0));
        dr[u][j] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(drs, od + cj, 0, 0));
      }
    } else {
      vt[u] = v0;
      if (kl0 != kPadEmpty) {
        RO::load(cr[u], Cm, int32_t(kl0 >> 16), c, Rr);
        RO::load(dr[u], Dm, int32_t(kl0 & 0xFFFFu), c, Rr);
      } else {
        RO::zero(cr[u]);
        RO::zero(dr[u]);
        vt[u] = 0.f;
      }
    }
  }
  V acc[NV];
  RO::zero(acc);
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    V w[NV];
    RO::zero(w);
    RO::axpy(w, vt[u], dr[u]);
    RO::hfma(acc, w, cr[u]);
  }
  RO::wave_sum(acc);
  if constexpr (nwv == 1) {
    if (gi == 0) RO::store(A, row, c, Rr, acc);
    return;
  }
  if (gi == 0) {
    RO::put(red[wv], c, acc);
  }
  __syncthreads();
  if (wv == 0 && gi == 0) {
#pragma unroll
    for (int w = 1; w < nwv; ++w) {
      V o[NV];
      RO::get(red[w], c, o);
      RO::add(acc, o);
    }
    RO::store(A, row, c, Rr, acc);
  }
}

// Two root nodes per workgroup over the paired slice layout: 2 waves, each
// lane taking two slots (t and t + 128) in two halves, rows by buffer loads
// at 32-bit offsets (an empty slot passes an offset past the end, which reads
// zeros, so no branch). Every product goes to the first or the second slice's
// accumulator by its slot index; both are reduced over the wave and through
// LDS and stored once. With 4096 slices of at most 192 nonzeros the 2048
// two-wave workgroups are all resident at once, where one 192-thread
// workgroup per slice takes about 2.7 rounds of the GPU (83 VGPRs).
template <int R>
__global__ __launch_bounds__(128) void slice_pair_kernel(const uint2* __restrict__ slots,
                                                         const int4* __restrict__ info,
                                                         FactorsDev F, float* __restrict__ A,
                                                         int Rr) {
  using RO = Row<R>;
  using V = typename RO::V;
  constexpr int NV = RO::NV;
  constexpr int LPR = RO::LPR;
  constexpr int NG = 64 / LPR;
  constexpr int NT = 64 / NG;
  constexpr int NW = 2;
  __shared__ __align__(16) float red[NW][2][Lay<R>::kMaxRank];
  const int32_t g = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  const int gi = lane / LPR;
  const int c = lane % LPR;
  uint2 e[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) e[h] = slots[int64_t(g) * kPairSlots + h * 128 + threadIdx.x];
  const int4 inf = info[g];
  const float* __restrict__ Cm = F.M[1];
  const float* __restrict__ Dm = F.M[2];
  const int32_t nrec = int32_t(65535u * uint32_t(R) * 4u);
  const __amdgpu_buffer_rsrc_t crs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(Cm), int16_t(0), nrec, 0x00020000);
  const __amdgpu_buffer_rsrc_t drs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(Dm), int16_t(0), nrec, 0x00020000);
  V aa[NV], ab[NV];
  RO::zero(aa);
  RO::zero(ab);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    V cr[NT][NV], dr[NT][NV];
    float vt[NT];
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const int src = u * NG + gi;
      const uint32_t kl = __shfl(e[h].x, src);
      const float v0 = __uint_as_float(__shfl(e[h].y, src));
      // coordinates below 65535, so byte offsets fit 32 bits
      const bool real = kl != kPadEmpty;
      vt[u] = real ? v0 : 0.f;
      const uint32_t oc = real ? (kl >> 16) * uint32_t(R * 4) : 0x80000000u;
      const uint32_t od = real ? (kl & 0xFFFFu) * uint32_t(R * 4) : 0x80000000u;
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const uint32_t cj = uint32_t(RO::slot(j, c) * 4);
        cr[u][j] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(crs, oc + cj, 0, 0));
        dr[u][j] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(drs, od + cj, 0, 0));
      }
    }
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const int slot = h * 128 + wv * 64 + u * NG + gi;
      const float va = slot < inf.z ? vt[u] : 0.f;
      const float vb = vt[u] - va;
      V w[NV];
      RO::zero(w);
      RO::axpy(w, va, dr[u]);
      RO::hfma(aa, w, cr[u]);
      RO::zero(w);
      RO::axpy(w, vb, dr[u]);
      RO::hfma(ab, w, cr[u]);
    }
  }
  RO::wave_sum(aa);
  RO::wave_sum(ab);
  if (gi == 0) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      *reinterpret_cast<float4*>(&red[wv][0][RO::slot(j, c)]) = aa[j];
      *reinterpret_cast<float4*>(&red[wv][1][RO::slot(j, c)]) = ab[j];
    }
  }
  __syncthreads();
  // wave 0 stores the first slice's row, wave 1 the second's
  if (gi == 0) {
    V t[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const float4 o0 = *reinterpret_cast<const float4*>(&red[0][wv][RO::slot(j, c)]);
      const float4 o1 = *reinterpret_cast<const float4*>(&red[1][wv][RO::slot(j, c)]);
      t[j] = make_float4(o0.x + o1.x, o0.y + o1.y, o0.z + o1.z, o0.w + o1.w);
    }
    const int32_t row = wv == 0 ? inf.x : inf.y;
    if (row >= 0) RO::store(A, row, c, Rr, t);
  }
}


// Persistent workgroups over the items of one order's tasks (the device
// task table is sorted by order: tasks [t_lo, t_hi) hold items [i_lo, i_hi)),
// so each order runs with its own register and LDS footprint. schedule 0
// pulls items from the order's device counter (reset by the prep launch) in
// arrival order; schedule 1 is a static cyclic assignment (item = i_lo +
// block + k * grid). Either way a workgroup's items increase, so its task
// cursor only moves forward.
template <int N, int R, bool EP>
__global__ __launch_bounds__(512) void batch_kernel(const BatchTaskDev* __restrict__ tasks,
                                                    int32_t t_lo, int32_t t_hi,
                                                    const int64_t* __restrict__ item_off,
                                                    int32_t i_lo, int32_t i_hi,
                                                    int32_t* __restrict__ counter, int Rr,
                                                    int32_t G, int32_t NB, int dynamic) {
  // the batch has no FP64 row buffer, which the edge-serial walk needs
  static_assert(EP, "the batch runs the edge-parallel walk only");
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int32_t s_item;
  int32_t t = -1;
  int64_t t_end = 0;
  int32_t item = i_lo + int32_t(blockIdx.x);
  for (;;) {
    __syncthreads();  // the previous item's LDS reads are done
    if (dynamic) {
      if (threadIdx.x == 0) s_item = i_lo + atomicAdd(counter, 1);
      __syncthreads();
      item = __builtin_amdgcn_readfirstlane(s_item);
    }
    if (item >= i_hi) break;
    if (t < 0) {
      t = t_lo + upper_index(item_off + t_lo, t_hi - t_lo, item);
      t_end = item_off[t + 1];
    }
    while (item >= t_end) {
      ++t;
      t_end = item_off[t + 1];
    }
    const BatchTaskDev& T = tasks[t];
    const int32_t b = item - int32_t(item_off[t]);
    edge_block<N, R, EP>(T.B, T.F, T.A, Rr, T.brk, b, G, NB, smem, nullptr);
    if (!dynamic) item += int32_t(gridDim.x);
  }
}

template <int N, int R>
int launch_batch_order(const BatchLaunch& L, hipStream_t st) {
  const int32_t i_lo = L.grp_item[N], i_hi = L.grp_item[N + 1];
  if (i_hi <= i_lo) return TENTACO_OK;
  const int lpr = Row<R>::LPR;
  const int blk = L.blk[N];
  const size_t lds = edge_stage_ints(N, L.nb[N]) * sizeof(int32_t) + edge_ep_bytes(blk, lpr, L.R);
  if (lds > 65536) return fail(TENTACO_EUNSUPPORTED, "batch LDS %zu B", lds);
  const int grid = std::max(1, std::min<int>(L.grp_grid[N], i_hi - i_lo));
  batch_kernel<N, R, true><<<grid, blk, lds, st>>>(
      L.tasks, L.grp_task[N], L.grp_task[N + 1], L.item_off, i_lo, i_hi, L.counter + N, L.R,
      L.grp[N], L.nb[N], L.sch[N] == 0);
  TT_HIP_CHECK(hipGetLastError());
  return TENTACO_OK;
}

template <int N, int R>
int batch_occupancy_order(int family, int block, int Rr, int32_t NB, int* per_cu) {
  const int lpr = Row<R>::LPR;
  if (family != kEdgeParallel)
    return fail(TENTACO_EUNSUPPORTED, "the batch runs the edge-parallel walk only");
  const size_t lds = edge_stage_ints(N, NB) * sizeof(int32_t) + edge_ep_bytes(block, lpr, Rr);
  const hipError_t e =
      hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, batch_kernel<N, R, true>, block, lds);
  if (e != hipSuccess) return fail(TENTACO_EHIP, "occupancy query: %s", hipGetErrorString(e));
  return TENTACO_OK;
}

template <int N, int R>
int launch_typed(const CsfDev& B, const FactorsDev& F, int Rr, float* A,
                 int32_t a_rows, bool dense_root, const Variant& vr, void* ws,
                 hipStream_t st) {
  const int64_t a_elems = int64_t(a_rows) * Rr;
  if (vr.family == kSliceRow) {
    if (!dense_root) {
      const int rc = launch_fill(A, a_elems, 0.f, st);
      if (rc) return rc;
    }
    if (B.nodes[0] > 0) {
      ktimer_begin(st);
      if constexpr (N == 3 && R > 0) {
        // short fibres (nnz <= 1.25 x fibres) with the expansion built: the
        // kernel that skips the pos -> crd chain
        if (B.crd1_of_nnz && int64_t(B.nnz) * 4 <= int64_t(B.nodes[1]) * 5) {
          if constexpr (R == 16 || R == 32 || R == 64) {
            if (B.pair && vr.block >= 256) {
              slice_pair_kernel<R><<<B.npairs, 128, 0, st>>>(B.pair, B.pair_info, F, A, Rr);
              TT_HIP_CHECK(hipGetLastError());
              ktimer_end(st, "slice_pair_kernel");
              return TENTACO_OK;
            }
          }
          if (B.pad && B.pad_width <= vr.block && B.pad_width % 64 == 0 && B.pad_width <= 512) {
            const int id = dense_root ? 1 : 0;
            switch (B.pad_width / 64) {
              case 1: slice_pad_kernel<R, 1><<<B.nodes[0], 64, 0, st>>>(B, F, A, Rr, id); break;
              case 2: slice_pad_kernel<R, 2><<<B.nodes[0], 128, 0, st>>>(B, F, A, Rr, id); break;
              case 3: slice_pad_kernel<R, 3><<<B.nodes[0], 192, 0, st>>>(B, F, A, Rr, id); break;
              case 4: slice_pad_kernel<R, 4><<<B.nodes[0], 256, 0, st>>>(B, F, A, Rr, id); break;
              case 5: slice_pad_kernel<R, 5><<<B.nodes[0], 320, 0, st>>>(B, F, A, Rr, id); break;
              case 6: slice_pad_kernel<R, 6><<<B.nodes[0], 384, 0, st>>>(B, F, A, Rr, id); break;
              case 7: slice_pad_kernel<R, 7><<<B.nodes[0], 448, 0, st>>>(B, F, A, Rr, id); break;
              default: slice_pad_kernel<R, 8><<<B.nodes[0], 512, 0, st>>>(B, F, A, Rr, id); break;
            }
            TT_HIP_CHECK(hipGetLastError());
            ktimer_end(st, "slice_pad_kernel");
            return TENTACO_OK;
          }
          slice_short_kernel<R><<<B.nodes[0], vr.block, 0, st>>>(B, F, A, Rr);
          TT_HIP_CHECK(hipGetLastError());
          ktimer_end(st, "slice_short_kernel");
          return TENTACO_OK;
        }
      }
      slice_kernel<N, R><<<B.nodes[0], vr.block, 0, st>>>(B, F, A, Rr);
      TT_HIP_CHECK(hipGetLastError());
      ktimer_end(st, "slice_kernel");
    }
    return TENTACO_OK;
  }
  const int64_t NB = nnz_per_block(vr, Rr);
  const int64_t nblk = (int64_t(B.nnz) + NB - 1) / NB;
  int32_t* brk = static_cast<int32_t*>(ws);
  // edge-serial: rows accumulate in FP64 (W, after the brackets), narrowed
  // to A at the end; the prep zeroes W instead of A
  double* W = (vr.family == kEdgeSerial && nblk > 0)
                  ? reinterpret_cast<double*>(static_cast<char*>(ws) + edge_brk_bytes(B, NB))
                  : nullptr;
  {
    float* Z = W ? reinterpret_cast<float*>(W) : A;
    const int64_t z_elems = W ? 2 * a_elems : a_elems;
    const int rc = launch_edge_prep(B, Z, z_elems, brk, int32_t(nblk), int32_t(NB), st);
    if (rc) return rc;
  }
  if (nblk == 0) return TENTACO_OK;
  const int lpr = Row<R>::LPR;
  const size_t stage = edge_stage_ints(N, int32_t(NB)) * sizeof(int32_t);
  if (vr.family == kEdgeSerial) {
    if (stage > 65536)
      return fail(TENTACO_EUNSUPPORTED, "edge-serial tile of %lld nonzeros needs %zu B of LDS",
                  (long long)NB, stage);
    ktimer_begin(st);
    edge_kernel<N, R, false><<<int(nblk), vr.block, stage, st>>>(
        B, F, A, Rr, brk, vr.group, int32_t(NB), W);
    TT_HIP_CHECK(hipGetLastError());
    ktimer_end(st, "edge_kernel");
    return launch_narrow(W, A, a_elems, st);
  } else {
    const size_t lds = edge_ep_bytes(vr.block, lpr, Rr) + stage;
    if (lds > 65536)
      return fail(TENTACO_EUNSUPPORTED, "edge-parallel block %d at rank %d needs %zu B of LDS",
                  vr.block, Rr, lds);
    ktimer_begin(st);
    edge_kernel<N, R, true><<<int(nblk), vr.block, lds, st>>>(
        B, F, A, Rr, brk, vr.group, int32_t(NB), nullptr);
  }
  TT_HIP_CHECK(hipGetLastError());
  ktimer_end(st, "edge_kernel");
  return TENTACO_OK;
}

template <int N, int L, int R>
int launch_inner_typed(const CsfDev& B, const LevelIndex& X, const FactorsDev& F, int Rr, float* A,
                       int32_t a_rows, hipStream_t st) {
  if (a_rows <= 0) return TENTACO_OK;
  // 1-4 waves per row, from the mean level-L nodes per row
  const int64_t mean = (int64_t(B.nodes[L]) + X.dim - 1) / std::max<int32_t>(X.dim, 1);
  const int per_wave = 64 / Row<R>::LPR;
  const int nwv = int(std::max<int64_t>(1, std::min<int64_t>(4, (mean + 4 * per_wave - 1) /
                                                                   (4 * per_wave))));
  ktimer_begin(st);
  inner_kernel<N, L, R><<<a_rows, 64 * nwv, 0, st>>>(X.tpos, X.dim, X.node, X.anc, B, F, A, Rr);
  TT_HIP_CHECK(hipGetLastError());
  ktimer_end(st, "inner_kernel");
  return TENTACO_OK;
}

template <int N, int R>
int launch_inner_order(const CsfDev& B, const LevelIndex& X, const FactorsDev& F, int level,
                       int Rr, float* A, int32_t a_rows, hipStream_t st) {
  if constexpr (N >= 3) {
    if (level == 1) return launch_inner_typed<N, 1, R>(B, X, F, Rr, A, a_rows, st);
  }
  if constexpr (N >= 4) {
    if (level == 2) return launch_inner_typed<N, 2, R>(B, X, F, Rr, A, a_rows, st);
  }
  if constexpr (N >= 5) {
    if (level == 3) return launch_inner_typed<N, 3, R>(B, X, F, Rr, A, a_rows, st);
  }
  return fail(TENTACO_EINVAL, "level %d is not an inner level of an order-%d tensor", level, N);
}

template <int N, int L, int R>
int launch_level_typed(const CsfDev& B, const FactorsDev& F, int Rr, float* A, int32_t a_rows,
                       hipStream_t st) {
  const int64_t a_elems = int64_t(a_rows) * Rr;
  const int rc = launch_fill(A, a_elems, 0.f, st);
  if (rc) return rc;
  const int32_t ny = B.nodes[L];
  if (ny <= 0) return TENTACO_OK;
  // chunks of CH level-L nodes, about 2^16 row groups in all
  const int32_t CH = int32_t(std::max<int64_t>(4, (int64_t(ny) + 65535) / 65536));
  const int64_t groups = (int64_t(ny) + CH - 1) / CH;
  const int per_block = 256 / Row<R>::LPR;
  const int grid = grid_for(groups, per_block, 65536);
  ktimer_begin(st);
  level_kernel<N, L, R><<<grid, 256, 0, st>>>(B, F, A, Rr, CH);
  TT_HIP_CHECK(hipGetLastError());
  ktimer_end(st, "level_kernel");
  return TENTACO_OK;
}

template <int N, int R>
int launch_level_order(const CsfDev& B, const FactorsDev& F, int level, int Rr, float* A,
                       int32_t a_rows, hipStream_t st) {
  if constexpr (N >= 2) {
    if (level == 1) return launch_level_typed<N, 1, R>(B, F, Rr, A, a_rows, st);
  }
  if constexpr (N >= 3) {
    if (level == 2) return launch_level_typed<N, 2, R>(B, F, Rr, A, a_rows, st);
  }
  if constexpr (N >= 4) {
    if (level == 3) return launch_level_typed<N, 3, R>(B, F, Rr, A, a_rows, st);
  }
  if constexpr (N >= 5) {
    if (level == 4) return launch_level_typed<N, 4, R>(B, F, Rr, A, a_rows, st);
  }
  return fail(TENTACO_EINVAL, "level %d outside 1..%d", level, N - 1);
}

}  // namespace

// ---- one tensor order's entry points (mttkrp_dispatch.h) --------------------
template <int N>
int order_mttkrp(const CsfDev& B, const FactorsDev& F, int R, float* A, int32_t a_rows,
                 bool dense_root, const Variant& vr, void* ws, hipStream_t st) {
  return with_rank_layout(R, [&](auto r) {
    return launch_typed<N, r()>(B, F, R, A, a_rows, dense_root, vr, ws, st);
  });
}

template <int N>
int order_inner(const CsfDev& B, const LevelIndex& X, const FactorsDev& F, int level, int R,
                float* A, int32_t a_rows, hipStream_t st) {
  return with_rank_layout(
      R, [&](auto r) { return launch_inner_order<N, r()>(B, X, F, level, R, A, a_rows, st); });
}

template <int N>
int order_level(const CsfDev& B, const FactorsDev& F, int level, int R, float* A, int32_t a_rows,
                hipStream_t st) {
  return with_rank_layout(
      R, [&](auto r) { return launch_level_order<N, r()>(B, F, level, R, A, a_rows, st); });
}

template <int N>
int order_batch(const BatchLaunch& L, hipStream_t st) {
  switch (L.R) {
    case 16: return launch_batch_order<N, 16>(L, st);
    case 32: return launch_batch_order<N, 32>(L, st);
    default: return launch_batch_order<N, 64>(L, st);
  }
}

template <int N>
int order_batch_occupancy(int family, int block, int R, int32_t NB, int* per_cu) {
  switch (R) {
    case 16: return batch_occupancy_order<N, 16>(family, block, R, NB, per_cu);
    case 32: return batch_occupancy_order<N, 32>(family, block, R, NB, per_cu);
    default: return batch_occupancy_order<N, 64>(family, block, R, NB, per_cu);
  }
}

}  // namespace tt

// Instantiates order N's entry points (one source per order).
#define TT_INSTANTIATE_ORDER(N)                                                                 \
  template int tt::order_mttkrp<N>(const CsfDev&, const FactorsDev&, int, float*, int32_t, bool, \
                                   const Variant&, void*, hipStream_t);                         \
  template int tt::order_inner<N>(const CsfDev&, const LevelIndex&, const FactorsDev&, int, int, \
                                  float*, int32_t, hipStream_t);                                \
  template int tt::order_level<N>(const CsfDev&, const FactorsDev&, int, int, float*, int32_t,  \
                                  hipStream_t);                                                 \
  template int tt::order_batch<N>(const BatchLaunch&, hipStream_t);                             \
  template int tt::order_batch_occupancy<N>(int, int, int, int32_t, int*);
