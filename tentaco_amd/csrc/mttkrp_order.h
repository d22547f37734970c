// The MTTKRP kernels templated on tensor order and rank layout, with their
// launches (the kernels' overview is in mttkrp.hip). Each order N is
// instantiated in its own source, mttkrp_o<N>.hip, so that the orders compile
// in parallel.
#pragma once

#include <algorithm>
#include <cfloat>
#include <climits>

#include "index_range.h"
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
// Every wave owns a contiguous run of NGW*G nonzeros (NGW row groups) and
// walks it in chunks of up to 64, one nonzero per lane. A chunk's leaf pairs
// and, per level, the next 64 node bounds and coordinates arrive in coalesced
// loads one chunk ahead. A lane's node at a level is the chunk's first node
// plus the number of later nodes that start at or before its child: a
// histogram of the starts over the chunk's children and a lane scan, so no
// lane searches or branches on its own. The chunk then splits into pieces of
// one slice and at most PF fibres (a whole chunk where slices are long). For
// a piece, the product of the upper levels' rows is formed once per fibre and
// kept in LDS (P); the row groups take the piece's nonzeros in turn, each
// step one leaf row by a global load and one P row from LDS:
//   acc += (val * M_{N-1}(l, :)) (.) P(fibre, :).
// (At orders 4 and 5 P is a product of rows itself. Where it passes FP32's range,
// or falls below the normal numbers under a value times leaf row above kSafe, the
// rows multiply the value's leaf row one by one: 1e30 * 1e-15 * 1e-15 * 1e-15 *
// 1e-15 is no 0. The check is an instruction a column and product. Products that
// underflow under ordinary values are common, in CP-ALS on skewed tensors columns
// concentrate within a few sweeps, and what is lost there is below 2^-139: a sweep
// of three tensors 560 us without the check, 690 with the rows one by one whenever
// a product underflows.)
// Slice changes are uniform over the wave: the row groups' accumulators are
// summed over the wave and the row is stored.
//
// The serial walk it replaces gave every row group a run of its own and
// closed fibres per group; some group of a wave closed one on most steps, and
// the closing's instructions bound it where the factors fit L2, and drained
// the row gathers in flight where they do not. Per call, before and after:
// 2M nonzeros, 3-mode, rank 32 (10007 x 20011 x 5003) 61 and 45 us; 100M,
// 3-mode, rank 32 (500k^3) 2281 and 2099 us (of 1960 us at the random-row rate
// of a 64 MB factor); 60M, 4-mode, rank 64 (200k^4) 2845 and 2415 us; 5M at
// rank 50 229 and 165 us. What is left where the factors fit L2 is the
// latency of a chunk's dependent steps and about 4 vector instructions a
// nonzero.
//
// Rows: the workgroups' shared rows are FP64 ones. Without them a long slice's
// row takes an FP32 addition per workgroup, and a run is summed in two levels
// to leave that the room it had: a chunk's nonzeros, then (in LDS, a lane each)
// the chunks. One chain over a run of 512 had 1.2 to 1.4 times the error at the
// same tile: 1.85 and 1.43e-7 against FP64 for 400k nonzeros, 2.14 and 1.85 for
// 12M at rank 128, in two levels 1.25 and 1.79. With FP64 rows the chain stays
// (1.0 and 1.5e-7, 2044 us for 100M nonzeros; 2083 in two levels).
//
// LDS per wave (edge_wave_lds bytes): a record per nonzero of the chunk
// (leaf row, value, fibre), the histogram, P, the wave's first slice's row, and
// without Rows the earlier chunks' sums; the block's combine reuses P and the
// histogram.
constexpr int kRecBytes = 64 * 16;
constexpr int kHistBytes = 64 * 4;
constexpr int kFibBytes = 4096;

template <int R, bool Rows>
constexpr size_t edge_wave_lds() {
  return kRecBytes + kHistBytes + kFibBytes + Lay<R>::kMaxRank * sizeof(float) +
         (Rows ? 0 : 64 * Row<R>::NV * sizeof(typename Row<R>::V));
}

// Largest x in [lo, hi] with a[x] <= key (requires a[lo] <= key), 64 probes a
// step, uniform over the wave.
__device__ __forceinline__ int32_t wave_search_le(const int32_t* __restrict__ a, int32_t lo,
                                                  int32_t hi, int32_t key, int lane) {
  while (lo < hi) {
    const uint32_t n = uint32_t(hi - lo);
    const uint32_t step = (n + 63u) >> 6;
    const uint32_t off = uint32_t(lane + 1) * step;
    const bool le = off <= n && a[lo + int32_t(off <= n ? off : n)] <= key;
    const uint32_t cnt = uint32_t(__popcll(__ballot(le)));
    const uint32_t next = cnt * step;
    hi = lo + int32_t(min(n, next + step - 1u));
    lo += int32_t(next);
  }
  return lo;
}

// Where a wave's run starts comes from `starts` (the node of its first
// nonzero at every level, N-1 per wave, waves in order), a table that depends
// on the CSF and the run length only and that a handle or a batch keeps; or,
// with starts null, from the block's brackets brk (the same per block) by a
// search of its own.
template <int N, int R, bool EP, bool Rows, bool Batch = false>
__device__ __forceinline__ void edge_block(const CsfDev& B, const FactorsDev& F, float* out_a,
                                           int Rr, const int32_t* brk_p, const int32_t* starts_p,
                                           int32_t b, int32_t G, int32_t NB, unsigned char* smem,
                                           double* out_w, const int2* slots) {
  using RO = Row<R>;
  using V = typename RO::V;
  constexpr int NV = RO::NV;
  constexpr int LPR = RO::LPR;
  constexpr int KR = Lay<R>::kMaxRank;
  constexpr int NGW = 64 / LPR;             // row groups of a wave
  constexpr int NL = N - 1;                 // levels 0..N-2 hold nodes
  constexpr int FL = N - 2;                 // the nonzeros' parents (fibres)
  constexpr int PF0 = kFibBytes / (KR * 4); // fibres whose product rows fit P
  constexpr int PF = PF0 < 64 ? PF0 : 64;
  // slices of a chunk from which their nonzeros' products are summed from LDS,
  // PF at a time: about twice as many as the chunk has such rounds
  constexpr int kManySlices = 128 / PF < 3 ? 3 : 128 / PF;
  // leaf rows in flight per row group, at most 32 VGPRs of them
  constexpr int SB = NV >= 4 ? 2 : NV == 2 ? 4 : LPR < 8 ? LPR : 8;
  float* __restrict__ A = global_ptr(out_a);
  double* __restrict__ W = global_ptr(out_w);
  const int32_t* __restrict__ brk = global_ptr(brk_p);
  const int32_t* __restrict__ starts = global_ptr(starts_p);

  // read here: at the end its latency would stand alone
  const int2 slot = Rows ? *slots : make_int2(0, 0);

  const int lane = int(threadIdx.x) & 63;
  const int wv = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int nwv = int(blockDim.x) >> 6;
  const int gi = lane / LPR;
  const int c = lane % LPR;
  auto wave_mem = [&](int w) { return smem + size_t(w) * edge_wave_lds<R, Rows>(); };
  int4* rec = reinterpret_cast<int4*>(wave_mem(wv));
  int32_t* hist = reinterpret_cast<int32_t*>(wave_mem(wv) + kRecBytes);
  float* P = reinterpret_cast<float*>(wave_mem(wv) + kRecBytes + kHistBytes);
  float* head_row = P + kFibBytes / 4;
  V* earlier = reinterpret_cast<V*>(head_row + KR) + lane * NV;  // this lane's

  // the wave's run [w0, w1)
  const int32_t blk0 = b * NB;
  const int32_t len = min(NB, B.nnz - blk0);
  const int32_t off = wv * (NGW * G);
  const bool active = off < len;
  const int32_t w0 = blk0 + off;
  const int32_t w1 = active ? w0 + min(NGW * G, len - off) : w0;

  V acc[NV];
  RO::zero(acc);
  int32_t head = INT_MAX, open = INT_MAX;
  bool head_closed = false;
  bool has_earlier = false;  // of the open slice
  auto take_earlier = [&]() {
    if (!has_earlier) return;
    has_earlier = false;
    V t[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) t[j] = earlier[j];
    RO::add(acc, t);
  };

  if (active) {
    const int32_t* __restrict__ lcrd = global_ptr(B.crd[N - 1]);
    const float* __restrict__ vals = global_ptr(B.vals);
    const float* __restrict__ Mleaf = global_ptr(F.M[N - 1]);
    // per level: its nodes' child ranges, their coordinates and factor
    const int32_t* __restrict__ pos[NL];
    const int32_t* __restrict__ crd[NL];
    const float* __restrict__ M[NL];
#pragma unroll
    for (int k = 0; k < NL; ++k) {
      pos[k] = global_ptr(B.pos[k + 1]);
      crd[k] = global_ptr(k == 0 ? B.crd0 : B.crd[k]);
      M[k] = global_ptr(F.M[k]);
    }
    // cur[k]: the node at level k that holds the chunk's first nonzero
    int32_t cur[NL];
    if (starts) {
      const int32_t* st = starts + (int64_t(b) * nwv + wv) * NL;
#pragma unroll
      for (int k = 0; k < NL; ++k) cur[k] = __builtin_amdgcn_readfirstlane(st[k]);
    } else {
      int32_t key = w0;
#pragma unroll
      for (int k = FL; k >= 0; --k) {
        const int32_t lo = brk[b * NL + k];
        const int32_t hi = wv == 0 ? lo : brk[(b + 1) * NL + k];
        cur[k] = wave_search_le(pos[k], lo, hi, key, lane);
        key = cur[k];
      }
    }
    head = open = cur[0];

    // The windows of a chunk: wp[k] lane j = where node cur[k]+1+j starts
    // among the level's children (the level's total past its last node),
    // wc[k] lane j = coordinate of node cur[k]+j.
    int32_t wp[NL], wc[NL];
    auto window = [&](int k, int32_t x, int32_t& p, int32_t& cc) {
      p = pos[k][index_ahead(x, 1 + lane, B.nodes[k])];
      cc = crd[k][index_ahead(x, lane, B.nodes[k] - 1)];
    };
    auto pairs = [&](int32_t q, int32_t& l, float& v) {
      const int32_t t = index_ahead(q, lane, w1 - 1);
      l = lcrd[t];
      v = vals[t];
    };
    // lane x: how many of the starts p (ascending over the lanes) are <= base + x
    auto rank = [&](int32_t p, int32_t base) -> int32_t {
      const uint32_t s = uint32_t(p - base);
      hist[lane] = 0;
      wave_lds_sync();
      if (s < 64u) atomicAdd(&hist[s], 1);
      wave_lds_sync();
      const int32_t n = hist[lane];
      wave_lds_sync();
      return wave_scan_add(n);
    };
    auto lane_of = [&](int32_t x, int32_t src) { return __builtin_amdgcn_readlane(x, src); };

    int32_t open_row = 0;
    auto close_slice = [&]() {
      take_earlier();
      RO::wave_sum(acc);
      if (open == head && !head_closed) {
        head_closed = true;
        if (gi == 0) RO::put(head_row, c, acc);
      } else if (gi == 0) {
        if constexpr (EP) RO::store(A, open_row, c, Rr, acc);
        else RO::store_f64(W, open_row, c, Rr, acc);
      }
      RO::zero(acc);
    };

    int32_t l, lnext = 0;
    float v, vnext = 0.f;
    pairs(w0, l, v);
#pragma unroll
    for (int k = 0; k < NL; ++k) window(k, cur[k], wp[k], wc[k]);

    for (int32_t q = w0; q < w1;) {
      // move past nodes that end at or before the chunk's first child (empty
      // nodes, or a window the last chunk used up)
#pragma unroll
      for (int k = FL; k >= 0; --k) {
        const int32_t key = k == FL ? q : cur[k + 1];
        const int past = __popcll(__ballot(wp[k] <= key));
        if (past) {
          cur[k] += past;
          if (past == 64)
            cur[k] = wave_search_le(pos[k], cur[k], B.nodes[k] - 1, key, lane);
          window(k, cur[k], wp[k], wc[k]);
        }
      }
      // the chunk ends where a level's window does
      int32_t n = 64;
#pragma unroll
      for (int k = 0; k < NL; ++k) {
        const int32_t key = k == FL ? q : cur[k + 1];
        n = min(64, lane_of(wp[k], n - 1) - key);
      }
      n = min(n, w1 - q);
      // local node of every child, bottom up; then the fibres' ancestors
      int32_t loc[NL];  // loc[k] lane x: node of child x of the chunk
      int32_t cnt[NL];  // nodes of the chunk
#pragma unroll
      for (int k = FL; k >= 0; --k) {
        const int32_t key = k == FL ? q : cur[k + 1];
        const int32_t m = k == FL ? n : cnt[k + 1];
        loc[k] = 0;
        if (lane_of(wp[k], 0) - key < m) loc[k] = rank(wp[k], key);
        cnt[k] = lane_of(loc[k], m - 1) + 1;
      }
      int32_t fc[NL];      // fc[k] lane f: coordinate at level k above fibre f
      int32_t root = loc[0];  // lane f: root node of fibre f (of nonzero f for N = 2)
      {
        int32_t an = lane;
        fc[FL] = wc[FL];
#pragma unroll
        for (int k = FL - 1; k >= 0; --k) {
          an = k == FL - 1 ? loc[k] : __shfl(loc[k], an);
          fc[k] = __shfl(wc[k], an);
        }
        if constexpr (N > 2) root = an;
      }
      rec[lane] = make_int4(l, __float_as_int(v), loc[FL], 0);
      wave_lds_sync();
      // the next chunk's loads
      const int32_t qn = q + n;
      int32_t curn[NL], wpn[NL], wcn[NL];
      if (qn < w1) {
        pairs(qn, lnext, vnext);
#pragma unroll
        for (int k = FL; k >= 0; --k) {
          const int32_t key = k == FL ? qn : curn[k + 1];
          curn[k] = cur[k] + __popcll(__ballot(wp[k] <= key));
          window(k, curn[k], wpn[k], wcn[k]);
        }
      }
      // slices of the chunk: the mask of their first nonzeros
      const int32_t rq = N > 2 ? __shfl(root, loc[FL]) : root;  // lane q: nonzero q's root
      const int32_t rbefore = __shfl_up(rq, 1);
      const bool first_of = lane < n && (lane == 0 || rq != rbefore);
      const uint64_t starts_of = __ballot(first_of);
      const int32_t ns = __popcll(starts_of);
      const bool many = ns >= kManySlices;
      if (many) {
        // Many slices: the products of PB nonzeros at a time go to LDS, all
        // their rows in flight at once, and the row groups then sum a slice
        // each. Taken as pieces, every slice would wait for its own rows.
        const int32_t ord = __popcll(starts_of & ((2ull << lane) - 1ull)) - 1;
        if (first_of) hist[ord] = lane;  // first nonzero of slice `ord`
        wave_lds_sync();
        constexpr int PB = PF;
        constexpr int U = PB / NGW;
        for (int32_t s0 = 0; s0 < n; s0 += PB) {
          const int32_t m = min(PB, n - s0);
          V d[U][NV];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int4 x = rec[s0 + min(u * NGW + gi, m - 1)];
            RO::load(d[u], Mleaf, x.x, c, Rr);
            RO::scale(d[u], __int_as_float(x.y));
#pragma unroll
            for (int k = FL; k >= 1; --k) {
              V p[NV];
              RO::load(p, M[k], __shfl(fc[k], x.z), c, Rr);
              RO::hmul(d[u], p);
            }
          }
#pragma unroll
          for (int u = 0; u < U; ++u)
            if (u * NGW + gi < m) RO::put(P + (u * NGW + gi) * KR, c, d[u]);
          wave_lds_sync();
          const int32_t o0 = lane_of(ord, s0), o1 = lane_of(ord, s0 + m - 1);
          const int32_t r0 = lane_of(rq, s0);
          if (cur[0] + r0 != open) {
            close_slice();
            open = cur[0] + r0;
            open_row = lane_of(wc[0], r0);
          }
          // slice o0 continues the open one, o1 stays open
          V last[NV];
          RO::zero(last);
          for (int32_t ob = o0; ob <= o1; ob += NGW) {
            const int32_t o = min(ob + gi, o1);
            const int32_t a = max(hist[o], s0);
            const int32_t e = o + 1 < ns ? min(hist[min(o + 1, 63)], s0 + m) : s0 + m;
            const int32_t row = __shfl(wc[0], __shfl(rq, a));
            // (in FP64: in FP32 a serial sum of 20 had 1.2 times the error of the
            // nested sums before; the batch, where it costs 20%, stays with FP32)
            std::conditional_t<Batch, V[NV], typename RO::D> total = {};
            if (ob + gi <= o1)
              for (int32_t i = a; i < e; ++i) {
                V p[NV];
                RO::get(P + (i - s0) * KR, c, p);
                RO::add(total, p);
              }
            V sum[NV];
            RO::narrow(sum, total);
            if (o == o0) {
              RO::add(acc, sum);
            } else if (o == o1) {
              RO::add(last, sum);
            } else if constexpr (EP) {
              RO::store(A, row, c, Rr, sum);
            } else {
              RO::store_f64(W, row, c, Rr, sum);
            }
          }
          if (o1 > o0) {
            close_slice();
#pragma unroll
            for (int j = 0; j < NV; ++j) acc[j] = last[j];
            const int32_t r1 = lane_of(rq, s0 + m - 1);
            open = cur[0] + r1;
            open_row = lane_of(wc[0], r1);
          }
          wave_lds_sync();
        }
      }
      // few: pieces, nonzeros [a, e) of one slice in fibres [fa, fe)
      const int32_t nf = N > 2 ? cnt[FL] : n;
      for (int32_t a = many ? n : 0, fa = 0; a < n;) {
        const int32_t r = lane_of(root, fa);
        const int32_t fe =
            fa + __popcll(__ballot(lane >= fa && lane < min(nf, N > 2 ? fa + PF : 64) && root == r));
        const int32_t e = N == 2 ? fe : (fe >= nf ? n : lane_of(wp[FL], fe - 1) - q);
        if (cur[0] + r != open) {
          close_slice();
          open = cur[0] + r;
        }
        open_row = lane_of(wc[0], r);
        bool staged = N == 2;
        bool odd = false, over = false;  // P has products that are no normal numbers, or past them
        auto stage = [&]() {
          constexpr int U = NV >= 4 ? 1 : 2;
          float least = FLT_MAX, most = 0.f;
          for (int32_t f0 = fa; f0 < fe; f0 += U * NGW) {
            V p[U][NV];
#pragma unroll
            for (int u = 0; u < U; ++u) {
              const int32_t f = min(f0 + u * NGW + gi, fe - 1);
              RO::load(p[u], M[FL], __shfl(fc[FL], f), c, Rr);
#pragma unroll
              for (int k = FL - 1; k >= 1; --k) {
                V m[NV];
                RO::load(m, M[k], __shfl(fc[k], f), c, Rr);
                RO::hmul(p[u], m);
                RO::extent(p[u], c, Rr, least, most);
              }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
              const int32_t f = f0 + u * NGW + gi;
              if (f < fe) RO::put(P + (f - fa) * KR, c, p[u]);
            }
          }
          if constexpr (N > 3) {
            odd = __ballot(!(least >= FLT_MIN && most <= FLT_MAX)) != 0;
            over = odd && __ballot(!(most <= FLT_MAX)) != 0;
          }
          wave_lds_sync();
        };
        // (cold) whether a product of the piece's rows left the normal numbers
        // where no row has a 0
        auto product_lost = [&]() {
          bool l = false;
          for (int32_t f0 = fa; f0 < fe; f0 += NGW) {
            const int32_t f = min(f0 + gi, fe - 1);
            V p[NV];
            RO::load(p, M[FL], __shfl(fc[FL], f), c, Rr);
#pragma unroll
            for (int k = FL - 1; k >= 1; --k) {
              V m[NV];
              RO::load(m, M[k], __shfl(fc[k], f), c, Rr);
              l = RO::hmul_lost(p, m) || l;
            }
          }
          return __ballot(l) != 0;
        };
        // (cold) whether a row that multiplies a product of others is above 1
        auto raised = [&]() {
          float peak = 0.f;
          for (int32_t f0 = fa; N > 4 && f0 < fe; f0 += NGW) {
            V m[NV];
            RO::load(m, M[1], __shfl(fc[1], min(f0 + gi, fe - 1)), c, Rr);
            peak = RO::peak(m, peak);
          }
          return __ballot(!(peak <= 1.f)) != 0;
        };
        // (cold) nonzeros [t, e) with P, unless a value times leaf row is above
        // kSafe: whether they are added
        auto with_p = [&](int32_t t) {
          constexpr int S = SB < 4 ? 2 : 4;
          V sum[NV];
#pragma unroll
          for (int j = 0; j < NV; ++j) sum[j] = acc[j];
          float peak = 0.f;
          for (; t < e; t += S * NGW) {
            V d[S][NV];
            int4 x[S];
#pragma unroll
            for (int u = 0; u < S; ++u) {
              x[u] = rec[min(t + u * NGW + gi, e - 1)];
              RO::load(d[u], Mleaf, x[u].x, c, Rr);
            }
#pragma unroll
            for (int u = 0; u < S; ++u) {
              V p[NV];
              RO::get(P + (x[u].z - fa) * KR, c, p);
              RO::scale(d[u], __int_as_float(x[u].y));
              peak = RO::peak(d[u], peak);
              RO::hfma_if(t + u * NGW + gi < e, sum, d[u], p);
            }
          }
          if (__ballot(!(peak <= kSafe))) return false;
#pragma unroll
          for (int j = 0; j < NV; ++j) acc[j] = sum[j];
          return true;
        };
        // (cold) nonzeros [t, te) without P: the rows multiply each value's leaf
        // row in turn
        auto rows_apart = [&](int32_t t, int32_t te) {
          for (; t < te; t += NGW) {
            const int4 x = rec[min(t + gi, te - 1)];
            V s[NV];
            RO::load(s, Mleaf, x.x, c, Rr);
            RO::scale(s, __int_as_float(x.y));
#pragma unroll
            for (int k = FL; k >= 1; --k) {
              V m[NV];
              RO::load(m, M[k], __shfl(fc[k], x.z), c, Rr);
              RO::hmul(s, m);
            }
            if (t + gi < te) RO::add(acc, s);
          }
        };
        // S steps of the row groups from nonzero t0. `whole`: none of them is past
        // the piece, as most are; the batch, whose registers already spill, has
        // no form for those (5-mode 1.5M nonzeros 30.6 us a call without the
        // form and 28.2 with it, the batch of 8 tensors 546 and 580)
        // False, with nothing done, where P may not do.
        auto steps = [&](auto S, auto whole, int32_t t0) -> bool {
          V d[S()][NV];
          auto record = [&](int u) {
            return rec[whole() ? t0 + u * NGW + gi : min(t0 + u * NGW + gi, e - 1)];
          };
#pragma unroll
          for (int u = 0; u < S(); ++u) RO::load(d[u], Mleaf, record(u).x, c, Rr);
          if constexpr (N > 2) {
            if (!staged) stage();
            staged = true;
            if (N > 3 && __builtin_expect(odd, 0)) return false;
          }
          // (the records are read again rather than held: 16 registers less)
#pragma unroll
          for (int u = 0; u < S(); ++u) {
            const int4 x = record(u);
            const float w = __int_as_float(x.y);
            // a step past the piece adds nothing (not its weight 0: the row it
            // repeats may hold infinities)
            const bool ok = whole() || t0 + u * NGW + gi < e;
            if constexpr (N > 2) {
              V p[NV];
              RO::get(P + (x.z - fa) * KR, c, p);
              RO::scale(d[u], w);
              if constexpr (whole()) RO::hfma(acc, d[u], p);
              else RO::hfma_if(ok, acc, d[u], p);
            } else {
              if constexpr (whole()) RO::axpy(acc, w, d[u]);
              else RO::axpy_if(ok, acc, w, d[u]);
            }
          }
          return true;
        };
        for (int32_t t0 = a; t0 < e;) {
          bool done;
          int32_t t1;
          if (!Batch && SB >= 4 && e - t0 >= SB * NGW) {
            done = steps(std::integral_constant<int, SB>(), std::true_type(), t0);
            t1 = t0 + SB * NGW;
          } else if (SB == 8 && e - t0 > 4 * NGW) {
            done = steps(std::integral_constant<int, SB>(), std::false_type(), t0);
            t1 = t0 + SB * NGW;
          } else if (SB >= 4 && e - t0 > 2 * NGW) {
            done = steps(std::integral_constant<int, SB < 4 ? SB : 4>(), std::false_type(), t0);
            t1 = t0 + 4 * NGW;
          } else {
            done = steps(std::integral_constant<int, 2>(), std::false_type(), t0);
            t1 = t0 + 2 * NGW;
          }
          if (N > 3 && __builtin_expect(!done, 0)) {
            t1 = e;
            if (over || raised() || !with_p(t0)) {
              if (!product_lost()) {
                odd = false;
                continue;
              }
              rows_apart(t0, e);
            }
          }
          t0 = t1;
        }
        wave_lds_sync();
        a = e;
        fa = fe;
      }
      if (!Rows && !many && qn < w1) {
        take_earlier();
#pragma unroll
        for (int j = 0; j < NV; ++j) earlier[j] = acc[j];
        RO::zero(acc);
        has_earlier = true;
      }
      q = qn;
      l = lnext;
      v = vnext;
#pragma unroll
      for (int k = 0; k < NL; ++k) {
        cur[k] = curn[k];
        wp[k] = wpn[k];
        wc[k] = wcn[k];
      }
    }
    take_earlier();
    RO::wave_sum(acc);
  }

  // The workgroup's slices: two entries per wave (its first slice, complete
  // or 0 where it is still open; the slice open at the run's end), keys in
  // ascending order. Every column sums runs of equal keys in FP64; only the
  // workgroup's first and last slice can be shared with another workgroup.
  if (gi == 0) {
    V h[NV];
    RO::zero(h);
    if (head_closed) RO::get(head_row, c, h);
    RO::put(P, c, h);
    RO::put(P + KR, c, acc);
    if (c == 0) {
      hist[0] = head;
      hist[1] = open;
    }
  }
  __syncthreads();
  auto key_of = [&](int en) {
    return reinterpret_cast<const int32_t*>(wave_mem(en >> 1) + kRecBytes)[en & 1];
  };
  auto row_of = [&](int en) {
    return reinterpret_cast<const float*>(wave_mem(en >> 1) + kRecBytes + kHistBytes) +
           (en & 1) * KR;
  };
  const int nent = 2 * int(min(int64_t(nwv), (int64_t(len) + NGW * G - 1) / (NGW * G)));
  const int32_t first = key_of(0), last = key_of(nent - 1);
  const int cols = R > 0 ? R : Rr;
  for (int col = int(threadIdx.x); col < cols; col += int(blockDim.x)) {
    const int at = RO::slot_of(col, Rr);
    double s = 0.0;
    int32_t key = first;
    auto out = [&]() {
      const int64_t o = int64_t(global_ptr(B.crd0)[key]) * cols + col;
      const bool shared = key == first || key == last;
      if constexpr (EP) {
        if (!shared) A[o] = float(s);
        else if (Rows) unsafeAtomicAdd(W + int64_t(key == first ? slot.x : slot.y) * cols + col, s);
        else unsafeAtomicAdd(A + o, float(s));
      } else {
        if (shared) unsafeAtomicAdd(W + o, s);
        else W[o] = s;
      }
    };
    for (int en = 0; en < nent; ++en) {
      const int32_t k = key_of(en);
      if (k != key) {
        out();
        s = 0.0;
        key = k;
      }
      s += double(row_of(en)[at]);
    }
    out();
  }
}

// Waves per SIMD asked of the compiler (its register budget is 512 over this):
// left alone it takes 114 registers at order 3 and 140 at order 5.
template <int N, int R>
constexpr int edge_waves() {
  return Row<R>::NV >= 4 ? 2 : Row<R>::NV == 2 ? 4 : N <= 3 ? 5 : 4;
}

template <int N, int R, bool EP, bool Rows>
__global__ __launch_bounds__(512, (edge_waves<N, R>())) void edge_kernel(CsfDev B, FactorsDev F,
                                                   float* __restrict__ A, int Rr,
                                                   const int32_t* __restrict__ brk,
                                                   const int32_t* __restrict__ starts,
                                                   int32_t G, int32_t NB,
                                                   double* __restrict__ W,
                                                   const int2* __restrict__ slots) {
  extern __shared__ __align__(16) unsigned char smem[];
  edge_block<N, R, EP, Rows>(B, F, A, Rr, brk, starts, blockIdx.x, G, NB, smem, W,
                             Rows ? slots + blockIdx.x : nullptr);
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
      for (int u = 0; u < U; ++u)
        RO::axpy_if(q0 + u < e, out, v[u], d[u]);
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
  constexpr int TB = NV >= 4 ? 2 : NT < 8 ? NT : 8;  // fibers whose rows are in flight per batch
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
  // (unsigned: a base past the slice may pass 2^31 - 1)
  for (uint32_t base = uint32_t(q0) + 64 * wv; base < uint32_t(q1); base += 64 * nwv) {
    const uint32_t q = base + lane;
    const bool okq = q < uint32_t(q1);
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
      RO::hfma_if(base + u * NG + gi < uint32_t(q1), acc, w, cr[u]);
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
      for (int t = 0; t < NT; ++t)
        RO::axpy_if(base + t * NG + gi < e, acc, vt[t], d[t]);
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

// Slice-row kernel for 3-mode tensors of short fibres and short slices, over
// the expansion: a wave takes the consecutive slices that start among its WN
// nonzeros (whole, the empty ones too), PB nonzeros at a time. Their products
// val * C(k,:) (.) D(l,:) go to LDS with all rows in flight, and the row
// groups then sum a slice each and store its row; a slice that runs past the
// batch is carried to the next. A row group's serial sum is in FP64: in FP32 it
// had 12 to 17% more error than slices summed over the wave. No atomics, no zero
// fill on a dense root, deterministic. A workgroup per slice (slice_short_kernel) leaves most of its
// lanes idle below some 12 nonzeros a slice: 40000 slices of 7.5, rank 32:
// 50 us a call with 256 threads a slice, 32 with 128, 13 here.
template <int R>
constexpr int group_batch() {
  constexpr int p = 4096 / (Lay<R>::kMaxRank * 4);
  return p > 64 ? 64 : Lay<R>::kMaxRank == 128 ? 16 : Lay<R>::kMaxRank == 256 ? 8 : p;
}

template <int R>
__global__ __launch_bounds__(256) void slice_group_kernel(CsfDev B, FactorsDev F,
                                                          float* __restrict__ A, int Rr,
                                                          int32_t WN) {
  using RO = Row<R>;
  using V = typename RO::V;
  constexpr int NV = RO::NV;
  constexpr int LPR = RO::LPR;
  constexpr int KR = Lay<R>::kMaxRank;
  constexpr int NGW = 64 / LPR;
  constexpr int PB = group_batch<R>();
  constexpr int U = PB / NGW;
  static_assert(U >= 1 && PB % NGW == 0, "whole steps");
  __shared__ __align__(16) float lds[4][PB * KR];
  const int lane = int(threadIdx.x) & 63;
  const int wv = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int gi = lane / LPR;
  const int c = lane % LPR;
  float* P = lds[wv];
  const int32_t* __restrict__ nzr = B.nnz_of_root;
  const int32_t* __restrict__ kq = B.crd1_of_nnz;
  const int32_t* __restrict__ lq = B.crd[2];
  const float* __restrict__ vq = B.vals;
  const int32_t n0 = B.nodes[0];
  const int32_t nnz = B.nnz;
  const int64_t w = int64_t(blockIdx.x) * 4 + wv;
  if (w * WN >= nnz) return;
  // slices [x0, x1): those whose first nonzero is in [w*WN, (w+1)*WN); the
  // first wave takes the leading empty ones, the last the trailing ones
  const int64_t hi = (w + 1) * WN;
  const int32_t x0 = w == 0 ? 0 : wave_search_le(nzr, 0, n0 - 1, int32_t(w * WN) - 1, lane) + 1;
  const int32_t x1 =
      hi >= nnz ? n0 : wave_search_le(nzr, max(x0 - 1, 0), n0 - 1, int32_t(hi) - 1, lane) + 1;
  double carry[NV * RO::NC] = {};
  bool carried = false;
  for (uint32_t xb = x0; xb < uint32_t(x1); xb += 64) {
    // a window of slices, one per lane
    const int32_t nx = min(64, x1 - int32_t(xb));
    const int32_t x = index_ahead(int32_t(xb), lane, x1 - 1);
    const int32_t st = nzr[x];
    const int32_t en = nzr[x + 1];
    const int32_t row = B.crd0[x];
    for (int32_t rb = 0; rb < nx; rb += NGW) {
      const int32_t r = min(rb + gi, nx - 1);
      const int32_t len = __shfl(en - st, r);
      const int32_t rr = __shfl(row, r);
      if (rb + gi < nx && len == 0) {
        V z[NV];
        RO::zero(z);
        RO::store(A, rr, c, Rr, z);
      }
    }
    const int32_t q0 = __builtin_amdgcn_readlane(st, 0);
    const int32_t q1 = __builtin_amdgcn_readlane(en, nx - 1);
    for (int32_t s0 = q0, m = 0; s0 < q1; s0 += m) {
      m = min(PB, q1 - s0);
      V cr[U][NV], dr[U][NV];
      float vt[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int32_t q = s0 + min(u * NGW + gi, m - 1);
        vt[u] = vq[q];
        RO::load(cr[u], F.M[1], kq[q], c, Rr);
        RO::load(dr[u], F.M[2], lq[q], c, Rr);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        V p[NV];
        RO::zero(p);
        RO::axpy(p, vt[u], dr[u]);
        RO::hmul(p, cr[u]);
        if (u * NGW + gi < m) RO::put(P + (u * NGW + gi) * KR, c, p);
      }
      wave_lds_sync();
      const int32_t s1 = s0 + m;
      // slices that reach into the batch
      const int32_t r0 = __popcll(__ballot(lane < nx && en <= s0));
      const int32_t r1 = __popcll(__ballot(lane < nx && st < s1)) - 1;
      double last[NV * RO::NC] = {};
      for (int32_t rb = r0; rb <= r1; rb += NGW) {
        const int32_t r = min(rb + gi, r1);
        const int32_t a = max(__shfl(st, r), s0);
        const int32_t b = __shfl(en, r);
        const int32_t rr = __shfl(row, r);
        if (rb + gi > r1) continue;
        double sum[NV * RO::NC] = {};
        if (r == r0 && carried) {
#pragma unroll
          for (int k = 0; k < NV * RO::NC; ++k) sum[k] = carry[k];
        }
        for (int32_t i = a; i < min(b, s1); ++i) {
          V p[NV];
          RO::get(P + (i - s0) * KR, c, p);
          RO::add(sum, p);
        }
        if (b > s1) {
#pragma unroll
          for (int k = 0; k < NV * RO::NC; ++k) last[k] = sum[k];
        } else if (a < b) {
          V row[NV];
          RO::narrow(row, sum);
          RO::store(A, rr, c, Rr, row);
        }
      }
      carried = __builtin_amdgcn_readlane(en, r1) > s1;
      if (carried) {
        // to every row group, since the next batch's first one takes it
        const int from = (r1 - r0) % NGW * LPR + c;
#pragma unroll
        for (int k = 0; k < NV * RO::NC; ++k) carry[k] = __shfl(last[k], from);
      }
      wave_lds_sync();
    }
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
      // (the other slice adds nothing rather than 0 times the rows, which may
      // hold infinities; an empty slot's are zeros)
      V w[NV];
      RO::zero(w);
      RO::axpy(w, vt[u], dr[u]);
      const bool first = h * 128 + wv * 64 + u * NG + gi < inf.z;
      RO::hfma_if(first, aa, w, cr[u]);
      RO::hfma_if(!first, ab, w, cr[u]);
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


// Persistent workgroups over the items [i_lo, i_hi) of tasks [t_lo, t_hi):
// item(T, b) runs item b of task T. Items go out in chunks of `chunk`
// consecutive ones: a workgroup's first chunk is its own index; later ones
// come from the device counter (schedule 0, zero between runs; not
// touched when the first chunks cover every item) or by a static cyclic
// assignment (schedule 1). Either way a workgroup's items increase, so its
// task cursor only moves forward.
template <class F>
__device__ __forceinline__ void batch_items(const BatchTaskDev* __restrict__ tasks, int32_t t_lo,
                                            int32_t t_hi, const int64_t* __restrict__ item_off,
                                            int32_t i_lo, int32_t i_hi,
                                            int32_t* __restrict__ counter, int32_t chunk,
                                            int dynamic, F&& run) {
  __shared__ int32_t s_chunk;
  const int32_t nchunks = (i_hi - i_lo + chunk - 1) / chunk;
  const int32_t grid = int32_t(gridDim.x);
  int32_t t = -1;
  int64_t t_end = 0;
  for (int32_t ch = int32_t(blockIdx.x); ch < nchunks;) {
    const int32_t first = i_lo + ch * chunk;
    const int32_t last = min(i_hi - first, chunk) + first;
    for (int32_t item = first; item < last; ++item) {
      __syncthreads();  // the previous item's LDS reads are done
      if (t < 0) {
        t = t_lo + upper_index(item_off + t_lo, t_hi - t_lo, item);
        t_end = item_off[t + 1];
      }
      while (item >= t_end) {
        ++t;
        t_end = item_off[t + 1];
      }
      run(tasks[t], item - int32_t(item_off[t]));
    }
    if (dynamic) {
      if (nchunks <= grid) break;
      __syncthreads();  // every thread has read the previous s_chunk
      if (threadIdx.x == 0) s_chunk = grid + atomicAdd(counter, 1);
      __syncthreads();
      ch = __builtin_amdgcn_readfirstlane(s_chunk);
    } else {
      ch += grid;
    }
  }
}

// An add to the one counter takes 10-12 ns whatever the workgroups do, so
// items taken one at a time cost that each (8 tensors, 38k items of 512
// nonzeros: 815 us a replay, 676 us in chunks and with the starts kept). About
// eight chunks per workgroup keep the ends even.
inline int32_t batch_chunk(int32_t items, int grid, int schedule) {
  return schedule == 0 ? std::max(1, items / (8 * grid)) : 1;
}

// One order's tasks (the device task table is sorted by order: tasks [t_lo,
// t_hi) hold items [i_lo, i_hi)), with the order's own register footprint:
// batches of one order, and those whose orders differ in block or schedule.
// The batch has FP64 rows for the slices that items share only, not for all
// that the edge-serial walk adds to, so it runs the edge-parallel walk only.
template <int N, int R>
__global__ __launch_bounds__(512, (edge_waves<N, R>())) void batch_kernel(
    const BatchTaskDev* __restrict__ tasks, int32_t t_lo, int32_t t_hi,
    const int64_t* __restrict__ item_off, int32_t i_lo, int32_t i_hi, int32_t* __restrict__ counter,
    int Rr, int32_t G, int32_t NB, int32_t chunk, int dynamic) {
  extern __shared__ __align__(16) unsigned char smem[];
  batch_items(tasks, t_lo, t_hi, item_off, i_lo, i_hi, counter, chunk, dynamic,
              [&](const BatchTaskDev& T, int32_t b) {
                edge_block<N, R, true, true, true>(T.B, T.F, T.A, Rr, nullptr, T.starts, b, G, NB, smem, T.W,
                                       T.slots + b);
              });
}

template <int N, int R>
int launch_batch_order(const BatchLaunch& L, hipStream_t st) {
  const int32_t i_lo = L.grp_item[N], i_hi = L.grp_item[N + 1];
  if (i_hi <= i_lo) return TENTACO_OK;
  const int blk = L.blk[N];
  const size_t lds = size_t(blk / 64) * edge_wave_lds<R, true>();
  const int grid = std::max(1, std::min<int>(L.grp_grid[N], i_hi - i_lo));
  const int32_t chunk = batch_chunk(i_hi - i_lo, grid, L.sch[N]);
  batch_kernel<N, R><<<grid, blk, lds, st>>>(
      L.tasks, L.grp_task[N], L.grp_task[N + 1], L.item_off, i_lo, i_hi, L.counter + N, L.R,
      L.grp[N], L.nb[N], chunk, L.sch[N] == 0);
  TT_HIP_CHECK(hipGetLastError());
  return TENTACO_OK;
}

template <int N, int R>
int batch_occupancy_order(int family, int block, int Rr, int32_t NB, int* per_cu) {
  if (family != kEdgeParallel)
    return fail(TENTACO_EUNSUPPORTED, "the batch runs the edge-parallel walk only");
  const size_t lds = size_t(block / 64) * edge_wave_lds<R, true>();
  const hipError_t e =
      hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, batch_kernel<N, R>, block, lds);
  if (e != hipSuccess) return fail(TENTACO_EHIP, "occupancy query: %s", hipGetErrorString(e));
  return TENTACO_OK;
}

template <int N, int R>
int launch_typed(const CsfDev& B, const FactorsDev& F, int Rr, float* A,
                 int32_t a_rows, bool dense_root, const Variant& vr, void* ws,
                 const WalkTables& wt, hipStream_t st) {
  const int64_t a_elems = int64_t(a_rows) * Rr;
  if (vr.family == kSliceRow) {
    if (!dense_root) {
      const int rc = launch_fill(A, a_elems, 0.f, st);
      if (rc) return rc;
    }
    if (B.nodes[0] > 0) {
      ktimer_begin(st);
      // short fibres (nnz <= 1.25 x fibres) with the expansion built: the
      // kernels that skip the pos -> crd chain
      const bool expanded =
          N == 3 && B.crd1_of_nnz && int64_t(B.nnz) * 4 <= int64_t(B.nodes[1]) * 5 && B.nnz > 0;
      if constexpr (N == 3) {
        if (expanded && vr.group > 0) {
          const int64_t waves = (int64_t(B.nnz) + vr.group - 1) / vr.group;
          slice_group_kernel<R><<<int((waves + 3) / 4), 256, 0, st>>>(B, F, A, Rr, vr.group);
          TT_HIP_CHECK(hipGetLastError());
          ktimer_end(st, "slice_group_kernel");
          return TENTACO_OK;
        }
      }
      if constexpr (N == 3 && (R > 0 || Row<R>::NV == 1)) {
        if (expanded) {
          if constexpr (R == 16 || R == 32 || R == 64) {
            if (B.pair && vr.block >= 256) {
              slice_pair_kernel<R><<<B.npairs, 128, 0, st>>>(B.pair, B.pair_info, F, A, Rr);
              TT_HIP_CHECK(hipGetLastError());
              ktimer_end(st, "slice_pair_kernel");
              return TENTACO_OK;
            }
          }
          if constexpr (R > 0) {
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
  const int32_t* starts = wt.starts;
  const bool shared = vr.family == kEdgeParallel && starts && wt.slots && nblk > 0;
  // edge-serial: rows accumulate in FP64 (W, after the brackets), narrowed
  // to A at the end; the prep zeroes W instead of A
  double* W = (vr.family == kEdgeSerial && nblk > 0)
                  ? reinterpret_cast<double*>(static_cast<char*>(ws) + edge_brk_bytes(B, NB))
                  : nullptr;
  if (!shared) {
    float* Z = W ? reinterpret_cast<float*>(W) : A;
    const int64_t z_elems = W ? 2 * a_elems : a_elems;
    const int rc = starts ? launch_fill(Z, z_elems, 0.f, st)
                          : launch_edge_prep(B, Z, z_elems, brk, int32_t(nblk), int32_t(NB), st);
    if (rc) return rc;
  }
  if (nblk == 0) return TENTACO_OK;
  // the variant table's tile limit (tentaco_variant_fits)
  if (!edge_tile_fits(N, Rr, vr)) {
    return fail(TENTACO_EUNSUPPORTED, "edge tile of block %d and group %d at rank %d is over the "
                "tile limit of order %d", vr.block, vr.group, Rr, N);
  }
  const size_t lds =
      size_t(vr.block / 64) * (shared ? edge_wave_lds<R, true>() : edge_wave_lds<R, false>());
  const int32_t nb = int32_t(NB), grid = int32_t(nblk);
  ktimer_begin(st);
  if (shared)
    edge_kernel<N, R, true, true><<<grid, vr.block, lds, st>>>(B, F, A, Rr, brk, starts, vr.group, nb,
                                                               wt.W, wt.slots);
  else if (vr.family == kEdgeParallel)
    edge_kernel<N, R, true, false><<<grid, vr.block, lds, st>>>(B, F, A, Rr, brk, starts, vr.group, nb,
                                                                nullptr, nullptr);
  else
    edge_kernel<N, R, false, false><<<grid, vr.block, lds, st>>>(B, F, A, Rr, brk, starts, vr.group, nb,
                                                                 W, nullptr);
  TT_HIP_CHECK(hipGetLastError());
  ktimer_end(st, "edge_kernel");
  if (shared) return launch_edge_rows(wt, int32_t(nblk), A, a_rows, Rr, st);
  return W ? launch_narrow(W, A, a_elems, st) : TENTACO_OK;
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

// Writes nothing; holds as much scratch as the walk's kernels spill at most, which
// the runtime allocates for a queue on its first use (1.8 ms).
__global__ __launch_bounds__(512) void order_warm_kernel(int n) {
  volatile int32_t spill[40];
  for (int i = 0; i < n; ++i) spill[(i * 7 + int(threadIdx.x)) % 40] = i;
}

}  // namespace

// ---- one tensor order's entry points (mttkrp_dispatch.h) --------------------
template <int N>
int order_warm(hipStream_t st) {
  order_warm_kernel<<<2048, 512, 0, st>>>(0);
  TT_HIP_CHECK(hipGetLastError());
  return TENTACO_OK;
}

template <int N>
int order_mttkrp(const CsfDev& B, const FactorsDev& F, int R, float* A, int32_t a_rows,
                 bool dense_root, const Variant& vr, void* ws, const WalkTables& wt,
                 hipStream_t st) {
  return with_rank_layout(R, [&](auto r) {
    return launch_typed<N, r()>(B, F, R, A, a_rows, dense_root, vr, ws, wt, st);
  });
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
  template int tt::order_warm<N>(hipStream_t);                                                  \
  template int tt::order_mttkrp<N>(const CsfDev&, const FactorsDev&, int, float*, int32_t, bool, \
                                   const Variant&, void*, const WalkTables&, hipStream_t);         \
  template int tt::order_level<N>(const CsfDev&, const FactorsDev&, int, int, float*, int32_t,  \
                                  hipStream_t);                                                 \
  template int tt::order_batch<N>(const BatchLaunch&, hipStream_t);                             \
  template int tt::order_batch_occupancy<N>(int, int, int, int32_t, int*);
