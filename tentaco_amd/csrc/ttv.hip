// CSF TTV for gfx950: y(f) = sum_k B(f,k) * c(k) over the level N-2 positions
// f of B (the (i,j) fibers of a 3-mode tensor), i.e. a CSR SpMV whose rows
// are the innermost fibers. Replaces ttv_kernel / ttv_csf_gpu_taco
// (tensor_kernels/ttv_csf_gpu_taco.h:2-121).
//
// Two kernels. The unit kernel (below, ttv_unit_kernel) is the main path: it
// reads a per-handle fibre-start bitmap instead of searching pos and writes
// every y entry exactly once (no zero fill, no atomics). It has two forms: up to
// a million nonzeros without long or empty fibres a wave sums whole fibres;
// otherwise a wave walks a range of units, with a window of c in LDS, and with
// empty fibres the plan indexes the non-empty ones and maps them to output
// positions. The bracket kernel (ttv_kernel) covers calls
// captured before a handle's plan exists and c beyond 2^30 entries:
//
// Work split: each workgroup owns 8*BS consecutive nonzeros, each lane 8
// consecutive ones (two dwordx4 loads of crd and of vals per lane, fully
// coalesced per wavefront). The nonzero loads and the c gathers are issued
// first, so their latency overlaps the bracket load and the staging of the
// workgroup's fiber bounds in LDS. A lane sums its nonzeros per fiber; fibers that
// start and end inside a lane are stored directly, the lane's first and last
// partial sums are merged across the wavefront by a segmented shuffle scan
// keyed by fiber id, and the lane holding a fiber's last nonzero writes the
// total. Only the wavefront's first fiber (when it began in an earlier
// wavefront) and its open last fiber are added atomically into the
// zero-filled output. A prep launch zero-fills y and scatters, per fiber, the
// workgroup boundaries that fall inside it (no binary-search pre-pass).

#include <algorithm>
#include <climits>
#include <cstring>
#include <type_traits>
#include <vector>

#include <rocprim/device/device_scan.hpp>

#include "internal.h"
#include "rowops.h"

namespace tt {
namespace {

constexpr int kTtvBlock = 256;
constexpr int kTtvPerLane = 8;
constexpr int kTtvNB = kTtvBlock * kTtvPerLane;

// y[0..nf) = 0; brk[b] = fiber containing min(b*NB, nnz-1), b in 0..nblk.
__global__ __launch_bounds__(256) void ttv_prep_kernel(
    const int32_t* __restrict__ pos, float* __restrict__ y, int32_t nf,
    int32_t nnz, int32_t* __restrict__ brk, int32_t nblk) {
  const int64_t tid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t f = tid; f < nf; f += nthr) {
    y[f] = 0.f;
    const int32_t s = pos[f];
    const int32_t e = pos[f + 1];
    if (s >= e) continue;
    for (int64_t b = (int64_t(s) + kTtvNB - 1) / kTtvNB; b * kTtvNB < e; ++b)
      brk[b] = int32_t(f);
    if (s <= nnz - 1 && nnz - 1 < e) brk[nblk] = int32_t(f);
  }
}

__global__ __launch_bounds__(kTtvBlock) void ttv_kernel(
    const int32_t* __restrict__ pos, const int32_t* __restrict__ crd,
    const float* __restrict__ vals, const float* __restrict__ cv,
    float* __restrict__ y, int32_t nnz, const int32_t* __restrict__ brk) {
  constexpr int U = kTtvPerLane;
  // fiber bounds pos[lo..hi+1] of the workgroup, staged once; a CSF built
  // from coordinates has at most NB+1 non-empty fibers starting in a
  // workgroup, larger brackets (runs of empty fibers) read pos directly
  __shared__ int32_t s_pos[kTtvNB + 2];
  const int32_t b = blockIdx.x;
  const int32_t P = b * kTtvNB;
  const int32_t Pend = min(P + kTtvNB, nnz);
  const int lane = threadIdx.x & 63;
  const int32_t p0 = P + int32_t(threadIdx.x) * U;
  const int32_t p1 = min(p0 + U, Pend);
  const bool active = p0 < p1;
  // nonzeros and c gathers first: independent of the fiber bounds
  int32_t k[U];
  float v[U];
  float cg[U];
  if (active) {
    if (p0 + U <= nnz) {
#pragma unroll
      for (int h = 0; h < U; h += 4) {
        const int4 kk = *reinterpret_cast<const int4*>(crd + p0 + h);
        const float4 vv = *reinterpret_cast<const float4*>(vals + p0 + h);
        k[h] = kk.x; k[h + 1] = kk.y; k[h + 2] = kk.z; k[h + 3] = kk.w;
        v[h] = vv.x; v[h + 1] = vv.y; v[h + 2] = vv.z; v[h + 3] = vv.w;
      }
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool ok = p0 + u < nnz;
        k[u] = ok ? crd[p0 + u] : 0;
        v[u] = ok ? vals[p0 + u] : 0.f;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) cg[u] = cv[k[u]];
  }
  const int32_t lo = brk[b];
  const int32_t hi = brk[b + 1];
  const int32_t nstage = hi - lo + 2;
  const bool staged = nstage <= kTtvNB + 2;
  if (staged)
    for (int32_t j = threadIdx.x; j < nstage; j += kTtvBlock) s_pos[j] = pos[lo + j];
  __syncthreads();
  auto P_at = [&](int32_t x) -> int32_t { return staged ? s_pos[x - lo] : pos[x]; };
  auto search = [&](int32_t a, int32_t z, int32_t key) {
    while (a < z) {
      const int32_t mid = a + ((z - a + 1) >> 1);
      if (P_at(mid) <= key) a = mid;
      else z = mid - 1;
    }
    return a;
  };

  int32_t f = INT_MAX, nxt = 0, first = INT_MAX;
  float sum = 0.f, vf = 0.f;
  bool closed_first = false, ends_here = false, starts_before = false;
  if (active) {
    f = search(lo, hi, p0);
    nxt = P_at(f + 1);
    first = f;
    starts_before = P_at(f) < p0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int32_t p = p0 + u;
      if (p >= p1) break;
      if (p >= nxt) {
        if (!closed_first) {
          vf = sum;
          closed_first = true;
        } else {
          y[f] = sum;  // started and ended inside this lane
        }
        sum = 0.f;
        int32_t x = f + 1;
        int32_t e = P_at(x + 1);
        if (e <= p) {
          x = search(x + 1, hi, p);
          e = P_at(x + 1);
        }
        f = x;
        nxt = e;
      }
      sum = fmaf(v[u], cg[u], sum);
    }
    ends_here = (nxt == p1);
  }
  // inclusive segmented scan of the lanes' open (last) segments
  const int32_t tkey = f;
  float incl = active ? sum : 0.f;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const float ov = __shfl_up(incl, d);
    const int32_t ok = __shfl_up(tkey, d);
    if (lane >= d && ok == tkey) incl += ov;
  }
  const float pv = __shfl_up(incl, 1);
  const int32_t pk = __shfl_up(tkey, 1);
  const int32_t wfirst = __shfl(first, 0);
  const bool wbefore = __shfl(int(starts_before), 0) != 0;
  if (!active) return;
  const float carry = (lane > 0 && pk == first) ? pv : 0.f;
  const bool is_last = (lane == 63) || (p0 + U >= Pend);
  auto emit = [&](int32_t key, float val, bool shared) {
    if (shared || (key == wfirst && wbefore)) unsafeAtomicAdd(y + key, val);
    else y[key] = val;
  };
  if (closed_first) emit(first, vf + carry, false);
  if (ends_here) emit(f, incl, false);
  else if (is_last) emit(f, incl, true);
}

// ---- unit kernel ---------------------------------------------------------
// Each wave owns a contiguous range of 512-nonzero units and walks it in
// order, 8 nonzeros per lane per unit. The fibre of a lane's first nonzero is
// the unit's first fibre plus the fibre starts before it in the unit: an
// exclusive prefix count of the lanes' start bits (per-lane popcounts 0..8,
// summed over lanes as 4 bit-plane ballots). A lane closes the fibres that
// start and end inside it with a plain store; fibres spanning lanes are
// summed by a segmented scan keyed by fibre id, and the fibre still open at
// the end of a unit is carried in registers into the next. Fibres crossing
// the wave's range bounds leave their pieces in a per-wave table (head:
// the fibre that began before the range; tail: the one open at its end),
// which a second small launch folds into y. The c entries inside the
// plan's window are read from LDS, the rest from global memory.
constexpr int kUnit = 512;
constexpr int kUnitWaves = 16;
constexpr int kUnitThreads = 64 * kUnitWaves;
constexpr uint32_t kOutOfRange = 0xFFFFFFF0u;  // buffer offset past any c (c < 2^30 - 8 entries)
constexpr int32_t kUnitMaxC = (1 << 30) - 8;
// outputs the unit kernels write through a buffer descriptor: byte offsets
// and the descriptor's size in bytes stay below 2^31
constexpr int32_t kUnitMaxY = 1 << 29;
// units of a wave's range loaded ahead of the one being summed in the banded
// layout (its gathers are LDS reads, so the loads ahead are waited for only
// when their unit is summed)
constexpr int kBandPF = 2;

__global__ __launch_bounds__(256) void ttv_plan_kernel(
    const int32_t* __restrict__ pos, int32_t nf, uint32_t* __restrict__ flags,
    int32_t* __restrict__ unit_fid, uint32_t* __restrict__ bad) {
  const int64_t tid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t f = tid; f < nf; f += nthr) {
    const int32_t s = pos[f];
    const int32_t e = pos[f + 1];
    if (s >= e) {
      atomicOr(bad, 1u);
      continue;
    }
    atomicOr(flags + (s >> 5), 1u << (s & 31));
    for (int64_t u = (int64_t(s) + kUnit - 1) / kUnit; u * kUnit < e; ++u)
      unit_fid[u] = int32_t(f);
  }
}

// histogram of every `step`-th leaf coordinate in bins of 2^shift (picks the
// c window; a sample of about 2^20 nonzeros is enough for that)
__global__ __launch_bounds__(256) void ttv_hist_kernel(
    const int32_t* __restrict__ crd, int32_t nnz, int32_t step, int shift,
    uint32_t* __restrict__ hist) {
  const int64_t tid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t p = tid * step; p < nnz; p += nthr * step) atomicAdd(hist + (crd[p] >> shift), 1u);
}

// Lane moves through DPP (a VALU operand modifier: no LDS traffic). CTRL is
// the DPP control (0x111 + s - 1: row shift right by s within rows of 16;
// 0x142 / 0x143: lane 15 / 31 broadcast to the following rows; 0x130 /
// 0x138: whole-wave shift left / right by one); lanes without a source, or
// in rows outside ROWS, get `old`.
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ int32_t dpp_i(int32_t old, int32_t v) {
  return __builtin_amdgcn_update_dpp(old, v, CTRL, ROWS, 0xF, false);
}
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ float dpp_f(float old, float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v), CTRL,
                                                    ROWS, 0xF, false));
}
// one step of a segmented inclusive scan: v += the source lane's v when the
// source has the same key (keys never decrease with the lane, so equal keys
// are one contiguous run and the step adds only that run's lanes)
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ void seg_scan_step(float& v, int32_t key) {
  const float ov = dpp_f<CTRL, ROWS>(0.f, v);
  const int32_t ok = dpp_i<CTRL, ROWS>(INT_MIN, key);
  v = ok == key ? v + ov : v;
}
// inclusive scan over the wave of v among the lanes with the same key: row
// shifts 1, 2, 4, 8 within rows of 16, then lane 15's sum into rows 1 and 3,
// then lane 31's into rows 2 and 3
__device__ __forceinline__ float seg_scan(float v, int32_t key) {
  seg_scan_step<0x111>(v, key);
  seg_scan_step<0x112>(v, key);
  seg_scan_step<0x114>(v, key);
  seg_scan_step<0x118>(v, key);
  seg_scan_step<0x142, 0xA>(v, key);
  seg_scan_step<0x143, 0xC>(v, key);
  return v;
}

// exclusive prefix sum over the wave of cnt in 0..15
__device__ inline int32_t wave_excl_count(uint32_t cnt) {
  int32_t r = 0;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const uint64_t m = __ballot((cnt >> b) & 1u);
    r += int32_t(__builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32),
                                           __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u)))
         << b;
  }
  return r;
}

// c through a buffer descriptor: lanes served from LDS pass an offset past
// the end, which returns 0 without a memory access, so the LDS and global
// gathers of a lane need no branch between them
__device__ __forceinline__ __amdgpu_buffer_rsrc_t c_rsrc(const float* cv, int32_t cdim) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(cv), int16_t(0),
                                           int32_t(uint32_t(cdim) * 4u), 0x00020000);
}

// s_c[0 .. lc) = c[k0 .. k0 + lc) for lc <= LC (s_c[lc .. LC) = 0): every
// load of a thread is issued before any is stored, so the window costs one
// round trip to memory
template <int LC>
__device__ __forceinline__ void stage_window(float* s_c, __amdgpu_buffer_rsrc_t crs, int32_t k0,
                                             int32_t lc) {
  static_assert(LC % kUnitThreads == 0, "the window is whole rows of the workgroup");
  constexpr int kPer = LC / kUnitThreads;
  float t[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int32_t i = j * kUnitThreads + int32_t(threadIdx.x);
    t[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
        crs, i < lc ? uint32_t(k0 + i) * 4u : kOutOfRange, 0, 0));
  }
#pragma unroll
  for (int j = 0; j < kPer; ++j) s_c[j * kUnitThreads + int32_t(threadIdx.x)] = t[j];
}

// One wave's units [ub, ue): fibre sums into y[0 .. ny) (through ne_fid
// when given), the pieces of fibres crossing the range bounds into
// crossing-table slots 2w (head) and 2w + 1 (tail).
// WIN16 (the banded layouts): crd holds 16-bit indexes into the window s_c,
// padding the index of a slot that holds 0, so every gather is one LDS read
// and the index stream is half the size of the coordinates'. Otherwise crd
// holds 32-bit leaf coordinates: those in [k0, k0 + lc) are read from s_c,
// the others through crs.
// The units' streams are loaded PF units ahead of the one being summed, into
// PF + 1 register sets used in rotation (the loop is unrolled over the
// rotation, so no set is copied while its loads are in flight). Every store
// is issued whether or not its lanes write (a buffer store to an offset past
// the end writes nothing), so the compiler's count of memory operations in
// flight is exact and a wait for a unit's loads never waits for the later
// units'. stage() is called by every thread once the first PF units' loads
// are issued: it fills s_c and ends with the workgroup barrier, so the window
// and the first units arrive in one round trip. close_tail() (evaluated after
// the last unit) says whether the range ends where a fibre starts or the
// data end. With WHOLE_UNITS nnz is a multiple of the unit (padded layouts).
template <bool WIN16, bool WHOLE_UNITS, int PF, typename CloseTail, typename Stage>
__device__ __forceinline__ void ttv_units_wave(
    const std::conditional_t<WIN16, uint16_t, int32_t>* __restrict__ crd,
    const float* __restrict__ vals,
    const uint32_t* __restrict__ flags, const int32_t* __restrict__ unit_fid,
    __amdgpu_buffer_rsrc_t crs, const float* s_c, int32_t k0, int32_t lc,
    float* __restrict__ y, int32_t ny, int32_t nnz, int32_t ub, int32_t ue, int32_t w,
    int32_t* __restrict__ bnd_fid, float* __restrict__ bnd_val,
    const int32_t* __restrict__ ne_fid, CloseTail&& close_tail, Stage&& stage) {
  constexpr int NB = PF + 1;
  // The loaded words are used only when their unit is summed: any use
  // sooner (even a shift of the start-bit word) would wait for the load.
  struct UnitRegs {
    int32_t k[WIN16 ? 4 : 8];  // WIN16: two 16-bit indexes a word
    float v[8];
    uint32_t fw;   // the start-bit word holding this lane's 8 positions
    int32_t ufid;  // the unit's first fibre
  };
  const int lane = threadIdx.x & 63;
  int32_t cfid = -1;  // fibre open at the end of the previous unit
  float cval = 0.f;   // its sum so far
  int32_t hfid = -1;  // fibre that began before this range (its pieces go to the table)
  float hval = 0.f;
  bool hset = false;  // (per lane) this lane closed hfid
  const __amdgpu_buffer_rsrc_t yrs = __builtin_amdgcn_make_buffer_rsrc(
      y, int16_t(0), int32_t(uint32_t(ny) * 4u), 0x00020000);
  // y of fibre f when cond (the instruction is issued either way)
  auto put = [&](int32_t f, float val, bool cond) {
    if (ne_fid) {
      if (cond) y[ne_fid[f]] = val;
    } else {
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(val), yrs,
                                            cond ? int32_t(uint32_t(f) * 4u) : int32_t(kOutOfRange),
                                            0, 0);
    }
  };
  // a closed fibre's sum when cond: the table's head entry for hfid
  auto emit = [&](bool cond, int32_t fid, float val) {
    const bool h = cond && fid == hfid;
    hval = h ? val : hval;
    hset = hset || h;
    put(fid, val, cond && !h);
  };
  // a unit's coordinates, values, start bits and first fibre
  auto fetch = [&](int32_t u, UnitRegs& r) {
    const int32_t p0 = u * kUnit + lane * 8;
    if constexpr (WIN16) {
      static_assert(WHOLE_UNITS, "16-bit indexes come in whole units");
      const int4 kk = *reinterpret_cast<const int4*>(crd + p0);
      r.k[0] = kk.x; r.k[1] = kk.y; r.k[2] = kk.z; r.k[3] = kk.w;
#pragma unroll
      for (int h = 0; h < 8; h += 4) {
        const float4 vv = *reinterpret_cast<const float4*>(vals + p0 + h);
        r.v[h] = vv.x; r.v[h + 1] = vv.y; r.v[h + 2] = vv.z; r.v[h + 3] = vv.w;
      }
    } else if (WHOLE_UNITS || p0 + 8 <= nnz) {
#pragma unroll
      for (int h = 0; h < 8; h += 4) {
        const int4 kk = *reinterpret_cast<const int4*>(crd + p0 + h);
        const float4 vv = *reinterpret_cast<const float4*>(vals + p0 + h);
        r.k[h] = kk.x; r.k[h + 1] = kk.y; r.k[h + 2] = kk.z; r.k[h + 3] = kk.w;
        r.v[h] = vv.x; r.v[h + 1] = vv.y; r.v[h + 2] = vv.z; r.v[h + 3] = vv.w;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const bool ok = p0 + j < nnz;
        r.k[j] = ok ? crd[p0 + j] : -1;  // gathers 0 (out-of-range offset)
        r.v[j] = ok ? vals[p0 + j] : 0.f;
      }
    }
    r.fw = flags[min(p0, nnz - 1) >> 5];
    r.ufid = unit_fid[u];
  };
  // this lane's start bits of unit u (none past the end of the data)
  auto bits = [&](int32_t u, const UnitRegs& r) -> uint32_t {
    const int32_t p0 = u * kUnit + lane * 8;
    return WHOLE_UNITS || p0 < nnz ? (r.fw >> (p0 & 31)) & 0xFFu : 0u;
  };
  // sums of unit u
  auto work = [&](int32_t u, const UnitRegs& r) {
    const int32_t P = u * kUnit;
    const int32_t p0 = P + lane * 8;
    const bool active = p0 < nnz;
    const uint32_t fb = bits(u, r);
    const int32_t ufid = r.ufid;
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if constexpr (WIN16) {
        x[j] = r.v[j] * s_c[(uint32_t(r.k[j >> 1]) >> (16 * (j & 1))) & 0xFFFFu];
      } else {
        const int32_t kk = r.k[j] - k0;
        const bool win = r.k[j] >= 0 && uint32_t(kk) < uint32_t(lc);
        const float g = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
            crs, (win || r.k[j] < 0) ? kOutOfRange : uint32_t(r.k[j]) * 4u, 0, 0));
        const float l = s_c[win ? kk : 0];
        x[j] = r.v[j] * (win ? l : g);
      }
    }
    const uint32_t s0 = uint32_t(__builtin_amdgcn_readfirstlane(int(fb))) & 1u;
    // a range that begins inside a fibre: that fibre's pieces go to the table
    // (selects, not a branch: the trip's units stay one block of code that
    // the compiler can interleave)
    const bool inside = u == ub && !s0;
    cfid = inside ? ufid : cfid;
    hfid = inside ? ufid : hfid;
    const int32_t fid0 = ufid + wave_excl_count(uint32_t(__popc(fb))) + int32_t(fb & 1u) -
                         int32_t(s0);
    // the carried fibre ends at the unit boundary, or continues in lane 0
    emit(s0 && cfid >= 0 && lane == 0, cfid, cval);
    float sum = (lane == 0 && !s0 && cfid >= 0) ? cval : 0.f;
    float head = 0.f;
    bool closed = false;
    int32_t f = fid0;
#pragma unroll
    for (int j = 1; j < 8; ++j) {
      sum += x[j - 1];
      const bool b = (fb >> j) & 1u;
      put(f, sum, b && closed);  // began and ended inside this lane
      head = (b && !closed) ? sum : head;
      closed = closed || b;
      f += b ? 1 : 0;
      sum = b ? 0.f : sum;
    }
    sum += x[7];
    // segmented inclusive scan of the lanes' open (last) fibres
    const int32_t key = active ? f : INT_MAX;
    const float incl = seg_scan(active ? sum : 0.f, key);
    const float prev = dpp_f<0x138>(0.f, incl);                    // lane - 1 (lane 0: 0)
    const uint32_t nb0 = uint32_t(dpp_i<0x130>(0, int32_t(fb))) & 1u;  // lane + 1
    const int32_t lastl = __builtin_amdgcn_readfirstlane(min(63, (nnz - 1 - P) >> 3));
    emit(active && closed, fid0, head + ((!(fb & 1u) && lane > 0) ? prev : 0.f));
    emit(active && lane < lastl && nb0, f, incl);
    cfid = __builtin_amdgcn_readlane(key, lastl);
    cval = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(incl), lastl));
  };
  // unit u lives in q[(u - ub) % NB]
  UnitRegs q[NB];
#pragma unroll
  for (int s = 0; s < PF; ++s)
    if (ub + s < ue) fetch(ub + s, q[s]);
  stage();
  // every step of a trip runs, so a set is never reloaded while the wait
  // for its previous loads could be pending on some path
  int32_t u0 = ub;
  for (; u0 + NB <= ue; u0 += NB) {
#pragma unroll
    for (int s = 0; s < NB; ++s) {
      const int32_t u = u0 + s;
      // past the range the last unit is loaded again (from cache): with
      // every trip's loads issued, each wait counts only this unit's loads
      fetch(min(u + PF, ue - 1), q[(s + PF) % NB]);
      work(u, q[s]);
    }
  }
  // the last (fewer than NB) units, already loaded
#pragma unroll
  for (int s = 0; s < NB - 1; ++s)
    if (u0 + s < ue) work(u0 + s, q[s]);
  // a range that ends where a fibre starts (or at the end of the data)
  // completes its open fibre, unless that fibre also began before the range
  if (close_tail() && cfid >= 0 && cfid != hfid) {
    put(cfid, cval, lane == 0);
    cfid = -1;
    cval = 0.f;
  }
  // this range's entries of the crossing-fibre table
  const uint64_t hm = __ballot(hset);
  float hsum = 0.f;
  if (hm) hsum = __shfl(hval, int(__ffsll(static_cast<unsigned long long>(hm)) - 1));
  if (lane == 0) {
    bnd_fid[2 * w] = hm ? hfid : -1;
    bnd_val[2 * w] = hsum;
    bnd_fid[2 * w + 1] = cfid;
    bnd_val[2 * w + 1] = cval;
  }
}

template <int LC>
__global__ __launch_bounds__(kUnitThreads) void ttv_unit_kernel(
    const int32_t* __restrict__ crd, const float* __restrict__ vals,
    const uint32_t* __restrict__ flags, const int32_t* __restrict__ unit_fid,
    const float* __restrict__ cv, int32_t cdim, int32_t k0, int32_t lc, float* __restrict__ y,
    int32_t ny, int32_t nnz, int32_t nunits, int32_t* __restrict__ bnd_fid,
    float* __restrict__ bnd_val, const int32_t* __restrict__ ne_fid) {
  __shared__ float s_c[LC];
  const __amdgpu_buffer_rsrc_t crs = c_rsrc(cv, cdim);
  const int32_t W = int32_t(gridDim.x) * kUnitWaves;
  const int32_t w = int32_t(blockIdx.x) * kUnitWaves + int32_t(threadIdx.x >> 6);
  const int32_t ub = int32_t(int64_t(nunits) * w / W);
  const int32_t ue = int32_t(int64_t(nunits) * (w + 1) / W);
  // the global gathers of a unit are waited for with the loads issued
  // before them, so one unit ahead is as far as loading ahead reaches here
  ttv_units_wave<false, false, 1>(crd, vals, flags, unit_fid, crs, s_c, k0, lc, y, ny, nnz, ub, ue,
                                  w, bnd_fid, bnd_val, ne_fid, [] { return false; }, [&] {
                                    stage_window<LC>(s_c, crs, k0, lc);
                                    __syncthreads();
                                  });
}

// The unit kernel's form for tensors of few units and no long fibre: a wave sums
// whole fibres, those that start in its unit, so there is no crossing table
// and no second launch, and waves need neither each other nor a window of c
// (which L2 serves at these sizes). The unit's products go to LDS in FP64
// (exact) and a lane sums a fibre; one of more than kFibreLane nonzeros, and
// what the last fibre has past the unit, is summed by the whole wave. y is
// written once per entry, coalesced, without atomics (bitwise reproducible).
// Two dependent rounds of loads bound it: 200k nonzeros, 27k fibres: 5.3 us
// against 8.5 for the form with the window (25 workgroups of 16 waves) and its fold;
// the plan takes 0.1 ms, bands another 0.5 to 2 ms.
// kFibreLane: 8 11.1 us, 16 6.9, 24 6.1, 48 5.3, 100 5.5 (a wave's sum is 12
// cross-lane moves of latency, a lane's a serial chain).
// Taken up to kFibreUnits units, us of this and of the other form (banded
// where c is past its window): 24k nonzeros 4.8 and 7.7, 445k 7.0 and 20.9, 1M
// 6.2 and 8.9 (c of 4000) or 9.2 and 15.4 (c of 150000), 2M 10.1 and 9.7 or
// 13.8 and 16.3, 4M 17.2 and 14.0 or 24.6 and 19.4. And up to fibres of
// kFibreMax nonzeros, since a wave sums the rest of its last fibre alone.
constexpr int kFibreWaves = 4;
constexpr int32_t kFibreUnits = 2048;
constexpr int64_t kFibreMax = 2048;
constexpr int32_t kFibreLane = 48;
__global__ __launch_bounds__(64 * kFibreWaves) void ttv_unit_kernel(
    const int32_t* __restrict__ crd, const float* __restrict__ vals,
    const uint32_t* __restrict__ flags, const int32_t* __restrict__ unit_fid,
    const int32_t* __restrict__ pos, const float* __restrict__ cv, float* __restrict__ y,
    int32_t nf, int32_t nnz, int32_t nunits) {
  __shared__ double s_x[kFibreWaves][kUnit];
  const int lane = int(threadIdx.x) & 63;
  const int wv = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int32_t u = int32_t(blockIdx.x) * kFibreWaves + wv;
  if (u >= nunits) return;
  double* x = s_x[wv];
  const int32_t P = u * kUnit;
  int32_t k[8];
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int32_t p = min(P + j * 64 + lane, nnz - 1);
    k[j] = crd[p];
    v[j] = vals[p];
  }
  // fibres [f0, f1) start in this unit
  const bool last = u + 1 == nunits;
  const int32_t un = last ? u : u + 1;
  const int32_t f0 = unit_fid[u] + ((flags[u * (kUnit / 32)] & 1u) ? 0 : 1);
  const int32_t f1 = last ? nf : unit_fid[un] + ((flags[un * (kUnit / 32)] & 1u) ? 0 : 1);
  if (f0 >= f1) return;  // one fibre that started earlier covers the unit
  const int32_t end = pos[f1];
#pragma unroll
  for (int j = 0; j < 8; ++j) x[j * 64 + lane] = double(v[j]) * cv[k[j]];
  // the last fibre's nonzeros past the unit
  double t = 0.0;
  for (int32_t p0 = P + kUnit; p0 < end; p0 += 4 * 64) {
    double a[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int32_t p = p0 + j * 64 + lane;
      const int32_t q = min(p, end - 1);
      a[j] = p < end ? double(vals[q]) * cv[crd[q]] : 0.0;
    }
    t += (a[0] + a[1]) + (a[2] + a[3]);
  }
  if (end > P + kUnit) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) t += __shfl_xor(t, o);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  for (int32_t fb = f0; fb < f1; fb += 64) {
    const int32_t f = fb + lane;
    const int32_t a = f < f1 ? pos[f] - P : 0;
    const int32_t e = f < f1 ? min(pos[f + 1] - P, kUnit) : 0;
    double s = 0.0;
    if (e - a <= kFibreLane) {
      double s1 = 0.0;
      int32_t i = a;
      for (; i + 4 <= e; i += 4) {
        const double x0 = x[i], x1 = x[i + 1], x2 = x[i + 2], x3 = x[i + 3];
        s += x0 + x1;
        s1 += x2 + x3;
      }
      if (i + 2 <= e) {
        s1 += x[i] + x[i + 1];
        i += 2;
      }
      if (i < e) s += x[i];
      s += s1;
    }
    for (uint64_t big = __ballot(e - a > kFibreLane); big; big &= big - 1) {
      const int l = __builtin_ctzll(big);
      const int32_t ba = __builtin_amdgcn_readlane(a, l);
      const int32_t be = __builtin_amdgcn_readlane(e, l);
      double b = 0.0;
      for (int32_t i = ba + lane; i < be; i += 64) b += x[i];
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) b += __shfl_xor(b, o);
      if (lane == l) s = b;
    }
    if (f < f1) y[f] = float(s + (f == f1 - 1 ? t : 0.0));
  }
}

// First unit of wave i of the nwav waves that split a band's units
// [unit0, unit0 + units) evenly; i = nwav gives the band's end. The plan
// builder places the crossing table by the same function.
__host__ __device__ inline int32_t band_wave_start(int32_t unit0, int32_t units, int32_t nwav,
                                                   int32_t i) {
  return unit0 + int32_t(int64_t(units) * i / (nwav > 0 ? nwav : 1));
}

// The bands of the banded layout, by value (kernel argument).
struct BandArgs {
  int nb;
  int32_t band_w;
  int32_t cdim;
  int32_t unit0[kMaxBands + 1];
  int32_t wg0[kMaxBands + 1];
};

// The banded layout: workgroups wg0[b] .. wg0[b+1) stage band b of c and
// split its units among their waves; crd holds each nonzero's index in its
// band's window (padding: LC - 1, a slot past every band that stays 0), so
// every gather is an LDS read. Output: the nseg segment sums.
template <int LC>
__global__ __launch_bounds__(kUnitThreads) void ttv_band_kernel(
    const uint16_t* __restrict__ crd, const float* __restrict__ vals,
    const uint32_t* __restrict__ flags, const int32_t* __restrict__ unit_fid,
    const float* __restrict__ cv, BandArgs ba, float* __restrict__ seg, int32_t nseg,
    int32_t len, int32_t* __restrict__ bnd_fid, float* __restrict__ bnd_val) {
  __shared__ float s_c[LC];
  const int32_t g = int32_t(blockIdx.x);
  int b = 0;
  while (b + 1 < ba.nb && g >= ba.wg0[b + 1]) ++b;
  const int32_t k0 = b * ba.band_w;
  const int32_t lc = min(ba.band_w, ba.cdim - k0);
  const __amdgpu_buffer_rsrc_t crs = c_rsrc(cv, ba.cdim);
  // the wave's units: its share of the even split of the band's units
  const int32_t w = g * kUnitWaves + int32_t(threadIdx.x >> 6);
  const int32_t wb = w - ba.wg0[b] * kUnitWaves;
  const int32_t nwav = (ba.wg0[b + 1] - ba.wg0[b]) * kUnitWaves;
  const int32_t units = ba.unit0[b + 1] - ba.unit0[b];
  const int32_t ub = band_wave_start(ba.unit0[b], units, nwav, wb);
  const int32_t ue = band_wave_start(ba.unit0[b], units, nwav, wb + 1);
  // the start-bit word after the range (len > 0), loaded now and read after
  // the last unit; an unconditional load keeps its use out of any branch
  // here, where the compiler would wait for it at once
  const int32_t pe = ue * kUnit;
  const uint32_t tw = flags[min(pe, len - 1) >> 5];
  ttv_units_wave<true, true, kBandPF>(
      crd, vals, flags, unit_fid, crs, s_c, k0, lc, seg, nseg, len, ub, ue, w, bnd_fid, bnd_val,
      nullptr, [&] { return ub < ue && (pe >= len || ((tw >> (pe & 31)) & 1u)); },
      [&] {
        stage_window<LC>(s_c, crs, k0, lc);
        __syncthreads();
      });
}

// y(f) = sum of the crossing-table entries of f, for every fibre in the
// table (entries in position order, -1 = none); runs after the unit kernel,
// so the launch boundary makes its entries visible (no fences between
// workgroups on different XCDs)
__global__ __launch_bounds__(256) void ttv_fold_kernel(
    const int32_t* __restrict__ bnd_fid, const float* __restrict__ bnd_val, int32_t E,
    float* __restrict__ y, const int32_t* __restrict__ ne_fid,
    const int32_t* __restrict__ empty_ids, int32_t n_empty) {
  const int32_t e = int32_t(blockIdx.x) * 256 + int32_t(threadIdx.x);
  if (e < n_empty) y[empty_ids[e]] = 0.f;  // empty fibres
  if (e >= E) return;
  // the entry and its neighbours in one round of loads (runs are short:
  // a fibre has at most one entry per wave range it touches, and invalid
  // entries are heads only)
  auto fid_at = [&](int32_t i) { return (i >= 0 && i < E) ? bnd_fid[i] : -2; };
  const int32_t fm2 = fid_at(e - 2), fm1 = fid_at(e - 1), f = bnd_fid[e];
  const int32_t f1 = fid_at(e + 1), f2 = fid_at(e + 2);
  const float v0 = bnd_val[e];
  const float v1 = e + 1 < E ? bnd_val[e + 1] : 0.f;
  const float v2 = e + 2 < E ? bnd_val[e + 2] : 0.f;
  if (f < 0) return;
  // the previous valid entry: e-1, else e-2 when e-1 is invalid, else further
  int32_t prev = fm1 >= 0 ? fm1 : (fm1 == -2 ? -2 : fm2);
  if (fm1 == -1 && fm2 == -1) {
    int32_t q = e - 3;
    while (q >= 0 && bnd_fid[q] < 0) --q;
    prev = q >= 0 ? bnd_fid[q] : -2;
  }
  if (prev == f) return;  // not the first entry of f
  float s = v0;
  int32_t r = e + 1;
  if (f1 == f || f1 == -1) {
    if (f1 == f) s += v1;
    r = e + 2;
    if (f2 == f || f2 == -1) {
      if (f2 == f) s += v2;
      for (r = e + 3; r < E; ++r) {
        const int32_t g = bnd_fid[r];
        if (g < 0) continue;
        if (g != f) break;
        s += bnd_val[r];
      }
    }
  }
  y[ne_fid ? ne_fid[f] : f] = s;
}

// ---------------------------------------------------------------------------
// Building the banded layout (once per handle, from B alone)

// Band boundaries for the build kernels: each band's first place in band
// order (the nonzeros of bands before it) and its first padded position.
struct BandOff {
  int nb;
  int32_t start[kMaxBands + 1];
  int32_t off[kMaxBands + 1];
};

__device__ __forceinline__ int band_of_position(const BandOff& bo, int32_t d) {
  int b = 0;
  while (b + 1 < bo.nb && d >= bo.off[b + 1]) ++b;
  return b;
}

// fib[p] = f for every nonzero p of fibre f
__global__ __launch_bounds__(256) void band_fib_kernel(const int32_t* __restrict__ pos, int32_t nf,
                                                       int32_t* __restrict__ fib) {
  const int64_t tid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t f = tid; f < nf; f += nthr)
    for (int32_t p = pos[f]; p < pos[f + 1]; ++p) fib[p] = int32_t(f);
}

// The nonzeros go to their bands by a stable partition over chunks of
// kPartChunk nonzeros, one 256-thread workgroup per chunk.
constexpr int kPartChunk = 4096;

// cblk[b * nblk + k] = nonzeros of chunk k in band b; cnt[b] = band b's total
__global__ __launch_bounds__(256) void band_count_kernel(const int32_t* __restrict__ crd,
                                                         int32_t nnz, int32_t band_w, int nb,
                                                         int32_t nblk, int32_t* __restrict__ cblk,
                                                         uint32_t* __restrict__ cnt) {
  __shared__ uint32_t h[kMaxBands];
  if (threadIdx.x < kMaxBands) h[threadIdx.x] = 0u;
  __syncthreads();
  const int64_t p0 = int64_t(blockIdx.x) * kPartChunk;
  const int64_t p1 = p0 + kPartChunk < int64_t(nnz) ? p0 + kPartChunk : int64_t(nnz);
  uint32_t c[kMaxBands];
#pragma unroll
  for (int j = 0; j < kMaxBands; ++j) c[j] = 0u;
  for (int64_t p = p0 + threadIdx.x; p < p1; p += blockDim.x) {
    const int b = min(crd[p] / band_w, nb - 1);
#pragma unroll
    for (int j = 0; j < kMaxBands; ++j) c[j] += b == j;
  }
#pragma unroll
  for (int j = 0; j < kMaxBands; ++j)
    if (c[j]) atomicAdd(&h[j], c[j]);
  __syncthreads();
  if (int(threadIdx.x) < nb) {
    cblk[int64_t(threadIdx.x) * nblk + blockIdx.x] = int32_t(h[threadIdx.x]);
    if (h[threadIdx.x]) atomicAdd(cnt + threadIdx.x, h[threadIdx.x]);
  }
}

// padding everywhere first: coordinate -1 (gathers 0), value 0, no fibre
__global__ __launch_bounds__(256) void band_pad_kernel(uint16_t* __restrict__ bcrd,
                                                       float* __restrict__ bvals,
                                                       int32_t* __restrict__ bfib, int32_t len,
                                                       uint16_t pad_off) {
  const int64_t tid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t d = tid; d < len; d += nthr) {
    bcrd[d] = pad_off;
    bvals[d] = 0.f;
    bfib[d] = -1;
  }
}

// Each chunk's nonzeros, in their order, go to their band's padded range
// after the chunks before (oblk: exclusive prefix of cblk, band-major, so
// oblk[b * nblk + k] - bo.start[b] is chunk k's first place in band b); a
// nonzero's rank among its chunk's nonzeros of its band comes from wave
// ballots, 256 nonzeros a round. Its leaf coordinate is stored as an index
// in its band's window of band_w (< 2^16) coordinates. blockDim.x = 256.
__global__ __launch_bounds__(256) void band_part_kernel(
    const int32_t* __restrict__ crd, const float* __restrict__ vals,
    const int32_t* __restrict__ fib, int32_t nnz, int32_t band_w, BandOff bo, int32_t nblk,
    const int32_t* __restrict__ oblk, uint16_t* __restrict__ bcrd, float* __restrict__ bvals,
    int32_t* __restrict__ bfib) {
  __shared__ int32_t run[kMaxBands];    // next place of each band
  __shared__ int32_t wc[4][kMaxBands];  // the round's count per wave and band
  const int nb = bo.nb;
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  const int t = threadIdx.x;
  if (t < nb) run[t] = bo.off[t] + (oblk[int64_t(t) * nblk + blockIdx.x] - bo.start[t]);
  __syncthreads();
  const int64_t p0 = int64_t(blockIdx.x) * kPartChunk;
  const int64_t p1 = p0 + kPartChunk < int64_t(nnz) ? p0 + kPartChunk : int64_t(nnz);
  const uint64_t below = (uint64_t(1) << lane) - 1u;
  for (int64_t r = p0; r < p1; r += 256) {
    const int64_t p = r + t;
    const bool in = p < p1;
    const int32_t cv = in ? crd[p] : 0;
    const int b = in ? min(cv / band_w, nb - 1) : -1;
    int rank = 0;
    for (int j = 0; j < nb; ++j) {
      const uint64_t m = __ballot(b == j);
      if (b == j) rank = __popcll(m & below);
      if (lane == 0) wc[wv][j] = __popcll(m);
    }
    __syncthreads();
    if (in) {
      int32_t d = run[b] + rank;
      for (int v = 0; v < wv; ++v) d += wc[v][b];
      bcrd[d] = uint16_t(cv - b * band_w);
      bvals[d] = vals[p];
      bfib[d] = fib[p];
    }
    __syncthreads();
    if (t < nb) run[t] += wc[0][t] + wc[1][t] + wc[2][t] + wc[3][t];
    __syncthreads();
  }
}

// segment starts: a real position whose fibre differs from the previous
// position's, or the first position of its band. One position per lane: a
// wave's 64 consecutive positions make two words of flags (bit j of word w
// is position 32 w + j; len is a multiple of 64), wcnt[w] = the word's
// count. Each start also sets its fibre's bit in its band's presence bitmap
// (present[b * fwords + f / 32], cleared before).
__global__ __launch_bounds__(256) void band_flags_kernel(const int32_t* __restrict__ bfib,
                                                         int32_t nwords, BandOff bo,
                                                         int32_t fwords,
                                                         uint32_t* __restrict__ flags,
                                                         int32_t* __restrict__ wcnt,
                                                         uint32_t* __restrict__ present) {
  const int64_t n = int64_t(nwords) * 32;
  const int lane = threadIdx.x & 63;
  const int64_t wave = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
  const int64_t nwave = (int64_t(gridDim.x) * blockDim.x) >> 6;
  for (int64_t base = wave * 64; base < n; base += nwave * 64) {
    const int64_t d = base + lane;
    const int32_t f = bfib[d];
    const int32_t fp = d > 0 ? bfib[d - 1] : -1;
    bool start = false;
    if (f >= 0) {
      bool first = false;
      for (int b = 0; b < bo.nb; ++b) first |= d == bo.off[b];
      start = first || f != fp;
    }
    const uint64_t m = __ballot(start);
    if ((lane & 31) == 0) {
      const uint32_t word = uint32_t(m >> lane);
      flags[(base >> 5) + (lane >> 5)] = word;
      wcnt[(base >> 5) + (lane >> 5)] = __popc(word);
    }
    // one atomic per presence word the wave's starts touch (a wave's
    // positions are consecutive, so its starts' fibres share few words): the
    // lowest remaining start's word, the OR of the bits of every start with
    // that word, until none remain
    const int64_t pw = start ? int64_t(band_of_position(bo, int32_t(d))) * fwords + (f >> 5) : -1;
    const uint32_t bit = start ? 1u << (f & 31) : 0u;
    uint64_t left = m;
    while (left) {
      const int L = __ffsll(static_cast<unsigned long long>(left)) - 1;
      const int64_t w = __shfl(pw, L);
      const bool mine = start && pw == w;
      uint32_t v = mine ? bit : 0u;
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) v |= __shfl_xor(v, o);
      if (lane == L) atomicOr(present + w, v);
      left &= ~__ballot(mine);
    }
  }
}

// unit_fid[u] = segment holding unit u's first position (wpre: exclusive
// prefix of the segment starts per word)
__global__ __launch_bounds__(256) void band_unit_kernel(const uint32_t* __restrict__ flags,
                                                        const int32_t* __restrict__ wpre,
                                                        int32_t nunits,
                                                        int32_t* __restrict__ unit_fid) {
  const int64_t tid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t u = tid; u < nunits; u += nthr) {
    const int64_t w = u * (kUnit / 32);
    unit_fid[u] = wpre[w] + int32_t(flags[w] & 1u) - 1;
  }
}

__global__ __launch_bounds__(256) void popc_kernel(const uint32_t* __restrict__ words, int32_t n,
                                                   int32_t* __restrict__ cnt) {
  const int64_t tid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t i = tid; i < n; i += nthr) cnt[i] = __popc(words[i]);
}

// A crossing piece's sum slot holds a signalling NaN whose payload is its
// index + 1 in the crossing list; arithmetic never produces a signalling
// NaN, so no computed sum reads as a marker.
constexpr uint32_t kMarkExp = 0x7F800000u;
__global__ __launch_bounds__(256) void band_mark_kernel(const int4* __restrict__ crl, int32_t n,
                                                        float* __restrict__ seg) {
  const int64_t tid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t nthr = int64_t(gridDim.x) * blockDim.x;
  for (int64_t i = tid; i < n; i += nthr)
    seg[crl[i].z] = __uint_as_float(kMarkExp | uint32_t(i + 1));
}

// wst: first unit of each of the nw wave ranges (wst[nw]: the end). For the
// range of wave w > 0 that starts inside a piece (its first position is no
// piece start), out[w] = (2 w0 + 1, 2 w1 + 1, piece, 0) with w0, w1 the waves
// holding the piece's first and last positions; out[w].z = -1 otherwise.
// Range starts are unit starts, bit 0 of their word; a piece starts at every
// band's first position, so the backward scan ends; padding carries no
// start bits and belongs to the piece before it.
__global__ __launch_bounds__(256) void band_cross_kernel(const uint32_t* __restrict__ flags,
                                                         const int32_t* __restrict__ wpre,
                                                         int32_t nwords,
                                                         const int32_t* __restrict__ wst, int32_t nw,
                                                         int4* __restrict__ out) {
  const int32_t w = int32_t(blockIdx.x) * int32_t(blockDim.x) + int32_t(threadIdx.x);
  if (w >= nw) return;
  int4 r = make_int4(0, 0, -1, 0);
  const int32_t t = wst[w];
  const int32_t qw = t * (kUnit / 32);
  if (w > 0 && t < wst[w + 1] && (flags[qw] & 1u) == 0u) {
    int32_t j = qw - 1;
    while (j > 0 && flags[j] == 0u) --j;
    const int64_t a = flags[j] != 0u ? int64_t(j) * 32 + 31 - __clz(int(flags[j])) : 0;
    int64_t e = int64_t(nwords) * 32;
    if (flags[qw] != 0u) {
      e = int64_t(qw) * 32 + __ffs(int(flags[qw])) - 1;
    } else {
      for (int32_t k = qw + 1; k < nwords; ++k)
        if (flags[k] != 0u) {
          e = int64_t(k) * 32 + __ffs(int(flags[k])) - 1;
          break;
        }
    }
    auto wave_of = [&](int64_t x) {  // last wave whose first unit <= x's unit
      const int32_t u = int32_t(x / kUnit);
      int32_t lo = 0, hi = nw - 1;
      while (lo < hi) {
        const int32_t mid = lo + ((hi - lo + 1) >> 1);
        if (wst[mid] <= u) lo = mid;
        else hi = mid - 1;
      }
      return lo;
    };
    r = make_int4(2 * wave_of(a) + 1, 2 * wave_of(e - 1) + 1, wpre[qw] - 1, 0);
  }
  out[w] = r;
}

// The sum of a piece read from its slot: a marker sends it to the crossing
// table, whose parts of the piece are added in position order.
__device__ __forceinline__ float piece_sum(float v, const int4* __restrict__ crl, int32_t ncrl,
                                           const int32_t* __restrict__ bnd_fid,
                                           const float* __restrict__ bnd_val) {
  const uint32_t bits = __float_as_uint(v);
  const uint32_t idx = (bits & 0x003FFFFFu) - 1u;
  if ((bits & 0x7FC00000u) != kMarkExp || idx >= uint32_t(ncrl)) return v;
  const int4 L = crl[idx];
  float s = 0.f;
  // four slots' loads in flight at a time (most pieces have 3 slots)
  for (int32_t k0 = L.x; k0 <= L.y; k0 += 4) {
    int32_t f[4];
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bool in = k0 + j <= L.y;
      f[j] = in ? bnd_fid[k0 + j] : -1;
      v[j] = in ? bnd_val[k0 + j] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (f[j] == L.z) s += v[j];
  }
  return s;
}

// y[f] = sum over the bands, in band order, of fibre f's segment sums
// (0 for fibres without nonzeros). A wave covers kCombU x 64 consecutive
// fibres, lane-contiguous per step. With the band count known at compile
// time (NBT > 0) a wave issues every band's presence and prefix loads, then
// every band's segment loads, and only then resolves markers and sums: two
// rounds of loads in flight per wave. NBT = 0 (a run-time count up to
// kMaxBands) goes band by band.
constexpr int kCombU = 8;
template <int NBT>
__global__ __launch_bounds__(256) void band_combine_kernel(const uint32_t* __restrict__ present,
                                                           const int32_t* __restrict__ prefix,
                                                           int32_t fwords, int nb_rt,
                                                           const float* __restrict__ seg,
                                                           int32_t nf, float* __restrict__ y,
                                                           const int4* __restrict__ crl, int32_t ncrl,
                                                           const int32_t* __restrict__ bnd_fid,
                                                           const float* __restrict__ bnd_val) {
  constexpr int NBL = NBT > 0 ? NBT : 1;  // bands loaded together
  const int nb = NBT > 0 ? NBT : nb_rt;
  const int lane = threadIdx.x & 63;
  const int64_t nwave = int64_t(gridDim.x) * (blockDim.x >> 6);
  for (int64_t wv = int64_t(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
       wv * (64 * kCombU) < nf; wv += nwave) {
    float s[kCombU];
    for (int b0 = 0; b0 < nb; b0 += NBL) {
      uint32_t word[NBL][kCombU];
      int32_t base[NBL][kCombU];
#pragma unroll
      for (int i = 0; i < NBL; ++i)
#pragma unroll
        for (int u = 0; u < kCombU; ++u) {
          const int64_t f = wv * (64 * kCombU) + u * 64 + lane;
          const int64_t wi = (f < nf ? f : 0) >> 5;
          word[i][u] = present[int64_t(b0 + i) * fwords + wi];
          base[i][u] = prefix[int64_t(b0 + i) * fwords + wi];
        }
      float v[NBL][kCombU];
#pragma unroll
      for (int i = 0; i < NBL; ++i)
#pragma unroll
        for (int u = 0; u < kCombU; ++u) {
          const int64_t f = wv * (64 * kCombU) + u * 64 + lane;
          const uint32_t bit = uint32_t(f & 31);
          const bool has = f < nf && ((word[i][u] >> bit) & 1u);
          v[i][u] = has ? seg[base[i][u] + __popc(word[i][u] & ((1u << bit) - 1u))] : 0.f;
        }
#pragma unroll
      for (int i = 0; i < NBL; ++i)
#pragma unroll
        for (int u = 0; u < kCombU; ++u) {
          const float t = piece_sum(v[i][u], crl, ncrl, bnd_fid, bnd_val);
          s[u] = b0 + i == 0 ? t : s[u] + t;
        }
    }
#pragma unroll
    for (int u = 0; u < kCombU; ++u) {
      const int64_t f = wv * (64 * kCombU) + u * 64 + lane;
      if (f < nf) y[f] = s[u];
    }
  }
}

}  // namespace

int warm_ttv_module(hipStream_t st) {
  // no fibres: the launch touches no memory, it only loads the code object
  ttv_prep_kernel<<<1, 256, 0, st>>>(nullptr, nullptr, 0, 0, nullptr, 0);
  TT_HIP_CHECK(hipGetLastError());
  return TENTACO_OK;
}

size_t ttv_workspace_bytes(const CsfDev& B) {
  const int64_t nblk = (int64_t(B.nnz) + kTtvNB - 1) / kTtvNB;
  return size_t(nblk + 1) * sizeof(int32_t);
}

int launch_ttv(const CsfDev& B, const float* c, float* y, void* ws,
               hipStream_t st) {
  if (B.order < 2 || B.order > kMaxOrder)
    return fail(TENTACO_EUNSUPPORTED, "TTV order %d outside 2..5", B.order);
  const int32_t nf = B.nodes[B.order - 2];
  const int32_t* pos = B.pos[B.order - 1];
  const int32_t* crd = B.crd[B.order - 1];
  const int64_t nblk = (int64_t(B.nnz) + kTtvNB - 1) / kTtvNB;
  int32_t* brk = static_cast<int32_t*>(ws);
  int64_t g = (int64_t(nf) + 255) / 256;
  if (g < 1) g = 1;
  if (g > 16384) g = 16384;
  ttv_prep_kernel<<<int(g), 256, 0, st>>>(pos, y, nf, B.nnz, brk, int32_t(nblk));
  TT_HIP_CHECK(hipGetLastError());
  if (nblk == 0) return TENTACO_OK;
  ktimer_begin(st);
  ttv_kernel<<<int(nblk), kTtvBlock, 0, st>>>(pos, crd, B.vals, c, y, B.nnz, brk);
  TT_HIP_CHECK(hipGetLastError());
  ktimer_end(st, "ttv_kernel");
  return TENTACO_OK;
}

}  // namespace tt

namespace tt {
namespace {

constexpr int kTtvLdsMax = 38912;  // 152 KB of c per workgroup, one workgroup per CU
static_assert(kTtvLdsMax <= 65536, "band windows are indexed by 16 bits");

size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

// LDS instance of a band of band_w < kTtvLdsMax coordinates: its window
// keeps at least one slot past the band, which stays zero (the padding reads)
int band_inst(int32_t band_w) { return band_w < 4096 ? 4096 : band_w < 16384 ? 16384 : kTtvLdsMax; }

template <int LC>
int launch_units_typed(const CsfDev& B, const TtvPlan& P, const float* c, float* y,
                       hipStream_t st) {
  ktimer_begin(st);
  ttv_unit_kernel<LC><<<P.grid, kUnitThreads, 0, st>>>(
      B.crd[B.order - 1], B.vals, P.flags, P.unit_fid, c, P.cdim, P.k0, P.lc, y,
      B.nodes[B.order - 2], B.nnz, P.nunits, P.bnd_fid, P.bnd_val, P.ne_fid);
  TT_HIP_CHECK(hipGetLastError());
  ktimer_end(st, "ttv_unit_kernel");
  const int32_t E = 2 * P.grid * kUnitWaves;
  const int32_t nth = std::max(E, P.n_empty);
  ttv_fold_kernel<<<(nth + 255) / 256, 256, 0, st>>>(P.bnd_fid, P.bnd_val, E, y, P.ne_fid,
                                                       P.empty_ids, P.n_empty);
  TT_HIP_CHECK(hipGetLastError());
  return TENTACO_OK;
}

template <int LC>
int launch_bands_typed(const CsfDev& B, const TtvPlan& P, const float* c, float* y,
                       hipStream_t st) {
  BandArgs ba{};
  ba.nb = P.nbands;
  ba.band_w = P.band_w;
  ba.cdim = P.cdim;
  for (int b = 0; b <= P.nbands; ++b) {
    ba.unit0[b] = P.b_unit0[b];
    ba.wg0[b] = P.b_wg0[b];
  }
  ktimer_begin(st);
  ttv_band_kernel<LC><<<P.b_grid, kUnitThreads, 0, st>>>(P.b_crd, P.b_vals, P.b_flags,
                                                         P.b_unit_fid, c, ba, P.b_seg, P.b_nseg,
                                                         P.b_len, P.b_bnd_fid, P.b_bnd_val);
  TT_HIP_CHECK(hipGetLastError());
  ktimer_end(st, "ttv_band_kernel");
  // the crossing pieces are summed by the combine (no fold pass)
  const int32_t nf = B.nodes[B.order - 2];
  if (nf > 0) {
    const int64_t waves = (int64_t(nf) + 64 * kCombU - 1) / (64 * kCombU);
    const int g = int(std::max<int64_t>(1, std::min<int64_t>((waves + 3) / 4, 16384)));
    switch (P.nbands) {
      case 2:
        band_combine_kernel<2><<<g, 256, 0, st>>>(P.b_present, P.b_prefix, P.b_fwords, 2, P.b_seg,
                                                  nf, y, P.b_crossing, P.b_cross, P.b_bnd_fid,
                                                  P.b_bnd_val);
        break;
      case 3:
        band_combine_kernel<3><<<g, 256, 0, st>>>(P.b_present, P.b_prefix, P.b_fwords, 3, P.b_seg,
                                                  nf, y, P.b_crossing, P.b_cross, P.b_bnd_fid,
                                                  P.b_bnd_val);
        break;
      case 4:
        band_combine_kernel<4><<<g, 256, 0, st>>>(P.b_present, P.b_prefix, P.b_fwords, 4, P.b_seg,
                                                  nf, y, P.b_crossing, P.b_cross, P.b_bnd_fid,
                                                  P.b_bnd_val);
        break;
      default:
        band_combine_kernel<0><<<g, 256, 0, st>>>(P.b_present, P.b_prefix, P.b_fwords, P.nbands,
                                                  P.b_seg, nf, y, P.b_crossing, P.b_cross,
                                                  P.b_bnd_fid, P.b_bnd_val);
        break;
    }
    TT_HIP_CHECK(hipGetLastError());
  }
  return TENTACO_OK;
}

}  // namespace

void free_ttv_plan(TtvPlan* P) {
  if (!P) return;
  (void)hipFree(P->mem);
  (void)hipFree(P->mem2);
  (void)hipFree(P->bmem);
  (void)hipFree(P->bmem2);
  *P = TtvPlan{};
}

namespace {

// The banded layout of nb bands of band_w leaf coordinates (nb * band_w >=
// cdim, band_w < the LDS instance), built on `st` and waited for. On
// failure the plan keeps its one-window arrays (nbands stays 0).
int build_ttv_bands(const CsfDev& B, int nb, int32_t band_w, int cus, TtvPlan* P,
                    hipStream_t st) {
  const int32_t nnz = B.nnz;
  const int32_t nf = B.nodes[B.order - 2];
  const int32_t* pos = B.pos[B.order - 1];
  const int32_t* crd = B.crd[B.order - 1];
  auto grid_of = [](int64_t n) {
    return int(std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 16384)));
  };
  struct Free {
    void* p = nullptr;
    ~Free() { (void)hipFree(p); }
  } t1;
  // temporaries, in one allocation (sized by the bounds of the padded length
  // and of the wave count): for the stable partition by band, the fibre per
  // nonzero, per-chunk band counts and their prefix, band totals and the
  // scans' workspace; then the fibre of every padded position, per-word
  // counts and their prefix, the wave range starts and what starts inside a
  // piece
  const size_t b_n = align256(sizeof(int32_t) * size_t(nnz));
  const int32_t nblk = int32_t((int64_t(nnz) + kPartChunk - 1) / kPartChunk);
  const int64_t npart = int64_t(nb) * nblk;
  const size_t b_pc = align256(sizeof(int32_t) * size_t(npart));
  const int32_t fwords = (nf + 31) / 32;
  // upper bounds of the padded length and its words, for the scans' size
  const int64_t len_max = int64_t(nnz) + int64_t(nb) * kUnit;
  const int64_t nscan_max = std::max<int64_t>({len_max / 32, int64_t(nb) * fwords + 1, npart});
  size_t scan_bytes = 0;
  if (rocprim::exclusive_scan(nullptr, scan_bytes, static_cast<const int32_t*>(nullptr),
                              static_cast<int32_t*>(nullptr), 0, size_t(nscan_max),
                              rocprim::plus<int32_t>(), st) != hipSuccess)
    return fail(TENTACO_EHIP, "TTV bands: scan size query failed");
  const size_t b_ws = align256(std::max<size_t>(scan_bytes, 1));
  const size_t b_len = align256(sizeof(int32_t) * size_t(len_max));
  const size_t b_sc = align256(sizeof(int32_t) * size_t(std::max<int64_t>(len_max / 32, int64_t(nb) * fwords) + 1));
  const int64_t waves_max = (int64_t(std::max(cus, 1)) + 2 * nb) * kUnitWaves;  // given <= G + nb
  const size_t b_wst = align256(sizeof(int32_t) * size_t(waves_max + 1));
  const size_t b_xs = align256(sizeof(int4) * size_t(waves_max));
  const size_t o_t2 = b_n + 2 * b_pc + 256 + b_ws;
  if (hipMalloc(&t1.p, o_t2 + b_len + 2 * b_sc + b_wst + b_xs) != hipSuccess)
    return fail(TENTACO_ENOMEM, "TTV bands: temporary allocation failed");
  char* t = static_cast<char*>(t1.p);
  int32_t* fib = reinterpret_cast<int32_t*>(t);
  int32_t* cblk = reinterpret_cast<int32_t*>(t + b_n);
  int32_t* oblk = reinterpret_cast<int32_t*>(t + b_n + b_pc);
  uint32_t* cnt = reinterpret_cast<uint32_t*>(t + b_n + 2 * b_pc);
  void* wsp = t + b_n + 2 * b_pc + 256;
  TT_HIP_CHECK(hipMemsetAsync(cnt, 0, sizeof(uint32_t) * kMaxBands, st));
  band_fib_kernel<<<grid_of(nf), 256, 0, st>>>(pos, nf, fib);
  TT_HIP_CHECK(hipGetLastError());
  band_count_kernel<<<nblk, 256, 0, st>>>(crd, nnz, band_w, nb, nblk, cblk, cnt);
  TT_HIP_CHECK(hipGetLastError());
  if (rocprim::exclusive_scan(wsp, scan_bytes, static_cast<const int32_t*>(cblk), oblk, 0,
                              size_t(npart), rocprim::plus<int32_t>(), st) != hipSuccess)
    return fail(TENTACO_EHIP, "TTV bands: scan failed");
  uint32_t cnt_h[kMaxBands] = {};
  TT_HIP_CHECK(hipMemcpyAsync(cnt_h, cnt, sizeof(cnt_h), hipMemcpyDeviceToHost, st));
  TT_HIP_CHECK(hipStreamSynchronize(st));
  BandOff bo{};
  bo.nb = nb;
  int32_t units[kMaxBands] = {};
  int64_t len = 0, start = 0;
  for (int b = 0; b < nb; ++b) {
    bo.start[b] = int32_t(start);
    bo.off[b] = int32_t(len);
    units[b] = int32_t((int64_t(cnt_h[b]) + kUnit - 1) / kUnit);
    start += cnt_h[b];
    len += int64_t(units[b]) * kUnit;
  }
  bo.start[nb] = int32_t(start);
  bo.off[nb] = int32_t(len);
  if (start != nnz || len > len_max) return fail(TENTACO_EINVAL, "TTV bands: band counts do not add up");
  const int32_t nunits = int32_t(len / kUnit);
  const int32_t nwords = int32_t(len / 32);
  // workgroups per band in proportion to its units, at least one per
  // non-empty band, about one per CU in all
  int nonempty = 0;
  for (int b = 0; b < nb; ++b) nonempty += units[b] > 0;
  int64_t G = std::max<int64_t>(1, std::min<int64_t>(std::max(cus, 1), nunits / kUnitWaves));
  G = std::max<int64_t>(G, nonempty);
  int32_t wg[kMaxBands] = {};
  int64_t given = 0;
  for (int b = 0; b < nb; ++b) {
    if (!units[b]) continue;
    wg[b] = int32_t(std::max<int64_t>(1, (G * units[b]) / nunits));
    given += wg[b];
  }
  while (given < G) {  // what rounding left, to the most loaded bands
    int best = -1;
    double most = -1.0;
    for (int b = 0; b < nb; ++b)
      if (units[b] && double(units[b]) / wg[b] > most) {
        most = double(units[b]) / wg[b];
        best = b;
      }
    ++wg[best];
    ++given;
  }
  const int32_t max_waves = int32_t(given) * kUnitWaves;
  if (max_waves > waves_max) return fail(TENTACO_EINVAL, "TTV bands: %d waves", max_waves);
  // the layout
  const size_t o_crd = 0;
  const size_t o_vals = o_crd + align256(sizeof(uint16_t) * size_t(len));
  const size_t o_flags = o_vals + align256(sizeof(float) * size_t(len));
  const size_t o_unit = o_flags + align256(sizeof(uint32_t) * size_t(nwords));
  const size_t o_bfid = o_unit + align256(sizeof(int32_t) * size_t(nunits));
  const size_t o_bval = o_bfid + align256(sizeof(int32_t) * 2 * size_t(max_waves));
  const size_t o_pres = o_bval + align256(sizeof(float) * 2 * size_t(max_waves));
  const size_t o_pref = o_pres + align256(sizeof(uint32_t) * size_t(nb) * fwords);
  const size_t o_crl = o_pref + align256(sizeof(int32_t) * (size_t(nb) * fwords + 1));
  const size_t total = o_crl + align256(sizeof(int4) * size_t(max_waves));
  void* mem = nullptr;
  if (hipMalloc(&mem, total) != hipSuccess)
    return fail(TENTACO_ENOMEM, "TTV bands: hipMalloc of %zu bytes failed", total);
  struct Keep {
    void* p;
    bool keep = false;
    ~Keep() {
      if (!keep) (void)hipFree(p);
    }
  } kmem{mem};
  char* base = static_cast<char*>(mem);
  uint16_t* b_crd = reinterpret_cast<uint16_t*>(base + o_crd);
  float* b_vals = reinterpret_cast<float*>(base + o_vals);
  uint32_t* b_flags = reinterpret_cast<uint32_t*>(base + o_flags);
  int32_t* b_unit = reinterpret_cast<int32_t*>(base + o_unit);
  uint32_t* b_pres = reinterpret_cast<uint32_t*>(base + o_pres);
  int32_t* b_pref = reinterpret_cast<int32_t*>(base + o_pref);
  char* t2 = t + o_t2;
  int32_t* bfib = reinterpret_cast<int32_t*>(t2);
  int32_t* wcnt = reinterpret_cast<int32_t*>(t2 + b_len);
  int32_t* wpre = reinterpret_cast<int32_t*>(t2 + b_len + b_sc);
  int32_t* d_wst = reinterpret_cast<int32_t*>(t2 + b_len + 2 * b_sc);
  int4* d_xs = reinterpret_cast<int4*>(t2 + b_len + 2 * b_sc + b_wst);
  // padding reads the window's last slot, past every band (band_w < inst)
  band_pad_kernel<<<grid_of(len), 256, 0, st>>>(b_crd, b_vals, bfib, int32_t(len),
                                                uint16_t(band_inst(band_w) - 1));
  TT_HIP_CHECK(hipGetLastError());
  band_part_kernel<<<nblk, 256, 0, st>>>(crd, B.vals, fib, nnz, band_w, bo, nblk, oblk, b_crd, b_vals,
                                         bfib);
  TT_HIP_CHECK(hipGetLastError());
  // segment starts and which fibres have a segment in each band, the starts'
  // prefix per word, the unit table
  TT_HIP_CHECK(hipMemsetAsync(b_pres, 0, sizeof(uint32_t) * size_t(nb) * fwords, st));
  band_flags_kernel<<<grid_of(len), 256, 0, st>>>(bfib, nwords, bo, fwords, b_flags, wcnt, b_pres);
  TT_HIP_CHECK(hipGetLastError());
  if (rocprim::exclusive_scan(wsp, scan_bytes, static_cast<const int32_t*>(wcnt), wpre, 0,
                              size_t(nwords), rocprim::plus<int32_t>(), st) != hipSuccess)
    return fail(TENTACO_EHIP, "TTV bands: scan failed");
  band_unit_kernel<<<grid_of(nunits), 256, 0, st>>>(b_flags, wpre, nunits, b_unit);
  TT_HIP_CHECK(hipGetLastError());
  int32_t segs_h[2] = {0, 0};
  TT_HIP_CHECK(hipMemcpyAsync(&segs_h[0], wpre + nwords - 1, sizeof(int32_t), hipMemcpyDeviceToHost, st));
  TT_HIP_CHECK(hipMemcpyAsync(&segs_h[1], wcnt + nwords - 1, sizeof(int32_t), hipMemcpyDeviceToHost, st));
  // the segment index of each presence word's first set bit (band-major,
  // which is segment order)
  const int32_t npw = nb * fwords;
  popc_kernel<<<grid_of(npw), 256, 0, st>>>(b_pres, npw, wcnt);
  TT_HIP_CHECK(hipGetLastError());
  if (rocprim::exclusive_scan(wsp, scan_bytes, static_cast<const int32_t*>(wcnt), b_pref, 0,
                              size_t(npw), rocprim::plus<int32_t>(), st) != hipSuccess)
    return fail(TENTACO_EHIP, "TTV bands: scan failed");
  // wave ranges: the even split of each band's units, which the band kernel
  // computes by band_wave_start (moving starts to piece starts unbalances the
  // waves: up to 1.6x slower on 20M nonzeros); a range that starts inside a
  // piece leaves that piece's parts in the crossing table
  std::vector<int32_t> wst(size_t(max_waves) + 1);
  {
    int32_t u0 = 0, g0 = 0;
    for (int b = 0; b < nb; ++b) {
      const int32_t nwav = wg[b] * kUnitWaves;
      int32_t prev = u0;
      for (int32_t i = 0; i < nwav; ++i) {
        const int32_t t = std::max(band_wave_start(u0, units[b], nwav, i), prev);
        wst[size_t(g0) * kUnitWaves + size_t(i)] = t;
        prev = t;
      }
      u0 += units[b];
      g0 += wg[b];
    }
    wst[size_t(max_waves)] = u0;
  }
  // the pieces that cross a range start: their parts sit in the crossing
  // table at slots [2 w0 + 1, 2 w1 + 1] (w0, w1: the waves holding the
  // piece's first and last positions), and the combine sums them there;
  // found on the device (the piece-start bitmap stays there), listed once
  // each on the host
  std::vector<int4> xs(static_cast<size_t>(max_waves));
  TT_HIP_CHECK(hipMemcpyAsync(d_wst, wst.data(), sizeof(int32_t) * wst.size(), hipMemcpyHostToDevice,
                              st));
  band_cross_kernel<<<(max_waves + 255) / 256, 256, 0, st>>>(b_flags, wpre, nwords, d_wst, max_waves,
                                                             d_xs);
  TT_HIP_CHECK(hipGetLastError());
  TT_HIP_CHECK(hipMemcpyAsync(xs.data(), d_xs, sizeof(int4) * xs.size(), hipMemcpyDeviceToHost, st));
  TT_HIP_CHECK(hipStreamSynchronize(st));
  std::vector<int4> crl;
  for (int32_t w = 1; w < max_waves; ++w) {
    const int4 x = xs[size_t(w)];
    if (x.z < 0 || (!crl.empty() && crl.back().z == x.z)) continue;
    crl.push_back(x);
  }
  int4* b_crl = reinterpret_cast<int4*>(base + o_crl);
  if (!crl.empty())
    TT_HIP_CHECK(hipMemcpyAsync(b_crl, crl.data(), sizeof(int4) * crl.size(), hipMemcpyHostToDevice, st));
  TT_HIP_CHECK(hipStreamSynchronize(st));
  const int32_t nseg = segs_h[0] + segs_h[1];
  if (nseg >= kUnitMaxY)
    return fail(TENTACO_EUNSUPPORTED, "TTV bands: %d pieces (the band kernel's limit is %d)", nseg,
                kUnitMaxY);
  void* mem2 = nullptr;
  if (hipMalloc(&mem2, align256(sizeof(float) * size_t(std::max(nseg, 1)))) != hipSuccess)
    return fail(TENTACO_ENOMEM, "TTV bands: hipMalloc of the segment sums failed");
  // mark the crossing pieces' sums (the band kernel never writes them)
  if (!crl.empty()) {
    band_mark_kernel<<<grid_of(int64_t(crl.size())), 256, 0, st>>>(b_crl, int32_t(crl.size()),
                                                                   static_cast<float*>(mem2));
    const hipError_t e = hipGetLastError();
    if (e == hipSuccess && hipStreamSynchronize(st) == hipSuccess) {
    } else {
      (void)hipFree(mem2);
      return fail(TENTACO_EHIP, "TTV bands: marking the crossing pieces failed");
    }
  }
  kmem.keep = true;
  P->bmem = mem;
  P->bmem2 = mem2;
  P->b_crd = b_crd;
  P->b_vals = b_vals;
  P->b_flags = b_flags;
  P->b_unit_fid = b_unit;
  P->b_bnd_fid = reinterpret_cast<int32_t*>(base + o_bfid);
  P->b_bnd_val = reinterpret_cast<float*>(base + o_bval);
  P->b_seg = static_cast<float*>(mem2);
  P->b_present = b_pres;
  P->b_prefix = b_pref;
  P->b_fwords = fwords;
  P->b_len = int32_t(len);
  P->b_nseg = nseg;
  P->b_grid = int(given);
  P->b_crossing = b_crl;
  P->b_cross = int32_t(crl.size());
  P->band_w = band_w;
  int32_t u0 = 0, g0 = 0;
  for (int b = 0; b < nb; ++b) {
    P->b_unit0[b] = u0;
    P->b_wg0[b] = g0;
    u0 += units[b];
    g0 += wg[b];
  }
  P->b_unit0[nb] = u0;
  P->b_wg0[nb] = g0;
  P->nbands = nb;
  return TENTACO_OK;
}

}  // namespace

int build_ttv_plan(const CsfDev& B, int32_t cdim, int bands, int64_t max_fibre, TtvPlan* P,
                   hipStream_t st) {
  free_ttv_plan(P);
  P->built = true;
  if (B.order < 2 || B.order > kMaxOrder || B.nnz <= 0 || cdim <= 0 || cdim > kUnitMaxC ||
      B.nodes[B.order - 2] >= kUnitMaxY)
    return TENTACO_OK;
  P->cdim = cdim;
  const int32_t nf = B.nodes[B.order - 2];
  int dev = 0, cus = 0;
  TT_HIP_CHECK(hipGetDevice(&dev));
  TT_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const int lds = cdim <= 4096 ? 4096 : cdim <= 16384 ? 16384 : kTtvLdsMax;
  const int per_cu = size_t(lds) * sizeof(float) <= 80 * 1024 ? 2 : 1;
  const int32_t nunits = int32_t((int64_t(B.nnz) + kUnit - 1) / kUnit);
  int64_t grid = nunits / kUnitWaves;
  grid = std::max<int64_t>(1, std::min<int64_t>(grid, int64_t(std::max(cus, 1)) * per_cu));
  const int32_t max_waves = int32_t(grid) * kUnitWaves;
  const size_t words = size_t(nunits) * (kUnit / 32);
  const size_t o_flags = 0;
  const size_t o_unit = o_flags + align256(words * sizeof(uint32_t));
  const size_t o_bfid = o_unit + align256(size_t(nunits) * sizeof(int32_t));
  const size_t o_bval = o_bfid + align256(size_t(2) * max_waves * sizeof(int32_t));
  const size_t o_bad = o_bval + align256(size_t(2) * max_waves * sizeof(float));
  // the leaf-coordinate histogram that places the window (when c does not
  // fit it): bins of 2^shift coordinates, at most 65536 + 1
  int shift = 5;
  while ((int64_t(cdim) >> shift) + 1 > 65536) ++shift;
  const int64_t nbins = (int64_t(cdim) >> shift) + 1;
  const size_t o_hist = o_bad + 256;
  const size_t total = o_hist + (cdim > lds ? align256(size_t(nbins) * sizeof(uint32_t)) : 0);
  void* mem = nullptr;
  if (hipMalloc(&mem, total) != hipSuccess)
    return fail(TENTACO_ENOMEM, "TTV plan: hipMalloc of %zu bytes failed", total);
  char* base = static_cast<char*>(mem);
  P->mem = mem;
  P->flags = reinterpret_cast<uint32_t*>(base + o_flags);
  P->unit_fid = reinterpret_cast<int32_t*>(base + o_unit);
  P->bnd_fid = reinterpret_cast<int32_t*>(base + o_bfid);
  P->bnd_val = reinterpret_cast<float*>(base + o_bval);
  uint32_t* bad = reinterpret_cast<uint32_t*>(base + o_bad);
  P->nunits = nunits;
  P->max_waves = max_waves;
  P->grid = int(grid);
  P->lds_floats = lds;
  TT_HIP_CHECK(hipMemsetAsync(P->flags, 0, words * sizeof(uint32_t), st));
  TT_HIP_CHECK(hipMemsetAsync(bad, 0, sizeof(uint32_t), st));
  {
    int64_t g = (int64_t(nf) + 255) / 256;
    g = std::max<int64_t>(1, std::min<int64_t>(g, 16384));
    ttv_plan_kernel<<<int(g), 256, 0, st>>>(B.pos[B.order - 1], nf, P->flags, P->unit_fid, bad);
    TT_HIP_CHECK(hipGetLastError());
  }
  P->k0 = 0;
  P->lc = std::min(cdim, lds);
  if (bands == 0 && max_fibre <= kFibreMax && nunits <= kFibreUnits) {
    // whole fibres by the wave, unless there are empty ones to write too
    uint32_t empty = 1;
    TT_HIP_CHECK(hipMemcpyAsync(&empty, bad, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
    TT_HIP_CHECK(hipStreamSynchronize(st));
    if (!empty) {
      P->whole = P->ok = true;
      return TENTACO_OK;
    }
  }
  double window_share = 1.0;  // share of the sampled gathers the window serves
  if (cdim > lds) {
    // the window of `lds` consecutive entries of c that the most nonzeros
    // gather from (first best on ties), from a histogram of leaf coordinates
    const int64_t wb = std::max<int64_t>(1, lds >> shift);
    uint32_t* hist = reinterpret_cast<uint32_t*>(base + o_hist);
    std::vector<uint32_t> h(static_cast<size_t>(nbins));
    hipError_t e = hipMemsetAsync(hist, 0, size_t(nbins) * sizeof(uint32_t), st);
    if (e == hipSuccess) {
      const int32_t step = std::max<int32_t>(1, B.nnz >> 20);
      const int64_t n = (int64_t(B.nnz) + step - 1) / step;
      int64_t g = std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 4096));
      ttv_hist_kernel<<<int(g), 256, 0, st>>>(B.crd[B.order - 1], B.nnz, step, shift, hist);
      e = hipGetLastError();
    }
    if (e == hipSuccess)
      e = hipMemcpyAsync(h.data(), hist, size_t(nbins) * sizeof(uint32_t), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    TT_HIP_CHECK(e);
    uint64_t run = 0, best = 0, all = 0;
    int64_t best_b = 0;
    for (int64_t b = 0; b < nbins; ++b) {
      all += h[size_t(b)];
      run += h[size_t(b)];
      if (b >= wb) run -= h[size_t(b - wb)];
      const int64_t start = std::max<int64_t>(0, b - wb + 1);
      if (run > best) {
        best = run;
        best_b = start;
      }
    }
    P->k0 = int32_t(std::min<int64_t>(best_b << shift, int64_t(cdim) - 1));
    P->lc = int32_t(std::min<int64_t>(lds, int64_t(cdim) - P->k0));
    window_share = all ? double(best) / double(all) : 1.0;
  }
  uint32_t bad_h = 0;
  TT_HIP_CHECK(hipMemcpyAsync(&bad_h, bad, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
  TT_HIP_CHECK(hipStreamSynchronize(st));
  if (bad_h != 0) {
    // empty fibres: rebuild the bitmap and unit table over the non-empty
    // fibres (their starts are distinct), with the map back to output
    // positions and the list of fibres to write as zero
    std::vector<int32_t> pos(static_cast<size_t>(nf) + 1);
    TT_HIP_CHECK(hipMemcpy(pos.data(), B.pos[B.order - 1], sizeof(int32_t) * pos.size(),
                           hipMemcpyDeviceToHost));
    std::vector<int32_t> pos_ne, ne, empty;
    for (int32_t f = 0; f < nf; ++f) {
      if (pos[size_t(f)] < pos[size_t(f) + 1]) {
        pos_ne.push_back(pos[size_t(f)]);
        ne.push_back(f);
      } else if (pos[size_t(f)] == pos[size_t(f) + 1]) {
        empty.push_back(f);
      } else {
        return TENTACO_OK;  // decreasing bounds: not a CSF the kernel can read
      }
    }
    pos_ne.push_back(pos[size_t(nf)]);
    const int32_t nne = int32_t(ne.size());
    const size_t b_pos = align256(pos_ne.size() * sizeof(int32_t));
    const size_t b_ne = align256(ne.size() * sizeof(int32_t) + 4);
    const size_t b_em = align256(empty.size() * sizeof(int32_t) + 4);
    if (hipMalloc(&P->mem2, b_pos + b_ne + b_em) != hipSuccess) {
      P->mem2 = nullptr;
      return fail(TENTACO_ENOMEM, "TTV plan: hipMalloc of the non-empty fibre map failed");
    }
    char* b2 = static_cast<char*>(P->mem2);
    int32_t* d_pos_ne = reinterpret_cast<int32_t*>(b2);
    P->ne_fid = reinterpret_cast<int32_t*>(b2 + b_pos);
    P->empty_ids = reinterpret_cast<int32_t*>(b2 + b_pos + b_ne);
    P->n_empty = int32_t(empty.size());
    TT_HIP_CHECK(hipMemcpy(d_pos_ne, pos_ne.data(), sizeof(int32_t) * pos_ne.size(),
                           hipMemcpyHostToDevice));
    TT_HIP_CHECK(hipMemcpy(P->ne_fid, ne.data(), sizeof(int32_t) * ne.size(), hipMemcpyHostToDevice));
    if (!empty.empty())
      TT_HIP_CHECK(hipMemcpy(P->empty_ids, empty.data(), sizeof(int32_t) * empty.size(),
                             hipMemcpyHostToDevice));
    TT_HIP_CHECK(hipMemsetAsync(P->flags, 0, words * sizeof(uint32_t), st));
    int64_t g = (int64_t(nne) + 255) / 256;
    g = std::max<int64_t>(1, std::min<int64_t>(g, 16384));
    ttv_plan_kernel<<<int(g), 256, 0, st>>>(d_pos_ne, nne, P->flags, P->unit_fid, bad);
    TT_HIP_CHECK(hipGetLastError());
    TT_HIP_CHECK(hipStreamSynchronize(st));
  }
  P->ok = true;
  // the banded layout: forced (bands >= 2), or picked when c does not fit
  // one window and the best window would serve under 3/4 of the gathers
  int nb = 0;
  if (bands >= 2) {
    nb = std::min(bands, kMaxBands);
    while (nb <= kMaxBands && (int64_t(cdim) + nb - 1) / nb > kTtvLdsMax - 1) ++nb;
  } else if (bands == 0 && cdim > kTtvLdsMax && window_share < 0.75) {
    nb = int((int64_t(cdim) + kTtvLdsMax - 2) / (kTtvLdsMax - 1));
  }
  if (nb >= 2 && nb <= kMaxBands && nb <= cdim) {
    const int32_t band_w = int32_t((int64_t(cdim) + nb - 1) / nb);
    const int inst = band_inst(band_w);
    const int per = size_t(inst) * sizeof(float) <= 80 * 1024 ? 2 : 1;
    // an optimisation: when it cannot be built (memory), the one-window
    // plan serves (tentaco_csf_ttv_layout reports which)
    if (build_ttv_bands(B, nb, band_w, std::max(cus, 1) * per, P, st) != TENTACO_OK) {
      (void)hipStreamSynchronize(st);
      clear_error();
    }
  }
  return TENTACO_OK;
}

int launch_ttv_units(const CsfDev& B, const TtvPlan& P, const float* c, float* y,
                     hipStream_t st) {
  if (!P.ok) return fail(TENTACO_EINVAL, "TTV unit kernel: plan does not apply");
  if (P.nbands >= 2) {
    switch (band_inst(P.band_w)) {
      case 4096: return launch_bands_typed<4096>(B, P, c, y, st);
      case 16384: return launch_bands_typed<16384>(B, P, c, y, st);
      default: return launch_bands_typed<kTtvLdsMax>(B, P, c, y, st);
    }
  }
  if (P.whole) {
    ktimer_begin(st);
    ttv_unit_kernel<<<(P.nunits + kFibreWaves - 1) / kFibreWaves, 64 * kFibreWaves, 0, st>>>(
        B.crd[B.order - 1], B.vals, P.flags, P.unit_fid, B.pos[B.order - 1], c, y,
        B.nodes[B.order - 2], B.nnz, P.nunits);
    TT_HIP_CHECK(hipGetLastError());
    ktimer_end(st, "ttv_unit_kernel");
    return TENTACO_OK;
  }
  switch (P.lds_floats) {
    case 4096: return launch_units_typed<4096>(B, P, c, y, st);
    case 16384: return launch_units_typed<16384>(B, P, c, y, st);
    case kTtvLdsMax: return launch_units_typed<kTtvLdsMax>(B, P, c, y, st);
    default: return fail(TENTACO_EINVAL, "TTV unit kernel: bad LDS instance %d", P.lds_floats);
  }
}

}  // namespace tt
