// Register-resident factor-row fragments for wave64 MTTKRP kernels.
//
// A factor row of rank R is spread over LPR consecutive lanes of a wavefront
// ("row group"); each lane holds NV float4 fragments, so one
// global_load_dwordx4 per fragment reads LPR*16 contiguous bytes of the row.
// The template argument names the layout:
//   R > 0   exactly rank R: fragment j of lane c covers columns
//           (j*LPR + c)*4 .. +3 (R=16 -> 4 lanes, R=32 -> 8 lanes, R=64 -> 16
//           lanes, R=128 -> 16 lanes x 2 fragments);
//   R < 0   any runtime rank 4 <= Rr <= -R on rank -R's lanes: a fragment
//           that would pass the row's end is moved back to columns
//           Rr-4 .. Rr-1. It then repeats columns of the lane before it
//           (computed from the same data in the same order, so the copies
//           are equal): stores write them twice, atomics only the columns a
//           lane owns. No load is predicated and none leaves the row, at
//           4-byte alignment;
//   R == 0  ranks 1..3: one column per lane of 4.
// Ranks 4..256 used to share one scalar layout of 16 column-predicated loads
// per lane and row: a 5M-nonzero 3-mode MTTKRP at rank 50 took 598 us with it
// and 229 us with the float4 layout (the walk of that time).
#pragma once

#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>
#include <type_traits>

namespace tt {

// The pointer as one to global memory. Loads through a pointer that was itself
// read from memory (the task and job tables) are flat loads otherwise, whose
// waits also drain the LDS reads in flight.
template <class T>
__device__ __forceinline__ T* global_ptr(T* p) {
  typedef __attribute__((address_space(1))) T* G;
  return (T*)reinterpret_cast<G>(reinterpret_cast<uintptr_t>(p));
}

// Orders the wave's LDS accesses: what its lanes wrote before is read after.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Inclusive sum over the lanes up to this one (DPP row shifts, then the rows'
// last lanes broadcast to the next rows).
__device__ __forceinline__ int32_t wave_scan_add(int32_t x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
  return x;
}

constexpr int kMaxRankAny = 256;

// Where a product of factor rows underflows, a value times leaf row up to this
// makes of what is lost (2^-150) no more than 2^-140.
constexpr float kSafe = 1024.f;

template <int R>
struct Lay {
  static constexpr int K = R < 0 ? -R : R;
  static_assert(K == 16 || K == 32 || K == 64 || K == 128 || (R < 0 && K == kMaxRankAny),
                "rank layouts");
  static constexpr int LPR = (K / 4 >= 16) ? 16 : K / 4;
  static constexpr int NV = K / (4 * LPR);
  static constexpr int kMaxRank = K;
  using V = float4;
};

template <>
struct Lay<0> {
  static constexpr int LPR = 4;
  static constexpr int NV = 1;
  static constexpr int kMaxRank = 4;
  using V = float;
};

// f(std::integral_constant<int, layout>) for the layout of rank R in
// 1..kMaxRankAny.
template <class Fn>
auto with_rank_layout(int R, Fn&& f) {
  switch (R) {
    case 16: return f(std::integral_constant<int, 16>());
    case 32: return f(std::integral_constant<int, 32>());
    case 64: return f(std::integral_constant<int, 64>());
    case 128: return f(std::integral_constant<int, 128>());
  }
  if (R < 4) return f(std::integral_constant<int, 0>());
  if (R < 16) return f(std::integral_constant<int, -16>());
  if (R < 32) return f(std::integral_constant<int, -32>());
  if (R < 64) return f(std::integral_constant<int, -64>());
  if (R < 128) return f(std::integral_constant<int, -128>());
  return f(std::integral_constant<int, -256>());
}

// Four floats at any 4-byte address (one dwordx4 access on gfx950).
struct __attribute__((packed, aligned(4))) float4u {
  float x, y, z, w;
};
__device__ __forceinline__ float4 load4(const float* p) {
  const float4u v = *reinterpret_cast<const float4u*>(p);
  return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ void store4(float* p, const float4& v) {
  *reinterpret_cast<float4u*>(p) = float4u{v.x, v.y, v.z, v.w};
}

template <int R>
struct Row {
  using L = Lay<R>;
  using V = typename L::V;
  static constexpr int NV = L::NV;
  static constexpr int LPR = L::LPR;

  // Fragment j of lane c in the layout's full width (LDS rows of kMaxRank).
  __device__ __forceinline__ static int slot(int j, int c) {
    if constexpr (R == 0) return c;
    else return (j * LPR + c) * 4;
  }
  // Its first column in a row of rank Rr.
  __device__ __forceinline__ static int col(int j, int c, int Rr) {
    if constexpr (R < 0) return min(slot(j, c), Rr - 4);
    else return slot(j, c);
  }

  // Where column k is in such a row.
  __device__ __forceinline__ static int slot_of(int k, int Rr) {
    if constexpr (R < 0) return (k & ~3) + (k - min(k & ~3, Rr - 4));
    else return k;
  }

  // base[slot] = a, a += base[slot]: a row of kMaxRank floats, 16-byte
  // aligned (LDS).
  __device__ __forceinline__ static void put(float* base, int c, const V (&a)[NV]) {
#pragma unroll
    for (int j = 0; j < NV; ++j) *reinterpret_cast<V*>(base + slot(j, c)) = a[j];
  }
  __device__ __forceinline__ static void get(const float* base, int c, V (&a)[NV]) {
#pragma unroll
    for (int j = 0; j < NV; ++j) a[j] = *reinterpret_cast<const V*>(base + slot(j, c));
  }

  __device__ __forceinline__ static void zero(V (&a)[NV]) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if constexpr (R == 0) a[j] = 0.f;
      else a[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }

  // d = M[row, this lane's columns]; Rr is the runtime rank (== R when R>0).
  __device__ __forceinline__ static void load(V (&d)[NV],
                                              const float* __restrict__ M,
                                              int64_t row, int c, int Rr) {
    if constexpr (R == 0) {
      d[0] = (c < Rr) ? M[row * Rr + c] : 0.f;
    } else if constexpr (R < 0) {
      const float* p = M + row * Rr;
#pragma unroll
      for (int j = 0; j < NV; ++j) d[j] = load4(p + col(j, c, Rr));
    } else {
      const float* p = M + row * R;
#pragma unroll
      for (int j = 0; j < NV; ++j)
        d[j] = *reinterpret_cast<const float4*>(p + col(j, c, Rr));
    }
  }

  // a *= s
  __device__ __forceinline__ static void scale(V (&a)[NV], float s) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if constexpr (R == 0) {
        a[j] *= s;
      } else {
        a[j].x *= s;
        a[j].y *= s;
        a[j].z *= s;
        a[j].w *= s;
      }
    }
  }

  // The smallest and largest magnitude of a's columns, with what least and most
  // hold.
  __device__ __forceinline__ static void extent(const V (&a)[NV], int c, int Rr, float& least,
                                                float& most) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if constexpr (R == 0) {
        if (c < Rr) least = fminf(least, fabsf(a[j]));
        most = fmaxf(most, fabsf(a[j]));
      } else {
        least = fminf(fminf(least, fabsf(a[j].x)), fabsf(a[j].y));
        least = fminf(fminf(least, fabsf(a[j].z)), fabsf(a[j].w));
        most = fmaxf(fmaxf(most, fabsf(a[j].x)), fabsf(a[j].y));
        most = fmaxf(fmaxf(most, fabsf(a[j].z)), fabsf(a[j].w));
      }
    }
  }

  // The largest magnitude of a's columns and m.
  __device__ __forceinline__ static float peak(const V (&a)[NV], float m) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if constexpr (R == 0) {
        m = fmaxf(m, fabsf(a[j]));
      } else {
        m = fmaxf(fmaxf(m, fabsf(a[j].x)), fabsf(a[j].y));
        m = fmaxf(fmaxf(m, fabsf(a[j].z)), fabsf(a[j].w));
      }
    }
    return m;
  }

  // a = a (.) y; whether a column left the normal numbers that neither a nor y
  // has as 0.
  __device__ __forceinline__ static bool hmul_lost(V (&a)[NV], const V (&y)[NV]) {
    bool lost = false;
    auto mul = [&](float& x, float z) {
      const bool zero = x == 0.f || z == 0.f;
      x *= z;
      lost = lost || !(zero || (fabsf(x) >= FLT_MIN && fabsf(x) <= FLT_MAX));
    };
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if constexpr (R == 0) {
        mul(a[j], y[j]);
      } else {
        mul(a[j].x, y[j].x);
        mul(a[j].y, y[j].y);
        mul(a[j].z, y[j].z);
        mul(a[j].w, y[j].w);
      }
    }
    return lost;
  }

  // a += s * d
  __device__ __forceinline__ static void axpy(V (&a)[NV], float s,
                                              const V (&d)[NV]) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if constexpr (R == 0) {
        a[j] = fmaf(s, d[j], a[j]);
      } else {
        a[j].x = fmaf(s, d[j].x, a[j].x);
        a[j].y = fmaf(s, d[j].y, a[j].y);
        a[j].z = fmaf(s, d[j].z, a[j].z);
        a[j].w = fmaf(s, d[j].w, a[j].w);
      }
    }
  }

  // a += x (.) y   (Hadamard product accumulate)
  __device__ __forceinline__ static void hfma(V (&a)[NV], const V (&x)[NV],
                                              const V (&y)[NV]) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if constexpr (R == 0) {
        a[j] = fmaf(x[j], y[j], a[j]);
      } else {
        a[j].x = fmaf(x[j].x, y[j].x, a[j].x);
        a[j].y = fmaf(x[j].y, y[j].y, a[j].y);
        a[j].z = fmaf(x[j].z, y[j].z, a[j].z);
        a[j].w = fmaf(x[j].w, y[j].w, a[j].w);
      }
    }
  }

  // axpy and hfma where ok, else a as it is, whatever the operands (weight 0
  // would turn infinities and NaN of an idle lane's row into NaN). Selects, not a
  // branch: behind one, the compiler moves the operands' loads to it, each waited
  // for by itself (300k nonzeros in 40000 slices, 256 threads a slice: 84 us a
  // call against 42).
  __device__ __forceinline__ static void axpy_if(bool ok, V (&a)[NV], float s, const V (&d)[NV]) {
    V t[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) t[j] = a[j];
    axpy(t, s, d);
    select(ok, a, t);
  }
  __device__ __forceinline__ static void hfma_if(bool ok, V (&a)[NV], const V (&x)[NV],
                                                 const V (&y)[NV]) {
    V t[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) t[j] = a[j];
    hfma(t, x, y);
    select(ok, a, t);
  }
  __device__ __forceinline__ static void select(bool ok, V (&a)[NV], const V (&t)[NV]) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if constexpr (R == 0) {
        a[j] = ok ? t[j] : a[j];
      } else {
        a[j].x = ok ? t[j].x : a[j].x;
        a[j].y = ok ? t[j].y : a[j].y;
        a[j].z = ok ? t[j].z : a[j].z;
        a[j].w = ok ? t[j].w : a[j].w;
      }
    }
  }

  // a = a (.) y
  __device__ __forceinline__ static void hmul(V (&a)[NV], const V (&y)[NV]) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if constexpr (R == 0) {
        a[j] = a[j] * y[j];
      } else {
        a[j].x *= y[j].x;
        a[j].y *= y[j].y;
        a[j].z *= y[j].z;
        a[j].w *= y[j].w;
      }
    }
  }

  __device__ __forceinline__ static void add(V (&a)[NV], const V (&b)[NV]) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if constexpr (R == 0) {
        a[j] += b[j];
      } else {
        a[j].x += b[j].x;
        a[j].y += b[j].y;
        a[j].z += b[j].z;
        a[j].w += b[j].w;
      }
    }
  }

  // Sums in FP64, a lane's 4 (layout 0: 1) columns per fragment.
  static constexpr int NC = R == 0 ? 1 : 4;
  using D = double[NV * NC];
  __device__ __forceinline__ static void add(D& a, const V (&b)[NV]) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if constexpr (R == 0) {
        a[j] += double(b[j]);
      } else {
        a[4 * j] += double(b[j].x);
        a[4 * j + 1] += double(b[j].y);
        a[4 * j + 2] += double(b[j].z);
        a[4 * j + 3] += double(b[j].w);
      }
    }
  }
  __device__ __forceinline__ static void narrow(V (&a)[NV], const V (&b)[NV]) {
#pragma unroll
    for (int j = 0; j < NV; ++j) a[j] = b[j];
  }
  __device__ __forceinline__ static void narrow(V (&a)[NV], const D& b) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if constexpr (R == 0) a[j] = float(b[j]);
      else a[j] = make_float4(float(b[4 * j]), float(b[4 * j + 1]), float(b[4 * j + 2]), float(b[4 * j + 3]));
    }
  }

  __device__ __forceinline__ static void store(float* __restrict__ A,
                                               int64_t row, int c, int Rr,
                                               const V (&a)[NV]) {
    if constexpr (R == 0) {
      if (c < Rr) A[row * Rr + c] = a[0];
    } else if constexpr (R < 0) {
      float* p = A + row * Rr;
#pragma unroll
      for (int j = 0; j < NV; ++j)
        if (slot(j, c) < Rr) store4(p + col(j, c, Rr), a[j]);
    } else {
      float* p = A + row * R;
#pragma unroll
      for (int j = 0; j < NV; ++j)
        *reinterpret_cast<float4*>(p + col(j, c, Rr)) = a[j];
    }
  }

  // Device-scope float atomics (global_atomic_add_f32) on coarse-grained
  // memory: correct across XCDs, no CAS loop.
  __device__ __forceinline__ static void atomic_add(float* __restrict__ A,
                                                    int64_t row, int c, int Rr,
                                                    const V (&a)[NV]) {
    if constexpr (R == 0) {
      if (c < Rr) unsafeAtomicAdd(A + row * Rr + c, a[0]);
    } else if constexpr (R < 0) {
      float* p = A + row * Rr;
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const int own = slot(j, c);  // columns from here on are this lane's
        const int k = col(j, c, Rr);
        if (k >= own) unsafeAtomicAdd(p + k, a[j].x);
        if (k + 1 >= own) unsafeAtomicAdd(p + k + 1, a[j].y);
        if (k + 2 >= own) unsafeAtomicAdd(p + k + 2, a[j].z);
        if (k + 3 >= own) unsafeAtomicAdd(p + k + 3, a[j].w);
      }
    } else {
      float* p = A + row * R;
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        float* q = p + col(j, c, Rr);
        unsafeAtomicAdd(q + 0, a[j].x);
        unsafeAtomicAdd(q + 1, a[j].y);
        unsafeAtomicAdd(q + 2, a[j].z);
        unsafeAtomicAdd(q + 3, a[j].w);
      }
    }
  }

  // FP64 row output (the edge-serial family's accumulation buffer).
  __device__ __forceinline__ static void store_f64(double* __restrict__ W, int64_t row, int c,
                                                   int Rr, const V (&a)[NV]) {
    if constexpr (R == 0) {
      if (c < Rr) W[row * Rr + c] = double(a[0]);
    } else if constexpr (R < 0) {
      double* p = W + row * Rr;
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        if (slot(j, c) >= Rr) continue;
        double* q = p + col(j, c, Rr);
        q[0] = double(a[j].x);
        q[1] = double(a[j].y);
        q[2] = double(a[j].z);
        q[3] = double(a[j].w);
      }
    } else {
      double* p = W + row * R;
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        double2* q = reinterpret_cast<double2*>(p + col(j, c, Rr));
        q[0] = make_double2(double(a[j].x), double(a[j].y));
        q[1] = make_double2(double(a[j].z), double(a[j].w));
      }
    }
  }

  // Sum a over the row groups of a wavefront (xor butterfly over the lane
  // bits above log2(LPR)); every lane ends with the wave total of its slots.
  __device__ __forceinline__ static void wave_sum(V (&a)[NV]) {
#pragma unroll
    for (int off = LPR; off < 64; off <<= 1) {
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        if constexpr (R == 0) {
          a[j] += __shfl_xor(a[j], off);
        } else {
          a[j].x += __shfl_xor(a[j].x, off);
          a[j].y += __shfl_xor(a[j].y, off);
          a[j].z += __shfl_xor(a[j].z, off);
          a[j].w += __shfl_xor(a[j].w, off);
        }
      }
    }
  }
};

// Largest x in [lo, hi] with a[x] <= key; requires a[lo] <= key. With runs of
// equal values (empty nodes) this is the last node that starts at or before
// key, i.e. the node that contains key (upper-bound semantics; the
// reference's taco_binarySearchBefore may return any of the equal slots).
__device__ __forceinline__ int32_t search_le(const int32_t* __restrict__ a,
                                             int32_t lo, int32_t hi,
                                             int32_t key) {
  while (lo < hi) {
    const int32_t mid = lo + ((hi - lo + 1) >> 1);
    if (a[mid] <= key) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

}  // namespace tt
