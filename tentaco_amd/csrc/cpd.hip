// CP-ALS around the batched MTTKRP: the caller that splatt_cpd_als stands in
// for in the reference (ds.h:395), for many tensors at once.
//
// One ALS sweep updates every factor of every tensor in mode order
// m = 0 .. 4. Mode step m runs
//   1. one batched, graph-replayed MTTKRP over every tensor with order > m
//      (M_t = B_t x_{k != m} A_t,k, from the tensor's mode-m CSF),
//   2. per tensor: V = Hadamard product of the other modes' Grams, its
//      inverse by Cholesky (FP64, in LDS), A_t,m = M_t V^-1,
//   3. column normalisation (2-norm on the first sweep, max(1, max |a|)
//      afterwards) into lambda_t, and the new Gram A^T A.
// Steps 2-3 read and write the factor rows twice: one fused pass computes
// A = M V^-1 and per-block partials of A^T A, of the column max and of the
// fit's inner product; a per-job kernel reduces them (the 2-norms are the
// Gram diagonal, and the normalised Gram is (A^T A) ./ (lambda lambda^T));
// a last pass divides A by lambda.
// Row-parallel kernels cover every tensor of a step in one launch through a
// job table; their reductions write per-block partials that a second kernel
// sums in block order, so results do not depend on scheduling. The fit
// after a sweep is 1 - ||X - model|| / ||X|| with
// ||X - model||^2 = ||X||^2 + lambda^T (*_k G_k) lambda - 2 <X, model> and
// <X, model> = sum_r lambda_r sum_i M_N[i,r] A_N[i,r] for the last mode N.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

#include "handle.h"
#include "host_copy.h"
#include "internal.h"
#include "rowops.h"

namespace tt {
namespace {

constexpr int kMaxR = 64;
constexpr int kApplyRows = 64;    // rows per block of the apply / scale kernels
constexpr int kStatRows = 2048;   // rows per block of the reduction kernels
// Blocks of a mode step's fused update: the rows per block are chosen so that
// about 256 cover the chip without many partials to sum, and for long modes up
// to 1024, four a CU, to keep enough bytes in flight (64 tensors, 9.3M rows and
// less per step, R = 32: 689 and 413 us a step, the finish 10 and 18).
constexpr int kUpdBlocks = 256, kUpdBlocksMax = 1024;
constexpr int kUpdUnit = 128;     // rows per block: a multiple of this

struct CpdJob {
  const float* M = nullptr;  // MTTKRP result, rows x R
  float* A = nullptr;        // factor being updated, rows x R
  float* G = nullptr;        // its Gram, R x R
  float* lam = nullptr;      // lambda, R
  float* Vinv = nullptr;     // R x R scratch
  const float* Gk[kMaxOrder - 1] = {};
  int nG = 0;
  double* inner = nullptr;   // <M, A diag(lambda)> of this update, when the fit needs it
  int32_t rows = 0;
  int32_t ablk0 = 0, nablk = 0;  // apply blocks (kApplyRows rows each)
  int32_t sblk0 = 0, nsblk = 0;  // reduction blocks (kStatRows rows each)
  int32_t ublk0 = 0, nublk = 0;  // update blocks (urows rows each)
  int32_t urows = 0;
};

// Sum over the wave, in a fixed order; every lane gets it.
__device__ __forceinline__ double wave_sum_f64(double x) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) x += __shfl_xor(x, o);
  return x;
}

__device__ __forceinline__ int find_job(const int32_t* __restrict__ off, int n, int32_t blk) {
  int lo = 0, hi = n - 1;  // largest j with off[j] <= blk
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (off[mid] <= blk) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// V = Hadamard product of the job's Grams; Vinv = V^-1 by Gauss-Jordan
// elimination in FP64 (V is symmetric positive semidefinite, so the diagonal
// is the pivot). A pivot at or below 1e-12 times the largest diagonal (a
// rank-deficient V) is lifted to that value, which keeps the solve finite; the
// pivots are those of a Cholesky factorisation.
//
// A chain of R dependent steps bounds it, so a step is one barrier: every
// thread keeps EPT entries of a row in registers, the owners of the step's
// row and column publish them in one of two LDS buffers in turn, and every
// thread eliminates its own entries. One workgroup per job, R*R / EPT threads.
// (A Cholesky factorisation with a thread per pivot and a forward substitution
// per column took 69 us at R = 32, this 18 us.)
template <int R>
__global__ __launch_bounds__(R * R / (R == 16 ? 1 : 4)) void hadamard_inverse_kernel(
    const CpdJob* __restrict__ jobs) {
  constexpr int EPT = R == 16 ? 1 : 4;
  __shared__ double rowk[2][R], colk[2][R];
  __shared__ double diag[R];
  const CpdJob& J = jobs[blockIdx.x];
  const int i = int(threadIdx.x) / (R / EPT), j0 = int(threadIdx.x) % (R / EPT) * EPT;
  double v[EPT];
#pragma unroll
  for (int u = 0; u < EPT; ++u) {
    v[u] = 1.0;
    for (int g = 0; g < J.nG; ++g) v[u] *= double(J.Gk[g][i * R + j0 + u]);
    if (i == j0 + u) diag[i] = v[u];
  }
  __syncthreads();
  double dmax = 0.0;
  for (int q = 0; q < R; ++q) dmax = fmax(dmax, diag[q]);
  const double least = 1e-12 * (dmax > 0.0 ? dmax : 1.0);
  for (int k = 0; k < R; ++k) {
    double* rk = rowk[k & 1];
    double* ck = colk[k & 1];
    if (i == k) {
#pragma unroll
      for (int u = 0; u < EPT; ++u) rk[j0 + u] = v[u];
    }
#pragma unroll
    for (int u = 0; u < EPT; ++u)
      if (j0 + u == k) ck[i] = v[u];
    __syncthreads();  // (the other buffer's readers are past the last barrier)
    const double d = rk[k];
    const double p = 1.0 / (d > least ? d : least);
    const double f = ck[i] * p;
#pragma unroll
    for (int u = 0; u < EPT; ++u) {
      const int j = j0 + u;
      if (i == k) v[u] = j == k ? p : v[u] * p;
      else v[u] = j == k ? -f : v[u] - f * rk[j];
    }
  }
#pragma unroll
  for (int u = 0; u < EPT; ++u) J.Vinv[i * R + j0 + u] = float(v[u]);
}

// Gram partials: part[block][i*R + j] = sum over the block's rows of
// A[r,i] A[r,j] (upper triangle computed, mirrored), FP64 accumulation.
__global__ __launch_bounds__(256) void gram_partial_kernel(const CpdJob* __restrict__ jobs,
                                                           const int32_t* __restrict__ sblk0,
                                                           int njobs, int R,
                                                           double* __restrict__ part) {
  constexpr int kTile = 32;
  __shared__ float As[kTile][kMaxR + 1];
  const int j = find_job(sblk0, njobs, blockIdx.x);
  const CpdJob& J = jobs[j];
  const int32_t r0 = (int32_t(blockIdx.x) - J.sblk0) * kStatRows;
  const int32_t r1 = min(r0 + kStatRows, J.rows);
  constexpr int kPer = (kMaxR * kMaxR + 255) / 256;
  double acc[kPer];
#pragma unroll
  for (int q = 0; q < kPer; ++q) acc[q] = 0.0;
  for (int32_t t0 = r0; t0 < r1; t0 += kTile) {
    const int nt = min(kTile, r1 - t0);
    __syncthreads();
    for (int e = threadIdx.x; e < kTile * R; e += blockDim.x) {
      const int r = e / R, c = e % R;
      As[r][c] = r < nt ? J.A[int64_t(t0 + r) * R + c] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
      const int e = threadIdx.x + q * 256;
      if (e >= R * R) break;
      const int a = e / R, b = e % R;
      if (a > b) continue;
      double s = 0.0;
      for (int r = 0; r < kTile; ++r) s += double(As[r][a]) * double(As[r][b]);
      acc[q] += s;
    }
  }
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int e = threadIdx.x + q * 256;
    if (e >= R * R) break;
    const int a = e / R, b = e % R;
    if (a > b) continue;
    part[int64_t(blockIdx.x) * R * R + a * R + b] = acc[q];
    part[int64_t(blockIdx.x) * R * R + b * R + a] = acc[q];
  }
}

__global__ __launch_bounds__(256) void gram_reduce_kernel(const CpdJob* __restrict__ jobs, int R,
                                                          const double* __restrict__ part) {
  const CpdJob& J = jobs[blockIdx.x];
  for (int e = threadIdx.x; e < R * R; e += blockDim.x) {
    double s = 0.0;
    for (int b = 0; b < J.nsblk; ++b) s += part[int64_t(J.sblk0 + b) * R * R + e];
    J.G[e] = float(s);
  }
}

// Pass 1 of a mode step, urows rows of one job per block, in tiles of
// TR = 1024 / R rows (one float4 of M per thread per tile):
//   A = M V^-1, written unnormalised;
//   per-block FP64 partials of A^T A (FP32 within a tile), of the column
//   max |a|, and of <M, A> (the fit's inner product, since the stored factor
//   is A / lambda and the model carries lambda).
// Partials go to pg[block][R*R], pm[block][R], pi[block]; finish_kernel sums
// them in block order, so the results do not depend on scheduling.
template <int R>
__global__ __launch_bounds__(256) void update_kernel(const CpdJob* __restrict__ jobs,
                                                     const int32_t* __restrict__ ublk0, int njobs,
                                                     double* __restrict__ pg,
                                                     double* __restrict__ pm,
                                                     double* __restrict__ pi) {
  constexpr int Q = R / 4;           // float4 quads per row
  constexpr int TR = 256 / Q;        // rows per tile
  constexpr int EPT = R * R / 256 > 0 ? R * R / 256 : 1;  // Gram entries per thread
  __shared__ __align__(16) float Vs[R][R];
  __shared__ float Ms[TR][R + 1];
  __shared__ float As[TR][R + 1];
  __shared__ double red[4];
  const int j = find_job(ublk0, njobs, blockIdx.x);
  const CpdJob& J = jobs[j];
  const int32_t r0 = (int32_t(blockIdx.x) - J.ublk0) * J.urows;
  const int32_t r1 = min(r0 + J.urows, J.rows);
  for (int e = threadIdx.x; e < R * R; e += 256) Vs[e / R][e % R] = J.Vinv[e];
  const int rr = int(threadIdx.x) / Q, q = int(threadIdx.x) % Q;
  double g[EPT];
#pragma unroll
  for (int k = 0; k < EPT; ++k) g[k] = 0.0;
  float cmax[4] = {0.f, 0.f, 0.f, 0.f};
  double inner = 0.0;
  for (int32_t t0 = r0; t0 < r1; t0 += TR) {
    const int32_t row = t0 + rr;
    const bool ok = row < r1;
    __syncthreads();  // the previous tile's LDS reads are done (and Vs is loaded)
    {
      float4 m4 = make_float4(0.f, 0.f, 0.f, 0.f);
      if (ok) m4 = *reinterpret_cast<const float4*>(J.M + int64_t(row) * R + 4 * q);
      Ms[rr][4 * q] = m4.x;
      Ms[rr][4 * q + 1] = m4.y;
      Ms[rr][4 * q + 2] = m4.z;
      Ms[rr][4 * q + 3] = m4.w;
    }
    __syncthreads();
    float o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int k = 0; k < R; ++k) {
      const float mk = Ms[rr][k];
      const float4 v = *reinterpret_cast<const float4*>(&Vs[k][4 * q]);
      o[0] = fmaf(mk, v.x, o[0]);
      o[1] = fmaf(mk, v.y, o[1]);
      o[2] = fmaf(mk, v.z, o[2]);
      o[3] = fmaf(mk, v.w, o[3]);
    }
    if (ok) {
      *reinterpret_cast<float4*>(J.A + int64_t(row) * R + 4 * q) = make_float4(o[0], o[1], o[2], o[3]);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        cmax[u] = fmaxf(cmax[u], fabsf(o[u]));
        inner += double(Ms[rr][4 * q + u]) * double(o[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) As[rr][4 * q + u] = ok ? o[u] : 0.f;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
      const int e = int(threadIdx.x) + 256 * k;
      if (e < R * R) {
        const int a = e / R, b = e % R;
        float sf = 0.f;
#pragma unroll 8
        for (int r = 0; r < TR; ++r) sf = fmaf(As[r][a], As[r][b], sf);
        g[k] += double(sf);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < EPT; ++k) {
    const int e = int(threadIdx.x) + 256 * k;
    if (e < R * R) pg[int64_t(blockIdx.x) * R * R + e] = g[k];
  }
  // column max over the block: per column, the TR row threads in order
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 4; ++u) As[rr][4 * q + u] = cmax[u];
  inner = wave_sum_f64(inner);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = inner;
  __syncthreads();
  if (threadIdx.x < R) {
    float mx = 0.f;
    for (int r = 0; r < TR; ++r) mx = fmaxf(mx, As[r][threadIdx.x]);
    pm[int64_t(blockIdx.x) * R + threadIdx.x] = double(mx);
  }
  if (threadIdx.x == 0) pi[blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
}

// update_kernel for R = 32 on the matrix cores. Each wave takes 32-row tiles
// (tile w + 4k of the block) on its own, the next tile's M loaded while this
// one is computed; per tile:
//   A = M V^-1 as 16 v_mfma_f32_32x32x2f32 steps (operands from LDS: M tile
//   and V^-1), then A^T A as 16 more on the A tile staged in LDS; the Gram
//   accumulators are added into FP64 registers after every tile.
// Accumulator layout of the 32x32 result: lane l holds column l % 32 and,
// in register r, row (r % 4) + 4 * (l / 32) + 8 * (r / 4). Operand layout:
// lane l supplies A[l % 32][k = l / 32] and B[k = l / 32][l % 32] for the
// step's two k values.
typedef float f32x16 __attribute__((ext_vector_type(16)));

__global__ __launch_bounds__(256) void update32_mfma_kernel(const CpdJob* __restrict__ jobs,
                                                            const int32_t* __restrict__ ublk0,
                                                            int njobs, double* __restrict__ pg,
                                                            double* __restrict__ pm,
                                                            double* __restrict__ pi) {
  constexpr int R = 32;
  constexpr int W = 4;  // waves per block
  __shared__ float Vs[R][R + 1];
  __shared__ float Ts[W][32][R + 1];  // per wave: the M tile, then the A tile
  __shared__ double Gs[R][R];         // cross-wave Gram reduction
  __shared__ float Cm[W][64];
  __shared__ double Is[W];
  const int j = find_job(ublk0, njobs, blockIdx.x);
  const CpdJob& J = jobs[j];
  const int32_t r0 = (int32_t(blockIdx.x) - J.ublk0) * J.urows;
  const int32_t r1 = min(r0 + J.urows, J.rows);
  const int lane = int(threadIdx.x) & 63;
  const int w = int(threadIdx.x) >> 6;
  const int col = lane & 31, half = lane >> 5;
  const float* __restrict__ M = global_ptr(J.M);
  float* __restrict__ A = global_ptr(J.A);
  const float* __restrict__ Vinv = global_ptr(J.Vinv);
  for (int e = threadIdx.x; e < R * R; e += 256) Vs[e / R][e % R] = Vinv[e];
  double gd[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) gd[r] = 0.0;
  float cmax = 0.f;
  double inner = 0.0;
  // M tile: 32 rows x 32 floats, float4 per lane, 4 passes
  float4 mt[4];
  auto load_tile = [&](int32_t t0) {
#pragma unroll
    for (int pss = 0; pss < 4; ++pss) {
      const int e = pss * 64 + lane;  // float4 index in the tile
      const int32_t row = t0 + (e >> 3);
      mt[pss] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (row < r1) mt[pss] = *reinterpret_cast<const float4*>(M + int64_t(row) * R + 4 * (e & 7));
    }
  };
  load_tile(r0 + w * 32);
  __syncthreads();  // Vs is loaded
  for (int32_t t0 = r0 + w * 32; t0 < r1; t0 += W * 32) {
#pragma unroll
    for (int pss = 0; pss < 4; ++pss) {
      const int e = pss * 64 + lane;
      float* row = &Ts[w][e >> 3][4 * (e & 7)];
      row[0] = mt[pss].x;
      row[1] = mt[pss].y;
      row[2] = mt[pss].z;
      row[3] = mt[pss].w;
    }
    wave_lds_sync();
    if (t0 + W * 32 < r1) load_tile(t0 + W * 32);
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (int s = 0; s < R / 2; ++s) {
      const float a = Ts[w][col][2 * s + half];
      const float b = Vs[2 * s + half][col];
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
    }
    // store A, column max, <M, A>; then stage A for the Gram
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int i = (r & 3) + 4 * half + 8 * (r >> 2);
      if (t0 + i < r1) {
        A[int64_t(t0 + i) * R + col] = acc[r];
        cmax = fmaxf(cmax, fabsf(acc[r]));
        inner += double(Ts[w][i][col]) * double(acc[r]);
      }
    }
    wave_lds_sync();  // every lane has read its M values
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int i = (r & 3) + 4 * half + 8 * (r >> 2);
      Ts[w][i][col] = (t0 + i < r1) ? acc[r] : 0.f;
    }
    wave_lds_sync();
    f32x16 g;
#pragma unroll
    for (int r = 0; r < 16; ++r) g[r] = 0.f;
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      const float v = Ts[w][2 * s + half][col];
      g = __builtin_amdgcn_mfma_f32_32x32x2f32(v, v, g, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) gd[r] += double(g[r]);
    wave_lds_sync();  // the tile's readers are done
  }
  // the block's partials, waves summed in order
  for (int ww = 0; ww < W; ++ww) {
    __syncthreads();
    if (w == ww) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = (r & 3) + 4 * half + 8 * (r >> 2);
        Gs[i][col] = (ww == 0 ? 0.0 : Gs[i][col]) + gd[r];
      }
    }
  }
  Cm[w][lane] = cmax;
  inner = wave_sum_f64(inner);
  if (lane == 0) Is[w] = inner;
  __syncthreads();
  for (int e = threadIdx.x; e < R * R; e += 256) pg[int64_t(blockIdx.x) * R * R + e] = Gs[e / R][e % R];
  if (threadIdx.x < R) {
    float mx = 0.f;
    for (int ww = 0; ww < W; ++ww) mx = fmaxf(mx, fmaxf(Cm[ww][threadIdx.x], Cm[ww][threadIdx.x + 32]));
    pm[int64_t(blockIdx.x) * R + threadIdx.x] = double(mx);
  }
  if (threadIdx.x == 0) pi[blockIdx.x] = ((Is[0] + Is[1]) + Is[2]) + Is[3];
}

// Per job and chunk of 256 Gram entries (grid = jobs x ceil(R*R / 256), 1024
// threads): lambda (2-norms from the Gram diagonal on the first sweep, else
// max(1, max |a|)), the Gram of the normalised factor G = (A^T A) ./
// (lambda lambda^T), and the fit's inner product. The partials of an entry
// are summed in four contiguous segments by four threads, each in block order,
// and the segments in order, so the results do not depend on scheduling. Every
// block of a job computes the same lambda; the chunk-0 block stores it.
__global__ __launch_bounds__(1024) void finish_kernel(const CpdJob* __restrict__ jobs, int R,
                                                      int use_max,
                                                      const double* __restrict__ pg,
                                                      const double* __restrict__ pm,
                                                      const double* __restrict__ pi) {
  __shared__ double part[4][256];
  __shared__ double lam[kMaxR];
  const int chunks = (R * R + 255) / 256;
  const int chunk = int(blockIdx.x) % chunks;
  const CpdJob& J = jobs[blockIdx.x / chunks];
  const int t = int(threadIdx.x) & 255, seg = int(threadIdx.x) >> 8;
  const int per = (J.nublk + 3) / 4;
  const int b0 = min(seg * per, J.nublk), b1 = min(b0 + per, J.nublk);
  // this segment's partials, sixteen loaded ahead of their adds
  auto segment = [&](const double* base, int64_t stride, auto&& add) {
    double s = 0.0;
    int b = b0;
    for (; b + 16 <= b1; b += 16) {
      double v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = base[int64_t(J.ublk0 + b + u) * stride];
#pragma unroll
      for (int u = 0; u < 16; ++u) s = add(s, v[u]);
    }
    for (; b < b1; ++b) s = add(s, base[int64_t(J.ublk0 + b) * stride]);
    return s;
  };
  auto plus = [](double x, double y) { return x + y; };
  auto larger = [](double x, double y) { return fmax(x, y); };
  // lambda
  if (t < R) part[seg][t] = use_max ? segment(pm + t, R, larger)
                                    : segment(pg + t * R + t, int64_t(R) * R, plus);
  __syncthreads();
  if (int(threadIdx.x) < R) {
    double l;
    if (use_max) l = fmax(fmax(fmax(part[0][t], part[1][t]), fmax(part[2][t], part[3][t])), 1.0);
    else l = sqrt(((part[0][t] + part[1][t]) + part[2][t]) + part[3][t]);
    if (!(l > 0.0)) l = 1.0;
    lam[t] = double(float(l));
    if (chunk == 0) J.lam[t] = float(l);
  }
  __syncthreads();
  const int e = chunk * 256 + t;
  if (e < R * R) part[seg][t] = segment(pg + e, int64_t(R) * R, plus);
  __syncthreads();
  if (seg == 0 && e < R * R) {
    const double s = ((part[0][t] + part[1][t]) + part[2][t]) + part[3][t];
    J.G[e] = float(s / (lam[e / R] * lam[e % R]));
  }
  if (chunk == 0 && J.inner) {
    __syncthreads();
    if (t == 0) part[seg][0] = segment(pi, 1, plus);
    __syncthreads();
    if (threadIdx.x == 0) *J.inner = ((part[0][0] + part[1][0]) + part[2][0]) + part[3][0];
  }
}

// A /= lambda over every job's rows, float4 at a time (kApplyRows rows per
// block).
__global__ __launch_bounds__(256) void scale4_kernel(const CpdJob* __restrict__ jobs,
                                                     const int32_t* __restrict__ ablk0, int njobs,
                                                     int R) {
  const int j = find_job(ablk0, njobs, blockIdx.x);
  const CpdJob& J = jobs[j];
  const int32_t r0 = (int32_t(blockIdx.x) - J.ablk0) * kApplyRows;
  const int nr = min(kApplyRows, J.rows - r0);
  const int Q = R / 4;
  float4* A4 = reinterpret_cast<float4*>(J.A + int64_t(r0) * R);
  for (int e = threadIdx.x; e < nr * Q; e += blockDim.x) {
    const int qq = e % Q;
    float4 a = A4[e];
    a.x /= J.lam[4 * qq];
    a.y /= J.lam[4 * qq + 1];
    a.z /= J.lam[4 * qq + 2];
    a.w /= J.lam[4 * qq + 3];
    A4[e] = a;
  }
}

template <class T>
int dalloc(T** p, int64_t n) {
  *p = nullptr;
  if (hipMalloc(reinterpret_cast<void**>(p), size_t(std::max<int64_t>(n, 1)) * sizeof(T)) !=
      hipSuccess) {
    *p = nullptr;
    return fail(TENTACO_ENOMEM, "cpd: hipMalloc of %lld elements failed", (long long)n);
  }
  return TENTACO_OK;
}

// sq[t] = |model of tensor t|^2 = sum over (a, b) of lam_a lam_b prod_m G_m[a][b],
// one workgroup per tensor (a job names all its Grams), FP64. It is read back
// with the inner products in one copy; copying the Grams and summing on the
// host took 16 copies of 15 us for three tensors.
__global__ __launch_bounds__(256) void model_norm_kernel(const CpdJob* __restrict__ jobs, int R,
                                                         double* __restrict__ sq) {
  __shared__ double part[256];
  const CpdJob& J = jobs[blockIdx.x];
  double s = 0.0;
  for (int e = int(threadIdx.x); e < R * R; e += 256) {
    double h = double(J.G[e]);
    for (int k = 0; k < J.nG; ++k) h *= double(J.Gk[k][e]);
    s += double(J.lam[e / R]) * double(J.lam[e % R]) * h;
  }
  part[threadIdx.x] = s;
  for (int w = 128; w > 0; w >>= 1) {
    __syncthreads();
    if (int(threadIdx.x) < w) part[threadIdx.x] += part[threadIdx.x + w];
  }
  if (threadIdx.x == 0) sq[blockIdx.x] = part[0];
}

}  // namespace
}  // namespace tt

using namespace tt;

struct tentaco_cpd {
  int nt = 0, R = 0;
  std::vector<int> order;
  std::vector<std::vector<int32_t>> dims;                  // per tensor, tensor mode
  std::vector<std::vector<std::vector<int>>> lvl;          // [t][m][level] -> tensor mode
  std::vector<std::vector<tentaco_csf*>> h;                // [t][m]
  std::vector<std::vector<float*>> A, G;                   // [t][mode]
  std::vector<float*> lam, Vinv;                           // [t]
  // MTTKRP outputs per tensor mode, written only by that mode's batch, which
  // keeps them in retained-output mode (rows no nonzero reaches zeroed once)
  std::vector<std::vector<float*>> M;                      // [t][mode]
  std::vector<double> xnorm2;                              // ||X_t||^2
  double* d_inner = nullptr;                               // [t] <X_t, model>, then [t] |model|^2
  int sweeps = 0;
  // per mode step
  struct Step {
    std::vector<int> tensors;
    tentaco_batch* batch = nullptr;
    bool captured = false;
    CpdJob* d_jobs = nullptr;
    int32_t *d_ablk0 = nullptr, *d_sblk0 = nullptr, *d_ublk0 = nullptr;
    int32_t nablk = 0, nsblk = 0, nublk = 0;
    std::vector<CpdJob> jobs;
  } step[kMaxOrder];
  // jobs for the Grams of every factor (initialisation)
  double* part = nullptr;
  int64_t part_len = 0;
  // partials of the fused update (Gram, column max, inner product)
  double *upg = nullptr, *upm = nullptr, *upi = nullptr;
  hipStream_t own = nullptr;
  // V^-1 needs only the other modes' Grams: it runs beside the batched MTTKRP
  // on this stream (default priority), forked from and joined to the sweep's
  hipStream_t side = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
  // tentaco_cpd_factor copies through it, one caller at a time
  mutable std::mutex stage_mu;
  mutable HostStage stage;

  ~tentaco_cpd() {
    for (auto& s : step) {
      if (s.batch) tentaco_batch_free(s.batch);
      (void)hipFree(s.d_jobs);
      (void)hipFree(s.d_ablk0);
      (void)hipFree(s.d_sblk0);
      (void)hipFree(s.d_ublk0);
    }
    for (auto& v : A)
      for (float* p : v) (void)hipFree(p);
    for (auto& v : G)
      for (float* p : v) (void)hipFree(p);
    for (float* p : lam) (void)hipFree(p);
    for (auto& v : M)
      for (float* p : v) (void)hipFree(p);
    for (float* p : Vinv) (void)hipFree(p);
    (void)hipFree(part);
    (void)hipFree(upg);
    (void)hipFree(upm);
    (void)hipFree(upi);
    (void)hipFree(d_inner);
    if (own) (void)hipStreamDestroy(own);
    if (side) (void)hipStreamDestroy(side);
    if (fork) (void)hipEventDestroy(fork);
    if (join) (void)hipEventDestroy(join);
  }
};

namespace tt {
namespace {

// Fill a job table for `tensors` updating mode m; out-of-place Grams are the
// other modes' Grams.
int build_jobs(tentaco_cpd* c, int m, const std::vector<int>& tensors, std::vector<CpdJob>& jobs,
               std::vector<int32_t>& ablk0, std::vector<int32_t>& sblk0, int32_t& nablk,
               int32_t& nsblk, std::vector<int32_t>* ublk0 = nullptr, int32_t* nublk = nullptr) {
  jobs.clear();
  ablk0.clear();
  sblk0.clear();
  if (ublk0) ublk0->clear();
  nablk = nsblk = 0;
  int32_t nu = 0;
  int64_t total = 0;
  for (int t : tensors) total += c->dims[size_t(t)][size_t(m)];
  const int64_t blocks = std::min<int64_t>(kUpdBlocksMax, std::max<int64_t>(kUpdBlocks, total / 4096));
  const int64_t per = (total + blocks - 1) / blocks;
  const int32_t urows = int32_t((per + kUpdUnit - 1) / kUpdUnit * kUpdUnit);
  for (int t : tensors) {
    CpdJob J;
    J.M = c->M[size_t(t)][size_t(m)];
    J.A = c->A[size_t(t)][size_t(m)];
    J.G = c->G[size_t(t)][size_t(m)];
    J.lam = c->lam[size_t(t)];
    J.Vinv = c->Vinv[size_t(t)];
    for (int k = 0; k < c->order[size_t(t)]; ++k)
      if (k != m) J.Gk[J.nG++] = c->G[size_t(t)][size_t(k)];
    J.rows = c->dims[size_t(t)][size_t(m)];
    J.ablk0 = nablk;
    J.nablk = (J.rows + kApplyRows - 1) / kApplyRows;
    J.sblk0 = nsblk;
    J.nsblk = (J.rows + kStatRows - 1) / kStatRows;
    J.ublk0 = nu;
    J.urows = urows;
    J.nublk = (J.rows + urows - 1) / urows;
    // the fit needs <X, model> from each tensor's last mode update
    if (c->d_inner && m == c->order[size_t(t)] - 1) J.inner = c->d_inner + t;
    ablk0.push_back(J.ablk0);
    sblk0.push_back(J.sblk0);
    if (ublk0) ublk0->push_back(J.ublk0);
    nablk += J.nablk;
    nsblk += J.nsblk;
    nu += J.nublk;
    jobs.push_back(J);
  }
  if (nublk) *nublk = nu;
  return TENTACO_OK;
}

int upload_jobs(const std::vector<CpdJob>& jobs, const std::vector<int32_t>& ablk0,
                const std::vector<int32_t>& sblk0, CpdJob** dj, int32_t** da, int32_t** ds) {
  (void)hipFree(*dj);
  (void)hipFree(*da);
  (void)hipFree(*ds);
  *dj = nullptr;
  *da = *ds = nullptr;
  int rc = 0;
  if ((rc = dalloc(dj, int64_t(jobs.size()))) || (rc = dalloc(da, int64_t(ablk0.size()))) ||
      (rc = dalloc(ds, int64_t(sblk0.size()))))
    return rc;
  TT_HIP_CHECK(hipMemcpy(*dj, jobs.data(), sizeof(CpdJob) * jobs.size(), hipMemcpyHostToDevice));
  TT_HIP_CHECK(hipMemcpy(*da, ablk0.data(), sizeof(int32_t) * ablk0.size(), hipMemcpyHostToDevice));
  TT_HIP_CHECK(hipMemcpy(*ds, sblk0.data(), sizeof(int32_t) * sblk0.size(), hipMemcpyHostToDevice));
  return TENTACO_OK;
}

int ensure_part(tentaco_cpd* c, int64_t n) {
  if (n <= c->part_len) return TENTACO_OK;
  // only reached before any kernel reads the buffer (create)
  (void)hipFree(c->part);
  c->part = nullptr;
  c->part_len = 0;
  int rc = dalloc(&c->part, n);
  if (rc) return rc;
  c->part_len = n;
  return TENTACO_OK;
}

// Grams of the jobs' A (all rows), on st.
int grams(tentaco_cpd* c, const CpdJob* dj, const int32_t* ds, int njobs, int32_t nsblk,
          hipStream_t st) {
  if (njobs == 0 || nsblk == 0) return TENTACO_OK;
  const int R = c->R;
  int rc = ensure_part(c, int64_t(nsblk) * R * R);
  if (rc) return rc;
  gram_partial_kernel<<<nsblk, 256, 0, st>>>(dj, ds, njobs, R, c->part);
  TT_HIP_CHECK(hipGetLastError());
  gram_reduce_kernel<<<njobs, 256, 0, st>>>(dj, R, c->part);
  TT_HIP_CHECK(hipGetLastError());
  return TENTACO_OK;
}

}  // namespace
}  // namespace tt

extern "C" {

int tentaco_cpd_create(tentaco_csf* const* handles, const int* level_modes, int ntensors, int R,
                       uint64_t seed, tentaco_cpd** out) {
  clear_error();
  if (!handles || !level_modes || !out || ntensors < 1)
    return fail(TENTACO_EINVAL, "cpd: NULL argument or no tensors");
  *out = nullptr;
  if (R != 16 && R != 32 && R != 64) return fail(TENTACO_EUNSUPPORTED, "cpd: R must be 16, 32 or 64");
  auto* c = new tentaco_cpd();
  c->nt = ntensors;
  c->R = R;
  auto bail = [&](int rc) {
    delete c;
    return rc;
  };
  for (int t = 0; t < ntensors; ++t) {
    const tentaco_csf* h0 = handles[size_t(t) * kMaxOrder];
    if (!h0) return bail(fail(TENTACO_EINVAL, "cpd: tensor %d has no mode-0 CSF", t));
    const int N = h0->order;
    c->order.push_back(N);
    std::vector<int32_t> dims(size_t(N), 0);
    std::vector<std::vector<int>> lv(static_cast<size_t>(N));
    std::vector<tentaco_csf*> hs(static_cast<size_t>(N));
    for (int m = 0; m < N; ++m) {
      tentaco_csf* h = handles[size_t(t) * kMaxOrder + m];
      if (!h || h->order != N) return bail(fail(TENTACO_EINVAL, "cpd: tensor %d mode %d CSF missing or of another order", t, m));
      const int* L = level_modes + (size_t(t) * kMaxOrder + m) * kMaxOrder;
      bool seen[kMaxOrder] = {};
      if (L[0] != m) return bail(fail(TENTACO_EINVAL, "cpd: tensor %d mode %d CSF must have mode %d at its root", t, m, m));
      for (int l = 0; l < N; ++l) {
        if (L[l] < 0 || L[l] >= N || seen[L[l]]) return bail(fail(TENTACO_EINVAL, "cpd: tensor %d mode %d level map is not a permutation", t, m));
        seen[L[l]] = true;
        lv[size_t(m)].push_back(L[l]);
      }
      hs[size_t(m)] = h;
    }
    // mode dims from the level dims; every CSF must agree
    for (int m = 0; m < N; ++m)
      for (int l = 0; l < N; ++l) {
        const int md = lv[size_t(m)][size_t(l)];
        const int32_t d = hs[size_t(m)]->dims[l];
        if (dims[size_t(md)] == 0) dims[size_t(md)] = d;
        else if (dims[size_t(md)] != d) return bail(fail(TENTACO_EINVAL, "cpd: tensor %d mode %d dimension disagrees between CSFs", t, md));
      }
    if (hs[0]->nodes[N - 1] <= 0) return bail(fail(TENTACO_EINVAL, "cpd: tensor %d is empty", t));
    c->dims.push_back(dims);
    c->lvl.push_back(lv);
    c->h.push_back(hs);
  }
  // factors (U[0,1) from seed, like gen_factor_matrices, ds.h:386-409),
  // lambda = 1, scratch; ||X||^2 from the mode-0 CSF's values
  uint64_t s = seed ^ 0x2545F4914F6CDD1Dull;
  auto next = [&]() {
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
  };
  c->A.resize(size_t(ntensors));
  c->G.resize(size_t(ntensors));
  for (int t = 0; t < ntensors; ++t) {
    const int N = c->order[size_t(t)];
    for (int m = 0; m < N; ++m) {
      const int32_t d = c->dims[size_t(t)][size_t(m)];
      std::vector<float> host(size_t(d) * R);
      for (auto& v : host) v = float(double(next() >> 11) * (1.0 / 9007199254740992.0));
      float *a = nullptr, *g = nullptr;
      int rc = 0;
      if ((rc = dalloc(&a, int64_t(d) * R)) || (rc = dalloc(&g, int64_t(R) * R))) {
        (void)hipFree(a);
        return bail(rc);
      }
      c->A[size_t(t)].push_back(a);
      c->G[size_t(t)].push_back(g);
      if (hipMemcpy(a, host.data(), sizeof(float) * host.size(), hipMemcpyHostToDevice) != hipSuccess)
        return bail(fail(TENTACO_EHIP, "cpd: factor upload failed"));
    }
    float *lam = nullptr, *vi = nullptr;
    int rc = 0;
    if ((rc = dalloc(&lam, R)) || (rc = dalloc(&vi, int64_t(R) * R))) {
      (void)hipFree(lam);
      return bail(rc);
    }
    c->lam.push_back(lam);
    c->Vinv.push_back(vi);
    c->M.emplace_back();
    for (int m = 0; m < N; ++m) {
      float* Mt = nullptr;
      if ((rc = dalloc(&Mt, int64_t(c->dims[size_t(t)][size_t(m)]) * R))) return bail(rc);
      c->M.back().push_back(Mt);
    }
    std::vector<float> ones(size_t(R), 1.f);
    if (hipMemcpy(lam, ones.data(), sizeof(float) * R, hipMemcpyHostToDevice) != hipSuccess)
      return bail(fail(TENTACO_EHIP, "cpd: lambda upload failed"));
    // ||X||^2 (host copy of the values of the mode-0 CSF)
    const tentaco_csf* h0 = c->h[size_t(t)][0];
    const int64_t nnz = h0->nodes[N - 1];
    std::vector<float> vals(static_cast<size_t>(nnz));
    if (hipMemcpy(vals.data(), h0->d_vals, sizeof(float) * size_t(nnz), hipMemcpyDeviceToHost) != hipSuccess)
      return bail(fail(TENTACO_EHIP, "cpd: value download failed"));
    double x2 = 0.0;
    for (float v : vals) x2 += double(v) * double(v);
    c->xnorm2.push_back(x2);
  }
  {
    int rc = dalloc(&c->d_inner, 2 * ntensors);
    if (rc) return bail(rc);
  }
  // mode steps: one batch and one job table each
  for (int m = 0; m < kMaxOrder; ++m) {
    auto& S = c->step[m];
    for (int t = 0; t < ntensors; ++t)
      if (c->order[size_t(t)] > m) S.tensors.push_back(t);
    if (S.tensors.empty()) continue;
    std::vector<tentaco_csf*> tasks;
    std::vector<const float*> facs;
    std::vector<float*> outs;
    std::vector<int32_t> rows;
    for (int t : S.tensors) {
      tasks.push_back(c->h[size_t(t)][size_t(m)]);
      const auto& L = c->lvl[size_t(t)][size_t(m)];
      for (int l = 1; l < kMaxOrder; ++l)
        facs.push_back(l < int(L.size()) ? c->A[size_t(t)][size_t(L[size_t(l)])] : nullptr);
      outs.push_back(c->M[size_t(t)][size_t(m)]);
      rows.push_back(c->dims[size_t(t)][size_t(m)]);
    }
    int rc = tentaco_batch_create(tasks.data(), int(tasks.size()), R, &S.batch);
    if (!rc) rc = tentaco_batch_set_operands(S.batch, facs.data(), outs.data(), rows.data());
    if (!rc) rc = tentaco_batch_set_output_mode(S.batch, TENTACO_BATCH_OUTPUTS_RETAINED);
    if (rc) return bail(rc);
    std::vector<int32_t> ab, sb, ub;
    build_jobs(c, m, S.tensors, S.jobs, ab, sb, S.nablk, S.nsblk, &ub, &S.nublk);
    rc = upload_jobs(S.jobs, ab, sb, &S.d_jobs, &S.d_ablk0, &S.d_sblk0);
    if (!rc) rc = dalloc(&S.d_ublk0, int64_t(ub.size()));
    if (rc) return bail(rc);
    TT_HIP_CHECK(hipMemcpy(S.d_ublk0, ub.data(), sizeof(int32_t) * ub.size(), hipMemcpyHostToDevice));
  }
  {
    int64_t nu = 1;
    for (auto& S : c->step) nu = std::max<int64_t>(nu, S.nublk);
    int rc = 0;
    if ((rc = dalloc(&c->upg, nu * R * R)) || (rc = dalloc(&c->upm, nu * R)) ||
        (rc = dalloc(&c->upi, nu)))
      return bail(rc);
  }
  // the reduction partials, sized once for the largest step (never
  // reallocated while kernels may still read them)
  {
    int64_t need = 1;
    for (auto& S : c->step) need = std::max<int64_t>(need, int64_t(S.nsblk) * R * R);
    int rc = ensure_part(c, need);
    if (rc) return bail(rc);
  }
  // initial Grams of every factor
  for (int m = 0; m < kMaxOrder; ++m) {
    auto& S = c->step[m];
    if (S.tensors.empty()) continue;
    int rc = grams(c, S.d_jobs, S.d_sblk0, int(S.jobs.size()), S.nsblk, nullptr);
    if (rc) return bail(rc);
  }
  TT_HIP_CHECK(hipDeviceSynchronize());
  *out = c;
  return TENTACO_OK;
}

int tentaco_cpd_tune(tentaco_cpd* c, int reps) {
  clear_error();
  if (!c) return fail(TENTACO_EINVAL, "cpd: NULL handle");
  for (auto& S : c->step) {
    if (!S.batch) continue;
    int f, b, g;
    float ms;
    int rc = tentaco_batch_autotune(S.batch, reps, nullptr, &f, &b, &g, &ms);
    if (rc) return rc;
    S.captured = false;
  }
  return TENTACO_OK;
}

int tentaco_cpd_iterate(tentaco_cpd* c, int sweeps, int use_graphs, void* stream, double* fits) {
  clear_error();
  if (!c) return fail(TENTACO_EINVAL, "cpd: NULL handle");
  if (sweeps < 1) return fail(TENTACO_EINVAL, "cpd: sweeps must be >= 1");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (use_graphs && !st) {
    if (!c->own) TT_HIP_CHECK(hipStreamCreate(&c->own));
    st = c->own;
  }
  if (!c->side) {
    TT_HIP_CHECK(hipEventCreateWithFlags(&c->fork, hipEventDisableTiming));
    TT_HIP_CHECK(hipEventCreateWithFlags(&c->join, hipEventDisableTiming));
    TT_HIP_CHECK(hipStreamCreateWithFlags(&c->side, hipStreamNonBlocking));
  }
  const int R = c->R;
  for (int it = 0; it < sweeps; ++it) {
    const int use_max = c->sweeps > 0 ? 1 : 0;
    for (int m = 0; m < kMaxOrder; ++m) {
      auto& S = c->step[m];
      if (S.tensors.empty()) continue;
      const int nj = int(S.jobs.size());
      int rc;
      if (use_graphs && !S.captured) {
        rc = tentaco_batch_capture(S.batch, st);
        if (rc) return rc;
        S.captured = true;
      }
      TT_HIP_CHECK(hipEventRecord(c->fork, st));
      TT_HIP_CHECK(hipStreamWaitEvent(c->side, c->fork, 0));
      switch (R) {
        case 16: hadamard_inverse_kernel<16><<<nj, 256, 0, c->side>>>(S.d_jobs); break;
        case 32: hadamard_inverse_kernel<32><<<nj, 256, 0, c->side>>>(S.d_jobs); break;
        default: hadamard_inverse_kernel<64><<<nj, 1024, 0, c->side>>>(S.d_jobs); break;
      }
      TT_HIP_CHECK(hipGetLastError());
      TT_HIP_CHECK(hipEventRecord(c->join, c->side));
      rc = use_graphs ? tentaco_batch_launch(S.batch, st) : tentaco_batch_run(S.batch, st);
      if (rc) return rc;
      TT_HIP_CHECK(hipStreamWaitEvent(st, c->join, 0));
      switch (R) {
        case 16:
          update_kernel<16><<<S.nublk, 256, 0, st>>>(S.d_jobs, S.d_ublk0, nj, c->upg, c->upm, c->upi);
          break;
        case 32:
          update32_mfma_kernel<<<S.nublk, 256, 0, st>>>(S.d_jobs, S.d_ublk0, nj, c->upg, c->upm,
                                                        c->upi);
          break;
        default:
          update_kernel<64><<<S.nublk, 256, 0, st>>>(S.d_jobs, S.d_ublk0, nj, c->upg, c->upm, c->upi);
          break;
      }
      TT_HIP_CHECK(hipGetLastError());
      finish_kernel<<<nj * ((R * R + 255) / 256), 1024, 0, st>>>(S.d_jobs, R, use_max, c->upg,
                                                                 c->upm, c->upi);
      TT_HIP_CHECK(hipGetLastError());
      scale4_kernel<<<S.nablk, 256, 0, st>>>(S.d_jobs, S.d_ablk0, nj, R);
      TT_HIP_CHECK(hipGetLastError());
    }
    ++c->sweeps;
  }
  if (fits) {
    // step 0 holds a job of every tensor
    model_norm_kernel<<<c->nt, 256, 0, st>>>(c->step[0].d_jobs, R, c->d_inner + c->nt);
    TT_HIP_CHECK(hipGetLastError());
  }
  TT_HIP_CHECK(hipStreamSynchronize(st));
  if (fits) {
    std::vector<double> sums(size_t(c->nt) * 2, 0.0);
    {
      std::lock_guard<std::mutex> lk(c->stage_mu);
      const int rc = c->stage.to_host(sums.data(), c->d_inner, sizeof(double) * sums.size());
      if (rc) return rc;
    }
    for (int t = 0; t < c->nt; ++t) {
      const double inner = sums[size_t(t)], mnorm = sums[size_t(c->nt + t)];
      const double resid = std::max(0.0, c->xnorm2[size_t(t)] + mnorm - 2.0 * inner);
      fits[t] = c->xnorm2[size_t(t)] > 0.0 ? 1.0 - std::sqrt(resid) / std::sqrt(c->xnorm2[size_t(t)]) : 0.0;
    }
  }
  return TENTACO_OK;
}

int tentaco_cpd_factor(const tentaco_cpd* c, int t, int m, float* factor, float* lambda) {
  clear_error();
  if (!c || t < 0 || t >= c->nt) return fail(TENTACO_EINVAL, "cpd: bad tensor index");
  if (m < 0 || m >= c->order[size_t(t)]) return fail(TENTACO_EINVAL, "cpd: bad mode");
  std::lock_guard<std::mutex> lk(c->stage_mu);
  return c->stage.to_host(
      factor, c->A[size_t(t)][size_t(m)],
      factor ? sizeof(float) * size_t(c->dims[size_t(t)][size_t(m)]) * c->R : 0, lambda,
      c->lam[size_t(t)], lambda ? sizeof(float) * c->R : 0);
}

int tentaco_cpd_set_factor(tentaco_cpd* c, int t, int m, const float* factor) {
  clear_error();
  if (!c || !factor || t < 0 || t >= c->nt) return fail(TENTACO_EINVAL, "cpd: bad argument");
  if (m < 0 || m >= c->order[size_t(t)]) return fail(TENTACO_EINVAL, "cpd: bad mode");
  TT_HIP_CHECK(hipMemcpy(c->A[size_t(t)][size_t(m)], factor,
                         sizeof(float) * size_t(c->dims[size_t(t)][size_t(m)]) * c->R,
                         hipMemcpyHostToDevice));
  // refresh this factor's Gram through a one-job table
  std::vector<CpdJob> jobs;
  std::vector<int32_t> ab, sb;
  int32_t na = 0, ns = 0;
  std::vector<int> one{t};
  build_jobs(c, m, one, jobs, ab, sb, na, ns);
  CpdJob* dj = nullptr;
  int32_t *da = nullptr, *ds = nullptr;
  int rc = upload_jobs(jobs, ab, sb, &dj, &da, &ds);
  if (!rc) rc = grams(c, dj, ds, 1, ns, nullptr);
  if (!rc && hipDeviceSynchronize() != hipSuccess) rc = fail(TENTACO_EHIP, "cpd: synchronize failed");
  (void)hipFree(dj);
  (void)hipFree(da);
  (void)hipFree(ds);
  return rc;
}

int tentaco_cpd_free(tentaco_cpd* c) {
  if (c && c->side) (void)hipStreamSynchronize(c->side);
  delete c;
  return TENTACO_OK;
}

}  // extern "C"
