// The batch of several orders in one launch.
#include "mttkrp_order.h"

namespace tt {
namespace {

struct OrderTiles {
  int32_t G[kMaxOrder + 1], NB[kMaxOrder + 1];
};

// batch_kernel over the tasks of every order: a workgroup takes whichever
// item is next and branches on its task's order, so no order waits for the
// workgroups of another to end (a launch per order on its own queue gave the
// 123 workgroups of three-mode tensors their places only as the others
// finished), and one queue needs no fork and join. The price is the largest
// order's registers for all: 161 at R=32, where three waves a SIMD without
// spills beat four with 37 registers spilled (569 and 649 us for 8 uneven
// tensors; at R=16 453 and 395, at R=64 933 and 877, so four there). A sweep of
// three tensors, five mode steps: 800 us with launches per order, 566 with this
// (220 of them the fit's); small batches 86 -> 79 us, with written outputs
// 131 -> 84. launch_batch_orders has the sizes up to which it is the faster.
template <int R>
__global__ __launch_bounds__(512, (R == 32 ? 3 : 4)) void batch_all_kernel(
    const BatchTaskDev* __restrict__ tasks, int32_t ntasks, const int64_t* __restrict__ item_off,
    int32_t items, int32_t* __restrict__ counter, int Rr, OrderTiles tl, int32_t chunk, int dynamic) {
  extern __shared__ __align__(16) unsigned char smem[];
  batch_items(tasks, 0, ntasks, item_off, 0, items, counter, chunk, dynamic,
              [&](const BatchTaskDev& T, int32_t b) {
                switch (T.B.order) {
                  case 2:
                    edge_block<2, R, true, true, true>(T.B, T.F, T.A, Rr, nullptr, T.starts, b, tl.G[2],
                                                       tl.NB[2], smem, T.W, T.slots + b);
                    break;
                  case 3:
                    edge_block<3, R, true, true, true>(T.B, T.F, T.A, Rr, nullptr, T.starts, b, tl.G[3],
                                                       tl.NB[3], smem, T.W, T.slots + b);
                    break;
                  case 4:
                    edge_block<4, R, true, true, true>(T.B, T.F, T.A, Rr, nullptr, T.starts, b, tl.G[4],
                                                       tl.NB[4], smem, T.W, T.slots + b);
                    break;
                  default:
                    edge_block<5, R, true, true, true>(T.B, T.F, T.A, Rr, nullptr, T.starts, b, tl.G[5],
                                                       tl.NB[5], smem, T.W, T.slots + b);
                    break;
                }
              });
}

template <int R>
int launch_all(const BatchLaunch& L, int block, int schedule, hipStream_t st) {
  OrderTiles tl{};
  for (int N = 2; N <= kMaxOrder; ++N) {
    tl.G[N] = L.grp[N];
    tl.NB[N] = L.nb[N];
  }
  const size_t lds = size_t(block / 64) * edge_wave_lds<R, true>();
  const int grid = std::max(1, std::min<int>(L.all_grid, L.total_items));
  batch_all_kernel<R><<<grid, block, lds, st>>>(L.tasks, L.ntasks, L.item_off, L.total_items, L.counter + 2,
                                                L.R, tl, batch_chunk(L.total_items, grid, schedule),
                                                schedule == 0);
  TT_HIP_CHECK(hipGetLastError());
  return TENTACO_OK;
}

template <int R>
int occupancy_all(int block, int* per_cu) {
  const size_t lds = size_t(block / 64) * edge_wave_lds<R, true>();
  const hipError_t e =
      hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, batch_all_kernel<R>, block, lds);
  if (e != hipSuccess) return fail(TENTACO_EHIP, "occupancy query: %s", hipGetErrorString(e));
  return TENTACO_OK;
}

}  // namespace

int all_orders_batch(const BatchLaunch& L, int block, int schedule, hipStream_t st) {
  switch (L.R) {
    case 16: return launch_all<16>(L, block, schedule, st);
    case 32: return launch_all<32>(L, block, schedule, st);
    default: return launch_all<64>(L, block, schedule, st);
  }
}

int all_orders_batch_occupancy(int block, int R, int* per_cu) {
  switch (R) {
    case 16: return occupancy_all<16>(block, per_cu);
    case 32: return occupancy_all<32>(block, per_cu);
    default: return occupancy_all<64>(block, per_cu);
  }
}

}  // namespace tt
