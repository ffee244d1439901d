// spmm_vals.hip — FP32 SpMM of a value-carrying bitmap (vals_tile.hpp): one problem
// or a grouped launch (gfx950).
#include "vals_tile.hpp"

namespace bws {
namespace {

template <int VR>
__global__ void __launch_bounds__(kVW * 64)
k_spmm_vals(const uint32_t* __restrict__ W, int64_t M, int64_t K, int64_t ldw,
            const int64_t* __restrict__ row_ptr, const float* __restrict__ values,
            const float* __restrict__ B, int64_t ldb, int64_t N, float* __restrict__ C,
            int64_t ldc, float alpha, float beta, int64_t row_blocks, int64_t col_blocks,
            int64_t per_xcd) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kValsLds];
  const int64_t tile = xcd_tile(blockIdx.x, per_xcd);
  if (tile >= row_blocks * col_blocks) return;
  vals_tile<VR>(W, M, K, ldw, row_ptr, values, B, ldb, N, C, ldc, alpha, beta, tile, row_blocks,
                smem);
}

// Grouped launch: a workgroup finds its problem and tile with batch_tile.
template <int VR, bool RANGE>
__global__ void __launch_bounds__(kVW * 64)
k_spmm_vals_batch(const BatchEntry* __restrict__ entries, const int64_t* __restrict__ off,
                  int count, int64_t range) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kValsLds];
  int lo;
  int64_t tile;
  if (!batch_tile<RANGE>(entries, off, count, range, lo, tile)) return;
  const BatchEntry& e = entries[lo];
  vals_tile<VR>(e.W, e.M, e.K, e.ldw, e.row_ptr, e.values, static_cast<const float*>(e.B), e.ldb,
                e.N, e.C, e.ldc, 1.0f, 0.0f, tile, e.row_blocks, smem);
}

template <int VR>
bws_status launch_vals(const bws_bitmap* A, const float* B, int64_t ldb, int64_t N, float* C,
                       int64_t ldc, float alpha, float beta, hipStream_t s) {
  const int64_t row_blocks = ceil_div(A->rows, kVW * VR), col_blocks = ceil_div(N, kVBN);
  const int64_t per_xcd = ceil_div(row_blocks * col_blocks, 8);
  if (8 * per_xcd > kMaxGrid) return BWS_ECAPACITY;
  hipLaunchKernelGGL(k_spmm_vals<VR>, dim3((unsigned)(8 * per_xcd)), dim3(kVW * 64), 0, s,
                     A->words, A->rows, A->cols, A->ldw, A->row_ptr, A->values, B, ldb, N, C, ldc,
                     alpha, beta, row_blocks, col_blocks, per_xcd);
  return launch_check();
}

}  // namespace

bool spmm_vals_ok(int64_t K) { return K <= kValsMaxK; }

// Rows per workgroup of the value product's tile.  A workgroup has a CU to itself,
// so the time is the number of rounds over 256 CUs times a tile's: 143, 242 and
// 421 us for 64, 128 and 256 rows at K = 4096 and 10% density (80, 120, 189 at 1%;
// 394, 735, 1412 at 50%), of which 100 us do not depend on the rows.  The 256-row
// form keeps 28 bytes a lane in scratch (16 waves leave a lane 128 registers, 64 of
// them sums); the other two keep none.
int32_t spmm_vals_rows(int64_t M, int64_t N) {
  static const int32_t rows[3] = {256, 128, 64}, cost[3] = {26, 15, 9};
  int32_t best = 0;
  int64_t best_cost = 0;
  for (int i = 0; i < 3; ++i) {
    const int64_t c = ceil_div(ceil_div(M, rows[i]) * ceil_div(N, kVBN), 256) * cost[i];
    if (best == 0 || c < best_cost) {
      best = rows[i];
      best_cost = c;
    }
  }
  return best;
}

bws_status spmm_vals_f32(const bws_bitmap* A, const float* B, int64_t ldb, int64_t N, float* C,
                         int64_t ldc, float alpha, float beta, int32_t rows, hipStream_t s) {
  switch (rows) {
    case 256: return launch_vals<16>(A, B, ldb, N, C, ldc, alpha, beta, s);
    case 128: return launch_vals<8>(A, B, ldb, N, C, ldc, alpha, beta, s);
    case 64: return launch_vals<4>(A, B, ldb, N, C, ldc, alpha, beta, s);
    default: return BWS_EINVAL;
  }
}

bws_status spmm_vals_f32_batch(const BatchEntry* entries, const int64_t* off, int count,
                               int64_t total_tiles, int32_t rows, hipStream_t s) {
  const int64_t range = batch_range(total_tiles, count);
  const int64_t grid = batch_grid(total_tiles, count, range);
  if (grid > kMaxGrid) return BWS_ECAPACITY;
  if (total_tiles == 0) return BWS_OK;
  auto launch = [&](auto ranges, auto shares) {
    hipLaunchKernelGGL(range ? ranges : shares, dim3((unsigned)grid), dim3(kVW * 64), 0, s, entries,
                       off, count, range);
  };
  switch (rows) {
    case 256: launch(k_spmm_vals_batch<16, true>, k_spmm_vals_batch<16, false>); break;
    case 128: launch(k_spmm_vals_batch<8, true>, k_spmm_vals_batch<8, false>); break;
    case 64: launch(k_spmm_vals_batch<4, true>, k_spmm_vals_batch<4, false>); break;
    default: return BWS_EINVAL;
  }
  return launch_check();
}

}  // namespace bws
