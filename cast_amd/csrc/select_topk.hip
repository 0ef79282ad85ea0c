// Fixed-budget top-k block selector (gfx950): one wavefront per row; the
// selection itself is in select_core.h.
#include "select_core.h"

namespace rcsa {

template <int PER, bool RANK, bool MIXED>
__global__ void __launch_bounds__(kSelWaves * kWave)
select_kernel(SelArgs a) {
  extern __shared__ __attribute__((aligned(16))) char s_rank[];  // RANK: kSelWaves rank lists
  select_rows<PER, RANK, MIXED>(a, blockIdx.x, s_rank);
}

// The selection's certificate: per row the repeated neighbours of its list
// (first counts[row] entries), the stencil's blocks it keeps and the sum of its
// scores; a second launch adds the rows up in order.
struct CheckArgs {
  const int32_t* selected;  // [n_rows][max_k]
  const int32_t* counts;    // [n_rows]
  const uint8_t* local;     // [n_q][n_k]
  const float* score;       // [n_rows][n_k]
  int64_t n_rows, n_q, n_k, max_k;
  double* rows;             // [n_rows][3]
  double* out;              // [3]
};

__device__ __forceinline__ double wave_sum_d(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  return v;
}

__global__ void __launch_bounds__(kSelWaves * kWave) check_rows_kernel(CheckArgs a) {
  const int lane = threadIdx.x % kWave;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kSelWaves + threadIdx.x / kWave;
  if (row >= a.n_rows) return;
  const int32_t* sel = a.selected + row * a.max_k;
  const uint8_t* local = a.local + row % a.n_q * a.n_k;
  int64_t n = a.counts[row];
  n = n < 0 ? 0 : (n > a.max_k ? a.max_k : n);
  int dup = 0, kept = 0;
  for (int64_t e = lane; e < n; e += kWave) {
    const int32_t j = sel[e];
    dup += e > 0 && sel[e - 1] == j;
    kept += j >= 0 && j < a.n_k && local[j] != 0;
  }
  double sum = 0.0;
  for (int64_t j = lane; j < a.n_k; j += kWave) sum += static_cast<double>(a.score[row * a.n_k + j]);
  const double d = wave_sum_d(dup), c = wave_sum_d(kept);
  sum = wave_sum_d(sum);
  if (lane == 0) {
    a.rows[row * 3] = d;
    a.rows[row * 3 + 1] = c;
    a.rows[row * 3 + 2] = sum;
  }
}

__global__ void __launch_bounds__(1024) check_sum_kernel(CheckArgs a) {
  __shared__ double s_sum[16][3];
  double v[3] = {0.0, 0.0, 0.0};
  for (int64_t r = threadIdx.x; r < a.n_rows; r += 1024)
#pragma unroll
    for (int i = 0; i < 3; ++i) v[i] += a.rows[r * 3 + i];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    v[i] = wave_sum_d(v[i]);
    if (threadIdx.x % kWave == 0) s_sum[threadIdx.x / kWave][i] = v[i];
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    double t = 0.0;
    for (int w = 0; w < 16; ++w) t += s_sum[w][threadIdx.x];
    a.out[threadIdx.x] = t;
  }
}

template <bool RANK, bool MIXED = false>
static void launch_select(const SelArgs& a, hipStream_t stream) {
  const int64_t per = (a.n_k + kWave - 1) / kWave;
  dim3 grid(static_cast<unsigned>((a.n_rows + kSelWaves - 1) / kSelWaves));
  dim3 block(kSelWaves * kWave);
  const size_t lds = RANK ? static_cast<size_t>(kSelWaves * rank_slots(a.max_k) * kRankSlotBytes)
                          : 0;
  if (per <= 1) select_kernel<1, RANK, MIXED><<<grid, block, lds, stream>>>(a);
  else if (per <= 2) select_kernel<2, RANK, MIXED><<<grid, block, lds, stream>>>(a);
  else if (per <= 4) select_kernel<4, RANK, MIXED><<<grid, block, lds, stream>>>(a);
  else if (per <= 6) select_kernel<6, RANK, MIXED><<<grid, block, lds, stream>>>(a);
  else if (per <= 8) select_kernel<8, RANK, MIXED><<<grid, block, lds, stream>>>(a);
  else if (per <= 16) select_kernel<16, RANK, MIXED><<<grid, block, lds, stream>>>(a);
  else if (per <= 32) select_kernel<32, RANK, MIXED><<<grid, block, lds, stream>>>(a);
  else select_kernel<0, RANK, MIXED><<<grid, block, lds, stream>>>(a);
}

}  // namespace rcsa

using namespace rcsa;

extern "C" int rcsa_select_topk(const float* score, int64_t n_bh, int64_t n_qblocks,
                                int64_t n_kblocks, const int32_t* row_k,
                                int64_t row_k_stride_bh, int64_t k_fixed,
                                const uint8_t* forced, const uint8_t* allowed,
                                int64_t mask_stride_bh, int32_t* indices,
                                int64_t max_k, int32_t* counts, int order,
                                hipStream_t stream) {
  if (!score || !indices || !counts) return RCSA_ERR_NULL;
  if (n_bh <= 0 || n_qblocks <= 0 || n_kblocks <= 0 || max_k <= 0) return RCSA_ERR_SHAPE;
  if (n_kblocks > 65536) return RCSA_ERR_SHAPE;
  if (order != RCSA_ORDER_INDEX && order != RCSA_ORDER_RANK && order != RCSA_ORDER_RANK_LOCAL &&
      order != RCSA_ORDER_SPLIT)
    return RCSA_ERR_SHAPE;
  if (order != RCSA_ORDER_INDEX && max_k > 2048) return RCSA_ERR_SHAPE;
  if (mask_stride_bh < 0 || row_k_stride_bh < 0) return RCSA_ERR_STRIDE;
  SelArgs a{score, n_bh * n_qblocks, n_qblocks, n_kblocks, row_k, row_k_stride_bh,
            k_fixed, forced, allowed, mask_stride_bh, indices, max_k, counts,
            order == RCSA_ORDER_RANK_LOCAL, 0, 0};
  if (order == RCSA_ORDER_SPLIT) {
    a.xcd_items = (a.n_rows + kNumXcd - 1) / kNumXcd;
    a.xcd_direct = whole_items(a.xcd_items, cus_per_xcd());
    launch_select<true, true>(a, stream);
  } else if (order != RCSA_ORDER_INDEX) {
    launch_select<true>(a, stream);
  } else {
    launch_select<false>(a, stream);
  }
  return launch_status();
}

extern "C" int rcsa_select_check(const int32_t* selected, const int32_t* counts,
                                 const uint8_t* local, const float* score, int64_t n_bh,
                                 int64_t n_qblocks, int64_t n_kblocks, int64_t max_k,
                                 double* row_sums, double* out, hipStream_t stream) {
  if (!selected || !counts || !local || !score || !row_sums || !out) return RCSA_ERR_NULL;
  if (n_bh <= 0 || n_qblocks <= 0 || n_kblocks <= 0 || max_k <= 0) return RCSA_ERR_SHAPE;
  const CheckArgs a{selected, counts, local, score, n_bh * n_qblocks, n_qblocks, n_kblocks,
                    max_k, row_sums, out};
  check_rows_kernel<<<dim3(static_cast<unsigned>((a.n_rows + kSelWaves - 1) / kSelWaves)),
                      dim3(kSelWaves * kWave), 0, stream>>>(a);
  check_sum_kernel<<<dim3(1), dim3(1024), 0, stream>>>(a);
  return launch_status();
}
