// Block lists and key validity in the form the attention reads fastest
// (gfx950): every list in ascending block order, the validity flags as bits.
//
// The attention streams the key blocks of a list in the list's order, and the
// lists of neighbouring query blocks share blocks.  In ascending order the
// workgroups of a head sweep its keys together and share them in their XCD's
// L2; in score order each re-reads them from the Infinity Cache or HBM.
//
// One wavefront sorts one list (or one share of it) by counting: entries are
// tallied per block in LDS, and every block number is written as often as it is
// listed, at the wavefront's running prefix.  A list of n entries over nb blocks
// costs n + nb LDS accesses whatever its order.
//
// A list that the attention cuts into shares is ordered share by share: which
// entries a share holds stays the caller's.  The shares' partial outputs are
// rounded to bf16, and those of a run of neighbouring blocks, whose keys resemble
// each other, are larger than those of a mixture: from float64, 1 head x 1 query
// block x 89 of 215 key blocks in random order 1.89e-3 as given, 2.21e-3 where the
// shares are cut from the ascending list, 1.89e-3 so.
#include "rcsa_common.h"

namespace rcsa {

struct ListArgs {
  const int32_t* idx;
  const int32_t* lens;
  int64_t sbz, sbh, sbm, slz, slh, slm;
  const int64_t* rows;  // output row r is row rows[r] of the source (nullable: r)
  int64_t n_src_rows;
  int64_t H, n_rows, max_k;
  int32_t n_blocks;     // key blocks
  int64_t n_lists;      // B * H * n_rows
  // lists [x xcd_items + xcd_direct, (x + 1) xcd_items) of XCD x are cut into n_split shares
  int64_t xcd_items, xcd_direct;
  uint32_t n_split;
  int32_t* out_idx;     // [n_lists][max_k]
  int32_t* out_lens;    // [n_lists]
  const uint8_t* valid;  // nullable
  int64_t n_valid;
  uint32_t* bits;       // [ceil(n_valid / 32)]
};

constexpr int kListWaves = 4;
constexpr int64_t kListMaxBlocks = 4096;  // LDS tallies: 4 x 16 KiB

// Workgroups [0, list_wgs): kListWaves wavefronts, n_split for each list (of a
// list that is not cut all but the first end at once).  The shares of a list side
// by side take as long as one: 3 heads x 7 lists of 2048 blocks in 8 shares, one
// after the other by one wavefront, took 85 us.  The rest: 256 flags each.
__global__ void __launch_bounds__(kListWaves * kWave)
order_lists_kernel(ListArgs a, int64_t list_wgs) {
  extern __shared__ uint32_t s_tally[];  // kListWaves * n_blocks
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  if (blockIdx.x >= list_wgs) {
    const int64_t first = (static_cast<int64_t>(blockIdx.x) - list_wgs) * 256 + wave * kWave;
    const int64_t i = first + lane;
    const uint64_t m = __ballot(i < a.n_valid && a.valid[i] != 0);
    if (lane < 2 && first + 32 * lane < a.n_valid)
      a.bits[first / 32 + lane] = static_cast<uint32_t>(m >> (32 * lane));
    return;
  }
  const int64_t unit = static_cast<int64_t>(blockIdx.x) * kListWaves + wave;
  const int64_t list = unit / a.n_split;
  const uint32_t s = static_cast<uint32_t>(unit % a.n_split);
  if (list >= a.n_lists) return;  // whole wavefronts; no barrier below
  const bool cut = a.n_split > 1 && list % a.xcd_items >= a.xcd_direct;
  if (!cut && s > 0) return;
  const uint32_t ns = cut ? a.n_split : 1;
  const int64_t r = list % a.n_rows, bh = list / a.n_rows;
  const int64_t b = bh / a.H, h = bh % a.H;
  int64_t row = a.rows ? a.rows[r] : r;
  row = row < 0 ? 0 : (row < a.n_src_rows ? row : a.n_src_rows - 1);
  const int32_t* src = a.idx + b * a.sbz + h * a.sbh + row * a.sbm;
  int64_t n64 = a.lens[b * a.slz + h * a.slh + row * a.slm];
  n64 = n64 < 0 ? 0 : (n64 > a.max_k ? a.max_k : n64);
  const uint32_t n = static_cast<uint32_t>(n64);  // (< 2^24, ns <= 16)
  const uint32_t first = n * s / ns, end = n * (s + 1) / ns;  // the attention's shares
  uint32_t* tally = s_tally + wave * a.n_blocks;
  for (int j = lane; j < a.n_blocks; j += kWave) tally[j] = 0;
  // the tallies are this wavefront's own: its LDS operations stay in order
  __builtin_amdgcn_wave_barrier();
  for (uint32_t e = first + lane; e < end; e += kWave) {
    const uint32_t j = static_cast<uint32_t>(src[e]);
    if (j < static_cast<uint32_t>(a.n_blocks)) atomicAdd(&tally[j], 1u);
  }
  __builtin_amdgcn_wave_barrier();
  int32_t* out = a.out_idx + list * a.max_k;
  uint32_t base = first;
  for (int j0 = 0; j0 < a.n_blocks; j0 += kWave) {
    const int j = j0 + lane;
    const uint32_t c = j < a.n_blocks ? tally[j] : 0u;
    uint32_t pre = c;  // inclusive prefix over the wavefront
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const uint32_t up = __shfl_up(pre, o, kWave);
      if (lane >= o) pre += up;
    }
    for (uint32_t t = 0; t < c; ++t) out[base + pre - c + t] = j;
    base += __shfl(pre, kWave - 1, kWave);
  }
  // entries that name no block leave a whole list; a share keeps its place in it
  const int64_t stop = s + 1 < ns ? end : a.max_k;
  for (int64_t e = base + lane; e < stop; e += kWave) out[e] = -1;
  if (s == 0 && lane == 0) a.out_lens[list] = static_cast<int32_t>(cut ? n : base);
}

}  // namespace rcsa

using namespace rcsa;

extern "C" int64_t rcsa_order_lists_max_blocks(void) { return kListMaxBlocks; }

extern "C" int rcsa_order_split_lists(const int32_t* block_indices,
                                      const int32_t* block_indices_lens,
                                      int64_t stride_bz, int64_t stride_bh, int64_t stride_bm,
                                      int64_t stride_lz, int64_t stride_lh, int64_t stride_lm,
                                      const int64_t* rows, int64_t n_src_rows, int64_t B,
                                      int64_t H, int64_t n_rows, int64_t max_k,
                                      int64_t n_kblocks, int64_t n_split, int32_t* out_indices,
                                      int32_t* out_lens, const uint8_t* valid, int64_t n_valid,
                                      uint32_t* valid_bits, hipStream_t stream) {
  if ((valid == nullptr) != (valid_bits == nullptr)) return RCSA_ERR_NULL;
  if (block_indices == nullptr && valid == nullptr) return RCSA_ERR_NULL;
  ListArgs a{};
  int64_t list_wgs = 0;
  size_t lds = 0;
  if (block_indices) {
    if (!block_indices_lens || !out_indices || !out_lens) return RCSA_ERR_NULL;
    if (B <= 0 || H <= 0 || n_rows <= 0 || n_src_rows <= 0 || max_k <= 0 ||
        max_k >= (int64_t{1} << 24) || n_kblocks <= 0 || n_kblocks > kListMaxBlocks)
      return RCSA_ERR_SHAPE;
    if (!rows && n_rows > n_src_rows) return RCSA_ERR_SHAPE;
    if (n_split < 1 || n_split > 16) return RCSA_ERR_SHAPE;
    a.idx = block_indices;
    a.lens = block_indices_lens;
    a.sbz = stride_bz; a.sbh = stride_bh; a.sbm = stride_bm;
    a.slz = stride_lz; a.slh = stride_lh; a.slm = stride_lm;
    a.rows = rows;
    a.n_src_rows = n_src_rows;
    a.H = H;
    a.n_rows = n_rows;
    a.max_k = max_k;
    a.n_blocks = static_cast<int32_t>(n_kblocks);
    a.n_lists = B * H * n_rows;
    a.xcd_items = (a.n_lists + kNumXcd - 1) / kNumXcd;
    a.xcd_direct = n_split > 1 ? whole_items(a.xcd_items, cus_per_xcd()) : a.xcd_items;
    a.n_split = static_cast<uint32_t>(n_split);
    a.out_idx = out_indices;
    a.out_lens = out_lens;
    list_wgs = (a.n_lists * n_split + kListWaves - 1) / kListWaves;
    lds = static_cast<size_t>(kListWaves * n_kblocks) * sizeof(uint32_t);
  }
  int64_t valid_wgs = 0;
  if (valid) {
    if (n_valid <= 0) return RCSA_ERR_SHAPE;
    a.valid = valid;
    a.n_valid = n_valid;
    a.bits = valid_bits;
    valid_wgs = (n_valid + 255) / 256;
  }
  if (list_wgs + valid_wgs >= (int64_t{1} << 31)) return RCSA_ERR_SHAPE;
  order_lists_kernel<<<dim3(static_cast<unsigned>(list_wgs + valid_wgs)),
                       dim3(kListWaves * kWave), lds, stream>>>(a, list_wgs);
  return launch_status();
}

extern "C" int rcsa_order_lists(const int32_t* block_indices, const int32_t* block_indices_lens,
                                int64_t stride_bz, int64_t stride_bh, int64_t stride_bm,
                                int64_t stride_lz, int64_t stride_lh, int64_t stride_lm,
                                const int64_t* rows, int64_t n_src_rows, int64_t B, int64_t H,
                                int64_t n_rows, int64_t max_k, int64_t n_kblocks,
                                int32_t* out_indices, int32_t* out_lens, const uint8_t* valid,
                                int64_t n_valid, uint32_t* valid_bits, hipStream_t stream) {
  return rcsa_order_split_lists(block_indices, block_indices_lens, stride_bz, stride_bh, stride_bm,
                                stride_lz, stride_lh, stride_lm, rows, n_src_rows, B, H, n_rows,
                                max_k, n_kblocks, 1, out_indices, out_lens, valid, n_valid,
                                valid_bits, stream);
}
