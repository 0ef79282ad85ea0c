// Fixed-budget top-k selection of one (head, query block) row per wavefront,
// shared by rcsa_select_topk and the fused key-quantiser + selection launch.
//
// Forced columns rank before the others; inside either class a column's 32-bit
// value orders it: the order-preserving image of its fp32 score (0: not allowed,
// never selected), ties to the lower index.  The forced columns fill the row
// first, so only one class has a cut; its k-th largest value T is found by a
// bisection of the value's bits, whose counts are wavefront ballots + popcounts
// (scalar unit, no LDS, no shuffles), ended as soon as a prefix counts exactly k.
// The selected set is {value > T} and the first of the columns at T; it is
// written in ascending column order by ballot prefix counts, or in rank order.
// (32-bit compares of one class instead of 50 steps over 64-bit keys of both:
// 24 x 330 rows of 330 columns, rank order, take 30 against 37 us, index order
// 24 x 300 rows of 300 columns 16 us against 38 in rank order before.)
#pragma once
#include "rcsa_common.h"

namespace rcsa {


struct SelArgs {
  const float* score;
  int64_t n_rows;       // n_bh * n_q
  int64_t n_q, n_k;
  const int32_t* row_k;
  int64_t row_k_stride_bh;
  int64_t k_fixed;
  const uint8_t* forced;
  const uint8_t* allowed;
  int64_t mask_stride_bh;
  int32_t* indices;
  int64_t max_k;
  int32_t* counts;
  // forced columns rank among themselves by fl(score + 1e6) (RCSA_ORDER_RANK_LOCAL)
  bool coarse_forced;
  // MIXED: rank order for rows [x xcd_items + xcd_direct, (x + 1) xcd_items) only, index
  // order for the others (RCSA_ORDER_SPLIT)
  int64_t xcd_items, xcd_direct;
};

constexpr int kSelWaves = 4;

// Value of column j of a row (0 when it is not allowed), and whether it is forced.
__device__ __forceinline__ uint32_t column_value(const SelArgs& a, int64_t row, int64_t bh,
                                                 int64_t i, int64_t j, bool& forced) {
  forced = false;
  if (j >= a.n_k) return 0u;
  float s = a.score[row * a.n_k + j];
  const int64_t moff = bh * a.mask_stride_bh + i * a.n_k + j;
  if (a.allowed && a.allowed[moff] == 0) return 0u;
  forced = a.forced && a.forced[moff] != 0;
  if (a.coarse_forced && forced) s = (s + 1e6f) - 1e6f;
  if (s == 0.0f) s = 0.0f;                          // -0 and +0: one image
  if (s != s) s = __uint_as_float(0x7fc00000u);     // every NaN ranks highest
  const uint32_t u = __float_as_uint(s);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);  // never 0: NaN is positive here
}

// LDS words of a wavefront's rank lists: values (both classes padded to whole
// 16-byte groups), then 16-bit columns.
__host__ __device__ __forceinline__ int64_t rank_slots(int64_t max_k) {
  return (max_k + 8 + 3) / 4 * 4;
}
constexpr int64_t kRankSlotBytes = 6;

// Rank order of one class of n selected columns (ascending in index): values at
// v, columns at c; out[rank] = column.  Every lane ranks two columns at a time
// against all of them, four per LDS read.
__device__ __forceinline__ void write_ranked(const uint32_t* v, const uint16_t* c, int64_t n,
                                             int32_t* out, int lane) {
  for (int64_t e0 = 0; e0 < n; e0 += 2 * kWave) {
    const int64_t ea = e0 + lane, eb = ea + kWave;
    const uint32_t ma = ea < n ? v[ea] : 0xffffffffu, mb = eb < n ? v[eb] : 0xffffffffu;
    int32_t ra = 0, rb = 0;
    for (int64_t f = 0; f < n; f += 4) {
      const uint4 w = *reinterpret_cast<const uint4*>(v + f);
      const uint32_t wv[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int t = 0; t < 4; ++t) {  // an equal value earlier in the class ranks first
        ra += wv[t] > ma - static_cast<uint32_t>(f + t < ea);
        rb += wv[t] > mb - static_cast<uint32_t>(f + t < eb);
      }
    }
    if (ea < n) out[ra] = c[ea];
    if (eb < n) out[rb] = c[eb];
  }
}

// PER > 0: values held in registers (PER per lane, n_k <= 64 * PER).
// PER == 0: values recomputed from memory on every pass (any n_k <= 65536).
template <int PER, bool RANK, bool MIXED = false>
__device__ __forceinline__ void select_rows(const SelArgs& a, int64_t block, char* s_rank) {
  static_assert(PER <= 32, "one forced bit per pass");
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int64_t row = block * kSelWaves + wave;
  if (row >= a.n_rows) return;  // whole wavefront exits together
  const int64_t bh = row / a.n_q, i = row % a.n_q;
  const int passes = PER > 0 ? PER : static_cast<int>((a.n_k + kWave - 1) / kWave);

  uint32_t vals[PER > 0 ? PER : 1];
  uint32_t fbits = 0;  // this lane's forced columns (PER > 0)
  int n_allowed = 0, n_forced = 0;
#pragma unroll PER > 0 ? PER : 1
  for (int p = 0; p < passes; ++p) {
    bool f;
    const uint32_t v = column_value(a, row, bh, i, lane + int64_t{kWave} * p, f);
    f = f && v != 0;
    if (PER > 0) {
      vals[p] = v;
      fbits |= static_cast<uint32_t>(f) << p;
    }
    n_allowed += __popcll(__ballot(v != 0));
    n_forced += __popcll(__ballot(f));
  }
  int64_t k = a.row_k ? static_cast<int64_t>(a.row_k[bh * a.row_k_stride_bh + i]) : a.k_fixed;
  k = k < 0 ? 0 : (k > a.max_k ? a.max_k : k);
  const int k_eff = k < n_allowed ? static_cast<int>(k) : n_allowed;
  int32_t* out = a.indices + row * a.max_k;

  if (k_eff > 0) {
    const bool cut_forced = k_eff <= n_forced;  // the class with the cut
    const int kk = cut_forced ? k_eff : k_eff - n_forced;
    // a column's value and class in pass p
    auto column = [&](int p, bool& f) __attribute__((always_inline)) -> uint32_t {
      if constexpr (PER > 0) {
        f = (fbits >> p) & 1u;
        return vals[p];
      } else {
        const uint32_t v = column_value(a, row, bh, i, lane + int64_t{kWave} * p, f);
        f = f && v != 0;
        return v;
      }
    };
    uint32_t cls[PER > 0 ? PER : 1];  // the cut class's values, 0 for the others
    if constexpr (PER > 0) {
#pragma unroll
      for (int p = 0; p < PER; ++p) {
        bool f;
        const uint32_t v = column(p, f);
        cls[p] = f == cut_forced ? v : 0u;
      }
    }
    auto cut_value = [&](int p) __attribute__((always_inline)) -> uint32_t {
      if constexpr (PER > 0) {
        return cls[p];
      } else {
        bool f;
        const uint32_t v = column(p, f);
        return f == cut_forced ? v : 0u;
      }
    };
    uint32_t thr = 0;
    for (int bit = 31; bit >= 0; --bit) {
      const uint32_t cand = thr | (1u << bit);
      int cnt = 0;
#pragma unroll PER > 0 ? PER : 1
      for (int p = 0; p < passes; ++p) cnt += __popcll(__ballot(cut_value(p) >= cand));
      if (cnt >= kk) thr = cand;
      if (cnt == kk) break;
    }
    int above = 0;
#pragma unroll PER > 0 ? PER : 1
    for (int p = 0; p < passes; ++p) above += __popcll(__ballot(cut_value(p) > thr));
    const int ties = kk - above;  // columns at the threshold to take, lowest first

    const bool ranked = RANK && (!MIXED || row % a.xcd_items >= a.xcd_direct);
    const uint64_t lt_mask = (1ull << lane) - 1ull;
    const int64_t slots = RANK ? rank_slots(a.max_k) : 0;
    uint32_t* rv = RANK ? reinterpret_cast<uint32_t*>(s_rank) + wave * slots : nullptr;
    uint16_t* rc = RANK ? reinterpret_cast<uint16_t*>(s_rank + kSelWaves * slots * 4) +
                              wave * slots : nullptr;
    const int n_a = cut_forced ? k_eff : n_forced;  // selected forced columns
    const int b0 = (n_a + 3) / 4 * 4;               // the others' first rank slot
    int base = 0, base_f = 0, taken = 0;
#pragma unroll PER > 0 ? PER : 1
    for (int p = 0; p < passes; ++p) {
      const int64_t j = lane + int64_t{kWave} * p;
      bool f;
      const uint32_t v = column(p, f);
      const bool in_cut = f == cut_forced && v != 0;
      const uint64_t eq = __ballot(in_cut && v == thr);
      const bool sel = (in_cut && (v > thr || (v == thr && taken + __popcll(eq & lt_mask) < ties)))
                       || (f && !cut_forced);
      taken += __popcll(eq);
      const uint64_t m = __ballot(sel);
      if (ranked) {
        const uint64_t mf = __ballot(sel && f);
        if (sel) {
          const int s = f ? base_f + __popcll(mf & lt_mask)
                          : b0 + (base - base_f) + __popcll(m & ~mf & lt_mask);
          rv[s] = v;
          rc[s] = static_cast<uint16_t>(j);
        }
        base_f += __popcll(mf);
      } else if (sel) {
        out[base + __popcll(m & lt_mask)] = static_cast<int32_t>(j);
      }
      base += __popcll(m);
    }
    if (ranked) {
      // the padding of both classes' last groups outranks nothing
      const int n_b = k_eff - n_a;
      if (lane < b0 - n_a) rv[n_a + lane] = 0;
      if (lane < (4 - n_b % 4) % 4) rv[b0 + n_b + lane] = 0;
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      write_ranked(rv, rc, n_a, out, lane);
      write_ranked(rv + b0, rc + b0, n_b, out + n_a, lane);
    }
  }
  for (int64_t s = k_eff + lane; s < a.max_k; s += kWave) out[s] = -1;
  if (lane == 0) a.counts[row] = k_eff;
}

}  // namespace rcsa
