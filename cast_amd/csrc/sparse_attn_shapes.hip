// The attention kernel of sparse_attn_kernel.h for the block shapes other
// than D 128 with 128 x 128 blocks: head_dim 64 or 64-row / 64-key blocks.
//
// Two forms per shape, chosen as for the main shape by the query blocks of an
// XCD.  With at least two rounds of them, small workgroups of one key half
// share a compute unit (MANY): each waits for its own copies only, so the
// others' MFMAs cover the wait.  Below that, workgroups of two key halves and
// longer ring steps (FEW) walk a list in half as many steps.  us, MANY / FEW /
// the one 2-slot workgroup per compute unit they replace, 24 heads, 80 x 128
// keys a row, validity bits:
//                                1792 query rows       256 query rows
//   bf16 D 128, 64 x 128         360 / 406 / 608       84 /  85 / 122
//   bf16 D 128, 64 x 64          349 / 433 / 593       80 /  93 / 113
//   bf16 D 64, 64 x 64           215 / 203 / 263       54 /  45 /  53
//   int8 D 128, 64 x 128         298 / 355 / 522       64 /  75 / 102
//   int8 D 64, 64 x 64           202 / 214 / 261       51 /  47 /  53
// and at 8 heads x 1024 rows x 32 of 64 key blocks, int8 D 128, 64 x 128:
// 51 / 41 / 48.  bf16 D 64 keeps FEW throughout: 24 heads, FEW / MANY,
//                1792 query rows    3584 query rows
//   128 x 128    165 / 165          294 / 288
//   128 x 64     203 / 211          288 / 281
//   64 x 128     180 / 211          317 / 280
//   64 x 64      202 / 198          350 / 279
// (64-row blocks pass to MANY's side between 84 and 168 query blocks an XCD; no
// line is drawn there.)
// Validity bytes: FEW.
//
// Wavefronts per SIMD that MANY's register budget allows: as many as the
// workgroups that the LDS holds come to, three at most (159 to 170 VGPRs).  A
// bf16 ring of D 128 takes 50 KiB, so three workgroups share a compute unit: 128-row
// blocks (four wavefronts) three, 64-row blocks (two) two.  int8 rings take 38 KiB,
// four workgroups: 64-row blocks two.  D 64 rings of 19 to 38 KiB: three.
#include "sparse_attn_kernel.h"

namespace rcsa {

template <bool INT8, int D, int BM, int BN, int BNS, int NKH, int WPE>
static int launch_form(AttnArgs& a, dim3 grid, hipStream_t s) {
  constexpr int kThreads = BM / 32 * NKH * 64;
  if (a.kmask != nullptr)
    sparse_attn_kernel<INT8, D, BM, BN, BNS, NKH, true, false, WPE>
        <<<grid, dim3(kThreads), 0, s>>>(a);
  else
    sparse_attn_kernel<INT8, D, BM, BN, BNS, NKH, false, false, WPE>
        <<<grid, dim3(kThreads), 0, s>>>(a);
  return launch_status();
}

// 64-row query blocks over gathered sources, any number of them (a relay layer whose
// blocks hold at most 64 query tokens uses them for two rounds and more of query
// blocks: two frames, int8, 24 heads x 30 blocks, the relay call takes 401 us
// against 472 with 128-row blocks)
template <bool INT8>
static int launch_half_gather(AttnArgs& a, dim3 grid, hipStream_t s) {
  sparse_attn_kernel<INT8, 128, 64, 128, 32, 1, true, true, 2><<<grid, dim3(128), 0, s>>>(a);
  return launch_status();
}

template <bool INT8, int D, int BM, int BN, int BNS, int WPE>
static int launch_many(AttnArgs& a, dim3 grid, hipStream_t s) {
  sparse_attn_kernel<INT8, D, BM, BN, BNS, 1, true, false, WPE>
      <<<grid, dim3(BM / 32 * 64), 0, s>>>(a);
  return launch_status();
}

int launch_attn_shape(AttnArgs& a, bool int8, int64_t D, int64_t BM, int64_t BN, bool many,
                      dim3 grid, hipStream_t s) {
  if (a.kv_tok != nullptr)
    return int8 ? launch_half_gather<true>(a, grid, s) : launch_half_gather<false>(a, grid, s);
  many = many && a.kmask != nullptr;
#define RCSA_SHAPE(D_, BM_, BN_) if (D == D_ && BM == BM_ && BN == BN_)
  if (int8) {
    RCSA_SHAPE(128, 128, 64) return many ? launch_many<true, 128, 128, 64, 32, 3>(a, grid, s) : launch_form<true, 128, 128, 64, 64, 2, 0>(a, grid, s);
    RCSA_SHAPE(128, 64, 128) return many ? launch_many<true, 128, 64, 128, 32, 2>(a, grid, s) : launch_form<true, 128, 64, 128, 64, 2, 0>(a, grid, s);
    RCSA_SHAPE(128, 64, 64) return many ? launch_many<true, 128, 64, 64, 32, 2>(a, grid, s) : launch_form<true, 128, 64, 64, 64, 2, 0>(a, grid, s);
    RCSA_SHAPE(64, 128, 128) return many ? launch_many<true, 64, 128, 128, 64, 3>(a, grid, s) : launch_form<true, 64, 128, 128, 128, 2, 0>(a, grid, s);
    // (a 64-key step has too few K copies for the eight wavefronts of two halves)
    RCSA_SHAPE(64, 128, 64) return launch_form<true, 64, 128, 64, 64, 1, 3>(a, grid, s);
    RCSA_SHAPE(64, 64, 128) return many ? launch_many<true, 64, 64, 128, 32, 3>(a, grid, s) : launch_form<true, 64, 64, 128, 64, 2, 0>(a, grid, s);
    RCSA_SHAPE(64, 64, 64) return many ? launch_many<true, 64, 64, 64, 32, 3>(a, grid, s) : launch_form<true, 64, 64, 64, 64, 2, 0>(a, grid, s);
  } else {
    RCSA_SHAPE(128, 128, 64) return many ? launch_many<false, 128, 128, 64, 32, 3>(a, grid, s) : launch_form<false, 128, 128, 64, 64, 2, 0>(a, grid, s);
    RCSA_SHAPE(128, 64, 128) return many ? launch_many<false, 128, 64, 128, 32, 2>(a, grid, s) : launch_form<false, 128, 64, 128, 64, 2, 0>(a, grid, s);
    RCSA_SHAPE(128, 64, 64) return many ? launch_many<false, 128, 64, 64, 32, 2>(a, grid, s) : launch_form<false, 128, 64, 64, 64, 2, 0>(a, grid, s);
    RCSA_SHAPE(64, 128, 128) return launch_form<false, 64, 128, 128, 64, 2, 0>(a, grid, s);
    RCSA_SHAPE(64, 128, 64) return launch_form<false, 64, 128, 64, 64, 2, 0>(a, grid, s);
    RCSA_SHAPE(64, 64, 128) return launch_form<false, 64, 64, 128, 64, 2, 0>(a, grid, s);
    RCSA_SHAPE(64, 64, 64) return launch_form<false, 64, 64, 64, 64, 2, 0>(a, grid, s);
  }
#undef RCSA_SHAPE
  return RCSA_ERR_SHAPE;
}

}  // namespace rcsa
