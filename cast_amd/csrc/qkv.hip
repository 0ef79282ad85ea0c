// Shared int8 Q/K/V projection (gfx950): one per-token int8 quantisation of
// the activations, then int8 GEMMs with a dequantising epilogue.
//
// quant_rows_kernel: one wavefront per token row; scale = absmax / 127 (1 for
// an all-zero row), q = rne(x * 127 / absmax) clamped to [-127, 127].
//
// int8_linear_kernel: out[m][n] = bf16(bf16(acc * xs[m] * ws[n]) + bias[n]),
// acc = sum_k x[m][k] w[n][k] in int32, for up to four projections of one x.  A
// workgroup of four wavefronts, one per SIMD, computes a tile of 256 (tokens) x
// 256 (channels) or 128 x 128 with v_mfma_i32_32x32x32_i8, the weights as the A
// operand, so a lane ends up holding one token and runs of 4 consecutive
// channels.  A wavefront's quarter of 128 x 128 reads 8 operand tiles from LDS
// for 16 MFMAs: half the matrix cores' time at 128 bytes a clock (64 x 128
// quarters of eight wavefronts take three quarters of it and run at 42% of the
// matrix cores' cycles).  Both operands are staged by direct-to-LDS copies
// through a ring of 128-byte K steps (one whole line of every row); 16-byte
// chunks of each 128-byte row are XORed by (row / 2) mod 8 so the ds_read_b128
// operand reads are conflict free.  The launch is persistent: a compute unit's
// workgroups walk its XCD's tiles of all projections, and the ring runs on from
// one tile to the next.  Three projections of 3072 x 3072, one launch,
// against three launches of the eight-wavefront kernel: 38,720 tokens 1034
// against 1199 us (2.1 POP/s), 3520 tokens 92 against 155, 880 tokens (128 x 128
// tiles) 31 against 144 us.  What bounds it: the matrix cores' clock under load
// (1.9 GHz) and the epilogue, which no MFMA of the same SIMD covers.
#include <type_traits>

#include "rcsa_common.h"

#define RCSA_QKV_LDS(T, p) ((__attribute__((address_space(3))) T*)(p))

namespace rcsa {

constexpr int kQThreads = 256;       // quantiser: 4 rows per workgroup
constexpr int kGemmWaves = 4;        // 2 (tokens) x 2 (channels), one per SIMD
constexpr int kGemmThreads = kGemmWaves * kWave;
constexpr int kKS = 128;             // bytes of K per ring step (one 128-byte line per row)

typedef unsigned int v4u __attribute__((ext_vector_type(4)));

// Two floats as packed bf16 (round to nearest even), low half = a.
__device__ __forceinline__ uint32_t cvt_bf16x2(float a, float b) {
  typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
  const v2bf v = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
  return __builtin_bit_cast(uint32_t, v);
}

// Eight floats as int8 (two words).
__device__ __forceinline__ uint2 quant8(const float (&v)[8], float inv) {
  uint32_t lo = 0, hi = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    lo |= (static_cast<uint32_t>(quant_i8(v[j], inv)) & 0xffu) << (8 * j);
    hi |= (static_cast<uint32_t>(quant_i8(v[j + 4], inv)) & 0xffu) << (8 * j);
  }
  return make_uint2(lo, hi);
}

// NC > 0: rows of at most NC 512-channel chunks stay in registers between the
// two passes (all loads in flight at once, one read of x); NC == 0: any length,
// read twice.  HBM-bound: 38,720 x 3072 bf16 takes 69 us (5.2 TB/s), read twice
// 86 us.
template <typename T, int NC>
__global__ void __launch_bounds__(kQThreads)
quant_rows_kernel(const T* x, int64_t M, int64_t C, int64_t ldx, int8_t* q, float* scale) {
  const int lane = threadIdx.x % kWave;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * (kQThreads / kWave) + threadIdx.x / kWave;
  if (row >= M) return;
  const T* xr = x + row * ldx;
  int8_t* qr = q + row * C;
  float amax = 0.0f;
  if constexpr (NC > 0) {
    float v[NC][8];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int64_t c = (i * kWave + lane) * 8;
      if (c < C) {
        Vec8<T>::load(xr + c, v[i]);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] = 0.0f;
      }
    }
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[i][j]));
    amax = wave_max(amax);
    const float inv = amax > 0.0f ? 127.0f / amax : 1.0f;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int64_t c = (i * kWave + lane) * 8;
      if (c < C) *reinterpret_cast<uint2*>(qr + c) = quant8(v[i], inv);
    }
  } else {
    for (int64_t c = lane * 8; c < C; c += kWave * 8) {
      float v[8];
      Vec8<T>::load(xr + c, v);
#pragma unroll
      for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
    }
    amax = wave_max(amax);
    const float inv = amax > 0.0f ? 127.0f / amax : 1.0f;
    for (int64_t c = lane * 8; c < C; c += kWave * 8) {
      float v[8];
      Vec8<T>::load(xr + c, v);
      *reinterpret_cast<uint2*>(qr + c) = quant8(v, inv);
    }
  }
  if (lane == 0) scale[row] = amax > 0.0f ? amax / 127.0f : 1.0f;
}

constexpr int kMaxLinear = 4;  // projections of one launch

// The projections of one input: out_g[m][n] for g < n_lin, n < N_g.
struct LinearArgs {
  const int8_t* x;      // [M, K]
  const float* xs;      // [M]
  int64_t M, K;
  int32_t n_lin;
  int32_t steps;        // K steps of a tile, padded to the ring's slots with empty ones
  int64_t tiles[kMaxLinear + 1];  // first tile of each projection; [n_lin]: all tiles
  const int8_t* w[kMaxLinear];    // [N, K]
  const float* ws[kMaxLinear];    // [N]
  const u16* bias[kMaxLinear];    // [N] bf16 or NULL
  void* out[kMaxLinear];          // [M, ldo], bf16 or the same values as fp32
  int64_t N[kMaxLinear], ldo[kMaxLinear];
};

constexpr int kQkvRsrc3 = 0x00020000;  // raw untyped buffer, 32-bit data format

__device__ __forceinline__ void dma16(const int8_t* base, int bytes, uint32_t voff, int soff,
                                      char* dst) {
  const __amdgpu_buffer_rsrc_t r =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(base), 0, bytes, kQkvRsrc3);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, RCSA_QKV_LDS(void, dst), 16, voff, soff, 0, 0);
}

// chunk XOR of a 128-byte row: (row / 2) mod 8
__device__ __forceinline__ int qkv_swz(int row) { return (row >> 1) & 7; }

// Wait until at most N copies of this wavefront are outstanding and its LDS
// reads have returned, then barrier: unlike __syncthreads() the younger copies
// stay in flight.
template <int N>
__device__ __forceinline__ void lin_wait_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// A workgroup tile of 4 wavefronts (2 along tokens x 2 along channels), each
// T x T MFMA tiles of 32 x 32, over a ring of two K steps.
// WGS workgroups share a compute unit.
template <int T_, int WGS_>
struct LinTile {
  static constexpr int T = T_, WGS = WGS_;
  static constexpr int SLOTS = 2;                      // (the ring is unrolled by hand)
  static constexpr int B = 2 * 32 * T;                 // tokens and channels of a tile
  static constexpr int OB = B * kKS;                   // bytes of one operand's step
  static constexpr int U = OB / 1024 / kGemmWaves;     // 1 KiB copies per wavefront and operand
  static constexpr int OPS = 2 * U;                    // copies per wavefront and step
  static constexpr int KS = kKS / 32;                  // MFMA k-steps per ring step
  static constexpr int CH = 8;                         // 16-byte chunks of an epilogue row
  static constexpr int ROWS = 32 * CH * 16;            // 32 epilogue rows of a wavefront
  static constexpr int EN = WGS == 1 ? 2 : 1;          // in one or two buffers
  static constexpr int EB = EN * ROWS;
  static_assert((SLOTS - 2) * OPS < 64, "vmcnt range");
  static_assert(WGS * (SLOTS * 2 * OB + kGemmWaves * EB) <= 160 * 1024, "LDS of a compute unit");
};

using BigTile = LinTile<4, 1>;  // 256 x 256, 64 KiB steps
// 128 x 128, 32 KiB steps: two workgroups fill each other's waits (three
// projections of 880 tokens 31.4 us against 33.1 with one of four slots, 2640
// tokens 81 against 87)
using MidTile = LinTile<2, 2>;

// Where a tile's operands are and where its outputs go.
struct TileSrc {
  const int8_t* xb;
  const int8_t* wb;
  int xbytes, wbytes;
  int32_t g, m0, n0;
};

// Tile `work` of the launch.  Consecutive tiles walk groups of kGroupM token
// blocks for one channel block, then the next, so the 32 workgroups of an XCD
// share 4 token blocks and 8 weight blocks in its L2.
template <class L>
__device__ __forceinline__ TileSrc tile_src(const LinearArgs& a, uint32_t work) {
  constexpr uint32_t kGroupM = 4;
  int32_t g = 0;
#pragma unroll
  for (int i = 1; i < kMaxLinear; ++i)
    if (i < a.n_lin && work >= static_cast<uint32_t>(a.tiles[i])) g = i;
  work -= static_cast<uint32_t>(a.tiles[g]);
  const uint32_t n_m = static_cast<uint32_t>((a.M + L::B - 1) / L::B);
  const uint32_t n_n = static_cast<uint32_t>(a.N[g]) / L::B;
  const uint32_t group = work / (kGroupM * n_n), in_group = work % (kGroupM * n_n);
  const uint32_t group_m = n_m - group * kGroupM < kGroupM ? n_m - group * kGroupM : kGroupM;
  const int32_t m0 = static_cast<int32_t>((group * kGroupM + in_group % group_m) * L::B);
  const int32_t n0 = static_cast<int32_t>(in_group / group_m * L::B);
  const int64_t rows = a.M - m0 < L::B ? a.M - m0 : L::B;  // rows past M read as zeros
  return {a.x + m0 * a.K, a.w[g] + n0 * a.K, static_cast<int>(rows * a.K),
          static_cast<int>(L::B * a.K), g, m0, n0};
}

// L::WGS persistent workgroups per compute unit: workgroup j of XCD x takes the
// XCD's tiles j, j + per_wg, ...  The copy ring runs on from tile to tile, so a
// tile's first steps land during the previous tile's last MFMAs and epilogue.
template <class L, bool OUT32>
__global__ void __launch_bounds__(kGemmThreads) __attribute__((amdgpu_waves_per_eu(L::WGS, L::WGS)))
int8_linear_kernel(LinearArgs a, int32_t per_wg, int32_t per_xcd) {
  constexpr int T = L::T, SLOTS = L::SLOTS, KS = L::KS;
  // (slots in arrays of their own: the compiler then knows that reads of one do
  // not alias the copies in flight into the others)
  __shared__ __attribute__((aligned(1024))) char s_0[2 * L::OB];
  __shared__ __attribute__((aligned(1024))) char s_1[2 * L::OB];
  __shared__ __attribute__((aligned(1024))) char s_e[kGemmWaves * L::EB];
  const int32_t first = static_cast<int32_t>(blockIdx.x % kNumXcd) * per_xcd;
  const int32_t all = static_cast<int32_t>(a.tiles[a.n_lin]);
  const int32_t end = first + per_xcd < all ? first + per_xcd : all;
  int32_t item = first + static_cast<int32_t>(blockIdx.x / kNumXcd);
  if (item >= end) return;

  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wm = wave & 1, wn = wave >> 1, hf = lane >> 5, li = lane & 31;
  // each operand's step is units of 1 KiB (8 rows of 128 bytes); lane l lands at
  // row 8 u + l / 8, chunk l % 8 of its unit and loads the chunk that the
  // swizzle puts there (the same rows of both operands)
  uint32_t off[L::U];
#pragma unroll
  for (int i = 0; i < L::U; ++i) {
    const int r = (wave * L::U + i) * 8 + lane / 8;
    off[i] = static_cast<uint32_t>(r * a.K + ((lane & 7) ^ qkv_swz(r)) * 16);
  }
  // Row 32 i + li of a wavefront's rows has the chunk swizzle (li / 2) mod 8 for
  // every i, so its 32-row tiles sit 4 KiB apart and one lane offset per k-step
  // serves them all (the 4 KiB steps become instruction immediates).
  int xk[KS], wk[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int c = ((ks * 2 + hf) ^ qkv_swz(li)) * 16;
    xk[ks] = (wm * 32 * T + li) * kKS + c;
    wk[ks] = L::OB + (wn * 32 * T + li) * kKS + c;
  }
  const int real_steps = static_cast<int>(a.K / kKS), steps = a.steps;

  // the copies of k-step s of a tile (none of the bytes of a step past K: zeros)
  auto stage = [&](const TileSrc& t, int s, char* dst) __attribute__((always_inline)) {
    const int xbytes = s < real_steps ? t.xbytes : 0, wbytes = s < real_steps ? t.wbytes : 0;
    const int k0 = s * kKS;
#pragma unroll
    for (int i = 0; i < L::U; ++i)
      dma16(t.xb, xbytes, off[i], k0, dst + (wave * L::U + i) * 1024);
#pragma unroll
    for (int i = 0; i < L::U; ++i)
      dma16(t.wb, wbytes, off[i], k0, dst + L::OB + (wave * L::U + i) * 1024);
  };
  v4i xf[2][T], wf[2][T];
  auto read = [&](const char* slot, auto ks_c, auto set_c) __attribute__((always_inline)) {
    constexpr int ks = decltype(ks_c)::value, set = decltype(set_c)::value;
#pragma unroll
    for (int i = 0; i < T; ++i)
      xf[set][i] = *reinterpret_cast<const v4i*>(slot + xk[ks] + i * 32 * kKS);
#pragma unroll
    for (int i = 0; i < T; ++i)
      wf[set][i] = *reinterpret_cast<const v4i*>(slot + wk[ks] + i * 32 * kKS);
  };
  v16i acc[T][T];  // [channel tile][token tile]
  auto mfma = [&](auto set_c) __attribute__((always_inline)) {
    constexpr int set = decltype(set_c)::value;
#pragma unroll
    for (int n = 0; n < T; ++n)
#pragma unroll
      for (int m = 0; m < T; ++m)
        acc[n][m] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf[set][n], xf[set][m], acc[n][m],
                                                          0, 0, 0);
  };
  using std::integral_constant;
  // Step s in slot `cur`: each k-step's operands are read during the MFMAs of
  // the one before.  Before the last k-step every wavefront has read the slot
  // and step s + 1 has landed (one barrier): the slot is refilled with step
  // s + SLOTS of the stream and the next slot's first operands are read beside
  // the last MFMAs.
  auto step = [&](char* cur, const char* nxt, const TileSrc& ft,
                  int fs) __attribute__((always_inline)) {
    read(cur, integral_constant<int, 1>{}, integral_constant<int, 1>{});
    mfma(integral_constant<int, 0>{});
    read(cur, integral_constant<int, 2>{}, integral_constant<int, 0>{});
    mfma(integral_constant<int, 1>{});
    read(cur, integral_constant<int, 3>{}, integral_constant<int, 1>{});
    mfma(integral_constant<int, 0>{});
    // (operand reads first, then spread the rest of each group over the MFMAs)
#pragma unroll
    for (int q = 0; q < 3; ++q) {
#pragma unroll
      for (int i = 0; i < 2 * T; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, T * T / (2 * T), 0);
      }
    }
    lin_wait_barrier<(SLOTS - 2) * L::OPS>();
    stage(ft, fs, cur);
    read(nxt, integral_constant<int, 0>{}, integral_constant<int, 0>{});
    mfma(integral_constant<int, 1>{});
#pragma unroll
    for (int i = 0; i < 2 * T; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, T * T / (2 * T), 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x020, L::OPS / (2 * T), 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // Epilogue: a lane holds token li of each 32-token tile and channels
  // 8 g + 4 hf + (0..3) of each 32-channel tile; lanes l and l + 32 swap halves
  // (8 consecutive channels each), and 32 tokens x 64 channels at a time go
  // through the wavefront's own LDS rows so that stores write whole lines.
  auto store = [&](const TileSrc& t) __attribute__((always_inline)) {
    char* const eb = s_e + wave * L::EB;
    const u16* const bias = a.bias[t.g];
    const u16* const bias_or_ws =
        bias != nullptr ? bias : reinterpret_cast<const u16*>(a.ws[t.g]);
    uint32_t keep = bias != nullptr ? 0xffffffffu : 0u;
    asm volatile("" : "+v"(keep));  // (masks, not sixteen branches)
    const uint32_t none = ~keep & 0x80008000u;
    const int64_t nw = t.n0 + wn * 32 * T, mw = t.m0 + wm * 32 * T;
    float xs[T];
#pragma unroll
    for (int m = 0; m < T; ++m) {
      const int64_t r = mw + m * 32 + li;
      xs[m] = a.xs[r < a.M ? r : a.M - 1];
    }
    // stores through a buffer that ends after the tile's last row: rows past M
    // are dropped
    constexpr uint32_t kOutBytes = OUT32 ? 4 : 2;
    const uint32_t row_bytes = static_cast<uint32_t>(a.ldo[t.g]) * kOutBytes;
    const int64_t left = a.M - t.m0;
    const uint32_t rows_left = static_cast<uint32_t>(left < L::B ? left : L::B);
    const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(
        static_cast<char*>(a.out[t.g]) + static_cast<int64_t>(t.m0) * row_bytes, 0, static_cast<int>(rows_left * row_bytes), kQkvRsrc3);
    const uint32_t lane_out = (lane / L::CH) * row_bytes + (lane % L::CH) * 8u * kOutBytes +
                              static_cast<uint32_t>(nw) * kOutBytes;
#pragma unroll
    for (int np = 0; np < T / 2; ++np) {  // 64 channels: whole 128-byte lines
      float4 ws[2][4];
      uint2 bb[2][4];
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int64_t c = nw + (2 * np + n) * 32 + 8 * g + 4 * hf;
          ws[n][g] = *reinterpret_cast<const float4*>(a.ws[t.g] + c);
          // (no bias: -0, which adds nothing to any value; the load then reads
          // the scales, which are there and long enough)
          const uint2 b = *reinterpret_cast<const uint2*>(bias_or_ws + c);
          bb[n][g] = make_uint2((b.x & keep) | none, (b.y & keep) | none);
        }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < T; ++m) {
        char* const rows = eb + (m & (L::EN - 1)) * L::ROWS;
        // (the accumulators leave their AGPRs here, not all before the epilogue)
        asm volatile("" : "+a"(acc[2 * np][m]), "+a"(acc[2 * np + 1][m]));
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            uint32_t pk[2][2];
#pragma unroll
            for (int gg = 0; gg < 2; ++gg) {
              const int g = 2 * p + gg;
              const float wv[4] = {ws[n][g].x, ws[n][g].y, ws[n][g].z, ws[n][g].w};
              float y[4];
#pragma unroll
              for (int e = 0; e < 4; ++e)
                y[e] = static_cast<float>(acc[2 * np + n][m][4 * g + e]) * xs[m] * wv[e];
              pk[gg][0] = cvt_bf16x2(y[0], y[1]);
              pk[gg][1] = cvt_bf16x2(y[2], y[3]);
              const uint32_t bw[2] = {bb[n][g].x, bb[n][g].y};
#pragma unroll
              for (int w = 0; w < 2; ++w)
                pk[gg][w] = cvt_bf16x2(
                    __uint_as_float(pk[gg][w] << 16) + __uint_as_float(bw[w] << 16),
                    __uint_as_float(pk[gg][w] & 0xffff0000u) +
                        __uint_as_float(bw[w] & 0xffff0000u));
            }
            // lane l (half 0) keeps channels 8(2p) + 0..3 and takes + 4..7 from
            // lane l + 32, which keeps 8(2p + 1) + 4..7 and takes + 0..3
            v4u st;
#pragma unroll
            for (int w = 0; w < 2; ++w) {
              const auto r = __builtin_amdgcn_permlane32_swap(pk[0][w], pk[1][w], false, false);
              st[w] = r[0];
              st[2 + w] = r[1];
            }
            const int c = n * 4 + 2 * p + hf;
            *reinterpret_cast<v4u*>(rows + (li * L::CH + (c ^ (li & (L::CH - 1)))) * 16) = st;
          }
        // (the rows are this wavefront's own: its LDS operations stay in order)
#pragma unroll
        for (int i = 0; i < 32 * L::CH / kWave; ++i) {
          const int r = i * (kWave / L::CH) + lane / L::CH, c = lane % L::CH;
          const v4u v = *reinterpret_cast<const v4u*>(
              rows + (r * L::CH + (c ^ (r & (L::CH - 1)))) * 16);
          const uint32_t row = wm * 32 * T + m * 32 + i * (kWave / L::CH);
          // (no scalar offset: with one, the compiler lets the next instruction
          // overwrite the registers that a 16-byte store is still reading)
          const int voff = static_cast<int>(row * row_bytes + lane_out + np * 64u * kOutBytes);
          if constexpr (OUT32) {
            const v4u lo = {v[0] << 16, v[0] & 0xffff0000u, v[1] << 16, v[1] & 0xffff0000u};
            const v4u hi = {v[2] << 16, v[2] & 0xffff0000u, v[3] << 16, v[3] & 0xffff0000u};
            __builtin_amdgcn_raw_buffer_store_b128(lo, out, voff, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b128(hi, out, voff + 16, 0, 0);
          } else {
            __builtin_amdgcn_raw_buffer_store_b128(v, out, voff, 0, 0);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  TileSrc cur = tile_src<L>(a, static_cast<uint32_t>(item));
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) {
    stage(cur, i, i == 0 ? s_0 : s_1);
    __builtin_amdgcn_sched_barrier(0);  // the steps' copies stay in order
  }
  lin_wait_barrier<(SLOTS - 1) * L::OPS>();
  read(s_0, integral_constant<int, 0>{}, integral_constant<int, 0>{});
  while (true) {
#pragma unroll
    for (int n = 0; n < T; ++n)
#pragma unroll
      for (int m = 0; m < T; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[n][m][r] = 0;
    const int32_t next = item + per_wg;
    const bool has_next = next < end;
    TileSrc nt = has_next ? tile_src<L>(a, static_cast<uint32_t>(next)) : cur;
    if (!has_next) nt.xbytes = nt.wbytes = 0;  // the last fills read nothing
    int s = 0;
    do {  // (steps >= SLOTS)
      const bool last = s + SLOTS >= steps;  // refill with the next tile's first steps
      TileSrc ft = cur;
      ft.xb = last ? nt.xb : cur.xb;
      ft.wb = last ? nt.wb : cur.wb;
      ft.xbytes = last ? nt.xbytes : cur.xbytes;
      ft.wbytes = last ? nt.wbytes : cur.wbytes;
      const int fs = last ? 0 : s + SLOTS;
      step(s_0, s_1, ft, fs);
      step(s_1, s_0, ft, fs + 1);
      s += SLOTS;
    } while (s < steps);
    store(cur);
    if (!has_next) break;
    item = next;
    cur = nt;
  }
  // the trailing copies (empty ranges) land before the slots are freed
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

}  // namespace rcsa

using namespace rcsa;

template <typename T>
static void launch_quant_rows(const void* x, int64_t M, int64_t C, int64_t ldx, int8_t* q,
                              float* scale, hipStream_t stream) {
  const int64_t rows_per = kQThreads / kWave;
  const dim3 grid(static_cast<unsigned>((M + rows_per - 1) / rows_per)), block(kQThreads);
  const T* xt = static_cast<const T*>(x);
  const int64_t chunks = (C + 511) / 512;
  if (chunks <= 2) quant_rows_kernel<T, 2><<<grid, block, 0, stream>>>(xt, M, C, ldx, q, scale);
  else if (chunks <= 4) quant_rows_kernel<T, 4><<<grid, block, 0, stream>>>(xt, M, C, ldx, q, scale);
  else if (chunks <= 6) quant_rows_kernel<T, 6><<<grid, block, 0, stream>>>(xt, M, C, ldx, q, scale);
  else if (chunks <= 10) quant_rows_kernel<T, 10><<<grid, block, 0, stream>>>(xt, M, C, ldx, q, scale);
  else quant_rows_kernel<T, 0><<<grid, block, 0, stream>>>(xt, M, C, ldx, q, scale);
}

extern "C" int rcsa_quantize_rows_int8(const void* x, int dtype, int64_t M, int64_t C, int64_t ldx,
                                       int8_t* q, float* scale, hipStream_t stream) {
  if (!x || !q || !scale) return RCSA_ERR_NULL;
  if (M <= 0 || C <= 0 || C % 8 || ldx < C || ldx % 8) return RCSA_ERR_SHAPE;
  if ((reinterpret_cast<uintptr_t>(x) & 15u) || (reinterpret_cast<uintptr_t>(q) & 7u))
    return RCSA_ERR_ALIGN;
  if (dtype == RCSA_BF16) launch_quant_rows<u16>(x, M, C, ldx, q, scale, stream);
  else if (dtype == RCSA_F32) launch_quant_rows<float>(x, M, C, ldx, q, scale, stream);
  else return RCSA_ERR_DTYPE;
  return launch_status();
}

// Compute units of the current device (256 when it cannot be read).
static int64_t device_cus() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus < kNumXcd)
    return 256;
  return cus;
}

template <class L>
static int64_t count_tiles(LinearArgs& a) {
  a.tiles[0] = 0;
  for (int g = 0; g < a.n_lin; ++g)
    a.tiles[g + 1] = a.tiles[g] + (a.M + L::B - 1) / L::B * (a.N[g] / L::B);
  return a.tiles[a.n_lin];
}

template <class L>
static int launch_linear(LinearArgs& a, int64_t cus, bool out_f32, hipStream_t stream) {
  const int64_t tiles = count_tiles<L>(a);
  if (tiles >= (int64_t{1} << 30)) return RCSA_ERR_SHAPE;
  a.steps = static_cast<int32_t>((a.K / kKS + L::SLOTS - 1) / L::SLOTS * L::SLOTS);
  // the compute units' workgroups, the same number on every XCD
  const int64_t per_xcd = (tiles + kNumXcd - 1) / kNumXcd;
  const int64_t slots = cus / kNumXcd * L::WGS;
  const int64_t per_wg = per_xcd < slots ? per_xcd : slots;
  const dim3 grid(static_cast<unsigned>(per_wg * kNumXcd)), block(kGemmThreads);
  const int32_t wg = static_cast<int32_t>(per_wg), px = static_cast<int32_t>(per_xcd);
  if (out_f32) int8_linear_kernel<L, true><<<grid, block, 0, stream>>>(a, wg, px);
  else int8_linear_kernel<L, false><<<grid, block, 0, stream>>>(a, wg, px);
  return launch_status();
}

extern "C" int rcsa_int8_linear_group(const int8_t* x, const float* x_scale, int64_t n_linear,
                                      const int8_t* const* w, const float* const* w_scale,
                                      const void* const* bias, const int64_t* N,
                                      void* const* out, const int64_t* ldo, int out_f32,
                                      int64_t M, int64_t K, hipStream_t stream) {
  if (!x || !x_scale || !w || !w_scale || !bias || !N || !out || !ldo) return RCSA_ERR_NULL;
  if (n_linear <= 0 || n_linear > kMaxLinear || M <= 0 || M >= (int64_t{1} << 31) - 256 ||
      K <= 0 || K % kKS)
    return RCSA_ERR_SHAPE;
  // the copies address a tile with 32-bit offsets
  if (static_cast<int64_t>(BigTile::B) * K >= (int64_t{1} << 31)) return RCSA_ERR_SHAPE;
  if (reinterpret_cast<uintptr_t>(x) & 15u) return RCSA_ERR_ALIGN;
  LinearArgs a{};
  a.x = x;
  a.xs = x_scale;
  a.M = M;
  a.K = K;
  a.n_lin = static_cast<int32_t>(n_linear);
  for (int g = 0; g < a.n_lin; ++g) {
    if (!w[g] || !w_scale[g] || !out[g]) return RCSA_ERR_NULL;
    if (N[g] <= 0 || N[g] % BigTile::B || ldo[g] < N[g] || ldo[g] % 4) return RCSA_ERR_SHAPE;
    if ((reinterpret_cast<uintptr_t>(w[g]) & 15u) ||
        (reinterpret_cast<uintptr_t>(w_scale[g]) & 15u) ||
        (reinterpret_cast<uintptr_t>(out[g]) & 7u) || (reinterpret_cast<uintptr_t>(bias[g]) & 7u))
      return RCSA_ERR_ALIGN;
    a.w[g] = w[g];
    a.ws[g] = w_scale[g];
    a.bias[g] = static_cast<const u16*>(bias[g]);
    a.out[g] = out[g];
    a.N[g] = N[g];
    a.ldo[g] = ldo[g];
  }
  // The stores address a tile's rows with offsets below 2^31.  Rows 8 MiB and more
  // apart (so they are few) go one by one, in parts of a row.
  constexpr int64_t kFarBytes = (int64_t{1} << 31) / BigTile::B, kPart = kFarBytes / 8;
  const int64_t elt = out_f32 != 0 ? 4 : 2;
  bool far = false;
  for (int g = 0; g < a.n_lin; ++g) far = far || ldo[g] * elt >= kFarBytes;
  if (far) {
    for (int g = 0; g < a.n_lin; ++g)
      for (int64_t r = 0; r < M; ++r)
        for (int64_t n = 0; n < N[g]; n += kPart) {
          const int64_t part = N[g] - n < kPart ? N[g] - n : kPart;
          const int8_t* const wn = w[g] + n * K;
          const float* const wsn = w_scale[g] + n;
          const void* const bn = bias[g] ? static_cast<const char*>(bias[g]) + n * 2 : nullptr;
          void* const on = static_cast<char*>(out[g]) + (r * ldo[g] + n) * elt;
          const int st = rcsa_int8_linear_group(x + r * K, x_scale + r, 1, &wn, &wsn, &bn, &part,
                                                &on, &part, out_f32, 1, K, stream);
          if (st != RCSA_OK) return st;
        }
    return RCSA_OK;
  }
  // The tile size that needs less time for its whole rounds: a round of 128 x 128
  // tiles takes 5/16 of a round of 256 x 256 tiles (14 and 44 us at K 3072; three
  // projections of 880 tokens: 2 rounds, 31 us, against 1 round, 44 us; of 1760
  // tokens: 4 rounds, 59 us, against 1 round, 51 us).
  const int64_t cus = device_cus();
  const int64_t big = (count_tiles<BigTile>(a) + cus - 1) / cus * 16;
  const int64_t mid = (count_tiles<MidTile>(a) + cus - 1) / cus * 5;
  return big <= mid ? launch_linear<BigTile>(a, cus, out_f32 != 0, stream)
                    : launch_linear<MidTile>(a, cus, out_f32 != 0, stream);
}

extern "C" int rcsa_int8_linear(const int8_t* x, const float* x_scale, const int8_t* w,
                                const float* w_scale, const void* bias, int64_t M, int64_t N,
                                int64_t K, void* out, int64_t ldo, hipStream_t stream) {
  return rcsa_int8_linear_group(x, x_scale, 1, &w, &w_scale, &bias, &N, &out, &ldo, 0, M, K,
                                stream);
}
