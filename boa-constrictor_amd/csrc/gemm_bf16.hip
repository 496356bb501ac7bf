// bf16 GEMM on CDNA4 matrix cores with the codec's fused epilogues:
//
//   C[m][n] = act(sum_k X[m][k] * W[n][k] + bias[n]) (+ R[m][n])
//
// X and W are bf16; accumulation is fp32 in v_mfma_f32_16x16x32_bf16.  W is
// stored n-major ([N_pad][K], k contiguous) so that both operands of an MFMA
// are 16-byte rows.  Every output is the chain of MFMAs over k-steps of 32 in
// ascending order from 0, with k = 32 s + 8 g + e in operand slot (g, e) of
// lane (i, g); the decode-step GEMM issues the same chain, so the compress and
// decompress passes produce identical logits.  The epilogue (bias, activation,
// residual) is the fp32 one; the output is stored in fp32 or bf16, and the
// last layer's FF2 can also store a bf16 copy of its fp32 output (head1's
// input).
//
// Operand roles as in the fp32 kernel: weights are the A operand (16 n-rows),
// activations the B operand (16 m-columns); a lane's accumulators are 4
// consecutive n of one row m.  LDS: [rows][BK + 8] u16 per operand (the pad
// staggers 16-byte row reads across banks), double-buffered.
#include <algorithm>
#include <type_traits>

#include "block_device.h"
#include "boa_kernels.h"
#include "coder_device.h"

namespace boa {

typedef float floatx4 __attribute__((ext_vector_type(4)));

// Epilogue mode of head.2 fused with the CDF (not a user activation): the
// block's logits rows pass through LDS 64 at a time and each row's (low,
// prob) pair of the next input byte is computed there (cdf_row_lowprob); the
// logits never reach memory.
constexpr int ACT_CDF = 3;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Epilogue of one tile: lane owns C[m][n .. n+3], m = m_blk + wm0 + 16p + j,
// n = n_blk + wn0 + 16q + 4g.  `sbias` holds the block's bias values
// (column c of the block at c, clamped at N - 1); the activation is a
// template argument, so the epilogue has no branch on it.
template <int TM, int TN, int ACT>
__device__ __forceinline__ void b16_epilogue(const GemmB16Args& a, const floatx4 (&acc)[TM][TN],
                                             int m_blk, int n_blk, int wm0, int wn0, int j, int g,
                                             const float* sbias) {
  const bool res4 = a.res && (a.ldr & 3) == 0;
#pragma unroll
  for (int p = 0; p < TM; ++p) {
    const int m = m_blk + wm0 + 16 * p + j;
    if (m >= a.M) continue;
#pragma unroll
    for (int q = 0; q < TN; ++q) {
      const int n = n_blk + wn0 + 16 * q + 4 * g;
      if (n >= a.N) continue;
      float rv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      if (res4 && n + 4 <= a.N) {
        const float4 t = *reinterpret_cast<const float4*>(a.res + (size_t)m * a.ldr + n);
        rv[0] = t.x; rv[1] = t.y; rv[2] = t.z; rv[3] = t.w;
      } else if (a.res) {
#pragma unroll
        for (int e = 0; e < 4; ++e) rv[e] = n + e < a.N ? a.res[(size_t)m * a.ldr + n + e] : 0.0f;
      }
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float t = acc[p][q][e] + sbias[n - n_blk + e];
        if (ACT == ACT_GELU) t = gelu<MATH_HW>(t);
        else if (ACT == ACT_RELU) t = fmaxf(0.0f, t);
        if (a.res) t = t + rv[e];
        v[e] = t;
      }
      const size_t o = (size_t)m * a.ldc + n;
      if (n + 4 <= a.N) {
        if (a.c_bf16)
          *reinterpret_cast<ushort4*>(reinterpret_cast<uint16_t*>(a.C) + o) =
              make_ushort4(f32_to_bf16(v[0]), f32_to_bf16(v[1]), f32_to_bf16(v[2]), f32_to_bf16(v[3]));
        else
          *reinterpret_cast<float4*>(reinterpret_cast<float*>(a.C) + o) =
              make_float4(v[0], v[1], v[2], v[3]);
        if (a.C2)
          *reinterpret_cast<ushort4*>(a.C2 + o) =
              make_ushort4(f32_to_bf16(v[0]), f32_to_bf16(v[1]), f32_to_bf16(v[2]), f32_to_bf16(v[3]));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (n + e >= a.N) break;
          if (a.c_bf16) reinterpret_cast<uint16_t*>(a.C)[o + e] = f32_to_bf16(v[e]);
          else reinterpret_cast<float*>(a.C)[o + e] = v[e];
          if (a.C2) a.C2[o + e] = f32_to_bf16(v[e]);
        }
      }
    }
  }
}

template <int BM, int BN, int WAVES_M, int WAVES_N, int BK, int NBUF, int ACT>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N) void gemm_bf16_kernel(GemmB16Args a,
                                                                           int swizzle,
                                                                           CdfEpi cdf) {
  constexpr int NT = 64 * WAVES_M * WAVES_N;
  constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
  constexpr int TM = WM / 16, TN = WN / 16;
  constexpr int S = BK + 8;                          // LDS row stride (u16)
  constexpr int XQ = BM * BK / 8, WQ = BN * BK / 8;  // 16-byte chunks per tile
  constexpr int XL = (XQ + NT - 1) / NT, WL = (WQ + NT - 1) / NT;
  static_assert(BK % 32 == 0, "BK must be a multiple of the MFMA k-step");
  // NBUF = 1 keeps one LDS stage (the next k-tile waits in registers), so
  // two workgroups fit in a CU's LDS and one's epilogue overlaps the
  // other's main loop.  The CDF epilogue reuses the words for 64 logits
  // rows of LS floats.
  constexpr int LS = BN + 4;
  constexpr int MAIN_B = NBUF * (BM + BN) * S * 2;
  constexpr int EPI_B = ACT == ACT_CDF ? 64 * LS * 4 : 0;
  __shared__ __attribute__((aligned(16))) uint16_t smem[(MAIN_B > EPI_B ? MAIN_B : EPI_B) / 2];
  uint16_t(*xs)[BM * S] = reinterpret_cast<uint16_t(*)[BM * S]>(smem);
  uint16_t(*ws)[BN * S] = reinterpret_cast<uint16_t(*)[BN * S]>(smem + NBUF * BM * S);
  __shared__ float sbias[BN];  // the block's bias values, for the epilogue

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm0 = (wave / WAVES_N) * WM, wn0 = (wave % WAVES_N) * WN;
  const int g = lane >> 4, j = lane & 15;
  // workgroup w runs on XCD w % 8; the swizzle gives each XCD a contiguous
  // range of tiles so an activation row-block stays in one XCD's L2
  const int nb = (a.N + BN - 1) / BN;
  int w = blockIdx.x;
  if (swizzle) {
    const int total = gridDim.x, per = total / 8;
    if (w < per * 8) w = (w % 8) * per + w / 8;
  }
  const int m_blk = (w / nb) * BM, n_blk = (w % nb) * BN;
  for (int c = tid; c < BN; c += NT) sbias[c] = a.bias ? a.bias[min(n_blk + c, a.N - 1)] : 0.0f;

  floatx4 acc[TM][TN];
#pragma unroll
  for (int p = 0; p < TM; ++p)
#pragma unroll
    for (int q = 0; q < TN; ++q) acc[p][q] = floatx4{0.f, 0.f, 0.f, 0.f};

  u32x4 xr[XL], wr[WL];
#define BOA_B16_LOAD(K0)                                                               \
  _Pragma("unroll") for (int i = 0; i < XL; ++i) {                                     \
    const int q = tid + i * NT;                                                        \
    if (XQ % NT == 0 || q < XQ) {                                                      \
      const int row = q / (BK / 8), c8 = q % (BK / 8);                                 \
      const int gm = min(m_blk + row, a.M - 1);                                        \
      xr[i] = *reinterpret_cast<const u32x4*>(a.X + (size_t)gm * a.ldx + (K0) + 8 * c8); \
    }                                                                                  \
  }                                                                                    \
  _Pragma("unroll") for (int i = 0; i < WL; ++i) {                                     \
    const int q = tid + i * NT;                                                        \
    if (WQ % NT == 0 || q < WQ) {                                                      \
      const int row = q / (BK / 8), c8 = q % (BK / 8);                                 \
      wr[i] = *reinterpret_cast<const u32x4*>(a.W + (size_t)(n_blk + row) * a.ldw + (K0) + 8 * c8); \
    }                                                                                  \
  }
#define BOA_B16_STORE(BUF)                                                             \
  _Pragma("unroll") for (int i = 0; i < XL; ++i) {                                     \
    const int q = tid + i * NT;                                                        \
    if (XQ % NT == 0 || q < XQ)                                                        \
      *reinterpret_cast<u32x4*>(&xs[BUF][(q / (BK / 8)) * S + 8 * (q % (BK / 8))]) = xr[i]; \
  }                                                                                    \
  _Pragma("unroll") for (int i = 0; i < WL; ++i) {                                     \
    const int q = tid + i * NT;                                                        \
    if (WQ % NT == 0 || q < WQ)                                                        \
      *reinterpret_cast<u32x4*>(&ws[BUF][(q / (BK / 8)) * S + 8 * (q % (BK / 8))]) = wr[i]; \
  }

  const int n_kt = a.K / BK;
  BOA_B16_LOAD(0)
  BOA_B16_STORE(0)
  __syncthreads();
  for (int kt = 0; kt < n_kt; ++kt) {
    const int cur = NBUF == 2 ? (kt & 1) : 0;
    if (kt + 1 < n_kt) { BOA_B16_LOAD((kt + 1) * BK) }
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks) {
      bf16x8 af[TN], bf[TM];
#pragma unroll
      for (int q = 0; q < TN; ++q)
        af[q] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(
                                               &ws[cur][(wn0 + 16 * q + j) * S + 32 * ks + 8 * g]));
#pragma unroll
      for (int p = 0; p < TM; ++p)
        bf[p] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(
                                               &xs[cur][(wm0 + 16 * p + j) * S + 32 * ks + 8 * g]));
#pragma unroll
      for (int p = 0; p < TM; ++p)
#pragma unroll
        for (int q = 0; q < TN; ++q)
          acc[p][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[q], bf[p], acc[p][q], 0, 0, 0);
    }
    if (NBUF == 1 && kt + 1 < n_kt) __syncthreads();
    if (kt + 1 < n_kt) { BOA_B16_STORE(NBUF == 2 ? (cur ^ 1) : 0) }
    __syncthreads();
  }
#undef BOA_B16_LOAD
#undef BOA_B16_STORE

  if constexpr (ACT == ACT_CDF) {
    // the logits rows, acc + bias as the unfused epilogue stores them,
    // 64 rows (one wave row of the block) at a time; the K loop ended with
    // a barrier, so its buffers are free
    static_assert(BN == 256 && WM == 64, "whole logits rows, 64 per wave row");
    float* lg = reinterpret_cast<float*>(smem);
    const int hw = tid >> 5, l = tid & 31;
    for (int h = 0; h < BM / 64; ++h) {
      if (wm0 == 64 * h) {
#pragma unroll
        for (int p = 0; p < TM; ++p)
#pragma unroll
          for (int q = 0; q < TN; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int col = wn0 + 16 * q + 4 * g + e;
              lg[(16 * p + j) * LS + col] = acc[p][q][e] + sbias[col];
            }
      }
      __syncthreads();
      for (int r = hw; r < 64; r += NT / 32)
        cdf_row_lowprob(lg + r * LS, cdf, m_blk + 64 * h + r, a.M, l);
      __syncthreads();  // the next 64 rows reuse the buffer
    }
    return;
  }
  b16_epilogue<TM, TN, ACT>(a, acc, m_blk, n_blk, wm0, wn0, j, g, sbias);
}

template <int BM, int BN, int WM_, int WN_, int BK, int NBUF = 2>
static hipError_t launch_b16(const GemmB16Args& a, hipStream_t s, int swizzle = 1,
                             const CdfEpi* cdf = nullptr) {
  if (a.K % BK || a.ldx % 8 || a.ldw % 8 || a.ldw < a.K) return hipErrorInvalidValue;
  const long long tiles = (long long)((a.N + BN - 1) / BN) * ((a.M + BM - 1) / BM);
  if (tiles >= (1ll << 31)) return hipErrorInvalidValue;
  const CdfEpi ce = cdf ? *cdf : CdfEpi{};
#define BOA_B16_GO(ACTv)                                                                  \
  BOA_LAUNCH((gemm_bf16_kernel<BM, BN, WM_, WN_, BK, NBUF, ACTv>), dim3((unsigned)tiles), \
                     dim3(64 * WM_ * WN_), 0, s, a, swizzle, ce)
  if (cdf) {
    if constexpr (BN == 256 && BM / WM_ == 64) {
      if (a.N != 256 || a.act != ACT_NONE) return hipErrorInvalidValue;
      BOA_B16_GO(ACT_CDF);
      return hipGetLastError();
    } else {
      return hipErrorInvalidValue;
    }
  }
  switch (a.act) {
    case ACT_NONE: BOA_B16_GO(ACT_NONE); break;
    case ACT_GELU: BOA_B16_GO(ACT_GELU); break;
    case ACT_RELU: BOA_B16_GO(ACT_RELU); break;
    default: return hipErrorInvalidValue;
  }
#undef BOA_B16_GO
  return hipGetLastError();
}

// ------------------------------------------------------- persistent blocks
// 256 rows x 256 features a tile, eight waves of 64 x 128 (128 accumulators,
// two waves per SIMD), one block per CU that walks over tiles.  What the
// shape is chosen for, on MI355X:
//   - LDS: a k-step's 32 MFMAs of a wave read 12 fragments (1 KB each); the
//     64 x 64 wave tiles of gemm_bf16_kernel read 8 for 16, which alone
//     filled the LDS.
//   - Vector memory: 64-k stages of 128-byte rows are copied straight to LDS
//     (global rows as whole cache lines).  Fragments loaded to registers
//     instead (64-byte pieces of 16 rows) kept the texture-address units 86 %
//     busy at a third of the MFMA rate.
//   - Stores: a lane holds four features of a row; stored from there a wave
//     writes 32-byte pieces of 16 rows, and those took longer than a short K
//     loop (262,144 x 1024, K = 256: 368 us, 175 without them).  The tile
//     turns round in LDS, 16 rows x 128 bytes at a time per wave, and leaves
//     in whole lines.
//   - K is short (256 to 2048): the next tile's first stage is copied while
//     this tile's last one is multiplied and its epilogue runs.
// LDS: two 64 KB stages (activations, then weights; the 16-byte chunk c of
// row r at slot c ^ (r & 7), so that eight lanes of a fragment read hit eight
// slots), 2 KB per wave for the epilogue, the bias of every feature.
// The chains are gemm_bf16_kernel's (k-steps of 32 in ascending order), and
// so are the bits.
constexpr int GP_STAGE = 65536, GP_EPI = 2048, GP_MAX_N = 2048;
constexpr int GP_LDS = 2 * GP_STAGE + 8 * GP_EPI + 4 * GP_MAX_N + 256;

struct GpTile {
  __amdgpu_buffer_rsrc_t x, w;  // the tile's activation rows, the wave's weight rows
  int m, n;
};

template <int ACT, bool F32>
__global__ __launch_bounds__(512, 2) void gemm_bf16_persist_kernel(GemmB16Args a, int m_blocks) {
  constexpr int TM = 4, TN = 8;
  __shared__ __attribute__((aligned(16))) unsigned char gp_smem[GP_LDS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, j = lane & 15;
  const int wm = wave >> 1, wn = wave & 1;  // rows 64 wm .., features 128 wn ..
  float* const sbias = reinterpret_cast<float*>(gp_smem + 2 * GP_STAGE + 8 * GP_EPI);
  for (int c = tid; c < a.N; c += 512) sbias[c] = a.bias ? a.bias[c] : 0.0f;
  __syncthreads();

  // Tiles: XCD x (blocks x, x + 8, ..) takes the m blocks x per .. x per +
  // per - 1, features fastest, so that the tiles in flight on an XCD share
  // activation rows and weights in its L2.
  const int nb = a.N / 256, per = (m_blocks + 7) / 8;
  const int x0 = (blockIdx.x & 7) * per;
  const int n_tiles = max(0, min(per, m_blocks - x0)) * nb;  // of this XCD
  const int step = gridDim.x / 8;
  const int n_st = a.K / 64;

  // copies: copy i of a wave fills rows 32 wave + 8 i .. + 7 of a stage's
  // activations and of its weights
  const int crow = 32 * wave + (lane >> 3), cchunk = ((lane & 7) ^ (lane >> 3)) * 16;
  const int woff = (lane >> 3) * a.ldw * 2 + cchunk;
  auto tile_at = [&](int t) {
    GpTile T;
    T.m = (x0 + t / nb) * 256;
    T.n = (t % nb) * 256;
    T.x = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.X) + (size_t)T.m * a.ldx,
                                            (short)0, -1, 0x00027000);
    T.w = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(a.W) + (size_t)(T.n + 32 * wave) * a.ldw, (short)0, -1, 0x00027000);
    return T;
  };
  auto copy = [&](const GpTile& T, int st, int slot) {
    unsigned char* const base = gp_smem + slot * GP_STAGE + wave * 4096;
    const int last = a.M - 1 - T.m;  // rows past M repeat the last one
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          T.x, (__attribute__((address_space(3))) void*)(base + i * 1024), 16,
          min(crow + 8 * i, last) * a.ldx * 2 + cchunk, st * 128, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          T.w, (__attribute__((address_space(3))) void*)(base + 32768 + i * 1024), 16, woff,
          st * 128 + i * 16 * a.ldw, 0, 0);
  };
  // fragments of k-step ks: rows 64 wm + 16 p + j (128 wn + 16 q + j of the
  // weights), chunk 4 ks + g
  const uint32_t lds0 = lds_addr(gp_smem);
  uint32_t xfrag[2], wfrag[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const uint32_t s = j * 128 + ((4 * ks + g) ^ (j & 7)) * 16;
    xfrag[ks] = lds0 + wm * 8192 + s;
    wfrag[ks] = lds0 + 32768 + wn * 16384 + s;
  }

  int t = blockIdx.x >> 3;
  if (t >= n_tiles) return;  // the whole block
  GpTile T = tile_at(t);
  copy(T, 0, 0);
  int slot = 0;
  int pending = 0;  // accesses newer than the next stage's copies (0, 1, 16 or 17)
  while (true) {
    floatx4 acc[TM][TN];
#pragma unroll
    for (int p = 0; p < TM; ++p)
#pragma unroll
      for (int q = 0; q < TN; ++q) acc[p][q] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int t_next = t + step;
    const bool more = t_next < n_tiles;
    const GpTile Tn = more ? tile_at(t_next) : T;
    // Wave 0 fetches a 64-row group of the next tile's activations into L2, a
    // stage's 128-byte line per row and stage (a copy to LDS that nobody
    // reads), where four or more blocks share those rows: the copies proper
    // run one stage ahead, too late for HBM behind the stores (1.2 M x 1024,
    // K = 256: 1009 -> 907 us; with one or two blocks a row the extra
    // requests cost more than they save, K = 512, N = 256: 384 -> 521 us).
    const bool ahead = more && wave == 0 && nb >= 4 && T.n < 4 * 256;
    const int poff = min(64 * (T.n / 256) + lane, a.M - 1 - Tn.m) * a.ldx * 2;
    for (int st = 0; st < n_st; ++st, slot ^= 1) {
      // this wave's copies of the stage have landed (newer are only the last
      // epilogue's 16 stores and the fetch ahead), then everyone's
      switch (pending) {
        case 17: asm volatile("s_waitcnt vmcnt(17)" ::: "memory"); break;
        case 16: asm volatile("s_waitcnt vmcnt(16)" ::: "memory"); break;
        case 1: asm volatile("s_waitcnt vmcnt(1)" ::: "memory"); break;
        default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      pending = 0;
      lds_barrier();  // and everyone is past the other slot's reads
      if (st + 1 < n_st) copy(T, st + 1, slot ^ 1);
      else if (more) copy(Tn, 0, slot ^ 1);
      if (ahead) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            Tn.x, (__attribute__((address_space(3))) void*)(gp_smem + GP_LDS - 256), 4, poff,
            st * 128, 0, 0);
        pending = 1;
      }
      const uint32_t so = (uint32_t)slot * GP_STAGE;
      const uint32_t xa[2] = {xfrag[0] + so, xfrag[1] + so}, wa[2] = {wfrag[0] + so, wfrag[1] + so};
      lds_u32x4 xf[2][TM], f[2][2];
      auto read_x = [&](auto KS) {
        constexpr int ks = decltype(KS)::value;
        xf[ks][0] = lds_read128_at<0>(xa[ks]);
        xf[ks][1] = lds_read128_at<2048>(xa[ks]);
        xf[ks][2] = lds_read128_at<4096>(xa[ks]);
        xf[ks][3] = lds_read128_at<6144>(xa[ks]);
      };
      auto read_w = [&](auto H) {  // feature tiles 2 (H % 4) and the next of k-step H / 4
        constexpr int h = decltype(H)::value;
        f[h & 1][0] = lds_read128_at<(2 * (h & 3)) * 2048>(wa[h >> 2]);
        f[h & 1][1] = lds_read128_at<(2 * (h & 3) + 1) * 2048>(wa[h >> 2]);
      };
      auto part = [&](auto H) {
        constexpr int h = decltype(H)::value, q0 = 2 * (h & 3), b = h & 1, ks = h >> 2;
        if constexpr (h == 2) read_x(std::integral_constant<int, 1>{});
        if constexpr (h < 7) read_w(std::integral_constant<int, h + 1>{});
        if constexpr (h == 0)
          asm volatile("s_waitcnt lgkmcnt(2)"
                       : "+v"(f[b][0]), "+v"(f[b][1]), "+v"(xf[0][0]), "+v"(xf[0][1]),
                         "+v"(xf[0][2]), "+v"(xf[0][3])::"memory");
        else if constexpr (h == 2)
          asm volatile("s_waitcnt lgkmcnt(6)" : "+v"(f[b][0]), "+v"(f[b][1])::"memory");
        else if constexpr (h == 4)
          asm volatile("s_waitcnt lgkmcnt(2)"
                       : "+v"(f[b][0]), "+v"(f[b][1]), "+v"(xf[1][0]), "+v"(xf[1][1]),
                         "+v"(xf[1][2]), "+v"(xf[1][3])::"memory");
        else if constexpr (h == 7)
          asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f[b][0]), "+v"(f[b][1])::"memory");
        else
          asm volatile("s_waitcnt lgkmcnt(2)" : "+v"(f[b][0]), "+v"(f[b][1])::"memory");
#pragma unroll
        for (int p = 0; p < TM; ++p)
#pragma unroll
          for (int q = 0; q < 2; ++q)
            acc[p][q0 + q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8, f[b][q]), __builtin_bit_cast(bf16x8, xf[ks][p]),
                acc[p][q0 + q], 0, 0, 0);
      };
      read_x(std::integral_constant<int, 0>{});
      read_w(std::integral_constant<int, 0>{});
      part(std::integral_constant<int, 0>{});
      part(std::integral_constant<int, 1>{});
      part(std::integral_constant<int, 2>{});
      part(std::integral_constant<int, 3>{});
      part(std::integral_constant<int, 4>{});
      part(std::integral_constant<int, 5>{});
      part(std::integral_constant<int, 6>{});
      part(std::integral_constant<int, 7>{});
    }

    // Epilogue, per wave without barriers, its LDS accesses outside the
    // compiler's view (it would wait for the next tile's copies).  A group of
    // 16 rows x 128 bytes goes to the wave's 2 KB with chunk c of row r at
    // slot c ^ (r & 7) and comes back eight lanes a row, two 8-row reads.
    const uint32_t epi = lds0 + 2 * GP_STAGE + wave * GP_EPI;
    const uint32_t bat = lds_addr(sbias) + (T.n + 128 * wn + 4 * g) * 4;
    const int m0 = T.m + 64 * wm, n0 = T.n + 128 * wn;
    const int er = lane >> 3, ec = lane & 7;  // row and chunk of a read
    const uint32_t erd = epi + er * 128 + ((ec ^ er) * 16);  // rows er and er + 8: the same slot
    const bool full = T.m + 256 <= a.M;
    auto act = [&](float v, float b) {
      float t = v + b;
      if (ACT == ACT_GELU) t = gelu<MATH_HW>(t);
      else if (ACT == ACT_RELU) t = fmaxf(0.0f, t);
      return t;
    };
    if (!full && m0 >= a.M) {  // padding rows only: no activations, no stores
      pending = 0;
    } else if constexpr (!F32) {
#pragma unroll
      for (int half = 0; half < 2; ++half) {  // features 64 half .. of the wave's 128
        lds_u32x4 bv[4];
        bv[0] = half ? lds_read128_at<256>(bat) : lds_read128_at<0>(bat);
        bv[1] = half ? lds_read128_at<320>(bat) : lds_read128_at<64>(bat);
        bv[2] = half ? lds_read128_at<384>(bat) : lds_read128_at<128>(bat);
        bv[3] = half ? lds_read128_at<448>(bat) : lds_read128_at<192>(bat);
        lds_wait4(bv[0], bv[1], bv[2], bv[3]);
#pragma unroll
        for (int p = 0; p < TM; ++p) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const floatx4 c = acc[p][4 * half + q];
            const uint32_t lo =
                (uint32_t)f32_to_bf16(act(c[0], u2f(bv[q][0]))) |
                ((uint32_t)f32_to_bf16(act(c[1], u2f(bv[q][1]))) << 16);
            const uint32_t hi =
                (uint32_t)f32_to_bf16(act(c[2], u2f(bv[q][2]))) |
                ((uint32_t)f32_to_bf16(act(c[3], u2f(bv[q][3]))) << 16);
            lds_write64_at<0>(epi + j * 128 + (((2 * q + (g >> 1)) ^ (j & 7)) * 16) + (g & 1) * 8,
                              lo, hi);
          }
          lds_u32x4 v0 = lds_read128_at<0>(erd), v1 = lds_read128_at<1024>(erd);
          asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(v0), "+v"(v1)::"memory");
          uint16_t* const o =
              reinterpret_cast<uint16_t*>(a.C) + (size_t)(m0 + 16 * p + er) * a.ldc + n0 + 64 * half + 8 * ec;
          if (full || m0 + 16 * p + er < a.M) *reinterpret_cast<lds_u32x4*>(o) = v0;
          if (full || m0 + 16 * p + er + 8 < a.M)
            *reinterpret_cast<lds_u32x4*>(o + (size_t)8 * a.ldc) = v1;
        }
      }
      pending = full ? pending + 16 : 0;
    } else {
      pending = 0;
#pragma unroll
      for (int qq = 0; qq < 4; ++qq) {  // features 32 qq .. of the wave's 128
        lds_u32x4 bv[2];
        bv[0] = qq == 0 ? lds_read128_at<0>(bat) : qq == 1 ? lds_read128_at<128>(bat)
              : qq == 2 ? lds_read128_at<256>(bat) : lds_read128_at<384>(bat);
        bv[1] = qq == 0 ? lds_read128_at<64>(bat) : qq == 1 ? lds_read128_at<192>(bat)
              : qq == 2 ? lds_read128_at<320>(bat) : lds_read128_at<448>(bat);
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(bv[0]), "+v"(bv[1])::"memory");
        float4 rs[TM][2];
        if (a.res) {
#pragma unroll
          for (int p = 0; p < TM; ++p)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int m = min(m0 + 16 * p + er + 8 * h, a.M - 1);
              rs[p][h] = *reinterpret_cast<const float4*>(a.res + (size_t)m * a.ldr + n0 + 32 * qq + 4 * ec);
            }
        }
#pragma unroll
        for (int p = 0; p < TM; ++p) {
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const floatx4 c = acc[p][2 * qq + q];
            lds_u32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = f2u(act(c[e], u2f(bv[q][e])));
            lds_write128_at<0>(epi + j * 128 + (((4 * q + g) ^ (j & 7)) * 16), v);
          }
          lds_u32x4 v[2];
          v[0] = lds_read128_at<0>(erd);
          v[1] = lds_read128_at<1024>(erd);
          asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(v[0]), "+v"(v[1])::"memory");
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int m = m0 + 16 * p + er + 8 * h;
            float4 o = make_float4(u2f(v[h][0]), u2f(v[h][1]), u2f(v[h][2]), u2f(v[h][3]));
            if (a.res) {
              const float4 e = rs[p][h];
              o = make_float4(o.x + e.x, o.y + e.y, o.z + e.z, o.w + e.w);
            }
            if (full || m < a.M) {
              const size_t at = (size_t)m * a.ldc + n0 + 32 * qq + 4 * ec;
              *reinterpret_cast<float4*>(reinterpret_cast<float*>(a.C) + at) = o;
              if (a.C2)
                *reinterpret_cast<ushort4*>(a.C2 + at) = make_ushort4(
                    f32_to_bf16(o.x), f32_to_bf16(o.y), f32_to_bf16(o.z), f32_to_bf16(o.w));
            }
          }
        }
      }
    }
    if (!more) break;
    t = t_next;
    T = Tn;
  }
}

// What the kernel's addressing takes: whole 256-feature tiles up to
// GP_MAX_N, whole 64-k stages, 16-byte rows, a tile's rows within 32-bit byte
// offsets; a residual or a bf16 copy only beside fp32 output, an activation
// only beside bf16 output (the model has no others).
static bool b16_persist_fits(const GemmB16Args& a) {
  return a.N % 256 == 0 && a.N <= GP_MAX_N && a.K % 64 == 0 && a.K >= 64 && a.ldx % 8 == 0 &&
         a.ldw % 8 == 0 && a.ldw >= a.K && a.ldx <= (1 << 20) && a.ldw <= (1 << 20) &&
         a.ldc % 8 == 0 && (!a.res || a.ldr % 4 == 0) &&
         (a.c_bf16 ? !a.res && !a.C2 : a.act == ACT_NONE);
}

static hipError_t launch_b16_persist(const GemmB16Args& a, hipStream_t s) {
  const int m_blocks = (int)(((long long)a.M + 255) / 256);
  // a multiple of eight blocks (one share of the XCDs each), at most one per CU
  const long long tiles = (long long)((m_blocks + 7) / 8) * (a.N / 256) * 8;
  const unsigned grid = (unsigned)std::min<long long>(tiles, 256);
#define BOA_B16_GO(ACTv, F32v)                                                                  \
  BOA_LAUNCH((gemm_bf16_persist_kernel<ACTv, F32v>), dim3(grid), dim3(512), 0, s, a, m_blocks)
  if (!a.c_bf16) {
    BOA_B16_GO(ACT_NONE, true);
    return hipGetLastError();
  }
  switch (a.act) {
    case ACT_NONE: BOA_B16_GO(ACT_NONE, false); break;
    case ACT_GELU: BOA_B16_GO(ACT_GELU, false); break;
    case ACT_RELU: BOA_B16_GO(ACT_RELU, false); break;
    default: return hipErrorInvalidValue;
  }
#undef BOA_B16_GO
  return hipGetLastError();
}

// W must hold round_up(N, 256) rows (zero padded) for every configuration.
// Outputs of whole 256-feature tiles run on the persistent blocks (TFLOP/s at
// M = 2^20, against the 16-wave 256 x 256 blocks of gemm_bf16_kernel: K 256 N
// 1024 492 -> 766, K 512 N 256 625 -> 842, K 512 N 2048 688 -> 1007, K 1024 N
// 512 839 -> 1066, K 2048 N 512 with residual 822 -> 982, GELU K 512 N 2048
// 590 -> 781; M 255 to 1300 as fast or faster); narrower or unaligned ones
// (x_proj, d_model 64's and 128's narrow outputs) on 128 x 64 blocks with 8
// waves.
hipError_t gemm_bf16(const GemmB16Args& a, hipStream_t s) {
  if (a.M <= 0 || a.N <= 0) return hipSuccess;
  if (b16_persist_fits(a)) return launch_b16_persist(a, s);
  return launch_b16<128, 64, 4, 2, 64>(a, s);
}

// head.2 (N = 256) fused with the CDF: the head GEMM's tile and stages, the
// epilogue of ACT_CDF; writes cdf.lowprob instead of the logits
hipError_t gemm_bf16_head_cdf(const GemmB16Args& a, const CdfEpi& cdf, hipStream_t s) {
  if (a.M <= 0) return hipSuccess;
  if (a.K >= 512) return launch_b16<256, 256, 4, 4, 64, 1>(a, s, 1, &cdf);
  return launch_b16<256, 256, 4, 4, 64>(a, s, 1, &cdf);
}

// ------------------------------------------------------ FF1 + GELU + FF2
// The feed-forward pair in one kernel: a block of 1024 threads owns BM rows
// and keeps their FF2 accumulators (BM x D fp32) in registers while the
// hidden layer passes through LDS HC columns at a time:
//   h = bf16(gelu(x . W1[c]^T + b1[c]))   (HC hidden columns of chunk c)
//   acc += h . W2[:, c]^T
// then acc + b2 + residual.  The hidden layer (4 D bf16 per row) never
// reaches HBM.  Every MFMA chain is the unfused GEMMs' (k-steps of 32 in
// ascending order from 0, k = 32 s + 8 g + e in operand slot (g, e); FF2's
// chain continues from chunk to chunk), and both epilogues are theirs, so
// the bits are those of gemm_bf16(FF1, GELU) + gemm_bf16(FF2).
// LDS rows are K-contiguous bf16 with 8 elements of padding.
// LNF bit 1: the block's rows of X are out_proj's output and LN2 runs on them
// in LDS before FF1, in ln2_kernel's order (one thread per row, elements in
// order, statistics from the bf16 values) and with its bf16 rounding of the
// result.  LNF bit 2: the fp32 output rows also pass through LDS, where the
// next layer's LN1 runs in ln1_kernel's order (half-wave per row, the
// 32-lane tree) and stores xn in bf16.
template <int D, int BM, int HC, int WM2, int WN2, int WM1, int WN1, int LNF>
__global__ __launch_bounds__(1024) void ffn_bf16_kernel(FfnB16Args a) {
  constexpr int H = 4 * D;
  // Row strides (bf16) of the LDS tiles.  The bank conflicts measured on
  // MI355X fit 16-byte fragment reads served 32 lanes at a time (16 rows j,
  // two 16-byte column groups g) over 128 four-byte banks: a row stride of
  // 8 mod 128 words (D + 16 bf16 at D = 256) puts those 32 reads on
  // distinct banks, while D + 8 (4 mod 128 words) paired them up.  C3
  // probe: FFN bank-conflict cycles 21.6 -> 8.9 % of its active cycles,
  // compress 19.32 -> 19.81 MB/s.  HP keeps HC + 8 (the tiles fill the LDS).
  constexpr int XP = D + 16, HP = HC + 8;
  constexpr int NC = H / HC;
  constexpr int TM2 = BM / WM2 / 16, TN2 = D / WN2 / 16;    // FF2 tiles per wave
  constexpr int TM1 = BM / WM1 / 16, TN1 = HC / WN1 / 16;   // FF1 tiles per wave
  static_assert(WM2 * WN2 == 16 && WM1 * WN1 <= 16, "16 waves");
  static_assert(TM2 >= 1 && TN2 >= 1 && TM1 >= 1 && TN1 >= 1, "tile shapes");
  constexpr int XQ = BM * D / 8, W1Q = HC * D / 8, W2Q = D * HC / 8;  // 16-byte chunks
  constexpr int XL = (XQ + 1023) / 1024, W1L = (W1Q + 1023) / 1024, W2L = (W2Q + 1023) / 1024;
  // one LDS buffer: the K loop's xs, w1s, hs, w2s; after it, the LN1
  // epilogue's fp32 rows (stride RS)
  constexpr int XS_B = BM * XP * 2, W1S_B = HC * XP * 2, HS_B = BM * HP * 2, W2S_B = D * HP * 2;
  constexpr int MAIN_B = XS_B + W1S_B + HS_B + W2S_B;
  constexpr int RS = D + 4;
  constexpr int EPI_B = (LNF & 2) ? BM * RS * 4 : 0;
  static_assert(XS_B % 16 == 0 && W1S_B % 16 == 0 && HS_B % 16 == 0, "16-byte aligned parts");
  __shared__ __attribute__((aligned(16))) unsigned char smem[MAIN_B > EPI_B ? MAIN_B : EPI_B];
  uint16_t* const xs = reinterpret_cast<uint16_t*>(smem);
  uint16_t* const w1s = reinterpret_cast<uint16_t*>(smem + XS_B);
  uint16_t* const hs = reinterpret_cast<uint16_t*>(smem + XS_B + W1S_B);
  uint16_t* const w2s = reinterpret_cast<uint16_t*>(smem + XS_B + W1S_B + HS_B);
  __shared__ float b1s[HC], b2s[D];
  __shared__ float lnst[2 * BM];  // LN2: per-row (mean, 1 / std)

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, j = lane & 15;
  const int m_blk = blockIdx.x * BM;

  // the block's rows and b2
#pragma unroll
  for (int it = 0; it < XL; ++it) {
    const int q = tid + it * 1024;
    if (XQ % 1024 == 0 || q < XQ) {
      const int row = q / (D / 8), c8 = q % (D / 8);
      const int gm = min(m_blk + row, a.M - 1);
      *reinterpret_cast<u32x4*>(&xs[row * XP + 8 * c8]) =
          *reinterpret_cast<const u32x4*>(a.X + (size_t)gm * D + 8 * c8);
    }
  }
  for (int c = tid; c < D; c += 1024) b2s[c] = a.b2 ? a.b2[c] : 0.0f;

  u32x4 w1r[W1L], w2r[W2L];
  float b1r = 0.0f;
  auto load_chunk = [&](int ch) {
#pragma unroll
    for (int it = 0; it < W1L; ++it) {
      const int q = tid + it * 1024;
      if (W1Q % 1024 == 0 || q < W1Q) {
        const int row = q / (D / 8), c8 = q % (D / 8);
        w1r[it] = *reinterpret_cast<const u32x4*>(a.W1 + (size_t)(ch * HC + row) * D + 8 * c8);
      }
    }
#pragma unroll
    for (int it = 0; it < W2L; ++it) {
      const int q = tid + it * 1024;
      if (W2Q % 1024 == 0 || q < W2Q) {
        const int row = q / (HC / 8), c8 = q % (HC / 8);
        w2r[it] = *reinterpret_cast<const u32x4*>(a.W2 + (size_t)row * H + ch * HC + 8 * c8);
      }
    }
    if (tid < HC) b1r = a.b1 ? a.b1[ch * HC + tid] : 0.0f;
  };
  auto store_chunk = [&]() {
#pragma unroll
    for (int it = 0; it < W1L; ++it) {
      const int q = tid + it * 1024;
      if (W1Q % 1024 == 0 || q < W1Q)
        *reinterpret_cast<u32x4*>(&w1s[(q / (D / 8)) * XP + 8 * (q % (D / 8))]) = w1r[it];
    }
#pragma unroll
    for (int it = 0; it < W2L; ++it) {
      const int q = tid + it * 1024;
      if (W2Q % 1024 == 0 || q < W2Q)
        *reinterpret_cast<u32x4*>(&w2s[(q / (HC / 8)) * HP + 8 * (q % (HC / 8))]) = w2r[it];
    }
    if (tid < HC) b1s[tid] = b1r;
  };

  // FF2 accumulators: wave (wm2, wn2) owns rows 16 TM2 wm2 + 16 p + j, features
  // 16 TN2 wn2 + 16 q + 4 g + v
  const int wm2 = wave / WN2, wn2 = wave % WN2;
  const int wm1 = wave / WN1, wn1 = wave % WN1;
  const bool ff1_wave = wave < WM1 * WN1;
  floatx4 acc2[TM2][TN2];
#pragma unroll
  for (int p = 0; p < TM2; ++p)
#pragma unroll
    for (int q = 0; q < TN2; ++q) acc2[p][q] = floatx4{0.f, 0.f, 0.f, 0.f};

  load_chunk(0);
  if constexpr ((LNF & 1) != 0) {
    // LN2 in place in xs while chunk 0's weights load (splitting the sums
    // and the sums of squares over two waves measured the same)
    __syncthreads();
    if (tid < BM) {
      const uint16_t* row = xs + tid * XP;
      float sm = 0.0f, sq = 0.0f;
      for (int c8 = 0; c8 < D / 8; ++c8) {
        const u32x4 w = *reinterpret_cast<const u32x4*>(row + 8 * c8);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float lo = u2f(w[e] << 16), hi = u2f(w[e] & 0xFFFF0000u);
          sm = sm + lo;
          sq = sq + lo * lo;
          sm = sm + hi;
          sq = sq + hi * hi;
        }
      }
      const float mean = sm / (float)a.n;
      const float var = sq / (float)a.n - mean * mean;
      lnst[2 * tid] = mean;
      lnst[2 * tid + 1] = 1.0f / __builtin_sqrtf(var + 1e-5f);
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < XL; ++it) {
      const int q = tid + it * 1024;
      if (XQ % 1024 == 0 || q < XQ) {
        const int row = q / (D / 8), c8 = q % (D / 8);
        u32x4* px = reinterpret_cast<u32x4*>(&xs[row * XP + 8 * c8]);
        const u32x4 w = *px;
        const float mean = lnst[2 * row], inv_std = lnst[2 * row + 1];
        const float4 wa = *reinterpret_cast<const float4*>(a.ln2_w + 8 * c8);
        const float4 wb = *reinterpret_cast<const float4*>(a.ln2_w + 8 * c8 + 4);
        const float4 ba = *reinterpret_cast<const float4*>(a.ln2_b + 8 * c8);
        const float4 bb = *reinterpret_cast<const float4*>(a.ln2_b + 8 * c8 + 4);
        const float wv[8] = {wa.x, wa.y, wa.z, wa.w, wb.x, wb.y, wb.z, wb.w};
        const float bv[8] = {ba.x, ba.y, ba.z, ba.w, bb.x, bb.y, bb.z, bb.w};
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float lo = u2f(w[e] << 16), hi = u2f(w[e] & 0xFFFF0000u);
          const uint32_t ol = f32_to_bf16(((lo - mean) * inv_std) * wv[2 * e] + bv[2 * e]);
          const uint32_t oh = f32_to_bf16(((hi - mean) * inv_std) * wv[2 * e + 1] + bv[2 * e + 1]);
          o[e] = ol | (oh << 16);
        }
        *px = o;
      }
    }
    // the chunk loop's first barrier orders these stores before FF1's reads
  }
  for (int ch = 0; ch < NC; ++ch) {
    __syncthreads();  // the previous chunk's w1s, hs and w2s are no longer read
    store_chunk();
    if (ch + 1 < NC) load_chunk(ch + 1);
    __syncthreads();
    // FF1 on chunk ch: hidden columns ch HC + 16 TN1 wn1 + 16 q + 4 g + v
    if (ff1_wave) {
      floatx4 acc1[TM1][TN1];
#pragma unroll
      for (int p = 0; p < TM1; ++p)
#pragma unroll
        for (int q = 0; q < TN1; ++q) acc1[p][q] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < D / 32; ++ks) {
        bf16x8 af[TN1], bf[TM1];
#pragma unroll
        for (int q = 0; q < TN1; ++q)
          af[q] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(
                                                 &w1s[(16 * (TN1 * wn1 + q) + j) * XP + 32 * ks + 8 * g]));
#pragma unroll
        for (int p = 0; p < TM1; ++p)
          bf[p] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(
                                                 &xs[(16 * (TM1 * wm1 + p) + j) * XP + 32 * ks + 8 * g]));
#pragma unroll
        for (int p = 0; p < TM1; ++p)
#pragma unroll
          for (int q = 0; q < TN1; ++q)
            acc1[p][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[q], bf[p], acc1[p][q], 0, 0, 0);
      }
#pragma unroll
      for (int p = 0; p < TM1; ++p)
#pragma unroll
        for (int q = 0; q < TN1; ++q) {
          const int n = 16 * (TN1 * wn1 + q) + 4 * g;
          uint16_t o[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) o[v] = f32_to_bf16(gelu<MATH_HW>(acc1[p][q][v] + b1s[n + v]));
          *reinterpret_cast<ushort4*>(&hs[(16 * (TM1 * wm1 + p) + j) * HP + n]) =
              make_ushort4(o[0], o[1], o[2], o[3]);
        }
    }
    __syncthreads();
    // FF2's k-steps of chunk ch
#pragma unroll
    for (int ks = 0; ks < HC / 32; ++ks) {
      bf16x8 af[TN2], bf[TM2];
#pragma unroll
      for (int q = 0; q < TN2; ++q)
        af[q] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(
                                               &w2s[(16 * (TN2 * wn2 + q) + j) * HP + 32 * ks + 8 * g]));
#pragma unroll
      for (int p = 0; p < TM2; ++p)
        bf[p] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(
                                               &hs[(16 * (TM2 * wm2 + p) + j) * HP + 32 * ks + 8 * g]));
#pragma unroll
      for (int p = 0; p < TM2; ++p)
#pragma unroll
        for (int q = 0; q < TN2; ++q)
          acc2[p][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[q], bf[p], acc2[p][q], 0, 0, 0);
    }
  }
  // FF2's epilogue: + b2, + residual, fp32 out (and the bf16 copy)
  float* const rows = reinterpret_cast<float*>(smem);
  if constexpr ((LNF & 2) != 0) __syncthreads();  // every wave is past its last reads of hs, w2s
#pragma unroll
  for (int p = 0; p < TM2; ++p) {
    const int rl = 16 * (TM2 * wm2 + p) + j;
    const int m = m_blk + rl;
    if (m >= a.M) continue;
#pragma unroll
    for (int q = 0; q < TN2; ++q) {
      const int n = 16 * (TN2 * wn2 + q) + 4 * g;
      const float4 rv = *reinterpret_cast<const float4*>(a.res + (size_t)m * D + n);
      const float r4[4] = {rv.x, rv.y, rv.z, rv.w};
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (acc2[p][q][e] + b2s[n + e]) + r4[e];
      *reinterpret_cast<float4*>(a.C + (size_t)m * D + n) = make_float4(v[0], v[1], v[2], v[3]);
      if ((LNF & 2) != 0)
        *reinterpret_cast<float4*>(rows + rl * RS + n) = make_float4(v[0], v[1], v[2], v[3]);
      if (a.C2)
        *reinterpret_cast<ushort4*>(a.C2 + (size_t)m * D + n) =
            make_ushort4(f32_to_bf16(v[0]), f32_to_bf16(v[1]), f32_to_bf16(v[2]), f32_to_bf16(v[3]));
    }
  }
  if constexpr ((LNF & 2) != 0) {
    __syncthreads();
    // the next layer's LN1: half-wave hw takes rows hw, hw + 32, ...; lane l
    // sums elements l, l + 32, ... in order, then the shuffle-down tree, and
    // lane 0's totals are broadcast; the normalised rows overwrite the LDS rows
    const int hw = tid >> 5, l = tid & 31;
#pragma unroll 1
    for (int rl = hw; rl < BM; rl += 32) {
      float* row = rows + rl * RS;
      float sm = 0.0f, sq = 0.0f;
#pragma unroll
      for (int e = 0; e < D / 32; ++e) {
        const float v = row[l + 32 * e];
        sm = sm + v;
        sq = sq + v * v;
      }
#pragma unroll
      for (int off = 16; off > 0; off >>= 1) {
        sm = sm + __shfl_down(sm, off, 32);
        sq = sq + __shfl_down(sq, off, 32);
      }
      sm = __shfl(sm, 0, 32);
      sq = __shfl(sq, 0, 32);
      const float mean = sm / (float)a.n;
      const float var = sq / (float)a.n - mean * mean;
      const float inv_std = 1.0f / __builtin_sqrtf(var + 1e-5f);
#pragma unroll
      for (int e = 0; e < D / 32; ++e) {
        const int idx = l + 32 * e;
        row[idx] = ((row[idx] - mean) * inv_std) * a.ln1_w[idx] + a.ln1_b[idx];
      }
    }
    __syncthreads();
    // bf16 xn, eight features (16 bytes) per store
#pragma unroll
    for (int it = 0; it < XL; ++it) {
      const int q = tid + it * 1024;
      if (XQ % 1024 == 0 || q < XQ) {
        const int rl = q / (D / 8), c8 = q % (D / 8);
        const int m = m_blk + rl;
        if (m < a.M) {
          const float* v = rows + rl * RS + 8 * c8;
          u32x4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            o[e] = (uint32_t)f32_to_bf16(v[2 * e]) | ((uint32_t)f32_to_bf16(v[2 * e + 1]) << 16);
          *reinterpret_cast<u32x4*>(a.xn + (size_t)m * D + 8 * c8) = o;
        }
      }
    }
  }
}

// ------------------------------------------- FF1 + GELU + FF2 by rows
// The same pair, 256 wide, in blocks of 128 rows and four waves, two blocks
// per CU: one's loads, LayerNorms and stores run under the other's MFMAs.  A
// wave holds 32 rows of X (LN2 applied) and their FF2 accumulators in
// registers and shares nothing with the others but the weights: 32 hidden
// columns a time go from FF1's accumulators through GELU into FF2's operand by
// lane swaps and never touch LDS.  LDS holds the rows, then two stages of the
// weights (32 hidden columns of both matrices, 32 KB, copied there one stage
// ahead); a stage is 32 fragment reads for 64 MFMAs of a wave, where the
// 16-wave blocks above read 3 for 2 in FF1 and 6 for 8 in FF2 and pass the
// hidden layer through LDS, which filled it.  The last rows leave through LDS
// as whole 1 KB lines.  The chains and the LayerNorms' orders are the same,
// and so are the bits.
// All 24 calls of a compress pass over 8192 lanes x 512 bytes, 8 layers: 73.0
// -> 55.5 ms (256-row blocks of eight waves, one per CU: 61.7, of which 29
// outside the MFMA loop; fragments read two steps ahead instead of one: no
// change; GELU taken out: 12.6 ms less).
constexpr int FR_STAGE = 32768, FR_B1 = 2 * FR_STAGE, FR_B2 = FR_B1 + 4096, FR_ST = FR_B2 + 1024;
constexpr int FR_LDS = FR_ST + 1024;

template <int LNF>
__global__ __launch_bounds__(256, 2) void ffn_bf16_rows_kernel(FfnB16Args a) {
  static_assert((LNF & 1) != 0, "LN2 is always applied here");
  constexpr int D = 256, H = 1024;
  __shared__ __attribute__((aligned(16))) unsigned char fr_smem[FR_LDS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, j = lane & 15;
  const int m_blk = blockIdx.x * 128, last = a.M - 1 - m_blk;  // rows past M repeat the last one
  float* const b1s = reinterpret_cast<float*>(fr_smem + FR_B1);
  float* const b2s = reinterpret_cast<float*>(fr_smem + FR_B2);
  float* const lnst = reinterpret_cast<float*>(fr_smem + FR_ST);
  const uint32_t lds0 = lds_addr(fr_smem);

  // The block's rows through both stages: four 64-k blocks of 128 rows x 128
  // bytes, chunk c of row r at slot c ^ (r & 7)
  const int cchunk = ((lane & 7) ^ (lane >> 3)) * 16;
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(a.X) + (size_t)m_blk * D, (short)0, -1, 0x00027000);
#pragma unroll
  for (int kq = 0; kq < 4; ++kq)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          xr, (__attribute__((address_space(3))) void*)(fr_smem + kq * 16384 + wave * 4096 + i * 1024),
          16, min(32 * wave + 8 * i + (lane >> 3), last) * (D * 2) + cchunk, kq * 128, 0, 0);
  for (int c = tid; c < H; c += 256) b1s[c] = a.b1 ? a.b1[c] : 0.0f;
  b2s[tid] = a.b2 ? a.b2[tid] : 0.0f;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  {  // one thread per row, elements in order
    if (tid < 128) {
      const unsigned char* row = fr_smem + tid * 128;
      float sm = 0.0f, sq = 0.0f;
      for (int c8 = 0; c8 < D / 8; ++c8) {
        const u32x4 w = *reinterpret_cast<const u32x4*>(row + (c8 >> 3) * 16384 +
                                                        (((c8 & 7) ^ (tid & 7)) * 16));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float lo = u2f(w[e] << 16), hi = u2f(w[e] & 0xFFFF0000u);
          sm = sm + lo;
          sq = sq + lo * lo;
          sm = sm + hi;
          sq = sq + hi * hi;
        }
      }
      const float mean = sm / (float)a.n;
      const float var = sq / (float)a.n - mean * mean;
      lnst[2 * tid] = mean;
      lnst[2 * tid + 1] = 1.0f / __builtin_sqrtf(var + 1e-5f);
    }
    __syncthreads();
  }
  u32x4 xf[2][8];  // rows 32 wave + 16 p + j, k = 32 s + 8 g ..
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int s = 0; s < 8; ++s)
      xf[p][s] = *reinterpret_cast<const u32x4*>(fr_smem + (s >> 1) * 16384 +
                                                 (32 * wave + 16 * p + j) * 128 +
                                                 (((4 * (s & 1) + g) ^ (j & 7)) * 16));
  __syncthreads();  // the stages are the weights' from here

  // copies of a stage: W1's 32 rows as four 64-k blocks, W2's 256 rows of 64
  // bytes, two a line, chunk c of row r at slot c ^ ((r >> 1) & 3)
  const __amdgpu_buffer_rsrc_t w1r = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(a.W1), (short)0, -1, 0x00027000);
  const __amdgpu_buffer_rsrc_t w2r = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(a.W2), (short)0, -1, 0x00027000);
  const int w1off = (lane >> 3) * (D * 2) + wave * 128 + cchunk;
  const int w2off = (64 * wave + (lane >> 2)) * (H * 2) + ((lane & 3) ^ ((lane >> 3) & 3)) * 16;
  auto copy = [&](int ch, int slot) {
    unsigned char* const base = fr_smem + slot * FR_STAGE + wave * 4096;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          w1r, (__attribute__((address_space(3))) void*)(base + i * 1024), 16, w1off,
          ch * (32 * D * 2) + i * (8 * D * 2), 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          w2r, (__attribute__((address_space(3))) void*)(base + 16384 + i * 1024), 16, w2off,
          ch * 64 + i * (16 * H * 2), 0, 0);
  };
  copy(0, 0);
  {  // LN2 in the registers while the first stage lands
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int row = 32 * wave + 16 * p + j;
      const float mean = lnst[2 * row], inv_std = lnst[2 * row + 1];
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const int k = 32 * s + 8 * g;
        const float4 wa = *reinterpret_cast<const float4*>(a.ln2_w + k);
        const float4 wb = *reinterpret_cast<const float4*>(a.ln2_w + k + 4);
        const float4 ba = *reinterpret_cast<const float4*>(a.ln2_b + k);
        const float4 bb = *reinterpret_cast<const float4*>(a.ln2_b + k + 4);
        const float wv[8] = {wa.x, wa.y, wa.z, wa.w, wb.x, wb.y, wb.z, wb.w};
        const float bv[8] = {ba.x, ba.y, ba.z, ba.w, bb.x, bb.y, bb.z, bb.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t w = xf[p][s][e];
          const float lo = u2f(w << 16), hi = u2f(w & 0xFFFF0000u);
          const uint32_t ol = f32_to_bf16(((lo - mean) * inv_std) * wv[2 * e] + bv[2 * e]);
          const uint32_t oh = f32_to_bf16(((hi - mean) * inv_std) * wv[2 * e + 1] + bv[2 * e + 1]);
          xf[p][s][e] = ol | (oh << 16);
        }
      }
    }
  }

  floatx4 acc2[2][16];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int q = 0; q < 16; ++q) acc2[p][q] = floatx4{0.f, 0.f, 0.f, 0.f};
  uint32_t frag[2];  // of W1: chunk 4 h + g of row j
#pragma unroll
  for (int h = 0; h < 2; ++h) frag[h] = lds0 + j * 128 + (((4 * h + g) ^ (j & 7)) * 16);
  const uint32_t frag2 = lds0 + 16384 + j * 64 + ((g ^ ((j >> 1) & 3)) * 16);  // of W2
  const uint32_t b1at = lds0 + FR_B1 + 16 * g;

  for (int ch = 0; ch < H / 32; ++ch) {  // 32 hidden columns
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's copies of the stage
    lds_barrier();  // everyone's, and everyone is past the other slot's reads
    if (ch + 1 < H / 32) copy(ch + 1, (ch + 1) & 1);
    const uint32_t so = (uint32_t)(ch & 1) * FR_STAGE;
    const uint32_t f0 = frag[0] + so, f1 = frag[1] + so;
    floatx4 acc1[2][2];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int q = 0; q < 2; ++q) acc1[p][q] = floatx4{0.f, 0.f, 0.f, 0.f};
    lds_u32x4 f[2][2], bv[2];
    const uint32_t bat = b1at + ch * 128;
    bv[0] = lds_read128_at<0>(bat);
    bv[1] = lds_read128_at<64>(bat);
    auto read1 = [&](auto S) {
      constexpr int s = decltype(S)::value;
      const uint32_t at = s & 1 ? f1 : f0;
      f[s & 1][0] = lds_read128_at<(s >> 1) * 4096>(at);
      f[s & 1][1] = lds_read128_at<(s >> 1) * 4096 + 2048>(at);
    };
    auto step1 = [&](auto S) {
      constexpr int s = decltype(S)::value;
      if constexpr (s < 7) {
        read1(std::integral_constant<int, s + 1>{});
        asm volatile("s_waitcnt lgkmcnt(2)" : "+v"(f[s & 1][0]), "+v"(f[s & 1][1])::"memory");
      } else {
        asm volatile("s_waitcnt lgkmcnt(0)"
                     : "+v"(f[1][0]), "+v"(f[1][1]), "+v"(bv[0]), "+v"(bv[1])::"memory");
      }
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q)
          acc1[p][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, f[s & 1][q]), __builtin_bit_cast(bf16x8, xf[p][s]),
              acc1[p][q], 0, 0, 0);
    };
    read1(std::integral_constant<int, 0>{});
    step1(std::integral_constant<int, 0>{});
    step1(std::integral_constant<int, 1>{});
    step1(std::integral_constant<int, 2>{});
    step1(std::integral_constant<int, 3>{});
    step1(std::integral_constant<int, 4>{});
    step1(std::integral_constant<int, 5>{});
    step1(std::integral_constant<int, 6>{});
    step1(std::integral_constant<int, 7>{});
    // FF2's first weights, under GELU
    const uint32_t at2 = frag2 + so;
    lds_u32x4 w[2][2];
    w[0][0] = lds_read128_at<0>(at2);
    w[0][1] = lds_read128_at<1024>(at2);
    // A lane holds columns 16 q + 4 g .. + 3 of row j (two words a tile) and
    // takes 8 g .. + 7: swap the tiles' halves, then their odd and even
    // quarters
    lds_u32x4 hf[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      uint32_t h[2][2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = gelu<MATH_HW>(acc1[p][q][e] + u2f(bv[q][e]));
        h[q][0] = (uint32_t)f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16);
        h[q][1] = (uint32_t)f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16);
      }
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const auto s32 = __builtin_amdgcn_permlane32_swap(h[0][r], h[1][r], false, false);
        const auto s16 = __builtin_amdgcn_permlane16_swap(s32[0], s32[1], false, false);
        hf[p][r] = s16[0];
        hf[p][2 + r] = s16[1];
      }
    }
    auto step2 = [&](auto Q) {  // feature tiles 2 i, 2 i + 1
      constexpr int i = decltype(Q)::value, b = i & 1;
      if constexpr (i < 7) {
        w[b ^ 1][0] = lds_read128_at<(2 * i + 2) * 1024>(at2);
        w[b ^ 1][1] = lds_read128_at<(2 * i + 3) * 1024>(at2);
        asm volatile("s_waitcnt lgkmcnt(2)" : "+v"(w[b][0]), "+v"(w[b][1])::"memory");
      } else {
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(w[b][0]), "+v"(w[b][1])::"memory");
      }
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int p = 0; p < 2; ++p)
          acc2[p][2 * i + q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, w[b][q]), __builtin_bit_cast(bf16x8, hf[p]),
              acc2[p][2 * i + q], 0, 0, 0);
    };
    step2(std::integral_constant<int, 0>{});
    step2(std::integral_constant<int, 1>{});
    step2(std::integral_constant<int, 2>{});
    step2(std::integral_constant<int, 3>{});
    step2(std::integral_constant<int, 4>{});
    step2(std::integral_constant<int, 5>{});
    step2(std::integral_constant<int, 6>{});
    step2(std::integral_constant<int, 7>{});
  }
  __syncthreads();  // every wave is past its last reads of the stages

  // Epilogue, per wave without barriers: 16 rows of fp32 in its 16 KB, chunk c
  // of row r at slot c ^ (r & 7), and back as whole rows
  unsigned char* const epi = fr_smem + wave * 16384;
  const float4 b2v = *reinterpret_cast<const float4*>(b2s + 4 * lane);
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int m0 = m_blk + 32 * wave + 16 * p;
#pragma unroll
    for (int q = 0; q < 16; ++q)
      *reinterpret_cast<floatx4*>(epi + j * 1024 + (((4 * q + g) ^ (j & 7)) * 16)) = acc2[p][q];
    __builtin_amdgcn_wave_barrier();
#pragma unroll 8
    for (int r = 0; r < 16; ++r) {
      const int m = min(m0 + r, a.M - 1);
      float4* const at = reinterpret_cast<float4*>(epi + r * 1024 + ((lane ^ (r & 7)) * 16));
      const float4 c = *at;
      const float4 rv = *reinterpret_cast<const float4*>(a.res + (size_t)m * D + 4 * lane);
      const float4 o = make_float4((c.x + b2v.x) + rv.x, (c.y + b2v.y) + rv.y,
                                   (c.z + b2v.z) + rv.z, (c.w + b2v.w) + rv.w);
      if constexpr ((LNF & 2) != 0) *at = o;
      if (m0 + r < a.M) {
        *reinterpret_cast<float4*>(a.C + (size_t)m * D + 4 * lane) = o;
        if (a.C2)
          *reinterpret_cast<ushort4*>(a.C2 + (size_t)m * D + 4 * lane) =
              make_ushort4(f32_to_bf16(o.x), f32_to_bf16(o.y), f32_to_bf16(o.z), f32_to_bf16(o.w));
      }
    }
    if constexpr ((LNF & 2) != 0) {
      // the next layer's LN1: a half-wave per row, lane l sums elements l, l +
      // 32, ... in order, then the shuffle-down tree and lane 0's totals
      __builtin_amdgcn_wave_barrier();
      const int hw = lane >> 5, l = lane & 31;
#pragma unroll 4
      for (int i = 0; i < 8; ++i) {
        const int r = 2 * i + hw;
        float v[8], sm = 0.0f, sq = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          v[e] = *reinterpret_cast<const float*>(epi + r * 1024 + (((8 * e + (l >> 2)) ^ (r & 7)) * 16) +
                                                 4 * (l & 3));
          sm = sm + v[e];
          sq = sq + v[e] * v[e];
        }
#pragma unroll
        for (int off = 16; off > 0; off >>= 1) {
          sm = sm + __shfl_down(sm, off, 32);
          sq = sq + __shfl_down(sq, off, 32);
        }
        sm = __shfl(sm, 0, 32);
        sq = __shfl(sq, 0, 32);
        const float mean = sm / (float)a.n;
        const float var = sq / (float)a.n - mean * mean;
        const float inv_std = 1.0f / __builtin_sqrtf(var + 1e-5f);
        if (l == 0) {
          lnst[2 * (32 * wave + 16 * p + r)] = mean;
          lnst[2 * (32 * wave + 16 * p + r) + 1] = inv_std;
        }
      }
      __builtin_amdgcn_wave_barrier();
      const float4 lw = *reinterpret_cast<const float4*>(a.ln1_w + 4 * lane);
      const float4 lb = *reinterpret_cast<const float4*>(a.ln1_b + 4 * lane);
#pragma unroll 8
      for (int r = 0; r < 16; ++r) {
        const float4 c = *reinterpret_cast<const float4*>(epi + r * 1024 + ((lane ^ (r & 7)) * 16));
        const float mean = lnst[2 * (32 * wave + 16 * p + r)];
        const float inv_std = lnst[2 * (32 * wave + 16 * p + r) + 1];
        if (m0 + r < a.M)
          *reinterpret_cast<ushort4*>(a.xn + (size_t)(m0 + r) * D + 4 * lane) =
              make_ushort4(f32_to_bf16(((c.x - mean) * inv_std) * lw.x + lb.x),
                           f32_to_bf16(((c.y - mean) * inv_std) * lw.y + lb.y),
                           f32_to_bf16(((c.z - mean) * inv_std) * lw.z + lb.z),
                           f32_to_bf16(((c.w - mean) * inv_std) * lw.w + lb.w));
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// More blocks than CUs: by rows.  Up to one block per CU the 16 waves hide
// more of a block's own latencies (a forward call, two layers: 32,768 rows 1809
// us against 1824, 1000 rows 259 against 271; 33,000 rows 1950 against 1888,
// 65,535 rows 3519 against 3449).  By rows only with LN2 in the kernel.
hipError_t ffn_bf16(const FfnB16Args& args, hipStream_t s) {
  FfnB16Args a = args;
  if (a.n <= 0) a.n = a.D;  // the LayerNorms' width defaults to the row width
  if (a.M <= 0) return hipSuccess;
  const unsigned blocks = (unsigned)((a.M + 127) / 128);
  switch (a.D) {
    case 256: {
      const bool ln2 = a.ln2_w && a.ln2_b, ln1 = a.xn && a.ln1_w && a.ln1_b;
      if ((a.ln2_w || a.ln2_b) && !ln2) return hipErrorInvalidValue;
      if ((a.xn || a.ln1_w || a.ln1_b) && !ln1) return hipErrorInvalidValue;
      const bool rows = blocks > 256 && ln2;
#define BOA_FFN(F)                                                                            \
  BOA_LAUNCH((ffn_bf16_kernel<256, 128, 64, 4, 4, 4, 4, F>), dim3(blocks), dim3(1024), 0, s, a)
#define BOA_FFN_ROWS(F) \
  BOA_LAUNCH((ffn_bf16_rows_kernel<F>), dim3(blocks), dim3(256), 0, s, a)
      if (rows && ln1) BOA_FFN_ROWS(3);
      else if (rows) BOA_FFN_ROWS(1);
      else if (ln2 && ln1) BOA_FFN(3);
      else if (ln2) BOA_FFN(1);
      else if (ln1) BOA_FFN(2);
      else BOA_FFN(0);
#undef BOA_FFN_ROWS
#undef BOA_FFN
      break;
    }
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// Weight relayout for the bf16 compress GEMM: W [K][ldw_in] fp32 (the fp32
// compress layout) -> [n_pad][K] bf16, rows n >= N zero.
__global__ void b16_weight_nk_kernel(const float* __restrict__ w, int ldw_in, int N, int K,
                                     int n_pad, uint16_t* out) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)n_pad * K) return;
  const int n = (int)(idx / K), k = (int)(idx % K);
  out[idx] = n < N ? f32_to_bf16(w[(size_t)k * ldw_in + n]) : (uint16_t)0;
}

hipError_t launch_b16_weight_nk(const float* w, int ldw_in, int N, int K, int n_pad, uint16_t* out,
                                hipStream_t s) {
  if (n_pad < N || N > ldw_in) return hipErrorInvalidValue;
  const size_t n = (size_t)n_pad * K;
  BOA_LAUNCH(b16_weight_nk_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, w,
                     ldw_in, N, K, n_pad, out);
  return hipGetLastError();
}

}  // namespace boa
