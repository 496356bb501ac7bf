// fp32 GEMM on CDNA4 matrix cores with the codec's fused epilogues.
//
//   C[m][n] = act(sum_k X[m][k] * W[k][n] + bias[n]) (+ R[m][n])
//
// Rounding contract (replaces gemm_kernels.cu:283-313 of the reference):
// every output is the K-ordered fused multiply-add chain acc = fma(x_k, w_k,
// acc) starting from 0, then `acc + bias` (0 when absent), then the
// activation, then `+ residual`.  v_mfma_f32_16x16x4_f32 on gfx950 evaluates
// its four products as exactly that sequential fma chain (k ascending), and
// the kernel issues the MFMAs of one output strictly in ascending k, never
// splitting K.  The result of an output row therefore does not depend on M,
// on the tile shape or on the row's position in the tile: the compress
// (M = lanes x tile) and decompress (M = lanes) passes produce bit-identical
// logits, and so does the CPU restatement that runs the same fma chain.
//
// Operand roles: the weight tile is the MFMA A operand (16 n-rows x 4 k) and
// the activation tile the B operand (4 k x 16 m-columns), so a lane's 4
// accumulators are 4 consecutive n of one row m and the epilogue stores a
// float4 per lane.  LDS: activations [BM][BK+4] (16-byte rows for b128
// stores), weights [BK][BN+16]; both double-buffered, one barrier per K step.
#include <algorithm>
#include <type_traits>

#include "block_device.h"
#include "boa_kernels.h"
#include "coder_device.h"

namespace boa {

typedef float floatx4 __attribute__((ext_vector_type(4)));

// Epilogue mode of head.2 fused with the CDF (not a user activation): the
// block's logits rows go to LDS, and each row's (low, prob) pair of the
// next input byte is computed there (cdf_row_lowprob).
constexpr int ACT_CDF = 3;
// Epilogue modes of a 256-wide GEMM followed by a LayerNorm (see gemm_f32_ln).
constexpr int ACT_LN1 = 4, ACT_LN2 = 5;

// Eight waves per SIMD (64 VGPRs): two 16-wave blocks share a CU.
template <int BM, int BN, int WAVES_M, int WAVES_N, int BK, int ACT>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N) __attribute__((amdgpu_waves_per_eu(8, 8)))
void gemm_f32_kernel(
    const float* __restrict__ X, int ldx, const float* __restrict__ W, int ldw, float* C, int ldc,
    const float* __restrict__ bias, const float* res, int ldr, int M, int N, int K,
    int vec_store, int swizzle, CdfEpi cdf, LnEpi ln) {
  constexpr int NT = 64 * WAVES_M * WAVES_N;
  constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
  constexpr int TM = WM / 16, TN = WN / 16;
  constexpr int XS = BK + 4;   // activation row stride in LDS (floats)
  constexpr int WS = BN + 16;  // weight row stride in LDS (floats)
  constexpr int XQ = BM * (BK / 4), WQ = BK * (BN / 4);  // float4s per tile
  constexpr int XL = (XQ + NT - 1) / NT;  // float4 activation loads per thread
  constexpr int WL = (WQ + NT - 1) / NT;  // float4 weight loads per thread
  // LDS: the K loop's double-buffered tiles; the CDF epilogue reuses the
  // same words for the block's logits rows (stride LS)
  constexpr int LS = BN + 4;
  constexpr int MAIN = 2 * BM * XS + 2 * BK * WS;
  constexpr int EPI = ACT == ACT_CDF ? BM * LS : ((ACT == ACT_LN1 || ACT == ACT_LN2) ? 64 * (BN + 3) : 0);
  __shared__ __attribute__((aligned(16))) float smem[MAIN > EPI ? MAIN : EPI];
  float(*xs)[BM * XS] = reinterpret_cast<float(*)[BM * XS]>(smem);
  float(*ws)[BK * WS] = reinterpret_cast<float(*)[BK * WS]>(smem + 2 * BM * XS);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm0 = (wave / WAVES_N) * WM;
  const int wn0 = (wave % WAVES_N) * WN;
  const int g = lane >> 4, j = lane & 15;
  // Workgroup w runs on XCD w % 8.  With the swizzle, each XCD gets a
  // contiguous range of tiles (all n-blocks of its m-blocks), so an activation
  // row-block is fetched into one XCD's L2 instead of into all eight.
  const int nb = (N + BN - 1) / BN;
  int w = blockIdx.x;
  if (swizzle) {
    const int total = gridDim.x, per = total / 8;
    if (w < per * 8) w = (w % 8) * per + w / 8;
  }
  const int m_blk = (w / nb) * BM, n_blk = (w % nb) * BN;

  floatx4 acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b) acc[a][b] = floatx4{0.f, 0.f, 0.f, 0.f};

  // The block's bias values (clamped at N - 1) in LDS before the K loop, so
  // that the epilogue does not wait on global loads.
  __shared__ float sbias[BN];
  for (int c = tid; c < BN; c += NT) sbias[c] = bias ? bias[min(n_blk + c, N - 1)] : 0.0f;

  float4 xr[XL], wr[WL];
  auto load_tile = [&](int k0) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      int q = tid + i * NT;
      if (XQ % NT && q >= XQ) break;
      int row = q / (BK / 4), k4 = q % (BK / 4);
      int gm = m_blk + row;
      gm = gm < M ? gm : M - 1;  // rows past M are computed but never stored
      xr[i] = *reinterpret_cast<const float4*>(X + (size_t)gm * ldx + k0 + 4 * k4);
    }
#pragma unroll
    for (int i = 0; i < WL; ++i) {
      int q = tid + i * NT;
      if (WQ % NT && q >= WQ) break;
      int kr = q / (BN / 4), n4 = q % (BN / 4);
      wr[i] = *reinterpret_cast<const float4*>(W + (size_t)(k0 + kr) * ldw + n_blk + 4 * n4);
    }
  };
  auto store_tile = [&](int buf) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      int q = tid + i * NT;
      if (XQ % NT && q >= XQ) break;
      int row = q / (BK / 4), k4 = q % (BK / 4);
      *reinterpret_cast<float4*>(&xs[buf][row * XS + 4 * k4]) = xr[i];
    }
#pragma unroll
    for (int i = 0; i < WL; ++i) {
      int q = tid + i * NT;
      if (WQ % NT && q >= WQ) break;
      int kr = q / (BN / 4), n4 = q % (BN / 4);
      *reinterpret_cast<float4*>(&ws[buf][kr * WS + 4 * n4]) = wr[i];
    }
  };

  const int n_kt = K / BK;
  load_tile(0);
  store_tile(0);
  __syncthreads();
  for (int kt = 0; kt < n_kt; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < n_kt) load_tile((kt + 1) * BK);
#pragma unroll
    for (int kk = 0; kk < BK / 4; ++kk) {
      float af[TN], bf[TM];
#pragma unroll
      for (int b = 0; b < TN; ++b) af[b] = ws[cur][(kk * 4 + g) * WS + wn0 + b * 16 + j];
#pragma unroll
      for (int a = 0; a < TM; ++a) bf[a] = xs[cur][(wm0 + a * 16 + j) * XS + kk * 4 + g];
#pragma unroll
      for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[b], bf[a], acc[a][b], 0, 0, 0);
    }
    if (kt + 1 < n_kt) store_tile(cur ^ 1);
    __syncthreads();
  }

  if constexpr (ACT == ACT_CDF) {
    // head.2 + bias into LDS (the K loop ended with a barrier, so the tile
    // buffers are free), then per row the CDF (cdf_row_lowprob)
    static_assert(BN == 256, "one block holds whole logits rows");
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int b = 0; b < TN; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int col = wn0 + b * 16 + 4 * g + e;
          smem[(wm0 + a * 16 + j) * LS + col] = acc[a][b][e] + sbias[col];
        }
    __syncthreads();
    const int hw = tid >> 5, l = tid & 31;
    for (int r = hw; r < BM; r += NT / 32) cdf_row_lowprob(smem + r * LS, cdf, m_blk + r, M, l);
    return;
  }

  if constexpr (ACT == ACT_LN1 || ACT == ACT_LN2) {
    // Whole 256-feature rows in the block, 64 rows at a time through LDS
    // (the K loop ended with a barrier, so the tile buffers are free).  Row
    // stride RS = 257 keeps LN2's thread-per-row reads conflict-free; the
    // rows' statistics follow the 64 rows.
    static_assert(BN == 256 && BM == 128 && WAVES_M == 4, "64-row halves of whole rows");
    constexpr int D = 256, RS = D + 1;
    float* stat = smem + 64 * RS;
    for (int half = 0; half < 2; ++half) {
      if (wm0 / 64 == half) {
#pragma unroll
        for (int a = 0; a < TM; ++a) {
          const int rl = wm0 - 64 * half + a * 16 + j;
#pragma unroll
          for (int b = 0; b < TN; ++b) {
            const int n = wn0 + b * 16 + 4 * g;
#pragma unroll
            for (int e = 0; e < 4; ++e) smem[rl * RS + n + e] = acc[a][b][e] + sbias[n + e];
          }
        }
      }
      __syncthreads();
      if (ACT == ACT_LN1) {  // + residual; the sum is the residual stream's next value
#pragma unroll 1
        for (int it = 0; it < 4; ++it) {
          const int rl = (tid >> 6) + 16 * it, c = 4 * (tid & 63);
          const int m = m_blk + 64 * half + rl;
          if (m < M) {
            float* v = smem + rl * RS + c;
            const float4 r = *reinterpret_cast<const float4*>(res + (size_t)m * ldr + c);
            const float4 o = make_float4(v[0] + r.x, v[1] + r.y, v[2] + r.z, v[3] + r.w);
            *reinterpret_cast<float4*>(C + (size_t)m * ldc + c) = o;
            v[0] = o.x; v[1] = o.y; v[2] = o.z; v[3] = o.w;
          }
        }
        __syncthreads();
        // ln1_kernel's order: half-wave per row, lane l sums l, l+32, ...,
        // then the shuffle-down tree; lane 0 holds the totals
        const int hw = tid >> 5, l = tid & 31;
#pragma unroll
        for (int rr = 0; rr < 2; ++rr) {
          const int row_i = hw + 32 * rr;
          const float* row = smem + row_i * RS;
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
          if (l == 0) {
            const float mean = sm / (float)ln.n;
            const float var = sq / (float)ln.n - mean * mean;
            stat[2 * row_i] = mean;
            stat[2 * row_i + 1] = 1.0f / __builtin_sqrtf(var + 1e-5f);
          }
        }
      } else if (tid < 64) {  // ln2_kernel's order: one thread per row, elements in order
        const float* row = smem + tid * RS;
        float sm = 0.0f, sq = 0.0f;
        for (int i = 0; i < D; ++i) {
          const float e = row[i];
          sm = sm + e;
          sq = sq + e * e;
        }
        const float mean = sm / (float)ln.n;
        const float var = sq / (float)ln.n - mean * mean;
        stat[2 * tid] = mean;
        stat[2 * tid + 1] = 1.0f / __builtin_sqrtf(var + 1e-5f);
      }
      __syncthreads();
      // normalise: thread t takes columns 4(t % 64) .. +3 of rows t / 64 + 16i
#pragma unroll 1
      for (int it = 0; it < 4; ++it) {
        const int rl = (tid >> 6) + 16 * it, c = 4 * (tid & 63);
        const int m = m_blk + 64 * half + rl;
        const float mean = stat[2 * rl], inv_std = stat[2 * rl + 1];
        const float* v = smem + rl * RS + c;
        const float4 wv = *reinterpret_cast<const float4*>(ln.w + c);
        const float4 bv = *reinterpret_cast<const float4*>(ln.b + c);
        float4 o;
        o.x = ((v[0] - mean) * inv_std) * wv.x + bv.x;
        o.y = ((v[1] - mean) * inv_std) * wv.y + bv.y;
        o.z = ((v[2] - mean) * inv_std) * wv.z + bv.z;
        o.w = ((v[3] - mean) * inv_std) * wv.w + bv.w;
        if (m < M) *reinterpret_cast<float4*>(ln.out + (size_t)m * ln.ldo + c) = o;
      }
      __syncthreads();  // the next half reuses the rows
    }
    return;
  }

  // Epilogue: lane owns C[m][n .. n+3], m = wm0 + a*16 + j, n = wn0 + b*16 + 4g.
#pragma unroll
  for (int a = 0; a < TM; ++a) {
    const int m = m_blk + wm0 + a * 16 + j;
    if (m >= M) continue;
#pragma unroll
    for (int b = 0; b < TN; ++b) {
      const int n = n_blk + wn0 + b * 16 + 4 * g;
      if (n >= N) continue;
      float v[4] = {acc[a][b][0], acc[a][b][1], acc[a][b][2], acc[a][b][3]};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float t = v[e] + sbias[wn0 + b * 16 + 4 * g + e];
        if (ACT == ACT_GELU) t = gelu(t);
        else if (ACT == ACT_RELU) t = fmaxf(0.0f, t);
        v[e] = t;
      }
      if (vec_store) {
        if (res) {
          float4 r = *reinterpret_cast<const float4*>(res + (size_t)m * ldr + n);
          v[0] = v[0] + r.x; v[1] = v[1] + r.y; v[2] = v[2] + r.z; v[3] = v[3] + r.w;
        }
        *reinterpret_cast<float4*>(C + (size_t)m * ldc + n) = make_float4(v[0], v[1], v[2], v[3]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (n + e >= N) break;
          float t = v[e];
          if (res) t = t + res[(size_t)m * ldr + n + e];
          C[(size_t)m * ldc + n + e] = t;
        }
      }
    }
  }
}

// ------------------------------------------------------- persistent blocks
// 256 rows x 256 features a tile, eight waves of 64 x 128 (two per SIMD), one
// block per CU that walks over tiles.  fp32 MFMAs and vector instructions
// share the SIMD's FMA units (they do not overlap, see boa_math.h), so the K
// loop holds little but MFMAs: 32-k stages are copied straight to LDS (no
// staging registers or LDS stores), most of an address is an instruction
// offset, and a 4-k step's 32 MFMAs read 12 operand dwords with six LDS
// instructions.  The loop runs at the MFMA rate (6.9 us a stage against 6.8);
// what costs besides is the output (256 KB a tile in 25 us, every CU at the
// same time, against 55 us of MFMAs at K = 256): the next tile's stages 0 and
// 1 are copied ahead of the stores, which drain behind them.  Keeping half a
// tile in registers and storing it between the next one's k-steps needed
// more registers than there are (spills; with 64 x 64 waves, where it fits,
// the loop took 11 % longer).
// LDS: two 64 KB stages.  Activations: rows of 128 bytes, the 16-byte chunk
// c of row r at slot c ^ ((r >> 1) & 7); weights: k rows of 1 KB, the 64-byte
// group q of row k at slot q ^ (k & 3): the 64 lanes of an operand read fall
// on the 64 banks either way.  Then the bias of every feature.
struct GfTile {
  __amdgpu_buffer_rsrc_t x, w;  // the tile's activation rows, its weight columns
  int m, n;
};
constexpr int GF_X = 32768, GF_STAGE = 2 * GF_X, GF_MAX_N = 2048;
constexpr int GF_LDS = 2 * GF_STAGE + 4 * GF_MAX_N;

template <int ACT>
__global__ __launch_bounds__(512, 2) void gemm_f32_persist_kernel(GemmArgs a, int m_blocks) {
  constexpr int TM = 4, TN = 8;
  __shared__ __attribute__((aligned(16))) unsigned char gf_smem[GF_LDS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, j = lane & 15;
  const int wm = wave >> 1, wn = wave & 1;  // rows 64 wm .., features 128 wn ..
  float* const sbias = reinterpret_cast<float*>(gf_smem + 2 * GF_STAGE);
  for (int c = tid; c < a.N; c += 512) sbias[c] = a.bias ? a.bias[c] : 0.0f;
  __syncthreads();

  // Tiles: XCD x (blocks x, x + 8, ..) takes the m blocks x per .. x per +
  // per - 1, features fastest, so that the tiles in flight on an XCD share
  // activation rows and weights in its L2.
  const int nb = a.N / 256, per = (m_blocks + 7) / 8;
  const int x0 = (blockIdx.x & 7) * per;
  const int n_tiles = max(0, min(per, m_blocks - x0)) * nb;  // of this XCD
  const int step = gridDim.x / 8;
  const int n_st = a.K / 32;

  // copies: copy i of a wave fills rows 32 wave + 8 i .. + 7 of a stage's
  // activations and k row 4 wave + i of its weights
  const int xrow = (32 * wave + (lane >> 3)) * a.ldx * 4;
  const int xoff[2] = {xrow + ((lane & 7) ^ (lane >> 4)) * 16,
                       xrow + ((lane & 7) ^ (4 + (lane >> 4))) * 16};
  auto tile_at = [&](int t) {
    GfTile T;
    // the last rows' tile starts early: rows that two tiles hold get the same
    // values from both
    T.m = min((x0 + t / nb) * 256, a.M - 256);
    T.n = (t % nb) * 256;
    T.x = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.X) + (size_t)T.m * a.ldx,
                                            (short)0, -1, 0x00027000);
    T.w = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.W) + T.n, (short)0, -1,
                                            0x00027000);
    return T;
  };
  auto copy_part = [&](const GfTile& T, int st, int slot, int i) {
    unsigned char* const base = gf_smem + slot * GF_STAGE + wave * 4096 + i * 1024;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        T.x, (__attribute__((address_space(3))) void*)base, 16, xoff[i & 1],
        st * 128 + 32 * i * a.ldx, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        T.w, (__attribute__((address_space(3))) void*)(base + GF_X), 16, (lane * 16) ^ (64 * i),
        (st * 32 + 4 * wave + i) * a.ldw * 4, 0, 0);
  };
  auto copy = [&](const GfTile& T, int st, int slot) {
#pragma unroll
    for (int i = 0; i < 4; ++i) copy_part(T, st, slot, i);
  };
  // operand addresses: activations of 4-k step s at xat ^ 16 s (row tiles are
  // instruction offsets), weights of feature tiles q and q + 4 at wat ^ 64 q
  // (so are steps); the stages start at multiples of 128 bytes
  const uint32_t lds0 = lds_addr(gf_smem);
  const uint32_t xat = lds0 + wm * 8192 + j * 128 + ((j >> 1) & 7) * 16 + 4 * g;
  const uint32_t wat = lds0 + GF_X + wn * 512 + g * 1024 + g * 64 + 4 * j;

  int t = blockIdx.x >> 3;
  if (t >= n_tiles) return;  // the whole block
  GfTile T = tile_at(t);
  copy(T, 0, 0);
  copy(T, 1, 1);
  int slot = 0;

  bool stores = false;  // the last epilogue's 32 stores, behind copies 0 and 1
  while (true) {
    floatx4 acc[TM][TN];
#pragma unroll
    for (int p = 0; p < TM; ++p)
#pragma unroll
      for (int q = 0; q < TN; ++q) acc[p][q] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int t_next = t + step;
    const bool more = t_next < n_tiles;
    const GfTile Tn = more ? tile_at(t_next) : T;
    for (int st = 0; st < n_st; ++st, slot ^= 1) {
      // this wave's copies of the stage have landed (newer may be, at stage 0,
      // the eight copies of stage 1 and the stores, at stage 1 those), then
      // everyone's
      if (st == 0) {
        if (stores) asm volatile("s_waitcnt vmcnt(40)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
      } else if (st == 1 && stores) {
        asm volatile("s_waitcnt vmcnt(32)" ::: "memory");
      } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      lds_barrier();  // and everyone is past the other slot's reads
      const bool here = st + 1 < n_st, copying = st > 0 && (here || more);
      const GfTile& Tc = here ? T : Tn;
      const int stc = here ? st + 1 : 0;
      const uint32_t so = (uint32_t)slot * GF_STAGE;
      const uint32_t wa = wat + so, xa = xat + so;
      lds_u32x2 xf[2][2], wf[2][4];
      auto read = [&](auto S) {
        constexpr int s = decltype(S)::value, b = s & 1;
        const uint32_t x = xa ^ (16 * s);
        xf[b][0] = lds_read2_at<0, 8>(x);    // row tiles 0, 1
        xf[b][1] = lds_read2_at<16, 24>(x);  // 2, 3
        wf[b][0] = lds_read2_at<16 * s, 16 * s + 1>(wa);  // feature tiles 0, 4
        wf[b][1] = lds_read2_at<16 * s, 16 * s + 1>(wa ^ 64);
        wf[b][2] = lds_read2_at<16 * s, 16 * s + 1>(wa ^ 128);
        wf[b][3] = lds_read2_at<16 * s, 16 * s + 1>(wa ^ 192);
      };
      auto kstep = [&](auto S) {
        constexpr int s = decltype(S)::value, b = s & 1;
        // the next step's operands are read while this one multiplies
        if constexpr (s < 7) read(std::integral_constant<int, s + 1>{});
        asm volatile("s_waitcnt lgkmcnt(%6)"
                     : "+v"(xf[b][0]), "+v"(xf[b][1]), "+v"(wf[b][0]), "+v"(wf[b][1]),
                       "+v"(wf[b][2]), "+v"(wf[b][3])
                     : "n"(s < 7 ? 6 : 0)
                     : "memory");
        if constexpr (s < 4)
          if (copying) copy_part(Tc, stc, slot ^ 1, s);
#pragma unroll
        for (int q = 0; q < TN; ++q)
#pragma unroll
          for (int p = 0; p < TM; ++p)
            acc[p][q] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                u2f(wf[b][q & 3][q >> 2]), u2f(xf[b][p >> 1][p & 1]), acc[p][q], 0, 0, 0);
      };
      read(std::integral_constant<int, 0>{});
      kstep(std::integral_constant<int, 0>{});
      kstep(std::integral_constant<int, 1>{});
      kstep(std::integral_constant<int, 2>{});
      kstep(std::integral_constant<int, 3>{});
      kstep(std::integral_constant<int, 4>{});
      kstep(std::integral_constant<int, 5>{});
      kstep(std::integral_constant<int, 6>{});
      kstep(std::integral_constant<int, 7>{});
    }

    // the tile's values: lane (g, j) has features n0 + 16 q .. + 3 of rows
    // m0 + 16 p, stored in 64-byte pieces
    if (more) {
      lds_barrier();  // everyone is past the last stage's reads
      copy(Tn, 1, slot ^ 1);
    }
    const uint32_t bat = lds_addr(sbias) + (T.n + 128 * wn + 4 * g) * 4;
    const int m0 = T.m + 64 * wm + j, n0 = T.n + 128 * wn + 4 * g;
    auto feature_tile = [&](auto Q) {
      constexpr int q = decltype(Q)::value;
      lds_u32x4 bv = lds_read128_at<64 * q>(bat);
      asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(bv)::"memory");
#pragma unroll
      for (int p = 0; p < TM; ++p) {
        floatx4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float x = acc[p][q][e] + u2f(bv[e]);
          if (ACT == ACT_GELU) x = gelu(x);
          else if (ACT == ACT_RELU) x = fmaxf(0.0f, x);
          v[e] = x;
        }
        *reinterpret_cast<floatx4*>(a.C + (size_t)(m0 + 16 * p) * a.ldc + n0 + 16 * q) = v;
      }
    };
    feature_tile(std::integral_constant<int, 0>{});
    feature_tile(std::integral_constant<int, 1>{});
    feature_tile(std::integral_constant<int, 2>{});
    feature_tile(std::integral_constant<int, 3>{});
    feature_tile(std::integral_constant<int, 4>{});
    feature_tile(std::integral_constant<int, 5>{});
    feature_tile(std::integral_constant<int, 6>{});
    feature_tile(std::integral_constant<int, 7>{});
    stores = true;
    if (!more) break;
    t = t_next;
    T = Tn;
  }
}

// What the kernel's addressing takes: whole 256-feature tiles up to GF_MAX_N,
// whole 32-k stages (two at least), 16-byte rows, a tile's rows and the
// weights within 32-bit byte offsets, a tile's worth of rows, no residual.
static bool f32_persist_fits(const GemmArgs& a) {
  return a.N % 256 == 0 && a.N <= GF_MAX_N && a.K % 32 == 0 && a.K >= 64 && a.ldx % 4 == 0 &&
         a.ldw % 4 == 0 && a.ldw >= a.N && a.ldx <= (1 << 20) &&
         (long long)a.K * a.ldw < (1 << 28) && a.ldc % 4 == 0 && !a.res && a.M >= 256 &&
         a.X != a.C;
}

// Blocks of bm x bn that the fullest of the 256 CUs gets (they are dispatched
// round-robin).  The MFMAs of a CU's blocks run one after another however many
// are resident, so a launch takes about that number times a block's time; a
// block too many for the CUs costs a whole one.
static long long cu_blocks(const GemmArgs& a, int bm, int bn) {
  return (((long long)a.M + bm - 1) / bm * ((a.N + bn - 1) / bn) + 255) / 256;
}

// Whether the persistent blocks beat the others.  `rounds`: tiles of the
// busiest CU (the 32 blocks of an XCD share its m blocks).  Below 16,384 rows
// the alternatives are fine-grained, and the tiles have to fill their rounds:
// N 2048 K 512 at 7177 rows (0.91 of a round) 132.5 us against 165.2, N 1024 K
// 256 at 14,441 rows (0.89) 72.6 against 86.1, at 9604 (0.59) 70.4 against
// 57.0.  From there on against two 128 x 256 blocks a tile, which take 1 /
// 0.91 of a tile's time; with K below 256 (the output is most of it) 1 / 0.88,
// with GELU, whose VALU work two resident blocks overlap in part, 1 / 0.96.
// 2700 points of 16,384 to 800,000 rows, 14 shapes: never more than 4.5 %
// slower than the 128 x 256 blocks (GELU, K 64), 5.2 % faster in the mean;
// with one line for all at 0.85 of whole rounds up to 11 % slower (GELU, K 64
// at 283,705 rows 181.8 us against 163.9; K 512 N 2048 at 35,584 rows 678
// against 643).
static bool f32_persist_pays(const GemmArgs& a) {
  const long long mb = ((long long)a.M + 255) / 256, nb = a.N / 256;
  const long long rounds = ((mb + 7) / 8 * nb + 31) / 32;
  if (a.M < 16384) return 100 * mb * nb >= 85 * 256 * rounds;
  const int cost = a.act == ACT_GELU ? 96 : a.K < 256 ? 88 : 91;
  return 2 * rounds * cost <= 100 * cu_blocks(a, 128, 256);
}

template <int ACT>
static hipError_t f32_persist_go(const GemmArgs& a, hipStream_t s) {
  const int m_blocks = (int)(((long long)a.M + 255) / 256);
  // a multiple of eight blocks (one share of the XCDs each), at most one per CU
  const long long tiles = (long long)((m_blocks + 7) / 8) * (a.N / 256) * 8;
  const unsigned grid = (unsigned)std::min<long long>(tiles, 256);
  BOA_LAUNCH((gemm_f32_persist_kernel<ACT>), dim3(grid), dim3(512), 0, s, a, m_blocks);
  return hipGetLastError();
}

template <int BM, int BN, int WM_, int WN_, int BK>
static hipError_t launch_cfg(const GemmArgs& a, hipStream_t s, int swizzle = 1) {
  if (a.K % BK || a.ldw < (a.N + BN - 1) / BN * BN) return hipErrorInvalidValue;
  const long long tiles = (long long)((a.N + BN - 1) / BN) * ((a.M + BM - 1) / BM);
  if (tiles >= (1ll << 31)) return hipErrorInvalidValue;
  int vec = (a.N % 4 == 0) && (a.ldc % 4 == 0) && (!a.res || a.ldr % 4 == 0);
  // the activation is a template argument: the epilogue has no branch on it
#define BOA_GEMM_GO(ACTv)                                                                     \
  BOA_LAUNCH((gemm_f32_kernel<BM, BN, WM_, WN_, BK, ACTv>), dim3((unsigned)tiles),     \
                     dim3(64 * WM_ * WN_), 0, s, a.X, a.ldx, a.W, a.ldw, a.C, a.ldc, a.bias,   \
                     a.res, a.ldr, a.M, a.N, a.K, vec, swizzle, CdfEpi{}, LnEpi{})
  switch (a.act) {
    case ACT_NONE: BOA_GEMM_GO(ACT_NONE); break;
    case ACT_GELU: BOA_GEMM_GO(ACT_GELU); break;
    case ACT_RELU: BOA_GEMM_GO(ACT_RELU); break;
    default: return hipErrorInvalidValue;
  }
#undef BOA_GEMM_GO
  return hipGetLastError();
}

// Tile choice only changes the schedule, never the numerics (see above).
// Large M (a compress tile), N >= 256: persistent 256x256 blocks where they
// pay (TFLOP/s at 1.6 M rows, against 128x256 blocks of 16 waves: K 256 N 1024
// 113.5 -> 126.6, with GELU at 400,000 rows 98.6 -> 105.9), the 128x256 blocks
// otherwise (the LayerNorm epilogues and FF2's residual, 256 wide: equal to
// 2 % at whole rounds of the CUs, slower between, and their epilogues overlap
// the other resident block's MFMAs); 128x64 with 8 waves for the narrow x_proj.
// Fewer rows (a forward call of some thousand tokens): 32x32 blocks with four
// waves, unless the fullest CU gets no more work in larger ones, whose MFMAs
// wait for fewer operands: 128x64 blocks hold eight times the work and are 10
// to 17 % cheaper for it from K 256 on, so they have to come to less than 1/7 of
// the number; 64x32 blocks of eight waves twice, 2 to 5 % cheaper from K 512
// on, so they have to come to half of it; at K 256 that holds for whole rounds
// of the four that a CU holds (N 256, 8064 rows, 4 on the fullest: 16.4 us
// against 17.7; 10,180 rows, 5: 21.1 against 20.6), below nowhere.  One of
// either on a CU exposes its latency (N 256 K 512, 3000 rows: 27.7 us of
// 128x64, 14.1 of 32x32).  us of 128x64 / 64x32 / 32x32 (blocks on the fullest
// CU): N 1024 K 256 at 8064 rows 46.7 / 50.5 / 50.8 (4, 16, 32), at 6387 46.1 /
// 42.0 / 41.6 (4, 13, 25), at 1178 16.4 / 12.8 / 11.4 (2, 3, 5); N 256 K 1024
// at 8064 rows 51.9 / 49.6 / 53.0 (1, 4, 8), at 4248 50.3 / 38.1 / 34.0 (1, 3,
// 5); N 2048 K 512 at 10,180 rows 192.8 / 222.4 / 231.5 (10, 40, 80).  2800
// points of 64 to 16,383 rows, 30 shapes: at most 1.5 % slower than 32x32, up
// to 18 % faster.
int gemm_f32_config(const GemmArgs& a) {
  if (a.M >= 16384) return a.N >= 256 ? 0 : 1;
  const long long n128 = cu_blocks(a, 128, 64), n64 = cu_blocks(a, 64, 32),
                  n32 = cu_blocks(a, 32, 32);
  if (a.K >= 256 && n128 >= 2 && 7 * n128 < n32) return 1;
  if (a.K % 32 == 0 && 2 * n64 == n32 &&
      (a.K >= 512 ? n64 >= 2 : a.K >= 256 && n64 % 4 == 0))
    return 3;
  return 2;
}

// head.2 of a compress tile fused with the CDF: rows of 256 logits (acc +
// bias) stay in LDS and each row's (low, prob) of the next byte is written
// to cdf.lowprob.  64-row blocks keep two blocks per CU (66.5 KB of LDS).
hipError_t gemm_f32_head_cdf(const GemmArgs& a, const CdfEpi& cdf, hipStream_t s) {
  if (a.M <= 0) return hipSuccess;
  if (a.N != 256 || a.K % 16 || a.ldx % 4 || a.ldw % 4 || !cdf.lowprob || cdf.T < 1)
    return hipErrorInvalidValue;
  constexpr int BM = 64, BN = 256;  // 128-row blocks (one per CU) measured the same
  if (a.ldw < BN) return hipErrorInvalidValue;
  const long long tiles = (a.M + BM - 1) / BM;
  if (tiles >= (1ll << 31)) return hipErrorInvalidValue;
  BOA_LAUNCH((gemm_f32_kernel<BM, BN, 4, 4, 16, ACT_CDF>), dim3((unsigned)tiles), dim3(1024),
                     0, s, a.X, a.ldx, a.W, a.ldw, nullptr, 0, a.bias, nullptr, 0, a.M, a.N, a.K,
                     0, 1, cdf, LnEpi{});
  return hipGetLastError();
}

hipError_t gemm_f32_ln(const GemmArgs& a, const LnEpi& ln, hipStream_t s) {
  if (a.M <= 0) return hipSuccess;
  if (a.N != 256 || a.K % 16 || a.ldx % 4 || a.ldw < 256 || a.ldw % 4 || !ln.out || !ln.w ||
      !ln.b || ln.ldo % 4 || ln.ldo < 256 || (ln.mode == 1 && (!a.res || !a.C || a.ldr % 4 ||
      a.ldc % 4)))
    return hipErrorInvalidValue;
  const long long tiles = (a.M + 127) / 128;
  if (tiles >= (1ll << 31)) return hipErrorInvalidValue;
  if (ln.mode == 1)
    BOA_LAUNCH((gemm_f32_kernel<128, 256, 4, 4, 16, ACT_LN1>), dim3((unsigned)tiles), dim3(1024),
               0, s, a.X, a.ldx, a.W, a.ldw, a.C, a.ldc, a.bias, a.res, a.ldr, a.M, a.N, a.K, 1, 1,
               CdfEpi{}, ln);
  else if (ln.mode == 2)
    BOA_LAUNCH((gemm_f32_kernel<128, 256, 4, 4, 16, ACT_LN2>), dim3((unsigned)tiles), dim3(1024),
               0, s, a.X, a.ldx, a.W, a.ldw, a.C, a.ldc, a.bias, a.res, a.ldr, a.M, a.N, a.K, 1, 1,
               CdfEpi{}, ln);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t gemm_f32(const GemmArgs& a, hipStream_t s) {
  if (a.M <= 0 || a.N <= 0) return hipSuccess;
  if (a.K % 16 != 0 || a.ldx % 4 != 0 || a.ldw % 4 != 0) return hipErrorInvalidValue;
  if (f32_persist_fits(a) && f32_persist_pays(a)) {
    switch (a.act) {
      case ACT_NONE: return f32_persist_go<ACT_NONE>(a, s);
      case ACT_GELU: return f32_persist_go<ACT_GELU>(a, s);
      case ACT_RELU: return f32_persist_go<ACT_RELU>(a, s);
      default: return hipErrorInvalidValue;
    }
  }
  switch (gemm_f32_config(a)) {
    case 0: return launch_cfg<128, 256, 4, 4, 16>(a, s);
    case 1: return launch_cfg<128, 64, 4, 2, 16>(a, s);
    case 3: return launch_cfg<64, 32, 4, 2, 32>(a, s);
    default:
      return a.K % 32 == 0 ? launch_cfg<32, 32, 2, 2, 32>(a, s) : launch_cfg<32, 32, 2, 2, 16>(a, s);
  }
}

}  // namespace boa
