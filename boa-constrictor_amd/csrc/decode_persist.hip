// Persistent decode for small models (d_model 64): one block of 1024 threads
// owns 16 lanes and runs every decode step of a batch for them -- embedding,
// the L blocks, the head, the CDF, the symbol search and the coder advance --
// with the step's activations in LDS and no synchronisation between blocks
// (decode lanes are independent).  It replaces the step's launch chain
// (6 L + 3 kernels per step, each a few microseconds of launch and drain at
// this size) by block barriers.
//
// It covers, for one batch, what the reference's decompress loop runs per
// step as a graph replay (portability_solved_cpp/boa.cpp:672-774):
// BoaPredictorGPU::step_batch (boa_gpu.hpp:1034-1053; blocks :835-843,
// Mamba step :227-247, feed-forward :739-764, head :1049-1052) and the fused
// decode step of range_coder_kernels.cu:491-629 (CDF, symbol search, coder
// advance).
//
// Every operation is the one of the step kernels (decode.hip, coder.hip),
// with the same operand arrangement and k order in every MFMA chain, the
// same LayerNorm reduction orders and the same epilogue order (bias,
// activation, residual), so the logits, and therefore the symbols, are
// bit-identical to the launch-chain step and to the compress pass.  The
// state layouts in global memory (conv, SSM, coder, token) are those of the
// step kernels, so either path can continue where the other stopped.
#include "block_device.h"
#include "coder_device.h"

namespace boa {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int PL = 16;  // MFMA rows of the block's tiles: the lane capacity of its LDS rows

// One 16 x 16 tile of the block's 16 lanes and features n0 .. n0 + 15.  A:
// activations in LDS, k-blocked with lane capacity 16 (feature k of lane m at
// ((k / 16) 16 + m) 16 + dperm(k % 16)); W: k-blocked decode weights in
// global memory with capacity ldw.  Lane (i, g) feeds W row n0 + i and lane
// i's float4 g of every 16-k block, four MFMAs per block in k order -- the
// arrangement of dec_mainloop.  The weights do not depend on the step: a wave
// loads its tile's (pd_load) phases ahead of the MFMAs (pd_mac), and the
// barriers between wait for LDS only.
template <int KB>
__device__ __forceinline__ void pd_load(float4* wv, const float* __restrict__ W, int ldw, int n0,
                                        int i, int g) {
  // uniform base, one 32-bit lane offset for all loads
  const char* base = reinterpret_cast<const char*>(W) + n0 * 64;
  const uint32_t off = (uint32_t)(i * 64 + g * 16);
#pragma unroll
  for (int q = 0; q < KB; ++q)
    wv[q] = *reinterpret_cast<const float4*>(base + (size_t)q * ldw * 64 + off);
}

// Registers that another wave fills: any value, from no instruction (without
// it they would keep, and spill, the last loop iteration's)
template <int KB>
__device__ __forceinline__ void pd_none(float4* wv) {
#pragma unroll
  for (int q = 0; q < KB; ++q)
    asm volatile("" : "=v"(wv[q].x), "=v"(wv[q].y), "=v"(wv[q].z), "=v"(wv[q].w));
}

template <int KB>
__device__ __forceinline__ floatx4 pd_mac(const float* A, const float4* wv, int i, int g) {
  floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < KB; ++q) {
    const float4 bv = reinterpret_cast<const float4*>(A + (q * PL + i) * 16)[g];
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[q].x, bv.x, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[q].y, bv.y, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[q].z, bv.z, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[q].w, bv.w, acc, 0, 0, 0);
  }
  return acc;
}

// The tile's float4 for lane i: k-blocked outputs (permuted weight rows) hold
// feature n0 + 4 e + g in component e, at in-block position 4 g + e.
__device__ __forceinline__ float4* pd_out(float* base, int n0, int i, int g) {
  return reinterpret_cast<float4*>(base + ((n0 >> 4) * PL + i) * 16) + g;
}

// LayerNorm statistics of the block's 16 lanes (xs k-blocked, d features).
// MODE 1 (LN1): 16 threads per lane, the reference's warp-tree order, stats =
// (mean, rstd).  MODE 2 (LN2): sequential sums (one thread for the sum, one
// for the squares), stats = (sum, sum of squares).  The orders of
// dec_ln_gemm_kernel.  n: the LayerNorm's width (features n .. d-1 are zero).
template <int MODE, int NB>
__device__ __forceinline__ void pd_ln_stats(const float* xs, float* stats, int tid, int n) {
  constexpr int d = NB * 16;
  if (MODE == 1) {
    if (tid >= 16 * PL) return;
    const int lj = tid >> 4, l = tid & 15;
    auto xat = [&](int f) { return xs[((f >> 4) * PL + lj) * 16 + dperm(f & 15)]; };
    float s0 = 0.0f, q0 = 0.0f, s1 = 0.0f, q1 = 0.0f;
#pragma unroll
    for (int f = l; f < d; f += 32) {
      const float x = xat(f);
      s0 = s0 + x;
      q0 = q0 + x * x;
    }
#pragma unroll
    for (int f = l + 16; f < d; f += 32) {
      const float x = xat(f);
      s1 = s1 + x;
      q1 = q1 + x * x;
    }
    float sum = s0 + s1, sq = q0 + q1;
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) {
      sum = sum + __shfl_down(sum, off, 16);
      sq = sq + __shfl_down(sq, off, 16);
    }
    if (l == 0) {
      const float mean = sum / (float)n;
      const float var = sq / (float)n - mean * mean;
      stats[2 * lj] = mean;
      stats[2 * lj + 1] = 1.0f / __builtin_sqrtf(var + 1e-5f);
    }
  } else {
    if (tid >= 2 * PL) return;
    const int lj = tid & 15;
    const bool squares = tid >= PL;
    float acc = 0.0f;
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const float4* row = reinterpret_cast<const float4*>(xs + (q * PL + lj) * 16);
      const float4 c0 = row[0], c1 = row[1], c2 = row[2], c3 = row[3];
      // position p holds feature dperm(p): features 16 q + 0, 1, 2, ... sit
      // at positions 0, 4, 8, 12, 1, 5, ...
      const float fv[16] = {c0.x, c1.x, c2.x, c3.x, c0.y, c1.y, c2.y, c3.y,
                            c0.z, c1.z, c2.z, c3.z, c0.w, c1.w, c2.w, c3.w};
#pragma unroll
      for (int j = 0; j < 16; ++j) acc = acc + (squares ? fv[j] * fv[j] : fv[j]);
    }
    stats[2 * lj + (squares ? 1 : 0)] = acc;
  }
}

template <int MODE, int NB>
__device__ __forceinline__ void pd_ln_apply(const float* xs, float* xn, const float* stats,
                                            const float* __restrict__ w,
                                            const float* __restrict__ b, int tid, int n) {
  for (int p = tid; p < NB * 256; p += 1024) {
    const int q = p >> 8, m = (p >> 4) & 15, f = 16 * q + dperm(p & 15);
    float mean, rstd;
    if (MODE == 1) {
      mean = stats[2 * m];
      rstd = stats[2 * m + 1];
    } else {
      mean = stats[2 * m] / (float)n;
      const float var = stats[2 * m + 1] / (float)n - mean * mean;
      rstd = 1.0f / __builtin_sqrtf(var + 1e-5f);
    }
    xn[p] = ((xs[p] - mean) * rstd) * w[f] + b[f];
  }
}

}  // namespace

// LP lanes per block (16, 8 or 4): rows LP .. 15 of every MFMA tile are
// inert (an MFMA output column depends on its own row of activations only;
// their loads read a lane of this block and nothing is stored for them), so
// a block's matrix-core chains cost the same for any LP, while its VALU
// phases (the scan's 16 exponentials per channel, GELU, the CDF) scale with
// LP.  Fewer lanes per block spread those phases over more CUs.
//
// What bounds it: a serial chain.  A step is 10 L + 4 phases between barriers
// (24 at two layers), in which an MFMA chain of K / 4 takes 42 cycles per MFMA
// (256 features at once: 2048 cycles a SIMD), and the elementwise phases their
// instruction latency.
// So everything that does not depend on the phase before is out of the chain:
// weights and recurrent states are loaded phases ahead into registers, MFMA
// outputs of LP < 16 lanes are spread over the wave before GELU and the conv
// step, the coder's division runs under out_proj, and the symbol search stays
// in the registers of the CDF (µs per step at 2 layers: 1 to 512 lanes 34.7 ->
// 25.5, 1024 lanes 42.8 -> 27.8, 4096 lanes 58.7 -> 39.9; 2 lanes per block
// gave 25.0 up to 300 lanes, 26.5 at 512).
template <int NB, int RB, int LP>
__global__ __launch_bounds__(1024) void dec_persist_kernel(PersistArgs a) {
  static_assert(LP == 4 || LP == 8 || LP == 16, "lanes per block");
  constexpr int LSH = LP == 4 ? 2 : LP == 8 ? 3 : 4;
  constexpr int VPL = LP / 4;  // values per thread of PD_SPREAD
  constexpr int d = NB * 16, DI = 2 * d, NBI = 2 * NB, NBF = 4 * NB, DS = 16;
  constexpr int NBX = (RB + 2 * DS + 15) / 16;  // 16-blocks of the x_proj row
  constexpr int RW = NBX * 16 + 1;              // LDS row stride of the x_proj rows
  __shared__ __align__(16) float xs[NB * 256];   // residual stream x
  __shared__ __align__(16) float xn[NB * 256];   // LayerNorm output
  __shared__ __align__(16) float zs[NBI * 256];  // z half of in_proj
  __shared__ __align__(16) float cvs[NBI * 256]; // conv + SiLU output
  __shared__ __align__(16) float rwn[PL * RW];   // x_proj rows (dt_in, B, C), natural order
  __shared__ __align__(16) float ys[NBI * 256];  // scan output
  __shared__ __align__(16) float os[NB * 256];   // out_proj / head1 output
  __shared__ __align__(16) float hid[NBF * 256]; // FF1 output
  __shared__ __align__(16) float lg[PL * 256];   // logits, row-major
  __shared__ float stats[2 * PL];
  __shared__ int tok_s[PL];
  // per-channel parameters of every layer and the head biases, staged once
  constexpr int O_LN1W = 0, O_LN1B = O_LN1W + d, O_BIN = O_LN1B + d, O_CONVW = O_BIN + 2 * DI,
                O_CONVB = O_CONVW + 4 * DI, O_BDT = O_CONVB + DI, O_DD = O_BDT + DI,
                O_NAQ = O_DD + DI, O_WDTQ = O_NAQ + DS * DI, O_BOUT = O_WDTQ + RB * DI,
                O_LN2W = O_BOUT + d, O_LN2B = O_LN2W + d, O_B1 = O_LN2B + d, O_B2 = O_B1 + 4 * d,
                PSZ = O_B2 + d;
  __shared__ __align__(16) float prm[PERSIST_MAX_LAYERS * PSZ];
  __shared__ float hb1[d], hb2[256];
  const int tid0 = threadIdx.x;
  const int m0 = blockIdx.x * LP;
  // coder: half-wave h < 16 decodes lane m0 + h; its lane 0 holds the state
  const int half = tid0 >> 5, l = tid0 & 31;
  const int mh = m0 + half;
  const bool coder_lane = half < LP && mh < a.lanes;
  RcDec st{};
  if (coder_lane && l == 0) st = a.states[mh];
  const int len_h = coder_lane ? a.lens[mh] : 0;
  // the lane's stream, read once (the byte stores of the step loop could
  // alias these arrays, so the compiler would reload them every step) and
  // its next word loaded ahead (dec_advance_ahead)
  const uint32_t* pin = nullptr;
  int32_t pn = 0;
  uint32_t nw = 0;
  uint32_t target0 = 0;
  if (coder_lane && l == 0) {
    pin = a.payload + a.offsets[mh];
    pn = a.sizes[mh];
    nw = st.read_idx_words < pn ? pin[st.read_idx_words] : 0u;
  }
  if (tid0 < PL) tok_s[tid0] = tid0 < LP ? a.tok[min(m0 + tid0, a.lanes - 1)] : 0;
  auto stage = [&](float* dst, const float* __restrict__ src, int n) {
    for (int k = tid0; k < n; k += 1024) dst[k] = src[k];
  };
#pragma unroll
  for (int li = 0; li < PERSIST_MAX_LAYERS; ++li) {
    if (li >= a.L) break;
    const PersistLayer& P = a.layer[li];
    float* q = prm + li * PSZ;
    stage(q + O_LN1W, P.ln1_w, d); stage(q + O_LN1B, P.ln1_b, d);
    stage(q + O_BIN, P.b_in, 2 * DI); stage(q + O_CONVW, P.conv_w, 4 * DI);
    stage(q + O_CONVB, P.conv_b, DI); stage(q + O_BDT, P.b_dt, DI); stage(q + O_DD, P.dd, DI);
    stage(q + O_NAQ, P.na_q, DS * DI); stage(q + O_WDTQ, P.wdt_q, RB * DI);
    stage(q + O_BOUT, P.b_out, d); stage(q + O_LN2W, P.ln2_w, d); stage(q + O_LN2B, P.ln2_b, d);
    stage(q + O_B1, P.b1, 4 * d); stage(q + O_B2, P.b2, d);
  }
  stage(hb1, a.hb1, d);
  stage(hb2, a.hb2, 256);
  __syncthreads();

  static_assert(2 * NBI == 16 && NBF == 16, "one in_proj and FF1 tile per wave");
  // Weight tiles in flight: every wave's tile of in_proj, FF1, then the next
  // layer's in_proj or head2; and, of waves 0 .. 3, head1's.
  float4 wa[NB], wh[NB];
  pd_load<NB>(wa, a.layer[0].w_in, 2 * DI, (tid0 >> 6) * 16, tid0 & 15, (tid0 >> 4) & 3);

  const int wv = __builtin_amdgcn_readfirstlane(tid0 >> 6);

  for (int t = 1; t < a.maxlen; ++t) {
    // the thread index passes through an opaque move in each phase (PD_IDX),
    // so that the many addresses derived from it are recomputed there instead
    // of being hoisted out of the loop (and spilled)
#define PD_IDX                  \
  int tid = tid0;               \
  asm volatile("" : "+v"(tid)); \
  [[maybe_unused]] const int i = tid & 15, g = (tid >> 4) & 3
    {  // x = embedding rows of the current tokens
      PD_IDX;
      for (int p = tid; p < NB * 256; p += 1024) {
        const int q = p >> 8, m = (p >> 4) & 15;
        xs[p] = a.emb[(size_t)tok_s[m] * d + 16 * q + dperm(p & 15)];
      }
    }
    __syncthreads();
    // An MFMA tile's 16 features of the block's LP lanes, spread over all
    // lanes of the wave (through its LDS tile) for the elementwise work on
    // it: thread (i, g) takes lane m, components e0 .. e0 + VPL - 1 of lane
    // m's float4 g
#define PD_SPREAD const int m = i & (LP - 1), e0 = (i >> LSH) * VPL
#pragma unroll 1
    for (int li = 0; li < a.L; ++li) {
      const PersistLayer& P = a.layer[li];
      const float* q = prm + li * PSZ;
      float4 s0[VPL];  // conv state of in_proj's tile
      float4 wx[NBI];  // x_proj's weights, waves 0 ..
      float4 wq[NBF];  // out_proj's (waves 8 .. 11) and FF2's (waves 12 .. 15)
      {
        PD_IDX;
        if (wv < NBX)
          pd_load<NBI>(wx, P.w_x, NBX * 16, wv * 16, i, g);
        else
          pd_none<NBI>(wx);
        if (wv < NBI) {
          PD_SPREAD;
#pragma unroll
          for (int k = 0; k < VPL; ++k)
            s0[k] = reinterpret_cast<const float4*>(P.conv)[(size_t)(wv * 16 + 4 * (e0 + k) + g) * a.ld_state +
                                                            min(m0 + m, a.lanes - 1)];
        } else {
          pd_none<VPL>(s0);
        }
        pd_ln_stats<1, NB>(xs, stats, tid, a.ln_n);
      }
      __syncthreads();
      {
        PD_IDX;
        pd_ln_apply<1, NB>(xs, xn, stats, q + O_LN1W, q + O_LN1B, tid, a.ln_n);
      }
      __syncthreads();
      // in_proj: features < DI run the conv step (state float4 [c][lane]),
      // features >= DI are z
      {
        PD_IDX;
        const int n0 = wv * 16;
        const floatx4 acc = pd_mac<NB>(xn, wa, i, g);
        pd_load<NB>(wa, P.w1, 4 * d, n0, i, g);
        if (n0 < DI) {
          PD_SPREAD;
          if (i < LP) *pd_out(cvs, n0, i, g) = make_float4(acc[0], acc[1], acc[2], acc[3]);
          __builtin_amdgcn_wave_barrier();
          float* const sp = reinterpret_cast<float*>(pd_out(cvs, n0, m, g)) + e0;
#pragma unroll
          for (int k = 0; k < VPL; ++k) {
            const int n = n0 + 4 * (e0 + k) + g;
            const float v = sp[k] + q[O_BIN + n];
            const float4 cw = reinterpret_cast<const float4*>(q + O_CONVW)[n];
            const float cv = conv_step_value<MATH_BR>(q[O_CONVB + n], s0[k], v, cw);
            sp[k] = cv;
            if (m0 + m < a.lanes)
              reinterpret_cast<float4*>(P.conv)[(size_t)n * a.ld_state + m0 + m] =
                  make_float4(s0[k].y, s0[k].z, s0[k].w, v);
          }
        } else {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[e] + q[O_BIN + n0 + 4 * e + g];
          *pd_out(zs, n0 - DI, i, g) = make_float4(v[0], v[1], v[2], v[3]);
        }
      }
      // scan item it: lane (it / 16) % LP, channel 16 (it / 16 / LP) + it % 16;
      // the first item's state is loaded here
      float4* const h4 = reinterpret_cast<float4*>(P.ssm);
      float4 hv[DS / 4];
      auto load_h = [&](int it) {
        const int cl = it & 15, lm = (it >> 4) & (LP - 1), cb = it >> (4 + LSH);
        const int m = min(m0 + lm, a.lanes - 1);
#pragma unroll
        for (int n4 = 0; n4 < DS / 4; ++n4)
          hv[n4] = h4[((size_t)(cb * (DS / 4) + n4) * a.ld_state + m) * 16 + cl];
      };
      auto load_after_scan = [&](int i, int g) {  // out_proj's and FF2's weights
        if (wv >= 12) {
          pd_load<NBF>(wq, P.w2, d, (wv - 12) * 16, i, g);
        } else if (wv >= 8) {
          pd_load<NBI>(wq, P.w_out, d, (wv - 8) * 16, i, g);
          pd_none<NBF - NBI>(wq + NBI);
        } else {
          pd_none<NBF>(wq);
        }
      };
      if (LP * DI >= 1024 || wv < LP * DI / 64) {
        PD_IDX;
        load_h(tid);
      } else {
        pd_none<DS / 4>(hv);
      }
      __syncthreads();
      // x_proj (no bias: + 0 as the step's epilogue)
      if (wv < NBX) {
        PD_IDX;
        const floatx4 acc = pd_mac<NBI>(cvs, wx, i, g);
#pragma unroll
        for (int e = 0; e < 4; ++e) rwn[i * RW + wv * 16 + 4 * e + g] = acc[e] + 0.0f;
      }
      __syncthreads();
      // scan: the operations of dec_scan_kernel
      if (LP * DI >= 1024 || wv < LP * DI / 64) {
        PD_IDX;
#pragma unroll 1
        for (int it = tid; it < LP * DI; it += 1024) {
          const int cl = it & 15, lm = (it >> 4) & (LP - 1), cb = it >> (4 + LSH);
          const int c = cb * 16 + cl;
          const int m = min(m0 + lm, a.lanes - 1);
          const float4* na4 = reinterpret_cast<const float4*>(q + O_NAQ);
          const float4* w4 = reinterpret_cast<const float4*>(q + O_WDTQ);
          ScanCtx<DS, RB> sc;
#pragma unroll
          for (int n4 = 0; n4 < DS / 4; ++n4) {
            sc.h[4 * n4] = hv[n4].x; sc.h[4 * n4 + 1] = hv[n4].y;
            sc.h[4 * n4 + 2] = hv[n4].z; sc.h[4 * n4 + 3] = hv[n4].w;
            const float4 av = na4[(cb * (DS / 4) + n4) * 16 + cl];
            sc.na[4 * n4] = av.x; sc.na[4 * n4 + 1] = av.y; sc.na[4 * n4 + 2] = av.z; sc.na[4 * n4 + 3] = av.w;
          }
#pragma unroll
          for (int j4 = 0; j4 < RB / 4; ++j4) {
            const float4 wd = w4[(cb * (RB / 4) + j4) * 16 + cl];
            sc.wdt[4 * j4] = wd.x; sc.wdt[4 * j4 + 1] = wd.y; sc.wdt[4 * j4 + 2] = wd.z; sc.wdt[4 * j4 + 3] = wd.w;
          }
          sc.bdt = q[O_BDT + c];
          sc.dd = q[O_DD + c];
          const float* row = rwn + lm * RW;
          const int cp = ((c >> 4) * PL + lm) * 16 + dperm(c & 15);
          ys[cp] = scan_token<DS, RB, MATH_BR>(sc, row, row + RB, a.r, cvs[cp], zs[cp]);
          if (m0 + lm < a.lanes) {
#pragma unroll
            for (int n4 = 0; n4 < DS / 4; ++n4)
              h4[((size_t)(cb * (DS / 4) + n4) * a.ld_state + m) * 16 + cl] =
                  make_float4(sc.h[4 * n4], sc.h[4 * n4 + 1], sc.h[4 * n4 + 2], sc.h[4 * n4 + 3]);
          }
          if (LP * DI > 1024 && it + 1024 < LP * DI) load_h(it + 1024);
        }
        if (LP * DI >= 1024)
          load_after_scan(i, g);
        else
          pd_none<NBF>(wq);
      } else {
        PD_IDX;
        load_after_scan(i, g);  // these waves have no scan items
      }
      __syncthreads();
      // (the coder's division, on waves that have nothing else here)
      if (coder_lane && l == 0 && li == 0) target0 = dec_target(st);
      // out_proj + bias
      if (wv >= 8 && wv < 12) {
        PD_IDX;
        const int n0 = (wv - 8) * 16;
        const floatx4 acc = pd_mac<NBI>(ys, wq, i, g);
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[e] + q[O_BOUT + n0 + 4 * e + g];
        *pd_out(os, n0, i, g) = make_float4(v[0], v[1], v[2], v[3]);
      }
      __syncthreads();
      {
        PD_IDX;
        pd_ln_stats<2, NB>(os, stats, tid, a.ln_n);
      }
      __syncthreads();
      {
        PD_IDX;
        pd_ln_apply<2, NB>(os, xn, stats, q + O_LN2W, q + O_LN2B, tid, a.ln_n);
      }
      __syncthreads();
      // FF1 + bias + GELU
      {
        PD_IDX;
        const int n0 = wv * 16;
        const floatx4 acc = pd_mac<NB>(xn, wa, i, g);
        const bool more = li + 1 < a.L;
        pd_load<NB>(wa, more ? a.layer[li + 1 < PERSIST_MAX_LAYERS ? li + 1 : li].w_in : a.hw2, 256,
                    n0, i, g);
        PD_SPREAD;
        if (i < LP) *pd_out(hid, n0, i, g) = make_float4(acc[0], acc[1], acc[2], acc[3]);
        __builtin_amdgcn_wave_barrier();
        float* const sp = reinterpret_cast<float*>(pd_out(hid, n0, m, g)) + e0;
#pragma unroll
        for (int k = 0; k < VPL; ++k) {
          const float v = gelu<MATH_BR>(sp[k] + q[O_B1 + n0 + 4 * (e0 + k) + g]);
          sp[k] = v;
        }
        if (!more && wv < NB)
          pd_load<NB>(wh, a.hw1, d, n0, i, g);
        else
          pd_none<NB>(wh);
      }
      __syncthreads();
      // FF2 + bias + residual (each float4 of x read and written by one lane)
      if (wv >= 12) {
        PD_IDX;
        const int n0 = (wv - 12) * 16;
        const floatx4 acc = pd_mac<NBF>(hid, wq, i, g);
        float4* xp = pd_out(xs, n0, i, g);
        const float4 rv = *xp;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[e] + q[O_B2 + n0 + 4 * e + g];
        *xp = make_float4(v[0] + rv.x, v[1] + rv.y, v[2] + rv.z, v[3] + rv.w);
      }
      __syncthreads();
    }
    // head1 + bias + ReLU
    if (wv < NB) {
      PD_IDX;
      const int n0 = wv * 16;
      const floatx4 acc = pd_mac<NB>(xs, wh, i, g);
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = fmaxf(0.0f, acc[e] + hb1[n0 + 4 * e + g]);
      *pd_out(os, n0, i, g) = make_float4(v[0], v[1], v[2], v[3]);
    }
    __syncthreads();
    // head2, row-major (unpermuted weights: component e is feature n0 + 4 g + e),
    // without b2 (the CDF adds it)
    {
      PD_IDX;
      const int n0 = wv * 16;
      const floatx4 acc = pd_mac<NB>(os, wa, i, g);
      pd_load<NB>(wa, a.layer[0].w_in, 2 * DI, n0, i, g);
      *reinterpret_cast<float4*>(lg + i * 256 + n0 + 4 * g) =
          make_float4(acc[0] + 0.0f, acc[1] + 0.0f, acc[2] + 0.0f, acc[3] + 0.0f);
    }
    __syncthreads();
    // CDF of each lane's row on its half-wave (lane l: symbols 8 l .. 8 l + 7),
    // symbol search (the lowest symbol whose range holds the target: ballot,
    // first set bit, first of the lane's eight) and the coder advance
    if (half < LP) {
      double r[8];
      cdf_halfwave_regs(lg + half * 256, hb2, a.inv_t, l, r);
      if (coder_lane && t < len_h) {  // uniform over the half-wave
        const uint32_t target = __shfl(target0, 0, 32);
        uint32_t lo[9];
#pragma unroll
        for (int k = 0; k < 8; ++k) lo[k] = q_lower(r[k], 8 * l + k);
        const uint32_t next = __shfl_down(lo[0], 1, 32);
        lo[8] = l == 31 ? TOTAL : next;
        int sym = -1;
        uint32_t low = 0, high = 0;
#pragma unroll
        for (int k = 7; k >= 0; --k)
          if (target >= lo[k] && target < lo[k + 1]) {
            sym = 8 * l + k;
            low = lo[k];
            high = lo[k + 1];
          }
        const uint32_t mask = (uint32_t)(__ballot(sym >= 0) >> (tid0 & 32));
        const int winner = mask != 0u ? __ffs(mask) - 1 : 0;
        sym = __shfl(sym, winner, 32);
        low = __shfl(low, winner, 32);
        high = __shfl(high, winner, 32);
        if (mask == 0u) sym = 0, low = 0, high = 0;
        if (l == 0) {
          dec_advance_ahead(st, low, high, pin, pn, nw);
          a.out[(size_t)mh * a.out_stride + t] = (uint8_t)sym;
          tok_s[half] = sym;
        }
      }
    }
    __syncthreads();
  }
  if (coder_lane && l == 0) {
    a.states[mh] = st;
    a.tok[mh] = (uint8_t)tok_s[half];
  }
  if (blockIdx.x == 0 && tid0 == 0) *a.t_counter = a.maxlen > 1 ? a.maxlen - 1 : 0;
}

bool dec_persist_fits(int d, int ds, int r, int L) {
  return d == 64 && ds == 16 && dec_rb(r) == 8 && L >= 1 && L <= PERSIST_MAX_LAYERS;
}

int dec_persist_lanes_per_block(int lanes, int n_cus) {
  for (int lp = 4; lp < PL; lp *= 2)
    if ((lanes + lp - 1) / lp <= n_cus) return lp;
  return PL;
}

hipError_t launch_dec_persist(const PersistArgs& a, int d, int ds, int n_cus, hipStream_t s) {
  if (a.lanes <= 0 || a.maxlen <= 1) return hipSuccess;
  if (!dec_persist_fits(d, ds, a.r, a.L)) return hipErrorInvalidValue;
  const int lp = dec_persist_lanes_per_block(a.lanes, n_cus);
  const dim3 grid((a.lanes + lp - 1) / lp), block(1024);
  if (lp == 4)
    BOA_LAUNCH((dec_persist_kernel<4, 8, 4>), grid, block, 0, s, a);
  else if (lp == 8)
    BOA_LAUNCH((dec_persist_kernel<4, 8, 8>), grid, block, 0, s, a);
  else
    BOA_LAUNCH((dec_persist_kernel<4, 8, 16>), grid, block, 0, s, a);
  return hipGetLastError();
}

}  // namespace boa
