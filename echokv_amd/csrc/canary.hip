// Canary probe (echokv_vllm/canary.py:59-89) on gfx950: per layer and tier b,
// delta_b = mean over query rows and heads of KL(softmax(q K~_b^T s) || softmax(q K_ref^T s)),
// K~_b = per-channel storage round trip of the K_ref keys over whole k_group
// groups (oldest-first; the oldest window mod k_group keys are dropped).
//
// One workgroup of 4 waves per (layer, KV head): it scores the rep = Hq / H query heads
// of that KV head for all nq query rows, 64 rows at a time. The window's keys are staged in
// LDS a chunk (64 keys; 32 above head size 128) at a time, in float32, with each K
// group's storage statistics per tier, so any window length fits. Wave v takes one variant
// (reference, then a tier): it holds the chunk's keys -- the reference's as they are, a
// tier's as its codes' round trip -- in the operand layout of v_mfma_f32_16x16x4_f32 and
// multiplies every block of 16 query rows with them, all in float32. The reference's
// logits and running max go through LDS to the tiers' waves, whose softmax statistics
// run online over the chunks against that max m:  s_v = sum exp(x_v - m),
// u_b = sum exp(x_b - m) (x_b - x_ref), so that KL_b = u_b / s_b - log(s_b / s_ref) (no
// difference of two large log-sum-exps). Each workgroup writes its KL sums per tier; a
// second kernel adds the heads of a layer in order (deterministic) and takes the mean.
// 32 layers, H 8, GQA 4, D 128, 8 rows, 64 keys: 126 us with one row at a time, a key
// per lane (its products on the vector unit, a barrier a row), 25 us here: start-up, two memory round
// trips and the statistics before 3.4 us of matrix products, one workgroup per CU.
#include "args.h"

namespace ek {

namespace {

constexpr int kCanRows = 64;  // query rows per pass

// LDS of one workgroup (dynamic), in floats: keys [C][LD] and queries [64][LD] (rows
// padded so that 16 rows' float4 reads spread over the banks), statistics [nbits][NG][DP]
// (fp16 scale, min), the reference's logits [4][C][17], per row the max before and after
// the chunk [64][2], the running max [64] and the running (s, u) [V][64][2].
struct CanaryLds {
  int C, DP, V, NG;
  __host__ __device__ int ld() const { return DP + 4; }
  __host__ __device__ size_t o_q() const { return (size_t)C * ld(); }
  __host__ __device__ size_t o_st() const { return o_q() + (size_t)kCanRows * ld(); }
  __host__ __device__ size_t o_ref() const { return o_st() + (size_t)(V - 1) * NG * DP; }
  __host__ __device__ size_t o_row() const { return o_ref() + (size_t)4 * C * 17; }
  __host__ __device__ size_t o_run() const { return o_row() + 2 * kCanRows; }
  __host__ __device__ size_t o_state() const { return o_run() + kCanRows; }
  __host__ __device__ size_t bytes() const { return 4 * (o_state() + (size_t)V * kCanRows * 2); }
};

__host__ __device__ inline int canary_chunk(int d) { return d <= 128 ? 64 : 32; }
__host__ __device__ inline int canary_dp(int d) { return d <= 64 ? 64 : (d <= 128 ? 128 : 256); }
// Most K groups that touch a chunk (a window's groups start at its first scored key).
// (0 for groups of one key: their statistics are the key itself.)
__host__ __device__ inline int canary_groups(int C, int kg) {
  return kg == 1 ? 0 : (C + kg - 1) / kg + (C % kg && kg % C ? 1 : 0);
}

__device__ __forceinline__ float rows4_sum(float x) {  // over lanes l, l ^ 16, l ^ 32, l ^ 48
  x += __shfl_xor(x, 16, 64);
  return x + __shfl_xor(x, 32, 64);
}

template <int KT>
__device__ __forceinline__ float tiles_sum(const f4_t* t) {
  f4_t v = t[0] + t[1];
  if constexpr (KT == 4) v = v + (t[2] + t[3]);
  return (v[0] + v[1]) + (v[2] + v[3]);
}

}  // namespace

// DG: 16-channel groups of the padded head size; KT: 16-key tiles per chunk.
template <int DG, int KT>
__global__ __launch_bounds__(256) void canary_kernel(CanaryArgs a) {
  constexpr int C = 16 * KT, DP = 16 * DG, LD = DP + 4;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int layer = blockIdx.x / a.h, h = blockIdx.x % a.h;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int c = lane >> 4, n = lane & 15;
  const int rep = a.hq / a.h;
  const int rows = rep * a.nq;
  const CanaryLds L{C, DP, 1 + a.nbits, canary_groups(C, a.kg)};
  float* const kv = lds;
  float* const qv = lds + L.o_q();
  uint32_t* const st = (uint32_t*)(lds + L.o_st());
  float* const xref = lds + L.o_ref();
  float* const mrow = lds + L.o_row();
  float* const mrun = lds + L.o_run();
  float* const state = lds + L.o_state();
  const int w = (a.window / a.kg) * a.kg;
  const int first = a.window - w;
  const long kbase = layer * a.k_sl + (long)h * a.k_s1;
  const int bits = wave >= 1 ? (a.bits_packed >> (8 * (wave - 1))) & 0xff : 8;
  const bool active = wave < L.V;
  float kl = 0.f;

  for (int r0 = 0; r0 < rows; r0 += kCanRows) {
    const int nr = rows - r0 < kCanRows ? rows - r0 : kCanRows;
    const int nrt = (nr + 15) / 16;
    __syncthreads();
    // The pass's query rows, in float32 (rows and channels past the end: zeros).
    for (int i = tid; i < 16 * nrt * (DP / 4); i += 256) {
      const int r = i / (DP / 4), ch = 4 * (i % (DP / 4));
      f4_t x = {0.f, 0.f, 0.f, 0.f};
      if (r < nr) {
        const long qb = layer * a.q_sl + (long)((r0 + r) % a.nq) * a.q_s0 + (long)(h * rep + (r0 + r) / a.nq) * a.q_s1;
        if (ch + 4 <= a.d) {
          float y[4];
          ld4(a.q, a.q_dtype, qb + ch, y);
          x = f4_t{y[0], y[1], y[2], y[3]};
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (ch + e < a.d) x[e] = ld(a.q, a.q_dtype, qb + ch + e);
        }
      }
      *(f4_t*)(qv + r * LD + ch) = x;
    }
    for (int i = tid; i < L.V * kCanRows * 2; i += 256) state[i] = 0.f;
    if (tid < kCanRows) mrun[tid] = -__builtin_inff();

    for (int c0 = 0; c0 < w; c0 += C) {
      const int nk = w - c0 < C ? w - c0 : C;
      __syncthreads();  // the previous chunk's keys and logits are no longer read
      for (int i = tid; i < C * (DP / 4); i += 256) {
        const int j = i / (DP / 4), ch = 4 * (i % (DP / 4));
        f4_t x = {0.f, 0.f, 0.f, 0.f};
        if (j < nk) {
          const float* src = a.kref + kbase + (long)(first + c0 + j) * a.k_s0 + ch;
          if (a.k_vec) {
            if (ch < a.d) x = *(const f4_t*)src;
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (ch + e < a.d) x[e] = src[e];
          }
        }
        *(f4_t*)(kv + j * LD + ch) = x;
      }
      __syncthreads();
      // Storage statistics of each K group touching the chunk, per channel: a group inside
      // the chunk from LDS, a longer one from memory.
      const int g0 = c0 / a.kg, g1 = (c0 + nk - 1) / a.kg;
      for (int i = tid; a.kg > 1 && i < (g1 - g0 + 1) * DP; i += 256) {
        const int g = g0 + i / DP, ch = i % DP;
        const bool in_chunk = g * a.kg >= c0 && (g + 1) * a.kg <= c0 + nk;
        float mn = __builtin_inff(), mx = -__builtin_inff();
        if (in_chunk) {
          const float* src = kv + (g * a.kg - c0) * LD + ch;
#pragma unroll 8
          for (int p = 0; p < a.kg; ++p) {
            mn = fminf(mn, src[p * LD]);
            mx = fmaxf(mx, src[p * LD]);
          }
        } else if (ch < a.d) {
          const float* src = a.kref + kbase + (long)(first + g * a.kg) * a.k_s0 + ch;
          for (int p = 0; p < a.kg; ++p) {
            const float x = src[(long)p * a.k_s0];
            mn = fminf(mn, x);
            mx = fmaxf(mx, x);
          }
        } else {
          mn = mx = 0.f;
        }
        for (int t = 0; t < a.nbits; ++t) {
          _Float16 s16, m16;
          float s, m;
          group_stats(mn, mx, (a.bits_packed >> (8 * t)) & 0xff, s16, m16, s, m);
          st[(t * L.NG + g - g0) * DP + ch] =
              (uint32_t)__builtin_bit_cast(uint16_t, s16) | (uint32_t)__builtin_bit_cast(uint16_t, m16) << 16;
        }
      }
      __syncthreads();

      f4_t x[4][KT];  // logits of row block rt: lane (c, n) holds keys 16 kt + 4c + i of row 16 rt + n
      if (active) {
        // The variant's keys as A operands: lane (c, n) holds key 16 kt + n, channels 16 g + 4c + u
        // at step (g, u); queries alike, so a step's four products cover 16 channels in any order.
        f4_t kf[KT][DG];
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
          const uint32_t* sp = st + ((wave - 1) * L.NG + (wave >= 1 ? (c0 + 16 * kt + n) / a.kg - g0 : 0)) * DP + 4 * c;
          const bool tier = wave >= 1 && 16 * kt + n < nk;
#pragma unroll
          for (int g = 0; g < DG; ++g) {
            f4_t y = *(const f4_t*)(kv + (16 * kt + n) * LD + 16 * g + 4 * c);
            if (tier && a.kg == 1) {
#pragma unroll
              for (int u = 0; u < 4; ++u) {
                _Float16 s16, m16;
                float s, m;
                group_stats(y[u], y[u], bits, s16, m16, s, m);
                y[u] = (float)quant_code(y[u], m, s, bits) * s + m;
              }
            } else if (tier) {
              const uint4 sm = *(const uint4*)(sp + 16 * g);
              const uint32_t pk[4] = {sm.x, sm.y, sm.z, sm.w};
#pragma unroll
              for (int u = 0; u < 4; ++u) {
                const float s = (float)__builtin_bit_cast(_Float16, (uint16_t)pk[u]);
                const float m = (float)__builtin_bit_cast(_Float16, (uint16_t)(pk[u] >> 16));
                bool tie = false;
                uint32_t q = quant_code_r(y[u], m, __builtin_amdgcn_rcpf(s), bits, tie);
                if (tie) q = quant_code(y[u], m, s, bits);
                y[u] = (float)q * s + m;
              }
            }
            kf[kt][g] = y;
          }
        }
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
          if (rt >= nrt) break;
          // Four accumulators per tile (a quarter of the steps each) and sums by pairs below: the
          // rounding of a chain of 32 products, and of 16 terms, grows with its length.
          f4_t acc[4][KT] = {};
#pragma unroll
          for (int g = 0; g < DG; ++g) {
            const f4_t qf = *(const f4_t*)(qv + (16 * rt + n) * LD + 16 * g + 4 * c);
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
              for (int kt = 0; kt < KT; ++kt)
                acc[g & 3][kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[kt][g][u], qf[u], acc[g & 3][kt], 0, 0, 0);
          }
#pragma unroll
          for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              x[rt][kt][i] = 16 * kt + 4 * c + i < nk ? ((acc[0][kt][i] + acc[1][kt][i]) + (acc[2][kt][i] + acc[3][kt][i])) * a.scale : -__builtin_inff();
          if (wave == 0) {  // the reference: running max and sum; publish its logits
            const int row = 16 * rt + n;
            float mt = -__builtin_inff();
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
              for (int i = 0; i < 4; ++i) mt = fmaxf(mt, x[rt][kt][i]);
            mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
            mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
            const float m_old = mrun[row], m_new = fmaxf(m_old, mt);
            f4_t et[KT];
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                et[kt][i] = expf(x[rt][kt][i] - m_new);
                xref[(rt * C + 16 * kt + 4 * c + i) * 17 + n] = x[rt][kt][i];
              }
            const float se = rows4_sum(tiles_sum<KT>(et));
            if (c == 0) {
              mrow[2 * row] = m_old;
              mrow[2 * row + 1] = m_new;
              mrun[row] = m_new;
              state[2 * row] = state[2 * row] * expf(m_old - m_new) + se;
            }
          }
        }
      }
      __syncthreads();
      if (wave >= 1 && active) {
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
          if (rt >= nrt) break;
          const int row = 16 * rt + n;
          const float m_old = mrow[2 * row], m_new = mrow[2 * row + 1];
          f4_t et[KT], ut[KT];
#pragma unroll
          for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int key = 16 * kt + 4 * c + i;
              const float e = key < nk ? expf(x[rt][kt][i] - m_new) : 0.f;
              et[kt][i] = e;
              ut[kt][i] = key < nk ? e * (x[rt][kt][i] - xref[(rt * C + key) * 17 + n]) : 0.f;
            }
          const float se = rows4_sum(tiles_sum<KT>(et)), su = rows4_sum(tiles_sum<KT>(ut));
          if (c == 0) {
            float* sv = state + (wave * kCanRows + row) * 2;
            const float f = expf(m_old - m_new);  // m_old = -inf on the first chunk: f = 0
            sv[0] = sv[0] * f + se;
            sv[1] = sv[1] * f + su;
          }
        }
      }
    }
    __syncthreads();
    if (wave >= 1 && active && lane < nr) {
      const float* sv = state + (wave * kCanRows + lane) * 2;
      kl += sv[1] / sv[0] - logf(sv[0] / state[2 * lane]);
    }
  }
  if (wave >= 1 && active) {
    for (int m = 32; m > 0; m >>= 1) kl += __shfl_xor(kl, m, 64);
    if (lane == 0) a.partial[((long)layer * a.h + h) * a.nbits + (wave - 1)] = kl;
  }
}

// out[layer][t] = max(sum over KV heads of the partial sums / (nq * Hq), 0), heads in order.
__global__ __launch_bounds__(64) void canary_reduce_kernel(CanaryArgs a, int num_layers) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  if (i >= num_layers * a.nbits) return;
  const int layer = i / a.nbits, t = i % a.nbits;
  float s = 0.f;
  for (int h = 0; h < a.h; ++h) s += a.partial[((long)layer * a.h + h) * a.nbits + t];
  a.out[i] = fmaxf(s / (float)(a.nq * a.hq), 0.f);
}

size_t canary_lds_bytes(int d, int nbits, int kg) {
  const int C = canary_chunk(d);
  return CanaryLds{C, canary_dp(d), 1 + nbits, canary_groups(C, kg)}.bytes();
}

template <int DG, int KT>
static hipError_t canary_d(const CanaryArgs& a, int num_layers, size_t lds, hipStream_t s) {
  static std::atomic<uint64_t> attr_done{0};
  const hipError_t e = ensure_lds_limit((const void*)canary_kernel<DG, KT>, (int)kLdsBytes, &attr_done);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((canary_kernel<DG, KT>), dim3((unsigned)(num_layers * a.h)), dim3(256), lds, s, a);
  return hipGetLastError();
}

hipError_t launch_canary(const CanaryArgs& a, int num_layers, hipStream_t s) {
  const size_t lds = canary_lds_bytes(a.d, a.nbits, a.kg);
  hipError_t e = a.d <= 64 ? canary_d<4, 4>(a, num_layers, lds, s)
                           : (a.d <= 128 ? canary_d<8, 4>(a, num_layers, lds, s) : canary_d<16, 2>(a, num_layers, lds, s));
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(canary_reduce_kernel, dim3((unsigned)((num_layers * a.nbits + 63) / 64)), dim3(64), 0, s, a,
                     num_layers);
  return hipGetLastError();
}

}  // namespace ek
