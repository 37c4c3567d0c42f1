// Paged decode attention for the layouts the MFMA decode kernels do not take
// (echokv_vllm/kernels/decode.py:95-129, the reference's PyTorch path for shapes
// its Triton kernel refuses): head sizes other than 64 / 128 / 256 (any multiple
// of 4 up to 256), V groups under D / 16 channels (at head size 256: outside 8 to
// 128), K groups under 16, block sizes or K groups that are not powers of two,
// more than 4 chunks per page.
//
// One workgroup per (sequence, KV head, split, group of query heads) in fp32 arithmetic,
// the split schedule of the MFMA kernels (splits of max(blocks_per_split, ceil(blocks /
// num_splits)) blocks, fewer for short sequences, so a sequence's result does not depend on
// its batch) and
// the same workspace rows: acc [S, Hq, splits, D] unnormalized, ml (running max
// in log2 units, sum). Keys and values go from codes to registers to products: a lane
// holds 8 channels of its query heads and of O, a row of 16 lanes (8 up to head size
// 64) a key's head, so a key costs its products, 4 lane sums per query head and one
// exponential, and no LDS. 16 sequences of 0.2-4K tokens, INT4, H 8, GQA 4, D 96, V group
// 24, with the merge: 2116 us with keys staged 64 at a time over scalar loads, 68 us now; a
// wave's batch of 16 keys takes 2 us (its waves, two a SIMD, issue in half of their cycles),
// and a split of 1024 tokens is 16 of them.
//
// Each token is dequantized as the reference's gather does: K codes with the
// group's per-channel (scale, min), or the residual row for the open group; V
// codes with the token's per-group (scale, min); a chunk id outside the layer's
// pages reads as zeros. Block ids outside the layer are left out.
#include "items.h"

namespace ek {
namespace {

constexpr int kAnyThreads = 256;  // prefill
constexpr int kAnyTile = 64;  // keys per tile
constexpr int kAnyCols = 16;  // query heads per pass (DecodeArgs::gs <= 16)

__device__ __forceinline__ float wave_max(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x = fmaxf(x, __shfl_xor(x, o, 64));
  return x;
}
__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}

// ---- decode -----------------------------------------------------------------
// One row of GW lanes takes an item at a time: 4 keys x 8 channels a lane (NO items, 128
// channels apart, above head size 128). A wave's 64 / GW rows take neighbouring items of
// a batch, the workgroup's waves the batches in turn. Each row keeps its own online
// softmax over its keys, in fp32 registers; rows meet by lane swaps and waves through
// LDS at the end.
constexpr int kDecThreads = 256;
constexpr int kDecWaves = kDecThreads / 64;

// x + x of another lane of the row: DPP quad_perm [1,0,3,2] / [2,3,0,1], row_half_mirror,
// row_mirror.
template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
  return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, true));
}
// Sum over the row's GW lanes; every lane gets it (the same bits: each step adds a pair).
template <int GW>
__device__ __forceinline__ float row_sum(float x) {
  x = dpp_add<0xB1>(x);
  x = dpp_add<0x4E>(x);
  x = dpp_add<0x141>(x);
  if constexpr (GW == 16) x = dpp_add<0x140>(x);
  return x;
}

// FAST (DecodeArgs::any_fast): power-of-two block size and K group of at least 4, whole
// octets inside one V group, aligned rows. Other layouts read their items by item_general.
template <int GW, int NO, int GS, bool FAST>
__global__ __launch_bounds__(kDecThreads, FAST && GS * NO == 1 ? 4 : 2) void decode_any_kernel(DecodeArgs a) {
  constexpr int RPW = 64 / GW;     // rows per wave
  constexpr int BK = RPW * 4;      // keys per batch
  constexpr int CH = 8 * NO;       // channels per lane
  const Lay& L = a.L;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int cg = blockIdx.y;  // the pass's query heads [GS cg, GS cg + GS)
  // Splits vary slowest: workgroups go to the 8 XCDs round-robin, and with the split
  // fastest the live ones (a sequence's first few of num_splits) met on one XCD
  // (16 sequences of 0.2-4K tokens at 32 splits, D 96: 390 -> 55 us).
  const long sh = blockIdx.x % (a.num_seqs * L.H);
  const int sp = (int)(blockIdx.x / (a.num_seqs * L.H));
  const int h = (int)(sh % L.H);
  const long seq = sh / L.H;
  const long seq_len = a.lens[seq];
  if (seq_len <= 0) return;
  const long n_blocks = (seq_len + L.BS - 1) / L.BS;
  const long bps = split_blocks(a.sp, (int)n_blocks);
  const long b0 = sp * bps;
  if (b0 >= n_blocks) return;
  const int t_begin = (int)(b0 * L.BS);
  const int t_end = (int)((b0 + bps) * L.BS < seq_len ? (b0 + bps) * L.BS : seq_len);

  const int D = L.D, G = D / L.VG;
  const int l = lane % GW, row = lane / GW;
  const long q_row = a.q_rows ? a.q_rows[seq] : seq;
  const long bt_row = a.bt_rows ? a.bt_rows[seq] : seq;
  const int g0 = a.g0 + cg * GS;
  const int gs = a.gs - cg * GS < GS ? a.gs - cg * GS : GS;
  const int qh0 = h * a.gqa + g0;
  // Item n's channels: [ch0(n), ch0(n) + 8); a lane past the head reads octet 0 and scores
  // zeros with it (not octet 0's keys times a query of 0: a key can be infinite).
  auto oct_of = [&](int n) { return l + n * GW; };
  auto ch0 = [&](int n) { return 8 * oct_of(n) < D ? 8 * oct_of(n) : 0; };
  auto past = [&](int n) { return 8 * oct_of(n) >= D; };

  // ---- the chain of loads: block table, header, codes ------------------------
  // As in prefill.hip: nothing loaded is looked at before the batch that needs it,
  // and no load sits in a branch (addresses are clamped), but for the K statistics' mask.
  auto block_of = [&](int kp) { return FAST ? kp >> a.bs_shift : kp / L.BS; };
  auto group_of = [&](int off) { return FAST ? off >> a.kg_shift : off / L.KG; };
  auto item_key = [&](int b) { return t_begin + b * BK + 4 * row; };
  auto item_off = [&](int b) {
    const int kp = item_key(b);
    return FAST ? kp & ((1 << a.bs_shift) - 1) : kp % L.BS;
  };
  auto load_blk = [&](int b) -> int {
    const int kp = item_key(b);
    return a.bt[bt_row * a.bt_s0 + block_of(kp < t_end ? kp : t_end - 1)];
  };
  struct Head {
    uint4 h;
    long rs;
    int blk;
    __device__ __forceinline__ Hdr hd() const { return Hdr{h.x & 0xffu, (int32_t)h.y, (int32_t)h.z, (int32_t)h.w}; }
  };
  auto page_of = [&](int blk) { return (unsigned)blk < (unsigned long)L.nb ? (long)blk : 0l; };
  auto load_head = [&](int blk) {
    const long b = page_of(blk);
    return Head{*(const uint4*)(a.pages + b * L.stride), a.block_res[b], blk};
  };
  auto item_row = [&](const Head& x, int off, int bits) -> long {
    if constexpr (!FAST) return row_base_h(L, page_of(x.blk), x.hd(), off, bits);
    const int tpc_shift = a.bs_shift + 1 - (bits == 8 ? 3 : bits == 4 ? 2 : 1);
    const int j = off >> tpc_shift;
    long cb = page_of(x.blk) * L.stride + L.o_data;
    if (j > 0) {
      const uint32_t id = (uint32_t)x.hd().id(j - 1);
      const uint32_t page = a.kc_mul ? __umulhi(id, a.kc_mul) : id;
      if ((int)id < 0 || (long)page >= L.nb) return -1;
      cb = (long)page * L.stride + L.o_data + (long)(id - page * (uint32_t)L.KC) * L.cb;
    }
    return cb + (long)((off & ((1 << tpc_shift) - 1)) * (L.H * (D / 4) * bits));
  };
  // Where an item's bytes are, from its header.
  struct At {
    const uint8_t *pg, *row;  // the block's page; the item's first row (no chunk: the page)
    int rowb;                 // bytes per row (no chunk: 0)
    int bits, off;
    bool ok;                  // the item can be read (its block and its chunk are in the layer)
  };
  auto at_of = [&](int b, const Head& x) {
    At t;
    t.off = item_off(b);
    t.bits = tier_of(x.hd().tag);
    const long rb = item_row(x, t.off, t.bits);
    t.ok = rb >= 0 && (unsigned)x.blk < (unsigned long)L.nb;
    t.pg = a.pages + page_of(x.blk) * L.stride;
    t.row = t.ok ? a.pages + rb : t.pg;
    t.rowb = t.ok ? L.H * (D / 4) * t.bits : 0;
    return t;
  };
  auto code_byte = [&](int n, int bits) { return (h * D + ch0(n)) * bits / 8; };
  // Each row's eight codes in the 8 bytes at or before them, and their statistics.
  struct RawK {
    uint2 k[NO][4];
    uint4 ks[NO], km[NO];
    int rg;
  } rk;
  struct RawV {
    uint2 v[NO][4];
    uint16_t vs[NO][4], vm[NO][4];
  } rv;
  auto load_k = [&](const Head& x, const At& t) {
    const long rs = (unsigned long)x.rs < (unsigned long)a.res.rows ? x.rs : 0;
    rk.rg = *(const int32_t*)(a.res_group + rs);
    if constexpr (!FAST) return;
#pragma unroll
    for (int n = 0; n < NO; ++n) {
      const uint8_t* p = t.ok ? t.row + (code_byte(n, t.bits) & ~7) : t.pg;
#pragma unroll
      for (int i = 0; i < 4; ++i) rk.k[n][i] = *(const uint2*)(p + i * t.rowb);
      const int se = (group_of(t.off) * L.H + h) * D + ch0(n);
      // Lanes past the head keep the zeros they began with (selects on the loaded words: 1 %
      // of the kernel's time more).
      if (!past(n)) {
        rk.ks[n] = *(const uint4*)(t.pg + L.o_ks + 2 * se);
        rk.km[n] = *(const uint4*)(t.pg + L.o_km + 2 * se);
      }
    }
  };
  auto load_v = [&](const At& t) {
    if constexpr (!FAST) return;
#pragma unroll
    for (int n = 0; n < NO; ++n) {
      const uint8_t* p = t.ok ? t.row + (code_byte(n, t.bits) & ~7) + t.rowb / 2 : t.pg;
      const int ve = (t.off * L.H + h) * G + ch0(n) / L.VG;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        rv.v[n][i] = *(const uint2*)(p + i * t.rowb);
        rv.vs[n][i] = *(const uint16_t*)(t.pg + L.o_vs + 2 * (ve + i * L.H * G));
        rv.vm[n][i] = *(const uint16_t*)(t.pg + L.o_vm + 2 * (ve + i * L.H * G));
      }
    }
  };
  // The four rows' codes of item n as fp16 pairs.
  auto pairs = [&](const uint2* w, int n, int bits, h2_t (*c)[4]) {
    const int sh = 8 * (code_byte(n, bits) & 7);
    if (bits == 4) {
#pragma unroll
      for (int i = 0; i < 4; ++i) code_pairs<4>(w[i], sh, c[i]);
    } else if (bits == 2) {
#pragma unroll
      for (int i = 0; i < 4; ++i) code_pairs<2>(w[i], sh, c[i]);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) code_pairs<8>(w[i], sh, c[i]);
    }
  };
  // The same for the other layouts (!FAST): the item's keys or values of octet n, `live` of them.
  auto general = [&](auto key, const Head& x, const At& t, int n, int live, float (*y)[8]) {
    item_general<decltype(key)::value>(L, a.pages, a.res, page_of(x.blk), x.hd(), x.rs, rk.rg, t.off, t.bits, live, h,
                                       8 * oct_of(n), y);
  };

  const int n_batches = (t_end - t_begin + BK - 1) / BK;
  Head head = load_head(load_blk(wv));
  Head head1 = load_head(load_blk(wv + kDecWaves));
  int blk2 = load_blk(wv + 2 * kDecWaves);
  At at = at_of(wv, head);
#pragma unroll
  for (int n = 0; n < NO; ++n) rk.ks[n] = rk.km[n] = uint4{};
  load_k(head, at);
  load_v(at);

  float q[GS][CH];
#pragma unroll
  for (int g = 0; g < GS; ++g) {
    const long qb = q_row * a.q_s0 + (long)(qh0 + (g < gs ? g : 0)) * a.q_s1;
#pragma unroll
    for (int n = 0; n < NO; ++n) {
      float x[8];
      if constexpr (FAST) {
        ld_n<8>(a.q, a.q_dtype, qb + ch0(n), x);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = ld(a.q, a.q_dtype, qb + (ch0(n) + e < D ? ch0(n) + e : 0));
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) q[g][8 * n + e] = g < gs && 8 * oct_of(n) + e < D ? x[e] * a.scale_log2 : 0.f;
    }
  }
  float m[GS], lsum[GS], o[GS][CH];
#pragma unroll
  for (int g = 0; g < GS; ++g) {
    m[g] = -__builtin_inff();
    lsum[g] = 0.f;
#pragma unroll
    for (int e = 0; e < CH; ++e) o[g][e] = 0.f;
  }

#pragma unroll 1
  for (int b = wv; b < n_batches; b += kDecWaves) {
    const int n_live = t_end - item_key(b);
    const bool opened = (unsigned)head.blk < (unsigned long)L.nb;  // else the block is left out
    const bool in_res = FAST && at.ok && (unsigned long)head.rs < (unsigned long)a.res.rows && rk.rg == group_of(at.off);
    // ---- scores
    float s[4][GS];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int g = 0; g < GS; ++g) s[i][g] = 0.f;
    auto score = [&](int n, int i, const float* x) {
#pragma unroll
      for (int g = 0; g < GS; ++g)
#pragma unroll
        for (int e = 0; e < 8; ++e) s[i][g] = __builtin_fmaf(q[g][8 * n + e], x[e], s[i][g]);
    };
#pragma unroll
    for (int n = 0; n < NO; ++n) {
      if constexpr (FAST) {
        h2_t c[4][4];
        pairs(rk.k[n], n, at.bits, c);
        const uint32_t sw[4] = {rk.ks[n].x, rk.ks[n].y, rk.ks[n].z, rk.ks[n].w};
        const uint32_t mw[4] = {rk.km[n].x, rk.km[n].y, rk.km[n].z, rk.km[n].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float x[8];
#pragma unroll
          for (int e = 0; e < 8; ++e)
            x[e] = __builtin_fmaf((float)c[i][e >> 1][e & 1], (float)u2h(sw[e >> 1])[e & 1], (float)u2h(mw[e >> 1])[e & 1]);
          score(n, i, x);
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
        float x[4][8];
        general(std::true_type{}, head, at, n, opened ? n_live : 0, x);
#pragma unroll
        for (int i = 0; i < 4; ++i) score(n, i, x[i]);
      }
    }
    if (FAST && __builtin_amdgcn_ballot_w64(in_res || !at.ok)) {
      // Rare: the sequence's open K group (keys from the residual), a chunk id outside the
      // pages (keys read as zeros).
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (in_res || !at.ok) {
#pragma unroll
          for (int g = 0; g < GS; ++g) s[i][g] = 0.f;
        }
        if (in_res && i < n_live) {
#pragma unroll
          for (int n = 0; n < NO; ++n) {
            float x[8];
            ld_n<8>(a.res.ptr, a.res.dtype,
                    head.rs * a.res.s0 + (long)((at.off + i) & (L.KG - 1)) * a.res.s1 + (long)h * a.res.s2 + ch0(n), x);
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = past(n) ? 0.f : x[e];
            score(n, i, x);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // The next batch's keys, requested as soon as this one's are used.
    const Head cur = head;
    const At cat = at;
    const bool more = b + kDecWaves < n_batches;
    if (more) {
      head = head1;
      at = at_of(b + kDecWaves, head);
      load_k(head, at);
      head1 = load_head(blk2);
      blk2 = load_blk(b + 3 * kDecWaves);
    }
    // ---- online softmax of the row
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int g = 0; g < GS; ++g) {
        s[i][g] = row_sum<GW>(s[i][g]);
        s[i][g] = opened && i < n_live ? s[i][g] : -__builtin_inff();
      }
#pragma unroll
    for (int g = 0; g < GS; ++g) {
      const float mt = fmaxf(fmaxf(s[0][g], s[1][g]), fmaxf(s[2][g], s[3][g]));
      if (__builtin_amdgcn_ballot_w64(mt > m[g])) {
        const float mn = fmaxf(m[g], mt);
        const float al = mn == -__builtin_inff() ? 1.f : __builtin_amdgcn_exp2f(m[g] - mn);
        lsum[g] *= al;
#pragma unroll
        for (int e = 0; e < CH; ++e) o[g][e] *= al;
        m[g] = mn;
      }
      const float ms = m[g] == -__builtin_inff() ? 0.f : m[g];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[i][g] = __builtin_amdgcn_exp2f(s[i][g] - ms);
        lsum[g] += s[i][g];
      }
    }
    // ---- O += P V
#pragma unroll
    for (int n = 0; n < NO; ++n) {
      auto add = [&](int i, const float* x) {
#pragma unroll
        for (int g = 0; g < GS; ++g)
#pragma unroll
          for (int e = 0; e < 8; ++e) o[g][8 * n + e] = __builtin_fmaf(s[i][g], x[e], o[g][8 * n + e]);
      };
      if constexpr (FAST) {
        h2_t c[4][4];
        pairs(rv.v[n], n, cat.bits, c);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          // Keys past the split, rows without a chunk and blocks left out (!ok) add zeros: their
          // bytes are arbitrary, and a weight of 0 times an infinity is not 0.
          const bool live = cat.ok && i < n_live;
          const float vs = live ? (float)u2h(rv.vs[n][i])[0] : 0.f, vm = live ? (float)u2h(rv.vm[n][i])[0] : 0.f;
          float x[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] = __builtin_fmaf((float)c[i][e >> 1][e & 1], vs, vm);
          add(i, x);
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
        float x[4][8];
        general(std::false_type{}, cur, cat, n, opened ? n_live : 0, x);
#pragma unroll
        for (int i = 0; i < 4; ++i) add(i, x[i]);
      }
    }
    if (more) load_v(at);
  }

  // ---- the rows of each wave, then the waves, added --------------------------
  __shared__ __align__(16) float part[kDecWaves][GS][CH * GW];
  __shared__ float2 part_ml[kDecWaves][GS];
#pragma unroll
  for (int g = 0; g < GS; ++g) {
    float mm = m[g];
#pragma unroll
    for (int x = GW; x < 64; x <<= 1) mm = fmaxf(mm, __shfl_xor(mm, x, 64));
    const float al = m[g] == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(m[g] - mm);
    float ls = lsum[g] * al;
#pragma unroll
    for (int x = GW; x < 64; x <<= 1) ls += __shfl_xor(ls, x, 64);
#pragma unroll
    for (int e = 0; e < CH; ++e) {
      float v = o[g][e] * al;
#pragma unroll
      for (int x = GW; x < 64; x <<= 1) v += __shfl_xor(v, x, 64);
      if (row == 0) part[wv][g][8 * oct_of(e >> 3) + (e & 7)] = v;
    }
    if (lane == 0) part_ml[wv][g] = float2{mm, ls};
  }
  __syncthreads();
  const long row0 = (seq * a.hq + qh0) * a.num_splits + sp;  // + g * num_splits for query head g
  for (int i = tid; i < gs * D; i += kDecThreads) {
    const int g = i / D, d = i - g * D;
    float mm = -__builtin_inff();
#pragma unroll
    for (int x = 0; x < kDecWaves; ++x) mm = fmaxf(mm, part_ml[x][g].x);
    float ls = 0.f, v = 0.f;
#pragma unroll
    for (int x = 0; x < kDecWaves; ++x) {
      const float2 p = part_ml[x][g];
      const float al = p.x == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(p.x - mm);
      ls += p.y * al;
      v += part[x][g][d] * al;
    }
    const long r = row0 + (long)g * a.num_splits;
    a.acc[r * D + d] = v;
    if (d == 0) {
      a.ml[r * 2] = mm;
      a.ml[r * 2 + 1] = ls;
    }
  }
}

// Log-sum-exp merge of a row's splits (any D <= 256): one wave per (sequence, query head).
__global__ __launch_bounds__(256) void merge_any_kernel(MergeArgs a) {
  const int lane = threadIdx.x & 63;
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);  // seq * hq + head
  if (row >= a.rows) return;
  const long seq = row / a.hq;
  const int head = (int)(row % a.hq);
  if (head % a.gqa < a.g0 || head % a.gqa >= a.g0 + a.gs) return;  // another pass's query heads
  const long seq_len = a.lens[seq];
  if (seq_len <= 0) return;
  const long n_blocks = (seq_len + a.BS - 1) / a.BS;
  const long bps = split_blocks(a.sp, (int)n_blocks);
  const int used = (int)((n_blocks + bps - 1) / bps);
  const long base = row * a.num_splits;
  const int D = a.D;
  float m = -__builtin_inff();
  for (int s = lane; s < used; s += 64) m = fmaxf(m, a.ml[(base + s) * 2]);
  m = wave_max(m);
  float den = 0.f, num[kMaxAnyD / 64];
#pragma unroll
  for (int e = 0; e < kMaxAnyD / 64; ++e) num[e] = 0.f;
  for (int s = 0; s < used; ++s) {
    const float w = __builtin_amdgcn_exp2f(a.ml[(base + s) * 2] - m);
    den += a.ml[(base + s) * 2 + 1] * w;
    const float* src = a.acc + (base + s) * D;
#pragma unroll
    for (int e = 0; e < kMaxAnyD / 64; ++e)
      if (lane + 64 * e < D) num[e] += src[lane + 64 * e] * w;
  }
  const long o_row = a.q_rows ? a.q_rows[seq] : seq;
#pragma unroll
  for (int e = 0; e < kMaxAnyD / 64; ++e)
    if (lane + 64 * e < D) st(a.out, a.out_dtype, o_row * a.o_s0 + head * a.o_s1 + lane + 64 * e, num[e] / den);
}

// Chunked prefill for the same layouts (echokv_vllm/kernels/prefill.py:210-236, the
// reference's gather + bottom-right causal SDPA): one workgroup per (tile of
// query tokens, KV head). Its columns are (token i, query head g) pairs, at most
// 16; column (i, g) sees keys < q_pos0 + i + 1 of its request's context. The
// keys stream once per tile in 64-key tiles: 64 threads locate their token (block, chunk
// row, tier, residual row), 4 threads per token score it against the columns, one wave
// per 4 columns runs the online softmax, each thread owns one channel of O for a share
// of the tile's tokens; each column's row is normalized and written at the end.
__global__ __launch_bounds__(kAnyThreads) void prefill_any_kernel(PrefillArgs a) {
  const Lay& L = a.L;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int h = (int)(blockIdx.x % L.H);
  const int32_t* td = a.tiles + (long)(blockIdx.x / L.H) * 5;
  const long q_row0 = td[0];
  const int q_pos0 = td[2], ctx = td[3];
  const long bt_row = td[4];
  const int gs = a.gs;
  // The host sizes tiles to at most 16 columns; a larger tile is cut to its first
  // 16 / gs tokens rather than overrun the LDS rows.
  const int max_tok = kAnyCols / gs > 0 ? kAnyCols / gs : 1;
  const int n_tok = td[1] < max_tok ? td[1] : max_tok;
  const int n_cols = n_tok * gs;
  const long kv_end = q_pos0 + n_tok < ctx ? q_pos0 + n_tok : ctx;

  __shared__ __align__(16) float qs[kAnyCols * kMaxAnyD];
  __shared__ float ps[kAnyCols][kAnyTile];
  __shared__ float alpha[kAnyCols];
  __shared__ long rbs[kAnyTile], pbs[kAnyTile], kres[kAnyTile];
  __shared__ int offs[kAnyTile], bits_s[kAnyTile];

  const int D = L.D, quads = D / 4, G = D / L.VG;
  const int qh0 = h * a.gqa + a.g0;
  for (int i = tid; i < n_cols * D; i += kAnyThreads) {
    const int c = i / D, d = i - c * D;
    const int tok = c / gs, g = c - tok * gs;
    qs[i] = ld(a.q, a.q_dtype, (q_row0 + tok) * a.q_s0 + (long)(qh0 + g) * a.q_s1 + d) * a.scale_log2;
  }

  float m_run[4], l_run[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    m_run[i] = -__builtin_inff();
    l_run[i] = 0.f;
  }
  const int NT = kAnyThreads / D;
  const int r = tid / D, d = tid - r * D;
  float o[kAnyCols];
#pragma unroll
  for (int c = 0; c < kAnyCols; ++c) o[c] = 0.f;

  for (long t0 = 0; t0 < kv_end; t0 += kAnyTile) {
    __syncthreads();
    if (tid < kAnyTile) {
      const long pos = t0 + tid;
      long rb = -2, pb = 0, kr = -1;
      int off = 0, bits = 2;
      if (pos < kv_end) {
        const long b = pos / L.BS;
        off = (int)(pos - b * L.BS);
        const long blk = a.bt[bt_row * a.bt_s0 + b];
        if (blk >= 0 && blk < L.nb) {
          pb = blk * L.stride;
          bits = tier_of(a.pages[pb]);
          rb = row_base(a.pages, L, blk, off, bits);
          const long rs = a.block_res[blk];
          if (rs >= 0 && rs < a.res.rows && a.res_group[rs] == off / L.KG)
            kr = rs * a.res.s0 + (long)(off % L.KG) * a.res.s1 + (long)h * a.res.s2;
        }
      }
      rbs[tid] = rb;
      pbs[tid] = pb;
      kres[tid] = kr;
      offs[tid] = off;
      bits_s[tid] = bits;
    }
    __syncthreads();

    {
      const int j = tid >> 2, p = tid & 3;
      float s[kAnyCols];
#pragma unroll
      for (int c = 0; c < kAnyCols; ++c) s[c] = 0.f;
      const long rb = rbs[j];
      if (rb >= 0) {
        const long kr = kres[j];
        const int bits = bits_s[j];
        const uint8_t* kp = a.pages + rb + (long)h * (D * bits / 8);
        const long se = pbs[j] + 2 * (((long)(offs[j] / L.KG) * L.H + h) * D);
        for (int q4 = p; q4 < quads; q4 += 4) {
          float k[4];
          if (kr >= 0) {
            ld4(a.res.ptr, a.res.dtype, kr + 4 * q4, k);
          } else {
            const uint32_t kc = load_codes4(kp + q4 * (bits / 2), bits);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float ks = (float)*f16p(a.pages, se + L.o_ks + 2 * (4 * q4 + e));
              const float km = (float)*f16p(a.pages, se + L.o_km + 2 * (4 * q4 + e));
              k[e] = code_at(kc, e, bits) * ks + km;
            }
          }
#pragma unroll
          for (int c = 0; c < kAnyCols; ++c) {
            if (c < n_cols) {
              const float4 q = *(const float4*)&qs[c * D + 4 * q4];
              s[c] += q.x * k[0] + q.y * k[1] + q.z * k[2] + q.w * k[3];
            }
          }
        }
      }
#pragma unroll
      for (int c = 0; c < kAnyCols; ++c) {
        s[c] += __shfl_xor(s[c], 1, 64);
        s[c] += __shfl_xor(s[c], 2, 64);
      }
      if (p == 0) {
        const long pos = t0 + j;
#pragma unroll
        for (int c = 0; c < kAnyCols; ++c) {
          if (c < n_cols) {
            const long lim = q_pos0 + c / gs + 1;  // bottom-right causal: keys <= the query's position
            ps[c][j] = (rb == -2 || pos >= lim) ? -__builtin_inff() : s[c];
          }
        }
      }
    }
    __syncthreads();

#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = wv + 4 * i;
      if (c < n_cols) {
        const float x = ps[c][lane];
        const float m_new = fmaxf(m_run[i], wave_max(x));
        const bool none = m_new == -__builtin_inff();
        const float pr = none ? 0.f : __builtin_amdgcn_exp2f(x - m_new);
        const float al = none ? 1.f : __builtin_amdgcn_exp2f(m_run[i] - m_new);
        l_run[i] = l_run[i] * al + wave_sum(pr);
        m_run[i] = m_new;
        ps[c][lane] = pr;
        if (lane == 0) alpha[c] = al;
      }
    }
    __syncthreads();

    if (r < NT) {
#pragma unroll
      for (int c = 0; c < kAnyCols; ++c)
        if (c < n_cols) o[c] *= alpha[c];
      for (int j = r; j < kAnyTile; j += NT) {
        const long rb = rbs[j];
        if (rb < 0) continue;
        const int bits = bits_s[j];
        const long vb = rb + (long)(L.H + h) * (D * bits / 8) + ((d * bits) >> 3);
        const float code = (float)((a.pages[vb] >> ((d * bits) & 7)) & ((1u << bits) - 1u));
        const long ve = ((long)offs[j] * L.H + h) * G + d / L.VG;
        const float v = code * (float)*f16p(a.pages, pbs[j] + L.o_vs + 2 * ve) +
                        (float)*f16p(a.pages, pbs[j] + L.o_vm + 2 * ve);
#pragma unroll
        for (int c = 0; c < kAnyCols; ++c)
          if (c < n_cols) o[c] += ps[c][j] * v;
      }
    }
  }

  // Sum O's token shares, normalize, write each column's row.
  __syncthreads();
  if (r < NT) {
#pragma unroll
    for (int c = 0; c < kAnyCols; ++c)
      if (c < n_cols) qs[(r * n_cols + c) * D + d] = o[c];
  }
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = wv + 4 * i;
      if (c < n_cols) alpha[c] = l_run[i] > 0.f ? 1.f / l_run[i] : 0.f;
    }
  }
  __syncthreads();
  for (int i = tid; i < n_cols * D; i += kAnyThreads) {
    const int c = i / D, dd = i - c * D;
    float x = 0.f;
    for (int rr = 0; rr < NT; ++rr) x += qs[(rr * n_cols + c) * D + dd];
    const int tok = c / gs, g = c - tok * gs;
    st(a.out, a.out_dtype, (q_row0 + tok) * a.o_s0 + (long)(qh0 + g) * a.o_s1 + dd, x * alpha[c]);
  }
}

}  // namespace

// GS query heads of a KV head per workgroup: q and O take GS x channels registers each,
// and with 4 heads x 8 channels (2 x 16) the kernel needs 190, two waves a SIMD; more
// query heads read the keys again (from L2).
template <int GW, int NO, int GS>
static hipError_t decode_any_t(const DecodeArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)(a.num_seqs * a.L.H * a.num_splits), (unsigned)((a.gs + GS - 1) / GS));
  if (a.any_fast) hipLaunchKernelGGL((decode_any_kernel<GW, NO, GS, true>), grid, dim3(kDecThreads), 0, s, a);
  else hipLaunchKernelGGL((decode_any_kernel<GW, NO, GS, false>), grid, dim3(kDecThreads), 0, s, a);
  return hipGetLastError();
}
template <int GW, int NO>
static hipError_t decode_any_d(const DecodeArgs& a, hipStream_t s) {
  if (a.gs == 1) return decode_any_t<GW, NO, 1>(a, s);
  return decode_any_t<GW, NO, 4 / NO>(a, s);
}

hipError_t launch_decode_any(const DecodeArgs& a, hipStream_t s) {
  if (a.L.D <= 64) return decode_any_d<8, 1>(a, s);
  if (a.L.D <= 128) return decode_any_d<16, 1>(a, s);
  return decode_any_d<16, 2>(a, s);
}

hipError_t launch_prefill_any(const PrefillArgs& a, long n_tiles, hipStream_t s) {
  hipLaunchKernelGGL(prefill_any_kernel, dim3((unsigned)(n_tiles * a.L.H)), dim3(kAnyThreads), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_merge_any(const MergeArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(merge_any_kernel, dim3((unsigned)((a.rows + 3) / 4)), dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace ek
