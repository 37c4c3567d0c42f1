// Chunked-prefill attention over the tiered pages on gfx950 MFMA tiles.
//
// One workgroup (4 waves) per (query tile, KV head, key range). A tile holds up to
// 128 / GQA query tokens; its rows are (token, GQA head) pairs, 128 rows, 32
// per wave (two 16-row blocks) -- at head size 256, 64 / GQA tokens and one
// 16-row block per wave (RB), so a wave's accumulators and query fragments take
// the registers they take at 128. The range's keys are walked in steps of 8192 / D
// keys: the workgroup dequantizes a step's keys once into LDS -- K row-major as an
// fp16 hi + lo pair (exact to ~2^-22), V transposed in fp16 -- and every wave then
// runs, per 16-row block and 32 keys (64 at head size 64),
//   S^T[key, row] = K Q^T         (v_mfma_f32_16x16x32_f16 on K hi and K lo)
//   O^T[d, row]  += V^T P^T       (v_mfma_f32_16x16x32_f16, D/16 per block)
// with a per-row online softmax and the bottom-right causal limit
// key <= query position (echokv_vllm/kernels/prefill.py:210-236 semantics).
// The S^T accumulator (lane = 4 keys x 1 row) is the P^T B-operand as is: the
// 32-key contraction maps lane group c's eight k-slots to keys
// {4c..4c+3, 16+4c..16+4c+3}, and V^T rows hold the keys in that order.
//
// Key ranges (PrefillArgs::items): short chunks over long contexts give few
// (tile, head) pairs, and a pair's context is a serial chain of steps. So a tile's
// context is cut into ranges, one workgroup each; a range leaves
// its rows' unnormalized output and (max, sum), and prefill_merge_kernel adds them.
// A tile whose context is one range writes its rows directly. 4 chunks of 5-64
// tokens over 0.7-8K-token INT4 contexts, H 8, D 128: 857 us in one range per pair, 55 us
// cut (about 50 in this kernel, whose waves, two a SIMD, issue in 38 % of their cycles and
// wait for loads, barriers and one another in the rest; 5 in the merge).
//
// A thread dequantizes one item of a step: 4 consecutive keys (one block, chunk and K
// group) x 8 channels, so one 16-byte load each of K scale and K min serves four
// keys, and V^T takes 8-byte stores. Its loads are a chain (block table, page
// header, codes) that is spread over the steps: step i + 1's codes, step i + 2's
// header and step i + 3's table entry are requested before step i's products.
// Items whose keys or channels straddle a group (K group not a multiple of 4, V
// group not of 8), and blocks or groups that are not powers of two, are read by
// item_general in the step that needs them (64 chunks of 16-32 tokens over 1-4K keys at
// block 48: 1190 us element by element, 614 so).
#include "items.h"

namespace ek {

namespace {

// max / sum over lanes l, l ^ 16, l ^ 32, l ^ 48 (every lane gets the result).
__device__ __forceinline__ float rows_max(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}

// LDS rows are unpadded; 16-byte slots are permuted by row so that the stores and the
// fragment reads (16 rows at one slot) both spread over the banks.
template <int D>
__device__ __forceinline__ int k_slot(int key, int slot) {
  return slot ^ (D == 64 ? (key >> 1) & 7 : key & 15);
}
template <int KEYS>
__device__ __forceinline__ int v_slot(int d, int slot) {
  return slot ^ (((d >> 1) ^ (d >> 4)) & (KEYS / 8 - 1) & 7);
}

// Four keys x eight channels: each row's eight codes in the 8 bytes at or before them.
struct Raw {
  uint2 k[4], v[4];
  uint4 ks, km;  // fp16 scale / min of the eight channels (the quad's K group)
  uint16_t vs[4], vm[4];  // the four tokens' V scale / min of the channels' V group
  int rg;                 // K group of the block's residual slot (if it has one)
  bool ok;                // the item's keys can be read
};

// Ranges of `per` keys of a tile of n_rows query rows over kv_end keys, of the `ranges` of
// `rows` query rows that it has partial rows for (0 or 1: it is taken in one piece).
__device__ __forceinline__ int tile_ranges(int ranges, int rows, int n_rows, int kv_end, int per) {
  if (ranges <= 1 || n_rows > rows) return 1;
  const int need = (kv_end + per - 1) / per;
  return need < ranges ? need : ranges;
}

// Query and output rows: vectors at any element's alignment.
typedef float f4_any_t __attribute__((ext_vector_type(4), aligned(4)));
typedef _Float16 h8_any_t __attribute__((ext_vector_type(8), aligned(2)));
typedef _Float16 h4_any_t __attribute__((ext_vector_type(4), aligned(2)));
typedef __bf16 b4_any_t __attribute__((ext_vector_type(4), aligned(2)));

// Four consecutive elements by one store. DT is a template parameter so that the dtype
// branch sits outside the caller's loop (the kernel's code is fetched cold at every
// launch: its size is time).
template <int DT>
__device__ __forceinline__ void st4v(void* p, long i, const f4_t x) {
  if constexpr (DT == ECHOKV_F32) {
    *(f4_any_t*)((float*)p + i) = x;
  } else if constexpr (DT == ECHOKV_F16) {
    *(h4_any_t*)((_Float16*)p + i) = h4_any_t{(_Float16)x[0], (_Float16)x[1], (_Float16)x[2], (_Float16)x[3]};
  } else {
    *(b4_any_t*)((__bf16*)p + i) = b4_any_t{(__bf16)x[0], (__bf16)x[1], (__bf16)x[2], (__bf16)x[3]};
  }
}

}  // namespace

// FAST (PrefillArgs::fast): power-of-two block size and K group, items inside one K group
// and V group. Other layouts take the same kernel with items read by item_general.
template <int D, bool QLO, int RB, bool FAST>
__global__ __launch_bounds__(256, QLO && D > 64 ? 1 : 2) void prefill_kernel(PrefillArgs a) {
  constexpr int KEYS = 8192 / D;            // keys per step: 256 items of 4 keys x 8 channels
  constexpr int SB = D == 64 ? 64 : 32;      // keys per softmax update (registers: no spill)
  constexpr int NKH = SB / 16;
  constexpr int NQK = D / 32;
  constexpr int NPV = D / 16;
  constexpr int OCTS = D / 8;
  __shared__ __attribute__((aligned(16))) _Float16 kt[KEYS * D];   // K, fp16 hi part
  __shared__ __attribute__((aligned(16))) _Float16 ktl[KEYS * D];  // K, fp16 lo part
  __shared__ __attribute__((aligned(16))) _Float16 vt[D * KEYS];

  const Lay& L = a.L;
  // Heads fastest: a request's tiles of one range and head are H workgroups apart, which
  // for 8 heads is the same XCD and its L2 (4 chunks over 0.7-8K keys 69 -> 65.5 us).
  const int h = blockIdx.x % a.L.H;
  int tile = blockIdx.x / a.L.H, z = 0, ranges = 1;
  long part0 = 0;  // the tile's partial rows: first, and rows per range
  int part_rows = 0, per = 0;
  if (a.items) {
    const int32_t* it = a.items + 5 * (long)tile;
    tile = it[0] / kPrefillMaxRanges;
    z = it[0] % kPrefillMaxRanges;
    ranges = it[1];
    per = it[2];
    part0 = it[3] - a.row0;
    part_rows = it[4];
  }
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int c = lane >> 4, n = lane & 15;
  const int32_t* td = a.tiles + tile * 5;
  const long q_row0 = td[0];
  const int n_tok = td[1], q_pos0 = td[2], ctx = td[3];
  const long req = td[4];
  const int gqa = a.gqa;
  const int n_rows = n_tok * gqa;
  int kv_end = q_pos0 + n_tok;
  kv_end = kv_end < ctx ? kv_end : ctx;
  ranges = tile_ranges(ranges, part_rows, n_rows, kv_end, per);
  if (z > 0 && z >= ranges) return;
  const int k_begin = z * per;
  const int k_end = z >= ranges - 1 ? kv_end : k_begin + per;  // the last takes the rest

  // ---- this thread's item of a step, and its chain of loads ----------------
  const int oct = tid % OCTS, quad = tid / OCTS;
  const int ch = 8 * oct;
  const int G = D / L.VG, vg = ch / L.VG;
  auto block_of = [&](int kp) { return FAST ? kp >> a.bs_shift : kp / L.BS; };
  auto group_of = [&](int off) { return FAST ? off >> a.kg_shift : off / L.KG; };
  auto item_key = [&](int step) { return k_begin + step * KEYS + 4 * quad; };
  auto item_off = [&](int step) {
    const int kp = item_key(step);
    return FAST ? kp & ((1 << a.bs_shift) - 1) : kp % L.BS;
  };
  // Nothing loaded is looked at before the step that needs it, and no load sits in a
  // branch (addresses are clamped instead): a value that is converted or merged where it
  // is loaded would be waited for there.
  auto load_blk = [&](int step) -> int {
    const int kp = item_key(step);
    const int last_key = k_end > 1 ? k_end - 1 : 0;
    return a.bt[req * a.bt_s0 + block_of(kp < last_key ? kp : last_key)];
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
  auto valid = [&](int step, const Head& x) { return (unsigned)x.blk < (unsigned long)L.nb && item_key(step) < k_end; };
  // Byte offset of the item's first token row (-1: its chunk id is out of range).
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
  auto load_raw = [&](int step, const Head& x, Raw& w) {
    const long rs = (unsigned long)x.rs < (unsigned long)a.res.rows ? x.rs : 0;
    w.rg = *(const int32_t*)(a.res_group + rs);  // the low word: groups are small
    if (!FAST) return;
    const int off = item_off(step), bits = tier_of(x.hd().tag);
    const long rb = item_row(x, off, bits);
    w.ok = rb >= 0 && valid(step, x);
    const uint8_t* pg = a.pages + page_of(x.blk) * L.stride;
    // A quad without a chunk reads its page's first bytes instead (dequantized to zero).
    const uint8_t* kp = rb >= 0 ? a.pages + rb + ((h * D + ch) * bits / 8 & ~7) : pg;
    const int rowb = rb >= 0 ? L.H * (D / 4) * bits : 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      w.k[i] = *(const uint2*)(kp + i * rowb);
      w.v[i] = *(const uint2*)(kp + i * rowb + rowb / 2);
    }
    const int se = (group_of(off) * L.H + h) * D + ch;
    w.ks = *(const uint4*)(pg + L.o_ks + 2 * se);
    w.km = *(const uint4*)(pg + L.o_km + 2 * se);
    const int ve = (off * L.H + h) * G + vg;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      w.vs[i] = *(const uint16_t*)(pg + L.o_vs + 2 * (ve + i * L.H * G));
      w.vm[i] = *(const uint16_t*)(pg + L.o_vm + 2 * (ve + i * L.H * G));
    }
  };
  // The item's keys, dequantized into LDS (keys past the range and blocks that cannot be
  // read: zeros).
  auto store_item = [&](int step, const Head& x, const Raw& w) {
    const int kp = item_key(step);
    const int off = item_off(step), bits = tier_of(x.hd().tag);
    const long pg = page_of(x.blk) * L.stride;
    const bool has_res = (unsigned long)x.rs < (unsigned long)a.res.rows;
    const int key0 = 4 * quad;
    auto put_k = [&](int i, const float* x8) {
      h8_t hi, lo;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        hi[e] = (_Float16)x8[e];
        lo[e] = (_Float16)(x8[e] - (float)hi[e]);
      }
      const int at = (key0 + i) * D + 8 * k_slot<D>(key0 + i, oct);
      *(h8_t*)&kt[at] = hi;
      *(h8_t*)&ktl[at] = lo;
    };
    // V^T: inside each 32 keys, keys 16 p + 4 c + i sit at 8 c + 4 p + i.
    const int q32 = quad & 7, pos = (quad >> 3) * 32 + 8 * (q32 & 3) + 4 * (q32 >> 2);
    auto v_at = [&](int e) { return (ch + e) * KEYS + 8 * v_slot<KEYS>(ch + e, pos >> 3) + (pos & 4); };
    if constexpr (FAST) {
      const bool in_res = w.ok && has_res && w.rg == group_of(off);
      const int n_live = w.ok ? k_end - kp : 0;
      const int sh = 8 * (((h * D + ch) * bits / 8) & 7);
      auto rows = [&](auto width) {
        constexpr int B = decltype(width)::value;
        const uint32_t sw[4] = {w.ks.x, w.ks.y, w.ks.z, w.ks.w}, mw[4] = {w.km.x, w.km.y, w.km.z, w.km.w};
        h2_t v[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          h2_t c[4];
          code_pairs<B>(w.k[i], sh, c);
          float x8[8];
#pragma unroll
          for (int e = 0; e < 8; ++e)
            x8[e] = __builtin_fmaf((float)c[e >> 1][e & 1], (float)u2h(sw[e >> 1])[e & 1], (float)u2h(mw[e >> 1])[e & 1]);
          put_k(i, x8);
          code_pairs<B>(w.v[i], sh, c);
          const h2_t vs = u2h(w.vs[i] * 0x10001u), vm = u2h(w.vm[i] * 0x10001u);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[i][e] = __builtin_elementwise_fma(c[e], vs, vm);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e)
          *(h4_t*)&vt[v_at(e)] = h4_t{v[0][e >> 1][e & 1], v[1][e >> 1][e & 1], v[2][e >> 1][e & 1], v[3][e >> 1][e & 1]};
      };
      if (bits == 4) rows(std::integral_constant<int, 4>{});
      else if (bits == 2) rows(std::integral_constant<int, 2>{});
      else rows(std::integral_constant<int, 8>{});
      if (n_live < 4) {  // rare: past the range's end, or a block that cannot be read
        const float z8[8] = {};
#pragma unroll 1
        for (int i = n_live > 0 ? n_live : 0; i < 4; ++i) {
          put_k(i, z8);
#pragma unroll
          for (int e = 0; e < 8; ++e) vt[v_at(e) + i] = (_Float16)0.f;
        }
      }
      if (in_res) {  // rare: the request's open K group
#pragma unroll 1
        for (int i = 0; i < 4 && kp + i < k_end; ++i) {
          float x8[8];
          ld_n<8>(a.res.ptr, a.res.dtype,
                  x.rs * a.res.s0 + (long)((off + i) & (L.KG - 1)) * a.res.s1 + h * a.res.s2 + ch, x8);
          put_k(i, x8);
        }
      }
      return;
    }
    const int n_live = valid(step, x) ? k_end - kp : 0;
    float y[4][8];
    item_general<true>(L, a.pages, a.res, page_of(x.blk), x.hd(), x.rs, w.rg, off, bits, n_live, h, ch, y);
#pragma unroll
    for (int i = 0; i < 4; ++i) put_k(i, y[i]);
    item_general<false>(L, a.pages, a.res, page_of(x.blk), x.hd(), x.rs, w.rg, off, bits, n_live, h, ch, y);
#pragma unroll
    for (int e = 0; e < 8; ++e)
      *(h4_t*)&vt[v_at(e)] = h4_t{(_Float16)y[0][e], (_Float16)y[1][e], (_Float16)y[2][e], (_Float16)y[3][e]};
  };

  const int n_steps = (k_end - k_begin + KEYS - 1) / KEYS;
  Raw raw;
  Head head = load_head(load_blk(0));
  Head head1 = load_head(load_blk(1));
  int blk2 = load_blk(2);
  load_raw(0, head, raw);

  // Scores are scaled inside the exponent, and the max is taken on unscaled scores,
  // which needs the scale positive: a negative one flips the query's sign (exact), a
  // zero one becomes 2^-100 (every weight equal, and masked scores stay -inf).
  constexpr float kTinyScale = 7.8886090522101181e-31f;
  const float scale = fabsf(a.scale_log2) < kTinyScale ? kTinyScale : fabsf(a.scale_log2);  // NaN stays

  // Query fragments (B operand of S^T): row = 16*RB*wave + 16*rb + n, channels
  // 32j + 8c .. +8 in natural order.
  h8_t qf[RB][NQK], qfl[QLO ? RB : 1][NQK];
  int qlim[RB];  // keys < qlim are visible
  #pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int r = 16 * RB * wave + 16 * rb + n;
    const int tok = r < n_rows ? r / gqa : 0;
    const int hh = h * gqa + (r < n_rows ? r % gqa : 0);
    qlim[rb] = og_limit(q_pos0 + tok, a.og_mask);
    const long qb = (q_row0 + tok) * a.q_s0 + (long)hh * a.q_s1;
    // Rows past the tile read its first row (never written out).
    if constexpr (QLO) {
#pragma unroll
      for (int j = 0; j < NQK; ++j) {
        const f4_any_t* src = (const f4_any_t*)((const float*)a.q + qb + 32 * j + 8 * c);
        const f4_t u = src[0], v = src[1];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float x = e < 4 ? u[e & 3] : v[e & 3];
          qf[rb][j][e] = (_Float16)x;
          qfl[rb][j][e] = (_Float16)(x - (float)qf[rb][j][e]);
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < NQK; ++j) qf[rb][j] = *(const h8_any_t*)((const _Float16*)a.q + qb + 32 * j + 8 * c);
    }
  }
  if (!QLO && a.q_dtype == ECHOKV_BF16) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int j = 0; j < NQK; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          qf[rb][j][e] = (_Float16)bf16_to_f32(__builtin_bit_cast(uint16_t, (_Float16)qf[rb][j][e]));
  }
  if (a.scale_log2 < 0.f) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int j = 0; j < NQK; ++j) {
        qf[rb][j] = -qf[rb][j];
        if constexpr (QLO) qfl[rb][j] = -qfl[rb][j];
      }
  }
  // The wave's rows: none (inactive), the keys any of them sees, and a bound below every
  // row's limit (no masking under it).
  const int r0 = 16 * RB * wave;
  const bool active = r0 < n_rows;
  const int r1 = r0 + 16 * RB - 1 < n_rows - 1 ? r0 + 16 * RB - 1 : n_rows - 1;
  const int kend_w = active ? (q_pos0 + r1 / gqa + 1 < k_end ? q_pos0 + r1 / gqa + 1 : k_end) : 0;
  const int qmin = q_pos0 + r0 / gqa;
  const int lim_min = a.og_mask ? (qmin & a.og_mask) : qmin + 1;

  f4_t acc[RB][NPV];
  float m_run[RB], l_lane[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
    for (int j = 0; j < NPV; ++j) acc[rb][j] = f4_t{0.f, 0.f, 0.f, 0.f};
    m_run[rb] = -__builtin_inff();
    l_lane[rb] = 0.f;
  }

  for (int step = 0; step < n_steps; ++step) {
    __syncthreads();  // every wave is done with the previous step's keys
    store_item(step, head, raw);
    __syncthreads();
    if (step + 1 < n_steps) {
      head = head1;
      load_raw(step + 1, head, raw);
      head1 = load_head(blk2);
      blk2 = load_blk(step + 3);
    }
#pragma unroll 1
    for (int sb = 0; sb < KEYS; sb += SB) {
      const int kb = k_begin + step * KEYS + sb;
      if (kb >= kend_w) break;
      f4_t s[RB][NKH];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int kh = 0; kh < NKH; ++kh) s[rb][kh] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NQK; ++j) {
        h8_t kf[NKH], kl[NKH];
#pragma unroll
        for (int kh = 0; kh < NKH; ++kh) {
          const int key = sb + 16 * kh + n;
          const int at = key * D + 8 * k_slot<D>(key, 4 * j + c);
          kf[kh] = *(const h8_t*)&kt[at];
          kl[kh] = *(const h8_t*)&ktl[at];
        }
        // The accumulators in turn, so that no product waits for the one before it.
        auto products = [&](const h8_t* kx, const h8_t (*qx)[NQK]) {
#pragma unroll
          for (int kh = 0; kh < NKH; ++kh)
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
              s[rb][kh] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kx[kh], qx[rb][j], s[rb][kh], 0, 0, 0);
        };
        products(kf, qf);
        products(kl, qf);
        if constexpr (QLO) products(kf, qfl);
        __builtin_amdgcn_sched_barrier(0);  // one block of channels' fragments live at a time
      }
      const bool masked = kb + SB > lim_min || kb + SB > k_end;  // wave-uniform
      h8_t pb[RB][SB / 32];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        float mt = -__builtin_inff();
#pragma unroll
        for (int kh = 0; kh < NKH; ++kh) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float v = s[rb][kh][i];
            if (masked) {
              const int kp = kb + 16 * kh + 4 * c + i;
              v = kp < k_end && kp < qlim[rb] ? v : -__builtin_inff();
            }
            s[rb][kh][i] = v;
            mt = fmaxf(mt, v);
          }
        }
        mt = rows_max(mt) * scale;
        // Exact running max: a row's largest weight is then 1, without a rounding (letting
        // it lag by up to 2^8 saved 2 us of 60 and cost 10-20 % in accuracy).
        if (__builtin_amdgcn_ballot_w64(mt > m_run[rb])) {
          const float m_new = fmaxf(m_run[rb], mt);
          const float alpha = m_new == -__builtin_inff() ? 1.f : __builtin_amdgcn_exp2f(m_run[rb] - m_new);
          l_lane[rb] *= alpha;
          m_run[rb] = m_new;
#pragma unroll
          for (int j = 0; j < NPV; ++j) acc[rb][j] *= alpha;
        }
        const float m_safe = m_run[rb] == -__builtin_inff() ? 0.f : m_run[rb];
        // The row sum takes the float32 weights: the log-sum-exp is made of it.
        float psum[2] = {0.f, 0.f};
#pragma unroll
        for (int kh = 0; kh < NKH; ++kh) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[rb][kh][i], scale, -m_safe));
            psum[i & 1] += p;
            pb[rb][kh >> 1][4 * (kh & 1) + i] = (_Float16)p;
          }
        }
        l_lane[rb] += psum[0] + psum[1];
      }
#pragma unroll
      for (int ps = 0; ps < SB / 32; ++ps) {
#pragma unroll
        for (int j = 0; j < NPV; ++j) {
          const int d = 16 * j + n;
          const h8_t vf = *(const h8_t*)&vt[d * KEYS + 8 * v_slot<KEYS>(d, sb / 8 + 4 * ps + c)];
#pragma unroll
          for (int rb = 0; rb < RB; ++rb)
            acc[rb][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pb[rb][ps], acc[rb][j], 0, 0, 0);
          if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }

  const bool direct = ranges <= 1;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    l_lane[rb] += __shfl_xor(l_lane[rb], 16, 64);
    l_lane[rb] += __shfl_xor(l_lane[rb], 32, 64);
    const float inv = !direct ? 1.f : l_lane[rb] > 0.f ? 1.f / l_lane[rb] : 0.f;
#pragma unroll
    for (int j = 0; j < NPV; ++j) acc[rb][j] *= inv;
  }
  auto rows = [&](auto put) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const int r = 16 * RB * wave + 16 * rb + n;
      if (r < n_rows) put(rb, r);
    }
  };
  if (!direct) {
    rows([&](int rb, int r) {
      const long pr = (part0 + (long)z * part_rows) * L.H + (long)h * part_rows + r;
      if (c == 0) *(float2*)(a.ml + 2 * pr) = float2{m_run[rb], l_lane[rb]};
#pragma unroll
      for (int j = 0; j < NPV; ++j) *(f4_t*)(a.acc + pr * D + 16 * j + 4 * c) = acc[rb][j];
    });
    return;
  }
  auto put_out = [&](auto dt) {
    constexpr int DT = decltype(dt)::value;
    rows([&](int rb, int r) {
      const long row = q_row0 + r / gqa;
      const int qh = h * gqa + r % gqa;
      const long ob = row * a.o_s0 + (long)qh * a.o_s1;
      if (a.lse && c == 0)
        a.lse[row * a.hq + qh] = l_lane[rb] > 0.f ? m_run[rb] + __log2f(l_lane[rb]) : -__builtin_inff();
#pragma unroll
      for (int j = 0; j < NPV; ++j) st4v<DT>(a.out, ob + 16 * j + 4 * c, acc[rb][j]);
    });
  };
  if (a.out_dtype == ECHOKV_BF16) put_out(std::integral_constant<int, ECHOKV_BF16>{});
  else if (a.out_dtype == ECHOKV_F16) put_out(std::integral_constant<int, ECHOKV_F16>{});
  else put_out(std::integral_constant<int, ECHOKV_F32>{});
}

// The ranges of a tile's rows added (log-sum-exp, in range order) and normalized: one
// wave per row, lane l channels [D/64 l, D/64 (l + 1)).
template <int D>
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillArgs a) {
  constexpr int C = D / 64;
  const int32_t* it = a.merges + 5 * (long)blockIdx.x;
  const int32_t* td = a.tiles + (long)(it[0] / kPrefillMaxRanges) * 5;
  const int n_tok = td[1], q_pos0 = td[2], ctx = td[3];
  const int kv_end = q_pos0 + n_tok < ctx ? q_pos0 + n_tok : ctx;
  const int ns = tile_ranges(it[1], it[4], n_tok * a.gqa, kv_end, it[2]);  // at most 64
  if (ns <= 1) return;  // written directly
  const int lane = threadIdx.x & 63;
  const int r = (int)blockIdx.z * 4 + (int)(threadIdx.x >> 6);
  if (r >= n_tok * a.gqa) return;
  const int h = blockIdx.y;
  const long row = td[0] + r / a.gqa;
  const int qh = h * a.gqa + r % a.gqa;
  const int rows = it[4];
  const long base = (long)(it[3] - a.row0) * a.L.H + (long)h * rows + r, per = (long)rows * a.L.H;
  // The (max, sum) pairs and the first 16 ranges' rows are requested together.
  const float2 p = lane < ns ? *(const float2*)(a.ml + 2 * (base + lane * per)) : float2{-__builtin_inff(), 0.f};
  float o[C] = {}, mm = 0.f, w = 0.f, den = 0.f;
  for (int s0 = 0; s0 < ns; s0 += 16) {
    float x[16][C];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const float* src = a.acc + (base + (s0 + u < ns ? s0 + u : 0) * per) * D + C * lane;
#pragma unroll
      for (int e = 0; e < C; ++e) x[u][e] = src[e];
    }
    if (s0 == 0) {
      mm = p.x;
#pragma unroll
      for (int m = 32; m > 0; m >>= 1) mm = fmaxf(mm, __shfl_xor(mm, m, 64));
      w = p.x == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(p.x - mm);
      den = w * p.y;
#pragma unroll
      for (int m = 32; m > 0; m >>= 1) den += __shfl_xor(den, m, 64);
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      if (s0 + u < ns) {
        const float wu = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w), s0 + u));
#pragma unroll
        for (int e = 0; e < C; ++e) o[e] += x[u][e] * wu;
      }
    }
  }
  const float inv = den > 0.f ? 1.f / den : 0.f;
#pragma unroll
  for (int e = 0; e < C; ++e) o[e] *= inv;
  if (a.lse && lane == 0) a.lse[row * a.hq + qh] = den > 0.f ? mm + __log2f(den) : -__builtin_inff();
  st_n<C>(a.out, a.out_dtype, row * a.o_s0 + (long)qh * a.o_s1 + C * lane, o);
}

template <int D, int RB>
static hipError_t prefill_d(const PrefillArgs& a, long n, long n_merges, hipStream_t s) {
  const dim3 grid((unsigned)(n * a.L.H));
  const bool f32 = a.q_dtype == ECHOKV_F32;
  if (f32 && a.fast) hipLaunchKernelGGL((prefill_kernel<D, true, RB, true>), grid, dim3(256), 0, s, a);
  else if (f32) hipLaunchKernelGGL((prefill_kernel<D, true, RB, false>), grid, dim3(256), 0, s, a);
  else if (a.fast) hipLaunchKernelGGL((prefill_kernel<D, false, RB, true>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((prefill_kernel<D, false, RB, false>), grid, dim3(256), 0, s, a);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || n_merges == 0) return e;
  const unsigned rows = (unsigned)prefill_rows(D);
  hipLaunchKernelGGL((prefill_merge_kernel<D>), dim3((unsigned)n_merges, (unsigned)a.L.H, rows / 4), dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_prefill(const PrefillArgs& a, long n, long n_merges, hipStream_t s) {
  if (a.L.D == 128) return prefill_d<128, 2>(a, n, n_merges, s);
  if (a.L.D == 64) return prefill_d<64, 2>(a, n, n_merges, s);
  if (a.L.D == 256) return prefill_d<256, 1>(a, n, n_merges, s);
  return hipErrorInvalidValue;
}

}  // namespace ek
