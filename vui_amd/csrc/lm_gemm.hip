// The matrix products of the token language models, one kernel template: C (M x N) = X (M x K) W^T (N x K) on the
// matrix cores (bf16 or true fp32), both operands tiled, K split over the waves of a workgroup (partial tiles meet in
// LDS and are added in wave order).  What a layer does with the sums is the epilogue.
//
// Parallel layers: the norm has a single number for its weight, so W norm(x) = s W x with one scale s per row: the product
// runs on the raw residual row and the epilogue scales.  The sum of squares behind s is left by whoever wrote the
// row, in pieces of 16 columns (LM_OUT, the embedding), so no launch is spent on norms.
#include "common.h"
#include "lm.h"
#include "wide.h"

__device__ __forceinline__ float lm_sigmoid(float v) { return 1.0f / (1.0f + expf(-v)); }

// gated feed-forward with clamped branches, two features from interleaved (gate, up) pairs
__device__ __forceinline__ float lm_ff(float g, float u, float limit) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g * lm_sigmoid(1.702f * g) * (u + 1.0f);
}

// rotates two pairs held as (u0, v0, u1, v1); pair indices i, i + 1; pairs at or beyond n pass
__device__ __forceinline__ void lm_rotate2(float* v, const float* rope, int pos, int n, int i) {
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if (i + k < n) {
      const float2 f = *reinterpret_cast<const float2*>(rope + ((size_t)pos * n + i + k) * 2);
      const float a = v[2 * k], b = v[2 * k + 1];
      v[2 * k] = a * f.x - b * f.y;
      v[2 * k + 1] = b * f.x + a * f.y;
    }
  }
}

// activations of ungated feed-forwards
__device__ __forceinline__ float lm_act(float z, int kind, float pos, float neg) {
  if (kind == VUI_LM_ACT_RELU2) { z = fmaxf(z, 0.f); return z * z; }
  const float m = fminf(z, 0.f);
  return (z > 0.f ? pos * z * z : neg * (expm1f(m) - m)) + 0.5f * z;
}

// Rows of a pass up to which sums of squares come as pairs (rows x np x 2), a half of a block's columns each, or the whole and 0: what half
// blocks of an output projection can leave.  With more rows there is one per block: two cost a prompt of 1999 positions 1.3 %.
#define LM_PAIRS 16

// What a unit's epilogue reads besides the sums, requested ahead of the operands (few rows).
struct LmPre {
  int slot, pos;
  float4 a, b, c;
};

// One unit of 16 rows x 16 features: a lane holds features n ... n + 3 of row m.  half: of the block's features, that half alone (LM_OUT).  mix: the unit is the update gate of a recurrence, xv and gv the candidate and the output gate beside it.
template <typename T, int EPI, bool PRE>
__device__ __forceinline__ void lm_unit(const LmGemm& p, const int m, const int nb, const int n, const int l16, const int kg,
                                        const bool live, const bool mix, float (&v)[4], const float (&xv)[4], const float (&gv)[4],
                                        const LmPre& e, const int half = -1) {
  constexpr bool GRU = EPI == LM_IN_GRU_STEP || EPI == LM_IN_GRU_SEQ;
  constexpr bool LOGITS = EPI == LM_LOGITS || EPI == LM_HEAD;
  if (GRU && mix) {
    const int ch = (nb / 3) * 16 + 4 * kg;  // blocks come in threes: update gate, candidate, output gate
    if (!live) return;
    const float4 b0 = PRE ? e.b : *reinterpret_cast<const float4*>(p.bz + ch), b1 = PRE ? e.c : *reinterpret_cast<const float4*>(p.bx + ch);
    const float zb[4] = {b0.x, b0.y, b0.z, b0.w}, xb[4] = {b1.x, b1.y, b1.z, b1.w};
    float keep[4], in[4], sg[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float zz = v[r] + zb[r], uu = xv[r] + xb[r];
      const float z = lm_sigmoid(zz);
      keep[r] = lm_sigmoid(-zz);
      in[r] = z * (uu >= 0.f ? uu + 0.5f : lm_sigmoid(uu));
      sg[r] = gv[r] * lm_sigmoid(gv[r]);
    }
    if (EPI == LM_IN_GRU_STEP) {
      float4* sp = reinterpret_cast<float4*>(p.state + (size_t)e.slot * p.d.gru16 + ch);
      const float4 old = e.pos > 0 ? e.a : make_float4(0.f, 0.f, 0.f, 0.f);
      const float4 nw = make_float4(fmaf(keep[0], old.x, in[0]), fmaf(keep[1], old.y, in[1]), fmaf(keep[2], old.z, in[2]),
                                    fmaf(keep[3], old.w, in[3]));
      *sp = nw;
      const float o[4] = {nw.x * sg[0], nw.y * sg[1], nw.z * sg[2], nw.w * sg[3]};
      Tl<T>::st4((T*)p.act + tl_off<T>(m, ch, p.d.out_k), o);
    } else {
      float4* up = reinterpret_cast<float4*>(p.upd + (size_t)m * p.d.gru16 + ch);
      up[0] = make_float4(keep[0], in[0], keep[1], in[1]);
      up[1] = make_float4(keep[2], in[2], keep[3], in[3]);
      Tl<T>::st4((T*)p.sg + (size_t)m * p.d.gru16 + ch, sg);
    }
    return;
  }
  if (EPI == LM_IN_ATTN || GRU) {
    if (!live) return;
    if (nb >= p.mix_blocks) {  // (gate, up) pairs
      const int f = (n - p.mix_blocks * 16) >> 1;
      Tl<T>::st2((T*)p.act + tl_off<T>(m, p.d.ff_off + f, p.d.out_k), lm_ff(v[0], v[1], p.limit), lm_ff(v[2], v[3], p.limit));
      return;
    }
    if (EPI == LM_IN_ATTN) {
      if (nb < p.b_qr) {
        const int dq = p.d.dim16 >> 4, h = nb / dq, o = (nb - h * dq) * 16 + 4 * kg;
        Tl<T>::st4((T*)p.qu + h * p.qu_z + tl_off<T>(m, o, p.d.dim64), v);
      } else if (nb < p.b_c) {
        const int dr = p.d.rot16 >> 4, b = nb - p.b_qr, h = b / dr, o = (b - h * dr) * 16 + 4 * kg;
        const int pos = min(max(PRE ? e.pos : lm_where(p.rows, m).y, 0), p.rows.S - 1);
        lm_rotate2(v, p.rope, pos, p.rot_pairs, o >> 1);
        Tl<T>::st4((T*)p.qr + h * p.qr_z + tl_off<T, 32>(m, o, p.d.rot32), v);
      } else if (nb < p.b_kr) {
        const int o = (nb - p.b_c) * 16 + 4 * kg;
        *reinterpret_cast<float4*>(p.craw + (size_t)m * p.d.rank16 + o) = make_float4(v[0], v[1], v[2], v[3]);
      } else if (nb < p.b_g) {
        const int o = (nb - p.b_kr) * 16 + 4 * kg;
        const int2 at = PRE ? make_int2(e.slot, e.pos) : lm_where(p.rows, m);
        const int slot = at.x, pos = at.y;
        if (pos >= 0 && pos < p.rows.S) {
          lm_rotate2(v, p.rope, pos, p.rot_pairs, o >> 1);
          Tl<T>::st4((T*)p.kr_cache + (size_t)slot * p.d.s64 * p.d.rot32 + tl_off<T, 32>(pos, o, p.d.rot32), v);
        }
      } else {
        const int o = (nb - p.b_g) * 16 + 4 * kg;
        if (o < p.d.heads16)  // the blocks behind the gates only fill the last tile of the mixer part
          *reinterpret_cast<float4*>(p.gate + (size_t)m * p.d.heads16 + o) =
              make_float4(lm_sigmoid(v[0]), lm_sigmoid(v[1]), lm_sigmoid(v[2]), lm_sigmoid(v[3]));
      }
    }
    return;
  }
  if (EPI == LM_OUT) {
    float sq = 0.f;
    if (live) {
      float4* xp = reinterpret_cast<float4*>(p.x + (size_t)m * p.d.w64 + n);
      const float4 old = PRE ? e.a : *xp;
      v[0] += old.x; v[1] += old.y; v[2] += old.z; v[3] += old.w;
      *xp = make_float4(v[0], v[1], v[2], v[3]);
      Tl<T>::st4((T*)p.xt + tl_off<T>(m, n, p.d.w64), v);
      sq = (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
      if (p.layer_out)
        for (int r = 0; r < 4; ++r) if (n + r < p.width) p.layer_out[(size_t)m * p.width + n + r] = v[r];
    }
    sq = rows_sum(sq);  // the 16 columns of this row's block
    if (live && kg == 0 && nb < p.np) {
      const size_t at = (size_t)m * p.np + nb;
      if (half >= 0) p.ssq_out[2 * at + half] = sq;
      else if (p.M <= LM_PAIRS) reinterpret_cast<float2*>(p.ssq_out)[at] = make_float2(sq, 0.f);
      else p.ssq_out[at] = sq;
    }
    return;
  }
  if (LOGITS) {
    if (live)
      for (int r = 0; r < 4; ++r) if (n + r < p.vocab) p.logits[(size_t)m * p.ldo + n + r] = v[r];
    return;
  }
  if (EPI == LM_PROJ || EPI == LM_PLAIN || EPI == LM_MOE_DOWN) {
    const int r = EPI != LM_MOE_DOWN ? m : p.choice ? e.slot : p.ent[m];
    if (!live || r < 0) return;
    if (EPI != LM_MOE_DOWN && p.bias) {
      const float4 b = *reinterpret_cast<const float4*>(p.bias + n);
      v[0] += b.x; v[1] += b.y; v[2] += b.z; v[3] += b.w;
    }
    if (EPI == LM_PROJ) Tl<T>::st4((T*)p.out + (size_t)r * p.ldo + n, v);
    else Tl<float>::st4((float*)p.out + (size_t)r * p.ldo + n, v);
    return;
  }
  if (EPI == LM_ACT || EPI == LM_MOE_UP) {
    if (!live) return;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = lm_act(v[r], p.act_kind, p.act_pos, p.act_neg);
    Tl<T>::st4((T*)p.act + tl_off<T>(m, n, p.act_k), v);
    return;
  }
}

// i / n with inv = lm_inv(n); the product is right or one too large
static uint32_t lm_inv(uint32_t n) { return n > 1 ? 0xFFFFFFFFu / n + 1u : 0u; }
__device__ __forceinline__ uint32_t lm_div(uint32_t i, uint32_t n, uint32_t inv) {
  const uint32_t q = inv ? __umulhi(i, inv) : i;
  return q - (q * n > i ? 1u : 0u);
}

// Tile of a workgroup.  Workgroups go round the eight XCDs, whose L2s are their own, so each XCD takes a contiguous range of the tiles, in
// bands of `band` feature tiles with all row tiles: those that run side by side on an XCD share both operands.  In order of dispatch
// every XCD met nearly all of both, and that, not the steps of a tile, bound the narrow products (650 x 1024 x 4224 on 176 tiles: 22 us
// with or without a second half of waves; in bands 19).  Whole prompts, us before / after: sakupel 2048 wide x 200 positions 770 / 650,
// 650 1186 / 1040, 1500 2025 / 1857; mabidra 1024 wide x 900 1216 / 1142, 2048 wide x 1200 2551 / 2419.
// The divisions are products with what the host knows: by runtime values they took a launch of few tiles 0.2-0.3 us, and made some
// short prompts slower than in order of dispatch (mabidra 768 wide, interleaved, in order / divided / so: 64 positions 544 / 554 / 550 us, 80
// 557 / 557 / 551, 120 587 / 586 / 579; 768 features of 64 rows 7.1 -> 6.8 us per launch).
__device__ __forceinline__ void lm_tile_at(const LmGemm& p, int i, int MT, int NT, int& t, int& nt) {
  const int n = MT * NT, x = i & 7, at = x * (n >> 3) + min(x, n & 7) + (i >> 3);
  const int b = lm_div(at, p.band * MT, p.inv_tiles), r = at - b * p.band * MT, w = min(p.band, NT - b * p.band);
  t = lm_div(r, w, w == p.band ? p.inv_band : p.inv_last);
  nt = b * p.band + r - t * w;
}
static void lm_set_order(LmGemm& g, int MT, int NT, int band) {
  g.band = band;
  g.inv_tiles = lm_inv(band * MT); g.inv_band = lm_inv(band); g.inv_last = lm_inv(NT % band ? NT % band : band);
}

// The first fourteen words of a kernel's scalar arguments are in registers when it starts, a struct is a trip to memory (0.2-0.35 us of a
// launch of 4-8): what the first loads need comes twice, ahead of the struct and in it.  aux0, aux1: of experts' products the choices, or
// the number of tiles and their experts, otherwise the sums of squares and the norm; np_band: of the same the entries' tiles.  The few bits
// of features and K (below LM_SIZES) keep the arithmetic of addresses short, too: with every size that an int holds 10-25 scalar instructions
// more, 8 steps of 36 launches 1306 -> 1313 us.
#define LM_SIZES (1 << 21)
#define LM_HOT const void *X, const void *W, const void *aux0, const void *aux1, int M, uint32_t nk, uint32_t np_band, uint32_t inv_tiles, uint32_t inv_band, uint32_t inv_last
#define LM_HOT_ARGS(g, moe)                                                                                                                 \
  g.X, g.W, (moe) ? (const void*)(g.choice ? g.choice : g.n_tiles) : (const void*)g.ssq, (moe) ? (const void*)g.tile_e : (const void*)g.norm, g.M,                   \
      (uint32_t)(g.N >> 4 | g.K >> 6 << 17), (uint32_t)((moe) ? g.max_tiles : g.np | g.band << 16), (uint32_t)((moe) ? (g.choice ? g.M * g.top : 0) : g.inv_tiles), g.inv_band, g.inv_last
#define LM_HOT_IN(p, moe)                                                                                    \
  p.X = X; p.W = W; p.M = M; p.N = (int)(nk & 0x1ffffu) * 16; p.K = (int)(nk >> 17) * 64;                    \
  p.inv_tiles = inv_tiles; p.inv_band = inv_band; p.inv_last = inv_last;                                     \
  if (moe) {                                                                                                 \
    p.choice = inv_tiles ? (const int32_t*)aux0 : nullptr; p.n_tiles = (const int32_t*)aux0; p.tile_e = (const int32_t*)aux1; \
    p.max_tiles = (int)np_band;                                                                              \
  }                                                                                                          \
  else { p.ssq = (const float*)aux0; p.norm = (const float*)aux1; p.np = (int)(np_band & 0xffffu); p.band = (int)(np_band >> 16); }

// sum within aligned groups of N lanes, in every lane, without LDS
template <int N>
__device__ __forceinline__ float lanes_sum(float v) {
  if (N >= 2) v += dpp_f<DPP_QUAD_XOR1>(v);
  if (N >= 4) v += dpp_f<DPP_QUAD_XOR2>(v);
  if (N >= 8) v += dpp_f<DPP_ROW_HALF_MIRROR>(v);
  if (N >= 16) v += dpp_f<DPP_ROW_MIRROR>(v);
  if (N >= 32) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  }
  if (N >= 64) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  }
  return v;
}

// a lane of 16 receives what the lane 16 - N above it (around the 16) holds
template <int N>
__device__ __forceinline__ uint4 row_ror(const uint4& v) {
  return make_uint4(dpp_i<0x120 + N>((int)v.x), dpp_i<0x120 + N>((int)v.y), dpp_i<0x120 + N>((int)v.z), dpp_i<0x120 + N>((int)v.w));
}

// n and the bits of a mask below this lane
__device__ __forceinline__ int lane_count(uint32_t lo, uint32_t hi, int n) { return __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, n)); }

// ALT, of LM_PLAIN and LM_OUT: HALF, a workgroup takes eight of a block's 16 features (few rows and few features, see pick); of experts'
// products: BITS, another way to the tile's entries (see experts).
// A CU's address unit takes a wave's load of 16 bytes per lane in 16 clocks whatever it fetches, and products of few rows wait for that: 176 such loads, 1.3 us,
// for 16 features of K 2816, half of them for the rows' operands.  So (bf16) half a block's weights fill the lanes of one load per step: lanes 8-15 of a
// group of 16 hold the second piece of the features of lanes 0-7, the matrix instruction meets them with both pieces of X, and
// either sum is right for half of its features.  FEW, of up to four rows: one load holds four steps of X, those of the later
// ones in the lanes of rows that there are not, and a rotation by lanes brings them to their place.  A step of the 768 wide model with one row, us: re-reading
// a wave's last step where it has no more 152, not so 140, all waves' parts read before the first is added 138, PACK and FEW 134; 16 rows
// of 1024 wide 225, 214, 212, 207; four rows of 2048 wide with experts 462, 441, 437, 431.
template <typename T, int MB, int NB, int WAVES, int EPI, bool ALT, bool FEW>
__global__ __launch_bounds__(64 * WAVES, sizeof(T) == 2 && MB == 1 && NB < 3 ? 4 : 1) void lm_gemm_kernel(LM_HOT, const LmGemm p0) {
  LmGemm p = p0;
  LM_HOT_IN(p, EPI == LM_MOE_UP || EPI == LM_MOE_DOWN);
  constexpr bool SCALED = EPI == LM_IN_ATTN || EPI == LM_IN_GRU_STEP || EPI == LM_IN_GRU_SEQ || EPI == LM_LOGITS;
  constexpr bool GRU = EPI == LM_IN_GRU_STEP || EPI == LM_IN_GRU_SEQ;
  constexpr bool LOGITS = EPI == LM_LOGITS || EPI == LM_HEAD, MOE = EPI == LM_MOE_UP || EPI == LM_MOE_DOWN;
  constexpr bool HALF = ALT && (EPI == LM_PLAIN || EPI == LM_OUT), BITS = ALT && MOE, PACK = HALF && sizeof(T) == 2;
  static_assert(ALT == (HALF || BITS) && (!HALF || NB == 1) && (!ALT || MB == 1), "half blocks are for features that are each by themselves");
  static_assert(!FEW || (MB == 1 && WAVES >= 8 && sizeof(T) == 2 && !MOE), "four rows of bf16");
  constexpr int EP = Tl<T>::EP, P = 16 / EP, TILE = MB * NB * 256;
  __shared__ __align__(16) float part[WAVES * TILE];
  __shared__ float srow[MB * 16];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l16 = lane & 15, kg = lane >> 4;
  const int MT = MOE ? p.max_tiles : MB == 1 ? 1 : (p.M + 16 * MB - 1) / (16 * MB);  // one block of rows: 16 at most
  // tiles of an expert that share features run on one XCD, whose cache then holds those weights: workgroup i is on XCD i % 8
  int t, nt;
  if (MOE) {
    t = ((int)blockIdx.x >> 3) % MT; nt = ((int)blockIdx.x >> 3) / MT * 8 + ((int)blockIdx.x & 7);
  } else if (MB == 1) {
    t = 0; nt = HALF ? (int)blockIdx.x >> 1 : (int)blockIdx.x;
  } else {
    lm_tile_at(p, blockIdx.x, MT, ((p.N >> 4) + NB - 1) / NB, t, nt);
  }
  const int half8 = HALF ? 8 * ((int)blockIdx.x & 1) : 0;
  const int m0 = t * 16 * MB, nb0 = nt * NB;
  size_t wz = 0;
  int entry = -1;  // of the tile's row l16, where the tile is found in the choices
  if (MOE && MB == 1 && p.choice) {
    // Experts in the order of their first entry, each with as many tiles of 16 entries as it needs; entries are lanes
    if (nb0 >= (p.N >> 4)) return;  // uniform, as what follows
    const int n = (int)inv_tiles, e = lane < n ? p.choice[lane] : -1;
    const uint64_t all = ~0ull >> (64 - n);
    uint64_t mine = 0;
    int expert = -1, sub = t;  // its tile
    if (!BITS) {  // from expert to expert up to the tile's own
      uint64_t left = all;
      while (left) {
        const int c = __builtin_amdgcn_readlane(e, __builtin_ctzll(left));
        const uint64_t same = __builtin_amdgcn_ballot_w64(e == c);
        const int tiles = (__popcll(same) + 15) >> 4;
        if (sub < tiles) { expert = c; mine = same; break; }
        sub -= tiles;
        left &= ~same;
      }
    } else {  // every lane finds the entries of its expert by the bits of its number (up to 128 experts, see lm_rows_routes)
      uint32_t lo = (uint32_t)all, hi = (uint32_t)(all >> 32);
#pragma unroll
      for (int b = 0; b < 7; ++b) {
        const uint64_t set = __builtin_amdgcn_ballot_w64(e >> b & 1);
        const uint32_t flip = (uint32_t)(e >> b & 1) - 1;
        lo &= (uint32_t)set ^ flip; hi &= (uint32_t)(set >> 32) ^ flip;
      }
      const bool leads = lane < n && lane_count(lo, hi, 0) == 0;
      const int tiles = leads ? (__popc(lo) + __popc(hi) + 15) >> 4 : 0;
      int first = 0;  // tiles of the experts before
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint64_t more = __builtin_amdgcn_ballot_w64(tiles > k);
        first = lane_count((uint32_t)more, (uint32_t)(more >> 32), first);
      }
      const uint64_t who = __builtin_amdgcn_ballot_w64((uint32_t)(t - first) < (uint32_t)tiles);
      if (who) {
        const int lead = __builtin_ctzll(who);
        expert = __builtin_amdgcn_readlane(e, lead); sub = t - __builtin_amdgcn_readlane(first, lead);
        mine = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)hi, lead) << 32 | (uint32_t)__builtin_amdgcn_readlane((int)lo, lead);
      }
    }
    if (expert < 0) return;
    wz = (size_t)expert * p.wz;
    const int at = lane_count((uint32_t)mine, (uint32_t)(mine >> 32), 0);
    const bool in = (mine >> lane & 1) && at >> 4 == sub;
    const int got = __builtin_amdgcn_ds_permute((in ? at & 15 : 63) * 4, lane + 1);  // lanes 0 ... 15: their entry + 1, or 0
    entry = __builtin_amdgcn_ds_bpermute(l16 * 4, got) - 1;
  } else if (MOE) {
    if (t >= p.n_tiles[0] || nb0 >= (p.N >> 4)) return;  // uniform
    wz = (size_t)p.tile_e[t] * p.wz;
  }
  const int nsteps = p.K >> 6;
  const int s0 = nsteps * wave / WAVES, s1 = nsteps * (wave + 1) / WAVES;
  const int MBL = (p.M + 15) >> 4, NBL = p.N >> 4;

  const T* xr[MB];
  const T* wr[NB];
#pragma unroll
  for (int j = 0; j < MB; ++j) {
    if (EPI == LM_MOE_UP && !p.sorted) {
      const int e = MB == 1 && p.choice ? entry : p.ent[m0 + 16 * j + l16], r = min(max(e, 0) / p.top, p.x_rows - 1);
      xr[j] = (const T*)p.X + (size_t)(r >> 4) * nsteps * 1024 + ((r & 15) + 16 * kg) * EP;
    } else if (MOE) {
      xr[j] = (const T*)p.X + (size_t)((m0 >> 4) + j) * nsteps * 1024 + lane * EP;
    } else if (LOGITS && p.rowmap) {
      const int r = min(max(p.rowmap[min(m0 + 16 * j + (FEW ? l16 & 3 : l16), p.M - 1)], 0), p.x_rows - 1);
      xr[j] = (const T*)p.X + (size_t)(r >> 4) * nsteps * 1024 + ((r & 15) + 16 * kg) * EP;
    } else {
      // few rows: lanes without a row re-read the last one instead of fetching a block that is mostly padding
      const int l = MB == 1 ? min(FEW ? l16 & 3 : l16, p.M - 1 - m0) + 16 * kg : lane;
      xr[j] = (const T*)p.X + (size_t)min((m0 >> 4) + j, MBL - 1) * nsteps * 1024 + l * EP;
    }
  }
#pragma unroll
  for (int i = 0; i < NB; ++i)
    wr[i] = (const T*)p.W + wz + (size_t)min(nb0 + i, NBL - 1) * nsteps * 1024 + (HALF ? (lane & 0x37) + half8 : lane) * EP + (PACK ? (l16 >> 3) * 512 : 0);

  // U steps' loads go out together, as far as the wave has steps (re-reading the last one instead was most of what launches of small K waited for);
  // the first ones now
  constexpr bool EARLY = WAVES >= 8 && sizeof(T) == 2;
  constexpr int U = !EARLY ? 1 : MB == 1 ? 4 : 2;
  static_assert(!FEW || U == 4, "a row's four steps lie in its lanes' places");
  constexpr int PW = PACK ? 1 : P, UX = FEW ? 1 : U;
  uint4 xa[UX][MB][P], wa[U][NB][PW];
  auto load = [&](int s) {
    if (FEW) {
      const size_t o = (size_t)min(s + (l16 >> 2), s1 - 1) * 1024;
#pragma unroll
      for (int h = 0; h < P; ++h) xa[0][0][h] = *reinterpret_cast<const uint4*>(xr[0] + o + 64 * EP * h);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u > 0 && s + u >= s1) break;  // uniform
      const size_t o = (size_t)(s + u) * 1024;
#pragma unroll
      for (int h = 0; h < P; ++h) {
#pragma unroll
        for (int i = 0; i < NB; ++i)
          if (h < PW) wa[u][i][h] = *reinterpret_cast<const uint4*>(wr[i] + o + 64 * EP * h);
        if (!FEW) {
#pragma unroll
          for (int j = 0; j < MB; ++j) xa[u % UX][j][h] = *reinterpret_cast<const uint4*>(xr[j] + o + 64 * EP * h);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // What the scale and the epilogue of this wave's first unit will need is requested now as well:
  // fetched where it is used, it would be a chain of dependent loads behind the last product.
  // Scale: TPR neighbouring threads add up one row's sums of squares, in a fixed order, while the operands are on their way.
  constexpr int TPR = WAVES * 64 / (MB * 16) > 64 ? 64 : WAVES * 64 / (MB * 16), NSQ = 4;
  const int sq_r = tid / TPR, sq_q = tid % TPR;
  int sq_m = 0;
  float2 sq[NSQ];
  float norm = 0.f;
  const bool pairs = LOGITS ? p.x_rows <= LM_PAIRS : MB == 1;  // of a block's columns there are two sums
  auto sq_at = [&](int i) {
    const size_t at = (size_t)sq_m * p.np + i;
    return pairs ? reinterpret_cast<const float2*>(p.ssq)[at] : make_float2(p.ssq[at], 0.f);
  };
  if (SCALED) {
    sq_m = min(m0 + min(sq_r, MB * 16 - 1), p.M - 1);
    if (LOGITS && p.rowmap) sq_m = min(max(p.rowmap[sq_m], 0), p.x_rows - 1);
#pragma unroll
    for (int i = 0; i < NSQ; ++i) sq[i] = sq_at(min(sq_q + TPR * i, p.np - 1));
    norm = p.norm[0];
  }
  if (EARLY && s0 < s1) load(s0);
  constexpr bool PRE = MB == 1 && (EPI == LM_IN_ATTN || EPI == LM_IN_GRU_STEP || EPI == LM_OUT);
  const int pm = min(m0 + l16, p.M - 1), pb = min(nb0 + min(wave, NB - 1), NBL - 1);  // row and block of unit `wave`
  LmPre e;
  e.slot = entry; e.pos = 0;
  e.a = e.b = e.c = make_float4(0.f, 0.f, 0.f, 0.f);
  if (PRE && EPI != LM_OUT) {
    const int2 at = lm_where(p.rows, pm);
    e.slot = at.x; e.pos = at.y;
  }
  if (PRE && EPI == LM_OUT) e.a = *reinterpret_cast<const float4*>(p.x + (size_t)pm * p.d.w64 + pb * 16 + (HALF ? half8 + 4 * (kg & 1) : 4 * kg));
  if (PRE && EPI == LM_IN_GRU_STEP && nb0 < p.mix_blocks) {
    const int ch = (nb0 / 3) * 16 + 4 * kg;
    e.a = *reinterpret_cast<const float4*>(p.state + (size_t)e.slot * p.d.gru16 + ch);
    e.b = *reinterpret_cast<const float4*>(p.bz + ch);
    e.c = *reinterpret_cast<const float4*>(p.bx + ch);
  }

  if (SCALED) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < NSQ; ++i) t += sq_q + TPR * i < p.np ? sq[i].x + sq[i].y : 0.f;
    for (int i = sq_q + TPR * NSQ; i < p.np; i += TPR) {
      const float2 v = sq_at(i);
      t += v.x + v.y;
    }
    t = lanes_sum<TPR>(t);
    if (sq_r < MB * 16 && sq_q == 0) srow[sq_r] = norm / sqrtf(t / (float)p.width + p.eps);
  }

  tl_f32x4 acc[NB][MB], odd = {0.f, 0.f, 0.f, 0.f};  // odd: of PACK, the sums with the second pieces of X
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j) acc[i][j] = tl_f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s = s0; s < s1; s += U) {
    if (!EARLY || s > s0) load(s);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (s + u >= s1) break;  // uniform
#pragma unroll
      for (int h = 0; h < P; ++h) {
        uint4 x[MB];
#pragma unroll
        for (int j = 0; j < MB; ++j) x[j] = FEW ? (u == 0 ? xa[0][0][h] : u == 1 ? row_ror<12>(xa[0][0][h]) : u == 2 ? row_ror<8>(xa[0][0][h]) : row_ror<4>(xa[0][0][h])) : xa[u % UX][j][h];
        if (PACK && h == 1) {
          odd = Tl<T>::mma(wa[u][0][0], x[0], odd);
          continue;
        }
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int j = 0; j < MB; ++j)
            acc[i][j] = Tl<T>::mma(wa[u][i][h % PW], x[j], acc[i][j]);
      }
    }
  }
  if (PACK) {  // features 0-7 with the first pieces (lanes of kg 0, 1) and with the second (kg 2, 3)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t v = __float_as_uint(kg < 2 ? acc[0][0][r] : odd[r]);
      const auto a = __builtin_amdgcn_permlane32_swap(v, v, false, false);
      acc[0][0][r] = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    }
  }
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j)
      *reinterpret_cast<tl_f32x4*>(&part[wave * TILE + ((i * MB + j) * 64 + lane) * 4]) = acc[i][j];
  __syncthreads();

  const bool mix = GRU && nb0 < p.mix_blocks;  // uniform: a tile is all mixer or all feed-forward (padded that way)
  const int units = mix ? MB : MB * NB;
  for (int u = wave; u < units; u += WAVES) {
    const int j = mix ? u : u % MB, i0 = mix ? 0 : u / MB;
    const int m = m0 + 16 * j + l16;
    const int nb = nb0 + i0;
    const int n = nb * 16 + (HALF ? half8 + 4 * (kg & 1) : 4 * kg);
    const bool live = (MOE || m < p.M) && nb < NBL && !(HALF && kg > 1);
    const float sc = SCALED ? srow[16 * j + l16] : 1.f;
    float v[4];
    // all waves' parts are read before the first is added: left to the compiler two reads were in flight at a time, 0.5 us for sixteen parts
    tl_f32x4 pt[WAVES];
    auto parts = [&](int i) {
      const float* q = part + ((i * MB + j) * 64 + lane) * 4;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) pt[w] = *reinterpret_cast<const tl_f32x4*>(q + w * TILE);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto gather = [&](int i, float* o) {
      parts(i);
      tl_f32x4 a = pt[0];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) a += pt[w];
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = a[r] * sc;
    };
    gather(i0, v);

    float xv[4] = {0.f, 0.f, 0.f, 0.f}, gv[4] = {0.f, 0.f, 0.f, 0.f};
    if (GRU && mix) {
      gather(NB > 1 ? 1 : 0, xv);
      gather(NB > 2 ? 2 : 0, gv);
    }
    lm_unit<T, EPI, PRE>(p, m, nb, n, l16, kg, live, mix, v, xv, gv, e, HALF ? half8 >> 3 : -1);
  }
  if (LOGITS && p.upd_lens && blockIdx.x == 0) {
    if (p.upd_inc) {
      for (int s = tid; s < p.rows.n_slots; s += 64 * WAVES) p.upd_lens[s] += p.upd_inc[s];
    } else {
      for (int b = tid; b < p.upd_rows; b += 64 * WAVES) atomicAdd(&p.upd_lens[lm_where(p.rows, b).x], 1);
    }
  }
}

// ---- many rows, bf16: large tiles through LDS (wide.h) ----
// G = 2: eight waves, each half of them with half of K and stages of its own, for tiles that are alone on their CU: a step of
// such a tile is a chain of barrier, LDS reads and products, and two chains side by side take little longer than one.
template <int EPI, int MBW, int NBW, int WM, int WN, int S, int KS, int G>
__global__ __launch_bounds__(256 * G, 2) void lm_wide_kernel(LM_HOT, const LmGemm p0) {
  LmGemm p = p0;
  LM_HOT_IN(p, EPI == LM_MOE_UP || EPI == LM_MOE_DOWN);
  constexpr bool SCALED = EPI == LM_IN_ATTN || EPI == LM_IN_GRU_SEQ;
  constexpr bool GRU = EPI == LM_IN_GRU_SEQ, MOE = EPI == LM_MOE_UP || EPI == LM_MOE_DOWN;
  typedef WideTile<MBW, NBW, WM, WN, S, KS> Tile;
  constexpr int MB = Tile::MB, NB = Tile::NB;
  static_assert(!GRU || NBW % 3 == 0, "a recurrence's blocks come in threes");
  __shared__ __align__(16) char lds[Tile::LDS * G];
  __shared__ float srow[MB * 16];
  const int tid = threadIdx.x, wave8 = __builtin_amdgcn_readfirstlane(tid >> 6), half = G == 2 ? wave8 >> 2 : 0, wave = wave8 & 3;
  const int lane = tid & 63, l16 = lane & 15, kg = lane >> 4, wm = wave % WM, wn = wave / WM;
  const bool val = EPI == LM_EXPAND && (int)blockIdx.z >= p.heads;  // values of a head behind the keys of all
  const int head = (int)blockIdx.z - (val ? p.heads : 0);
  const int MBL = (p.M + 15) >> 4, NBL = (val ? p.n_v : p.N) >> 4, MT = MOE ? p.max_tiles : (MBL + MB - 1) / MB, NT = (NBL + NB - 1) / NB;
  int t, nt;
  if (MOE) {
    // Tiles of one expert that share features run on one XCD (workgroup i is on XCD i % 8), which reads those weights from
    // HBM once; which feature tiles are an XCD's turns with the expert, so that NT need not be a multiple of 8.
    // (With an expert's tiles on whatever XCD they fell the up product of 2600 entries, 32 experts of 1024 x 1056, took 34.4 us
    // instead of 32.4.)
    const int per = (NT + 7) >> 3, slice = (int)blockIdx.x >> 3;
    t = slice / per;
    if (t >= p.n_tiles[0]) return;  // uniform
    nt = (((int)blockIdx.x - p.tile_e[t]) & 7) + 8 * (slice % per);
    if (nt >= NT) return;
  } else if (EPI == LM_EXPAND) {
    t = (int)blockIdx.x % MT; nt = (int)blockIdx.x / MT;
    if (nt >= NT) return;
  } else if (MB == 8 && p.band == 0) {  // every eighth feature tile with all rows
    const int slice = (int)blockIdx.x >> 3;
    t = slice % MT; nt = slice / MT * 8 + ((int)blockIdx.x & 7);
    if (nt >= NT) return;
  } else {
    lm_tile_at(p, blockIdx.x, MT, NT, t, nt);
  }
  const int mb0 = t * MB, nb0 = nt * NB, m0 = mb0 * 16;
  const int Q = p.K / (32 * KS);  // steps
  const size_t wz = MOE ? (size_t)p.tile_e[t] * p.wz : head * (val ? p.wz_v : p.wz);
  const char* weights = (const char*)(val ? p.w_v : p.W);

  const int n64 = p.K >> 6, mid = G == 2 ? (n64 >> 1) * 2 / KS : 0, first = half * mid, mine = G == 1 ? Q : half ? Q - mid : mid;
  Tile tile;
  tile.begin(lds + half * Tile::LDS, wave, lane,
             [&](int i) { return (const char*)p.X + ((size_t)(MOE ? mb0 + i : min(mb0 + i, MBL - 1)) * Q + first) * (KS * 1024); },
             [&](int i) { return weights + wz * 2 + ((size_t)min(nb0 + i, NBL - 1) * Q + first) * (KS * 1024); });
  tile.prologue(mine);

  if (SCALED && half == 0) {
    // 16 lanes add up one row's sums of squares, in a fixed order, the loads of all the wave's rows side by side (one
    // after the other they took longer than the products: 98 against 61 us at 1024 x 11776 x 2048)
    constexpr int NR = MB;  // rows per 16 lanes: 16 MB rows over 16 groups
    const int grp = wave * 4 + kg;
    float a[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) a[i] = 0.f;
    if ((p.np & 3) == 0) {
      for (int c = 4 * l16; c < p.np; c += 64) {
        float4 v[NR];
#pragma unroll
        for (int i = 0; i < NR; ++i) v[i] = *reinterpret_cast<const float4*>(p.ssq + (size_t)min(m0 + grp * NR + i, p.M - 1) * p.np + c);
#pragma unroll
        for (int i = 0; i < NR; ++i) a[i] += (v[i].x + v[i].y) + (v[i].z + v[i].w);
      }
    } else {
      for (int c = l16; c < p.np; c += 16) {
        float v[NR];
#pragma unroll
        for (int i = 0; i < NR; ++i) v[i] = p.ssq[(size_t)min(m0 + grp * NR + i, p.M - 1) * p.np + c];
#pragma unroll
        for (int i = 0; i < NR; ++i) a[i] += v[i];
      }
    }
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const float t = group16_sum(a[i]);
      if (l16 == 0) srow[grp * NR + i] = p.norm[0] / sqrtf(t / (float)p.width + p.eps);
    }
  }

  tl_f32x4 acc[NBW][MBW];
  if constexpr (G == 1) {
    tile.run(Q, acc);
  } else {  // the quarters are added in the same order
    static_assert(8 * NBW * MBW * 1024 <= Tile::LDS, "the other half's sums fit its stages");
    tl_f32x4 last[NBW][MBW];
    tile.steps(first, mine, Q - mid, n64, 1 + 2 * half, acc, last);
    __syncthreads();
    char* other = lds + Tile::LDS + wave * 2 * NBW * MBW * 1024 + lane * 16;
#pragma unroll
    for (int i = 0; i < NBW; ++i)
#pragma unroll
      for (int j = 0; j < MBW; ++j) {
        if (half) {
          *reinterpret_cast<tl_f32x4*>(other + (i * MBW + j) * 1024) = acc[i][j];
          *reinterpret_cast<tl_f32x4*>(other + (NBW * MBW + i * MBW + j) * 1024) = last[i][j];
        } else {
          acc[i][j] += last[i][j];
        }
      }
    __syncthreads();
    if (half) return;
#pragma unroll
    for (int i = 0; i < NBW; ++i)
#pragma unroll
      for (int j = 0; j < MBW; ++j) {
        acc[i][j] += *reinterpret_cast<const tl_f32x4*>(other + (i * MBW + j) * 1024);
        acc[i][j] += *reinterpret_cast<const tl_f32x4*>(other + (NBW * MBW + i * MBW + j) * 1024);
      }
  }
  // The sums pass through this wave's share of LDS, so that the epilogue is a loop: unrolled over the units it is 100 KB of
  // instructions, and fetching those took longer than the products (98 against 61 us at 1024 x 11776 x 2048).
  constexpr int ROOM = S * Tile::PIECES / 4, CH0 = ROOM / MBW < NBW ? ROOM / MBW : NBW, CH = GRU ? CH0 / 3 * 3 : CH0;  // blocks at a time
  static_assert(CH > 0, "a block of sums fits the wave's share");
  if (G == 1) __syncthreads();
  char* own = lds + wave * ROOM * 1024 + lane * 16;
#pragma unroll
  for (int c = 0; c < NBW; c += CH) {
#pragma unroll
    for (int i = c; i < c + CH && i < NBW; ++i)
#pragma unroll
      for (int j = 0; j < MBW; ++j) *reinterpret_cast<tl_f32x4*>(own + ((i - c) * MBW + j) * 1024) = acc[i][j];
    const int n_blocks = min(CH, NBW - c);
#pragma unroll 1
    for (int i = 0; i < n_blocks; ++i) {  // the MBW units of a block side by side: their loads and exponentials overlap
      const int nb = nb0 + wn * NBW + c + i, n = nb * 16 + 4 * kg;
      const bool mix = GRU && nb - i % 3 < p.mix_blocks;  // uniform
      if (nb >= NBL || (mix && i % 3)) continue;
      auto sums = [&](int blk, int j, float* o) {
        const tl_f32x4 a = *reinterpret_cast<const tl_f32x4*>(own + (blk * MBW + j) * 1024);
        const float sc = SCALED ? srow[(wm * MBW + j) * 16 + l16] : 1.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = a[r] * sc;
      };
      const int mw = m0 + wm * MBW * 16 + l16;
      if (EPI == LM_EXPAND) {
#pragma unroll
        for (int j = 0; j < MBW; ++j) {
          float v[4];
          if (val) {
            // Blocks of 16 value dims x 32 keys: a lane of the attention kernel reads the keys 4 kg .. + 3 of both halves.  The
            // unit is read from LDS the other way round, four rows of a feature.
            const float* q = reinterpret_cast<const float*>(own - lane * 16 + (i * MBW + j) * 1024) + 4 * (4 * kg + 16 * (l16 >> 2)) + (l16 & 3);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = q[4 * r];
            const int m = m0 + (wm * MBW + j) * 16 + 4 * kg;
            if (m < p.M)
              Tl<bf16_t>::st4((bf16_t*)p.v_out + head * p.v_z + ((size_t)nb * (p.d.s64 >> 5) + (m >> 5)) * 512 +
                              (l16 + 16 * ((m & 15) >> 2)) * 8 + 4 * ((m & 31) >> 4), v);
          } else {
            sums(i, j, v);
            if (mw + 16 * j < p.M) Tl<bf16_t>::st4((bf16_t*)p.kv_out + head * p.kv_z + tl_off<bf16_t>(mw + 16 * j, n, p.d.dim64), v);
          }
        }
        continue;
      }
      if ((EPI == LM_IN_ATTN || GRU) && nb >= p.mix_blocks) {  // (gate, up) pairs
        const int f = p.d.ff_off + ((n - p.mix_blocks * 16) >> 1);
#pragma unroll
        for (int j = 0; j < MBW; ++j) {
          float v[4];
          sums(i, j, v);
          if (mw + 16 * j < p.M)
            Tl<bf16_t>::st2((bf16_t*)p.act + tl_off<bf16_t>(mw + 16 * j, f, p.d.out_k), lm_ff(v[0], v[1], p.limit), lm_ff(v[2], v[3], p.limit));
        }
        continue;
      }
      LmPre e[MBW];
#pragma unroll
      for (int j = 0; j < MBW; ++j)
        if (EPI == LM_OUT) e[j].a = *reinterpret_cast<const float4*>(p.x + (size_t)min(mw + 16 * j, p.M - 1) * p.d.w64 + n);
#pragma unroll
      for (int j = 0; j < MBW; ++j) {
        float v[4], xv[4] = {0.f, 0.f, 0.f, 0.f}, gv[4] = {0.f, 0.f, 0.f, 0.f};
        sums(i, j, v);
        if (GRU && mix) { sums(i + 1, j, xv); sums(i + 2, j, gv); }
        lm_unit<bf16_t, EPI, EPI == LM_OUT>(p, mw + 16 * j, nb, n, l16, kg, MOE || mw + 16 * j < p.M, mix, v, xv, gv, e[j]);
      }
    }
  }
}

// Feature tiles from which an XCD takes every eighth of them with all rows, if a tile has 128 rows (with fewer, whole XCDs would have
// nothing or twice as much to do; tiles of 64 rows read their operands twice as often, and there what counts is how little the
// tiles side by side read together).  us, so / in bands: 1999 x 14400 x 2048 (128 x 192) 155 / 165, 1999 x 7744 x 1024 (128 x 128)
// 55 / 64; 1500 x 2048 x 6144 (64 x 64) 89 / 76.
#define WIDE_STRIDED 24
// Feature tiles of a band: the tiles that an XCD runs side by side (two per CU, or its share) as near to a square of the operands as
// they come.
static int lm_band(int MT, int NT, int bm, int bn) {
  const long side = std::min(64L, ((long)MT * NT + 7) / 8);
  int w = 1;
  while (w < NT && (long)w * w * bn < side * bm) ++w;
  return std::max(w, (int)std::min((long)NT, side / MT));  // few rows: all of them side by side
}
template <int EPI, int MBW, int NBW, int WM, int WN, int S, int KS, int G = 1>
static int go_wide(LmGemm g, hipStream_t st) {
  const int MT = (g.M + 16 * MBW * WM - 1) / (16 * MBW * WM), NT = ((EPI == LM_EXPAND && g.n_v > g.N ? g.n_v : g.N) / 16 + NBW * WN - 1) / (NBW * WN);
  const bool moe = EPI == LM_MOE_UP || EPI == LM_MOE_DOWN;
  const bool strided = MBW * WM == 8 && EPI != LM_EXPAND && NT >= WIDE_STRIDED;
  if (strided) g.band = 0;
  else lm_set_order(g, MT, NT, lm_band(MT, NT, MBW * WM, NBW * WN));
  const int tiles = moe ? g.max_tiles * ((NT + 7) & ~7) : MT * (strided ? (NT + 7) & ~7 : NT);
  const int heads = EPI == LM_EXPAND ? 2 * g.heads : 1;  // keys of every head, values of every head
  hipLaunchKernelGGL((lm_wide_kernel<EPI, MBW, NBW, WM, WN, S, KS, G>), dim3((unsigned)tiles, 1, heads), dim3(256 * G), 0, st, LM_HOT_ARGS(g, moe), g);
  HIP_TRY(hipGetLastError());
  return VUI_OK;
}

template <typename T, int MB, int NB, int WAVES, int EPI, bool ALT = false, bool FEW = false>
static int go(LmGemm g, hipStream_t st) {
  if constexpr (sizeof(T) == 2 && MB == 1 && !FEW && EPI != LM_MOE_UP && EPI != LM_MOE_DOWN)
    if (g.M <= 4) return go<T, MB, NB, WAVES, EPI, ALT, true>(g, st);
  const bool moe = EPI == LM_MOE_UP || EPI == LM_MOE_DOWN;
  const int nt = (g.N / 16 + NB - 1) / NB;
  const int mt = (g.M + 16 * MB - 1) / (16 * MB);
  lm_set_order(g, mt, nt, lm_band(mt, nt, MB, NB));
  const int tiles = moe ? g.max_tiles * ((nt + 7) & ~7) : mt * nt * (ALT ? 2 : 1);
  hipLaunchKernelGGL((lm_gemm_kernel<T, MB, NB, WAVES, EPI, ALT, FEW>), dim3((unsigned)tiles), dim3(64 * WAVES), 0, st, LM_HOT_ARGS(g, moe), g);
  HIP_TRY(hipGetLastError());
  return VUI_OK;
}

// Tile of a prompt's product (wide_pick).  The K-splitting kernel is counted 1.5 times: 28.4 against 23 us at 650 x 1024 x 4608
// with 18.4 estimated.  Whole prompts with 0.85 / 1.2 / 1.5 / 2 of the estimate, us: latent models of 2048 x 400 positions
// 1033 / 869 / 865 / 870 and of 1024 x 900 760 / 701 / 691 / 697, x 500 487 / 487 / 497 / 553; experts of 2048 x 300
// 1463 / 1404 / 1311 / 1320.
static int lm_tile(int epi, int M, int N, int K) {
  if (epi != LM_IN_GRU_SEQ) {
    // Tiles that are alone on their CU split K over two halves of waves.  Whole prompts, us, without / with (the same order of tiles):
    // sakupel 1024 wide x 900 positions 722 / 690, 2048 wide x 333 833 / 805; mabidra 2048 wide x 333 1371 / 1340.
    const int t = wide_pick(M, N, K, 1.5);
    const long MT = (M + 63) / 64;
    if (t == WIDE_64 && K >= 512 && MT * ((N + 63) / 64) <= 256) return WIDE_64_2;
    if (t == WIDE_64x128 && K >= 512 && MT * ((N + 127) / 128) <= 256) return WIDE_64x128_2;
    return t;
  }
  // A minGRU projection takes 128 x 192, whose tiles fill an XCD 64 at a time, or the K-splitting form, which is bound by the
  // weights' way to the chip and by its tiles.  us, K-splitting / large tile (50 products of 130 ... 2048
  // rows, the quicker form is taken in 49): 900 x 6400 x 768 27.6 / 30.0, 1200 32.1 / 31.1, 1600 39.7 / 46.5; 640 x 8704 x 1024 33.1 / 31.9; 300 x 11776 x 1024
  // 33.7 / 31.4, 1200 79 / 64; 130 x 14336 x 2048 51 / 44, 1024 154 / 93.
  if (M < 128) return WIDE_NONE;
  const long MT = (M + 127) / 128, NT = (N + 191) / 192;
  const long fills = NT >= WIDE_STRIDED ? ((NT + 7) / 8 * MT + 63) / 64 : (NT * MT + 511) / 512;
  const double split = 4 + 1e-6 * N * K + 0.26e-3 * ((M + 31) / 32) * ((N + 31) / 32) * (K / 64);
  return 6 + fills * (10 + 0.56 * (K / 32)) < split ? WIDE_128 : WIDE_NONE;
}
template <int EPI>
static int pick_wide(int tile, const LmGemm& g, hipStream_t st) {
  if constexpr (EPI != LM_EXPAND) {
    if (tile == WIDE_64x128_2) return go_wide<EPI, 4, 2, 1, 4, 3, 2, 2>(g, st);
    if (tile == WIDE_64_2) return go_wide<EPI, 2, 2, 2, 2, 4, 2, 2>(g, st);
  }
  switch (tile) {
    case WIDE_128: return go_wide<EPI, 4, 4, 2, 2, 4, 1>(g, st);
    case WIDE_64x128: return go_wide<EPI, 4, 2, 1, 4, 3, 2>(g, st);
    default: return go_wide<EPI, 2, 2, 2, 2, 4, 2>(g, st);
  }
}

// More rows, as long as no large tile is quicker.  Few tiles are a wave's chain of trips to memory, not its width: with one tile per CU at
// most eight waves split K and request two steps at a time, and where half the CUs would have none a tile is 16 features wide.  us per
// launch, four waves on 32 x 32 / eight / eight on 32 x 16: 50 x 2048 x 6144 18.2 / 15.5 / 12.3, 110 x 1024 x 4096 10.0 / 8.7 / 7.4,
// 30 x 768 x 2816 7.7 / 6.6 / 5.4; at 224 tiles 7.8 / 6.5 / 7.4 (200 x 1024 x 2048), at 256 11.4 / 9.2 / 10.6 (100 x 2048 x 4096).
// With more tiles than CUs they are each other's company: 400 x 6400 x 768 (1742 tiles) 16.2 with four waves, 23 with eight.
template <typename T, int NB, int EPI>
static int many(const LmGemm& g, hipStream_t st) {
  if constexpr (sizeof(T) == 2 && NB == 2) {
    const long tiles = (long)((g.M + 31) / 32) * ((g.N + 31) / 32);
    if (tiles <= 128) return go<T, 2, 1, 8, EPI>(g, st);
    if (tiles <= 256) return go<T, 2, 2, 8, EPI>(g, st);
  }
  return go<T, 2, NB, 4, EPI>(g, st);
}

// Experts' products of few rows, which find their entries themselves.  Up to 24 tiles are walked to from expert to expert; with more, that is a
// chain of up to 64 steps for the last of them.  Walked / by bits, us: 16 rows of 2048, 32 experts, up 29.3 / 28.2 and down 34.3 / 32.1 per
// launch; 8 steps with 64 experts 6410 / 6090, 768 wide with 128 4180 / 3995, 7 rows of 1024 (28 tiles) 3280 / 3241, but 4 rows of 768 2420 / 2447
// and 5 (20 tiles) 2471 / 2494.
template <typename T, int NB, int WAVES, int EPI>
static int experts(const LmGemm& g, hipStream_t st) {
  return g.choice && g.max_tiles > 24 ? go<T, 1, NB, WAVES, EPI, true>(g, st) : go<T, 1, NB, WAVES, EPI>(g, st);
}

// up to 16 rows: one row block, more waves per tile (the weights are streamed once, latency counts)
template <typename T>
static int pick(int epi, const LmGemm& g, hipStream_t st) {
  const bool few = g.M <= 16;
  const int tile = sizeof(T) == 2 ? lm_tile(epi, g.M, g.N, g.K) : WIDE_NONE;
  if (tile != WIDE_NONE) {
    if (epi == LM_IN_ATTN) return pick_wide<LM_IN_ATTN>(tile, g, st);
    if (epi == LM_IN_GRU_SEQ) return go_wide<LM_IN_GRU_SEQ, 4, 6, 2, 2, 3, 1>(g, st);
    if (epi == LM_OUT) return pick_wide<LM_OUT>(tile, g, st);
    if (epi == LM_PROJ) return pick_wide<LM_PROJ>(tile, g, st);
    if (epi == LM_PLAIN) return pick_wide<LM_PLAIN>(tile, g, st);
    if (epi == LM_ACT) return pick_wide<LM_ACT>(tile, g, st);
  }
  if (sizeof(T) == 2 && g.tile_rows == 32) {
    if (epi == LM_MOE_UP) return go_wide<LM_MOE_UP, 2, 2, 1, 4, 4, 2>(g, st);
    if (epi == LM_MOE_DOWN) return go_wide<LM_MOE_DOWN, 2, 2, 1, 4, 4, 2>(g, st);
  }
  if (sizeof(T) == 2 && g.tile_rows == 64) {
    if (epi == LM_MOE_UP) return go_wide<LM_MOE_UP, 4, 2, 1, 4, 3, 2>(g, st);
    if (epi == LM_MOE_DOWN) return go_wide<LM_MOE_DOWN, 4, 2, 1, 4, 3, 2>(g, st);
  }
  // few rows and few features: one block of features per workgroup, so that more of the chip takes part
  if (few && (long)g.N * (g.max_tiles > 0 ? g.max_tiles : 1) <= 4096) {
    if (epi == LM_PROJ) return go<T, 1, 1, 16, LM_PROJ>(g, st);
    if (epi == LM_ACT) return go<T, 1, 1, 16, LM_ACT>(g, st);
    if (epi == LM_MOE_UP) return experts<T, 1, 16, LM_MOE_UP>(g, st);
    if (epi == LM_MOE_DOWN) return experts<T, 1, 16, LM_MOE_DOWN>(g, st);
  }
  // few features still: half a block per workgroup where whole ones would leave half the CUs without, and the others take in a block's
  // weights at 45 KB a us (16 x 2048 x 6144 13.4 -> 11.7 us, the mean of a 2048 wide step's thirteen 7.8 -> 7.0, with 4 rows 6.8 -> 6.5; before half a
  // block's weights were one load per step)
  if (few && epi == LM_PLAIN && g.N / 16 <= 128) return go<T, 1, 1, 16, LM_PLAIN, true>(g, st);
  if constexpr (sizeof(T) == 2)
    if (few && epi == LM_OUT && g.N / 16 <= 128) return go<T, 1, 1, 16, LM_OUT, true>(g, st);
  switch (epi) {
    case LM_IN_ATTN: return few ? go<T, 1, 2, 8, LM_IN_ATTN>(g, st) : many<T, 2, LM_IN_ATTN>(g, st);
    case LM_IN_GRU_STEP: return go<T, 1, 3, 8, LM_IN_GRU_STEP>(g, st);
    case LM_IN_GRU_SEQ: return few ? go<T, 1, 3, 8, LM_IN_GRU_SEQ>(g, st) : many<T, 3, LM_IN_GRU_SEQ>(g, st);
    case LM_OUT: return few ? go<T, 1, 1, 16, LM_OUT>(g, st) : many<T, 2, LM_OUT>(g, st);
    case LM_LOGITS: return few ? go<T, 1, 2, 8, LM_LOGITS>(g, st) : many<T, 2, LM_LOGITS>(g, st);
    case LM_HEAD: return few ? go<T, 1, 2, 8, LM_HEAD>(g, st) : many<T, 2, LM_HEAD>(g, st);
    case LM_PROJ: return few ? go<T, 1, 2, 8, LM_PROJ>(g, st) : many<T, 2, LM_PROJ>(g, st);
    case LM_PLAIN: return few ? go<T, 1, 1, 16, LM_PLAIN>(g, st) : many<T, 2, LM_PLAIN>(g, st);
    case LM_ACT: return few ? go<T, 1, 2, 8, LM_ACT>(g, st) : many<T, 2, LM_ACT>(g, st);
    case LM_MOE_UP: return few ? experts<T, 2, 8, LM_MOE_UP>(g, st) : go<T, 2, 2, 4, LM_MOE_UP>(g, st);
    case LM_MOE_DOWN: return few ? experts<T, 2, 8, LM_MOE_DOWN>(g, st) : go<T, 2, 2, 4, LM_MOE_DOWN>(g, st);
  }
  vui_set_error("lm gemm: unknown epilogue %d", epi);
  return VUI_EINVAL;
}

int launch_lm_gemm(int dtype, int epi, const LmGemm& g, hipStream_t st) {
  if ((epi == LM_LOGITS || epi == LM_HEAD) && g.N >= LM_SIZES) {  // a larger vocabulary by parts, the lengths with the last
    const int part = LM_SIZES / 2;
    for (int n = 0, rc; n < g.N; n += part) {
      LmGemm h = g;
      h.N = std::min(part, g.N - n); h.W = (const char*)g.W + (size_t)n * g.K * (dtype == VUI_DTYPE_F32 ? 4 : 2);
      h.logits = g.logits + n; h.vocab = g.vocab - n;
      if (h.N < g.N - n) h.upd_lens = nullptr;
      if ((rc = launch_lm_gemm(dtype, epi, h, st))) return rc;
    }
    return VUI_OK;
  }
  if (g.M < 1 || g.N < 16 || (g.N & 15) || g.K < 64 || (g.K & 63) || g.N >= LM_SIZES || g.K >= LM_SIZES || g.np > 0xffff) {
    vui_set_error("lm gemm: bad shape M=%d N=%d K=%d", g.M, g.N, g.K);
    return VUI_EINVAL;
  }
  if (epi == LM_EXPAND) {
    if (dtype != VUI_DTYPE_BF16 || g.heads < 1 || g.n_v < 16 || (g.n_v & 15)) { vui_set_error("lm gemm: bad expansion"); return VUI_EINVAL; }
    // the largest tile that gives every CU two workgroups (16 heads of 128 + 128, rank 512, 1999 positions: 18 us, with 64 x 128 24)
    auto tiles = [&](int bm, int bn) { return (long)((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn + (g.n_v + bn - 1) / bn) * g.heads; };
    return pick_wide<LM_EXPAND>(g.N > 64 && tiles(128, 128) >= 512 ? WIDE_128 : g.N > 64 && tiles(64, 128) >= 512 ? WIDE_64x128 : WIDE_64, g, st);
  }
  const bool gru = epi == LM_IN_GRU_STEP || epi == LM_IN_GRU_SEQ;
  if ((gru && ((g.mix_blocks % 3) || (g.N / 16) % 3)) || (epi == LM_IN_ATTN && (g.mix_blocks % 2))) {
    vui_set_error("lm gemm: the input projection is not padded to its tile");
    return VUI_EINVAL;
  }
  if (epi == LM_IN_GRU_STEP && g.M > 16) { vui_set_error("lm gemm: a recurrence step takes at most 16 rows"); return VUI_EINVAL; }
  return dtype == VUI_DTYPE_F32 ? pick<float>(epi, g, st) : pick<bf16_t>(epi, g, st);
}

// ---- embedding rows: residual, operand copy, sums of squares per 16 columns ----
template <typename T>
__global__ __launch_bounds__(256) void lm_embed_kernel(const LmRows where, const int64_t* tokens, const T* table, float* x, T* xt, float* ssq,
                                                       int width, int w64, int np, int vocab, int rows) {
  const int m = blockIdx.x * 16 + (threadIdx.x >> 4), c = blockIdx.y * 64 + (threadIdx.x & 15) * 4;  // a block of the operand's layout
  if (m >= rows) return;
  if (c == 0) lm_set_where(where, m);
  int64_t t = tokens[m];
  t = t < 0 ? 0 : (t >= vocab ? vocab - 1 : t);
  if (c < np * 16) {  // a multiple of 16: four neighbouring lanes are there or absent together
    const T* row = table + (size_t)t * width;
    float v[4];
    if ((width & 3) == 0 && ((uintptr_t)table & (4 * sizeof(T) - 1)) == 0) {  // every row starts on a whole vector
      if (c < width) Tl<T>::ld4(row + c, v);
      else v[0] = v[1] = v[2] = v[3] = 0.f;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = c + r < width ? El<T>::ld(row + c + r) : 0.f;
    }
    *reinterpret_cast<float4*>(x + (size_t)m * w64 + c) = make_float4(v[0], v[1], v[2], v[3]);
    Tl<T>::st4(xt + tl_off<T>(m, c, w64), v);
    float s = (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
    s += dpp_f<DPP_QUAD_XOR1>(s);
    s += dpp_f<DPP_QUAD_XOR2>(s);
    if ((c & 15) == 0) {
      const size_t at = (size_t)m * np + (c >> 4);
      if (rows <= LM_PAIRS) reinterpret_cast<float2*>(ssq)[at] = make_float2(s, 0.f);
      else ssq[at] = s;
    }
  }
}
int launch_lm_embed(int dtype, const LmRows& where, const int64_t* tokens, const void* table, float* x, void* xt, float* ssq, int rows, int width,
                    int w64, int np, int vocab, hipStream_t st) {
  if (dtype == VUI_DTYPE_F32)
    hipLaunchKernelGGL(lm_embed_kernel<float>, dim3((rows + 15) / 16, (np + 3) / 4), dim3(256), 0, st, where, tokens, (const float*)table, x, (float*)xt, ssq, width, w64, np, vocab, rows);
  else
    hipLaunchKernelGGL(lm_embed_kernel<bf16_t>, dim3((rows + 15) / 16, (np + 3) / 4), dim3(256), 0, st, where, tokens, (const bf16_t*)table, x, (bf16_t*)xt, ssq, width, w64, np, vocab, rows);
  HIP_TRY(hipGetLastError());
  return VUI_OK;
}
