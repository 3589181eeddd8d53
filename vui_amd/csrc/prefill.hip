// Prompt ingestion: T > 1 new positions of one row through the backbone in one pass per layer.
//
//   Decoder.forward_flash / Engine._prefill_emb with T > 1  (src/vui/model.py:534-549, engine.py:674-694)
//
// bf16 activations; the layers' matrices bf16, or int8 with per-row scales (widened in registers inside the GEMMs,
// the scale on the finished sum).  Per layer: row RMSNorm, QKV GEMM whose epilogue rotates queries and keys, appends keys and
// values to the cache and leaves both in the attention's operand layout (behind earlier positions a kernel lays out the whole slot
// instead: the copy of those costs the launch anyway), causal attention of the new positions (scores never leave the registers; probabilities
// rounded to bf16 before they meet the values), out_proj GEMM with the residual add in its epilogue, row RMSNorm, one GEMM over
// W1 and W3 with the SwiGLU product in its epilogue, W2 GEMM with residual: seven launches, eight behind earlier positions.
// A short block (up to PF_SHORT positions) takes five: its GEMMs norm their rows themselves, and attention reads the cache as it is.
// Every GEMM is C (M x N) = X (M x K) W^T (N x K) on the matrix cores, both operands in the tiled layout below.
//
// Rounding points are those of the single-position step (one rounding after each linear, two in
// the norm, products of the rotation rounded before their sum, residual sums rounded).
#include "common.h"
#include "internal.h"
#include "wide.h"
#include <stdio.h>

typedef tl_bf16x8 pf_bf16x8;
typedef tl_f32x4 pf_floatx4;
__device__ __forceinline__ pf_bf16x8 pf_frag(const uint4& x) { return Tl<bf16_t>::frag(x); }

enum { PF_BF16 = 0, PF_RESID = 1, PF_QKV = 2 };

// Both operands of the GEMMs are in the tiled layout of tile.h (blocks of 16 rows x 64 columns).  Weights are brought
// into this form once per context, activations are written in it by their producers.
__host__ __device__ __forceinline__ size_t pf_toff(int r, int k, int K) { return tl_off<bf16_t>(r, k, K); }

struct PfGemm {
  const bf16_t* X;   // activations (M x K), tiled
  const void* W;     // weights (N x K), tiled: bf16, or int8 (the byte form of the layout: block (r / 16, k / 64) at
                     // ((r / 16) * (K / 64) + k / 64) * 1024 bytes, the 16 bytes k % 16 = 0..15 of lane (r % 16) + 16 * ((k % 64) / 16)
                     // at 16 * lane) with the per-row scales sc (and sc2 for the second matrix of a SwiGLU pair)
  const bf16_t *sc, *sc2;
  void* C;           // output (M x N) bf16: row-major with row stride ldc (PF_RESID: in place on the residual), or tiled
  int M, N, K, ldc;  // ldc: of PF_QKV
  int c_tiled;
  // X is the residual and is normed on its way: sums of squares of every 16 columns (M x K / 16), weights (K)
  const float* ssq;
  const bf16_t* nw;
  float eps;
  float* ssq_out;    // PF_RESID: the same sums of the new residual, or nullptr
  // PF_QKV: C receives the rotated queries alone; row m is position pos0 + m of the slot
  bf16_t *kc, *vc;   // its cache rows
  bf16_t *kt, *vt;   // operand copies of keys and transposed values (pf_stage_kv_kernel); nullptr unless the slot is empty (pos0 == 0)
  const float* rope;
  int nq, nkv, hd, rope_dim, pos0, Lpad;
  // pf_order: tiles of an XCD (the first xcd_more have one more), tiles of one step of the slower index
  uint32_t xcd_tiles, xcd_more, run, inv_run, inv_hd;
  int by_rows, n_tiles;
  int warm_gsz;         // heads per group, or 0 (see pf_warm)
  int warm, warm_from;  // the last `warm` workgroups only fetch the cached positions warm_from .. pos0 - 1 (see pf_warm)
};

// i / n for i < 65536 with inv = pf_inv(n): a division by a runtime value costs a workgroup 0.1 us
static uint32_t pf_inv(uint32_t n) { return n > 1 ? 0xFFFFFFFFu / n + 1u : 0u; }
__device__ __forceinline__ uint32_t pf_div(uint32_t i, uint32_t inv) { return inv ? __umulhi(i, inv) : i; }

// The attention of a short block is a few workgroups that wait for cached keys and values from memory (2.4 us of its first
// step, 0.85 where they are in the memory-side cache).  The QKV product before it leaves compute units idle: workgroups of
// its launch that have no tile read them ahead.
// Where XCD x attends to heads x, x + 8, ... (a number of heads that eight divides), its readers take those heads' columns, so that they lie in
// its L2: 16 positions behind up to 1500 in eight rows in turn, us a prompt, 550 -> 539 in bf16, 545 -> 537 in int8; one row behind 100, 700 or 2000 the same.
__device__ __forceinline__ void pf_warm(const PfGemm& p, int part) {
  if (p.warm_gsz > 0) {
    const int x = (int)blockIdx.x & 7, lead = p.n_tiles + ((x - p.n_tiles) & 7), mine = ((int)blockIdx.x - lead) >> 3, all = ((int)gridDim.x - 1 - lead) / 8 + 1;
    const int per = p.hd >> 3, rows = (int)blockDim.x / per, row = (int)threadIdx.x / per, col = ((int)threadIdx.x - row * per) * 8;
    if (row >= rows) return;
    for (int h = x, last = -1; h * p.hd < p.nq; h += 8) {
      const int g = h / p.warm_gsz;
      if (g == last) continue;  // heads of a group share keys
      last = g;
      for (int j = p.warm_from + mine * rows + row; j < p.pos0; j += all * rows) {
        const size_t at = (size_t)j * p.nkv + g * p.hd + col;
        const uint4 k = *reinterpret_cast<const uint4*>(p.kc + at), v = *reinterpret_cast<const uint4*>(p.vc + at);
        asm volatile("" ::"v"(k.x), "v"(v.x));
      }
    }
    return;
  }
  const size_t n = (size_t)(p.pos0 - p.warm_from) * p.nkv / 8, at = (size_t)p.warm_from * p.nkv;
  for (size_t i = (size_t)part * blockDim.x + threadIdx.x; i < n; i += (size_t)p.warm * blockDim.x) {
    const uint4 k = *reinterpret_cast<const uint4*>(p.kc + at + i * 8), v = *reinterpret_cast<const uint4*>(p.vc + at + i * 8);
    asm volatile("" ::"v"(k.x), "v"(v.x));
  }
}

// The first fourteen words of a kernel's scalar arguments are in registers when it starts; a struct behind them is a trip to memory.
// What the first loads of a product need therefore comes twice, ahead of the struct and in it: 0.2-0.35 us of a launch of 4-6 (16
// positions, us per launch: QKV 5.4 -> 5.1, W1 and W3 5.6 -> 5.2; whole pass of 576 positions 1160 -> 1121, of 1733 in int8 1976 -> 1952).
#define PF_HOT const bf16_t *X, const void *W, const void *aux, const bf16_t *nw, int M, uint32_t nk, uint32_t xcd, uint32_t run, uint32_t inv_run
#define PF_HOT_ARGS(g, aux) g.X, g.W, (const void*)(aux), g.nw, g.M, (uint32_t)(g.N >> 4 | g.K >> 6 << 16) | (uint32_t)g.c_tiled << 31, g.xcd_tiles | g.xcd_more << 28 | (uint32_t)g.by_rows << 31, g.run, g.inv_run
#define PF_HOT_IN(p)                                                                                                  \
  p.X = X; p.W = W; p.nw = nw; p.M = M; p.N = (int)(nk & 0xffffu) * 16; p.K = (int)(nk >> 16 & 0x7fffu) * 64; p.c_tiled = (int)(nk >> 31);                  \
  p.xcd_tiles = xcd & 0xfffffffu; p.xcd_more = xcd >> 28 & 7u; p.by_rows = (int)(xcd >> 31); p.run = run; p.inv_run = inv_run

// Which tile (of MT x NT) a workgroup takes: {row tile, feature tile}.  Workgroups go round the eight XCDs, whose L2s are their
// own, so each XCD gets a contiguous range of the tiles: of the feature tiles where the weights are more bytes than the rows - it then
// meets an eighth of the weights and all rows - and of the row tiles otherwise.
// Whole pass, us, in order of dispatch / so: bf16 300 positions 988 / 916, 576 1246 / 1145, 1733 2155 / 2070; int8 300 833 / 789, 1733
// 2194 / 1951.  The line lies at twice the rows' bytes, since the rows were written just before (576 positions at equal bytes: 1180).
__device__ __forceinline__ int2 pf_order(const PfGemm& p) {
  const uint32_t x = blockIdx.x & 7u;
  const uint32_t id = x * p.xcd_tiles + min(x, p.xcd_more) + (blockIdx.x >> 3), q = pf_div(id, p.inv_run), r = id - q * p.run;
  return p.by_rows ? make_int2(q, r) : make_int2(r, q);
}

// rotation factors of features n .. n + 3 (n % 4 == 0) of a head whose first rope_dim features turn: cos, sin of two pairs
struct PfRot { float4 a, b; };
__device__ __forceinline__ PfRot pf_rot(const float* rope, int pos, int rope_dim, int dd) {
  PfRot r;
  const float* f = rope + (size_t)pos * rope_dim * 2;
  r.a = *reinterpret_cast<const float4*>(f + min(dd, rope_dim - 2) * 2);
  r.b = *reinterpret_cast<const float4*>(f + min(dd + 2, rope_dim - 2) * 2);
  return r;
}
// Where a block of 16 features that begins at n (uniform over the wave) lies: queries, keys or values, its head there, its first
// dimension in the head (a multiple of 16), and for keys and values its column in a cache row
struct PfPart { int part, head, dim, col; };
__device__ __forceinline__ PfPart pf_part(const PfGemm& p, int n) {
  PfPart r;
  r.part = n < p.nq ? 0 : (n < p.nq + p.nkv ? 1 : 2);
  r.col = n - (r.part == 0 ? 0 : (r.part == 1 ? p.nq : p.nq + p.nkv));
  r.head = pf_div(r.col, p.inv_hd);
  r.dim = r.col - r.head * p.hd;
  return r;
}
// Epilogue of PF_QKV for features 4 kg .. 4 kg + 3 of such a block, row m: v is rounded, the interleaved pairs of queries and keys are
// rotated (src/vui/rope.py:16-77), keys and values appended to the cache (src/vui/model.py:234-247), keys laid out for pf_attn_kernel.
__device__ __forceinline__ void pf_qkv_out(const PfGemm& p, const PfPart& b, int m, int kg, const float* v, const PfRot& rot) {
  float o[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) o[r] = bf2f(f2bf(v[r]));
  const int dd = b.dim + 4 * kg, col = b.col + 4 * kg, j = p.pos0 + m;
  if (b.part < 2) {
    const float a = rope_mix(o[0], rot.a.x, -o[1], rot.a.y), c = rope_mix(o[1], rot.a.z, o[0], rot.a.w);
    const float e = rope_mix(o[2], rot.b.x, -o[3], rot.b.y), f = rope_mix(o[3], rot.b.z, o[2], rot.b.w);
    if (dd < p.rope_dim) { o[0] = a; o[1] = c; }
    if (dd + 2 < p.rope_dim) { o[2] = e; o[3] = f; }
  }
  const uint2 w = make_uint2(f2bf2(o[0], o[1]), f2bf2(o[2], o[3]));
  if (b.part == 0) {
    *reinterpret_cast<uint2*>((bf16_t*)p.C + (size_t)m * p.ldc + col) = w;
  } else if (b.part == 1) {
    *reinterpret_cast<uint2*>(p.kc + (size_t)j * p.nkv + col) = w;
    if (p.kt) {
      const size_t blk = ((size_t)b.head * (p.Lpad >> 4) + (m >> 4)) * (p.hd >> 5) + (dd >> 5);
      *reinterpret_cast<uint2*>(p.kt + blk * 512 + ((m & 15) + 16 * ((dd & 31) >> 3)) * 8 + (dd & 7)) = w;
    }
  } else {
    *reinterpret_cast<uint2*>(p.vc + (size_t)j * p.nkv + col) = w;
  }
}
// The values of feature l16 of such a block in rows m .. m + 3 (m % 4 == 0), into the transposed layout
__device__ __forceinline__ void pf_vt_out(const PfGemm& p, const PfPart& b, int m, int l16, const float* v) {
  const size_t blk0 = ((size_t)b.head * (p.hd >> 4) + (b.dim >> 4)) * (p.Lpad >> 5);
  bf16_t* dst = p.vt + (blk0 + (m >> 5)) * 512 + (l16 + 16 * ((m & 15) >> 2)) * 8 + 4 * ((m & 31) >> 4);
  if (m + 3 < p.M) { *reinterpret_cast<uint2*>(dst) = make_uint2(f2bf2(v[0], v[1]), f2bf2(v[2], v[3])); return; }
  for (int r = 0; r < 4; ++r) if (m + r < p.M) dst[r] = f2bf(v[r]);
}

// row-major (N x K) -> tiled; one 8-element piece per thread
__global__ __launch_bounds__(256) void pf_tile_kernel(const bf16_t* __restrict__ src, bf16_t* __restrict__ dst, int N, int K) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  const int per_row = K >> 3;
  if (i >= (size_t)N * per_row) return;
  const int n = (int)(i / per_row), k = (int)(i % per_row) * 8;
  *reinterpret_cast<uint4*>(dst + pf_toff(n, k, K)) = *reinterpret_cast<const uint4*>(src + (size_t)n * K + k);
}

// eight residual values of one row -> normed: rnd(rnd(x r) g)
__device__ __forceinline__ uint4 pf_norm8(const uint4& x, float r, const uint4& g) {
  uint4 o;
  uint32_t t;
  t = f2bf2(bf_lo(x.x) * r, bf_hi(x.x) * r); o.x = f2bf2(bf_lo(t) * bf_lo(g.x), bf_hi(t) * bf_hi(g.x));
  t = f2bf2(bf_lo(x.y) * r, bf_hi(x.y) * r); o.y = f2bf2(bf_lo(t) * bf_lo(g.y), bf_hi(t) * bf_hi(g.y));
  t = f2bf2(bf_lo(x.z) * r, bf_hi(x.z) * r); o.z = f2bf2(bf_lo(t) * bf_lo(g.z), bf_hi(t) * bf_hi(g.z));
  t = f2bf2(bf_lo(x.w) * r, bf_hi(x.w) * r); o.w = f2bf2(bf_lo(t) * bf_lo(g.w), bf_hi(t) * bf_hi(g.w));
  return o;
}

// C = X W^T for the projections (K = d_model ... ffn; 64 x 64 tiles would give only 9 x 12 ... 9 x 64
// workgroups at 576 positions, each a long serial walk over K): a workgroup owns 16 MB rows x 16 NB features and its waves
// split the K steps between them, so a wave's chain of dependent trips to memory is a fraction as long and more
// workgroups are in flight.  The partial tiles meet in LDS and are added in wave order (a fixed order:
// results do not depend on timing).
// DUAL: two weight matrices against the same activations, h = rnd(rnd(silu(rnd(a))) * rnd(c)) written once
// (SwiGLU, src/vui/model.py:282) instead of two products and a pass over both.
// NORM: X is the residual; every wave norms the fragments it multiplies (two roundings, src/vui/model.py:286-297) with the
// rows' factors from sums of squares that the residual's producer left in pieces of 16 columns.  That costs a launch of a
// short block 0.5-1.7 us (16 positions: QKV 3.8 -> 5.5, W1 and W3 5.0 -> 5.5) and saves the norm's own of 3.4; repeated for every
// tile of features it does not pay for longer ones.
template <int EPI, bool DUAL, bool I8, int WAVES, int MB, int NB, bool NORM>
__global__ __launch_bounds__(64 * WAVES) void pf_gemm_kernel(PF_HOT, const PfGemm p0) {
  PfGemm p = p0;
  PF_HOT_IN(p);
  if (EPI == PF_RESID) p.C = (void*)aux;
  else if (NORM) p.ssq = (const float*)aux;
  const char* W2 = (const char*)W + (size_t)p.N * p.K * (I8 ? 1 : 2);  // DUAL: the second matrix lies behind the first
  constexpr int TILE = MB * NB * 256;  // floats of one partial tile
  constexpr int PW = (DUAL ? 2 : 1) * TILE;
  __shared__ __align__(16) float part[WAVES * PW];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l16 = lane & 15, kg = lane >> 4;
  if (EPI == PF_QKV && NORM && (int)blockIdx.x >= p.n_tiles) { pf_warm(p, blockIdx.x - p.n_tiles); return; }
  const int2 tile = pf_order(p);
  const int m0 = tile.x * 16 * MB, n0 = tile.y * 16 * NB;
  // A step covers 64 values of k, one block of the tiled operands per 16 rows: the lane's 16-byte piece of half h
  // (k = 64 s + 16 kg + 8 h ...; any assignment of k to lanes is valid as long as both operands share it) is at
  // block + 512 h + 8 lane.
  const int nsteps = p.K >> 6;
  const int s0 = nsteps * wave / WAVES, s1 = nsteps * (wave + 1) / WAVES;
  const int MBL = (p.M + 15) >> 4, NBL = (p.N + 15) >> 4;  // 16-row blocks; a tile past the end reads the last block again
  const bf16_t* xr[MB];
  const char* wr[NB];  // byte addresses: a block is 2048 bytes of bf16 (two 16-byte pieces per lane) or 1024 of int8 (one)
  const char* vr[NB];
  constexpr int WB = I8 ? 1024 : 2048, WL = 16;
#pragma unroll
  for (int j = 0; j < MB; ++j) xr[j] = p.X + (size_t)min((m0 >> 4) + j, MBL - 1) * nsteps * 1024 + lane * 8;
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const size_t wo = (size_t)min((n0 >> 4) + j, NBL - 1) * nsteps * WB + lane * WL;
    wr[j] = (const char*)p.W + wo;
    vr[j] = (DUAL ? W2 : (const char*)p.W) + wo;
  }
  pf_floatx4 acc[NB][MB], acc2[NB][MB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j) { acc[i][j] = pf_floatx4{0.f, 0.f, 0.f, 0.f}; acc2[i][j] = acc[i][j]; }
  // Steps whose loads go out together, as far as the wave has them
  constexpr int U = WAVES >= 12 && MB * NB <= 2 ? 2 : 1;
  uint4 xs[U][MB][2], ws[U][NB][2], vs[U][NB][2], gs[U][2];
  auto load = [&](int s0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u, k = s << 10;
      if (u > 0 && s >= s1) break;  // uniform
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          if (I8 && h) continue;  // both halves of an int8 block are one piece
          ws[u][j][h] = *reinterpret_cast<const uint4*>(wr[j] + (size_t)s * WB + 1024 * h);
          if (DUAL) vs[u][j][h] = *reinterpret_cast<const uint4*>(vr[j] + (size_t)s * WB + 1024 * h);
        }
#pragma unroll
        for (int j = 0; j < MB; ++j) xs[u][j][h] = *reinterpret_cast<const uint4*>(xr[j] + k + 512 * h);
        if (NORM) gs[u][h] = *reinterpret_cast<const uint4*>(p.nw + 64 * s + 16 * kg + 8 * h);
      }
    }
  };
  // The operands of the first step go out before anything else is asked for, then the residual values this thread will add to (its
  // four outputs, see the epilogue), instead of after the last product; clamped to the matrix, unused where the thread has no output.
  if (WAVES >= 8 && s0 < s1) load(s0);
  if (WAVES >= 8) __builtin_amdgcn_sched_barrier(0);
  uint2 old = make_uint2(0, 0);
  PfRot rot = {};
  {
    const int em = min(m0 + 16 * (wave % MB) + l16, p.M - 1), en = min(n0 + 16 * (wave / MB % NB) + 4 * kg, p.N - 4);
    if (EPI == PF_RESID) old = *reinterpret_cast<const uint2*>((const bf16_t*)p.C + (p.c_tiled ? pf_toff(em, en, p.N) : (size_t)em * p.N + en));
    if (EPI == PF_QKV && p.rope_dim >= 2) rot = pf_rot(p.rope, p.pos0 + em, p.rope_dim, pf_part(p, min(n0 + 16 * (wave / MB % NB), p.N - 16)).dim + 4 * kg);
  }
  float rf[MB];
  if (NORM) {
    float ss[MB] = {};
    for (int i = kg; i < nsteps; i += 16) {
      float4 t[MB][4];
#pragma unroll
      for (int j = 0; j < MB; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          t[j][u] = reinterpret_cast<const float4*>(p.ssq + (size_t)min(m0 + 16 * j + l16, p.M - 1) * (p.K >> 4))[min(i + 4 * u, nsteps - 1)];
#pragma unroll
      for (int j = 0; j < MB; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) ss[j] += i + 4 * u < nsteps ? (t[j][u].x + t[j][u].y) + (t[j][u].z + t[j][u].w) : 0.f;
    }
#pragma unroll
    for (int j = 0; j < MB; ++j) rf[j] = 1.0f / sqrtf(rows_sum(ss[j]) / (float)p.K + p.eps);
  }
  for (int s = s0; s < s1; s += U) {
    if (WAVES < 8 || s > s0) load(s);
#pragma unroll
    for (int q = 0; q < U; ++q) {
    if (q > 0 && s + q >= s1) break;  // uniform
    uint4 (&xa)[MB][2] = xs[q], (&wa)[NB][2] = ws[q], (&va)[NB][2] = vs[q], (&g)[2] = gs[q];
    if (I8) {
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const uint4 w8 = wa[j][0];
        wa[j][0] = widen8_i8(w8.x, w8.y); wa[j][1] = widen8_i8(w8.z, w8.w);
        if (DUAL) {
          const uint4 v8 = va[j][0];
          va[j][0] = widen8_i8(v8.x, v8.y); va[j][1] = widen8_i8(v8.z, v8.w);
        }
      }
    }
    if (NORM) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < MB; ++j) xa[j][h] = pf_norm8(xa[j][h], rf[j], g[h]);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < MB; ++j) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf_frag(wa[i][h]), pf_frag(xa[j][h]), acc[i][j], 0, 0, 0);
          if (DUAL) acc2[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf_frag(va[i][h]), pf_frag(xa[j][h]), acc2[i][j], 0, 0, 0);
        }
    }
  }
  // partial tiles to LDS: [wave][(i, j)][lane] as float4
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j) {
      *reinterpret_cast<pf_floatx4*>(&part[wave * PW + ((i * MB + j) * 64 + lane) * 4]) = acc[i][j];
      if (DUAL) *reinterpret_cast<pf_floatx4*>(&part[wave * PW + TILE + ((i * MB + j) * 64 + lane) * 4]) = acc2[i][j];
    }
  __syncthreads();
  if (wave >= MB * NB) return;
  // thread: sub-tile (i, j) of its wave, features n0 + 16 i + 4 kg + r (r = 0..3) of row m0 + 16 j + l16
  const int i = wave / MB, j = wave % MB;
  const int m = m0 + 16 * j + l16, n = n0 + 16 * i + 4 * kg;
  float v[4], u[4];
  {  // all waves' parts are read before the first is added
    pf_floatx4 a[WAVES], b[DUAL ? WAVES : 1];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      a[w] = *reinterpret_cast<const pf_floatx4*>(&part[w * PW + tid * 4]);
      if (DUAL) b[w] = *reinterpret_cast<const pf_floatx4*>(&part[w * PW + TILE + tid * 4]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
      a[0] += a[w];
      if (DUAL) b[0] += b[w];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) { v[r] = a[0][r]; if (DUAL) u[r] = b[0][r]; }
  }
  const bool out = m < p.M && n < p.N;  // N is a multiple of 16
  if (EPI == PF_QKV && !NORM && p.vt && n0 + 16 * i >= p.nq + p.nkv && n0 + 16 * i < p.N) {
    // the tile transposed: feature l16 of rows 4 kg .. 4 kg + 3
    float t[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int e = (wave * 64 + 4 * kg + r + 16 * (l16 >> 2)) * 4 + (l16 & 3);
      t[r] = part[e];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) t[r] += part[w * PW + e];
      if (I8) t[r] *= bf2f(p.sc[n0 + 16 * i + l16]);
    }
    pf_vt_out(p, pf_part(p, n0 + 16 * i), m0 + 16 * j + 4 * kg, l16, t);
  }
  if (EPI != PF_RESID && !out) return;
  if (I8) {  // y[n] = scale[n] * sum_k q[n, k] x[k]
    const int ns = min(n, p.N - 4);
    for (int r = 0; r < 4; ++r) { v[r] *= bf2f(p.sc[ns + r]); if (DUAL) u[r] *= bf2f(p.sc2[ns + r]); }
  }
  if (EPI == PF_QKV) {
    const PfPart blk = pf_part(p, n0 + 16 * i);
    pf_qkv_out(p, blk, m, kg, v, rot);
    return;
  }
  bf16_t* c = (bf16_t*)p.C + (p.c_tiled ? pf_toff(m, n, p.N) : (size_t)m * p.N + n);  // n % 4 == 0: inside one piece
  if (DUAL) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float a = bf2f(f2bf(v[r])), b = bf2f(f2bf(u[r]));
      v[r] = bf2f(f2bf(a / (1.0f + expf(-a)))) * b;
    }
  }
  if (EPI == PF_RESID) {  // x = rnd(x + rnd(y)), src/vui/model.py:367, 374
    v[0] = bf_lo(old.x) + bf2f(f2bf(v[0])); v[1] = bf_hi(old.x) + bf2f(f2bf(v[1]));
    v[2] = bf_lo(old.y) + bf2f(f2bf(v[2])); v[3] = bf_hi(old.y) + bf2f(f2bf(v[3]));
  }
  const uint2 w = make_uint2(f2bf2(v[0], v[1]), f2bf2(v[2], v[3]));
  if (out) *reinterpret_cast<uint2*>(c) = w;
  if (EPI == PF_RESID && p.ssq_out) {  // uniform; a row's sixteen columns are in the four lanes of its column
    const float a = bf_lo(w.x), b = bf_hi(w.x), e = bf_lo(w.y), f = bf_hi(w.y);
    const float ss = rows_sum((a * a + b * b) + (e * e + f * f));
    if (out && kg == 0) p.ssq_out[(size_t)m * (p.N >> 4) + (n >> 4)] = ss;
  }
}

// The same product for prompts of a few hundred positions and more: large tiles through LDS (wide.h).  DUAL: a wave's first
// NBW / 2 blocks are features of the first matrix, the others the same features of the second.  The sums pass through
// the wave's share of LDS, so that the epilogue is a loop over blocks.
template <int EPI, bool DUAL, bool I8, int MBW, int NBW, int WM, int WN, int S, int KS>
__global__ __launch_bounds__(256, 2) void pf_wide_kernel(PF_HOT, const PfGemm p0) {
  PfGemm p = p0;
  PF_HOT_IN(p);
  const char* W2 = (const char*)W + (size_t)p.N * p.K * (I8 ? 1 : 2);
  typedef WideTile<MBW, NBW, WM, WN, S, KS, I8> Tile;
  constexpr int NF = DUAL ? NBW / 2 : NBW, MB = Tile::MB, NB = NF * WN;  // feature blocks of a wave and of the tile
  __shared__ __align__(16) char lds[Tile::LDS];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l16 = lane & 15, kg = lane >> 4, wm = wave % WM, wn = wave / WM;
  const int MBL = (p.M + 15) >> 4, NBL = p.N >> 4;
  const int2 tl = pf_order(p);
  const int mb0 = tl.x * MB, nb0 = tl.y * NB;
  const size_t xb = (size_t)p.K * 32, wb = (size_t)p.K * (I8 ? 16 : 32);  // bytes of a 16-row block
  Tile tile;
  tile.begin(lds, wave, lane, [&](int i) { return (const char*)p.X + min(mb0 + i, MBL - 1) * xb; },
             [&](int i) {
               const int w = i / NBW, b = i % NBW;  // wave and block of the tile's i-th
               return (DUAL && b >= NF ? W2 : (const char*)p.W) + min(nb0 + w * NF + b % NF, NBL - 1) * wb;
             });
  const int Q = p.K / (32 * KS);
  tile.prologue(Q);
  tl_f32x4 acc[NBW][MBW];
  tile.run(Q, acc);
  __syncthreads();
  constexpr int ROOM = S * Tile::PIECES / 4;
  static_assert(ROOM >= NBW * MBW, "a wave's sums fit its share");
  char* own = lds + wave * ROOM * 1024 + lane * 16;
#pragma unroll
  for (int i = 0; i < NBW; ++i)
#pragma unroll
    for (int j = 0; j < MBW; ++j) *reinterpret_cast<tl_f32x4*>(own + (i * MBW + j) * 1024) = acc[i][j];
#pragma unroll 1
  for (int i = 0; i < NF; ++i) {
    const int nb = nb0 + wn * NF + i, n = nb * 16 + 4 * kg, mw = (mb0 + wm * MBW) * 16 + l16;
    if (nb >= NBL) break;
    float s1[4], s2[4];
    if (I8) {
#pragma unroll
      for (int r = 0; r < 4; ++r) { s1[r] = bf2f(p.sc[n + r]); if (DUAL) s2[r] = bf2f(p.sc2[n + r]); }
    }
    uint2 old[MBW];
    PfRot rot[MBW] = {};
    PfPart blk = {};
    if (EPI == PF_QKV) blk = pf_part(p, nb * 16);
#pragma unroll
    for (int j = 0; j < MBW; ++j) {
      const int m = min(mw + 16 * j, p.M - 1);
      if (EPI == PF_QKV && p.rope_dim >= 2 && blk.part < 2) rot[j] = pf_rot(p.rope, p.pos0 + m, p.rope_dim, blk.dim + 4 * kg);
      if (EPI == PF_RESID) old[j] = *reinterpret_cast<const uint2*>((const bf16_t*)p.C + (p.c_tiled ? pf_toff(m, n, p.N) : (size_t)m * p.N + n));
    }
#pragma unroll
    for (int j = 0; j < MBW; ++j) {
      const int m = mw + 16 * j;
      const tl_f32x4 a = *reinterpret_cast<const tl_f32x4*>(own + (i * MBW + j) * 1024);
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = I8 ? a[r] * s1[r] : a[r];
      if (DUAL) {  // rnd(rnd(silu(rnd(a))) * rnd(c)), src/vui/model.py:282
        const tl_f32x4 c = *reinterpret_cast<const tl_f32x4*>(own + ((NF + i) * MBW + j) * 1024);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float g = bf2f(f2bf(v[r])), u = bf2f(f2bf(I8 ? c[r] * s2[r] : c[r]));
          v[r] = bf2f(f2bf(g / (1.0f + expf(-g)))) * u;
        }
      }
      if (EPI == PF_RESID) {  // x = rnd(x + rnd(y)), src/vui/model.py:367, 374
        v[0] = bf_lo(old[j].x) + bf2f(f2bf(v[0])); v[1] = bf_hi(old[j].x) + bf2f(f2bf(v[1]));
        v[2] = bf_lo(old[j].y) + bf2f(f2bf(v[2])); v[3] = bf_hi(old[j].y) + bf2f(f2bf(v[3]));
      }
      if (EPI == PF_QKV) {
        if (m < p.M) pf_qkv_out(p, blk, m, kg, v, rot[j]);
        if (blk.part == 2 && p.vt) {  // the block transposed: feature l16 of rows 4 kg .. 4 kg + 3
          const float* t = reinterpret_cast<const float*>(lds + wave * ROOM * 1024 + (i * MBW + j) * 1024) + (l16 >> 2) * 64 + (l16 & 3);
          const float sf = I8 ? bf2f(p.sc[nb * 16 + l16]) : 0.f;
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = I8 ? t[(4 * kg + r) * 4] * sf : t[(4 * kg + r) * 4];
          pf_vt_out(p, blk, (mb0 + wm * MBW + j) * 16 + 4 * kg, l16, v);
        }
      } else if (m < p.M) *reinterpret_cast<uint2*>((bf16_t*)p.C + (p.c_tiled ? pf_toff(m, n, p.N) : (size_t)m * p.N + n)) = make_uint2(f2bf2(v[0], v[1]), f2bf2(v[2], v[3]));
    }
  }
}

// the fields of pf_order for tiles of bm x bn; returns their number
static unsigned pf_set_order(PfGemm& g, int bm, int bn, size_t weight_bytes) {
  const unsigned MT = (g.M + bm - 1) / bm, NT = (g.N + bn - 1) / bn, n = MT * NT;
  g.by_rows = weight_bytes < (size_t)g.M * g.K * 4;
  g.xcd_tiles = n >> 3; g.xcd_more = n & 7; g.run = g.by_rows ? NT : MT; g.inv_run = pf_inv(g.run); g.n_tiles = (int)n;
  return n;
}

template <int EPI, bool DUAL, bool I8>
static int pf_wide(int tile, PfGemm& g, hipStream_t st) {
  const int bm = tile == WIDE_128 ? 128 : 64, bn = (tile == WIDE_64 ? 64 : 128) / (DUAL ? 2 : 1);
  const dim3 grid(pf_set_order(g, bm, bn, (size_t)g.N * g.K * ((DUAL ? 2 : 1) * (I8 ? 1 : 2))));
  if (tile == WIDE_128) hipLaunchKernelGGL((pf_wide_kernel<EPI, DUAL, I8, 4, 4, 2, 2, I8 ? 3 : 4, I8 ? 2 : 1>), grid, dim3(256), 0, st, PF_HOT_ARGS(g, nullptr), g);
  else if (tile == WIDE_64x128) hipLaunchKernelGGL((pf_wide_kernel<EPI, DUAL, I8, 4, 2, 1, 4, I8 ? 4 : 3, 2>), grid, dim3(256), 0, st, PF_HOT_ARGS(g, nullptr), g);
  else hipLaunchKernelGGL((pf_wide_kernel<EPI, DUAL, I8, 2, 2, 2, 2, 4, 2>), grid, dim3(256), 0, st, PF_HOT_ARGS(g, nullptr), g);
  HIP_TRY(hipGetLastError());
  return VUI_OK;
}

// two-rounding RMSNorm of rows (src/vui/model.py:286-297); one wave per row.  len != nullptr: the slot's new length goes there
// (where a row lies is known when compiled: asked for per piece it took a launch 0.3 us, 65 positions behind 600 3.57 -> 3.95)
// The row stays in registers, NP pieces of eight columns per lane, and the weights are asked for with it: one trip to memory instead of
// two, one after the other.  Whole prompts, us: 576 positions 1109 -> 1098, 1733 in int8 1955 -> 1917.  Four and eight rows per wave, which write
// whole lines of the tiled rows, were slower (576: 1115 and 1170).  NP 0: rows of more than 2048 columns, read twice.
template <bool X_TILED, int NP>
__global__ __launch_bounds__(256) void pf_rownorm_kernel(const bf16_t* x, const bf16_t* w, bf16_t* y, int M, int K, float eps, int y_tiled,
                                                         int32_t* len, int len_to) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (len && blockIdx.x == 0 && threadIdx.x == 0) *len = len_to;
  if (row >= M) return;
  const int nc = K >> 3;
  auto ld = [&](const bf16_t* q) { return *reinterpret_cast<const uint4*>(q); };
  auto xr = [&](int c) { return ld(x + (X_TILED ? pf_toff(row, c * 8, K) : (size_t)row * K + c * 8)); };
  uint4 xv[NP > 0 ? NP : 1], wv[NP > 0 ? NP : 1];
  if constexpr (NP > 0) {
#pragma unroll
    for (int i = 0; i < NP; ++i) xv[i] = xr(min(lane + WAVE * i, nc - 1));
#pragma unroll
    for (int i = 0; i < NP; ++i) wv[i] = ld(w + min(lane + WAVE * i, nc - 1) * 8);
    __builtin_amdgcn_sched_barrier(0);
  }
  float ss = 0.f;
  auto add = [&](const uint4& q) {
    float v[8];
    El<bf16_t>::ld8(reinterpret_cast<const bf16_t*>(&q), v);
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
  };
  if constexpr (NP > 0) {
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if (lane + WAVE * i < nc) add(xv[i]);
  } else {
    for (int c = lane; c < nc; c += WAVE) add(xr(c));
  }
  ss = wave_sum(ss);
  const float r = 1.0f / sqrtf(ss / (float)K + eps);
  auto put = [&](int c, const uint4& q, const uint4& g) {
    *reinterpret_cast<uint4*>(y + (y_tiled ? pf_toff(row, c * 8, K) : (size_t)row * K + c * 8)) = pf_norm8(q, r, g);
  };
  if constexpr (NP > 0) {
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if (lane + WAVE * i < nc) put(lane + WAVE * i, xv[i], wv[i]);
  } else {
    for (int c = lane; c < nc; c += WAVE) put(c, xr(c), ld(w + c * 8));
  }
}
template <bool X_TILED>
static void pf_rownorm(const bf16_t* x, const void* w, bf16_t* y, int M, int K, float eps, int y_tiled, int32_t* len, int len_to, hipStream_t st) {
#define PF_NORM(NP) hipLaunchKernelGGL((pf_rownorm_kernel<X_TILED, NP>), dim3((M + 3) / 4), dim3(256), 0, st, x, (const bf16_t*)w, y, M, K, eps, y_tiled, len, len_to)
  switch ((K / 8 + WAVE - 1) / WAVE) {
    case 1: PF_NORM(1); break;
    case 2: PF_NORM(2); break;
    case 3: PF_NORM(3); break;
    case 4: PF_NORM(4); break;
    default: PF_NORM(0);
  }
#undef PF_NORM
}

// The residual of the new positions.  Short block (ssq): tiled, with the sums of squares of every 16 columns of a row, and the
// attention's arrival counters cleared; otherwise row-major, and the values behind position L in the attention's copy cleared (their weights are zero).  8 columns per thread.
__global__ __launch_bounds__(256) void pf_begin_kernel(const bf16_t* __restrict__ emb, bf16_t* __restrict__ x, float* __restrict__ ssq,
                                                       bf16_t* __restrict__ vt, uint32_t* __restrict__ count, int n_count, int T, int d,
                                                       int nkv, int L, int Lpad) {
  const int i = blockIdx.x * 256 + threadIdx.x, per_row = d >> 3;
  if (i < n_count) count[i] = 0;
  if (i < T * per_row) {  // T d / 8 is a multiple of 8: both lanes of a pair are in
    const int t = i / per_row, k = (i - t * per_row) * 8;
    const uint4 v = *reinterpret_cast<const uint4*>(emb + (size_t)i * 8);
    if (ssq) {
      float f[8];
      El<bf16_t>::ld8(reinterpret_cast<const bf16_t*>(&v), f);
      float ss = ((f[0] * f[0] + f[1] * f[1]) + (f[2] * f[2] + f[3] * f[3])) + ((f[4] * f[4] + f[5] * f[5]) + (f[6] * f[6] + f[7] * f[7]));
      ss += dpp_f<DPP_QUAD_XOR1>(ss);
      if (!(k & 8)) ssq[(size_t)t * (d >> 4) + (k >> 4)] = ss;
      *reinterpret_cast<uint4*>(x + pf_toff(t, k, d)) = v;
    } else {
      *reinterpret_cast<uint4*>(x + (size_t)i * 8) = v;
    }
  }
  const int n = Lpad - L;
  if (vt && n > 0 && i < n * nkv) {  // dim by dim of all KV heads
    const int f = i / n, j = L + i - f * n;
    vt[((size_t)(f >> 4) * (Lpad >> 5) + (j >> 5)) * 512 + ((f & 15) + 16 * ((j & 15) >> 2)) * 8 + 4 * ((j & 31) >> 4) + (j & 3)] = 0;
  }
}

// Attention of the new positions against the row's cache without materialised scores: one workgroup per
// (16 queries, head), its waves (eight, four for head_dim 128) take 32 keys at a time in turn with a running maximum and sum each and
// meet in LDS at the end.  Per step: scores^T (keys x queries) = K q^T on the matrix cores, so that a lane holds
// eight keys of ONE query (its column) and the softmax bookkeeping is per lane plus a fold over the four lane
// rows; the probabilities, rounded to bf16, are then already in operand layout for out^T (dims x queries) =
// V^T p^T, with V^T read from the transposed copy in the same key order (any assignment of k to lanes is valid
// when both operands share it).  HD32 = head_dim / 32.
// Bound by the keys and values that every tile of queries fetches from L2 and by the instructions around the weights.
// Neighbouring workgroups take different heads, so that an XCD's L2 holds the keys and values of few (all heads together
// are 5.3 MB at eight heads of 96, 1733 positions); masks and the rescaling of the sums only in the steps that need them:
// 25.2 -> 19.0 us there, 9.4 -> 7.0 us at 576 positions.  Weights as powers of two, one fma and one v_exp_f32 each, took
// 16.3 / 6.3 us, but up to 2.7 times the error of expf against 64 bits (heads of 64, scores of deviation 12: 3.9e-7 against 1.4e-7).
// Two tiles of queries per wave or per workgroup, which halves the fetches, measured the same at 1733 and slower below.
#define PF_ATT_WAVES (HD32 <= 3 ? 8 : 4)  // the partial outputs of the waves must fit 64 KiB of LDS
template <int HD32>
__global__ __launch_bounds__(64 * PF_ATT_WAVES, 2) void pf_attn_kernel(const bf16_t* __restrict__ qr, const bf16_t* __restrict__ kt,
                                                      const bf16_t* __restrict__ vt, bf16_t* __restrict__ att, int T, int ldq,
                                                      int Lpad, int nq, int gsz, int pos0, int window, float scale) {
  constexpr int HD = 32 * HD32, DT = 2 * HD32;
  __shared__ float s_acc[PF_ATT_WAVES][DT * 256];
  __shared__ float s_m[PF_ATT_WAVES][16], s_l[PF_ATT_WAVES][16];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l16 = lane & 15, kg = lane >> 4;
  // neighbouring workgroups take different KV heads (one XCD meets few of them); the tiles with the most keys start first
  const int nkvh = gridDim.x / gsz, kvh = blockIdx.x % nkvh, h = kvh * gsz + blockIdx.x / nkvh;
  const int q0 = (gridDim.y - 1 - blockIdx.y) * 16;
  // this lane's query (column of every product below)
  const int tq = min(q0 + l16, T - 1);
  const int qlast = pos0 + tq;                                   // last visible key
  const int qfirst = window > 0 ? max(0, qlast - window) : 0;   // first visible key
  uint4 qf[HD32];
#pragma unroll
  for (int c = 0; c < HD32; ++c)
    qf[c] = *reinterpret_cast<const uint4*>(qr + (size_t)tq * ldq + h * HD + c * 32 + kg * 8);
  // keys any query of the tile can see
  const int t_hi = min(q0 + 15, T - 1);
  const int kend = pos0 + t_hi + 1;
  const int kbeg = (window > 0 ? max(0, pos0 + q0 - window) : 0) & ~31;
  // steps that start in [kall, kmid) are visible to every query of the tile
  const int kall = window > 0 ? max(0, pos0 + t_hi - window) : 0, kmid = pos0 + q0 - 30;
  // staged keys / values of this KV head (pf_stage_kv_kernel): a fragment is 16 bytes per lane, 1 KiB contiguous per wave
  const bf16_t* kb = kt + (size_t)kvh * (Lpad >> 4) * HD32 * 512 + lane * 8;
  const bf16_t* vb = vt + (size_t)kvh * DT * (Lpad >> 5) * 512 + lane * 8;

  pf_floatx4 acc[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) acc[d] = pf_floatx4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;
  for (int k0 = kbeg + 32 * wave; k0 < kend; k0 += 32 * PF_ATT_WAVES) {
    // every load of the step goes out before the first product (keys and values alike: the values do not depend
    // on the scores), so a step is one trip to memory
    uint4 kf[2][HD32], vf[DT];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int c = 0; c < HD32; ++c)
        kf[kt][c] = *reinterpret_cast<const uint4*>(kb + ((size_t)((k0 >> 4) + kt) * HD32 + c) * 512);
    // V^T of dims 16 d + l16: the lane's eight keys k0 + 4 kg + r and k0 + 16 + 4 kg + r, in the order of its scores
#pragma unroll
    for (int d = 0; d < DT; ++d) vf[d] = *reinterpret_cast<const uint4*>(vb + ((size_t)d * (Lpad >> 5) + (k0 >> 5)) * 512);
    __builtin_amdgcn_sched_barrier(0);
    // scores^T of 32 keys: two tiles of 16 keys x 16 queries
    pf_floatx4 sc[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      sc[kt] = pf_floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < HD32; ++c)
        sc[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf_frag(kf[kt][c]), pf_frag(qf[c]), sc[kt], 0, 0, 0);
    }
    // the lane holds keys k0 + 16 kt + 4 kg + r of its query
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int r = 0; r < 4; ++r) sc[kt][r] *= scale;
    if (k0 < kall || k0 >= kmid) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = k0 + 16 * kt + 4 * kg + r;
          if (j < qfirst || j > qlast) sc[kt][r] = -INFINITY;
        }
    }
    float mx = fmaxf(sc[0][0], sc[1][0]);
#pragma unroll
    for (int r = 1; r < 4; ++r) mx = fmaxf(mx, fmaxf(sc[0][r], sc[1][r]));
    mx = rows_max(mx);  // over the four lane rows: every key of the step for this query
    const float m_new = fmaxf(m_run, mx);
    const float m_use = (m_new == -INFINITY) ? 0.f : m_new;  // nothing visible yet: every weight below is zero
    const float alpha = expf(m_run - m_use);                  // 0 on the first visible step (m_run = -inf)
    float pv[8], ps = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) { pv[e] = expf(sc[e >> 2][e & 3] - m_use); ps += pv[e]; }
    l_run = l_run * alpha + ps;
    m_run = m_new;
    uint4 pf;
    pf.x = f2bf2(pv[0], pv[1]); pf.y = f2bf2(pv[2], pv[3]); pf.z = f2bf2(pv[4], pv[5]); pf.w = f2bf2(pv[6], pv[7]);
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {  // few steps raise a maximum
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[d][r] *= alpha;
    }
#pragma unroll
    for (int d = 0; d < DT; ++d) acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf_frag(vf[d]), pf_frag(pf), acc[d], 0, 0, 0);
  }
  // the waves' parts meet: lane holds dims 16 d + 4 kg + r of query l16
  l_run = rows_sum(l_run);
  if (kg == 0) { s_m[wave][l16] = m_run; s_l[wave][l16] = l_run; }
#pragma unroll
  for (int d = 0; d < DT; ++d) *reinterpret_cast<pf_floatx4*>(&s_acc[wave][(d * 64 + lane) * 4]) = acc[d];
  __syncthreads();
  for (int sl = tid; sl < DT * 64; sl += 64 * PF_ATT_WAVES) {
    const int d = sl >> 6, ln = sl & 63, q = ln & 15, g4 = ln >> 4;
    const int t = q0 + q;
    if (t >= T) continue;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < PF_ATT_WAVES; ++w) M = fmaxf(M, s_m[w][q]);
    float den = 0.f, o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < PF_ATT_WAVES; ++w) {
      const float f = (s_m[w][q] == -INFINITY) ? 0.f : expf(s_m[w][q] - M);
      den = fmaf(f, s_l[w][q], den);
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = fmaf(f, s_acc[w][sl * 4 + r], o[r]);
    }
    const float inv = 1.0f / den;
    bf16_t* dst = att + pf_toff(t, h * HD + 16 * d + 4 * g4, nq);  // tiled: operand of out_proj
    *reinterpret_cast<uint2*>(dst) = make_uint2(f2bf2(o[0] * inv, o[1] * inv), f2bf2(o[2] * inv, o[3] * inv));
  }
}

// The same attention for short blocks: keys and values come from the cache rows themselves.  A short block is one tile of
// queries per head or a few, so each cached value is fetched once or twice and a copy in operand layout costs more than it saves
// (4.8 us of 37 per layer for that launch alone).  A key fragment is 16 bytes of 16 rows (64 contiguous bytes each); values go through
// a wave's own 32 x HD share of LDS and come back transposed (ds_read_b64_tr_b16: 16 lanes read 4 rows of 16, lane i
// receives column i).  Bound by what one compute unit can fetch, so the keys of a (head, tile) are dealt to up to PF_SPLITS
// workgroups of four waves, 128 keys (a step of 32 per wave) for each as far as that reaches; the last one to arrive merges their parts.
// Whole pass of 16 positions behind 600 / 2000, us: by a staged copy 777 / 964; here with 8 splits of four waves 644 / 704 (with the
// cache read ahead, see pf_warm, 635 / 695), of eight waves and 256 keys 678 / 712, one workgroup of sixteen waves 830 / 1043.
#define PF_SPLITS 8
template <int HD32> struct PfDirect {
  static constexpr int HD = 32 * HD32, DT = 2 * HD32, WAVES = 4;
  static constexpr size_t VB = (size_t)WAVES * 32 * HD * 2, ML = (size_t)WAVES * 16 * 4;  // VB = WAVES * DT * 1024: the waves' parts
  static constexpr size_t LDS = VB + 2 * ML + 16;
};
struct PfDirectArgs {
  const bf16_t *q, *kc, *vc;
  bf16_t* att;
  int T, nq, nkv, gsz, pos0, window;
  float scale;
  float *part, *ml;  // (head, tile, split): sums (DT x 64 lanes x 4), {max, sum of weights} x 16
  uint32_t* count;   // arrivals of a (head, tile) in the pass; `before`: those of earlier layers (their splits differ: windows)
  uint32_t before;
  int nsp;           // splits; workgroups of higher blockIdx.z read ahead: `n_ahead` matrices, one behind the other
  const char* ahead;
  uint32_t ahead_bytes[5];
  int n_ahead;
};
// A short block's products wait for their weights (1-2 us of launches of 3-5), and its attention leaves most compute units idle: workgroups of its
// launch read the weights of the products up to the next attention into the L2s that will ask for them.  L2s keep what they hold
// from launch to launch; pf_order deals an eighth of a matrix's features to an XCD, and workgroup i is on XCD i % 8.  Measured, a whole prompt on
// the device, us without / with: bf16, an empty slot's 5, 16, 24 and 60 positions 491 / 480, 512 / 484, 591 / 549, 656 / 612, 16 behind 100, 700 and 2000
// cached ones 528 / 482, 580 / 517, 627 / 576; int8 (half the bytes) 434 / 440, 450 / 455, 533 / 543, 587 / 585, 467 / 465, 517 / 515, 594 / 592, 40 behind 2000
// 725 / 704, sixteen rows 549 / 549: nothing on average, 2 % lost at most and 3 % gained, so that the type makes no rule.  A vocoder on another stream loses
// nothing by what its L2s held: 16 behind 700 and six streamed frames beside each other 620 / 561 and 5046 / 4830, in int8 565 / 555 and 4833 / 4810.  No more
// than PF_AHEAD_BYTES: the L2s of a card hold 32 MB, and what does not stay is read twice.
// Workgroups per XCD, 20 / 32 / 48: an empty slot's 9, 23 and 60 positions in bf16 537 / 514 / 520, 604 / 569 / 562, 658 / 612 / 611 us, four turns behind
// 700 7204 / 7128 / 7129, sixteen in int8 14.95 / 14.96 / 15.09 ms.
#define PF_AHEAD 32
#define PF_AHEAD_BYTES (24u << 20)
__device__ __forceinline__ void pf_ahead(const PfDirectArgs& a) {
  const uint32_t plane = gridDim.x * gridDim.y, first = plane * a.nsp, i = blockIdx.x + gridDim.x * blockIdx.y + plane * blockIdx.z, x = i & 7u;
  const uint32_t lead = first + ((x - first) & 7u), mine = (i - lead) >> 3, all = ((plane * gridDim.z - 1 - lead) >> 3) + 1;  // of the XCD's readers
  const char* base = a.ahead;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    if (k >= a.n_ahead) break;
    const uint32_t n = a.ahead_bytes[k] >> 4, lo = (uint32_t)((uint64_t)n * x >> 3), hi = (uint32_t)((uint64_t)n * (x + 1) >> 3);  // in pieces of 16 bytes
    const uint4* src = reinterpret_cast<const uint4*>(base);
    for (uint32_t at = lo + mine * 4 * blockDim.x + threadIdx.x; at < hi; at += all * 4 * blockDim.x) {
      uint4 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = src[min(at + u * blockDim.x, hi - 1)];
#pragma unroll
      for (int u = 0; u < 4; ++u) asm volatile("" ::"v"(v[u].x));
    }
    base += a.ahead_bytes[k];
  }
}
template <int HD32>
__global__ __launch_bounds__(64 * PfDirect<HD32>::WAVES) void pf_direct_attn_kernel(const bf16_t* q, const bf16_t* kc, const bf16_t* vc, int T, int nq,
                                                                                    int nkv, int gsz, int pos0, int window, const PfDirectArgs a0) {
  PfDirectArgs a = a0;
  a.q = q; a.kc = kc; a.vc = vc; a.T = T; a.nq = nq; a.nkv = nkv; a.gsz = gsz; a.pos0 = pos0; a.window = window;  // (see PF_HOT)
  typedef PfDirect<HD32> P;
  constexpr int HD = P::HD, DT = P::DT, WAVES = P::WAVES;
  extern __shared__ __align__(16) char lds[];
  if ((int)blockIdx.z >= a.nsp) { pf_ahead(a); return; }
  float* s_m = (float*)(lds + P::VB);
  float* s_l = (float*)(lds + P::VB + P::ML);
  uint32_t* s_last = (uint32_t*)(lds + P::VB + 2 * P::ML);
  float* s_acc = (float*)lds;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l16 = lane & 15, kg = lane >> 4;
  const int h = blockIdx.x, kvh = h / a.gsz, q0 = blockIdx.y * 16, sp = blockIdx.z, nsp = a.nsp;
  const int tq = min(q0 + l16, a.T - 1);
  const int qlast = a.pos0 + tq, qfirst = a.window > 0 ? max(0, qlast - a.window) : 0;  // visible keys of this lane's query
  const int t_hi = min(q0 + 15, a.T - 1);
  const int kend = a.pos0 + t_hi + 1, kbeg = (a.window > 0 ? max(0, a.pos0 + q0 - a.window) : 0) & ~31;
  const int per = ((kend - kbeg + 31) / 32 + nsp - 1) / nsp * 32, lo = kbeg + sp * per, hi = min(lo + per, kend);
  uint4 qf[HD32];
#pragma unroll
  for (int c = 0; c < HD32; ++c) qf[c] = *reinterpret_cast<const uint4*>(a.q + (size_t)tq * a.nq + h * HD + c * 32 + kg * 8);
  const bf16_t* kb = a.kc + kvh * HD + kg * 8;
  const bf16_t* vb = a.vc + kvh * HD;
  char* own = lds + (size_t)wave * 32 * HD * 2;
  pf_floatx4 acc[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) acc[d] = pf_floatx4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;
  for (int k0 = lo + 32 * wave; k0 < hi; k0 += 32 * WAVES) {
    // a key behind the last visible one reads that one again; its weight is zero
    uint4 kf[2][HD32];
    tl_u32x4 vr[DT];  // native vectors: an array of HIP's structs stays in scratch memory
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int c = 0; c < HD32; ++c) kf[kt][c] = *reinterpret_cast<const uint4*>(kb + (size_t)min(k0 + 16 * kt + l16, kend - 1) * a.nkv + c * 32);
#pragma unroll
    for (int i = 0; i < DT; ++i) {  // 32 rows of HD values, in the order of LDS
      const int e = i * 512 + lane * 8, row = e / HD;
      vr[i] = *reinterpret_cast<const tl_u32x4*>(vb + (size_t)min(k0 + row, kend - 1) * a.nkv + (e - row * HD));
    }
    __builtin_amdgcn_sched_barrier(0);
    pf_floatx4 sc[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      sc[kt] = pf_floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < HD32; ++c) sc[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf_frag(kf[kt][c]), pf_frag(qf[c]), sc[kt], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < DT; ++i) *reinterpret_cast<tl_u32x4*>(own + i * 1024 + lane * 16) = vr[i];
    float mx = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = k0 + 16 * kt + 4 * kg + r;
        sc[kt][r] = (j < qfirst || j > qlast) ? -INFINITY : sc[kt][r] * a.scale;
        mx = fmaxf(mx, sc[kt][r]);
      }
    mx = rows_max(mx);
    const float m_new = fmaxf(m_run, mx);
    const float m_use = (m_new == -INFINITY) ? 0.f : m_new;  // nothing visible yet: every weight below is zero
    const float alpha = expf(m_run - m_use);
    float pv[8], ps = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) { pv[e] = expf(sc[e >> 2][e & 3] - m_use); ps += pv[e]; }
    l_run = l_run * alpha + ps;
    m_run = m_new;
    uint4 pf;
    pf.x = f2bf2(pv[0], pv[1]); pf.y = f2bf2(pv[2], pv[3]); pf.z = f2bf2(pv[4], pv[5]); pf.w = f2bf2(pv[6], pv[7]);
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[d][r] *= alpha;
    // V^T of dims 16 d + l16: keys 4 kg + r and 16 + 4 kg + r, in the order of the lane's scores
    const char* vrow = own + (4 * kg + (l16 >> 2)) * (HD * 2) + (l16 & 3) * 8;
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      const uint2 x = tl_read_tr(vrow + d * 32), y = tl_read_tr(vrow + 16 * HD * 2 + d * 32);
      acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf_frag(make_uint4(x.x, x.y, y.x, y.y)), pf_frag(pf), acc[d], 0, 0, 0);
    }
  }
  l_run = rows_sum(l_run);
  if (kg == 0) { s_m[wave * 16 + l16] = m_run; s_l[wave * 16 + l16] = l_run; }
  __syncthreads();  // the shares of the values become the waves' parts
#pragma unroll
  for (int d = 0; d < DT; ++d) *reinterpret_cast<pf_floatx4*>(&s_acc[((wave * DT + d) * 64 + lane) * 4]) = acc[d];
  __syncthreads();
  // blocks d = wave, wave + WAVES, ...: dims 16 d + 4 kg + r of query l16
  constexpr int ND = (DT + WAVES - 1) / WAVES;
  float M = -INFINITY, den = 0.f, o[ND][4] = {};
#pragma unroll
  for (int w = 0; w < WAVES; ++w) M = fmaxf(M, s_m[w * 16 + l16]);
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    const float m = s_m[w * 16 + l16], f = (m == -INFINITY) ? 0.f : expf(m - M);
    den = fmaf(f, s_l[w * 16 + l16], den);
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      const pf_floatx4 x = *reinterpret_cast<const pf_floatx4*>(&s_acc[((w * DT + min(wave + i * WAVES, DT - 1)) * 64 + lane) * 4]);
#pragma unroll
      for (int r = 0; r < 4; ++r) o[i][r] = fmaf(f, x[r], o[i][r]);
    }
  }
  if (nsp > 1) {
    const size_t set = (size_t)h * gridDim.y + blockIdx.y;
    const __amdgpu_buffer_rsrc_t part = dev_buffer(a.part + set * nsp * (DT * 256), (uint32_t)(nsp * DT * 1024));
    float* ml = a.ml + set * nsp * 32;
#pragma unroll
    for (int i = 0; i < ND; ++i)
      if (wave + i * WAVES < DT) st_dev4(part, (uint32_t)(((sp * DT + wave + i * WAVES) * 64 + lane) * 16), o[i]);
    if (tid < 16) st_dev(ml + sp * 32 + tid * 2, M, den);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) *s_last = __hip_atomic_fetch_add(a.count + set, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.before + nsp - 1;
    __syncthreads();
    if (!*s_last) return;
    // One compute unit takes in all parts, which is what this tail waits for: whole lines, and nothing for splits and blocks that are not
    // there.  (Eight bytes at a time of eight splits however many there are: 9.1 us per launch of 16 positions behind 700, so 8.4.)
    uint64_t xm[PF_SPLITS];
    dev_f32x4 xo[ND][PF_SPLITS];
#pragma unroll
    for (int s = 0; s < PF_SPLITS; ++s) {
      xm[s] = ld_dev(ml + min(s, nsp - 1) * 32 + l16 * 2);
#pragma unroll
      for (int i = 0; i < ND; ++i)
        xo[i][s] = ld_dev4(part, wave + i * WAVES < DT ? (uint32_t)(((s * DT + wave + i * WAVES) * 64 + lane) * 16) : DEV_NOWHERE);
    }
    M = -INFINITY;
#pragma unroll
    for (int s = 0; s < PF_SPLITS; ++s) M = fmaxf(M, lo_f(xm[s]));
    den = 0.f;
#pragma unroll
    for (int i = 0; i < ND; ++i) o[i][0] = o[i][1] = o[i][2] = o[i][3] = 0.f;
#pragma unroll
    for (int s = 0; s < PF_SPLITS; ++s) {
      const float m = lo_f(xm[s]), f = (s >= nsp || m == -INFINITY) ? 0.f : expf(m - M);
      den = fmaf(f, hi_f(xm[s]), den);
#pragma unroll
      for (int i = 0; i < ND; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) o[i][r] = fmaf(f, xo[i][s][r], o[i][r]);
      }
    }
  }
  const int t = q0 + l16;
  const float inv = 1.0f / den;
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    const int d = wave + i * WAVES;
    if (d < DT && t < a.T)
      *reinterpret_cast<uint2*>(a.att + pf_toff(t, h * HD + 16 * d + 4 * kg, a.nq)) =
          make_uint2(f2bf2(o[i][0] * inv, o[i][1] * inv), f2bf2(o[i][2] * inv, o[i][3] * inv));
  }
}
template <int HD32> static int pf_direct_attn(PfDirectArgs& a, int H, hipStream_t st) {
  constexpr size_t lds = PfDirect<HD32>::LDS;
  const int L = a.pos0 + a.T, keys = a.window > 0 && a.window + 48 < L ? a.window + 48 : L, n = (keys + 127) / 128;
  HIP_TRY(hipFuncSetAttribute((const void*)pf_direct_attn_kernel<HD32>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  const int splits = n > PF_SPLITS ? PF_SPLITS : n;
  a.nsp = splits;
  const int plane = H * ((a.T + 15) / 16), readers = (8 * PF_AHEAD + plane - 1) / plane;
  hipLaunchKernelGGL(pf_direct_attn_kernel<HD32>, dim3(H, (a.T + 15) / 16, splits + readers), dim3(64 * PfDirect<HD32>::WAVES), lds, st, a.q, a.kc, a.vc, a.T, a.nq,
                     a.nkv, a.gsz, a.pos0, a.window, a);
  if (splits > 1) a.before += splits;
  return VUI_OK;
}

// The cached keys and values before position L of one slot in the operand layouts of pf_attn_kernel (in a pass that starts an empty
// slot the QKV product's epilogue writes them).
// Keys of KV head g: blocks of 16 keys x 32 dims, block ((g * Lpad / 16 + j / 16) * hd / 32 + dim / 32) of 512
// elements, lane (j % 16) + 16 * ((dim % 32) / 8) holds its 8 dims at 8 * lane.  Values, transposed: blocks of 16
// dims x 32 keys, block ((g * hd / 16 + dim / 16) * Lpad / 32 + j / 32), lane (dim % 16) + 16 * ((j % 16) / 4)
// holds keys j % 4 of both halves (j % 32) / 16 of the step at 8 * lane + 4 * half + j % 4 - the order in which a
// lane of the attention kernel holds the scores of a step.  One workgroup: 32 keys x 32 features.
__global__ __launch_bounds__(256) void pf_stage_kv_kernel(const bf16_t* __restrict__ kc, const bf16_t* __restrict__ vc,
                                                          bf16_t* __restrict__ kt, bf16_t* __restrict__ vt, int L, int Lpad, int nkv, int hd) {
  __shared__ bf16_t tile[32][34];
  const int tid = threadIdx.x;
  const int j0 = blockIdx.x * 32, f0 = blockIdx.y * 32;  // f over nkv (= KV * hd); hd is a multiple of 32
  const int g = f0 / hd, dim0 = f0 % hd;
  if (tid < 128) {  // keys: 32 keys x four 8-dim pieces
    const int key = tid >> 2, pc = tid & 3, j = j0 + key;
    if (j < L) {
      const size_t blk = ((size_t)g * (Lpad >> 4) + (j >> 4)) * (hd >> 5) + (dim0 >> 5);
      *reinterpret_cast<uint4*>(kt + blk * 512 + ((j & 15) + 16 * pc) * 8) = *reinterpret_cast<const uint4*>(kc + (size_t)j * nkv + f0 + pc * 8);
    }
  }
  {
    const int tx = tid & 31, ty = tid >> 5;  // 32 x 8
    for (int r = ty; r < 32; r += 8) tile[r][tx] = vc[(size_t)min(j0 + r, L - 1) * nkv + f0 + tx];
  }
  __syncthreads();
  {
    // thread: dim dl of the 32, piece q = 4 * half + key group: four consecutive keys
    const int dl = tid >> 3, q = tid & 7, half = q >> 2, kgk = q & 3;
    const int dim = dim0 + dl;
    const int jj = half * 16 + kgk * 4;
    const size_t blk = ((size_t)g * (hd >> 4) + (dim >> 4)) * (Lpad >> 5) + (j0 >> 5);
    bf16_t* dst = vt + blk * 512 + ((dim & 15) + 16 * kgk) * 8 + 4 * half;
    if (j0 + jj + 3 < L) {
      const uint32_t lo = (uint32_t)tile[jj][dl] | ((uint32_t)tile[jj + 1][dl] << 16);
      const uint32_t hi = (uint32_t)tile[jj + 2][dl] | ((uint32_t)tile[jj + 3][dl] << 16);
      *reinterpret_cast<uint2*>(dst) = make_uint2(lo, hi);
    } else {
      for (int r = 0; r < 4; ++r) if (j0 + jj + r < L) dst[r] = tile[jj + r][dl];
    }
  }
}

// The form of a product of M rows (pair: two matrices of N features): estimated microseconds of the large tiles - a launch,
// and per step of 32 columns `wait` or `work` for each round of 256 tiles - and of the K-splitting form, whose time follows its
// trips to memory and its tiles; with an odd number of row tiles every XCD meets all rows, which costs where they exceed
// its L2.  Up to 256 tiles of 32 x 32 the K-splitting form runs with more waves and is quicker.
// Fitted to 384 products (130 ... 2048 rows, widths 512, 768, 1024, bf16 and int8, weights of 22 layers in turn): on average 2 %
// above the best form of each and 6 % below K-splitting alone; 6 products are more than 5 % above that, 19 % at most.
// The bf16 forms once more, beside each other in whole prompts of 200 ... 2048 positions at widths 512, 768 and 1024: of 204 products the form
// taken was 0.58 us above the quickest on average and is 0.1 now.  Prompts of width 768 with that and the norms' one trip, us: 1000 1514 -> 1450, 1500 1970 -> 1810, 1733 2091 -> 1970.
// us, K-splitting / 128 x 128 / 64 x 128 / 64 x 64, bf16 at width 768: W1 and W3 at 577 rows 13.3 / 13.5 / 14.5 / 14.0, at 1000
// 16.9 / 14.0 / 13.7 / 16.4, at 1733 25.3 / 19.3 / 22.7 / 25.6; W2 at 577 10.6 / 26.2 / 17.3 / 12.0, at 1733 29.4 / 26.3 / 17.6 / 17.8.
static int pf_pick(int M, int N, int K, bool pair, bool i8) {
  static const struct { int bm, bn; double base[2], wait[2], work[2]; } tile[] = {  // of bf16 and int8 weights
      {128, 128, {6.37, 7.3}, {0.393, 0.325}, {0.199, 0.274}},
      {64, 128, {5.63, 5.3}, {0.24, 0.204}, {0.171, 0.181}},
      {64, 64, {3.25, 4.8}, {0.163, 0.141}, {0.136, 0.112}}};
  static const double part[2] = {0.6, 0};  // of what a last round's missing tiles would take is saved: the others' workgroups end one by one
  static const struct { double base, k256, tile, over; } split[2] = {{2.75, 0.635, 0.233e-3, 2.08e-6}, {4.3, 0.146, 0.262e-3, 0.44e-6}};
  const long rows = (M + 31) / 32;
  if (M < 128 || K < 256 || rows * ((N + 31) / 32) <= 256) return WIDE_NONE;
  if (pair) N *= 2;
  int best = WIDE_NONE;
  double us = split[i8].base + split[i8].k256 * (K / 256.0) + split[i8].tile * rows * ((N + 31) / 32) * (K / 64);
  const double over = 2.0 * M * K - 3e6;
  if ((rows & 1) && over > 0) us += split[i8].over * over;
  for (int i = 0; i < 3; ++i) {
    const long tiles = (long)((M + tile[i].bm - 1) / tile[i].bm) * ((N + tile[i].bn - 1) / tile[i].bn), rounds = (tiles + 255) / 256;
    const double work = (rounds == 1 ? 1.0 : part[i8] * tiles / 256 + (1 - part[i8]) * rounds) * tile[i].work[i8], c = tile[i].base[i8] + (K / 32) * (work > tile[i].wait[i8] ? work : tile[i].wait[i8]);
    if (c < us) { best = i; us = c; }
  }
  return best;
}

// bf16 out, K split over the waves of a workgroup; DUAL: the SwiGLU pair, its second matrix behind g.W; i8: int8 matrices with g.sc / g.sc2;
// g.ssq != nullptr: rows are normed on their way (short blocks)
template <int EPI, bool DUAL, bool I8>
static int pf_go(PfGemm& g, hipStream_t st) {
  // Few tiles (short blocks): more waves, so that a wave's chain of dependent trips is one to three steps long, and 16
  // features per workgroup, so that more of the chip pulls weights.  us per launch, 32 x 32 and 4 waves / as chosen here:
  // 16 positions out_proj and W2 8.0 / 4.4, QKV 5.6 / 3.8, W1 and W3 5.9 / 5.0; whole pass of 16 positions 883 / 776
  // (int8 902 / 745), of 230 positions 1069 / 1060 (1013 / 931).
  const long t32 = (long)((g.M + 31) / 32) * ((g.N + 31) / 32);
  const bool norm = g.ssq != nullptr, some = t32 <= 256 && g.K >= 512, few = norm || (some && t32 <= 128);
  const int mb = few && g.M <= 16 ? 1 : 2, nb = few ? 1 : 2;
  const unsigned tiles = pf_set_order(g, 16 * mb, 16 * nb, (size_t)g.N * g.K * ((DUAL ? 2 : 1) * (I8 ? 1 : 2))) + g.warm;
  constexpr int W = EPI == PF_RESID ? 16 : 12;
#define PF_GO(WV, MB, NB, NORM) hipLaunchKernelGGL((pf_gemm_kernel<EPI, DUAL, I8, WV, MB, NB, NORM>), dim3(tiles), dim3(64 * (WV)), 0, st, PF_HOT_ARGS(g, EPI == PF_RESID ? (const void*)g.C : (const void*)g.ssq), g)
  if constexpr (EPI != PF_RESID) {
    if (norm) {
      // More tiles than CUs: eight waves, of which two workgroups fit a CU (33 ... 64 rows x 2304 features, 288 tiles: 11.1 -> 8.3 us; of twelve
      // waves each 32 CUs would take a second round alone)
      if (mb == 1) PF_GO(W, 1, 1, true);
      else if (g.n_tiles > 256) PF_GO(8, 2, 1, true);
      else PF_GO(W, 2, 1, true);
      HIP_TRY(hipGetLastError());
      return VUI_OK;
    }
  }
  if (few && mb == 1) PF_GO(W, 1, 1, false);
  else if (few) PF_GO(W, 2, 1, false);
  else if (some) PF_GO((DUAL ? 8 : 12), 2, 2, false);
  else PF_GO(4, 2, 2, false);
#undef PF_GO
  HIP_TRY(hipGetLastError());
  return VUI_OK;
}
template <int EPI, bool DUAL>
static int pf_gemm4(PfGemm& g, bool i8, hipStream_t st) {
  if (g.K % 64 || g.N % 16 || g.M < 1 || g.N < 1 || g.N >= 1 << 20 || g.K >= 1 << 21 || (g.c_tiled && g.N % 64)) { vui_set_error("prefill GEMM: bad shape N=%d K=%d", g.N, g.K); return VUI_EINVAL; }
  const int tile = g.ssq ? WIDE_NONE : pf_pick(g.M, g.N, g.K, DUAL, i8);
  if (tile != WIDE_NONE) return i8 ? pf_wide<EPI, DUAL, true>(tile, g, st) : pf_wide<EPI, DUAL, false>(tile, g, st);
  return i8 ? pf_go<EPI, DUAL, true>(g, st) : pf_go<EPI, DUAL, false>(g, st);
}

// Blocks of up to this many positions take the five-launch form.
// Whole pass, us, 65 positions in the long form / in this: bf16 738 / 800, behind 600 912 / 907, behind 2000 1063 / 1071; 100 positions
// 752 / 905; 64 positions in this form 724, 835, 899 (all by eight launches with a staged copy: 796, 882, 1034).
#define PF_SHORT 64
#define PF_WARM 64

static size_t pf_align(size_t b) { return (b + 255) & ~(size_t)255; }

// (head, tile of queries) pairs of a short block
static size_t pf_sets(const vui_config& c, int T) { return T <= PF_SHORT ? (size_t)c.n_heads * ((T + 15) / 16) : 0; }
// scratch: residual x, its sums of squares, normed xn, queries, attention output, FFN buffer, staged keys and values
size_t prefill_scratch_bytes(const vui_config& c, int T, int L) {
  const size_t d = c.d_model, nq = (size_t)c.n_heads * c.head_dim, nkv = (size_t)c.n_kv_heads * c.head_dim;
  const size_t Lpad = ((size_t)L + 63) & ~(size_t)63;
  const size_t T16 = ((size_t)T + 15) & ~(size_t)15;  // tiled operands come in blocks of 16 rows
  size_t b = 0;
  b += pf_align(T16 * d * 2) * 2 + pf_align(T16 * (d / 16) * 4);
  b += pf_align((size_t)T * nq * 2);
  b += pf_align(T16 * nq * 2);
  b += pf_align(T16 * c.ffn * 2);
  b += pf_align(nkv * Lpad * 2) * 2;
  const size_t sets = pf_sets(c, T);
  b += pf_align(sets * PF_SPLITS * 16 * c.head_dim * 4) + pf_align(sets * PF_SPLITS * 32 * 4) + pf_align(sets * 4);
  return b;
}

// elements of one layer's weights in tiled form (wqkv | wo | w1 | w3 | w2), and of all layers
static size_t pf_layer_elems(const vui_config& c) {
  const size_t d = c.d_model, nq = (size_t)c.n_heads * c.head_dim, nkv = (size_t)c.n_kv_heads * c.head_dim, F = c.ffn;
  return (nq + 2 * nkv) * d + d * nq + 2 * F * d + d * F;
}
// the pass's own tiled copy: bf16 matrices only (an int8 context reads the batched backbone kernel's tiled int8 copy)
size_t prefill_weight_bytes(const vui_config& c) {
  char why[96];
  return (!c.int8_backbone && prefill_supported(c, why, sizeof(why))) ? pf_layer_elems(c) * c.n_layers * 2 : 0;
}

// one-time: the layers' projection weights in the GEMMs' operand layout
int prefill_tile_weights(const vui_config& c, const vui_weights& w, void* dst, hipStream_t st) {
  const int d = c.d_model, nq = c.n_heads * c.head_dim, nkv = c.n_kv_heads * c.head_dim, F = c.ffn;
  bf16_t* o = (bf16_t*)dst;
  auto tile = [&](const void* src, int N, int K) {
    const size_t pieces = (size_t)N * (K / 8);
    hipLaunchKernelGGL(pf_tile_kernel, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, st, (const bf16_t*)src, o, N, K);
    o += (size_t)N * K;
  };
  for (int l = 0; l < c.n_layers; ++l) {
    const vui_layer_weights& lw = w.layers[l];
    tile(lw.wqkv, nq + 2 * nkv, d);
    tile(lw.wo, d, nq);
    tile(lw.w1, F, d);
    tile(lw.w3, F, d);
    tile(lw.w2, d, F);
  }
  HIP_TRY(hipGetLastError());
  return VUI_OK;
}

bool prefill_supported(const vui_config& c, char* why, size_t why_len) {
  const char* r = nullptr;
  const int nkv = c.n_kv_heads * c.head_dim;
  if (c.dtype != VUI_DTYPE_BF16) r = "bf16 activations only";
  else if (c.int8_backbone && !bb_batch_weight_bytes(c, 256)) r = "int8 weights: no tiled int8 copy (it belongs to the batched backbone kernel, which does not take this configuration)";
  else if ((c.d_model % 64) || (c.ffn % 64) || ((c.n_heads * c.head_dim) % 64) || (c.head_dim % 32) || c.head_dim > 128 || (nkv % 8) || (c.rope_dim & 1))
    r = "d_model, heads x head_dim and ffn must be multiples of 64, head_dim a multiple of 32 up to 128";
  else if (c.n_kv_heads < 1 || c.n_heads % c.n_kv_heads) r = "heads must be a multiple of KV heads";
  if (r && why) snprintf(why, why_len, "%s", r);
  return r == nullptr;
}

int launch_prefill(const vui_config& c, const vui_weights& w, const void* tiled_w, const void* emb, int T, int slot, int pos0,
                   int32_t* seq_lens, void* k_cache, void* v_cache, void* out, void* scratch, size_t scratch_bytes, hipStream_t st) {
  const int d = c.d_model, H = c.n_heads, KV = c.n_kv_heads, hd = c.head_dim, F = c.ffn, S = c.max_seqlen;
  const int nq = H * hd, nkv = KV * hd, L = pos0 + T, Lpad = (L + 63) & ~63;
  char why[96];
  if (!prefill_supported(c, why, sizeof(why))) { vui_set_error("prefill: %s", why); return VUI_EINVAL; }
  if (T < 1 || pos0 < 0 || L > S) { vui_set_error("prefill: positions %d..%d outside the cache (S=%d)", pos0, L, S); return VUI_EINVAL; }
  if (slot < 0 || slot >= c.n_slots) { vui_set_error("prefill: slot %d outside [0,%d)", slot, c.n_slots); return VUI_EINVAL; }
  if (scratch_bytes < prefill_scratch_bytes(c, T, L)) { vui_set_error("prefill: scratch of %zu bytes, %zu needed", scratch_bytes, prefill_scratch_bytes(c, T, L)); return VUI_EINVAL; }
  if (!tiled_w) { vui_set_error("prefill: the context holds no tiled weights"); return VUI_EINVAL; }
  const size_t T16 = ((size_t)T + 15) & ~(size_t)15;
  char* sp = (char*)scratch;
  auto take = [&](size_t bytes) { char* r = sp; sp += pf_align(bytes); return r; };
  bf16_t* x = (bf16_t*)take(T16 * d * 2);                       // residual stream: row-major, of a short block tiled
  float* ssq = (float*)take(T16 * (d / 16) * 4);
  bf16_t* xn = (bf16_t*)take(T16 * d * 2);                      // normed rows, tiled (rows past T are never written:
  bf16_t* q = (bf16_t*)take((size_t)T * nq * 2);                //  what a GEMM reads there only reaches output rows it drops)
  bf16_t* att = (bf16_t*)take(T16 * nq * 2);                    // attention output, tiled
  bf16_t* fa = (bf16_t*)take(T16 * F * 2);                      // SwiGLU product, tiled
  bf16_t* kt = (bf16_t*)take((size_t)nkv * Lpad * 2);           // keys and values of the slot in the attention's layout
  bf16_t* vt = (bf16_t*)take((size_t)nkv * Lpad * 2);
  const bool tiny = T <= PF_SHORT;
  const size_t sets = pf_sets(c, T);
  float* part = (float*)take(sets * PF_SPLITS * 16 * hd * 4);   // parts of a short block's attention
  float* ml = (float*)take(sets * PF_SPLITS * 32 * 4);
  uint32_t* count = (uint32_t*)take(sets * 4);
  const bool i8 = c.int8_backbone != 0;
  const size_t slab = (size_t)c.n_slots * S * nkv, wsz = i8 ? 1 : 2;
  const float scale = 1.0f / sqrtf((float)hd);
  if ((uintptr_t)emb & 15) {  // a caller's view may start anywhere
    HIP_TRY(hipMemcpyAsync(xn, emb, (size_t)T * d * 2, hipMemcpyDeviceToDevice, st));
    emb = xn;
  }
  {
    size_t n = (size_t)T * (d / 8);
    const size_t more = tiny ? sets : (size_t)(Lpad - L) * nkv;
    if (more > n) n = more;
    hipLaunchKernelGGL(pf_begin_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, (const bf16_t*)emb, x,
                       tiny ? ssq : nullptr, tiny ? nullptr : vt, count, (int)sets, T, d, nkv, L, Lpad);
  }
  auto norm = [&](const void* w, bf16_t* y, int y_tiled, int32_t* len) {
    if (tiny) pf_rownorm<true>(x, w, y, T, d, c.norm_eps, y_tiled, len, L, st);
    else pf_rownorm<false>(x, w, y, T, d, c.norm_eps, y_tiled, len, L, st);
  };
  PfDirectArgs da = {q, nullptr, nullptr, att, T, nq, nkv, H / KV, pos0, 0, scale, part, ml, count};
  int rc;
  for (int l = 0; l < c.n_layers; ++l) {
    const vui_layer_weights& lw = w.layers[l];
    const char* t_qkv = (const char*)tiled_w + pf_layer_elems(c) * wsz * l;
    const char* t_o = t_qkv + (size_t)(nq + 2 * nkv) * d * wsz;
    const char* t_1 = t_o + (size_t)d * nq * wsz;
    const char* t_3 = t_1 + (size_t)F * d * wsz;
    const char* t_2 = t_3 + (size_t)F * d * wsz;
    PfGemm g{};
    g.X = tiny ? x : xn; g.W = t_qkv; g.C = q; g.M = T; g.N = nq + 2 * nkv; g.K = d; g.ldc = nq; g.sc = (const bf16_t*)lw.s_qkv;
    if (tiny) { g.ssq = ssq; g.nw = (const bf16_t*)lw.attn_norm; g.eps = c.norm_eps; }
    else norm(lw.attn_norm, xn, 1, nullptr);
    g.kc = (bf16_t*)k_cache + slab * l + (size_t)slot * S * nkv;
    g.vc = (bf16_t*)v_cache + slab * l + (size_t)slot * S * nkv;
    const int win = layer_window(c, l);
    if (!tiny && pos0 == 0) { g.kt = kt; g.vt = vt; }
    if (tiny && pos0 > 0) { g.warm_from = win > 0 && pos0 > win ? pos0 - win : 0; g.warm = PF_WARM; g.warm_gsz = H % 8 == 0 ? H / KV : 0; }
    g.rope = layer_rope(c, w, l, &g.rope_dim);
    g.nq = nq; g.nkv = nkv; g.hd = hd; g.inv_hd = pf_inv(hd); g.pos0 = pos0; g.Lpad = Lpad;
    if ((rc = pf_gemm4<PF_QKV, false>(g, i8, st))) return rc;
    if (tiny) {
      da.kc = g.kc; da.vc = g.vc; da.window = win;
      da.ahead = t_o;
      const size_t ff = (size_t)F * d * wsz, sizes[5] = {(size_t)d * nq * wsz, ff, ff, ff, (size_t)(nq + 2 * nkv) * d * wsz};  // the last: the next layer's
      size_t sum = 0;
      for (da.n_ahead = 0; da.n_ahead < (l + 1 < c.n_layers ? 5 : 4); ++da.n_ahead) {
        if ((sum += sizes[da.n_ahead]) > PF_AHEAD_BYTES) break;
        da.ahead_bytes[da.n_ahead] = (uint32_t)sizes[da.n_ahead];
      }
      switch (hd / 32) {
        case 1: rc = pf_direct_attn<1>(da, H, st); break;
        case 2: rc = pf_direct_attn<2>(da, H, st); break;
        case 3: rc = pf_direct_attn<3>(da, H, st); break;
        default: rc = pf_direct_attn<4>(da, H, st); break;
      }
      if (rc) return rc;
    } else {
      if (pos0 > 0)
        hipLaunchKernelGGL(pf_stage_kv_kernel, dim3((L + 31) / 32, nkv / 32), dim3(256), 0, st, g.kc, g.vc, kt, vt, L, Lpad, nkv, hd);
      const dim3 grid(H, (T + 15) / 16);
      switch (hd / 32) {
        case 1: hipLaunchKernelGGL(pf_attn_kernel<1>, grid, dim3(512), 0, st, q, kt, vt, att, T, nq, Lpad, nq, H / KV, pos0, win, scale); break;
        case 2: hipLaunchKernelGGL(pf_attn_kernel<2>, grid, dim3(512), 0, st, q, kt, vt, att, T, nq, Lpad, nq, H / KV, pos0, win, scale); break;
        case 3: hipLaunchKernelGGL(pf_attn_kernel<3>, grid, dim3(512), 0, st, q, kt, vt, att, T, nq, Lpad, nq, H / KV, pos0, win, scale); break;
        default: hipLaunchKernelGGL(pf_attn_kernel<4>, grid, dim3(256), 0, st, q, kt, vt, att, T, nq, Lpad, nq, H / KV, pos0, win, scale); break;
      }
    }
    PfGemm wo{};
    wo.X = att; wo.W = t_o; wo.C = x; wo.c_tiled = tiny; wo.M = T; wo.N = d; wo.K = nq; wo.sc = (const bf16_t*)lw.s_o;
    if (tiny) wo.ssq_out = ssq;
    if ((rc = pf_gemm4<PF_RESID, false>(wo, i8, st))) return rc;
    PfGemm f1{};
    f1.X = tiny ? x : xn; f1.W = t_1; f1.C = fa; f1.c_tiled = 1; f1.M = T; f1.N = F; f1.K = d; f1.sc = (const bf16_t*)lw.s_1; f1.sc2 = (const bf16_t*)lw.s_3;
    if (tiny) { f1.ssq = ssq; f1.nw = (const bf16_t*)lw.mlp_norm; f1.eps = c.norm_eps; }
    else norm(lw.mlp_norm, xn, 1, nullptr);
    if ((rc = pf_gemm4<PF_BF16, true>(f1, i8, st))) return rc;  // written tiled: operand of W2
    PfGemm f2{};
    f2.X = fa; f2.W = t_2; f2.C = x; f2.c_tiled = tiny; f2.M = T; f2.N = d; f2.K = F; f2.sc = (const bf16_t*)lw.s_2;
    if (tiny) f2.ssq_out = ssq;
    if ((rc = pf_gemm4<PF_RESID, false>(f2, i8, st))) return rc;
  }
  norm(w.final_norm, (bf16_t*)out, 0, seq_lens + slot);
  HIP_TRY(hipGetLastError());
  return VUI_OK;
}
