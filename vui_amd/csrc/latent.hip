// Latent attention: per position the cache holds one normed latent c (kv_rank) and one rotated key part (rot_dim)
// common to the heads; head h's key is W_uk[h] c and its value W_uv[h] c.
//
// Two forms of the same sums.  Few rows attend in the latent space: the query goes through W_uk[h]^T once
// (latent_query_kernel), scores are its products with the cached latents, the softmax average of the latents goes
// through W_uv[h] (latent_value_kernel); nothing per key and head is ever formed.  Long blocks of a prompt expand
// keys and values of the whole slot once per layer (lm_gemm.hip) and run latent_prefill_kernel on them.
//
// Caches are tiled rows (tile.h), so that 16 keys x 64 latent columns are an operand of the matrix cores as they lie.
#include "common.h"
#include "lm.h"
#include "tile.h"

// ---- norm of the new latents and append; one wave per row ----
template <typename T>
__device__ __forceinline__ void latent_append_row(const LatentArgs& p, int m) {
  const int lane = threadIdx.x & 63;
  const float* src = p.craw + (size_t)m * p.d.rank16;
  float ss = 0.f;
  for (int k = lane * 4; k < p.d.rank16; k += 256) {  // columns beyond kv_rank hold zeros
    const float4 v = *reinterpret_cast<const float4*>(src + k);
    ss += (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w);
  }
  ss = wave_sum(ss);
  const float r = 1.0f / sqrtf(ss / (float)p.rank + p.eps);
  const int2 at = lm_where(p.rows, m);
  const int slot = at.x, pos = at.y;
  if (pos < 0 || pos >= p.rows.S) return;
  T* dst = (T*)p.c_cache + (size_t)slot * p.d.s64 * p.d.rank64;
  for (int k = lane * 4; k < p.d.rank16; k += 256) {
    const float4 v = *reinterpret_cast<const float4*>(src + k);
    const float4 w = *reinterpret_cast<const float4*>(p.latent_norm + k);
    const float o[4] = {v.x * r * w.x, v.y * r * w.y, v.z * r * w.z, v.w * r * w.w};
    Tl<T>::st4(dst + tl_off<T>(pos, k, p.d.rank64), o);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void latent_append_kernel(const LatentArgs p) {
  const int m = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (m < p.M) latent_append_row<T>(p, m);
}

// ---- queries into the latent space: qlat[h] (M x rank) = qu[h] (M x dim) W_uk[h]; a wave owns 16 latent columns ----
template <typename T>
__global__ __launch_bounds__(256) void latent_query_kernel(const void* w_uk_t, const void* qu, const float* craw, size_t qu_z, int heads, int M, int dim64, int rank16,
                                                           const LatentArgs p0) {
  LatentArgs p = p0;  // what the first loads need is in registers (see lm_gemm.hip)
  p.w_uk_t = w_uk_t; p.qu = qu; p.craw = craw; p.qu_z = qu_z; p.heads = heads; p.M = M; p.d.dim64 = dim64; p.d.rank16 = rank16;
  constexpr int EP = Tl<T>::EP, P = 16 / EP;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int h = blockIdx.x, mt = blockIdx.z;
  if (h == p.heads) {  // the extra workgroups append the new latents
    for (int r = blockIdx.y * 4 + wave; r < 16; r += 4 * gridDim.y)
      if (mt * 16 + r < p.M) latent_append_row<T>(p, mt * 16 + r);
    return;
  }
  const int nb = blockIdx.y * 4 + wave;
  if (nb >= p.d.rank16 >> 4) return;
  const int nk = p.d.dim64 >> 6;
  const T* w = (const T*)p.w_uk_t + ((size_t)h * (p.d.rank16 >> 4) + nb) * nk * 1024 + lane * EP;
  const T* x = (const T*)p.qu + h * p.qu_z + (size_t)mt * nk * 1024 + lane * EP;
  tl_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < nk; ++k) {
    uint4 a[P], b[P];
#pragma unroll
    for (int i = 0; i < P; ++i) {
      a[i] = *reinterpret_cast<const uint4*>(w + (size_t)k * 1024 + 64 * EP * i);
      b[i] = *reinterpret_cast<const uint4*>(x + (size_t)k * 1024 + 64 * EP * i);
    }
#pragma unroll
    for (int i = 0; i < P; ++i) acc = Tl<T>::mma(a[i], b[i], acc);
  }
  const int m = mt * 16 + (lane & 15);
  if (m >= p.M) return;
  const float v[4] = {acc[0], acc[1], acc[2], acc[3]};
  Tl<T>::st4((T*)p.qlat + (size_t)m * p.d.heads16 * p.d.rank64 + tl_off<T>(h, nb * 16 + 4 * (lane >> 4), p.d.rank64), v);
}

// A row that sees len keys is cut into pieces of this many (whole 32-key tiles), at most ns of them.  With more than
// four rows a piece has two tiles at least: there are pieces enough, and fewer are merged faster.
__host__ __device__ __forceinline__ int latent_least(int M) { return M > 4 ? 64 : 32; }
__host__ __device__ __forceinline__ int latent_chunk(int len, int ns, int M) { return max(((len + ns - 1) / ns + 31) & ~31, latent_least(M)); }
// keys [lo, hi) of piece sp
__device__ __forceinline__ void latent_range(int len, int ns, int M, int sp, int& lo, int& hi) {
  const int chunk = latent_chunk(len, ns, M);
  lo = min(sp * chunk, len);
  hi = min(lo + chunk, len);
}

// ---- attention in the latent space, any sizes: one workgroup per (row, head, split); fp32 arithmetic ----
#define LAT_TILE 256
#define LAT_ACC 8  // latent columns per thread: kv_rank up to 2048
template <typename T>
__global__ __launch_bounds__(256) void latent_attn_kernel(const LatentArgs p) {
  extern __shared__ __align__(16) float lq[];  // query: rank64 + rot32
  __shared__ float sc[LAT_TILE];
  __shared__ float red[4], red2[4];
  constexpr int EP = Tl<T>::EP;
  const int m = blockIdx.x, h = blockIdx.y, sp = blockIdx.z, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int R = p.d.rank64, RR = p.d.rot32;
  const int2 at = lm_where(p.rows, m);
  const int slot = at.x, len = min(max(at.y + 1, 1), p.rows.S);
  int lo, hi;
  latent_range(len, p.n_splits, p.M, sp, lo, hi);
  if (lo >= hi) return;  // no such piece: latent_value_kernel does not look for it
  for (int k = tid; k < R + RR; k += 256)
    lq[k] = k < R ? (k < p.d.rank16 ? El<T>::ld((const T*)p.qlat + (size_t)m * p.d.heads16 * R + tl_off<T>(h, k, R)) : 0.f)
                  : (k - R < p.d.rot16 ? El<T>::ld((const T*)p.qr + h * p.qr_z + tl_off<T, 32>(m, k - R, RR)) : 0.f);
  const T* cc = (const T*)p.c_cache + (size_t)slot * p.d.s64 * R;
  const T* kc = (const T*)p.kr_cache + (size_t)slot * p.d.s64 * RR;
  float acc[LAT_ACC];
#pragma unroll
  for (int i = 0; i < LAT_ACC; ++i) acc[i] = 0.f;
  float M = -INFINITY, L = 0.f;
  __syncthreads();
  for (int j0 = lo; j0 < hi; j0 += LAT_TILE) {
    const int j = j0 + tid, nj = min(LAT_TILE, hi - j0);
    float s = -INFINITY;
    if (j < hi) {
      float d = 0.f;
      for (int k = 0; k < R; k += EP) {
        const T* q = cc + tl_off<T>(j, k, R);
#pragma unroll
        for (int e = 0; e < EP; ++e) d = fmaf(lq[k + e], El<T>::ld(q + e), d);
      }
      for (int k = 0; k < RR; k += EP) {
        const T* q = kc + tl_off<T, 32>(j, k, RR);
#pragma unroll
        for (int e = 0; e < EP; ++e) d = fmaf(lq[R + k + e], El<T>::ld(q + e), d);
      }
      s = d * p.scale;
    }
    const float wm = wave_max(s);
    if (lane == 0) red[wave] = wm;
    __syncthreads();
    const float mn = fmaxf(M, fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])));
    const float e = j < hi ? expf(s - mn) : 0.f;
    sc[tid] = e;
    const float ws = wave_sum(e);
    if (lane == 0) red2[wave] = ws;
    __syncthreads();
    const float al = expf(M - mn);
    L = L * al + ((red2[0] + red2[1]) + (red2[2] + red2[3]));
    M = mn;
#pragma unroll
    for (int i = 0; i < LAT_ACC; ++i) {
      const int col = tid + 256 * i;
      if (col < R) {
        float a = acc[i] * al;
        for (int k = 0; k < nj; ++k) a = fmaf(sc[k], El<T>::ld(cc + tl_off<T>(j0 + k, col, R)), a);
        acc[i] = a;
      }
    }
    __syncthreads();
  }
  const size_t piece = ((size_t)m * p.heads + h) * p.n_splits + sp;
  if (tid == 0) *reinterpret_cast<float2*>(p.part_ml + 2 * piece) = make_float2(M, L);
#pragma unroll
  for (int i = 0; i < LAT_ACC; ++i)
    if (tid + 256 * i < R) p.part[piece * R + tid + 256 * i] = acc[i];
}

// ---- attention in the latent space on the matrix cores (bf16): one workgroup per (row, 16 heads, split) ----
// All heads read the same latents, so 32 KT keys are staged in LDS once and serve 16 heads.  Scores^T (keys x heads) =
// [c | k_rot] [q_lat | q_rot]^T, the four waves dealing key tiles (and, KT = 1, half of the columns) between them; every wave then
// has all scores of its lane's head and averages a quarter of the latent columns: out^T (columns x heads) = C^T p^T,
// the weights as a bf16 pair (value and remainder).  The transposed operand comes from LDS by ds_read_b64_tr_b16.
// RK = rank64 / 64, RB = rot32 / 32.  Pieces of 32 keys (up to four rows) take KT = 1, longer ones two tiles side by side instead of one
// after the other.  Bound by its chain: length, keys, LDS, scores, LDS, weights, average.  8 heads of rank 512, 16 rows behind up to 1400
// keys, us per launch: queries of a head each, values element by element, tile by tile 10.9, so 8.8; 16 heads 13.6 / 9.0 (of it two tiles
// side by side 0.4 us).
template <int RK, int RB, int KT>
__global__ __launch_bounds__(256, 2) void latent_attn_mfma_kernel(int2* where, const void* c_cache, const void* kr_cache, const void* qlat, uint32_t m_ns,
                                                                  int S, int s64, int heads16, const LatentArgs p0) {
  LatentArgs p = p0;  // what the first loads need is in registers (see lm_gemm.hip)
  p.rows.where = where; p.c_cache = const_cast<void*>(c_cache); p.kr_cache = const_cast<void*>(kr_cache); p.qlat = const_cast<void*>(qlat);
  p.M = (int)(m_ns & 0xffffffu); p.n_splits = (int)(m_ns >> 24); p.rows.S = S; p.d.s64 = s64; p.d.heads16 = heads16;
  constexpr int CT = RK * 2048, RT = RB * 1024;  // elements of the staged tiles (32 keys)
  constexpr int NT = 2 * KT, BUFS = KT == 1 ? 2 : 1, BUF = KT * (CT + RT);
  extern __shared__ __align__(16) bf16_t tile[];  // BUFS x KT x (CT + RT)
  __shared__ __align__(16) float sco[4][64 * 4];
  const int m = blockIdx.x, sp = blockIdx.z, tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l16 = lane & 15, kg = lane >> 4;
  const int t = wave % NT, half = wave / NT;  // KT = 2: every wave takes both halves
  const int head = blockIdx.y * 16 + l16, hq = min(head, p.heads - 1);
  const int2 at = lm_where(p.rows, m);
  const int slot = at.x, len = min(max(at.y + 1, 1), p.rows.S);
  int lo, hi;
  latent_range(len, p.n_splits, p.M, sp, lo, hi);
  const tl_u32x4* cc = reinterpret_cast<const tl_u32x4*>((const bf16_t*)p.c_cache + (size_t)slot * p.d.s64 * (RK * 64));
  const tl_u32x4* kc = reinterpret_cast<const tl_u32x4*>((const bf16_t*)p.kr_cache + (size_t)slot * p.d.s64 * (RB * 32));
  if (lo >= hi) return;  // no such piece
  // 32 keys are one contiguous run of either cache; a tile behind the piece's last re-reads that one, and its keys weigh nothing
  tl_u32x4 rc[KT][RK], rr[KT];
  auto fetch = [&](int j) {
#pragma unroll
    for (int k = 0; k < KT; ++k) {
      const size_t jt = (size_t)min((j >> 5) + k, (hi - 1) >> 5);
#pragma unroll
      for (int i = 0; i < RK; ++i) rc[k][i] = cc[jt * (CT / 8) + tid + 256 * i];
      rr[k] = kc[jt * (RT / 8) + min(tid, RT / 8 - 1)];
    }
  };
  auto stage = [&](bf16_t* dst) {
    tl_u32x4* sd = reinterpret_cast<tl_u32x4*>(dst);
#pragma unroll
    for (int k = 0; k < KT; ++k) {
#pragma unroll
      for (int i = 0; i < RK; ++i) sd[k * ((CT + RT) / 8) + tid + 256 * i] = rc[k][i];
      if (tid < RT / 8) sd[k * ((CT + RT) / 8) + CT / 8 + tid] = rr[k];
    }
  };
  fetch(lo);
  // this wave's columns: of every latent block piece `half` (or both), and a block of the rotated part (KT = 1: of one wave pair
  // without, RB = 1)
  const bool rot = KT == 2 || RB == 2 || half == 0;
  uint4 qf[KT][RK], qr[KT == 2 ? RB : 1];
  const int qrow = ((m & 15) + 16 * kg) * 8;
#pragma unroll
  for (int k = 0; k < KT; ++k)
#pragma unroll
    for (int i = 0; i < RK; ++i)
      qf[k][i] = *reinterpret_cast<const uint4*>((const bf16_t*)p.qlat + ((size_t)m * (p.d.heads16 >> 4) + blockIdx.y) * RK * 1024 + i * 1024 + (KT == 2 ? k : half) * 512 + lane * 8);
#pragma unroll
  for (int k = 0; k < (KT == 2 ? RB : 1); ++k)
    qr[k] = *reinterpret_cast<const uint4*>((const bf16_t*)p.qr + hq * p.qr_z + ((size_t)(m >> 4) * RB + (KT == 2 ? k : RB == 2 ? half : 0)) * 512 + qrow);
  tl_f32x4 acc[RK];
#pragma unroll
  for (int i = 0; i < RK; ++i) acc[i] = tl_f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;
  stage(tile);
  __syncthreads();
  int buf = 0;
  for (int j0 = lo; j0 < hi; j0 += 32 * KT) {
    const bf16_t* cur = tile + buf * BUF;
    const bool more = j0 + 32 * KT < hi;
    if (more) fetch(j0 + 32 * KT);
    tl_f32x4 s = {0.f, 0.f, 0.f, 0.f};
    const bf16_t* mine = cur + (t >> 1) * (CT + RT);  // tile of 16 keys t
#pragma unroll
    for (int k = 0; k < KT; ++k)
#pragma unroll
      for (int i = 0; i < RK; ++i)
        s = Tl<bf16_t>::mma(*reinterpret_cast<const uint4*>(mine + ((t & 1) * RK + i) * 1024 + (KT == 2 ? k : half) * 512 + lane * 8), qf[k][i], s);
    if (rot)  // uniform over the wave
#pragma unroll
      for (int k = 0; k < (KT == 2 ? RB : 1); ++k)
        s = Tl<bf16_t>::mma(*reinterpret_cast<const uint4*>(mine + CT + ((t & 1) * RB + (KT == 2 ? k : RB == 2 ? half : 0)) * 512 + lane * 8), qr[k], s);
    *reinterpret_cast<tl_f32x4*>(&sco[half * NT + t][lane * 4]) = s;
    __syncthreads();
    // keys j0 + 16 u + 4 kg + r of this lane's head
    float sv[4 * NT], mx = -INFINITY;
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      tl_f32x4 a = *reinterpret_cast<const tl_f32x4*>(&sco[u][lane * 4]);
      if (KT == 1) a += *reinterpret_cast<const tl_f32x4*>(&sco[(2 + u) & 3][lane * 4]);
      if (p.we.mul != 1.0f) a *= p.we.mul;  // uniform
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float v = j0 + 16 * u + 4 * kg + r < hi ? a[r] : -INFINITY;
        sv[4 * u + r] = v;
        mx = fmaxf(mx, v);
      }
    }
    mx = rows_max(mx);
    const float m_new = fmaxf(m_run, mx);  // finite: key j0 is in range
    const float alpha = weight_of(m_run, m_new, p.we);
    float pv[4 * NT], ps = 0.f;
#pragma unroll
    for (int e = 0; e < 4 * NT; ++e) { pv[e] = weight_of(sv[e], m_new, p.we); ps += pv[e]; }
    l_run = l_run * alpha + ps;
    m_run = m_new;
    uint4 hi4[KT], lo4[KT];
#pragma unroll
    for (int k = 0; k < KT; ++k) {
      const float* w = pv + 8 * k;
      uint4 &h = hi4[k], &l = lo4[k];
      h.x = f2bf2(w[0], w[1]); h.y = f2bf2(w[2], w[3]); h.z = f2bf2(w[4], w[5]); h.w = f2bf2(w[6], w[7]);
      l.x = f2bf2(w[0] - bf_lo(h.x), w[1] - bf_hi(h.x)); l.y = f2bf2(w[2] - bf_lo(h.y), w[3] - bf_hi(h.y));
      l.z = f2bf2(w[4] - bf_lo(h.z), w[5] - bf_hi(h.z)); l.w = f2bf2(w[6] - bf_lo(h.w), w[7] - bf_hi(h.w));
    }
    // 16 columns of block i, column group `wave`: column l16 of keys 4 kg + r and 16 + 4 kg + r; the lane reads four columns of a key
    const bf16_t* from = cur + (l16 >> 1 & 1) * 512 + (4 * kg + (l16 >> 2) + 16 * wave) * 8 + (l16 & 1) * 4;
#pragma unroll
    for (int i = 0; i < RK; ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][r] *= alpha;
#pragma unroll
      for (int k = 0; k < KT; ++k) {
        const uint2 a = tl_read_tr(from + k * (CT + RT) + i * 1024), b = tl_read_tr(from + k * (CT + RT) + (RK + i) * 1024);
        const uint4 v = make_uint4(a.x, a.y, b.x, b.y);
        acc[i] = Tl<bf16_t>::mma(v, hi4[k], acc[i]);
        acc[i] = Tl<bf16_t>::mma(v, lo4[k], acc[i]);
      }
    }
    if (BUFS == 1 && more) __syncthreads();
    if (more) stage(tile + (buf ^ (BUFS - 1)) * BUF);
    __syncthreads();
    buf ^= BUFS - 1;
  }
  l_run = rows_sum(l_run);
  if (head >= p.heads) return;
  const size_t piece = ((size_t)m * p.heads + head) * p.n_splits + sp;
  if (wave == 0 && kg == 0) *reinterpret_cast<float2*>(p.part_ml + 2 * piece) = make_float2(m_run, l_run);
#pragma unroll
  for (int i = 0; i < RK; ++i)
    *reinterpret_cast<tl_f32x4*>(p.part + piece * (RK * 64) + i * 64 + wave * 16 + 4 * kg) = acc[i];
}

// ---- merge of the pieces, value expansion through W_uv[h], head gate: up to 16 rows x 128 value dims of one head ----
template <typename T>
__global__ __launch_bounds__(512) void latent_value_kernel(int2* where, const void* w_uv, float* part, float* part_ml, int heads, int M, int S, uint32_t split,
                                                           int rank64, int vdim16, const LatentArgs p0) {
  LatentArgs p = p0;  // what the first loads need is in registers (see lm_gemm.hip)
  p.rows.where = where; p.w_uv = w_uv; p.part = part; p.part_ml = part_ml; p.heads = heads; p.M = M; p.rows.S = S;
  p.n_splits = (int)(split & 0xffu); p.d.rank64 = rank64; p.d.vdim16 = vdim16;
  const int rpw = (int)(split >> 8 & 0xffu), nbw = (int)(split >> 16);  // rows and blocks of 16 features of this workgroup
  extern __shared__ __align__(16) unsigned char lv_raw[];
  __shared__ __align__(16) float red[8][256];
  T* xs = (T*)lv_raw;  // 16 x rank64, tiled
  constexpr int EP = Tl<T>::EP, P = 16 / EP, PRE = sizeof(T) == 2 ? 8 : 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int h = blockIdx.x, m0 = blockIdx.z * rpw, R = p.d.rank64, ns = p.n_splits, nk = R >> 6;
  const int parts = 8 / nbw, kp = wave / nbw, k0 = nk * kp / parts, k1 = nk * (kp + 1) / parts;  // the waves of a block share its K
  const int nb = blockIdx.y * nbw + wave % nbw, nvb = p.d.vdim16 >> 4;
  const int nrow = min(rpw, p.M - m0);
  // the first weights are requested ahead of the merge
  const T* wv = (const T*)p.w_uv + ((size_t)h * nvb + min(nb, nvb - 1)) * nk * 1024 + lane * EP;
  uint4 wp[PRE][P];
#pragma unroll
  for (int k = 0; k < PRE; ++k)
    if (k0 + k < k1) {  // uniform
#pragma unroll
      for (int i = 0; i < P; ++i) wp[k][i] = *reinterpret_cast<const uint4*>(wv + (size_t)(k0 + k) * 1024 + 64 * EP * i);
    }
  const int m16 = min(m0 + (lane & 15), p.M - 1), pos16 = lm_where(p.rows, m16).y;  // of row lane % 16
  const float gate = p.gate[(size_t)m16 * p.d.heads16 + h];
  const int nc = (R + 255) >> 8;
  for (int it = wave; it < nrow * nc; it += 8) {  // a wave merges 256 columns of a row
    const int r = nc == 1 ? it : it / nc, c = (it - r * nc) * 256 + lane * 4;
    const int m = m0 + r, len = min(max(__builtin_amdgcn_readlane(pos16, r) + 1, 1), p.rows.S);
    const int chunk = latent_chunk(len, ns, p.M), np = (len + chunk - 1) / chunk;  // pieces that exist
    const size_t piece = ((size_t)m * p.heads + h) * ns;
    const float2 ml = *reinterpret_cast<const float2*>(p.part_ml + 2 * (piece + min(lane, np - 1)));
    const __amdgpu_buffer_rsrc_t pc = dev_buffer(p.part + piece * R, (uint32_t)(np * R * 4));  // nothing is fetched for pieces beyond the last
    auto load = [&](int s) {
      return __builtin_bit_cast(dev_f32x4, __builtin_amdgcn_raw_buffer_load_b128(pc, c < R ? (s * R + c) * 4 : (int)DEV_NOWHERE, 0, 0));
    };
    dev_f32x4 v[16];  // in flight together
#pragma unroll
    for (int u = 0; u < 16; ++u) v[u] = load(u);
    const float mx = wave_max(lane < np ? ml.x : -INFINITY);
    float w = lane < np ? weight_of(ml.x, mx, p.we) : 0.f;
    w /= wave_sum(w * ml.y);
    float o[4] = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0;;) {
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const float f = lane_f(w, min(s0 + u, 63));  // zero beyond the last piece
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = fmaf(f, v[u][e], o[e]);
      }
      s0 += 16;
      if (s0 >= np) break;
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = load(s0 + u);
    }
    if (c < R) Tl<T>::st4(xs + tl_off<T>(r, c, R), o);
  }
  // rows without a position: their products are dropped, but must be numbers
  for (int i = threadIdx.x; i < (16 - nrow) * (R / 4); i += 512) {
    const float z[4] = {0.f, 0.f, 0.f, 0.f};
    Tl<T>::st4(xs + tl_off<T>(nrow + i / (R / 4), (i % (R / 4)) * 4, R), z);
  }
  __syncthreads();
  tl_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  auto step = [&](int k, const uint4* a) {
#pragma unroll
    for (int i = 0; i < P; ++i)
      acc = Tl<T>::mma(a[i], *reinterpret_cast<const uint4*>(xs + (size_t)k * 1024 + 64 * EP * i + lane * EP), acc);
  };
#pragma unroll
  for (int k = 0; k < PRE; ++k)
    if (k0 + k < k1) step(k0 + k, wp[k]);
  for (int k = k0 + PRE; k < k1; ++k) {
    uint4 a[P];
#pragma unroll
    for (int i = 0; i < P; ++i) a[i] = *reinterpret_cast<const uint4*>(wv + (size_t)k * 1024 + 64 * EP * i);
    step(k, a);
  }
  if (parts > 1) {
    *reinterpret_cast<tl_f32x4*>(&red[wave][lane * 4]) = acc;
    __syncthreads();
    if (kp) return;
    for (int q = 1; q < parts; ++q) acc += *reinterpret_cast<const tl_f32x4*>(&red[wave + q * nbw][lane * 4]);
  }
  if (nb >= nvb || (lane & 15) >= nrow) return;
  const float v[4] = {acc[0] * gate, acc[1] * gate, acc[2] * gate, acc[3] * gate};
  Tl<T>::st4((T*)p.act + tl_off<T>(m0 + (lane & 15), h * p.d.vdim16 + nb * 16 + 4 * (lane >> 4), p.d.out_k), v);
}

// ---- expanded form for long blocks of one sequence (bf16): one workgroup per 16 queries and head ----
// Waves take 32 keys at a time in turn.  Scores^T (keys x queries) = K q^T leave a lane with eight keys of one query,
// which is operand layout for out^T = V^T p^T; the fp32 weights go in as a bf16 pair (value and remainder), so the
// average keeps about 16 bits of them.  DB = dim64 / 64, RB = rot32 / 32, VT >= vdim16 / 16.
// Bound by the keys and values that every tile of queries fetches from L2 (16 heads of 128 + 64 and 128, 1999 positions:
// 1.7 GB in 60 us).  Neighbouring workgroups take different heads, so that an XCD's L2 holds few of them, masks and the
// rescaling of the sums only in the steps that need them: 73 -> 60 us there; weights by weight_of instead of expf 63.7 -> 61.3 (another
// machine; 56 for 60 by the power of two alone, which is less exact than expf).  Two tiles of queries per wave were quicker there and slower at 600 positions of eight heads,
// and gave nothing of it in the whole prompt's time.
#define LPF_WAVES (VT <= 4 ? 8 : 4)
template <int DB, int RB, int VT>
__global__ __launch_bounds__(64 * LPF_WAVES, 2) void latent_prefill_kernel(const LatentArgs p, const WeightExp we) {
  __shared__ __align__(16) float s_acc[LPF_WAVES][VT * 256];
  __shared__ float s_m[LPF_WAVES][16], s_l[LPF_WAVES][16];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l16 = lane & 15, kg = lane >> 4;
  const int qt = gridDim.y - 1 - blockIdx.y, h = blockIdx.x;  // the tiles with the most keys start first
  const int q0 = qt * 16, T = p.M, pos0 = p.rows.pos0;
  const int nvb = p.d.vdim16 >> 4;
  const int qlast = pos0 + min(q0 + l16, T - 1);  // last visible key of this lane's query
  const int kend = pos0 + min(q0 + 15, T - 1) + 1;
  const bf16_t* qu = (const bf16_t*)p.qu + h * p.qu_z + (size_t)qt * DB * 1024 + lane * 8;
  const bf16_t* qr = (const bf16_t*)p.qr + h * p.qr_z + (size_t)qt * RB * 512 + lane * 8;
  uint4 qf[2 * DB + RB];
#pragma unroll
  for (int i = 0; i < 2 * DB; ++i) qf[i] = *reinterpret_cast<const uint4*>(qu + i * 512);
#pragma unroll
  for (int i = 0; i < RB; ++i) qf[2 * DB + i] = *reinterpret_cast<const uint4*>(qr + i * 512);
  const bf16_t* kb = (const bf16_t*)p.kx + h * p.kx_z + lane * 8;
  const bf16_t* rb = (const bf16_t*)p.kr_cache + (size_t)p.rows.slot * p.d.s64 * (RB * 32) + lane * 8;
  const bf16_t* vb = (const bf16_t*)p.vx + h * p.vx_z + lane * 8;
  const int vstep = (p.d.s64 >> 5) * 512;

  tl_f32x4 acc[VT];
#pragma unroll
  for (int d = 0; d < VT; ++d) acc[d] = tl_f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;
  for (int k0 = 32 * wave; k0 < kend; k0 += 32 * LPF_WAVES) {
    uint4 kf[2][2 * DB + RB], vf[VT];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int i = 0; i < 2 * DB; ++i) kf[t][i] = *reinterpret_cast<const uint4*>(kb + (size_t)((k0 >> 4) + t) * DB * 1024 + i * 512);
#pragma unroll
      for (int i = 0; i < RB; ++i) kf[t][2 * DB + i] = *reinterpret_cast<const uint4*>(rb + (size_t)((k0 >> 4) + t) * RB * 512 + i * 512);
    }
#pragma unroll
    for (int d = 0; d < VT; ++d) vf[d] = *reinterpret_cast<const uint4*>(vb + (size_t)min(d, nvb - 1) * vstep + (size_t)(k0 >> 5) * 512);
    __builtin_amdgcn_sched_barrier(0);
    tl_f32x4 sc[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      sc[t] = tl_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 2 * DB + RB; ++i) sc[t] = Tl<bf16_t>::mma(kf[t][i], qf[i], sc[t]);
      if (we.mul != 1.0f) sc[t] *= we.mul;  // uniform
    }
    if (k0 + 31 > pos0 + q0) {  // a key that some query of the tile does not see
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (k0 + 16 * t + 4 * kg + r > qlast) sc[t][r] = -INFINITY;
    }
    float mx = fmaxf(sc[0][0], sc[1][0]);
#pragma unroll
    for (int r = 1; r < 4; ++r) mx = fmaxf(mx, fmaxf(sc[0][r], sc[1][r]));
    mx = rows_max(mx);
    const float m_new = fmaxf(m_run, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = weight_of(m_run, m_use, we);
    float pv[8], lo[8], ps = 0.f;
    uint4 hi4, lo4;
#pragma unroll
    for (int e = 0; e < 8; ++e) { pv[e] = weight_of(sc[e >> 2][e & 3], m_use, we); ps += pv[e]; }
    l_run = l_run * alpha + ps;
    m_run = m_new;
    hi4.x = f2bf2(pv[0], pv[1]); hi4.y = f2bf2(pv[2], pv[3]); hi4.z = f2bf2(pv[4], pv[5]); hi4.w = f2bf2(pv[6], pv[7]);
    lo[0] = pv[0] - bf_lo(hi4.x); lo[1] = pv[1] - bf_hi(hi4.x); lo[2] = pv[2] - bf_lo(hi4.y); lo[3] = pv[3] - bf_hi(hi4.y);
    lo[4] = pv[4] - bf_lo(hi4.z); lo[5] = pv[5] - bf_hi(hi4.z); lo[6] = pv[6] - bf_lo(hi4.w); lo[7] = pv[7] - bf_hi(hi4.w);
    lo4.x = f2bf2(lo[0], lo[1]); lo4.y = f2bf2(lo[2], lo[3]); lo4.z = f2bf2(lo[4], lo[5]); lo4.w = f2bf2(lo[6], lo[7]);
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {  // few steps raise a maximum
#pragma unroll
      for (int d = 0; d < VT; ++d)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[d][r] *= alpha;
    }
#pragma unroll
    for (int d = 0; d < VT; ++d) {
      acc[d] = Tl<bf16_t>::mma(vf[d], hi4, acc[d]);
      acc[d] = Tl<bf16_t>::mma(vf[d], lo4, acc[d]);
    }
  }
  l_run = rows_sum(l_run);
  if (kg == 0) { s_m[wave][l16] = m_run; s_l[wave][l16] = l_run; }
#pragma unroll
  for (int d = 0; d < VT; ++d) *reinterpret_cast<tl_f32x4*>(&s_acc[wave][(d * 64 + lane) * 4]) = acc[d];
  __syncthreads();
  for (int sl = tid; sl < nvb * 64; sl += 64 * LPF_WAVES) {
    const int d = sl >> 6, ln = sl & 63, q = ln & 15, g4 = ln >> 4;
    const int t = q0 + q;
    if (t >= T) continue;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < LPF_WAVES; ++w) M = fmaxf(M, s_m[w][q]);
    float den = 0.f, o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < LPF_WAVES; ++w) {
      const float f = s_m[w][q] == -INFINITY ? 0.f : weight_of(s_m[w][q], M, we);
      den = fmaf(f, s_l[w][q], den);
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = fmaf(f, s_acc[w][sl * 4 + r], o[r]);
    }
    const float inv = p.gate[(size_t)t * p.d.heads16 + h] / den;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] *= inv;
    Tl<bf16_t>::st4((bf16_t*)p.act + tl_off<bf16_t>(t, h * p.d.vdim16 + 16 * d + 4 * g4, p.d.out_k), o);
  }
}

// ---- launchers ----
int launch_latent_append(const LatentArgs& a, hipStream_t st) {
  if (a.dtype == VUI_DTYPE_F32) hipLaunchKernelGGL(latent_append_kernel<float>, dim3((a.M + 3) / 4), dim3(256), 0, st, a);
  else hipLaunchKernelGGL(latent_append_kernel<bf16_t>, dim3((a.M + 3) / 4), dim3(256), 0, st, a);
  HIP_TRY(hipGetLastError());
  return VUI_OK;
}

int launch_latent_query(const LatentArgs& a, hipStream_t st) {
  const dim3 grid(a.heads + (a.own ? 1 : 0), (a.d.rank16 / 16 + 3) / 4, (a.M + 15) / 16);
  if (a.dtype == VUI_DTYPE_F32) hipLaunchKernelGGL(latent_query_kernel<float>, grid, dim3(256), 0, st, a.w_uk_t, a.qu, a.craw, a.qu_z, a.heads, a.M, a.d.dim64, a.d.rank16, a);
  else hipLaunchKernelGGL(latent_query_kernel<bf16_t>, grid, dim3(256), 0, st, a.w_uk_t, a.qu, a.craw, a.qu_z, a.heads, a.M, a.d.dim64, a.d.rank16, a);
  HIP_TRY(hipGetLastError());
  return VUI_OK;
}

bool latent_mfma_ok(const vui_lm_dims& d) { return d.rank64 <= 512 && d.rot32 <= 64; }

template <int RK, int RB, int KT>
static int lam_go(const LatentArgs& a, hipStream_t st) {
  constexpr int lds = 2 * (RK * 2048 + RB * 1024) * 2;
  if (lds > 60 * 1024)
    HIP_TRY(hipFuncSetAttribute((const void*)latent_attn_mfma_kernel<RK, RB, KT>, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  hipLaunchKernelGGL((latent_attn_mfma_kernel<RK, RB, KT>), dim3(a.M, (a.heads + 15) / 16, a.n_splits), dim3(256), lds, st, a.rows.where, a.c_cache, a.kr_cache, a.qlat,
                     (uint32_t)a.M | (uint32_t)a.n_splits << 24, a.rows.S, a.d.s64, a.d.heads16, a);
  HIP_TRY(hipGetLastError());
  return VUI_OK;
}
template <int RB, int KT>
static int lam_rank(const LatentArgs& a, hipStream_t st) {
  switch (a.d.rank64 / 64) {
    case 1: return lam_go<1, RB, KT>(a, st);
    case 2: return lam_go<2, RB, KT>(a, st);
    case 3: return lam_go<3, RB, KT>(a, st);
    case 4: return lam_go<4, RB, KT>(a, st);
    case 5: return lam_go<5, RB, KT>(a, st);
    case 6: return lam_go<6, RB, KT>(a, st);
    case 7: return lam_go<7, RB, KT>(a, st);
    default: return lam_go<8, RB, KT>(a, st);
  }
}

int launch_latent_attn(const LatentArgs& a, hipStream_t st) {
  if (a.n_splits < 1 || a.n_splits > 64 || a.M >= 1 << 24 || a.d.rank64 > 256 * LAT_ACC) { vui_set_error("latent attention: rank %d, splits %d out of range", a.d.rank64, a.n_splits); return VUI_EINVAL; }
  if (a.dtype == VUI_DTYPE_BF16 && latent_mfma_ok(a.d)) {
    const bool one = latent_least(a.M) == 32;
    if (a.d.rot32 == 32) return one ? lam_rank<1, 1>(a, st) : lam_rank<1, 2>(a, st);
    return one ? lam_rank<2, 1>(a, st) : lam_rank<2, 2>(a, st);
  }
  const dim3 grid(a.M, a.heads, a.n_splits);
  const size_t lds = (size_t)(a.d.rank64 + a.d.rot32) * 4;
  if (a.dtype == VUI_DTYPE_F32) hipLaunchKernelGGL(latent_attn_kernel<float>, grid, dim3(256), lds, st, a);
  else hipLaunchKernelGGL(latent_attn_kernel<bf16_t>, grid, dim3(256), lds, st, a);
  HIP_TRY(hipGetLastError());
  return VUI_OK;
}

// Rows and feature blocks of a workgroup: what a CU takes in (the rows' pieces, which every split of the features reads again, and W_uv,
// which every split of the rows does) at 60 KB a us, 1.2 us per round of merges, 3 us for the rest, all of it again for every 256
// workgroups, of which a CU holds one.  us per launch, a row and all 128 features until 192 workgroups / two merges of 64 columns side by side ->
// so: 16 heads of rank 512, 1 row behind 1200 7.8 -> 6.5 (two blocks), 16 rows behind 300 6.2 -> 5.4 (two rows, four blocks), a prompt of
// 50 15.3 -> 7.8 (eight rows, four blocks); 8 heads, 16 rows behind 1400 7.0 -> 6.0.
int launch_latent_value(const LatentArgs& a, hipStream_t st) {
  const bool f32 = a.dtype == VUI_DTYPE_F32;
  const int nvb = a.d.vdim16 / 16, R = a.d.rank64;
  int pieces = (a.n_splits + 1) / 2;  // of a row; known for a prompt
  if (a.rows.seq) {
    const int len = std::min(a.rows.pos0 + a.M, a.rows.S), chunk = latent_chunk(len, a.n_splits, a.M);
    pieces = (len + chunk - 1) / chunk;
  }
  int rpw = 1, nbw = 8;
  float best = 0;
  const float in_row = pieces * R * 4 / 60e3f, in_block = 16 * R * (f32 ? 4 : 2) / 60e3f;
  for (int rs = 0; rs <= 4 && (rs == 0 || 1 << (rs - 1) < a.M); ++rs) {
    const int tiles = (a.M + (1 << rs) - 1) >> rs, r = std::min(1 << rs, a.M);
    for (int bs = 3; bs >= 1; --bs) {
      const int n = a.heads * ((nvb + (1 << bs) - 1) >> bs) * tiles;
      const float c = ((n + 255) >> 8) * (3 + r * in_row + std::min(1 << bs, nvb) * in_block + 1.2f * ((r * ((R + 255) >> 8) + 7) >> 3));
      if (best == 0 || c < best) { best = c; rpw = 1 << rs; nbw = 1 << bs; }
    }
  }
  const dim3 grid(a.heads, (nvb + nbw - 1) / nbw, (a.M + rpw - 1) / rpw);
  const uint32_t split = (uint32_t)a.n_splits | (uint32_t)rpw << 8 | (uint32_t)nbw << 16;
  const size_t lds = (size_t)16 * a.d.rank64 * (f32 ? 4 : 2);
  if (lds > 56 * 1024) {  // beside it 8 KiB of the waves' sums
    HIP_TRY(hipFuncSetAttribute(f32 ? (const void*)latent_value_kernel<float> : (const void*)latent_value_kernel<bf16_t>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  }
  if (f32) hipLaunchKernelGGL(latent_value_kernel<float>, grid, dim3(512), lds, st, a.rows.where, a.w_uv, a.part, a.part_ml, a.heads, a.M, a.rows.S, split, a.d.rank64, a.d.vdim16, a);
  else hipLaunchKernelGGL(latent_value_kernel<bf16_t>, grid, dim3(512), lds, st, a.rows.where, a.w_uv, a.part, a.part_ml, a.heads, a.M, a.rows.S, split, a.d.rank64, a.d.vdim16, a);
  HIP_TRY(hipGetLastError());
  return VUI_OK;
}

bool latent_expand_ok(const vui_lm_dims& d) { return d.dim64 <= 128 && d.rot32 <= 64 && d.vdim16 <= 128; }

template <int DB, int RB>
static void lpf_go(const LatentArgs& a, hipStream_t st) {
  const dim3 grid(a.heads, (a.M + 15) / 16);
  const WeightExp we = weight_exp(a.scale);
  if (a.d.vdim16 <= 32) hipLaunchKernelGGL((latent_prefill_kernel<DB, RB, 2>), grid, dim3(512), 0, st, a, we);
  else if (a.d.vdim16 <= 64) hipLaunchKernelGGL((latent_prefill_kernel<DB, RB, 4>), grid, dim3(512), 0, st, a, we);
  else hipLaunchKernelGGL((latent_prefill_kernel<DB, RB, 8>), grid, dim3(256), 0, st, a, we);
}
int launch_latent_prefill_attn(const LatentArgs& a, hipStream_t st) {
  if (!latent_expand_ok(a.d) || a.dtype != VUI_DTYPE_BF16 || !a.rows.seq) { vui_set_error("latent prefill: sizes out of range"); return VUI_EINVAL; }
  if (a.d.dim64 == 64) { if (a.d.rot32 == 32) lpf_go<1, 1>(a, st); else lpf_go<1, 2>(a, st); }
  else { if (a.d.rot32 == 32) lpf_go<2, 1>(a, st); else lpf_go<2, 2>(a, st); }
  HIP_TRY(hipGetLastError());
  return VUI_OK;
}
