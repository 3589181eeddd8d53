// Streaming vocoder frame step: codes of one codec frame -> hop audio samples, fp32.
//
// Reference: QwenCodecDecoder.forward in streaming mode (src/vui/qwen_codec.py:1191-1224) with its
// building blocks CausalConv1d (:45-101), CausalTransConv1d (:112-158), SplitResidualVQ.decode (:263-270),
// DecTransformer._forward_streaming (:1048-1076), ConvNeXtBlock (:832-848), DecoderBlock (:863-879),
// SnakeBeta (:820-829).
//
// Layout.  Activations are channel-major (C, columns).  Every conv input lives in a ring of 2^k columns
// per channel that keeps the last `pad` columns of earlier frames in front of the current ones: frame f
// occupies columns (f*T + pad + t) mod 2^k, so no history is ever copied; a device counter holds f.
// The activation that precedes a conv (snake) is applied by the producer's epilogue, which writes the
// raw value (for residuals) and the activated value (into the consumer's ring) in one pass.
//
// One GEMM kernel serves every conv, transposed conv and linear layer: out (M x T) = W (M x taps*Cin) .
// X, X[(tap, ci)][t] = ring[ci][t + tap*dil].  Weights are repacked once to tap-major (taps, M, Cin) so a
// lane reads 32 contiguous bytes of one output row; a transposed conv with kernel 2*stride is the
// two-tap conv over (previous column, current column) with M = Cout*stride rows whose results are
// scattered to column t*stride + r.  A workgroup owns 16 output rows x 16*TT columns; its input columns go through
// LDS, its waves split the (tap, 32-channel) units, multiply on v_mfma_f32_16x16x4_f32 with the weights read straight from
// global memory, and add their parts through LDS in a fixed order.
//
// Several frames at once (vui_codec_decode_clip: offline calls, the seeding of a stream; vui_codec_decode_block up to 32): the same
// steps over frames x columns, on buffers that hold a whole pass with the histories in front; wide products run in
// cv_wide_kernel.  93 frames: 42.7 ms one after the other, 5.6 ms in blocks of 32, 4.1 in one pass (MI355X).
#include "common.h"
#include "internal.h"
#include "../../include/vui_codec.h"

#include <algorithm>
#include <math.h>
#include <new>
#include <stdio.h>
#include <string.h>
#include <vector>

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

struct Ring {
  float* p;
  int rs;     // columns per channel (power of two; a buffer of several frames: any)
  int mask;   // rs - 1 (a buffer of several frames: all ones)
  int pad;    // history columns in front of a frame
  int tstep;  // columns a frame adds (0: plain buffer, always at column 0)
  int id;     // host side: its place in vui_codec::twins
};

__device__ __forceinline__ int ring_base(const Ring& r, int f) { return (f * r.tstep) & r.mask; }
__device__ __forceinline__ float* ring_ptr(const Ring& r, int base, int c, int col) {
  return r.p + (size_t)c * r.rs + ((base + col) & r.mask);
}

// IN_RMS: the input column is RMS-normalised; the norm weight is folded into W when it is packed and
// 1/rms multiplies the sums.  EPI_SILU_PAIR: rows (2i, 2i+1) hold gate_i and up_i; channel i = silu(gate) * up.
enum { IN_PLAIN = 0, IN_RMS = 1 };
enum { EPI_NONE = 0, EPI_GELU = 1, EPI_RES = 2, EPI_SCALE_RES = 3, EPI_SILU_PAIR = 4 };

struct CvGemm {
  const float* W;     // (taps, M, Cin)
  const float* bias;  // row m uses bias[m / bias_div]; may be null
  int M, Cin, taps, dil, T;
  int bias_div;
  Ring in;
  int in_mode;
  float eps;
  int epi;
  const float* scale;  // per output channel (EPI_SCALE_RES)
  Ring res;
  int tc_stride;  // > 0: row m -> channel m / s, column t*s + m % s
  Ring out_raw;   // p may be null
  Ring out_act;   // p may be null: snake with (ea, ib) of the consumer
  const float* ea;
  const float* ib;
  const int* ctr;  // frames started; this pass is frames *ctr - nf ... *ctr - 1
  int nf;
  int splits;      // workgroups that share one tile's channel groups; > 1: parts meet in `part`
  int per, chunk;  // cv_cols_kernel: channel groups of a workgroup, and of those at a time
  int xcols;       // and the input columns of a tile
  uint32_t inv_xcols, inv_tc;
  float* part;     // (tiles, splits, TT*64*4) partial sums
  int* cnt;        // (tiles) arrival counters, zero between launches
  int tt;          // cv_cols_kernel: 16-column blocks per tile (picks the instantiation); 0: cv_wide_kernel with tile kWide[wide]
  int wide;
};

// A vocoder that shares the GPU with other kernels (vui_codec_workgroups) reads its weights - 423 MB per frame, each
// byte once - with non-temporal loads, so that they pass through the caches without pushing out what those kernels
// read again and again.  On its own the vocoder is 4 % slower with the hint (636 against 610 us per frame), so a
// vocoder that owns the GPU does not use it.
typedef float cv_f32x4 __attribute__((ext_vector_type(4)));
template <bool NT> __device__ __forceinline__ float4 cv_ld_w(const float* p) {
  if constexpr (NT) {
    const cv_f32x4 v = __builtin_nontemporal_load((const __attribute__((address_space(1))) cv_f32x4*)p);
    float4 r;
    __builtin_memcpy(&r, &v, sizeof(r));
    return r;
  } else {
    return *reinterpret_cast<const float4*>(p);
  }
}

#define CV_WIDE_T 64  // columns from which cv_wide_kernel takes a product of several frames

#define CV_NW 8        // waves of a workgroup of cv_cols_kernel
// sin(t)^2 for |t| below CV_SIN_FAR: t less a multiple of pi / 2 (in two parts, by fma), then s = r + r^3 P(r^2) on [-pi/4, pi/4], P of degree 2 fitted
// here to the least relative error (2^-28); s^2, or 1 - s^2 of an odd multiple.  Half of sinf's instructions, root mean square error
// 0.35 x 2^-24 (a correctly rounded sine, squared: 0.45).  93 frames, us with sinf / so: 7-tap convolutions of 768 / 384 / 192 / 96 channels
// 181 / 198 / 220 / 192 and 178 / 196 / 216 / 189, 1x1 59 / 47 / 63 / 74 and 57 / 45 / 58 / 70, the clip 4164 / 4092; six streamed frames 2736 / 2721.
// Error of the audio against 64 bits 3.24e-6 / 3.23e-6.
#define CV_SIN_FAR 25000.f
__device__ __forceinline__ float cv_sin2(float t) {
  const float k = rintf(t * 0.63661975f);
  const float r = fmaf(-k, -4.371139e-08f, fmaf(-k, 1.5707964f, t)), z = r * r;
  const float s = fmaf(fmaf(fmaf(-0.00019514957f, z, 0.008332158f), z, -0.16666655f) * z, r, r);
  return (int)k & 1 ? fmaf(-s, s, 1.f) : s * s;
}
// v = y + ib sin(ea y)^2
template <int N>
__device__ __forceinline__ void cv_snake(const float (&y)[N], const float (&ea)[N], const float (&ib)[N], float (&v)[N]) {
  float t[N];
  bool far = false;
#pragma unroll
  for (int e = 0; e < N; ++e) {
    t[e] = y[e] * ea[e];
    far |= !(fabsf(t[e]) < CV_SIN_FAR);
    v[e] = fmaf(ib[e], cv_sin2(t[e]), y[e]);
  }
  if (far) {
#pragma unroll
    for (int e = 0; e < N; ++e) {
      const float s = sinf(t[e]);
      v[e] = y[e] + ib[e] * s * s;
    }
  }
}

// Floats of staged columns, at most: 68 KiB, beside them 8 KiB of the waves' parts per block of columns.  Of tiles of one block two workgroups
// fit a CU whatever they stage, of two and four blocks where they stage less (7 taps 9 apart of 384 channels x 160 columns: 82 KiB, one).
#define CV_XROOM 17408
// (tap, 32-channel) units of a wave between two barriers
template <int TT> struct CvUnits { static constexpr int N = TT <= 2 ? 6 : 4; };

// i / n for i n < 2^32 with inv = cv_inv(n)
static uint32_t cv_inv(uint32_t n) { return n > 1 ? 0xFFFFFFFFu / n + 1u : 0u; }
__device__ __forceinline__ uint32_t cv_div(uint32_t i, uint32_t inv) { return inv ? __umulhi(i, inv) : i; }

// One tile of 16 output rows x 16 TT columns.  A workgroup takes `per` of the G = Cin / 32 channel groups with all their taps (splits
// workgroups share a tile), `chunk` groups at a time: their input columns, taps - 1 dilations of halo among them, are read once,
// coalesced, and laid into LDS with the channels side by side, from where every tap reads them as whole vectors; the chunk's units are dealt
// round the waves, whose weights are on their way meanwhile.
// Bound by its chain of trips: counter, columns, LDS, products, LDS, the parts' meeting.  With the columns read from memory by every tap
// (eight loads of a float per unit and block of columns, issuing which took 3-4 us) and the outputs four to a lane, us per launch of a
// single frame / so: 7 taps of 768 channels x 32 columns 16.5 / 11.8, 384 x 160 14.8 / 11.9, 192 x 640 13.0 / 10.7, 96 x 1920 10.7 / 9.2; one tap
// 9.1 / 6.4, 7.9 / 5.6, 8.3 / 5.9, 7.4 / 5.6; the frame 572 / 482.
// The first fourteen words of scalar arguments are in registers when a kernel starts, a struct is a trip to memory (0.2-0.35 us): what the
// counter's, the weights' and the columns' addresses need comes twice, ahead of the struct and in it, and the waves' shares of the
// (group, tap) units as numbers instead of divisions (at most seven taps): 0.5-0.9 us of a
// launch of 6-12, a streamed frame 481 -> 457 us.
#define CV_HOT const float *W, const float *in_p, const int *ctr, int M, int Cin, int T, uint32_t taps, int rs, int mask, uint32_t per_chunk, uint32_t inv_xcols
static uint32_t cv_taps(const CvGemm& g) {
  const uint32_t taps = g.taps, step = CV_NW / taps;
  return taps | (uint32_t)g.dil << 8 | step << 16 | (CV_NW - step * taps) << 20 | (256 / taps + 1) << 23;
}
#define CV_HOT_ARGS(g) g.W, g.in.p, g.ctr, g.M, g.Cin, g.T, cv_taps(g), g.in.rs, g.in.mask, (uint32_t)g.per | (uint32_t)g.chunk << 16, g.inv_xcols
template <int TT, bool NT>
__global__ __launch_bounds__(64 * CV_NW, 4) void cv_cols_kernel(CV_HOT, const CvGemm p0) {
  CvGemm p = p0;
  p.W = W; p.in.p = const_cast<float*>(in_p); p.ctr = ctr; p.M = M; p.Cin = Cin; p.T = T; p.taps = (int)(taps & 0xffu); p.dil = (int)(taps >> 8 & 0xffu);
  p.in.rs = rs; p.in.mask = mask; p.per = (int)(per_chunk & 0xffffu); p.chunk = (int)(per_chunk >> 16); p.inv_xcols = inv_xcols;
  p.xcols = min(T, 16 * TT) + (p.taps - 1) * p.dil;
  constexpr int NU = CvUnits<TT>::N, NTH = 64 * CV_NW, RED = CV_NW * TT * 256;
  extern __shared__ __align__(16) float lds[];
  float* red = lds;
  float* xs = lds + RED;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int r16 = lane & 15, g = lane >> 4;
  const int m0 = blockIdx.x * 16, t0 = blockIdx.y * (16 * TT), tile = blockIdx.y * gridDim.x + blockIdx.x, part_idx = blockIdx.z;
  const int G = Cin >> 5;
  const int gb = part_idx * p.per, ge = min(G, gb + p.per);
  const int halo = (p.taps - 1) * p.dil, cols = p.xcols - halo, S = p.chunk * 32 + 4;

  // The wave's unit i of a chunk is wave + CV_NW i: group (unit / taps), tap (unit % taps).  The weights do not depend on the frame
  // counter: those of the first chunk are asked for before the counter is needed.
  float4 a[NU][2];
  int off[NU];  // of the unit's first column in LDS
  const uint32_t w_lane = (uint32_t)(r16 * Cin + g * 8);
  const int g_step = (int)(taps >> 16 & 15u), t_step = (int)(taps >> 20 & 7u), g_first = (int)(wave * (taps >> 23) >> 8), t_first = wave - g_first * p.taps;
  auto load_a = [&](int gc, int n) {
    int gl = g_first, tap = t_first;
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const bool on = gl < n;  // uniform over the wave
      off[i] = on ? tap * p.dil * S + gl * 32 : -1;
      if (on) {
        const float* wp = p.W + ((size_t)tap * M + m0) * Cin + (gc + gl) * 32;
        a[i][0] = cv_ld_w<NT>(wp + w_lane);
        a[i][1] = cv_ld_w<NT>(wp + w_lane + 4);
      }
      gl += g_step; tap += t_step;
      if (tap >= p.taps) { tap -= p.taps; ++gl; }
    }
  };
  const int f = *p.ctr - p.nf;
  load_a(gb, min(p.chunk, ge - gb));
  const int ib_ = ring_base(p.in, f);
  floatx4 acc[TT];
#pragma unroll
  for (int tt = 0; tt < TT; ++tt) acc[tt] = floatx4{0.f, 0.f, 0.f, 0.f};
  // Every thread finishes NO of the tile's sums: row (tid / 16) % 16, column tid % 16 of block tid / 256 (+ 2).  (Four rows of a column per lane
  // of the first TT waves was 1 us more per launch: long chains of sines and stores in few waves; the frame 515 / 483.)
  constexpr int NO = TT == 4 ? 2 : 1;
  const int em = m0 + ((tid >> 4) & 15), ech = p.tc_stride > 0 ? (int)cv_div(em, p.inv_tc) : em;
  float e_bias = 0.f, e_sc = 1.f, e_ea = 0.f, e_ib = 0.f, e_res[NO];
  int ecol[NO];  // of the output, -1: none
  const float* xrow[TT];  // this lane's columns
#pragma unroll
  for (int tt = 0; tt < TT; ++tt) xrow[tt] = xs + min(tt * 16 + r16, cols - 1) * S + g * 8;
  float ss = 0.f;  // IN_RMS: this thread's share of its column's sum of squares
  constexpr int TPC = NTH / (16 * TT);

  for (int gc = gb; gc < ge; gc += p.chunk) {
    const int n = min(p.chunk, ge - gc);
    if (gc > gb) { load_a(gc, n); __syncthreads(); }  // the columns of the chunk before have been read
    // four channels of a column per thread and round
    const int total = n * 8 * p.xcols;
    const float *in0 = p.in.p + (size_t)gc * 32 * p.in.rs, *in1 = in0 + p.in.rs, *in2 = in1 + p.in.rs, *in3 = in2 + p.in.rs;
    for (int i0 = tid; i0 < total; i0 += 4 * NTH) {
      float4 v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = min(i0 + k * NTH, total - 1), q = (int)cv_div(i, p.inv_xcols), c = i - q * p.xcols;
        const uint32_t o = (uint32_t)(4 * q * p.in.rs + ((ib_ + min(t0 + c, p.T - 1 + halo)) & p.in.mask));
        v[k] = make_float4(in0[o], in1[o], in2[o], in3[o]);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = i0 + k * NTH, q = (int)cv_div(i, p.inv_xcols), c = i - q * p.xcols;
        if (i < total) *reinterpret_cast<float4*>(xs + c * S + 4 * q) = v[k];
      }
    }
    if (gc == gb) {  // what the epilogue adds is requested now as well
      const int rb = ring_base(p.res, f);
      if (p.bias) e_bias = p.bias[ech];
      if (p.epi == EPI_SCALE_RES) e_sc = p.scale[ech];
      if (p.out_act.p) { e_ea = p.ea[ech]; e_ib = p.ib[ech]; }
#pragma unroll
      for (int k = 0; k < NO; ++k) {
        const int tt = (tid >> 8) + 2 * k, t = t0 + tt * 16 + (tid & 15);
        ecol[k] = tt < TT && t < p.T ? (p.tc_stride > 0 ? t * p.tc_stride + em - ech * p.tc_stride : t) : -1;
        e_res[k] = 0.f;
        if ((p.epi == EPI_RES || p.epi == EPI_SCALE_RES) && ecol[k] >= 0) e_res[k] = *ring_ptr(p.res, rb, ech, p.res.pad + ecol[k]);
      }
    }
    __syncthreads();
    if (p.in_mode == IN_RMS) {  // one tap
      const float* col = xs + min(tid / TPC, cols - 1) * S;
      for (int q = tid % TPC; q < n * 8; q += TPC) {
        const float4 v = *reinterpret_cast<const float4*>(col + 4 * q);
        ss += (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w);
      }
    }
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      if (off[i] < 0) break;  // uniform over the wave
      const float av[8] = {a[i][0].x, a[i][0].y, a[i][0].z, a[i][0].w, a[i][1].x, a[i][1].y, a[i][1].z, a[i][1].w};
      float bv[TT][8];
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
        const float4 lo = *reinterpret_cast<const float4*>(xrow[tt] + off[i]), hi = *reinterpret_cast<const float4*>(xrow[tt] + off[i] + 4);
        bv[tt][0] = lo.x; bv[tt][1] = lo.y; bv[tt][2] = lo.z; bv[tt][3] = lo.w;
        bv[tt][4] = hi.x; bv[tt][5] = hi.y; bv[tt][6] = hi.z; bv[tt][7] = hi.w;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) acc[tt] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[j], bv[tt][j], acc[tt], 0, 0, 0);
      if (i & 1) __builtin_amdgcn_sched_barrier(0);  // more units' operands at a time do not fit the registers
    }
  }

  // add the waves' parts in a fixed order
#pragma unroll
  for (int tt = 0; tt < TT; ++tt)
    *reinterpret_cast<float4*>(red + ((size_t)(wave * TT + tt) * 64 + lane) * 4) =
        make_float4(acc[tt][0], acc[tt][1], acc[tt][2], acc[tt][3]);
  __shared__ float rms[16 * TT];
  if (p.in_mode == IN_RMS) {  // neighbouring threads share a column
#pragma unroll
    for (int o = TPC / 2; o >= 1; o >>= 1) ss += __shfl_xor(ss, o);
    if (tid % TPC == 0) rms[tid / TPC] = 1.0f / sqrtf(ss / (float)Cin + p.eps);
  }
  __syncthreads();
  float v[NO];
#pragma unroll
  for (int k = 0; k < NO; ++k) {
    v[k] = 0.f;
    const float* src = red + (size_t)(min((tid >> 8) + 2 * k, TT - 1) * 64 + ((tid >> 6) & 3) * 16 + (tid & 15)) * 4 + ((tid >> 4) & 3);
#pragma unroll
    for (int w = 0; w < CV_NW; ++w) v[k] += src[w * TT * 256];
  }
  const bool mine = TT > 1 || tid < 256;
  if (p.splits > 1) {
    // parts of a tile meet in memory; the workgroup that arrives last adds them in part order and finishes
    __shared__ int last;
    float* part = p.part + (size_t)tile * p.splits * TT * 256 + tid;
    if (mine)
#pragma unroll
      for (int k = 0; k < NO; ++k) __hip_atomic_store(part + part_idx * TT * 256 + 512 * k, v[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the write-through stores have completed
    __syncthreads();
    if (tid == 0) {
      const int old = __hip_atomic_fetch_add(p.cnt + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last = old == p.splits - 1;
      if (last) __hip_atomic_store(p.cnt + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!last) return;
    if (mine) {
      float q[NO][8];
#pragma unroll
      for (int k = 0; k < NO; ++k)
#pragma unroll
        for (int z = 0; z < 8; ++z) q[k][z] = z < p.splits ? __hip_atomic_load(part + z * TT * 256 + 512 * k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.f;
#pragma unroll
      for (int k = 0; k < NO; ++k) {
        v[k] = 0.f;
#pragma unroll
        for (int z = 0; z < 8; ++z) v[k] += q[k][z];
      }
    }
  }
  if (!mine) return;
  const int ob = ring_base(p.out_raw, f), ab = ring_base(p.out_act, f);
#pragma unroll
  for (int k = 0; k < NO; ++k) {
    if (p.in_mode == IN_RMS) v[k] *= rms[min((tid >> 8) + 2 * k, TT - 1) * 16 + (tid & 15)];
    if (p.epi == EPI_SILU_PAIR) {
      const float up = __shfl_xor(v[k], 16);  // the next row's, for the even ones
      if (!(tid & 16) && ecol[k] >= 0) *ring_ptr(p.out_raw, ob, em >> 1, p.out_raw.pad + ecol[k]) = v[k] / (1.0f + expf(-v[k])) * up;
      continue;
    }
    float y = v[k] + e_bias;
    if (p.epi == EPI_GELU) y = 0.5f * y * (1.0f + erff(y * 0.70710678118654752f));
    else if (p.epi == EPI_RES) y = e_res[k] + y;
    else if (p.epi == EPI_SCALE_RES) y = e_res[k] + e_sc * y;
    if (ecol[k] < 0) continue;
    if (p.out_raw.p) *ring_ptr(p.out_raw, ob, ech, p.out_raw.pad + ecol[k]) = y;
    if (p.out_act.p) {
      float sq = y * e_ea;
      if (fabsf(sq) < CV_SIN_FAR) {
        sq = cv_sin2(sq);
      } else {
        sq = sinf(sq);
        sq *= sq;
      }
      *ring_ptr(p.out_act, ab, ech, p.out_act.pad + ecol[k]) = fmaf(e_ib, sq, y);
    }
  }
}

// ---- the same product for many columns (several frames at once) ----
// On the bf16 matrix instructions, which are 16 times the rate of the fp32 ones (157 TFLOP/s): every fp32 operand is the sum of three
// bf16 numbers (8 bits each, nearest, so that the rest halves once more), and of their nine products the six that
// reach 2^-24 of the value are summed in fp32, small ones first (G. Henry, P. T. P. Tang, A. Heinecke, "Leveraging the bfloat16
// Artificial Intelligence Datatype for Higher-Precision Computations", ARITH 2019).  What is left out is 2^-26 of a product; the sums have
// fewer roundings than with v_mfma_f32_32x32x2_f32 (sixteen products per step instead of two).
// The sum is exact for every finite value from 2^-110 up.  Of a smaller one, what lies below bf16's least subnormal, 2^-133, is lost
// (weights of 2^-118: error of the product 1.4e-5, 2^-122: 2e-4; with fp32 instructions 2e-6).  A value that is not finite makes its
// columns or rows NaN, an infinite one too.
// 32 frames: 7-tap convolutions of 768 / 384 / 192 / 96 channels 86 / 105 / 121 / 91 us -> 55 / 63 / 83 / 62 (920 TFLOP/s
// of bf16 products in the first; hipBLASLt reaches 1125 at 8192^3), 1x1 19 / 30 / 32 / 33 -> 16 / 29 / 26 / 29 (3-4 % more with the clamp
// of cv_split2); error of 93 frames against 64 bits 4.1e-6 -> 3.9e-6.
// Tiles of BM x BN = 128 x 128 (or what divides M) of four waves through LDS, three planes of each operand: a K step is one (tap,
// 32-channel) unit, fetched into registers while the one before it is multiplied, split on the way to LDS.  A group's taps follow each
// other, so that its columns, with the taps' halo, are fetched, split and stored once for all of them (per tap they were two thirds of
// the vector instructions and a quarter of what LDS moves, beside matrix instructions that it nearly holds up); where two workgroups of a
// CU still fit, weights have a second buffer and a unit one barrier.  93 frames, 7-tap convolutions of 768 / 384 / 192 / 96 channels
// 214 / 247 / 275 / 227 -> 195 / 211 / 240 / 198 us, the clip 4681 -> 4259, 250 frames 10883 -> 9726.  Eight waves with two buffers of both
// and one to three units in flight: 75 us of the 384-channel convolution of 32 frames when this form took 63.
// Two fp16 parts of each operand, scaled by a power of two per matrix and per 32 channels of a tile, and three products took the clip 4110 -> 3225 us
// and the audio was no further off (3.1e-6).  But what is small beside something large in the same block lost its bits: a frame 2^30 larger than those
// before it put 2e-3 of error into their audio, rows 2^30 apart, or channels 2^40 apart and their weights the inverse, likewise.
// Where the tiles are fewer than the CUs their units are split over workgroups, and cv_finish_kernel adds the parts.
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 cv_bf16x8;

#define CVW_RUN 4
#define CVW_HALO 56  // columns that the taps reach beyond a tile: 6 x 9
// In LDS a row's (or column's) 32 channels of a plane are four pieces of 16 bytes; a piece's place turns with the row, so that 16-byte
// reads of eight rows fall on different banks.
__device__ __forceinline__ int cv_at(int row, int piece) { return row * 32 + 8 * (piece ^ (row >> 2 & 3)); }

// two fp32 values -> their three bf16 parts, packed.  The first part of a value above bf16's largest (3.39e38) is that largest: to the
// nearest it would be infinity, and the column NaN.  Two instructions per pair: the products take 3-4 % more, 93 frames 5960 -> 6050 us.
// (A tile computed once more with the clamp where a sum is not finite needs 40 registers more: 6070 us.)
__device__ __forceinline__ void cv_split2(float a, float b, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  const float top = __uint_as_float(0x7f7f0000u);
  hi = f2bf2(__builtin_amdgcn_fmed3f(a, -top, top), __builtin_amdgcn_fmed3f(b, -top, top));
  a -= bf_lo(hi); b -= bf_hi(hi);
  mid = f2bf2(a, b);
  lo = f2bf2(a - bf_lo(mid), b - bf_hi(mid));
}

// bias, activation or residual, and the outputs of one column of eight rows m, m + step, ... (uniform over a wave)
struct CvBases { int res, raw, act; };
__device__ __forceinline__ void cv_finish_rows(const CvGemm& p, const CvBases& b, int m, int step, int t, float (&y)[8]) {
  // one condition around eight rows each: with the conditions inside the rows every load was waited for by itself
  int ch[8], col[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) { ch[e] = m + e * step; col[e] = t; }
  if (p.bias) {
    float v[8];
    if (p.bias_div == 1) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = p.bias[ch[e]];
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = p.bias[ch[e] / p.bias_div];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] += v[e];
  }
  if (p.tc_stride > 0) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int c = ch[e] / p.tc_stride;
      col[e] = t * p.tc_stride + (ch[e] - c * p.tc_stride);
      ch[e] = c;
    }
  }
  if (p.epi == EPI_GELU) {
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = 0.5f * y[e] * (1.0f + erff(y[e] * 0.70710678118654752f));
  } else if (p.epi == EPI_RES || p.epi == EPI_SCALE_RES) {
    float v[8], sc[8] = {1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f};
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = *ring_ptr(p.res, b.res, ch[e], p.res.pad + col[e]);
    if (p.epi == EPI_SCALE_RES) {
#pragma unroll
      for (int e = 0; e < 8; ++e) sc[e] = p.scale[ch[e]];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = v[e] + sc[e] * y[e];
  }
  if (p.out_raw.p) {
#pragma unroll
    for (int e = 0; e < 8; ++e) *ring_ptr(p.out_raw, b.raw, ch[e], p.out_raw.pad + col[e]) = y[e];
  }
  if (p.out_act.p) {
    float ea[8], ib[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) { ea[e] = p.ea[ch[e]]; ib[e] = p.ib[ch[e]]; }
    float v[8];
    cv_snake(y, ea, ib, v);
#pragma unroll
    for (int e = 0; e < 8; ++e) *ring_ptr(p.out_act, b.act, ch[e], p.out_act.pad + col[e]) = v[e];
  }
}

template <int MI, int NI, int WM, int WN>
__global__ __launch_bounds__(256, 2) void cv_wide_kernel(const CvGemm p) {
  constexpr int NT = 256, BM = 32 * MI * WM, BN = 32 * NI * WN, BS = BN + 8, CW = BN + CVW_HALO;
  constexpr int NA = (BM * 8 + NT - 1) / NT, NB = (CW * 4 + NT - 1) / NT;  // 16-byte loads per thread and unit, pieces of 8 channels and group
  static_assert(WM * WN == 4 && NT % BN == 0, "four waves, whole columns per thread");
  constexpr int PA = BM * 64, PB = CW * 64;  // bytes of one plane of the weights, of the columns
  constexpr bool TWO = 2 * (6 * PA + 3 * PB) <= 160 * 1024;  // a second buffer for weights: two workgroups still share a CU
  constexpr int OPS = (TWO ? 6 : 3) * PA + 3 * PB;
  __shared__ __align__(16) char raw[OPS > BM * BS * 4 ? OPS : BM * BS * 4];  // the operands, then the sums
  float* const lds = reinterpret_cast<float*>(raw);
  auto la = [&](int buf, int plane, int row, int piece) { return reinterpret_cast<bf16_t*>(raw + 3 * PB + (buf * 3 + plane) * PA) + cv_at(row, piece); };
  auto lb = [&](int plane, int col, int piece) { return reinterpret_cast<bf16_t*>(raw + plane * PB) + cv_at(col, piece); };
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l32 = lane & 31, h = lane >> 5, wm = wave % WM, wn = wave / WM;
  // Workgroups go round the eight XCDs, whose L2s are their own: each gets a contiguous range of the tiles, columns slowest, so that
  // it meets an eighth of the input (or, of few columns, of the weights) instead of all of it.
  // (384 channels x 5120 columns: 66 -> 63 us, 768 x 1280 54 -> 53.)
  const int MT = p.M / BM, NTL = (p.T + BN - 1) / BN;
  const int n8 = MT * NTL * p.splits, x8 = blockIdx.x & 7, at = x8 * (n8 >> 3) + min(x8, n8 & 7) + (int)(blockIdx.x >> 3);
  const int tz = at / MT, tl = tz / p.splits;
  const int m0 = (at - tz * MT) * BM, t0 = tl * BN, z = tz - tl * p.splits, cols = NTL * BN;
  const int G = p.Cin >> 5, Uall = p.taps * G;
  const int ub = (int)((int64_t)Uall * z / p.splits), ue = (int)((int64_t)Uall * (z + 1) / p.splits);
  const int f = *p.ctr - p.nf;

  // acc: the products of CVW_RUN units; sum: those before.  One chain over all units (168 of them in block 1) would
  // round each step against the full sum: 1.4 times the error against 64 bits of the audio.
  floatx16 acc[MI][NI], sum[MI][NI];
  const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int n = 0; n < NI; ++n) acc[i][n] = sum[i][n] = zero;

  floatx4 ra[NA];  // native vectors: an array of HIP's float4 structs stayed in scratch memory
  float rb[NB][8];
  // This thread's pieces of a group's columns, BN and the taps' halo: eight channels of a column each.
  const int W = BN + (p.taps - 1) * p.dil;
  int pc[NB];  // column and piece
  uint32_t xoff[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int q = min(tid + i * NT, 4 * W - 1), k = (q >= W) + (q >= 2 * W) + (q >= 3 * W), c = q - k * W;
    pc[i] = c * 4 + k;
    xoff[i] = (uint32_t)(8 * k * p.in.rs + c);
  }
  const uint32_t woff = (tid >> 3) * p.Cin + (tid & 7) * 4;
  auto fetch_w = [&](int tap, int grp) {
    const float* wp = p.W + ((size_t)tap * p.M + m0) * p.Cin + grp * 32;  // uniform, with offsets of the thread's own
#pragma unroll
    for (int i = 0; i < NA; ++i)
      if ((i + 1) * (NT / 8) <= BM || (tid >> 3) + i * (NT / 8) < BM) ra[i] = *reinterpret_cast<const floatx4*>(wp + (size_t)i * (NT / 8) * p.Cin + woff);
  };
  auto fetch_x = [&](int grp) {
    // a block's buffer has no end to turn at; columns behind T are whatever is there: they reach no output
    const float* xp = p.in.p + (size_t)grp * 32 * p.in.rs + t0;
#pragma unroll
    for (int i = 0; i < NB; ++i)
      if ((i + 1) * NT <= 4 * BN || tid + i * NT < 4 * W) {
#pragma unroll
        for (int e = 0; e < 8; ++e) rb[i][e] = xp[(size_t)e * p.in.rs + xoff[i]];
      }
  };
  auto stage_w = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NA; ++i)
      if ((i + 1) * (NT / 8) <= BM || (tid >> 3) + i * (NT / 8) < BM) {
        uint2 q[3];
        cv_split2(ra[i][0], ra[i][1], q[0].x, q[1].x, q[2].x);
        cv_split2(ra[i][2], ra[i][3], q[0].y, q[1].y, q[2].y);
#pragma unroll
        for (int k = 0; k < 3; ++k) *reinterpret_cast<uint2*>(la(buf, k, (tid >> 3) + (NT / 8) * i, (tid & 7) >> 1) + (tid & 1) * 4) = q[k];
      }
  };
  auto stage_x = [&]() {
#pragma unroll
    for (int i = 0; i < NB; ++i)
      if ((i + 1) * NT <= 4 * BN || tid + i * NT < 4 * W) {
        uint4 q[3];
        cv_split2(rb[i][0], rb[i][1], q[0].x, q[1].x, q[2].x);
        cv_split2(rb[i][2], rb[i][3], q[0].y, q[1].y, q[2].y);
        cv_split2(rb[i][4], rb[i][5], q[0].z, q[1].z, q[2].z);
        cv_split2(rb[i][6], rb[i][7], q[0].w, q[1].w, q[2].w);
#pragma unroll
        for (int k = 0; k < 3; ++k) *reinterpret_cast<uint4*>(lb(k, pc[i] >> 2, pc[i] & 3)) = q[k];
      }
  };
  auto frag = [](const bf16_t* q) { return __builtin_bit_cast(cv_bf16x8, *reinterpret_cast<const uint4*>(q)); };
  int grp = ub / p.taps, tap = ub - grp * p.taps;  // a group's taps one after the other
  if (ub < ue) {
    fetch_w(tap, grp);
    fetch_x(grp);
    stage_w(0);
    stage_x();
  }
  __syncthreads();
  for (int u = ub; u < ue; ++u) {
    const int col = tap * p.dil, buf = TWO ? (u - ub) & 1 : 0;
    const bool more = u + 1 < ue, turn = tap + 1 == p.taps;  // uniform; turn: the next unit is another group's
    if (turn) { tap = 0; ++grp; } else ++tap;
    if (more) {
      fetch_w(tap, grp);
      if (turn) fetch_x(grp);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {  // 16 channels: a lane holds eight of its row or column
      cv_bf16x8 a[3][MI], x[3][NI];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
#pragma unroll
        for (int i = 0; i < MI; ++i) a[k][i] = frag(la(buf, k, (wm * MI + i) * 32 + l32, 2 * j + h));
#pragma unroll
        for (int n = 0; n < NI; ++n) x[k][n] = frag(lb(k, (wn * NI + n) * 32 + l32 + col, 2 * j + h));
      }
      // {part of the weight, part of the input}
      constexpr int PAIR[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};
#pragma unroll
      for (int c = 0; c < 6; ++c)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int n = 0; n < NI; ++n)
            acc[i][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[PAIR[c][0]][i], x[PAIR[c][1]][n], acc[i][n], 0, 0, 0);
    }
    if ((u - ub) % CVW_RUN == CVW_RUN - 1 || u + 1 == ue) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int n = 0; n < NI; ++n) { sum[i][n] += acc[i][n]; acc[i][n] = zero; }
    }
    if (TWO && more) stage_w(buf ^ 1);
    if (!TWO || turn || !more) __syncthreads();
    if (more) {
      if (!TWO) stage_w(0);
      if (turn) stage_x();
      __syncthreads();
    }
  }

  if (p.splits > 1) {  // cv_finish_kernel adds the parts
    float* part = p.part + ((size_t)z * p.M + m0) * cols + t0 + wn * NI * 32 + l32;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r)
#pragma unroll
        for (int n = 0; n < NI; ++n)
          part[(size_t)((wm * MI + i) * 32 + 8 * (r >> 2) + 4 * h + (r & 3)) * cols + n * 32] = sum[i][n][r];
    return;
  }
  // The sums go through LDS so that a wave finishes whole rows: what depends on the row is scalar, and 64 columns are
  // written in a run.
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int n = 0; n < NI; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        lds[((wm * MI + i) * 32 + 8 * (r >> 2) + 4 * h + (r & 3)) * BS + (wn * NI + n) * 32 + l32] = sum[i][n][r];
  __syncthreads();
  constexpr int RW = NT / BN;  // rows that the workgroup finishes side by side
  const int t = t0 + tid % BN, row0 = wave / (BN / 64);
  if (t >= p.T) return;
  const CvBases b{ring_base(p.res, f), ring_base(p.out_raw, f), ring_base(p.out_act, f)};
  static_assert(BM % (8 * RW) == 0, "whole batches of rows");
  for (int row = row0; row < BM; row += 8 * RW) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = lds[(row + e * RW) * BS + tid % BN];
    cv_finish_rows(p, b, m0 + row, RW, t, v);
  }
}

// Parts of the tiles of cv_wide_kernel, (splits, M, cols), added in order: a wave per 64 columns x 8 rows.  A launch of
// its own: with the last of a tile's workgroups adding and finishing 128 x 128 results by itself, the 1x1 convolutions of
// block 1 took 85 us per 32 frames, 7 us of it products.
__global__ __launch_bounds__(256) void cv_finish_kernel(const CvGemm p, int cols) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t = blockIdx.x * 64 + (threadIdx.x & 63);
  const int m = blockIdx.y * 32 + wave * 8;
  if (t >= p.T) return;
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int z = 0; z < p.splits; ++z) {
    const float* src = p.part + ((size_t)z * p.M + m) * cols + t;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] += src[(size_t)e * cols];
  }
  const int f = *p.ctr - p.nf;
  cv_finish_rows(p, CvBases{ring_base(p.res, f), ring_base(p.out_raw, f), ring_base(p.out_act, f)}, m, 1, t, v);
}

// ---- codebook rows of one frame per workgroup: [sum of the semantic rows | sum of the acoustic rows]; starts the pass ----
struct CvVq {
  const int64_t* codes;  // (nf, n_q)
  int n_q, n_sem, CS, cd;
  const float* embed;  // (n_codebooks, CS, cd)
  float* x;            // (2*cd, rs): a column per frame
  int rs, nf;
  int* ctr;
  int* err;
  int max_seq;
};

__global__ __launch_bounds__(256) void cv_vq_kernel(const CvVq p) {
  const int64_t* codes = p.codes + (size_t)blockIdx.x * p.n_q;
  for (int c = threadIdx.x; c < p.cd; c += blockDim.x) {
    float s0 = 0.f, s1 = 0.f;
    for (int i0 = 0; i0 < p.n_q; i0 += 16) {  // 16 codes, then their 16 rows, are requested together
      long code[16];
      float e[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) code[k] = i0 + k < p.n_q ? codes[i0 + k] : 0;
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        if (code[k] < 0 || code[k] >= p.CS) { code[k] = code[k] < 0 ? 0 : p.CS - 1; if (c == 0) *p.err = 1; }
        e[k] = i0 + k < p.n_q ? p.embed[((size_t)(i0 + k) * p.CS + code[k]) * p.cd + c] : 0.f;
      }
#pragma unroll
      for (int k = 0; k < 16; ++k) {  // the reference's order: codebook after codebook
        if (i0 + k < p.n_sem) s0 += e[k]; else s1 += e[k];
      }
    }
    p.x[(size_t)c * p.rs + blockIdx.x] = s0;
    p.x[(size_t)(p.cd + c) * p.rs + blockIdx.x] = s1;
  }
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    int f = *p.ctr;
    if (f + p.nf > p.max_seq) { *p.err = 2; f = p.max_seq - p.nf; }  // stay on the last positions: nothing runs out of bounds
    *p.ctr = f + p.nf;
  }
}

// ---- pre-transformer attention of nf new positions: rotate-half RoPE, cache append, softmax, P.V ----
struct CvAttn {
  const float* qkv;  // (3*A, rs): q | k | v, a column per position
  float* kc;         // (H, max_seq, hd)
  float* vc;
  float* out;        // (A, rs_out)
  const float* inv_freq;  // (hd/2)
  int rs, rs_out, H, hd, max_seq, nf;
  const int* ctr;
};

// keys and values of several positions, ahead of the launch that attends: workgroup (head, position)
__global__ __launch_bounds__(64) void cv_append_kernel(const CvAttn p) {
  const int h = blockIdx.x, i = blockIdx.y, d = threadIdx.x, hd = p.hd, half = hd >> 1, A = p.H * hd;
  const int pos = *p.ctr - p.nf + i;
  if (d >= hd) return;
  const float ang = (float)pos * p.inv_freq[d % half];
  const float* kk = p.qkv + (size_t)(A + h * hd) * p.rs + i;
  const float kr = d < half ? -kk[(size_t)(d + half) * p.rs] : kk[(size_t)(d - half) * p.rs];
  const size_t at = ((size_t)h * p.max_seq + pos) * hd + d;
  p.kc[at] = kk[(size_t)d * p.rs] * cosf(ang) + kr * sinf(ang);
  p.vc[at] = p.qkv[(size_t)(2 * A + h * hd + d) * p.rs + i];
}

__global__ __launch_bounds__(256) void cv_attn_kernel(const CvAttn p) {
  extern __shared__ float sm[];  // q[hd] | sc[max_seq] | part[4][hd] | red[8]
  float* q = sm;
  float* sc = q + p.hd;
  float* part = sc + p.max_seq;
  float* red = part + 4 * p.hd;
  const int h = blockIdx.x, tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int hd = p.hd, half = hd >> 1, A = p.H * hd;
  const int pos = *p.ctr - p.nf + (int)blockIdx.y;
  float* kh = p.kc + (size_t)h * p.max_seq * hd;
  float* vh = p.vc + (size_t)h * p.max_seq * hd;
  if (tid < hd) {
    const float ang = (float)pos * p.inv_freq[tid % half];
    const float cs = cosf(ang), sn = sinf(ang);
    const size_t rs = p.rs;
    const float* qq = p.qkv + h * hd * rs + blockIdx.y;
    const float qr = tid < half ? -qq[(tid + half) * rs] : qq[(tid - half) * rs];
    q[tid] = qq[tid * rs] * cs + qr * sn;
    if (p.nf == 1) {
      const float* kk = qq + A * rs;
      const float kr = tid < half ? -kk[(tid + half) * rs] : kk[(tid - half) * rs];
      kh[(size_t)pos * hd + tid] = kk[tid * rs] * cs + kr * sn;
      vh[(size_t)pos * hd + tid] = kk[(A + tid) * rs];
    }
  }
  __syncthreads();  // this workgroup's own cache row is visible to all its threads after the barrier
  // scores: a group of 16 lanes per key (features l16, l16 + 16, ...), four keys of a group in flight
  const float scale = 1.0f / sqrtf((float)hd);
  const int grp = tid >> 4, l16 = tid & 15, E = hd >> 4;
  float qe[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) qe[e] = e < E ? q[l16 + 16 * e] : 0.f;
  for (int j0 = grp; j0 <= pos; j0 += 64) {
    float kv[4][4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = j0 + 16 * u;
#pragma unroll
      for (int e = 0; e < 4; ++e) kv[u][e] = (j <= pos && e < E) ? kh[(size_t)j * hd + l16 + 16 * e] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = j0 + 16 * u;
      float d = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) d = fmaf(qe[e], kv[u][e], d);
      d = group16_sum(d);
      if (l16 == 0 && j <= pos) sc[j] = d * scale;
    }
  }
  __syncthreads();
  float mx = -INFINITY;
  for (int j = tid; j <= pos; j += 256) mx = fmaxf(mx, sc[j]);
  mx = wave_max(mx);
  if (lane == 0) red[wave] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float sum = 0.f;
  for (int j = tid; j <= pos; j += 256) { const float e = expf(sc[j] - mx); sc[j] = e; sum += e; }
  sum = wave_sum(sum);
  if (lane == 0) red[4 + wave] = sum;
  __syncthreads();
  sum = (red[4] + red[5]) + (red[6] + red[7]);
  // P.V: wave w takes keys w, w + 4, ...; eight rows in flight
  float o = 0.f;
  if (lane < hd) {
    for (int j0 = wave; j0 <= pos; j0 += 32) {
      float vv[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) { const int j = j0 + 4 * u; vv[u] = j <= pos ? vh[(size_t)j * hd + lane] : 0.f; }
#pragma unroll
      for (int u = 0; u < 8; ++u) { const int j = j0 + 4 * u; o = fmaf(j <= pos ? sc[j] : 0.f, vv[u], o); }
    }
    part[wave * hd + lane] = o;
  }
  __syncthreads();
  if (tid < hd) p.out[(size_t)(h * hd + tid) * p.rs_out + blockIdx.y] = ((part[tid] + part[hd + tid]) + (part[2 * hd + tid] + part[3 * hd + tid])) / sum;
}

// =============================================================================================
// The one-column trunk as ONE persistent kernel: codebook rows -> quantizer projection -> pre_conv
// -> input_proj -> the transformer layers -> output_proj -> first upsampling transposed conv.
// These 46 steps have one column each (1-3 MB of weights), so as separate launches they run at the
// cost of a dependent launch.  Here 256 workgroups (one per CU) walk the same list of phases; every
// workgroup owns a few rows of every matrix, keeps the residual stream and the current input vector
// in LDS, requests the weights of the next phase before it waits, and passes results as 8-byte
// words = fp32 payload + launch epoch (device-scope relaxed atomics: a word showing the epoch is the
// data).  Exchange buffers are never reused inside a launch.  Every wait is bounded.
// =============================================================================================
#include "ll.h"

struct TrunkLayer {
  const float* Wqkv; const float* Wo; const float* asc; const float* Wgu; const float* Wd; const float* msc;
  float* kc; float* vc;
};

struct CvTrunk {
  const int64_t* codes;
  int n_q, n_sem, CS, cd;
  const float* embed;
  int* ctr;
  int* err;
  int max_seq;
  const float* Wvq; int vq_dim;
  const float* Wpre; const float* bpre; int L;
  Ring pre_in;
  const float* Win; const float* bin; int D;
  int n_layers, H, hd, mlp;
  const TrunkLayer* layers;
  const float* inv_freq;
  const float* Wout; const float* bout;
  const float* Wt0; const float* bt0; int r0;  // Wt0 == nullptr: no upsampling stage, `out` takes the latent
  Ring out;
  uint64_t* ll;
  uint32_t* epoch; uint32_t* arrive; uint32_t* lerr;
  float eps;
};

#define TR_MAXC 6   // float4 chunks per lane and row: K <= 1536
#define TR_REGS 24  // float4 registers of a wave's rows of one phase: rows per wave x chunks per row

// Rows per wave, phase by phase.  The kernel is built for a whole GPU (256 workgroups) and for the share of one that a
// caller leaves to the vocoder beside other work (NARROW: 96 workgroups and more): a workgroup then owns 256 / 96
// times the rows, and every phase keeps its rows x chunks within TR_REGS registers.
template <bool NARROW> struct TrPlan {
  static constexpr int VQ = NARROW ? 2 : 1, PRE = NARROW ? 3 : 1, IN = NARROW ? 2 : 1, QKV = NARROW ? 10 : 4, O = NARROW ? 2 : 1,
                       GU = NARROW ? 6 : 4, DN = NARROW ? 2 : 1, OUT = NARROW ? 3 : 1, UP = NARROW ? 6 : 4;
};

struct TrRows { float4 w[TR_REGS]; };

// rows r_lo + wave, r_lo + wave + 4, ... below r_hi of W (M x K): request them
template <int MAXR, int MAXC>
__device__ __forceinline__ void tr_prefetch(const float* W, int K, int r_lo, int r_hi, TrRows& rr) {
  static_assert(MAXR * MAXC <= TR_REGS, "rows x chunks of a phase exceed the wave's registers");
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < MAXR; ++i) {
    const int row = r_lo + wave + 4 * i;
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
      const int k = (lane + 64 * c) * 4;
      const bool on = row < r_hi && k < K;
      rr.w[i * MAXC + c] = on ? *reinterpret_cast<const float4*>(W + (size_t)row * K + k) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
}
// dot products of those rows with xs (K floats in LDS); epi(row, sum) runs in every lane of the wave
template <int MAXR, int MAXC, typename F>
__device__ __forceinline__ void tr_compute(const float* xs, int K, int r_lo, int r_hi, const TrRows& rr, F&& epi) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < MAXR; ++i) {
    const int row = r_lo + wave + 4 * i;
    if (row < r_hi) {
      float s = 0.f;
#pragma unroll
      for (int c = 0; c < MAXC; ++c) {
        const int k = (lane + 64 * c) * 4;
        if (k < K) {
          const float4 x = *reinterpret_cast<const float4*>(xs + k);
          const float4 w = rr.w[i * MAXC + c];
          s = fmaf(w.x, x.x, s); s = fmaf(w.y, x.y, s);
          s = fmaf(w.z, x.z, s); s = fmaf(w.w, x.w, s);
        }
      }
      s = wave_sum(s);
      epi(row, s);
    }
  }
}

__device__ __forceinline__ void tr_rows(int M, int wg, int nwg, int& lo, int& hi) {
  const int per = (M + nwg - 1) / nwg;
  lo = min(M, wg * per);
  hi = min(M, lo + per);
}

// q/k/v rows: the head-owning workgroups (the first H) stay out of this phase when enough others exist; they
// use the time to fetch their key / value history
__device__ __forceinline__ void tr_rows_qkv(int M, int wg, int nwg, int H, int& lo, int& hi) {
  if (nwg >= 4 * H) {
    if (wg < H) { lo = hi = M; return; }
    tr_rows(M, wg - H, nwg - H, lo, hi);
  } else {
    tr_rows(M, wg, nwg, lo, hi);
  }
}

__device__ __forceinline__ float tr_rstd(const float* x, int n, float eps, float* red) {
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  float ss = 0.f;
  for (int i = tid; i < n; i += FR_THREADS) ss = fmaf(x[i], x[i], ss);
  ss = wave_sum(ss);
  __syncthreads();
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  return 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)n + eps);
}

template <bool NARROW>
__global__ __launch_bounds__(FR_THREADS) void cv_trunk_kernel(const CvTrunk a) {
  typedef TrPlan<NARROW> P;
  extern __shared__ __align__(16) float tsm[];
  // xs: current input vector (<= 1536) | x: residual stream (D) | q (hd) | sc (max_seq) | part (4*hd) | red (16)
  float* xs = tsm;
  float* x = xs + 1536;
  float* q = x + a.D;
  float* sc = q + 64;  // max_seq + 192: scores, and before them the raw q | k | v of the head
  float* part = sc + a.max_seq + 192;
  float* red = part + 4 * 64;
  const int wg = blockIdx.x, nwg = gridDim.x, tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  Ctl c;
  ctl_begin(c, a.epoch, a.lerr);
  const uint32_t ep = c.epoch;
  int f = *a.ctr;
  const bool over = f >= a.max_seq;
  if (over) f = a.max_seq - 1;  // stay on the last position: nothing runs out of bounds
  // the epoch and the frame counter have been read before this workgroup reports its arrival
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  if (tid == 0) __hip_atomic_fetch_add(a.arrive, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

  uint64_t* ll = a.ll;
  auto take = [&](int n) { uint64_t* p = ll; ll += n; return p; };
  auto put = [&](uint64_t* buf, int i, float v) { ll_st(buf + i, __float_as_uint(v), ep); };
  auto get = [&](const uint64_t* buf, int n, float* dst) {
    ll_poll_auto(buf, n, c, [&](int i, uint32_t v) { dst[i] = __uint_as_float(v); });
    __syncthreads();
  };
  TrRows rr;
  int lo, hi;
  const int cd = a.cd, V = a.vq_dim, L = a.L, D = a.D, A = a.H * a.hd, hd = a.hd, mlp = a.mlp;

  // ---- quantizer projection: rows of [W_sem | W_ac] against [sum of semantic rows | sum of acoustic rows] ----
  tr_rows(V, wg, nwg, lo, hi);
  tr_prefetch<P::VQ, 2>(a.Wvq, 2 * cd, lo, hi, rr);
  for (int ch = tid; ch < cd; ch += FR_THREADS) {  // every workgroup sums the codebook rows itself
    float s0 = 0.f, s1 = 0.f;
    for (int i0 = 0; i0 < a.n_q; i0 += 16) {
      long code[16];
      float e[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) code[k] = i0 + k < a.n_q ? a.codes[i0 + k] : 0;
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        if (code[k] < 0 || code[k] >= a.CS) { code[k] = code[k] < 0 ? 0 : a.CS - 1; if (ch == 0 && wg == 0) *a.err = 1; }
        e[k] = i0 + k < a.n_q ? a.embed[((size_t)(i0 + k) * a.CS + code[k]) * cd + ch] : 0.f;
      }
#pragma unroll
      for (int k = 0; k < 16; ++k) { if (i0 + k < a.n_sem) s0 += e[k]; else s1 += e[k]; }
    }
    xs[ch] = s0;
    xs[cd + ch] = s1;
  }
  __syncthreads();
  uint64_t* b_y1 = take(V);
  const int pbase = ring_base(a.pre_in, f);
  tr_compute<P::VQ, 2>(xs, 2 * cd, lo, hi, rr, [&](int row, float s) {
    if (lane == 0) { put(b_y1, row, s); *ring_ptr(a.pre_in, pbase, row, a.pre_in.pad) = s; }
  });
  // ---- pre_conv: three taps = the two previous frames' columns and this one ----
  tr_rows(L, wg, nwg, lo, hi);
#pragma unroll
  for (int i = 0; i < P::PRE; ++i) {
    const int wave_row = lo + wave + 4 * i;  // (3, L, V) tap-major
#pragma unroll
    for (int cc = 0; cc < TR_MAXC; ++cc) {
      const int k = (lane + 64 * cc) * 4;  // index into [tap][ci]
      const int tap = k / V, ci = k - tap * V;
      const bool on = wave_row < hi && k < 3 * V;
      rr.w[i * TR_MAXC + cc] = on ? *reinterpret_cast<const float4*>(a.Wpre + ((size_t)tap * L + wave_row) * V + ci) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  __syncthreads();  // xs is free again
  for (int i = tid; i < 2 * V; i += FR_THREADS) xs[i] = *ring_ptr(a.pre_in, pbase, i % V, i / V);
  ll_poll_auto(b_y1, V, c, [&](int i, uint32_t v) { xs[2 * V + i] = __uint_as_float(v); });
  __syncthreads();
  uint64_t* b_pre = take(L);
  tr_compute<P::PRE, TR_MAXC>(xs, 3 * V, lo, hi, rr, [&](int row, float s) { if (lane == 0) put(b_pre, row, s + a.bpre[row]); });
  // ---- input_proj ----
  tr_rows(D, wg, nwg, lo, hi);
  tr_prefetch<P::IN, 4>(a.Win, L, lo, hi, rr);
  __syncthreads();
  get(b_pre, L, xs);
  uint64_t* b_x = take(D);
  tr_compute<P::IN, 4>(xs, L, lo, hi, rr, [&](int row, float s) { if (lane == 0) put(b_x, row, s + a.bin[row]); });
  {
    int qlo, qhi;
    tr_rows_qkv(3 * A, wg, nwg, a.H, qlo, qhi);
    tr_prefetch<P::QKV, 2>(a.layers[0].Wqkv, D, qlo, qhi, rr);
  }
  get(b_x, D, x);

  const float att_scale = 1.0f / sqrtf((float)hd);
  // rotation of this position: the same for every layer, computed once and before any q arrives
  float rope_cs = 1.f, rope_sn = 0.f;
  if (wg < a.H && tid < hd) {
    const float ang = (float)f * a.inv_freq[tid % (hd >> 1)];
    rope_cs = cosf(ang);
    rope_sn = sinf(ang);
  }
  for (int l = 0; l < a.n_layers; ++l) {
    const TrunkLayer& W = a.layers[l];
    // The head's workgroup asks for its whole key / value history now (at most 256 earlier positions: 16 per
    // lane group, 4 features per lane), long before the new q arrives: attention then runs from registers,
    // whatever the position.
    float kreg[16][4], vreg[16][4];
    if (wg < a.H) {
      const float* kh = W.kc + (size_t)wg * a.max_seq * hd;
      const float* vh = W.vc + (size_t)wg * a.max_seq * hd;
      const int g16 = tid >> 4, c16 = tid & 15, E = hd >> 4;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int j = g16 + 16 * i;
#pragma unroll
        for (int e = 0; e < 4; ++e) { kreg[i][e] = 0.f; vreg[i][e] = 0.f; }
        if (16 * i < f) {  // uniform: blocks of 16 positions that do not exist yet cost nothing
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const bool on = j < f && e < E;
            kreg[i][e] = on ? kh[(size_t)j * hd + c16 + 16 * e] : 0.f;
            vreg[i][e] = on ? vh[(size_t)j * hd + c16 + 16 * e] : 0.f;
          }
        }
      }
    }
    // ---- q, k, v rows (norm weight folded in; 1/rms multiplies the sums) ----
    const float r1 = tr_rstd(x, D, a.eps, red);
    tr_rows_qkv(3 * A, wg, nwg, a.H, lo, hi);
    uint64_t* b_qkv = take(3 * A);
    tr_compute<P::QKV, 2>(x, D, lo, hi, rr, [&](int row, float s) { if (lane == 0) put(b_qkv, row, s * r1); });
    uint64_t* b_att = take(A);
    int olo, ohi;
    tr_rows(D, wg, nwg, olo, ohi);
    tr_prefetch<P::O, 4>(W.Wo, A, olo, ohi, rr);
    // ---- attention: workgroup h owns head h ----
    if (wg < a.H) {
      const int h = wg, half = hd >> 1, pos = f;
      float* kh = W.kc + (size_t)h * a.max_seq * hd;
      float* vh = W.vc + (size_t)h * a.max_seq * hd;
      float* kvn = part;  // this position's rotated key | value
      __syncthreads();
      if (tid < 3 * hd) {
        const int which = tid / hd, i = tid - which * hd;
        const uint64_t* src = b_qkv + which * A + h * hd + i;
        uint64_t v = ll_ld(src);
        int spins = 0;
        while ((uint32_t)(v >> 32) != ep && !c.dead) {
          v = ll_ld(src);
          if (++spins > SPIN_LIMIT) { c.dead = 1; __hip_atomic_store(c.err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
        }
        sc[which * hd + i] = __uint_as_float((uint32_t)v);  // raw q | k | v
      }
      __syncthreads();
      if (tid < hd) {
        const float cs = rope_cs, sn = rope_sn;
        const float* qq = sc;
        const float* kk = sc + hd;
        const float qr = tid < half ? -qq[tid + half] : qq[tid - half];
        const float kr = tid < half ? -kk[tid + half] : kk[tid - half];
        q[tid] = qq[tid] * cs + qr * sn;
        const float kn = kk[tid] * cs + kr * sn, vn = sc[2 * hd + tid];
        kvn[tid] = kn; kvn[hd + tid] = vn;
        kh[(size_t)pos * hd + tid] = kn;
        vh[(size_t)pos * hd + tid] = vn;
      }
      __syncthreads();
      const int grp = tid >> 4, l16 = tid & 15, E = hd >> 4;
      float qe[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) qe[e] = e < E ? q[l16 + 16 * e] : 0.f;
      __syncthreads();  // sc is rewritten below
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int j = grp + 16 * i;
        if (j <= pos) {  // uniform over the 16 lanes of a group
          float d = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e) d = fmaf(qe[e], (j == pos && e < E) ? kvn[l16 + 16 * e] : kreg[i][e], d);
          d = group16_sum(d);
          if (l16 == 0) sc[j] = d * att_scale;
        }
      }
      __syncthreads();
      float mx = -INFINITY;
      for (int j = tid; j <= pos; j += FR_THREADS) mx = fmaxf(mx, sc[j]);
      mx = wave_max(mx);
      if (lane == 0) red[wave] = mx;
      __syncthreads();
      mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
      float sum = 0.f;
      for (int j = tid; j <= pos; j += FR_THREADS) { const float e = expf(sc[j] - mx); sc[j] = e; sum += e; }
      sum = wave_sum(sum);
      if (lane == 0) red[4 + wave] = sum;
      __syncthreads();
      sum = (red[4] + red[5]) + (red[6] + red[7]);
      // P.V per lane group over its own keys, then the 16 groups are added in order (xs is free here)
      float o4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int j = grp + 16 * i;
        if (j <= pos) {
          const float pj = sc[j];
#pragma unroll
          for (int e = 0; e < 4; ++e) o4[e] = fmaf(pj, (j == pos && e < E) ? kvn[hd + l16 + 16 * e] : vreg[i][e], o4[e]);
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) if (e < E) xs[grp * hd + l16 + 16 * e] = o4[e];
      __syncthreads();
      if (tid < hd) {
        float o = 0.f;
#pragma unroll
        for (int gg = 0; gg < 16; ++gg) o += xs[gg * hd + tid];
        part[tid] = o / sum;  // kvn (= part) has been read by everyone
      }
      __syncthreads();
      if (tid < hd) put(b_att, h * hd + tid, part[tid]);
    }
    // ---- out_proj, residual with per-channel scale ----
    // the scales of this thread's channels (tid, tid + 256, ...) are asked for ahead of the waits: fetched when
    // the sums arrive, their pointer and then their value would be two trips to memory on the critical path
    float asc_r[6], msc_r[6];  // d_model <= 1536
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      const int i = tid + FR_THREADS * k;
      asc_r[k] = i < D ? W.asc[i] : 0.f;
      msc_r[k] = i < D ? W.msc[i] : 0.f;
    }
    get(b_att, A, xs);
    uint64_t* b_o = take(D);
    tr_compute<P::O, 4>(xs, A, olo, ohi, rr, [&](int row, float s) { if (lane == 0) put(b_o, row, s); });
    int glo, ghi;
    tr_rows(mlp, wg, nwg, glo, ghi);  // channels; rows 2i, 2i + 1 are gate_i, up_i
    glo *= 2; ghi *= 2;
    tr_prefetch<P::GU, 2>(W.Wgu, D, glo, ghi, rr);
    ll_poll_auto(b_o, D, c, [&](int i, uint32_t v) { x[i] += asc_r[i / FR_THREADS] * __uint_as_float(v); });
    // ---- gate / up rows interleaved: channel i = silu(gate_i) * up_i ----
    const float r2 = tr_rstd(x, D, a.eps, red);
    uint64_t* b_h = take(mlp);
    {
      // a wave's rows glo + wave + 4 i alternate between gate and up of different channels: pair through LDS
      float* pair = part;
      tr_compute<P::GU, 2>(x, D, glo, ghi, rr, [&](int row, float s) { if (lane == 0) pair[row - glo] = s * r2; });
      __syncthreads();
      for (int i = tid; 2 * i + 1 < ghi - glo; i += FR_THREADS) {
        const float ga = pair[2 * i], up = pair[2 * i + 1];
        put(b_h, (glo >> 1) + i, ga / (1.0f + expf(-ga)) * up);
      }
    }
    int dlo, dhi;
    tr_rows(D, wg, nwg, dlo, dhi);
    tr_prefetch<P::DN, 4>(W.Wd, mlp, dlo, dhi, rr);
    get(b_h, mlp, xs);
    uint64_t* b_d = take(D);
    tr_compute<P::DN, 4>(xs, mlp, dlo, dhi, rr, [&](int row, float s) { if (lane == 0) put(b_d, row, s); });
    if (l + 1 < a.n_layers) {
      int qlo, qhi;
      tr_rows_qkv(3 * A, wg, nwg, a.H, qlo, qhi);
      tr_prefetch<P::QKV, 2>(a.layers[l + 1].Wqkv, D, qlo, qhi, rr);
    } else {
      int plo, phi;
      tr_rows(L, wg, nwg, plo, phi);
      tr_prefetch<P::OUT, 2>(a.Wout, D, plo, phi, rr);
    }
    ll_poll_auto(b_d, D, c, [&](int i, uint32_t v) { x[i] += msc_r[i / FR_THREADS] * __uint_as_float(v); });
  }
  // ---- final norm (folded) + output_proj ----
  const float r3 = tr_rstd(x, D, a.eps, red);
  tr_rows(L, wg, nwg, lo, hi);
  const int obase = ring_base(a.out, f);
  if (a.Wt0 == nullptr) {
    tr_compute<P::OUT, 2>(x, D, lo, hi, rr, [&](int row, float s) {
      if (lane == 0) *ring_ptr(a.out, obase, row, a.out.pad) = s * r3 + a.bout[row];
    });
  } else {
    uint64_t* b_lat = take(L);
    tr_compute<P::OUT, 2>(x, D, lo, hi, rr, [&](int row, float s) { if (lane == 0) put(b_lat, row, s * r3 + a.bout[row]); });
    // ---- first upsampling stage: transposed conv with kernel = stride: row m -> channel m / r0, column m % r0 ----
    tr_rows(L * a.r0, wg, nwg, lo, hi);
    tr_prefetch<P::UP, 4>(a.Wt0, L, lo, hi, rr);
    __syncthreads();
    get(b_lat, L, xs);
    tr_compute<P::UP, 4>(xs, L, lo, hi, rr, [&](int row, float s) {
      if (lane == 0) *ring_ptr(a.out, obase, row / a.r0, a.out.pad + row % a.r0) = s + a.bt0[row / a.r0];
    });
  }
  if (wg == 0 && tid == 0) {
    // every workgroup has read the epoch and the frame counter before they may change
    ctl_finish(c, a.epoch, a.arrive, (uint32_t)nwg);
    if (over) *a.err = 2;
    *a.ctr = f + 1;
  }
}

// ---- depthwise causal conv (k taps) + LayerNorm over channels, one workgroup per column ----
struct CvDwLn {
  Ring in;           // pad = k - 1
  const float* w;    // (C, k)
  const float* b;    // (C)
  const float* lnw;
  const float* lnb;
  float* out;        // (C, rs_out) plain
  int rs_out, C, nf;
  float eps;
  const int* ctr;
};

#define DW_MAXC 8  // channels per thread
#define DW_K 7     // taps

__global__ __launch_bounds__(256) void cv_dwln_kernel(const CvDwLn p) {
  __shared__ float red[8];
  const int t = blockIdx.x, tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int f = *p.ctr - p.nf, base = ring_base(p.in, f);
  float v[DW_MAXC];
  float s = 0.f;
  // every load of four channels is requested before the first is needed (a loop over a tap count known only at run time
  // took a round trip per tap: 9.7 us per launch of one frame)
#pragma unroll
  for (int i0 = 0; i0 < DW_MAXC; i0 += 4) {
    if (256 * i0 >= p.C) break;
    float x[4][DW_K], w[4][DW_K], a[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = min(tid + 256 * (i0 + i), p.C - 1);
      a[i] = p.b[c];
#pragma unroll
      for (int k = 0; k < DW_K; ++k) { x[i][k] = *ring_ptr(p.in, base, c, t + k); w[i][k] = p.w[c * DW_K + k]; }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int k = 0; k < DW_K; ++k) a[i] = fmaf(w[i][k], x[i][k], a[i]);
      v[i0 + i] = a[i];
      if (tid + 256 * (i0 + i) < p.C) s += a[i];
    }
  }
  s = wave_sum(s);
  if (lane == 0) red[wave] = s;
  __syncthreads();
  const float mean = ((red[0] + red[1]) + (red[2] + red[3])) / (float)p.C;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < DW_MAXC; ++i) {
    const int c = tid + 256 * i;
    if (c < p.C) { const float d = v[i] - mean; q = fmaf(d, d, q); }
  }
  q = wave_sum(q);
  if (lane == 0) red[4 + wave] = q;
  __syncthreads();
  const float rstd = 1.0f / sqrtf(((red[4] + red[5]) + (red[6] + red[7])) / (float)p.C + p.eps);
#pragma unroll
  for (int i = 0; i < DW_MAXC; ++i) {
    const int c = tid + 256 * i;
    if (c < p.C) p.out[(size_t)c * p.rs_out + t] = (v[i] - mean) * rstd * p.lnw[c] + p.lnb[c];
  }
}

// ---- last conv: one output channel, k taps, clamp to [-1, 1]; 64 samples x 4 channel quarters per workgroup ----
struct CvFinal {
  Ring in;         // pad = k - 1
  const float* w;  // (C, k)
  const float* b;  // (1)
  float* audio;
  int C, k, T, nf;
  const int* ctr;
};

#define FIN_TW 16  // output columns per workgroup: 120 workgroups per frame, and a window small enough that every
                   // thread has all its loads in flight at once (64 columns: 30 workgroups, four rounds of loads)
__global__ __launch_bounds__(256) void cv_final_kernel(const CvFinal p) {
  extern __shared__ float xs[];  // C x (FIN_TW + k - 1) window of the ring | 16 x FIN_TW partial sums | C x k weights
  const int tid = threadIdx.x, qd = tid / FIN_TW, l = tid % FIN_TW;  // 16 channel groups x FIN_TW columns
  const int t0 = blockIdx.x * FIN_TW, W = FIN_TW + p.k - 1;
  const int n = p.C * W;
  float* part = xs + n;
  float* ws = part + 256;
  for (int i = tid; i < p.C * p.k; i += 256) ws[i] = p.w[i];
  const int f = *p.ctr - p.nf, base = ring_base(p.in, f);
  for (int i0 = tid; i0 < n; i0 += 256 * 12) {
    float v[12];
#pragma unroll
    for (int u = 0; u < 12; ++u) {
      const int i = i0 + 256 * u;
      v[u] = i < n ? *ring_ptr(p.in, base, i / W, t0 + i % W) : 0.f;
    }
#pragma unroll
    for (int u = 0; u < 12; ++u) { const int i = i0 + 256 * u; if (i < n) xs[i] = v[u]; }
  }
  __syncthreads();
  float a = 0.f;
  const int c0 = (p.C * qd) / 16, c1 = (p.C * (qd + 1)) / 16;
  for (int c = c0; c < c1; ++c)
    for (int k = 0; k < p.k; ++k) a = fmaf(ws[c * p.k + k], xs[c * W + l + k], a);
  part[qd * FIN_TW + l] = a;
  __syncthreads();
  const int t = t0 + l;
  if (qd == 0 && t < p.T) {
    float y = 0.f;
#pragma unroll
    for (int q = 0; q < 16; ++q) y += part[q * FIN_TW + l];  // group order: a fixed order of the sum
    y += p.b[0];
    p.audio[t] = fminf(1.0f, fmaxf(-1.0f, y));
  }
}

// ---- one-time repacking ----
__global__ void cv_pack_conv_kernel(const float* w, float* wp, int Cout, int Cin, int K) {  // (Cout,Cin,K) -> (K,Cout,Cin)
  const size_t n = (size_t)Cout * Cin * K;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const int ci = (int)(i % Cin);
    const int co = (int)((i / Cin) % Cout);
    const int k = (int)(i / ((size_t)Cin * Cout));
    wp[i] = w[((size_t)co * Cin + ci) * K + k];
  }
}
// ConvTranspose1d (Cin, Cout, K = taps*s) -> (taps, Cout*s, Cin); tap `taps-1` multiplies the current column
__global__ void cv_pack_tconv_kernel(const float* w, float* wp, int Cin, int Cout, int s, int taps) {
  const size_t n = (size_t)taps * Cout * s * Cin;
  const int K = taps * s;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const int ci = (int)(i % Cin);
    const int m = (int)((i / Cin) % ((size_t)Cout * s));
    const int tap = (int)(i / ((size_t)Cin * Cout * s));
    const int co = m / s, r = m % s;
    wp[i] = w[((size_t)ci * Cout + co) * K + r + (taps - 1 - tap) * s];
  }
}
// rows of src (M, K) into dst (M, ld) at column offset off
__global__ void cv_copy_rows_kernel(const float* src, float* dst, int M, int K, int ld, int off) {
  const size_t n = (size_t)M * K;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    dst[(i / K) * ld + off + (i % K)] = src[i];
}
// W (M, K) *= w (K) along every row
__global__ void cv_scale_cols_kernel(float* W, const float* w, int M, int K) {
  const size_t n = (size_t)M * K;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) W[i] *= w[i % K];
}
__global__ void cv_snake_tab_kernel(const float* alpha, const float* beta, float* ea, float* ib, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) { ea[i] = expf(alpha[i]); ib[i] = 1.0f / (expf(beta[i]) + 1e-9f); }
}
__global__ void cv_fill_kernel(float* p, size_t n, float v) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}
// The history columns of every ring into the buffer that stands for it during a block (out = 0), and those behind the
// block's last frame back into the ring.
struct CvHist { Ring ring; size_t at; int rs, C; };  // of a block length; at, rs: the buffer in the scratch memory of the block (floats), its row stride
__global__ void cv_history_kernel(const CvHist* h, float* scratch, const int* ctr, int nf, int out) {
  const CvHist r = h[blockIdx.y];
  const int base = ring_base(r.ring, *ctr - (out ? 0 : nf)), at = out ? nf * r.ring.tstep : 0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < r.C * r.ring.pad; i += gridDim.x * blockDim.x) {
    const int c = i / r.ring.pad, t = i - c * r.ring.pad;
    float* ring = ring_ptr(r.ring, base, c, t);
    float* buf = scratch + r.at + (size_t)c * r.rs + at + t;
    if (out) *ring = *buf; else *buf = *ring;
  }
}
__global__ void cv_set_int_kernel(int* p, int v0, int v1) { p[0] = v0; p[1] = v1; }

// =================================== host side ===================================
struct Step {
  int kind;  // 0 gemm, 1 attn, 2 dwln
  int ln;    // dwln: the twin of its output
  CvGemm g;
  CvAttn a;
  CvDwLn d;
};

// Where the twins of a block of frames lie in the scratch memory.
struct CvBlock {
  std::vector<Ring> twins;
  std::vector<size_t> at;  // floats from its start
  size_t floats = 0;
};

struct vui_codec {
  vui_codec_config cfg;
  int hop;
  char* ws;
  int64_t ws_bytes;
  float* state0;  // start of the zeroed-on-reset region (rings)
  size_t state_floats;
  // what stands for each ring and buffer while several frames are decoded at once, in the caller's scratch memory
  std::vector<CvBlock> blocks;  // of n frames at [n]
  CvHist* hist;                 // device: the rings and their twins, n_hist for every n
  int n_hist = 0;
  int* ctr;  // [0] frames started since reset, [1] error flag
  int* cnt;  // arrival counters of split tiles
  size_t part_floats = 0, cnt_ints = 0;
  CvVq vq;
  int vqx, qkv, att;  // twins of buffers that are not part of a product
  std::vector<Step> steps;
  CvFinal fin;
  // the persistent form of the one-column steps (0: the kernel sequence runs them)
  CvTrunk trunk;
  int trunk_steps = 0;  // leading entries of `steps` the trunk kernel replaces (the codebook kernel as well)
  int trunk_wgs = 0;
  int w_nt = 0;          // GEMM weights with non-temporal loads: set when the vocoder is given part of the GPU
  int trunk_narrow = 0;  // the row plan of the kernel instantiation that trunk_wgs workgroups take
  int trunk_cap = 0;     // workgroups that can be resident at once on the whole GPU (at most 256 are used)
  size_t trunk_lds = 0;
  int use_trunk = 1;
};

static int ipow2(int n) { int r = 1; while (r < n) r <<= 1; return r; }

// Whether nwg workgroups can take the one-column steps with the row plan TrPlan<narrow>: every phase's rows per wave
// within the plan, every vector within the kernel's LDS areas.
template <bool NARROW> static bool trunk_fits_t(const vui_codec_config& k, int nwg) {
  typedef TrPlan<NARROW> P;
  const int A = k.n_heads * k.head_dim;
  auto fits = [&](int M, int K, int maxr, int maxc, int n) { return n > 0 && ((M + n - 1) / n + 3) / 4 <= maxr && K <= 256 * maxc && K % 4 == 0; };
  const int nq = nwg >= 4 * k.n_heads ? nwg - k.n_heads : nwg;  // the head-owning workgroups stay out of the q/k/v rows
  return nwg >= k.n_heads && fits(k.vq_dim, 2 * k.codebook_dim, P::VQ, 2, nwg) && fits(k.latent_dim, 3 * k.vq_dim, P::PRE, TR_MAXC, nwg) &&
         fits(k.d_model, k.latent_dim, P::IN, 4, nwg) && fits(3 * A, k.d_model, P::QKV, 2, nq) && fits(k.d_model, A, P::O, 4, nwg) &&
         2 * ((k.mlp_dim + nwg - 1) / nwg) <= 4 * P::GU && fits(k.d_model, k.mlp_dim, P::DN, 4, nwg) &&
         fits(k.latent_dim, k.d_model, P::OUT, 2, nwg) && (k.n_up == 0 || fits(k.latent_dim * k.up_ratios[0], k.latent_dim, P::UP, 4, nwg)) &&
         k.head_dim <= 64 && k.max_seq <= 256 && k.d_model <= 1536 && A <= 1536 && k.mlp_dim <= 1536 && k.latent_dim <= 1536 &&
         3 * k.vq_dim <= 1536;
}
static bool trunk_fits(const vui_codec_config& k, int nwg, bool narrow) {
  return narrow ? trunk_fits_t<true>(k, nwg) : trunk_fits_t<false>(k, nwg);
}

static int cv_check(const vui_codec_config* c) {
  if (!c) { vui_set_error("NULL codec config"); return VUI_EINVAL; }
  if (c->n_up < 0 || c->n_up > 4 || c->n_rates < 1 || c->n_rates > 8) { vui_set_error("codec: n_up=%d / n_rates=%d outside the supported range", c->n_up, c->n_rates); return VUI_EINVAL; }
  if (c->n_codebooks < 1 || c->n_semantic < 1 || c->n_semantic > c->n_codebooks || c->codebook_size < 1) { vui_set_error("codec: bad codebook layout"); return VUI_EINVAL; }
  const int A = c->n_heads * c->head_dim;
  int dims32[] = {2 * c->codebook_dim, c->vq_dim, c->latent_dim, c->d_model, A, c->mlp_dim, 4 * c->latent_dim, c->decoder_dim};
  for (int v : dims32)
    if (v < 32 || (v % 32)) { vui_set_error("codec: every layer width must be a multiple of 32 (got %d)", v); return VUI_EINVAL; }
  if (c->head_dim > 64 || (c->head_dim & 15) || c->n_heads < 1) { vui_set_error("codec: head_dim=%d unsupported (a multiple of 16, <= 64)", c->head_dim); return VUI_EINVAL; }
  if ((c->decoder_dim >> c->n_rates) * (FIN_TW + 6 + 7) * 4 > 60000) { vui_set_error("codec: last stage too wide"); return VUI_EINVAL; }
  if (c->max_seq < 1 || c->max_seq > 4096) { vui_set_error("codec: max_seq=%d outside [1,4096]", c->max_seq); return VUI_EINVAL; }
  if (c->latent_dim > 256 * DW_MAXC) { vui_set_error("codec: latent_dim=%d above %d", c->latent_dim, 256 * DW_MAXC); return VUI_EINVAL; }
  int dim = c->decoder_dim;
  for (int i = 0; i < c->n_rates; ++i) {
    if (c->rates[i] < 1 || (dim % 64)) { vui_set_error("codec: decoder stage %d: width %d must be a multiple of 64, rate >= 1", i, dim); return VUI_EINVAL; }
    dim /= 2;
  }
  for (int i = 0; i < c->n_up; ++i)
    if (c->up_ratios[i] < 1) { vui_set_error("codec: bad upsample ratio"); return VUI_EINVAL; }
  return VUI_OK;
}

int32_t vui_codec_hop(const vui_codec_config* c) {
  if (cv_check(c)) return VUI_EINVAL;
  int h = 1;
  for (int i = 0; i < c->n_up; ++i) h *= c->up_ratios[i];
  for (int i = 0; i < c->n_rates; ++i) h *= c->rates[i];
  return h;
}

int32_t vui_codec_n_tensors(const vui_codec_config* c) {
  if (cv_check(c)) return VUI_EINVAL;
  return 2 * 2 + c->n_codebooks + 2 + 2 + 11 * c->n_layers + 3 + 11 * c->n_up + 2 + c->n_rates * (4 + 3 * 8) + 2 + 2;
}

// Bump allocator over the workspace; with base == nullptr it only measures.
struct Arena {
  char* base;
  size_t off = 0;
  float* take(size_t floats) {
    float* p = base ? (float*)(base + off) : nullptr;
    off += (floats * 4 + 255) & ~(size_t)255;
    return p;
  }
};

// Frames that one pass takes at most: CV_BLOCK by vui_codec_decode_block, CV_CLIP by vui_codec_decode_clip, which is as large as
// products still gain: the weights pass once, the trunk's hundred launches of 5-9 us for a few columns come once, and 32 frames of the
// last stages are a grid and a half.  us of a clip in passes of 32 / 64 / 96 / 128 / 250 frames: 250 frames 15775 / 13583 / 12500 / 11196 /
// 10380, 128 7856 / 6804 / 6536 / 5618, 93 5844 / 5329 / 4505.  The buffers, scratch memory of the caller's, take 8 MB per frame.
#define CV_BLOCK 32
#define CV_CLIP 256
static int block_frames(const vui_codec_config& k) { return k.max_seq < CV_BLOCK ? k.max_seq : CV_BLOCK; }
// A clip's buffers stay under 1 GiB each (offsets are 32 bits) and its tiles of 16 columns within a grid's second dimension.
static int clip_frames(const vui_codec_config& k) {
  long wide = std::max({2 * k.codebook_dim, k.vq_dim, k.latent_dim, k.d_model, 3 * k.n_heads * k.head_dim, k.mlp_dim}), T = 1;
  for (int i = 0; i < k.n_up; ++i) { T *= k.up_ratios[i]; wide = std::max(wide, 4 * T * k.latent_dim); }
  for (int i = 0, dim = k.decoder_dim; ; ++i, dim /= 2) {
    wide = std::max(wide, T * dim);
    if (i == k.n_rates) break;
    T *= k.rates[i];
    wide = std::max(wide, T * (dim / 2));
  }
  const long n = std::min({(long)CV_CLIP, (long)k.max_seq, (1l << 28) / (wide + 1), (1l << 19) / T});
  return (int)std::max(n, (long)block_frames(k));
}

// Rings and buffers of one frame, and of each its twin: a plain buffer of a whole block of frames with the history
// columns in front.  A ring of 32 frames for both would need no copies of histories (two launches per block), but its
// lines are never in the caches again when a single frame comes to them: 1 % of the streamed vocoder.
struct RingMaker {
  Arena& ar;
  struct Made { Ring ring; int C, T, share; };  // share: twins of one group >= 0 take turns in the same memory
  std::vector<Made> made;
  Ring make(int C, int pad, int T, bool stream, int group = -1) {
    Ring r;
    r.rs = ipow2(pad + T);
    r.mask = r.rs - 1;
    r.pad = pad;
    r.tstep = stream ? T : 0;
    r.id = (int)made.size();
    r.p = ar.take((size_t)C * r.rs);
    made.push_back(Made{r, C, T, group});
    return r;
  }
  static bool keeps(const Made& m) { return m.ring.tstep && m.ring.pad; }
  int histories() const {
    int n = 0;
    for (const Made& m : made) n += keeps(m);
    return n;
  }
  CvBlock block(int frames) const {  // once every ring is known
    CvBlock b;
    size_t common[2] = {0, 0};  // floats, then places of the shared groups
    auto rs = [&](const Made& m) { return (m.ring.pad + m.T * frames + 3) & ~3; };
    auto need = [&](const Made& m) { return (size_t)m.C * rs(m) + 256; };  // a tile reads up to 256 columns behind the last channel's
    auto take = [&](size_t n) { const size_t o = b.floats; b.floats += (n + 63) & ~(size_t)63; return o; };
    for (const Made& m : made)
      if (m.share >= 0 && need(m) > common[m.share]) common[m.share] = need(m);
    for (size_t& c : common) c = take(c);
    for (const Made& m : made) {
      Ring t = m.ring;
      t.p = nullptr;
      t.rs = rs(m);
      t.mask = 0x7fffffff;
      t.tstep = 0;
      b.twins.push_back(t);
      b.at.push_back(m.share >= 0 ? common[m.share] : take(need(m)));
    }
    return b;
  }
  void histories(const CvBlock& b, std::vector<CvHist>& out) const {
    for (const Made& m : made)
      if (keeps(m)) out.push_back(CvHist{m.ring, b.at[m.ring.id], b.twins[m.ring.id].rs, m.C});
  }
};
static Ring no_ring() { Ring r; r.p = nullptr; r.rs = 1; r.mask = 0; r.pad = 0; r.tstep = 0; r.id = -1; return r; }

static void grid_for(size_t n, dim3& g) { size_t b = (n + 255) / 256; g = dim3((unsigned)(b > 4096 ? 4096 : (b ? b : 1))); }

// ---- launch shapes ----
struct CvScratch { size_t part, cnt; };  // floats of partial sums, arrival counters
// tiles of cv_wide_kernel, and what one unit of a tile costs against 128 x 128
struct WideTile { int bm, bn; float unit; };
#define CVW_PAIR 2.6   // us of a unit of 128 x 128 for two workgroups of a CU, and for one
#define CVW_ALONE 1.6
#define CVW_PARTS (6u << 20)  // floats of the parts of a split product, which the workspace holds
static const WideTile kWide[] = {{128, 128, 1.0f}, {96, 128, 0.79f}, {64, 128, 0.63f}, {128, 64, 0.63f}, {32, 128, 0.55f}};

static int cv_lds(const CvGemm& g) { return (CV_NW * g.tt * 256 + g.xcols * (g.chunk * 32 + 4)) * 4; }
// The fields of cv_cols_kernel for a tile shared by up to `splits` workgroups: chunks whose units fit the waves' registers and whose
// columns fit LDS (one group always does: a tile of 64 columns and its halo of 6 x 9 take 118 x 36 floats).
static void cv_shape(CvGemm& g, int splits) {
  const int G = g.Cin / 32, units = (g.tt <= 2 ? CvUnits<2>::N : CvUnits<4>::N) * CV_NW;
  g.per = (G + splits - 1) / splits;
  g.splits = (G + g.per - 1) / g.per;
  g.xcols = (g.T < 16 * g.tt ? g.T : 16 * g.tt) + (g.taps - 1) * g.dil;
  g.inv_xcols = cv_inv(g.xcols);
  g.inv_tc = cv_inv(g.tc_stride);
  const int fit = std::max(1, std::min(units / g.taps, (CV_XROOM / g.xcols - 4) / 32)), rounds = (std::min(g.per, G) + fit - 1) / fit;
  g.chunk = (g.per + rounds - 1) / rounds;
}

// Chooses tile width, splits and kernel for g.T columns.
// A clip's products split no further than the scratch memory sized for blocks reaches.
static CvScratch cv_plan(CvGemm& g, size_t part_cap = CVW_PARTS, size_t cnt_cap = SIZE_MAX) {
  const int U = g.taps * (g.Cin / 32), M = g.M, T = g.T;
  auto tiles = [&](int tt) { return (M / 16) * ((T + 16 * tt - 1) / (16 * tt)); };
  // few units and few tiles: a launch of cv_cols_kernel is shorter than the large tiles' two (768 channels x 128 columns, 1x1: 14 / 8 us)
  const bool few = U <= 32 && tiles(1) <= 512;
  if (g.nf > 1 && T >= CV_WIDE_T && !few && M % 32 == 0 && g.in_mode == IN_PLAIN && g.epi != EPI_SILU_PAIR &&
      (g.taps - 1) * g.dil <= CVW_HALO) {
    // Tile and splits: what the workgroups of a CU take, in pairs, and for split tiles the second launch and its traffic.
    size_t part = 0;
    double cost = 0;
    for (int i = 0; i < 5; ++i) {
      const WideTile& w = kWide[i];
      if (M % w.bm) continue;
      const int cols = (T + w.bn - 1) / w.bn * w.bn, tiles = (M / w.bm) * (cols / w.bn);
      for (int sp = 1; sp <= 16 && (sp == 1 || (U / sp >= 4 && (size_t)sp * M * cols <= std::min(part_cap, (size_t)CVW_PARTS))); ++sp) {
        const int wgs = (tiles * sp + 255) / 256;
        const double c = (wgs / 2 * CVW_PAIR + wgs % 2 * CVW_ALONE) * ((U + sp - 1) / sp) * w.unit + (sp > 1 ? 6 + 1e-6 * sp * M * T : 0);
        if (cost && c >= cost) continue;
        cost = c;
        g.tt = 0; g.wide = i; g.splits = sp;
        part = sp > 1 ? (size_t)sp * M * cols : 0;
      }
    }
    return CvScratch{part, 0};
  }
  // The narrowest tiles that are no more than the CUs; products of many units start at 32 columns, where a weight meets two blocks of
  // columns.  Then workgroups share a tile's channels until the CUs are busy (twice that for one block of columns: the layer
  // streams weights), each with 32 units or so.
  const int G = g.Cin / 32, most = g.in_mode == IN_PLAIN ? (U + 16) / 32 : 1;  // a split norm would need the other workgroups' sums
  g.tt = T > 16 && U > 32 ? 2 : 1;
  while (g.tt < 4 && T > 16 * g.tt && tiles(g.tt) > 256) g.tt *= 2;
  const int target = T <= 16 ? 512 : 256;
  const int sp = std::max(1, std::min(std::min((2 * target + tiles(g.tt)) / (2 * tiles(g.tt)), most), std::min(8, G)));
  cv_shape(g, sp);
  if (g.splits > 1 && ((size_t)tiles(g.tt) * g.splits * g.tt * 256 > part_cap || (size_t)tiles(g.tt) > cnt_cap)) cv_shape(g, 1);
  return CvScratch{(size_t)tiles(g.tt) * g.splits * g.tt * 256, (size_t)tiles(g.tt)};
}

// Lays out the workspace and (when tensors != nullptr) packs weights and records the launch plan.
static int cv_build(vui_codec* cc, const vui_codec_config* c, const void* const* tensors, char* ws, hipStream_t st, int64_t* need,
                    size_t part_cap, size_t cnt_cap, size_t* part_need, size_t* cnt_need, int frames = 0, int64_t* block_need = nullptr) {
  Arena ar{ws};
  const bool real = ws != nullptr && tensors != nullptr;
  int ti = 0;
  auto next = [&]() -> const float* { return real ? (const float*)tensors[ti++] : (ti++, nullptr); };
  auto pack_copy = [&](const float* src, float* dst, int M, int K, int ld, int off) {
    if (!real) return;
    dim3 g; grid_for((size_t)M * K, g);
    hipLaunchKernelGGL(cv_copy_rows_kernel, g, dim3(256), 0, st, src, dst, M, K, ld, off);
  };
  auto pack_conv = [&](const float* src, int Cout, int Cin, int K) -> float* {
    float* dst = ar.take((size_t)Cout * Cin * K);
    if (real) { dim3 g; grid_for((size_t)Cout * Cin * K, g); hipLaunchKernelGGL(cv_pack_conv_kernel, g, dim3(256), 0, st, src, dst, Cout, Cin, K); }
    return dst;
  };
  auto pack_tconv = [&](const float* src, int Cin, int Cout, int s, int taps) -> float* {
    float* dst = ar.take((size_t)taps * Cout * s * Cin);
    if (real) { dim3 g; grid_for((size_t)taps * Cout * s * Cin, g); hipLaunchKernelGGL(cv_pack_tconv_kernel, g, dim3(256), 0, st, src, dst, Cin, Cout, s, taps); }
    return dst;
  };
  auto fold_norm = [&](float* W, const float* w, int M, int K) {
    if (!real) return;
    dim3 g; grid_for((size_t)M * K, g);
    hipLaunchKernelGGL(cv_scale_cols_kernel, g, dim3(256), 0, st, W, w, M, K);
  };
  auto vec = [&](const float* src, int n) -> float* { float* dst = ar.take(n); pack_copy(src, dst, 1, n, n, 0); return dst; };
  struct Snake { float* ea; float* ib; };
  auto snake = [&](int n) -> Snake {
    const float* al = next(); const float* be = next();
    Snake s{ar.take(n), ar.take(n)};
    if (real) hipLaunchKernelGGL(cv_snake_tab_kernel, dim3((n + 255) / 256), dim3(256), 0, st, al, be, s.ea, s.ib, n);
    return s;
  };
  int* ctr = (int*)ar.take(64);
  // meeting place of split tiles: sized by a first pass (the sizes do not depend on the pointers)
  size_t part_floats = 0, cnt_ints = 0;
  float* part = ar.take(part_cap);
  int* cnt = (int*)ar.take(cnt_cap);
  auto gemm = [&](const float* W, const float* bias, int M, int Cin, int taps, int dil, int T, const Ring& in) -> CvGemm {
    CvGemm g;
    memset(&g, 0, sizeof(g));
    g.W = W; g.bias = bias; g.M = M; g.Cin = Cin; g.taps = taps; g.dil = dil; g.T = T; g.bias_div = 1;
    g.in = in; g.in_mode = IN_PLAIN; g.eps = 1e-6f; g.epi = EPI_NONE;
    g.res = no_ring(); g.out_raw = no_ring(); g.out_act = no_ring(); g.ctr = ctr; g.nf = 1;
    g.part = part; g.cnt = cnt;
    for (int n = real || part_need ? block_frames(*c) : 1; n >= 1; --n) {  // the frame's own plan is made last and stays
      g.T = n * T;
      g.nf = n;
      const CvScratch need = cv_plan(g);
      if (need.part > part_floats) part_floats = need.part;
      if (need.cnt > cnt_ints) cnt_ints = need.cnt;
    }
    return g;
  };
  auto push_gemm = [&](CvGemm& g) {
    if (!real) return;
    cv_plan(g);  // with the norm known
    Step s; memset((void*)&s, 0, sizeof(s)); s.kind = 0; s.g = g; cc->steps.push_back(s);
  };

  const int cd = c->codebook_dim, CS = c->codebook_size, L = c->latent_dim, D = c->d_model, A = c->n_heads * c->head_dim;
  // ---- quantizer: [semantic | acoustic] rows times [W_sem | W_ac] ----
  float* embed = ar.take((size_t)c->n_codebooks * CS * cd);
  float* Wvq = ar.take((size_t)c->vq_dim * 2 * cd);
  {
    int cb = 0;
    for (int grp = 0; grp < 2; ++grp) {
      const int n = grp == 0 ? c->n_semantic : c->n_codebooks - c->n_semantic;
      next();  // input_proj: encoder side only
      const float* op = next();
      pack_copy(op, Wvq, c->vq_dim, cd, 2 * cd, grp * cd);
      for (int i = 0; i < n; ++i, ++cb) pack_copy(next(), embed + (size_t)cb * CS * cd, CS, cd, cd, 0);
    }
  }
  // ---- state region (zeroed by reset) starts here: all rings ----
  RingMaker rings{ar};
  const size_t state_begin = ar.off;
  Ring pre_in = rings.make(c->vq_dim, 2, 1, true);
  std::vector<Ring> dw_in, tc_in, ru_in;
  int T = 1;
  for (int i = 0; i < c->n_up; ++i) { T *= c->up_ratios[i]; dw_in.push_back(rings.make(L, 6, T, true)); }
  const int T_lat = T;
  Ring dec0_in = rings.make(L, 6, T_lat, true);
  {
    int dim = c->decoder_dim, t = T_lat;
    for (int i = 0; i < c->n_rates; ++i) {
      tc_in.push_back(rings.make(dim, 1, t, true));
      t *= c->rates[i];
      dim /= 2;
      for (int j = 0; j < 3; ++j) { const int dil = j == 0 ? 1 : (j == 1 ? 3 : 9); ru_in.push_back(rings.make(dim, 6 * dil, t, true)); }
    }
  }
  int fin_dim = c->decoder_dim >> c->n_rates;
  const int hop = vui_codec_hop(c);
  Ring fin_in = rings.make(fin_dim, 6, hop, true);
  const size_t state_end = ar.off;
  // ---- plain activation buffers ----
  Ring vqx = rings.make(2 * cd, 0, 1, false);
  Ring pre_out = rings.make(L, 0, 1, false);
  Ring xres = rings.make(D, 0, 1, false);
  Ring qkv = rings.make(3 * A, 0, 1, false);
  Ring att = rings.make(A, 0, 1, false);
  Ring gu = rings.make(c->mlp_dim, 0, 1, false);
  float* kc = ar.take((size_t)c->n_layers * A * c->max_seq);
  float* vc = ar.take((size_t)c->n_layers * A * c->max_seq);
  float* inv_freq = ar.take(c->head_dim / 2);
  // persistent trunk: exchange words (never reused inside a launch), layer table, epoch / arrival / error words
  const size_t ll_words = (size_t)c->vq_dim + L + D + (size_t)c->n_layers * (3 * A + A + D + c->mlp_dim + D) + L;
  uint64_t* ll = (uint64_t*)ar.take(ll_words * 2);
  TrunkLayer* tl_dev = (TrunkLayer*)ar.take((sizeof(TrunkLayer) * c->n_layers + 3) / 4);
  uint32_t* tctl = (uint32_t*)ar.take(64);
  if (real) {
    std::vector<float> h(c->head_dim / 2);
    // 1 / theta^(2i/dim) in fp32, as torch evaluates it (qwen_codec.py:164)
    for (int i = 0; i < c->head_dim / 2; ++i) h[i] = 1.0f / powf(c->rope_theta, (float)(2 * i) / (float)c->head_dim);
    HIP_TRY(hipMemcpyAsync(inv_freq, h.data(), h.size() * 4, hipMemcpyHostToDevice, st));
    HIP_TRY(hipStreamSynchronize(st));  // h goes out of scope
  }

  // ---- pre_conv, pre_transformer ----
  CvTrunk tk;
  memset((void*)&tk, 0, sizeof(tk));
  std::vector<TrunkLayer> tl(c->n_layers);
  {
    CvGemm g = gemm(Wvq, nullptr, c->vq_dim, 2 * cd, 1, 1, 1, vqx);
    g.out_raw = pre_in;
    push_gemm(g);
    const float* w = next(); const float* b = next();
    g = gemm(pack_conv(w, L, c->vq_dim, 3), vec(b, L), L, c->vq_dim, 3, 1, 1, pre_in);
    g.out_raw = pre_out;
    push_gemm(g);
    tk.Wvq = Wvq; tk.vq_dim = c->vq_dim; tk.Wpre = g.W; tk.bpre = g.bias; tk.L = L; tk.pre_in = pre_in;
    w = next(); b = next();
    float* Wi = ar.take((size_t)D * L);
    pack_copy(w, Wi, D, L, L, 0);
    g = gemm(Wi, vec(b, D), D, L, 1, 1, 1, pre_out);
    g.out_raw = xres;
    push_gemm(g);
    tk.Win = g.W; tk.bin = g.bias; tk.D = D;
  }
  for (int l = 0; l < c->n_layers; ++l) {
    const float* ln1 = next();
    float* Wqkv = ar.take((size_t)3 * A * D);
    for (int i = 0; i < 3; ++i) pack_copy(next(), Wqkv + (size_t)i * A * D, A, D, D, 0);
    fold_norm(Wqkv, ln1, 3 * A, D);
    float* Wo = ar.take((size_t)D * A);
    pack_copy(next(), Wo, D, A, A, 0);
    const float* asc = next();
    const float* ln2 = next();
    float* Wgu = ar.take((size_t)2 * c->mlp_dim * D);  // rows interleaved: gate_0, up_0, gate_1, up_1, ...
    for (int i = 0; i < 2; ++i) pack_copy(next(), Wgu, c->mlp_dim, D, 2 * D, i * D);
    fold_norm(Wgu, ln2, 2 * c->mlp_dim, D);
    float* Wd = ar.take((size_t)D * c->mlp_dim);
    pack_copy(next(), Wd, D, c->mlp_dim, c->mlp_dim, 0);
    const float* msc = next();
    CvGemm g = gemm(Wqkv, nullptr, 3 * A, D, 1, 1, 1, xres);
    g.in_mode = IN_RMS; g.out_raw = qkv;
    push_gemm(g);
    if (real) {
      Step s; memset((void*)&s, 0, sizeof(s)); s.kind = 1;
      s.a.qkv = qkv.p; s.a.kc = kc + (size_t)l * A * c->max_seq; s.a.vc = vc + (size_t)l * A * c->max_seq;
      s.a.out = att.p; s.a.inv_freq = inv_freq; s.a.H = c->n_heads; s.a.hd = c->head_dim; s.a.max_seq = c->max_seq; s.a.ctr = ctr;
      s.a.rs = qkv.rs; s.a.rs_out = att.rs; s.a.nf = 1;
      cc->steps.push_back(s);
    }
    g = gemm(Wo, nullptr, D, A, 1, 1, 1, att);
    g.epi = EPI_SCALE_RES; g.scale = vec(asc, D); g.res = xres; g.out_raw = xres;
    push_gemm(g);
    tl[l].Wqkv = Wqkv; tl[l].Wo = Wo; tl[l].asc = g.scale; tl[l].Wgu = Wgu; tl[l].Wd = Wd;
    tl[l].kc = kc + (size_t)l * A * c->max_seq; tl[l].vc = vc + (size_t)l * A * c->max_seq;
    g = gemm(Wgu, nullptr, 2 * c->mlp_dim, D, 1, 1, 1, xres);
    g.in_mode = IN_RMS; g.epi = EPI_SILU_PAIR; g.out_raw = gu;
    push_gemm(g);
    g = gemm(Wd, nullptr, D, c->mlp_dim, 1, 1, 1, gu);
    g.epi = EPI_SCALE_RES; g.scale = vec(msc, D); g.res = xres; g.out_raw = xres;
    push_gemm(g);
    tl[l].msc = g.scale;
  }
  Ring cur = rings.make(L, 0, 1, false);  // output of the transformer = input of the first upsample stage
  {
    const float* nw = next(); const float* w = next(); const float* b = next();
    float* Wout = ar.take((size_t)L * D);
    pack_copy(w, Wout, L, D, D, 0);
    fold_norm(Wout, nw, L, D);
    CvGemm g = gemm(Wout, vec(b, L), L, D, 1, 1, 1, xres);
    g.in_mode = IN_RMS;
    g.out_raw = c->n_up ? cur : dec0_in;
    push_gemm(g);
    tk.Wout = g.W; tk.bout = g.bias; tk.out = dec0_in;
  }
  int trunk_steps = real ? (int)cc->steps.size() : 0;
  // ---- upsample stages: transposed conv (kernel = stride) + ConvNeXt block ----
  T = 1;
  for (int i = 0; i < c->n_up; ++i) {
    const int r = c->up_ratios[i], Tin = T;
    T *= r;
    const float* w = next(); const float* b = next();
    CvGemm g = gemm(pack_tconv(w, L, L, r, 1), vec(b, L), L * r, L, 1, 1, Tin, cur);
    g.bias_div = r; g.tc_stride = r; g.out_raw = dw_in[i];
    push_gemm(g);
    if (i == 0) { tk.Wt0 = g.W; tk.bt0 = g.bias; tk.r0 = r; tk.out = dw_in[0]; if (real) trunk_steps = (int)cc->steps.size(); }
    const float* dww = next(); const float* dwb = next(); const float* lnw = next(); const float* lnb = next();
    Ring ln = rings.make(L, 0, T, false);
    float* dwwp = vec(dww, L * 7); float* dwbp = vec(dwb, L); float* lnwp = vec(lnw, L); float* lnbp = vec(lnb, L);
    if (real) {
      Step s; memset((void*)&s, 0, sizeof(s)); s.kind = 2;
      s.d.in = dw_in[i]; s.d.w = dwwp; s.d.b = dwbp; s.d.lnw = lnwp; s.d.lnb = lnbp;
      s.ln = ln.id; s.d.out = ln.p; s.d.rs_out = ln.rs; s.d.C = L; s.d.eps = 1e-6f; s.d.ctr = ctr; s.d.nf = 1;
      s.g.T = T;  // grid
      cc->steps.push_back(s);
    }
    const float* w1 = next(); const float* b1 = next(); const float* w2 = next(); const float* b2 = next(); const float* gam = next();
    Ring pw = rings.make(4 * L, 0, T, false);
    float* W1 = ar.take((size_t)4 * L * L);
    pack_copy(w1, W1, 4 * L, L, L, 0);
    g = gemm(W1, vec(b1, 4 * L), 4 * L, L, 1, 1, T, ln);
    g.epi = EPI_GELU; g.out_raw = pw;
    push_gemm(g);
    float* W2 = ar.take((size_t)L * 4 * L);
    pack_copy(w2, W2, L, 4 * L, 4 * L, 0);
    g = gemm(W2, vec(b2, L), L, 4 * L, 1, 1, T, pw);
    g.epi = EPI_SCALE_RES; g.scale = vec(gam, L); g.res = dw_in[i];
    if (i + 1 < c->n_up) { cur = rings.make(L, 0, T, false); g.out_raw = cur; } else g.out_raw = dec0_in;
    push_gemm(g);
  }
  // ---- BigVGAN-style decoder ----
  {
    int dim = c->decoder_dim;
    const float* w = next(); const float* b = next();
    CvGemm g0 = gemm(pack_conv(w, dim, L, 7), vec(b, dim), dim, L, 7, 1, T_lat, dec0_in);
    int t = T_lat;
    CvGemm pending = g0;  // its out_act is the first block's snake, known once the block's tensors are read
    for (int i = 0; i < c->n_rates; ++i) {
      const int rate = c->rates[i], out = dim / 2, tin = t;
      t *= rate;
      Snake s0 = snake(dim);
      pending.out_act = tc_in[i]; pending.ea = s0.ea; pending.ib = s0.ib;
      push_gemm(pending);
      const float* tw = next(); const float* tb = next();
      CvGemm tg = gemm(pack_tconv(tw, dim, out, rate, 2), vec(tb, out), out * rate, dim, 2, 1, tin, tc_in[i]);
      tg.bias_div = rate; tg.tc_stride = rate;
      Ring R = rings.make(out, 0, t, false, 0);  // a stage's own: the next stage's take their place
      Ring hbuf = rings.make(out, 0, t, false, 1);
      tg.out_raw = R;
      pending = tg;
      for (int j = 0; j < 3; ++j) {
        const int dil = j == 0 ? 1 : (j == 1 ? 3 : 9);
        const Ring& rin = ru_in[i * 3 + j];
        Snake a1 = snake(out);
        pending.out_act = rin; pending.ea = a1.ea; pending.ib = a1.ib;
        push_gemm(pending);
        const float* w1 = next(); const float* b1 = next();
        Snake a2 = snake(out);
        const float* w2 = next(); const float* b2 = next();
        CvGemm c1 = gemm(pack_conv(w1, out, out, 7), vec(b1, out), out, out, 7, dil, t, rin);
        c1.out_act = hbuf; c1.ea = a2.ea; c1.ib = a2.ib;
        push_gemm(c1);
        float* W2 = ar.take((size_t)out * out);
        pack_copy(w2, W2, out, out, out, 0);
        CvGemm c2 = gemm(W2, vec(b2, out), out, out, 1, 1, t, hbuf);
        c2.epi = EPI_RES; c2.res = R;
        if (j < 2) c2.out_raw = R;
        pending = c2;
      }
      dim = out;
    }
    Snake sf = snake(dim);
    pending.out_act = fin_in; pending.ea = sf.ea; pending.ib = sf.ib;
    push_gemm(pending);
    const float* fw = next(); const float* fb = next();
    float* fwp = vec(fw, dim * 7); float* fbp = vec(fb, 1);
    if (real) {
      cc->fin.in = fin_in; cc->fin.w = fwp; cc->fin.b = fbp; cc->fin.audio = nullptr; cc->fin.C = dim; cc->fin.k = 7; cc->fin.T = hop; cc->fin.ctr = ctr; cc->fin.nf = 1;
    }
  }
  if (block_need) *block_need = (int64_t)rings.block(frames).floats * 4;
  const int n_hist = rings.histories(), n_blocks = clip_frames(*c) + 1;
  CvHist* hist_dev = (CvHist*)ar.take((sizeof(CvHist) * n_hist * n_blocks + 3) / 4);
  if (need) *need = (int64_t)ar.off;
  if (part_need) *part_need = part_floats;
  if (cnt_need) *cnt_need = cnt_ints;
  if (real) {
    tk.codes = nullptr; tk.n_q = 0; tk.n_sem = c->n_semantic; tk.CS = CS; tk.cd = cd; tk.embed = embed;
    tk.ctr = ctr; tk.err = ctr + 1; tk.max_seq = c->max_seq;
    tk.n_layers = c->n_layers; tk.H = c->n_heads; tk.hd = c->head_dim; tk.mlp = c->mlp_dim;
    tk.layers = tl_dev; tk.inv_freq = inv_freq; tk.ll = ll; tk.epoch = tctl; tk.arrive = tctl + 1; tk.lerr = tctl + 2;
    tk.eps = 1e-6f;
    HIP_TRY(hipMemcpyAsync(tl_dev, tl.data(), sizeof(TrunkLayer) * c->n_layers, hipMemcpyHostToDevice, st));
    {
      dim3 g; grid_for(ll_words * 2, g);
      hipLaunchKernelGGL(cv_fill_kernel, g, dim3(256), 0, st, (float*)ll, ll_words * 2, 0.0f);
      hipLaunchKernelGGL(cv_fill_kernel, dim3(1), dim3(64), 0, st, (float*)tctl, (size_t)16, 0.0f);
    }
    std::vector<CvHist> hist;
    for (int n = 0; n < n_blocks; ++n) {
      cc->blocks.push_back(rings.block(n));
      rings.histories(cc->blocks[n], hist);
    }
    HIP_TRY(hipMemcpyAsync(hist_dev, hist.data(), sizeof(CvHist) * hist.size(), hipMemcpyHostToDevice, st));
    HIP_TRY(hipStreamSynchronize(st));  // tl and hist go out of scope
    cc->trunk = tk;
    cc->trunk_steps = trunk_steps;
    if (part_floats > part_cap || cnt_ints > cnt_cap) { vui_set_error("codec: internal scratch sizing"); return VUI_EINVAL; }
    cc->ctr = ctr; cc->cnt = cnt; cc->cnt_ints = cnt_cap; cc->part_floats = part_cap;
    cc->state0 = (float*)(ws + state_begin);
    cc->state_floats = (state_end - state_begin) / 4;
    cc->hist = hist_dev;
    cc->n_hist = n_hist;
    cc->vqx = vqx.id; cc->qkv = qkv.id; cc->att = att.id;
    cc->vq.codes = nullptr; cc->vq.n_q = 0; cc->vq.n_sem = c->n_semantic; cc->vq.CS = CS; cc->vq.cd = cd;
    cc->vq.embed = embed; cc->vq.x = vqx.p; cc->vq.rs = vqx.rs; cc->vq.nf = 1; cc->vq.ctr = ctr; cc->vq.err = ctr + 1; cc->vq.max_seq = c->max_seq;
    if (ti != vui_codec_n_tensors(c)) { vui_set_error("codec: internal tensor count %d != %d", ti, vui_codec_n_tensors(c)); return VUI_EINVAL; }
    HIP_TRY(hipGetLastError());
  }
  return VUI_OK;
}

int64_t vui_codec_workspace_bytes(const vui_codec_config* c) {
  if (cv_check(c)) return VUI_EINVAL;
  int64_t need = 0;
  size_t pf = 0, ci = 0;
  if (cv_build(nullptr, c, nullptr, nullptr, nullptr, nullptr, 0, 0, &pf, &ci)) return VUI_EINVAL;
  if (cv_build(nullptr, c, nullptr, nullptr, nullptr, &need, pf, ci, nullptr, nullptr)) return VUI_EINVAL;
  return need;
}

int vui_codec_reset(vui_codec* c, vui_stream_t stream) {
  if (!c) { vui_set_error("NULL codec"); return VUI_EINVAL; }
  hipStream_t st = (hipStream_t)stream;
  dim3 g; grid_for(c->state_floats, g);
  hipLaunchKernelGGL(cv_fill_kernel, g, dim3(256), 0, st, c->state0, c->state_floats, 0.0f);
  hipLaunchKernelGGL(cv_set_int_kernel, dim3(1), dim3(1), 0, st, c->ctr, 0, 0);
  HIP_TRY(hipGetLastError());
  return VUI_OK;
}

int vui_codec_init(const vui_codec_config* cfg, const void* const* tensors, int32_t n_tensors, void* workspace,
                   int64_t workspace_bytes, vui_stream_t stream, vui_codec** out) {
  if (!out) { vui_set_error("NULL out"); return VUI_EINVAL; }
  *out = nullptr;
  int rc = cv_check(cfg);
  if (rc) return rc;
  if (!tensors || !workspace) { vui_set_error("NULL argument"); return VUI_EINVAL; }
  if (n_tensors != vui_codec_n_tensors(cfg)) { vui_set_error("codec: %d tensors given, %d expected", n_tensors, vui_codec_n_tensors(cfg)); return VUI_EINVAL; }
  for (int i = 0; i < n_tensors; ++i)
    if (!tensors[i]) { vui_set_error("codec: tensor %d is NULL", i); return VUI_EINVAL; }
  const int64_t need = vui_codec_workspace_bytes(cfg);
  if (need < 0) return (int)need;
  if (workspace_bytes < need) { vui_set_error("workspace too small: %lld < %lld", (long long)workspace_bytes, (long long)need); return VUI_ENOMEM; }
  if (((uintptr_t)workspace) & 255) { vui_set_error("workspace must be 256-byte aligned"); return VUI_EINVAL; }
  vui_codec* c = new (std::nothrow) vui_codec();
  if (!c) { vui_set_error("out of host memory"); return VUI_ENOMEM; }
  c->cfg = *cfg; c->hop = vui_codec_hop(cfg); c->ws = (char*)workspace; c->ws_bytes = workspace_bytes;
  size_t pf = 0, ci = 0;
  rc = cv_build(nullptr, cfg, nullptr, nullptr, nullptr, nullptr, 0, 0, &pf, &ci);
  if (!rc) rc = cv_build(c, cfg, tensors, (char*)workspace, (hipStream_t)stream, nullptr, pf, ci, nullptr, nullptr);
  if (!rc) {
    dim3 g; grid_for(ci, g);
    hipLaunchKernelGGL(cv_fill_kernel, g, dim3(256), 0, (hipStream_t)stream, (float*)c->cnt, ci, 0.0f);
  }
  if (!rc) rc = vui_codec_reset(c, stream);
  if (rc) { delete c; return rc; }
  for (const void* k : {(const void*)cv_cols_kernel<1, false>, (const void*)cv_cols_kernel<1, true>, (const void*)cv_cols_kernel<2, false>,
                        (const void*)cv_cols_kernel<2, true>, (const void*)cv_cols_kernel<4, false>, (const void*)cv_cols_kernel<4, true>})
    HIP_TRY(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (CV_NW * 4 * 256 + CV_XROOM) * 4));
  // the persistent trunk needs all its workgroups resident at once and the per-wave row counts it was built for
  {
    const vui_codec_config& k = c->cfg;
    c->trunk_lds = (size_t)(1536 + k.d_model + 64 + k.max_seq + 192 + 256 + 16) * 4;
    int dev = 0, cus = 0, per_cu = 0;
    HIP_TRY(hipGetDevice(&dev));
    HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)cv_trunk_kernel<true>, FR_THREADS, c->trunk_lds));
    c->trunk_cap = cus * per_cu < 256 ? cus * per_cu : 256;
    c->trunk_wgs = 0;
    for (int narrow = 0; narrow < 2 && !c->trunk_wgs; ++narrow)
      if (trunk_fits(k, c->trunk_cap, narrow != 0)) { c->trunk_wgs = c->trunk_cap; c->trunk_narrow = narrow; }
    c->use_trunk = 1;
  }
  *out = c;
  return VUI_OK;
}

void vui_codec_destroy(vui_codec* c) { delete c; }

int vui_codec_workgroups(vui_codec* c, int nwg) {
  if (!c) { vui_set_error("NULL codec"); return VUI_EINVAL; }
  if (nwg < 1 || nwg > c->trunk_cap) { vui_set_error("codec: %d workgroups outside [1, %d]", nwg, c->trunk_cap); return VUI_EINVAL; }
  for (int narrow = 0; narrow < 2; ++narrow)
    if (trunk_fits(c->cfg, nwg, narrow != 0)) {
      c->trunk_wgs = nwg; c->trunk_narrow = narrow;
      c->w_nt = nwg < c->trunk_cap ? 1 : 0;
      return VUI_OK;
    }
  vui_set_error("codec: the persistent form of the one-column steps does not run on %d workgroups (too many rows per wave)", nwg);
  return VUI_EINVAL;
}

int vui_codec_persistent(vui_codec* c, int enable) {
  if (!c) { vui_set_error("NULL codec"); return 0; }
  if (enable >= 0) c->use_trunk = enable ? 1 : 0;
  return c->use_trunk && c->trunk_wgs > 0;
}

static int launch_cv_gemm(const CvGemm& g, bool w_nt, hipStream_t st) {
  if (g.M % 16 || g.Cin % 32 || g.T < 1) { vui_set_error("codec gemm: bad shape M=%d Cin=%d T=%d", g.M, g.Cin, g.T); return VUI_EINVAL; }
  if (g.tt == 0) {
    const WideTile& w = kWide[g.wide];
    const int tiles = (g.T + w.bn - 1) / w.bn;
    const dim3 grid(g.M / w.bm * tiles * g.splits);
#define CV_WIDE(...) hipLaunchKernelGGL((cv_wide_kernel<__VA_ARGS__>), grid, dim3(256), 0, st, g)
    if (g.wide == 0) CV_WIDE(2, 2, 2, 2);
    else if (g.wide == 1) CV_WIDE(3, 1, 1, 4);
    else if (g.wide == 2) CV_WIDE(1, 2, 2, 2);
    else if (g.wide == 3) CV_WIDE(2, 1, 2, 2);
    else CV_WIDE(1, 1, 1, 4);
#undef CV_WIDE
    if (g.splits > 1) hipLaunchKernelGGL(cv_finish_kernel, dim3((g.T + 63) / 64, g.M / 32), dim3(256), 0, st, g, tiles * w.bn);
    return VUI_OK;
  }
  const dim3 grid(g.M / 16, (g.T + 16 * g.tt - 1) / (16 * g.tt), g.splits), block(64 * CV_NW);
  const int lds = cv_lds(g);
#define CV_TT(TT_)                                                                              \
  do {                                                                                          \
    if (w_nt) hipLaunchKernelGGL((cv_cols_kernel<TT_, true>), grid, block, lds, st, CV_HOT_ARGS(g), g);         \
    else hipLaunchKernelGGL((cv_cols_kernel<TT_, false>), grid, block, lds, st, CV_HOT_ARGS(g), g);             \
  } while (0)
  if (g.tt == 1) CV_TT(1);
  else if (g.tt == 2) CV_TT(2);
  else CV_TT(4);
#undef CV_TT
  return VUI_OK;
}

int vui_codec_decode_frame(vui_codec* c, const int64_t* codes, int32_t n_q, float* audio_out, vui_stream_t stream) {
  if (!c) { vui_set_error("NULL codec"); return VUI_EINVAL; }
  if (!codes || !audio_out) { vui_set_error("NULL argument"); return VUI_EINVAL; }
  if (n_q < 1 || n_q > c->cfg.n_codebooks) { vui_set_error("n_q=%d outside [1,%d]", n_q, c->cfg.n_codebooks); return VUI_EINVAL; }
  hipStream_t st = (hipStream_t)stream;
  size_t first = 0;
  if (c->use_trunk && c->trunk_wgs > 0) {
    CvTrunk tk = c->trunk;
    tk.codes = codes; tk.n_q = n_q;
    if (c->trunk_narrow) hipLaunchKernelGGL(cv_trunk_kernel<true>, dim3(c->trunk_wgs), dim3(FR_THREADS), c->trunk_lds, st, tk);
    else hipLaunchKernelGGL(cv_trunk_kernel<false>, dim3(c->trunk_wgs), dim3(FR_THREADS), c->trunk_lds, st, tk);
    first = (size_t)c->trunk_steps;
  } else {
    CvVq vq = c->vq;
    vq.codes = codes; vq.n_q = n_q;
    hipLaunchKernelGGL(cv_vq_kernel, dim3(1), dim3(256), 0, st, vq);
  }
  for (size_t si = first; si < c->steps.size(); ++si) {
    const Step& s = c->steps[si];
    if (s.kind == 0) {
      int rc = launch_cv_gemm(s.g, c->w_nt != 0, st);
      if (rc) return rc;
    } else if (s.kind == 1) {
      const size_t lds = (size_t)(s.a.hd + s.a.max_seq + 4 * s.a.hd + 8) * 4;
      hipLaunchKernelGGL(cv_attn_kernel, dim3(s.a.H), dim3(256), lds, st, s.a);
    } else {
      hipLaunchKernelGGL(cv_dwln_kernel, dim3(s.g.T), dim3(256), 0, st, s.d);
    }
  }
  CvFinal fin = c->fin;
  fin.audio = audio_out;
  hipLaunchKernelGGL(cv_final_kernel, dim3((fin.T + FIN_TW - 1) / FIN_TW), dim3(256), (size_t)(fin.C * (FIN_TW + fin.k - 1) + 256 + fin.C * fin.k) * 4, st, fin);
  HIP_TRY(hipGetLastError());
  return VUI_OK;
}

int32_t vui_codec_block_frames(const vui_codec* c) {
  if (!c) { vui_set_error("NULL codec"); return VUI_EINVAL; }
  return block_frames(c->cfg);
}

int32_t vui_codec_clip_frames(const vui_codec* c) {
  if (!c) { vui_set_error("NULL codec"); return VUI_EINVAL; }
  return clip_frames(c->cfg);
}

static int frames_check(int32_t n_frames, int most) {
  if (n_frames >= 1 && n_frames <= most) return VUI_OK;
  vui_set_error("codec: %d frames outside [1, %d]", n_frames, most);
  return VUI_EINVAL;
}

static int64_t pass_scratch(const vui_codec_config* c, int32_t n_frames) {
  int64_t need = 0;
  if (n_frames > 1 && cv_build(nullptr, c, nullptr, nullptr, nullptr, nullptr, 0, 0, nullptr, nullptr, n_frames, &need)) return VUI_EINVAL;
  return need;
}

int64_t vui_codec_block_scratch_bytes(const vui_codec_config* c, int32_t n_frames) {
  if (cv_check(c) || frames_check(n_frames, block_frames(*c))) return VUI_EINVAL;
  return pass_scratch(c, n_frames);
}

int64_t vui_codec_clip_scratch_bytes(const vui_codec_config* c, int32_t n_frames) {
  if (cv_check(c) || frames_check(n_frames, clip_frames(*c))) return VUI_EINVAL;
  return pass_scratch(c, n_frames);
}

static int decode_pass(vui_codec* c, const int64_t* codes, int32_t n_frames, int32_t n_q, float* audio_out, void* scratch, int64_t scratch_bytes,
                       int most, vui_stream_t stream) {
  if (!codes || !audio_out) { vui_set_error("NULL argument"); return VUI_EINVAL; }
  if (n_q < 1 || n_q > c->cfg.n_codebooks) { vui_set_error("n_q=%d outside [1,%d]", n_q, c->cfg.n_codebooks); return VUI_EINVAL; }
  if (frames_check(n_frames, most)) return VUI_EINVAL;
  if (n_frames == 1) return vui_codec_decode_frame(c, codes, n_q, audio_out, stream);
  if (!scratch || ((uintptr_t)scratch) & 255) { vui_set_error("codec: the scratch memory must be given and 256-byte aligned"); return VUI_EINVAL; }
  const CvBlock& block = c->blocks[n_frames];
  const CvHist* hist = c->hist + (size_t)n_frames * c->n_hist;
  const int64_t need = (int64_t)block.floats * 4;
  if (scratch_bytes < need) { vui_set_error("codec: scratch too small: %lld < %lld", (long long)scratch_bytes, (long long)need); return VUI_ENOMEM; }
  hipStream_t st = (hipStream_t)stream;
  auto buf = [&](int id) { Ring t = block.twins[id]; t.p = (float*)scratch + block.at[id]; return t; };
  auto twin = [&](const Ring& r) { return r.id < 0 ? r : buf(r.id); };
  CvVq vq = c->vq;
  vq.codes = codes; vq.n_q = n_q; vq.nf = n_frames; vq.x = buf(c->vqx).p; vq.rs = buf(c->vqx).rs;
  hipLaunchKernelGGL(cv_vq_kernel, dim3(n_frames), dim3(256), 0, st, vq);
  hipLaunchKernelGGL(cv_history_kernel, dim3(16, c->n_hist), dim3(256), 0, st, hist, (float*)scratch, c->ctr, n_frames, 0);
  for (const Step& s0 : c->steps) {
    Step s = s0;
    if (s.kind == 0) {
      s.g.T *= n_frames; s.g.nf = n_frames;
      s.g.in = twin(s.g.in); s.g.res = twin(s.g.res); s.g.out_raw = twin(s.g.out_raw); s.g.out_act = twin(s.g.out_act);
      cv_plan(s.g, c->part_floats, c->cnt_ints);
      int rc = launch_cv_gemm(s.g, c->w_nt != 0, st);
      if (rc) return rc;
    } else if (s.kind == 1) {
      s.a.nf = n_frames;
      s.a.qkv = buf(c->qkv).p; s.a.rs = buf(c->qkv).rs; s.a.out = buf(c->att).p; s.a.rs_out = buf(c->att).rs;
      const size_t lds = (size_t)(s.a.hd + s.a.max_seq + 4 * s.a.hd + 8) * 4;
      hipLaunchKernelGGL(cv_append_kernel, dim3(s.a.H, n_frames), dim3(64), 0, st, s.a);
      hipLaunchKernelGGL(cv_attn_kernel, dim3(s.a.H, n_frames), dim3(256), lds, st, s.a);
    } else {
      const Ring ln = buf(s.ln);
      s.d.nf = n_frames; s.d.in = twin(s.d.in); s.d.out = ln.p; s.d.rs_out = ln.rs;
      hipLaunchKernelGGL(cv_dwln_kernel, dim3(s.g.T * n_frames), dim3(256), 0, st, s.d);
    }
  }
  hipLaunchKernelGGL(cv_history_kernel, dim3(16, c->n_hist), dim3(256), 0, st, hist, (float*)scratch, c->ctr, n_frames, 1);
  CvFinal fin = c->fin;
  fin.audio = audio_out; fin.nf = n_frames; fin.T *= n_frames; fin.in = twin(fin.in);
  hipLaunchKernelGGL(cv_final_kernel, dim3((fin.T + FIN_TW - 1) / FIN_TW), dim3(256), (size_t)(fin.C * (FIN_TW + fin.k - 1) + 256 + fin.C * fin.k) * 4, st, fin);
  HIP_TRY(hipGetLastError());
  return VUI_OK;
}

int vui_codec_decode_block(vui_codec* c, const int64_t* codes, int32_t n_frames, int32_t n_q, float* audio_out, void* scratch,
                           int64_t scratch_bytes, vui_stream_t stream) {
  if (!c) { vui_set_error("NULL codec"); return VUI_EINVAL; }
  return decode_pass(c, codes, n_frames, n_q, audio_out, scratch, scratch_bytes, block_frames(c->cfg), stream);
}

int vui_codec_decode_clip(vui_codec* c, const int64_t* codes, int32_t n_frames, int32_t n_q, float* audio_out, void* scratch,
                          int64_t scratch_bytes, vui_stream_t stream) {
  if (!c) { vui_set_error("NULL codec"); return VUI_EINVAL; }
  return decode_pass(c, codes, n_frames, n_q, audio_out, scratch, scratch_bytes, clip_frames(c->cfg), stream);
}

int64_t vui_codec_status(vui_codec* c, vui_stream_t stream) {
  if (!c) { vui_set_error("NULL codec"); return VUI_EINVAL; }
  int h[2] = {0, 0};
  uint32_t lerr = 0;
  HIP_TRY(hipMemcpyAsync(h, c->ctr, sizeof(h), hipMemcpyDeviceToHost, (hipStream_t)stream));
  if (c->trunk.lerr) HIP_TRY(hipMemcpyAsync(&lerr, c->trunk.lerr, sizeof(lerr), hipMemcpyDeviceToHost, (hipStream_t)stream));
  HIP_TRY(hipStreamSynchronize((hipStream_t)stream));
  if (lerr) {
    vui_set_error(lerr == 2 ? "codec: the persistent kernel's launch count wrapped; create the decoder again"
                            : "codec: an exchange wait of the persistent kernel timed out (is another kernel running on the device?)");
    return VUI_EHIP;
  }
  if (h[1] == 1) { vui_set_error("codec: a code outside [0, %d) was clamped", c->cfg.codebook_size); return VUI_EINVAL; }
  if (h[1] == 2) { vui_set_error("codec: more than max_seq=%d frames since the last reset", c->cfg.max_seq); return VUI_EINVAL; }
  return h[0];
}
