// deltanet.hip — the linear-attention layer parts of Qwen3.5 on gfx950: the
// depthwise causal conv1d (one decode step with its ring state, and the whole
// sequence) and the gated delta-rule recurrence (the fused decode step, the
// plain step and the whole sequence), plus the prefill's prep (l2 norms, gates)
// and its gated-RMSNorm epilogue.
//
// Reference: src/kernels/causal_conv1d.jl, src/kernels/deltanet_recurrent.jl,
// src/kernels/deltanet_fused.jl and their call sites in src/llm/qwen35.jl
// (decode!: :210-232, forward: :320-365).
//
// The recurrence: per (value head, sequence) a state S (Dk x Dv, fp32) with
//   S = decay S;  delta = beta (v - S^T k);  S += k delta^T;  o = S^T q.
// Every column of S evolves on its own given k, q, and its v entry, so the
// kernels split the columns over waves with no cross-wave traffic: wave w
// owns 2 NI columns; lane (j = lane % 32, h = lane / 32) holds rows 4j .. 4j+3
// of columns 2 NI w + 2 i + h, i < NI (one 16-byte load per i: two adjacent
// 512-byte columns per load instruction, 1 KB contiguous). The column sums
// S^T k and S^T q are butterfly reduce-scatters over the 32 lanes of a half:
// NI partial sums per lane become one full sum per lane group. The state is
// read once and written once per step (the reference makes two passes).
#include "common.h"
#include "kernels.h"

namespace vm {

namespace {

constexpr int DN_D = 128;  // Dk = Dv (Qwen3.5: deltanet.jl:12, qwen35.jl:19)

// v[l ^ M] within each 32-lane half: DPP quad permutes for M = 1, 2, the
// swizzle unit's bitmask mode (and 0x1f, xor M) for M = 4, 8, 16.
template <int M>
__device__ __forceinline__ float xor32(float v) {
  const int x = __float_as_int(v);
  if constexpr (M == 1) return __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0xB1, 0xF, 0xF, false));
  if constexpr (M == 2) return __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x4E, 0xF, 0xF, false));
  return __int_as_float(__builtin_amdgcn_ds_swizzle(x, 0x1F | (M << 10)));
}

__device__ __forceinline__ float half_sum(float v) {
  v += xor32<16>(v);
  v += xor32<8>(v);
  v += xor32<4>(v);
  v += xor32<2>(v);
  return v + xor32<1>(v);
}

// One scatter level over mask bit M: N values (index m + (N/2) * bit for the
// kept half) -> N / 2, each summed with the partner lane's matching value.
template <int M, int N>
__device__ __forceinline__ void scatter_level(float (&p)[16], bool bit) {
#pragma unroll
  for (int m = 0; m < N / 2; ++m) {
    const float keep = bit ? p[m + N / 2] : p[m];
    const float send = bit ? p[m] : p[m + N / 2];
    p[m] = keep + xor32<M>(send);
  }
}
template <int M>
__device__ __forceinline__ float sum_masks(float v) {  // plain sums over masks M, M/2, .., 1
  if constexpr (M >= 1) return sum_masks<M / 2>(v + xor32<M>(v));
  else return v;
}
template <int N, int M>
__device__ __forceinline__ float rs_level(float (&p)[16], int j) {
  if constexpr (N == 1) {
    return sum_masks<M>(p[0]);
  } else {
    scatter_level<M, N>(p, (j & M) != 0);
    return rs_level<N / 2, M / 2>(p, j);
  }
}
// p[0 .. NI-1]: this lane's partial sums of its NI columns. Scatter levels on
// masks 16, 8, .. (log2 NI of them) halve the values held, plain sums on the
// rest of the mask bits finish: every lane then holds the sum over the 32 lanes
// of its half for column index i = j >> (5 - log2 NI).
template <int NI>
__device__ __forceinline__ float reduce_scatter(float (&p)[16], int j) {
  static_assert(NI == 16 || NI == 8 || NI == 4 || NI == 2, "NI");
  return rs_level<NI, 16>(p, j);
}

// The sum of column index i sits in lanes (i << SH) .. of each half: lane
// (j, h) fetches index i of its own half.
template <int NI>
__device__ __forceinline__ float column_value(float v, int i, int h) {
  constexpr int SH = NI == 16 ? 1 : NI == 8 ? 2 : NI == 4 ? 3 : 4;
  const float lo = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), i << SH));
  const float hi = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32 + (i << SH)));
  return h ? hi : lo;
}

// One delta step of this lane's slice s[i][0..3] (rows 4j.., column index i):
// returns o = S'^T q for column index j >> SH (the lane group's column).
template <int NI>
__device__ __forceinline__ float delta_step(float (&s)[16][4], const float (&kn)[4],
                                            const float (&qn)[4], float v_col, float beta,
                                            float decay, int j, int h) {
  float p[16];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
#pragma unroll
    for (int e = 0; e < 4; ++e) s[i][e] *= decay;
    p[i] = s[i][0] * kn[0] + s[i][1] * kn[1] + s[i][2] * kn[2] + s[i][3] * kn[3];
  }
  const float acc = reduce_scatter<NI>(p, j);
  const float delta = beta * (v_col - acc);
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const float d = column_value<NI>(delta, i, h);
#pragma unroll
    for (int e = 0; e < 4; ++e) s[i][e] += kn[e] * d;
    p[i] = s[i][0] * qn[0] + s[i][1] * qn[1] + s[i][2] * qn[2] + s[i][3] * qn[3];
  }
  return reduce_scatter<NI>(p, j);
}

template <int NI>
__device__ __forceinline__ void load_state(float (&s)[16][4], const float* base, int w, int lane) {
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const f32x4 t = __builtin_nontemporal_load(
        reinterpret_cast<const f32x4*>(base + (int64_t)(2 * NI * w + 2 * i) * DN_D + 4 * lane));
    s[i][0] = t[0];
    s[i][1] = t[1];
    s[i][2] = t[2];
    s[i][3] = t[3];
  }
}
template <int NI>
__device__ __forceinline__ void store_state(const float (&s)[16][4], float* base, int w, int lane) {
#pragma unroll
  for (int i = 0; i < NI; ++i)
    __builtin_nontemporal_store(f32x4{s[i][0], s[i][1], s[i][2], s[i][3]},
                                reinterpret_cast<f32x4*>(base + (int64_t)(2 * NI * w + 2 * i) * DN_D + 4 * lane));
}

__device__ __forceinline__ void load4_bf16(const uint16_t* p, float (&x)[4]) {
  const uint2 u = *reinterpret_cast<const uint2*>(p);
  x[0] = __uint_as_float(u.x << 16);
  x[1] = __uint_as_float(u.x & 0xffff0000u);
  x[2] = __uint_as_float(u.y << 16);
  x[3] = __uint_as_float(u.y & 0xffff0000u);
}

}  // namespace

// ---- fused_deltanet_decode! (deltanet_fused.jl:27-141): one block of four
// waves per (value head, sequence), 32 columns per wave (NI = 16).
__global__ __launch_bounds__(256) void deltanet_fused_decode_kernel(DeltaFusedArgs a) {
  constexpr int NI = 16;
  const int hv = blockIdx.x, b = blockIdx.y;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, j = lane & 31, h = lane >> 5;
  const int hk = hv / (a.Hv / a.Hk);
  const int64_t sb = ((int64_t)b * a.Hv + hv) * DN_D * DN_D;
  float s[16][4];
  load_state<NI>(s, a.s_in + sb, w, lane);
  float q[4], k[4];
  load4_bf16(a.q + b * a.q_sb + hk * DN_D + 4 * j, q);
  load4_bf16(a.k + b * a.k_sb + hk * DN_D + 4 * j, k);
  const int col = 2 * NI * w + 2 * (j >> 1) + h;  // this lane group's column
  const float v_col = bf2f(a.v[b * a.v_sb + hv * DN_D + col]);
  const float z_col = bf2f(a.z[b * a.z_sb + hv * DN_D + col]);
  const float w_col = bf2f(a.norm_w[col]);
  // per-value-head gates (deltanet_fused.jl:52-59)
  const float spi = bf2f(a.alpha[b * a.a_sb + hv]) + a.dt_bias[hv];
  const float sp = spi > 20.0f ? spi : logf(1.0f + expf(spi));
  const float decay = expf(-expf(a.a_log[hv]) * sp);
  const float beta = accurate_sigmoid(bf2f(a.beta[b * a.b_sb + hv]));
  // l2 norms over the shared qk head (deltanet_fused.jl:61-71)
  const float qss = half_sum(q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3]);
  const float kss = half_sum(k[0] * k[0] + k[1] * k[1] + k[2] * k[2] + k[3] * k[3]);
  const float qsc = 1.0f / sqrtf(qss + 1e-6f) / sqrtf((float)DN_D);
  const float ksc = 1.0f / sqrtf(kss + 1e-6f);
  float qn[4], kn[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    qn[e] = q[e] * qsc;
    kn[e] = k[e] * ksc;
  }
  const float out = delta_step<NI>(s, kn, qn, v_col, beta, decay, j, h);
  store_state<NI>(s, a.s_out + sb, w, lane);
  // gated RMSNorm over the Dv columns (deltanet_fused.jl:98-105): lanes with j
  // even hold each column once
  __shared__ float red[4];
  const float ss = half_sum((j & 1) ? 0.f : out * out);
  const float wave_ss = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ss), 0)) +
                        __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ss), 32));
  if (lane == 0) red[w] = wave_ss;
  __syncthreads();
  const float tot = red[0] + red[1] + red[2] + red[3];
  const float rstd = 1.0f / sqrtf(tot / (float)DN_D + a.eps);
  if ((j & 1) == 0)
    a.o[b * a.o_sb + hv * DN_D + col] = f2bf(out * rstd * w_col * accurate_silu(z_col));
}

// ---- the DeltaNet layer's decode step after its projection in one kernel
// (qwen35.jl:212-232): one workgroup of 4 R waves per (qk head hk, sequence),
// R = Hv / Hk value heads. First every thread takes 4-channel groups of the
// projection [q | k | v | z | alpha | beta] of this head: the stream-K
// partials summed in workgroup order and rounded to bf16 (the value linear!
// stores), then for q, k and v the conv step as conv1d_update_sk_kernel
// (ring shift, silu, bf16), into LDS, the channels' ring columns written
// (each channel has one owner: the qk head's q and k, its R heads' v). The
// state loads are issued first and land meanwhile. Then wave group j runs
// fused_deltanet_decode! for value head hk R + j as deltanet_fused_decode_kernel,
// its inputs from LDS: bit for bit the results of linear_causal_conv1d
// followed by fused_deltanet_decode, one launch and the bf16 projection and
// conv output round trips fewer.
namespace {
__device__ __forceinline__ void unpack4(const uint2& u, float (&x)[4]) {
  x[0] = __uint_as_float(u.x << 16);
  x[1] = __uint_as_float(u.x & 0xffff0000u);
  x[2] = __uint_as_float(u.y << 16);
  x[3] = __uint_as_float(u.y & 0xffff0000u);
}
}  // namespace

template <int KC, int R>
__global__ __launch_bounds__(256 * R) void deltanet_decode_sk_kernel(DeltaDecodeSkArgs a) {
  constexpr int NI = 16;
  const DeltaFusedArgs& f = a.f;
  const Conv1dArgs& c = a.c;
  const int hk = blockIdx.x, b = blockIdx.y, tid = threadIdx.x;
  const int j = tid >> 8, t = tid & 255;  // value head hk R + j; thread t of its group
  const int lane = t & 63, w = t >> 6, jl = lane & 31, h = lane >> 5;
  const int hv = hk * R + j;
  const int64_t sb = ((int64_t)b * f.Hv + hv) * DN_D * DN_D;
  float s[16][4];
  load_state<NI>(s, f.s_in + sb, w, lane);
  // LDS: q, k, v[R], z[R] (DN_D each), alpha[R], beta[R]
  __shared__ float xs[(2 + 2 * R) * DN_D + 2 * R];
  __shared__ float red[R][4];
  constexpr int XA = (2 + 2 * R) * DN_D;
  for (int g = tid; g < 64 + 64 * R; g += 256 * R) {
    int ch, xo;  // projection channel and LDS slot of the group's first element
    if (g < 64) {  // q (g < 32) or k of head hk
      ch = (g < 32 ? 0 : f.Hk * DN_D) + hk * DN_D + 4 * (g & 31);
      xo = (g >> 5) * DN_D + 4 * (g & 31);
    } else if (g < 64 + 32 * R) {  // v of head hk R + jj
      const int jj = (g - 64) >> 5;
      ch = 2 * f.Hk * DN_D + (hk * R + jj) * DN_D + 4 * (g & 31);
      xo = (2 + jj) * DN_D + 4 * (g & 31);
    } else {  // z of head hk R + jj
      const int jj = (g - 64 - 32 * R) >> 5;
      ch = c.D + (hk * R + jj) * DN_D + 4 * (g & 31);
      xo = (2 + R + jj) * DN_D + 4 * (g & 31);
    }
    const float4 sum = gemv_sk_sum4(a.part, a.G, a.chunk, ch, b);
    const uint2 xr = make_uint2(pack2(sum.x, sum.y), pack2(sum.z, sum.w));  // bf16 projection
    float x4[4];
    if (g < 64 + 32 * R) {
      uint2 raw[KC];
#pragma unroll
      for (int i = 0; i < KC - 1; ++i)
        raw[i] = *reinterpret_cast<const uint2*>(c.s_in + b * c.s_sb + (int64_t)(i + 1) * c.s_cs + ch);
      raw[KC - 1] = xr;
      float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < KC; ++i) {
        float v[4], wf[4];
        unpack4(raw[i], v);
        unpack4(*reinterpret_cast<const uint2*>(c.w + (int64_t)i * c.w_cs + ch), wf);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += v[e] * wf[e];
      }
#pragma unroll
      for (int i = 0; i < KC; ++i)
        *reinterpret_cast<uint2*>(c.s_out + b * c.s_sb + (int64_t)i * c.s_cs + ch) = raw[i];
      if (c.bias) {
        float bf4[4];
        unpack4(*reinterpret_cast<const uint2*>(c.bias + ch), bf4);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += bf4[e];
      }
      if (c.act) {
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = accurate_silu(acc[e]);
      }
      unpack4(make_uint2(pack2(acc[0], acc[1]), pack2(acc[2], acc[3])), x4);  // bf16 conv output
    } else {
      unpack4(xr, x4);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) xs[xo + e] = x4[e];
  }
  if (tid < 2 * R) {  // alpha (tid < R) and beta of head hk R + tid % R
    const int ch = c.D + f.Hv * DN_D + (tid < R ? 0 : f.Hv) + hk * R + tid % R;
    xs[XA + tid] = __uint_as_float(pack2(gemv_sk_sum1(a.part, a.G, a.chunk, ch, b), 0.f) << 16);
  }
  __syncthreads();
  float q[4], k[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    q[e] = xs[4 * jl + e];
    k[e] = xs[DN_D + 4 * jl + e];
  }
  const int col = 2 * NI * w + 2 * (jl >> 1) + h;  // this lane group's column
  const float v_col = xs[(2 + j) * DN_D + col];
  const float z_col = xs[(2 + R + j) * DN_D + col];
  const float w_col = bf2f(f.norm_w[col]);
  const float spi = xs[XA + j] + f.dt_bias[hv];
  const float sp = spi > 20.0f ? spi : logf(1.0f + expf(spi));
  const float decay = expf(-expf(f.a_log[hv]) * sp);
  const float beta = accurate_sigmoid(xs[XA + R + j]);
  const float qss = half_sum(q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3]);
  const float kss = half_sum(k[0] * k[0] + k[1] * k[1] + k[2] * k[2] + k[3] * k[3]);
  const float qsc = 1.0f / sqrtf(qss + 1e-6f) / sqrtf((float)DN_D);
  const float ksc = 1.0f / sqrtf(kss + 1e-6f);
  float qn[4], kn[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    qn[e] = q[e] * qsc;
    kn[e] = k[e] * ksc;
  }
  const float out = delta_step<NI>(s, kn, qn, v_col, beta, decay, jl, h);
  store_state<NI>(s, f.s_out + sb, w, lane);
  const float ss = half_sum((jl & 1) ? 0.f : out * out);
  const float wave_ss = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ss), 0)) +
                        __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ss), 32));
  if (lane == 0) red[j][w] = wave_ss;
  __syncthreads();
  const float tot = red[j][0] + red[j][1] + red[j][2] + red[j][3];
  const float rstd = 1.0f / sqrtf(tot / (float)DN_D + f.eps);
  if ((jl & 1) == 0)
    f.o[b * f.o_sb + hv * DN_D + col] = f2bf(out * rstd * w_col * accurate_silu(z_col));
}

// ---- deltanet_sequence! (deltanet_recurrent.jl:109-198) and, at T = 1,
// deltanet_recurrent_decode! (:15-95): fp32 inputs already normed and gated.
// Grid (columns / (2 NI * 4), Hv, B), four independent waves per block; the
// state stays in registers across the T steps, the next step's inputs load
// while the current one computes.
template <int NI>
__global__ __launch_bounds__(256) void deltanet_sequence_kernel(DeltaSeqArgs a) {
  const int hv = blockIdx.y, b = blockIdx.z;
  const int lane = threadIdx.x & 63, j = lane & 31, h = lane >> 5;
  const int w = blockIdx.x * 4 + (threadIdx.x >> 6);  // wave index within the head
  const int hk = hv / (a.Hv / a.Hk);
  const int64_t sb = ((int64_t)b * a.Hv + hv) * DN_D * DN_D;
  constexpr int SH = NI == 16 ? 1 : NI == 8 ? 2 : NI == 4 ? 3 : 4;
  const int col = 2 * NI * w + 2 * (j >> SH) + h;
  float s[16][4];
  load_state<NI>(s, a.s_in + sb, w, lane);
  const float* qp = a.q + ((int64_t)b * a.Hk + hk) * a.T * DN_D + 4 * j;
  const float* kp = a.k + ((int64_t)b * a.Hk + hk) * a.T * DN_D + 4 * j;
  const float* vp = a.v + ((int64_t)b * a.Hv + hv) * a.T * DN_D + col;
  const float* bp = a.beta + (int64_t)b * a.T * a.Hv + hv;
  const float* gp = a.gate + (int64_t)b * a.T * a.Hv + hv;
  float* op = a.o + ((int64_t)b * a.Hv + hv) * a.T * DN_D + col;
  float4 qv = *reinterpret_cast<const float4*>(qp);
  float4 kv = *reinterpret_cast<const float4*>(kp);
  float v_col = *vp, beta = *bp, gate = *gp;
  for (int t = 0; t < a.T; ++t) {
    const float qn[4] = {qv.x, qv.y, qv.z, qv.w};
    const float kn[4] = {kv.x, kv.y, kv.z, kv.w};
    const float vc = v_col, bt = beta, decay = expf(gate);
    if (t + 1 < a.T) {  // the next step's inputs
      const int64_t o4 = (int64_t)(t + 1) * DN_D;
      qv = *reinterpret_cast<const float4*>(qp + o4);
      kv = *reinterpret_cast<const float4*>(kp + o4);
      v_col = vp[o4];
      beta = bp[(int64_t)(t + 1) * a.Hv];
      gate = gp[(int64_t)(t + 1) * a.Hv];
    }
    const float out = delta_step<NI>(s, kn, qn, vc, bt, decay, j, h);
    if ((j & ((1 << SH) - 1)) == 0) op[(int64_t)t * DN_D] = out;
  }
  store_state<NI>(s, a.s_out + sb, w, lane);
}

// ---- the chunked form of deltanet_sequence! ---------------------------------
// Over a chunk of C tokens (G the in-chunk cumulative log decay, gamma = exp G,
// D_ij = gamma_i / gamma_j) the recurrence's per-token corrections delta_i =
// beta_i (v_i - alpha_i S_{i-1}^T k_i) satisfy the lower-triangular system
//     (I + L) delta = beta (V - gamma K S_0),   L_ij = beta_i D_ij k_i.k_j (i > j)
// so delta = T R with T = (I + L)^-1 and R = beta V - beta gamma (K S_0); then
// O = gamma (Q S_0) + M delta with M_ij = D_ij q_i.k_j (j <= i), and
// S_C = gamma_C S_0 + K^T (e delta) with e_j = gamma_C / gamma_j (exact algebra
// of the sequential update). Two launches, and the gated norm as a third:
// Phase 1 (deltanet_chunk_kernel, chunk-parallel): what does not depend on the
// state: the Gram K K^T and Q K^T once per qk head, then per value head L, T by
// fp32 forward substitution, M, and the rows' decays.
// Phase 2 (deltanet_scan_kernel, sequential over chunks): one workgroup per 16
// state columns of a value head. Four waves carry the state chain (K S_0, T R,
// the state), four others form and store O beside them and stage the next K.
// Phase 3, fused form only: the layer's gated RMSNorm with z (qwen35.jl:360-364)
// on O, gated_rms_norm_*_kernel.
// Little passes between the phases: T, M and the decays, 33 KB per (chunk, value
// head), and K and Q split, 64 KB per (chunk, qk head), which the column blocks
// of all its value heads share in one XCD's L2. (-W, K~^T and U took 98 KB per
// value head, and S_0 and delta, passed on to an output kernel, another 98 KB.)
// The products run on the bf16 MFMA (v_mfma_f32_16x16x32_bf16) in split
// precision: each fp32 operand x is hi = bf16(x) and lo = bf16(x - hi), and a
// product is hi hi + hi lo + lo hi with fp32 accumulation (about 2^-16
// relative per product).
namespace {
constexpr int DC = 64;   // chunk length
constexpr int CBW = 16;  // state columns per scan workgroup
// per (chunk, value head, sequence) unit of phase 1's results, floats. T and M
// are split into bf16 hi / lo in the A operand order of
// v_mfma_f32_16x16x32_bf16: [row tile w 4][k step ks 2][hl 2][lane 64][8] with
// lane l element j = X[16 w + l % 16][32 ks + 8 (l / 16) + j]; the blocks ks >
// w / 2 lie above the diagonal and are neither written nor read
constexpr int UO_T = 0;
constexpr int UO_M = 4096;
constexpr int UO_SC = 8192;  // [beta 64][beta gamma 64][gamma_C / gamma 64][gamma 64]
constexpr int UNIT = 8448;   // floats per unit (33 792 B, a multiple of 256)
// per (chunk, qk head, sequence): K split, [hl 2][token 64][dk 128] bf16 (rows
// past the sequence's end 0), and Q split in A operand order, [row tile w 4][k
// step ks 4][hl 2][lane 64][8] bf16 (rows past the end repeat the last)
constexpr int KQ_Q = 8192;
constexpr int KQ_UNIT = 16384;  // floats per unit (64 KB)

// the chunk's inclusive cumulative log decay (one wave, one token per lane; log
// decays below -110 are taken as -110: expf underflows to exactly 0 below
// about -104, so every decay the recurrence applies is unchanged, while the
// cumulative sums stay finite; a -inf log decay, e.g. from softplus
// overflowing in log1p(exp(x)) at x > 88.7, would make their differences NaN)
__device__ __forceinline__ float chunk_cumsum(const DeltaSeqArgs& q, int b, int hv, int t0, int n,
                                              int t) {
  const int64_t g = ((int64_t)b * q.T + t0 + min(t, n - 1)) * q.Hv + hv;  // in bounds
  const float gt = t < n ? fmaxf(q.gate[g], -110.0f) : 0.f;
  float G = gt;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const float o = __shfl_up(G, off);
    if (t >= off) G += o;
  }
  return G;
}
}  // namespace

// the workspace: the units of every (sequence, value head, chunk), the K and Q
// units of every (sequence, qk head, chunk), then the fused form's O (fp32)
__device__ __forceinline__ float* dn_unit(const DeltaChunkArgs& a, int b, int hv, int NC, int c) {
  return a.ws + (((int64_t)b * a.s.Hv + hv) * NC + c) * UNIT;
}
__device__ __forceinline__ uint16_t* dn_kq(const DeltaChunkArgs& a, int b, int hk, int NC, int c) {
  return reinterpret_cast<uint16_t*>(a.ws + (int64_t)a.s.B * a.s.Hv * NC * UNIT +
                                     (((int64_t)b * a.s.Hk + hk) * NC + c) * KQ_UNIT);
}

namespace {
// 4 fp32 values as bf16 hi and lo parts (x = hi + lo to about 2^-16), 4 each
__device__ __forceinline__ void split4(const f32x4& x, uint2& hi, uint2& lo) {
  hi = make_uint2(pack2(x[0], x[1]), pack2(x[2], x[3]));
  lo = make_uint2(pack2(x[0] - __uint_as_float(hi.x << 16), x[1] - __uint_as_float(hi.x & 0xffff0000u)),
                  pack2(x[2] - __uint_as_float(hi.y << 16), x[3] - __uint_as_float(hi.y & 0xffff0000u)));
}
__device__ __forceinline__ void split8(const f32x4& a, const f32x4& b, uint4& hi, uint4& lo) {
  uint2 h0, l0, h1, l1;
  split4(a, h0, l0);
  split4(b, h1, l1);
  hi = make_uint4(h0.x, h0.y, h1.x, h1.y);
  lo = make_uint4(l0.x, l0.y, l1.x, l1.y);
}
// acc += A B in split precision (hi hi + hi lo + lo hi) on v_mfma_f32_16x16x32_bf16
// (A lane l = A[l % 16][8 (l / 16) + j], B lane l = B[8 (l / 16) + j][l % 16], D
// lane l reg r = D[4 (l / 16) + r][l % 16])
__device__ __forceinline__ f32x4 mfma_x3(const uint4& ah, const uint4& al, const uint4& bh,
                                         const uint4& bl, f32x4 acc) {
  acc = mfma16(al, bh, acc);
  acc = mfma16(ah, bl, acc);
  return mfma16(ah, bh, acc);
}
__device__ __forceinline__ uint4 lds16(const uint16_t* p) { return *reinterpret_cast<const uint4*>(p); }
constexpr int KW = DN_D + 8;  // LDS row of K hi / lo (bf16; 16-byte aligned, banks skewed)
constexpr int LSW = DC + 4;   // LDS row of L (floats)
constexpr int TW = DC + 8;    // LDS row of T hi / lo (bf16)
}  // namespace

// Phase 1. One workgroup per (chunk, two value heads of a qk head, sequence). Wave w
// takes rows i = 16 w .. of G = K K^T and P = Q K^T (lane l: row 16 w + l % 16, reg r of tile jt <=
// w: column 16 jt + 4 (l / 16) + r; tiles above the diagonal are not formed).
// Then every wave writes its rows of each head's L (LDS) and M (workspace); wave 3 solves (I + L) T = I for the first head and wave 2 for
// the second, lane c for column c, in fp32 (L's rows read from LDS ahead of
// their use); T, split, goes through LDS into the operand order.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
void deltanet_chunk_kernel(DeltaChunkArgs a) {
  const DeltaSeqArgs& q = a.s;
  const int R = q.Hv / q.Hk, RP = (R + 1) / 2;
  const int c = blockIdx.x, hk = blockIdx.y / RP, b = blockIdx.z, t = threadIdx.x;
  const int hv0 = hk * R + 2 * (blockIdx.y % RP);   // the workgroup's value heads
  const int nr = min(2, hk * R + R - hv0);
  const int lane = t & 63, l16 = lane & 15, r4 = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);  // wave-uniform: scalar branches
  const int t0 = c * DC, n = min(DC, q.T - t0);
  const int NC = (q.T + DC - 1) / DC;
  // K split (rows of KW), then in its place L and later T (hi, lo) of two heads
  __shared__ __attribute__((aligned(16))) float LT[2][DC * TW];
  static_assert(sizeof(LT) >= 2 * DC * KW * sizeof(uint16_t), "K hi, lo");
  static_assert(sizeof(LT[0]) >= DC * LSW * sizeof(float), "L");
  __shared__ __attribute__((aligned(16))) float Gs[2][DC], Bs[2][DC];
  uint16_t* const Kh = reinterpret_cast<uint16_t*>(LT);
  uint16_t* const Kl = Kh + DC * KW;
  const float* kp = q.k + (((int64_t)b * q.Hk + hk) * q.T + t0) * DN_D;
  const float* qp = q.q + (((int64_t)b * q.Hk + hk) * q.T + t0) * DN_D;
  const int i = 16 * w + l16;  // this lane's row of G, P, L and M
  uint4 qh[4], ql[4];          // Q[i][32 ks + 8 (l / 16) ..], split
  uint16_t* const kq = dn_kq(a, b, hk, NC, c);
  const bool first = blockIdx.y % RP == 0;  // this workgroup writes the qk head's K and Q
  {
    f32x4 kv[DC / 8], qv[8];
#pragma unroll
    for (int m = 0; m < DC / 8; ++m)  // float4 t + 256 m of the chunk's K
      kv[m] = *reinterpret_cast<const f32x4*>(kp + min((t >> 5) + 8 * m, n - 1) * DN_D + 4 * (t & 31));
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int u = 0; u < 2; ++u)
        qv[2 * ks + u] = *reinterpret_cast<const f32x4*>(qp + (int64_t)min(i, n - 1) * DN_D + 32 * ks +
                                                         8 * r4 + 4 * u);
    if (w < nr) {  // wave w: beta, the cumulative log decay and the decays of its value head
      const int hv = hv0 + w;
      const float bt = lane < n ? q.beta[((int64_t)b * q.T + t0 + lane) * q.Hv + hv] : 0.f;
      const float g = chunk_cumsum(q, b, hv, t0, n, lane), eg = expf(g);
      Gs[w][lane] = g;
      Bs[w][lane] = bt;
      float* sc = dn_unit(a, b, hv, NC, c) + UO_SC + lane;
      sc[0] = bt;
      sc[64] = bt * eg;
      sc[128] = expf(__shfl(g, DC - 1) - g);
      sc[192] = eg;
    }
#pragma unroll
    for (int m = 0; m < DC / 8; ++m) {  // rows past the end read as 0
      const int r = (t >> 5) + 8 * m;
      uint2 hi, lo;
      split4(kv[m], hi, lo);
      if (r >= n) hi = lo = make_uint2(0, 0);
      *reinterpret_cast<uint2*>(&Kh[r * KW + 4 * (t & 31)]) = hi;
      *reinterpret_cast<uint2*>(&Kl[r * KW + 4 * (t & 31)]) = lo;
      if (first) {
        *reinterpret_cast<uint2*>(kq + 4 * (t + 256 * m)) = hi;
        *reinterpret_cast<uint2*>(kq + DC * DN_D + 4 * (t + 256 * m)) = lo;
      }
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      split8(qv[2 * ks], qv[2 * ks + 1], qh[ks], ql[ks]);
      if (first) {
        uint16_t* const qo = kq + 2 * KQ_Q + (w * 4 + ks) * 1024 + lane * 8;
        *reinterpret_cast<uint4*>(qo) = qh[ks];
        *reinterpret_cast<uint4*>(qo + 512) = ql[ks];
      }
    }
  }
  __syncthreads();
  f32x4 G[4], P[4];
#pragma unroll
  for (int jt = 0; jt < 4; ++jt) G[jt] = P[jt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    const int o = 32 * ks + 8 * r4;
    const uint4 bh = lds16(&Kh[i * KW + o]), bl = lds16(&Kl[i * KW + o]);
#pragma unroll
    for (int jt = 0; jt < 4; ++jt) {
      if (jt > w) break;
      const uint4 ah = lds16(&Kh[(16 * jt + l16) * KW + o]), al = lds16(&Kl[(16 * jt + l16) * KW + o]);
      G[jt] = mfma_x3(ah, al, bh, bl, G[jt]);
      P[jt] = mfma_x3(ah, al, qh[ks], ql[ks], P[jt]);
    }
  }
  __syncthreads();  // K read: L takes its place
  for (int rr = 0; rr < nr; ++rr) {
    uint16_t* const mo =
        reinterpret_cast<uint16_t*>(dn_unit(a, b, hv0 + rr, NC, c) + UO_M) + w * 2048;
    const float Gi = Gs[rr][i], Bi = Bs[rr][i];
#pragma unroll
    for (int jt = 0; jt < 4; ++jt) {
      if (jt > (w | 1)) break;
      const f32x4 Gj = *reinterpret_cast<const f32x4*>(&Gs[rr][16 * jt + 4 * r4]);
      f32x4 l, m;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = 16 * jt + 4 * r4 + r;
        const float d = expf(Gi - Gj[r]);
        l[r] = i > j ? Bi * d * G[jt][r] : 0.f;
        m[r] = (j <= i && i < n) ? d * P[jt][r] : 0.f;
      }
      *reinterpret_cast<f32x4*>(&LT[rr][i * LSW + 16 * jt + 4 * r4]) = l;
      uint2 mh, ml;
      split4(m, mh, ml);
      const int l2 = 16 * (2 * (jt & 1) + (r4 >> 1)) + l16;  // operand lane of these 4 columns
      uint16_t* const d = mo + (jt >> 1) * 1024 + l2 * 8 + 4 * (r4 & 1);
      *reinterpret_cast<uint2*>(d) = mh;
      *reinterpret_cast<uint2*>(d + 512) = ml;
    }
  }
  __syncthreads();
  if (3 - w < nr) {
    // (I + L) T = I: lane c holds column c (rows above c stay 0, T[c][c] = 1).
    // The float4s of L's rows 1 .. 63 (j < i) are read in order through a ring
    // of SD registers, SD ahead of their use (the cursor (pi, pj) is a
    // constant once the loops are unrolled). All four lanes of a float4 enter
    // the sums: the ones at j >= i hold L's zeros above the diagonal (the Gram
    // tiles on it are written whole) times x[j] = 0, and a load whose every
    // register is used keeps the allocator from reloading into one in flight.
    constexpr int SD = 12;
    const float* const L = LT[3 - w];
    float x[DC];
#pragma unroll
    for (int k = 0; k < DC; ++k) x[k] = 0.f;
    f32x4 ring[SD];
    int pi = 1, pj = 0;  // next float4 to read: row pi, columns 4 pj ..
#pragma unroll
    for (int d = 0; d < SD; ++d) {
      ring[d] = *reinterpret_cast<const f32x4*>(&L[pi * LSW + 4 * pj]);
      if (4 * (pj + 1) < pi) ++pj; else { ++pi; pj = 0; }
    }
    x[0] = lane == 0 ? 1.f : 0.f;
    int idx = 0;
#pragma unroll
    for (int k = 1; k < DC; ++k) {
      float acc[4] = {k == lane ? 1.f : 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j4 = 0; 4 * j4 < k; ++j4) {
        const f32x4 l4 = ring[idx % SD];
        if (pi < DC) {
          ring[idx % SD] = *reinterpret_cast<const f32x4*>(&L[pi * LSW + 4 * pj]);
          if (4 * (pj + 1) < pi) ++pj; else { ++pi; pj = 0; }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] -= l4[e] * x[4 * j4 + e];
        ++idx;
      }
      x[k] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    }
    // T rows, split: columns (c & ~1, c | 1) as one pair, lane c even stores the
    // hi pair, odd the lo pair (L is dead: every read of it is above)
    uint16_t* const Tx = reinterpret_cast<uint16_t*>(LT[3 - w]) + ((lane & 1) ? DC * TW : 0);
#pragma unroll
    for (int k = 0; k < DC; ++k) {
      const float xo = xor32<1>(x[k]);
      const float x0 = (lane & 1) ? xo : x[k], x1 = (lane & 1) ? x[k] : xo;
      const uint32_t hi = pack2(x0, x1);
      const uint32_t lo = pack2(x0 - __uint_as_float(hi << 16), x1 - __uint_as_float(hi & 0xffff0000u));
      *reinterpret_cast<uint32_t*>(Tx + k * TW + (lane & ~1)) = (lane & 1) ? lo : hi;
    }
  }
  __syncthreads();
  for (int rr = 0; rr < nr; ++rr) {
    uint16_t* const to =
        reinterpret_cast<uint16_t*>(dn_unit(a, b, hv0 + rr, NC, c) + UO_T) + w * 2048;
    const uint16_t* const Th = reinterpret_cast<const uint16_t*>(LT[rr]);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      if (ks > (w >> 1)) break;
#pragma unroll
      for (int hl = 0; hl < 2; ++hl)
        *reinterpret_cast<uint4*>(to + (ks * 2 + hl) * 512 + lane * 8) =
            lds16(Th + hl * DC * TW + i * TW + 32 * ks + 8 * r4);
    }
  }
}

namespace {
constexpr int SSW = DN_D + 8;  // LDS row (one state column) of S hi / lo, bf16
constexpr int DSW = DC + 8;    // LDS row (one state column) of R, delta, e delta hi / lo, bf16
// accumulator tile rows k0 + 4 (l / 16) .. +3 of column l % 16, split, into LDS
// transposed (X[k][column] at [column][k], hi then lo)
__device__ __forceinline__ void lds_put(uint16_t* x, int ld, int k0, const f32x4& v, int lane) {
  uint2 hi, lo;
  split4(v, hi, lo);
  uint16_t* const p = x + (lane & 15) * ld + k0 + 4 * (lane >> 4);
  *reinterpret_cast<uint2*>(p) = hi;
  *reinterpret_cast<uint2*>(p + CBW * ld) = lo;
}
// the B operand of k step ks from such a buffer: lane l = X[32 ks + 8 (l / 16) ..][l % 16]
__device__ __forceinline__ void lds_get(const uint16_t* x, int ld, int ks, int lane, uint4& hi,
                                        uint4& lo) {
  const uint16_t* const p = x + (lane & 15) * ld + 32 * ks + 8 * (lane >> 4);
  hi = lds16(p);
  lo = lds16(p + CBW * ld);
}
// a load at a wave-uniform base and a 32-bit byte offset per lane
template <typename T>
__device__ __forceinline__ T ld_off(const void* base, uint32_t bytes) {
  return *reinterpret_cast<const T*>(static_cast<const char*>(base) + bytes);
}
// the scan's LDS: K (two chunks) and S (two chunks) split, R, delta and e delta
struct ScanLds {
  uint16_t k[2][2 * DC * KW];   // [parity][hi, lo][token][dk]
  uint16_t s[2][2 * CBW * SSW];
  uint16_t r[2 * CBW * DSW], d[2 * CBW * DSW], e[2 * CBW * DSW];
};
}  // namespace

// Phase 2. One workgroup of 8 waves per (16 state columns, value head, sequence);
// chunk c uses the LDS buffers of parity c % 2. Per chunk three barriers:
//   chain wave w (0 .. 3): X = K S_0 (rows 16 w), R = beta V - beta gamma X -> LDS | A |
//     delta = T R (rows 16 w), delta and e delta -> LDS | B |
//     S = gamma_C S_0 + K^T (e delta) (dk 32 w ..) -> LDS, other parity | C |
//   wave 4 + w: K of the next chunk into LDS, other parity | A | Q S_0 (rows 16 w) | B |
//     O = gamma (Q S_0) + M delta, stored | C |
// Every operand from memory is loaded one or two chunks ahead into registers.
// The chain's latency (three LDS round trips, three short MFMA chains) bounds a
// chunk; O's products fill its gaps. K goes through LDS because its rows serve
// both as they are (K S_0) and transposed (K^T delta).
// Measured at T = 4096, B = 1, 16 / 32 heads (kernel trace): 128 us, 2.0 us a chunk
// (1.1 us with every operand in cache and no O), after 49 us of phase 1 and before
// 25 us of gated norm: 202 us. The three kernels before (-W and U precomputed, S_0
// and delta passed on to an output kernel) took 86 + 145 + 94 = 325 us.
template <bool CHAIN>
__device__ __forceinline__ void scan_body(const DeltaChunkArgs& a, ScanLds& sm, int b, int hv,
                                          int hk, int cb, int w, int lane) {
  const DeltaSeqArgs& q = a.s;
  const int r4 = lane >> 4, col = lane & 15;
  const int NC = (q.T + DC - 1) / DC;
  const int dv0 = cb * CBW, i0 = 16 * w + 4 * r4;  // this lane's accumulator rows i0 .. i0 + 3
  const bool lower = w < 2;                        // rows below token 32: k step 1 is zero
  const float* const units = dn_unit(a, b, hv, NC, 0);
  if constexpr (CHAIN) {
    const float* const vp = q.v + ((int64_t)b * q.Hv + hv) * q.T * DN_D + dv0;
    const int64_t sb = ((int64_t)b * q.Hv + hv) * DN_D * DN_D;
    f32x4 St[2];  // state tiles d = 2w, 2w + 1: lane l reg e = S[16 d + 4 (l / 16) + e][l % 16]
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      St[x] = *reinterpret_cast<const f32x4*>(q.s_in + sb + (int64_t)(dv0 + col) * DN_D +
                                              16 * (2 * w + x) + 4 * r4);
      lds_put(sm.s[0], SSW, 16 * (2 * w + x), St[x], lane);
    }
    struct Ops {
      uint4 t[2][2];
      f32x4 v, be, bg, ek;
      float gc;
    } o0, o1;
    auto load_rows = [&](Ops& o, int c) __attribute__((always_inline)) {
      c = min(c, NC - 1);
      const int n = min(DC, q.T - c * DC);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        o.v[r] = ld_off<float>(vp + (int64_t)c * DC * DN_D, 4 * (min(i0 + r, n - 1) * DN_D + col));
      const float* sc = units + (int64_t)c * UNIT + UO_SC;
      o.be = ld_off<f32x4>(sc, 4 * i0);
      o.bg = ld_off<f32x4>(sc + 64, 4 * i0);
    };
    auto load_t = [&](Ops& o, int c) __attribute__((always_inline)) {
      c = min(c, NC - 1);
      const uint16_t* tp = reinterpret_cast<const uint16_t*>(units + (int64_t)c * UNIT + UO_T) + w * 2048;
#pragma unroll
      for (int hl = 0; hl < 2; ++hl) o.t[0][hl] = ld_off<uint4>(tp + hl * 512, 16 * lane);
      if (!lower) {
#pragma unroll
        for (int hl = 0; hl < 2; ++hl) o.t[1][hl] = ld_off<uint4>(tp + 1024 + hl * 512, 16 * lane);
      }
      const float* sc = units + (int64_t)c * UNIT + UO_SC;
      o.ek = ld_off<f32x4>(sc + 128, 4 * i0);
      o.gc = sc[192 + DC - 1];
    };
    uint4 kx[4][2];  // K rows 16 w + l % 16 of the coming chunk, A operands of X
    auto read_kx = [&](const uint16_t* k) __attribute__((always_inline)) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int hl = 0; hl < 2; ++hl)
          kx[ks][hl] = lds16(k + hl * DC * KW + (16 * w + col) * KW + 32 * ks + 8 * r4);
    };
    auto chunk = [&](Ops& o, int c, int p) __attribute__((always_inline)) {
      const uint16_t* const kb = sm.k[p];
      f32x4 xa = {0.f, 0.f, 0.f, 0.f}, xb = xa;
      uint4 sh[4], sl[4];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) lds_get(sm.s[p], SSW, ks, lane, sh[ks], sl[ks]);
      // K^T operands of the state product: lane l = K[32 ks + 8 (l / 16) + j][16 d + l % 16]
      uint2 kt[2][2][2][2];  // [x][ks][hl][j / 4]
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int hl = 0; hl < 2; ++hl)
#pragma unroll
            for (int h = 0; h < 2; ++h)
              kt[x][ks][hl][h] = lds_read_tr16(kb + hl * DC * KW +
                                               (32 * ks + 8 * r4 + 4 * h + (col >> 2)) * KW +
                                               16 * (2 * w + x) + 4 * (col & 3));
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        xa = mfma_x3(kx[ks][0], kx[ks][1], sh[ks], sl[ks], xa);
        xb = mfma_x3(kx[2 + ks][0], kx[2 + ks][1], sh[2 + ks], sl[2 + ks], xb);
      }
      lds_put(sm.r, DSW, 16 * w, o.be * o.v - o.bg * (xa + xb), lane);
      load_rows(o, c + 2);
      __syncthreads();  // A
      f32x4 d = {0.f, 0.f, 0.f, 0.f};
      uint4 rh[2], rl[2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) lds_get(sm.r, DSW, ks, lane, rh[ks], rl[ks]);
      d = mfma_x3(o.t[0][0], o.t[0][1], rh[0], rl[0], d);
      if (!lower) d = mfma_x3(o.t[1][0], o.t[1][1], rh[1], rl[1], d);
      lds_put(sm.e, DSW, 16 * w, d * o.ek, lane);
      lds_put(sm.d, DSW, 16 * w, d, lane);
      const float gc = o.gc;
      load_t(o, c + 2);
      __syncthreads();  // B
      uint4 eh[2], el[2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) lds_get(sm.e, DSW, ks, lane, eh[ks], el[ks]);
      read_kx(sm.k[p ^ 1]);  // staged before A
      St[0] = St[0] * gc;
      St[1] = St[1] * gc;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
        for (int x = 0; x < 2; ++x)
          St[x] = mfma_x3(make_uint4(kt[x][ks][0][0].x, kt[x][ks][0][0].y, kt[x][ks][0][1].x, kt[x][ks][0][1].y),
                          make_uint4(kt[x][ks][1][0].x, kt[x][ks][1][0].y, kt[x][ks][1][1].x, kt[x][ks][1][1].y),
                          eh[ks], el[ks], St[x]);
      }
#pragma unroll
      for (int x = 0; x < 2; ++x) lds_put(sm.s[p ^ 1], SSW, 16 * (2 * w + x), St[x], lane);
      __syncthreads();  // C
    };
    load_rows(o0, 0);
    load_t(o0, 0);
    load_rows(o1, 1);
    load_t(o1, 1);
    __syncthreads();
    read_kx(sm.k[0]);
    int c = 0;
    do {
      chunk(o0, c, 0);
      if (c + 1 >= NC) break;
      chunk(o1, c + 1, 1);
      c += 2;
    } while (c < NC);
#pragma unroll
    for (int x = 0; x < 2; ++x)
      *reinterpret_cast<f32x4*>(q.s_out + sb + (int64_t)(dv0 + col) * DN_D + 16 * (2 * w + x) +
                                4 * r4) = St[x];
  } else {
    const uint16_t* const kq = dn_kq(a, b, hk, NC, 0);
    float* const op = q.o + ((int64_t)b * q.Hv + hv) * q.T * DN_D + dv0 + col;
    struct OpsM {
      uint4 m[2][2];
      f32x4 g;
    } o0, o1;
    f32x4 k0[8], k1[8];  // 8 bf16 each
    uint4 q0[4][2], q1[4][2];
    // K: 16-byte pieces t + 256 u of the chunk's [hl][token][dk]
    auto load_k = [&](f32x4 (&k)[8], int c) __attribute__((always_inline)) {
      const uint16_t* p = kq + (int64_t)min(c, NC - 1) * (2 * KQ_UNIT);
#pragma unroll
      for (int u = 0; u < 8; ++u) k[u] = ld_off<f32x4>(p + 2048 * u, 16 * (64 * w + lane));
    };
    auto stage_k = [&](const f32x4 (&v)[8], uint16_t* k) __attribute__((always_inline)) {
      uint16_t* const p = k + (4 * w + (lane >> 4)) * KW + 8 * (lane & 15);
#pragma unroll
      for (int u = 0; u < 8; ++u) *reinterpret_cast<f32x4*>(p + 16 * u * KW) = v[u];
    };
    auto load_q = [&](uint4 (&q)[4][2], int c) __attribute__((always_inline)) {
      const uint16_t* p = kq + (int64_t)min(c, NC - 1) * (2 * KQ_UNIT) + 2 * KQ_Q + w * 4096;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int hl = 0; hl < 2; ++hl) q[ks][hl] = ld_off<uint4>(p + (ks * 2 + hl) * 512, 16 * lane);
    };
    auto load_m = [&](OpsM& o, int c) __attribute__((always_inline)) {
      c = min(c, NC - 1);
      const float* u = units + (int64_t)c * UNIT;
      const uint16_t* mp = reinterpret_cast<const uint16_t*>(u + UO_M) + w * 2048;
#pragma unroll
      for (int hl = 0; hl < 2; ++hl) o.m[0][hl] = ld_off<uint4>(mp + hl * 512, 16 * lane);
      if (!lower) {
#pragma unroll
        for (int hl = 0; hl < 2; ++hl) o.m[1][hl] = ld_off<uint4>(mp + 1024 + hl * 512, 16 * lane);
      }
      o.g = ld_off<f32x4>(u + UO_SC + 192, 4 * i0);
    };
    // qc, o: chunk c's operands; kn: K of chunk c + 1
    auto chunk = [&](f32x4 (&kn)[8], uint4 (&qc)[4][2], OpsM& o, int c, int p) __attribute__((always_inline)) {
      f32x4 oa = {0.f, 0.f, 0.f, 0.f}, ob = oa;
      stage_k(kn, sm.k[p ^ 1]);
      load_k(kn, c + 3);
      __syncthreads();  // A
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        uint4 sh, sl;
        lds_get(sm.s[p], SSW, ks, lane, sh, sl);
        oa = mfma_x3(qc[ks][0], qc[ks][1], sh, sl, oa);
        lds_get(sm.s[p], SSW, 2 + ks, lane, sh, sl);
        ob = mfma_x3(qc[2 + ks][0], qc[2 + ks][1], sh, sl, ob);
      }
      load_q(qc, c + 2);
      oa = (oa + ob) * o.g;
      __syncthreads();  // B
      uint4 dh, dl;
      lds_get(sm.d, DSW, 0, lane, dh, dl);
      oa = mfma_x3(o.m[0][0], o.m[0][1], dh, dl, oa);
      if (!lower) {
        lds_get(sm.d, DSW, 1, lane, dh, dl);
        oa = mfma_x3(o.m[1][0], o.m[1][1], dh, dl, oa);
      }
      float* const oc = op + ((int64_t)c * DC + i0) * DN_D;
      const int n = q.T - c * DC;
      if (n >= DC) {
#pragma unroll
        for (int r = 0; r < 4; ++r) oc[r * DN_D] = oa[r];
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (i0 + r < n) oc[r * DN_D] = oa[r];
      }
      load_m(o, c + 2);
      __syncthreads();  // C
    };
    load_k(k0, 0);
    stage_k(k0, sm.k[0]);
    load_k(k0, 1);
    load_k(k1, 2);
    load_q(q0, 0);
    load_q(q1, 1);
    load_m(o0, 0);
    load_m(o1, 1);
    __syncthreads();
    int c = 0;
    do {
      chunk(k0, q0, o0, c, 0);
      if (c + 1 >= NC) break;
      chunk(k1, q1, o1, c + 1, 1);
      c += 2;
    } while (c < NC);
  }
}

__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void deltanet_scan_kernel(DeltaChunkArgs a) {
  const DeltaSeqArgs& q = a.s;
  // a qk head's column blocks (of its R value heads) share an XCD (workgroup id
  // mod 8) when the (qk head, sequence) groups divide over the 8 XCDs
  const int R = q.Hv / q.Hk, R8 = R * (DN_D / CBW), id = blockIdx.x;
  const bool xcd = (q.Hk * q.B) % 8 == 0;
  const int grp = xcd ? (id & 7) + 8 * ((id >> 3) / R8) : id / R8;
  const int mem = xcd ? (id >> 3) % R8 : id % R8;
  const int hk = grp % q.Hk, b = grp / q.Hk;
  const int hv = hk * R + mem / (DN_D / CBW), cb = mem % (DN_D / CBW);
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  __shared__ __attribute__((aligned(16))) ScanLds sm;
  if (w < 4) {
    scan_body<true>(a, sm, b, hv, hk, cb, w, lane);
  } else {
    scan_body<false>(a, sm, b, hv, hk, cb, w - 4, lane);
  }
}

// ---- the prefill's inputs to the recurrence (qwen35.jl:347-356): one wave per
// (token, head): q / k heads l2-normed (q also by 1/sqrt(Dk)) from the conv
// output, v heads widened to fp32, gates from the alpha | beta projection.
__global__ __launch_bounds__(256) void deltanet_prep_kernel(DeltaPrepArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t wid = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int nh = 2 * a.Hk + a.Hv;  // q heads, k heads, v heads
  const int64_t tok = wid / nh;    // b * T + t
  if (tok >= (int64_t)a.B * a.T) return;
  const int hh = (int)(wid % nh);
  const int b = (int)(tok / a.T), t = (int)(tok % a.T);
  const uint16_t* row = a.cv + (int64_t)b * a.cv_sb + (int64_t)t * a.cv_st + hh * DN_D;
  const float x0 = bf2f(row[2 * lane]), x1 = bf2f(row[2 * lane + 1]);
  if (hh < 2 * a.Hk) {
    const int hk = hh % a.Hk;
    float ss = x0 * x0 + x1 * x1;
    ss += __shfl_xor(ss, 32);
    ss = half_sum(ss);
    const float den = sqrtf(ss + 1e-6f);
    const bool isq = hh < a.Hk;
    const float sc = isq ? 1.0f / sqrtf((float)DN_D) : 1.0f;
    float* dst = (isq ? a.qe : a.ke) + (((int64_t)b * a.Hk + hk) * a.T + t) * DN_D;
    *reinterpret_cast<float2*>(dst + 2 * lane) = make_float2(x0 / den * sc, x1 / den * sc);
  } else {
    const int hv = hh - 2 * a.Hk;
    float* dst = a.ve + (((int64_t)b * a.Hv + hv) * a.T + t) * DN_D;
    *reinterpret_cast<float2*>(dst + 2 * lane) = make_float2(x0, x1);
    if (lane == 0) {
      const uint16_t* ab = a.ab + (int64_t)b * a.ab_sb + (int64_t)t * a.ab_st;
      const int64_t g = ((int64_t)b * a.T + t) * a.Hv + hv;
      a.beta[g] = accurate_sigmoid(bf2f(ab[a.Hv + hv]));
      a.gate[g] = -expf(a.a_log[hv]) * log1pf(expf(bf2f(ab[hv]) + a.dt_bias[hv]));
    }
  }
}

// The same, vectorised for aligned operands (the conv output 16-byte aligned
// with strides of whole 8-element chunks, fp32 outputs 16-byte aligned; the
// launcher checks): one wave per token, four heads per pass (16 lanes of 8
// channels per head: 16-byte reads, 32-byte writes), the q / k sums of squares
// reduced over each 16-lane group, then lane l takes the gates of heads l, l + 64,
// ... The one-wave-per-(token, head) kernel above issued 64 times the waves
// for 4-byte reads, and ran at 2 TB/s.
__global__ __launch_bounds__(256) void deltanet_prep_vec_kernel(DeltaPrepArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t tok = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (tok >= (int64_t)a.B * a.T) return;
  const int b = (int)(tok / a.T), t = (int)(tok % a.T);
  const int nh = 2 * a.Hk + a.Hv, grp = lane >> 4, c = lane & 15;
  const uint16_t* row = a.cv + (int64_t)b * a.cv_sb + (int64_t)t * a.cv_st + 8 * c;
  const float qsc = 1.0f / sqrtf((float)DN_D);
  for (int h0 = 0; h0 < nh; h0 += 4) {
    const int hh = h0 + grp;  // uniform over the 16-lane group
    if (hh < nh) {
      float x[8];
      unpack8(*reinterpret_cast<const uint4*>(row + (int64_t)hh * DN_D), x);
      float* dst;
      float den = 1.0f, sc = 1.0f;
      if (hh < 2 * a.Hk) {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) ss += x[j] * x[j];
        ss += xor32<8>(ss);
        ss += xor32<4>(ss);
        ss += xor32<2>(ss);
        ss += xor32<1>(ss);
        den = sqrtf(ss + 1e-6f);
        const bool isq = hh < a.Hk;
        sc = isq ? qsc : 1.0f;
        dst = (isq ? a.qe : a.ke) + (((int64_t)b * a.Hk + (isq ? hh : hh - a.Hk)) * a.T + t) * DN_D;
      } else {
        dst = a.ve + (((int64_t)b * a.Hv + (hh - 2 * a.Hk)) * a.T + t) * DN_D;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = x[j] / den * sc;
      float4* d4 = reinterpret_cast<float4*>(dst + 8 * c);
      d4[0] = make_float4(x[0], x[1], x[2], x[3]);
      d4[1] = make_float4(x[4], x[5], x[6], x[7]);
    }
  }
  const uint16_t* ab = a.ab + (int64_t)b * a.ab_sb + (int64_t)t * a.ab_st;
  for (int hv = lane; hv < a.Hv; hv += 64) {
    const int64_t gi = ((int64_t)b * a.T + t) * a.Hv + hv;
    a.beta[gi] = accurate_sigmoid(bf2f(ab[a.Hv + hv]));
    a.gate[gi] = -expf(a.a_log[hv]) * log1pf(expf(bf2f(ab[hv]) + a.dt_bias[hv]));
  }
}

// ---- the prefill's epilogue (qwen35.jl:360-364): one wave per (head, token):
// y = o rstd norm_w silu(z) in bf16, written in the out projection's input
// layout (Dv, Hv, T, B).
__global__ __launch_bounds__(256) void gated_rms_norm_kernel(GatedNormArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t wid = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (wid >= (int64_t)a.B * a.T * a.Hv) return;
  const int hv = (int)(wid % a.Hv);
  const int64_t tok = wid / a.Hv;
  const int b = (int)(tok / a.T), t = (int)(tok % a.T);
  const float2 o = *reinterpret_cast<const float2*>(
      a.o + (((int64_t)b * a.Hv + hv) * a.T + t) * DN_D + 2 * lane);
  float ss = o.x * o.x + o.y * o.y;
  ss += __shfl_xor(ss, 32);
  ss = half_sum(ss);
  const float rstd = 1.0f / sqrtf(ss / (float)DN_D + a.eps);
  const uint16_t* z = a.z + (int64_t)b * a.z_sb + (int64_t)t * a.z_st + hv * DN_D + 2 * lane;
  const float w0 = bf2f(a.norm_w[2 * lane]), w1 = bf2f(a.norm_w[2 * lane + 1]);
  const float y0 = o.x * rstd * w0 * accurate_silu(bf2f(z[0]));
  const float y1 = o.y * rstd * w1 * accurate_silu(bf2f(z[1]));
  uint16_t* y = a.y + (int64_t)b * a.y_sb + (int64_t)t * a.y_st + hv * DN_D + 2 * lane;
  const uint32_t yp = pack2(y0, y1);
  y[0] = (uint16_t)yp;  // y may be 2-byte aligned
  y[1] = (uint16_t)(yp >> 16);
}

// The same, vectorised for aligned z and y (16-byte aligned, strides of whole
// 8-element chunks): one wave per token, four heads per pass (16 lanes of 8
// channels: 32-byte o reads, 16-byte z reads and y writes).
__global__ __launch_bounds__(256) void gated_rms_norm_vec_kernel(GatedNormArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t tok = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (tok >= (int64_t)a.B * a.T) return;
  const int b = (int)(tok / a.T), t = (int)(tok % a.T);
  const int grp = lane >> 4, c = lane & 15;
  float w[8];
  unpack8(*reinterpret_cast<const uint4*>(a.norm_w + 8 * c), w);
  for (int h0 = 0; h0 < a.Hv; h0 += 4) {
    const int hv = h0 + grp;
    if (hv < a.Hv) {
      const float4* op = reinterpret_cast<const float4*>(
          a.o + (((int64_t)b * a.Hv + hv) * a.T + t) * DN_D + 8 * c);
      const float4 o0 = op[0], o1 = op[1];
      const float o[8] = {o0.x, o0.y, o0.z, o0.w, o1.x, o1.y, o1.z, o1.w};
      float ss = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) ss += o[j] * o[j];
      ss += xor32<8>(ss);
      ss += xor32<4>(ss);
      ss += xor32<2>(ss);
      ss += xor32<1>(ss);
      const float rstd = 1.0f / sqrtf(ss / (float)DN_D + a.eps);
      float z[8], y[8];
      unpack8(*reinterpret_cast<const uint4*>(a.z + (int64_t)b * a.z_sb + (int64_t)t * a.z_st +
                                              hv * DN_D + 8 * c), z);
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = o[j] * rstd * w[j] * accurate_silu(z[j]);
      *reinterpret_cast<uint4*>(a.y + (int64_t)b * a.y_sb + (int64_t)t * a.y_st + hv * DN_D + 8 * c) =
          pack8(y);
    }
  }
}

// ---- causal_conv1d! (causal_conv1d.jl:7-61): one thread per 8 channels of one
// sequence. The ring's columns are all read before any is written, so the
// shifted ring may overwrite the one read (in place, as the reference runs it).
template <int K>
__global__ __launch_bounds__(256) void conv1d_update_kernel(Conv1dArgs a) {
  const int64_t c8 = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int b = blockIdx.y;
  if (c8 * 8 >= a.D) return;
  const int d = (int)c8 * 8;
  uint4 raw[K];
#pragma unroll
  for (int i = 0; i < K - 1; ++i)
    raw[i] = *reinterpret_cast<const uint4*>(a.s_in + b * a.s_sb + (int64_t)(i + 1) * a.s_cs + d);
  raw[K - 1] = *reinterpret_cast<const uint4*>(a.x + b * a.x_sb + d);
  float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < K; ++i) {
    float c[8], wf[8];
    unpack8(raw[i], c);
    unpack8(*reinterpret_cast<const uint4*>(a.w + (int64_t)i * a.w_cs + d), wf);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += c[e] * wf[e];
  }
#pragma unroll
  for (int i = 0; i < K; ++i)
    *reinterpret_cast<uint4*>(a.s_out + b * a.s_sb + (int64_t)i * a.s_cs + d) = raw[i];
  if (a.bias) {
    float bf8[8];
    unpack8(*reinterpret_cast<const uint4*>(a.bias + d), bf8);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += bf8[e];
  }
  if (a.act) {
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = accurate_silu(acc[e]);
  }
  *reinterpret_cast<uint4*>(a.y + b * a.y_sb + d) = pack8(acc);
}

// ---- linear! + causal_conv1d! (the decode step's in-projection and conv,
// qwen35.jl:212-223) from the projection's stream-K partials (gemv_sk_kernel,
// step.hip): thread = 8 channels of one sequence. Each thread adds its rows'
// partials in workgroup order, stores them rounded to bf16 as the projection's
// output (every channel: the conv's input, z, alpha, beta), and for the first
// D channels runs the conv step of conv1d_update_kernel on that bf16 input.
template <int K>
__global__ __launch_bounds__(256) void conv1d_update_sk_kernel(Conv1dSkArgs a) {
  const Conv1dArgs& c = a.c;
  const int64_t c8 = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int b = blockIdx.y;
  if (c8 * 8 >= a.M) return;
  const int d = (int)c8 * 8;
  const float4 lo = gemv_sk_sum4(a.part, a.G, a.chunk, d, b);
  const float4 hi = gemv_sk_sum4(a.part, a.G, a.chunk, d + 4, b);
  const float s8[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
  const uint4 xr = pack8(s8);
  *reinterpret_cast<uint4*>(a.yp + b * a.yp_sb + d) = xr;
  if (d >= c.D) return;
  uint4 raw[K];
#pragma unroll
  for (int i = 0; i < K - 1; ++i)
    raw[i] = *reinterpret_cast<const uint4*>(c.s_in + b * c.s_sb + (int64_t)(i + 1) * c.s_cs + d);
  raw[K - 1] = xr;
  float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < K; ++i) {
    float v[8], wf[8];
    unpack8(raw[i], v);
    unpack8(*reinterpret_cast<const uint4*>(c.w + (int64_t)i * c.w_cs + d), wf);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += v[e] * wf[e];
  }
#pragma unroll
  for (int i = 0; i < K; ++i)
    *reinterpret_cast<uint4*>(c.s_out + b * c.s_sb + (int64_t)i * c.s_cs + d) = raw[i];
  if (c.bias) {
    float bf8[8];
    unpack8(*reinterpret_cast<const uint4*>(c.bias + d), bf8);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += bf8[e];
  }
  if (c.act) {
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = accurate_silu(acc[e]);
  }
  *reinterpret_cast<uint4*>(c.y + b * c.y_sb + d) = pack8(acc);
}

// ---- causal_conv1d_sequence! (causal_conv1d.jl:73-149): thread = 8 channels x
// a run of CONV_TC tokens of one sequence, the window of the last K inputs in
// registers. The left context of token 0 is the ring's columns 2..K (s_in:
// the suffix prefill of qwen35.jl:333-344) or zeros. Only the threads of run 0
// read s_in (CONV_TC >= K - 1), and they also write the seeded ring (the last
// K inputs of the context-extended sequence) after reading, so s_out may alias
// s_in.
namespace {
template <int K>
__device__ __forceinline__ uint4 conv_ext(const Conv1dArgs& a, int b, int d, int t) {
  // ext(t), t in [-(K-1), T): x[t] for t >= 0, else ring column K + t (0-based)
  if (t >= 0) return *reinterpret_cast<const uint4*>(a.x + b * a.x_sb + (int64_t)t * a.x_st + d);
  if (a.s_in)
    return *reinterpret_cast<const uint4*>(a.s_in + b * a.s_sb + (int64_t)(K + t) * a.s_cs + d);
  return make_uint4(0, 0, 0, 0);
}
}  // namespace

template <int K>
__global__ __launch_bounds__(256) void conv1d_sequence_kernel(Conv1dArgs a) {
  static_assert(CONV_TC >= K - 1, "run 0 must cover the context reads");
  const int64_t c8 = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int run = blockIdx.y, b = blockIdx.z;
  if (c8 * 8 >= a.D) return;
  const int d = (int)c8 * 8;
  const int t0 = run * CONV_TC;
  const int t1 = min(t0 + CONV_TC, a.T);
  float wf[K][8];
#pragma unroll
  for (int i = 0; i < K; ++i)
    unpack8(*reinterpret_cast<const uint4*>(a.w + (int64_t)i * a.w_cs + d), wf[i]);
  float bias8[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (a.bias) unpack8(*reinterpret_cast<const uint4*>(a.bias + d), bias8);
  float win[K][8];  // win[i] = ext(t - K + 1 + i) for the current t
#pragma unroll
  for (int i = 0; i < K - 1; ++i) unpack8(conv_ext<K>(a, b, d, t0 - K + 1 + i), win[i]);
  for (int t = t0; t < t1; ++t) {
    unpack8(conv_ext<K>(a, b, d, t), win[K - 1]);
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float v = 0.f;
#pragma unroll
      for (int i = 0; i < K; ++i) v += win[i][e] * wf[i][e];
      v += bias8[e];
      acc[e] = a.act ? accurate_silu(v) : v;
    }
    *reinterpret_cast<uint4*>(a.y + b * a.y_sb + (int64_t)t * a.y_st + d) = pack8(acc);
#pragma unroll
    for (int i = 0; i + 1 < K; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) win[i][e] = win[i + 1][e];
  }
  if (run == 0 && a.s_out) {
    uint4 seed[K];  // column i = ext(T - K + i); every column read first (aliasing)
#pragma unroll
    for (int i = 0; i < K; ++i) seed[i] = conv_ext<K>(a, b, d, a.T - K + i);
#pragma unroll
    for (int i = 0; i < K; ++i)
      *reinterpret_cast<uint4*>(a.s_out + b * a.s_sb + (int64_t)i * a.s_cs + d) = seed[i];
  }
}

// ---- the prefill's conv and prep in one pass (qwen35.jl:333-356): thread = 8
// channels x a run of PREP_TC tokens (conv1d_sequence_kernel's form), the 16
// lanes of a head's 128 channels in one 16-lane group. Per token the conv
// output is rounded to bf16 (the value the two-kernel form stores between the
// kernels), then each q / k head row is scaled by its inverse L2 norm (q also
// by Dk^-1/2) over the group, and the row is written fp32 to Q / K / V, head
// major, as deltanet_prep_vec_kernel writes it: bit for bit the two-kernel
// result, without the conv output's round trip through memory. Workgroup column 0 also writes beta and the gate of its run's tokens.
// Bound by VALU issue (silu's exp and division are most of ~400 instructions per
// token and wave) beside 203 MB at T = 4096, so both are kept under way: the next
// K tokens' rows load while K are computed, the window turns through K fixed
// slots (no register moves), eight silus interleave, v skips the division and a
// row of q or k divides once. Runs of 8 tokens put 8 waves on a SIMD at T = 4096
// and 4 at 2000. B = 1, 8192 channels, T = 4096 / 2001: 66.5 / 41.0 -> 56.3 / 29.7
// us; runs of 16 as before 57.6 / 31.9, of 12 58.4 / 32.4; the shorter runs
// without the rest (9 tokens) 61.5 / 33.3. Runs of 8 against 16 over 2, 4 and 8 taps
// (8 re-read 7 rows of context a run), tokens B T: 16 to 64 10.5 to 12.1 against 17.7 to
// 19.4 us, 1024 17.1 to 20.3 against 20.7 to 23.5, 4096 43.0 / 47.4 / 56.6 against 44.3 / 48.0 /
// 56.6, 16384 199 / 205 / 230 against 199 / 200 / 226.
constexpr int PREP_TC = 8;

template <int K>
__global__ __launch_bounds__(256) void deltanet_conv_prep_kernel(ConvPrepArgs a) {
  static_assert(PREP_TC >= K - 1, "run 0 must cover the context reads");
  const Conv1dArgs& c = a.c;
  const DeltaPrepArgs& p = a.p;
  const int run = blockIdx.y, b = blockIdx.z;
  const int t0 = run * PREP_TC;
  const int t1 = min(t0 + PREP_TC, c.T);
  if (blockIdx.x == 0) {
    const uint16_t* ab = p.ab + (int64_t)b * p.ab_sb;
    for (int i = threadIdx.x; i < (t1 - t0) * p.Hv; i += 256) {
      const int t = t0 + i / p.Hv, hv = i % p.Hv;
      const int64_t gi = ((int64_t)b * p.T + t) * p.Hv + hv;
      p.beta[gi] = accurate_sigmoid(bf2f(ab[(int64_t)t * p.ab_st + p.Hv + hv]));
      p.gate[gi] = -expf(p.a_log[hv]) * log1pf(expf(bf2f(ab[(int64_t)t * p.ab_st + hv]) + p.dt_bias[hv]));
    }
  }
  const int64_t c8 = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c8 * 8 >= c.D) return;  // whole heads: a 16-lane group is all in or all out
  const int d = (int)c8 * 8;
  const int hh = d / DN_D, dc = d % DN_D;
  float* dst;  // this lane's 8 columns of head hh, token 0
  if (hh < p.Hk)
    dst = p.qe + ((int64_t)b * p.Hk + hh) * p.T * DN_D + dc;
  else if (hh < 2 * p.Hk)
    dst = p.ke + ((int64_t)b * p.Hk + hh - p.Hk) * p.T * DN_D + dc;
  else
    dst = p.ve + ((int64_t)b * p.Hv + hh - 2 * p.Hk) * p.T * DN_D + dc;
  const bool qk = hh < 2 * p.Hk;
  const float sc = hh < p.Hk ? 1.0f / sqrtf((float)DN_D) : 1.0f;
  float wf[K][8];
#pragma unroll
  for (int i = 0; i < K; ++i)
    unpack8(*reinterpret_cast<const uint4*>(c.w + (int64_t)i * c.w_cs + d), wf[i]);
  float bias8[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (c.bias) unpack8(*reinterpret_cast<const uint4*>(c.bias + d), bias8);
  float win[K][8];  // win[i] = ext(t - K + 1 + i) for the current t
#pragma unroll
  for (int i = 0; i < K - 1; ++i) unpack8(conv_ext<K>(c, b, d, t0 - K + 1 + i), win[i]);
  // the next block's K rows (past the run: its last row again, unused)
  const uint16_t* xr = c.x + b * c.x_sb + d;
  uint4 nx[K];
#pragma unroll
  for (int j = 0; j < K; ++j)
    nx[j] = *reinterpret_cast<const uint4*>(xr + (int64_t)min(t0 + j, t1 - 1) * c.x_st);
  for (int tb = t0; tb < t1; tb += K) {
    uint4 cur[K];
#pragma unroll
    for (int j = 0; j < K; ++j) cur[j] = nx[j];
    if (tb + K < t1) {
#pragma unroll
      for (int j = 0; j < K; ++j)
        nx[j] = *reinterpret_cast<const uint4*>(xr + (int64_t)min(tb + K + j, t1 - 1) * c.x_st);
    }
#pragma unroll
    for (int u = 0; u < K; ++u) {
      const int t = tb + u;
      if (t >= t1) break;
      unpack8(cur[u], win[(u + K - 1) % K]);  // ext(t - K + 1 + i) is in slot (u + i) % K
      float acc[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float v = 0.f;
#pragma unroll
        for (int i = 0; i < K; ++i) v += win[(u + i) % K][e] * wf[i][e];
        acc[e] = v + bias8[e];
      }
      if (c.act) {
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = accurate_silu(acc[e]);
      }
      float x[8];
      unpack8(pack8(acc), x);  // the conv output, bf16
      if (qk) {  // (v: the value itself)
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) ss += x[j] * x[j];
        ss += xor32<8>(ss);
        ss += xor32<4>(ss);
        ss += xor32<2>(ss);
        ss += xor32<1>(ss);
        const float den = sqrtf(ss + 1e-6f);
        if (den < INFINITY) {
          // x / den from the row's one reciprocal by Markstein's correction: y = x inv is
          // within an ulp, and the remainder x - y den, exact in an fma where |x| is
          // above 2^-102 (below that within 2^-150), brings it to the rounded quotient.
          // The remainder is formed negated, so that a zero keeps x's sign.
          const float inv = 1.0f / den;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float y = x[j] * inv;
            x[j] = fmaf(-fmaf(y, den, -x[j]), inv, y) * sc;
          }
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) x[j] = x[j] / den * sc;
        }
      }
      float4* d4 = reinterpret_cast<float4*>(dst + (int64_t)t * DN_D);
      d4[0] = make_float4(x[0], x[1], x[2], x[3]);
      d4[1] = make_float4(x[4], x[5], x[6], x[7]);
    }
  }
  if (run == 0 && c.s_out) {
    uint4 seed[K];  // column i = ext(T - K + i); every column read first (aliasing)
#pragma unroll
    for (int i = 0; i < K; ++i) seed[i] = conv_ext<K>(c, b, d, c.T - K + i);
#pragma unroll
    for (int i = 0; i < K; ++i)
      *reinterpret_cast<uint4*>(c.s_out + b * c.s_sb + (int64_t)i * c.s_cs + d) = seed[i];
  }
}

// ---- launchers -----------------------------------------------------------
hipError_t launch_deltanet_fused_decode(const DeltaFusedArgs& a, hipStream_t st) {
  if (a.B == 0) return hipSuccess;
  hipLaunchKernelGGL(deltanet_fused_decode_kernel, dim3(a.Hv, a.B), dim3(256), 0, st, a);
  return hipGetLastError();
}

#define VM_CONV_K_CASES(X) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8)

hipError_t launch_deltanet_decode_sk(const DeltaDecodeSkArgs& a, hipStream_t st) {
  if (a.f.B == 0) return hipSuccess;
  const int R = a.f.Hv / a.f.Hk;
  const dim3 grid(a.f.Hk, a.f.B);
#define DN_SK(kc, r) hipLaunchKernelGGL((deltanet_decode_sk_kernel<kc, r>), grid, dim3(256 * r), 0, st, a)
#define X(kc)                              \
  case kc:                                 \
    if (R == 1) DN_SK(kc, 1);              \
    else if (R == 2) DN_SK(kc, 2);         \
    else if (R == 4) DN_SK(kc, 4);         \
    else return hipErrorInvalidValue;      \
    break;
  switch (a.c.K) {
    VM_CONV_K_CASES(X)
    default: return hipErrorInvalidValue;
  }
#undef X
#undef DN_SK
  return hipGetLastError();
}

hipError_t launch_deltanet_sequence(const DeltaSeqArgs& a, hipStream_t st) {
  if (a.B == 0 || a.T == 0) {
    if (a.B > 0 && a.s_out != a.s_in)  // T = 0: the state passes through
      return hipMemcpyAsync(a.s_out, a.s_in, (size_t)a.B * a.Hv * DN_D * DN_D * sizeof(float),
                            hipMemcpyDeviceToDevice, st);
    return hipSuccess;
  }
  // few blocks (small B * Hv): 16 waves per head (NI = 4), else 4 (NI = 16)
  if ((int64_t)a.B * a.Hv >= 512) {
    hipLaunchKernelGGL(deltanet_sequence_kernel<16>, dim3(1, a.Hv, a.B), dim3(256), 0, st, a);
  } else {
    hipLaunchKernelGGL(deltanet_sequence_kernel<4>, dim3(4, a.Hv, a.B), dim3(256), 0, st, a);
  }
  return hipGetLastError();
}

size_t deltanet_chunk_workspace_bytes(int T, int Hv, int B) {
  // per (b, hv): the units, the K and Q units (Hk <= Hv) and the fused form's O
  const size_t NC = (T + DC - 1) / DC;
  return (NC * (UNIT + KQ_UNIT) + (size_t)T * DN_D) * Hv * B * sizeof(float);
}

// Up to this many tokens the sequential kernel is the faster form, by the scan's
// rounds (its 8 workgroups per value head and sequence, one on a CU at a time): the
// sequential kernel takes about 0.6 us a token up to 64 heads (B Hv) and from there
// on as well time in proportion to them, the two chunked launches the same for every
// T up to 64, one round after the other. Crossing points measured at 2 to 2048 heads,
// 1 to 4 value heads per qk head, 256 CUs: 35 to 38 tokens up to 32 heads (T = 36: 24.6 us
// sequential, 24.6 chunked), 43 at 48 and 64 (40: 27.2, 29.3; 48: 31.8, 29.6), 48 at 96 and 128
// (48: 38.6, 40.0), 52 at 144, 53 to 57 from 192 to 1024 (256 heads, 48: 52.1, 59.5; 56: 60.0,
// 60.1; 64: 66.7, 60.3), 60 and more beyond.
static int sequential_tokens(int64_t heads) {
  const int64_t cus = max(1, lm_head_waves() / 4);
  const int64_t rounds = (heads * (DN_D / CBW) + cus - 1) / cus;
  return (int)min((int64_t)54, 36 + 4 * (rounds - 1));
}
hipError_t launch_deltanet_sequence_chunked(const DeltaChunkArgs& args, hipStream_t st) {
  DeltaChunkArgs a = args;
  const DeltaSeqArgs& q = a.s;
  if (q.B == 0 || q.T == 0) return launch_deltanet_sequence(q, st);  // state copy / no-op
  const int NC = (q.T + DC - 1) / DC;
  if (a.g.y) {
    a.s.o = a.ws + (int64_t)q.B * NC * ((int64_t)q.Hv * UNIT + (int64_t)q.Hk * KQ_UNIT);
    a.g.o = a.s.o;
  }
  const int R = q.Hv / q.Hk;  // value heads per qk head, two a workgroup
  if (q.T <= sequential_tokens((int64_t)q.B * q.Hv)) {
    hipError_t e = launch_deltanet_sequence(a.s, st);
    if (e != hipSuccess || !a.g.y) return e;
    return launch_gated_rms_norm(a.g, st);
  }
  hipLaunchKernelGGL(deltanet_chunk_kernel, dim3(NC, q.Hk * ((R + 1) / 2), q.B), dim3(256), 0, st, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(deltanet_scan_kernel, dim3(q.Hv * q.B * (DN_D / CBW)), dim3(512), 0, st, a);
  e = hipGetLastError();
  if (e != hipSuccess || !a.g.y) return e;
  return launch_gated_rms_norm(a.g, st);
}

namespace {
bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
}  // namespace

hipError_t launch_deltanet_prep(const DeltaPrepArgs& a, hipStream_t st) {
  const int64_t toks = (int64_t)a.B * a.T;
  if (toks == 0) return hipSuccess;
  if (al16(a.cv) && a.cv_st % 8 == 0 && a.cv_sb % 8 == 0 && al16(a.qe) && al16(a.ke) && al16(a.ve)) {
    hipLaunchKernelGGL(deltanet_prep_vec_kernel, dim3((unsigned)((toks + 3) / 4)), dim3(256), 0, st, a);
  } else {
    const int64_t waves = toks * (2 * a.Hk + a.Hv);
    hipLaunchKernelGGL(deltanet_prep_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st, a);
  }
  return hipGetLastError();
}

hipError_t launch_gated_rms_norm(const GatedNormArgs& a, hipStream_t st) {
  const int64_t toks = (int64_t)a.B * a.T;
  if (toks == 0 || a.Hv == 0) return hipSuccess;
  if (al16(a.o) && al16(a.z) && al16(a.y) && al16(a.norm_w) && a.z_st % 8 == 0 && a.z_sb % 8 == 0 &&
      a.y_st % 8 == 0 && a.y_sb % 8 == 0) {
    hipLaunchKernelGGL(gated_rms_norm_vec_kernel, dim3((unsigned)((toks + 3) / 4)), dim3(256), 0, st, a);
  } else {
    const int64_t waves = toks * a.Hv;
    hipLaunchKernelGGL(gated_rms_norm_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st, a);
  }
  return hipGetLastError();
}


hipError_t launch_conv1d_update(const Conv1dArgs& a, hipStream_t st) {
  if (a.B == 0) return hipSuccess;
  const dim3 grid((unsigned)((a.D / 8 + 255) / 256), a.B);
  switch (a.K) {
#define X(k) \
  case k: hipLaunchKernelGGL(conv1d_update_kernel<k>, grid, dim3(256), 0, st, a); break;
    VM_CONV_K_CASES(X)
#undef X
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_conv1d_update_sk(const Conv1dSkArgs& a, hipStream_t st) {
  if (a.c.B == 0 || a.M == 0) return hipSuccess;
  const dim3 grid((unsigned)((a.M / 8 + 255) / 256), a.c.B);
  switch (a.c.K) {
#define X(k) \
  case k: hipLaunchKernelGGL(conv1d_update_sk_kernel<k>, grid, dim3(256), 0, st, a); break;
    VM_CONV_K_CASES(X)
#undef X
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_deltanet_conv_prep(const ConvPrepArgs& a, hipStream_t st) {
  if (a.c.B == 0 || a.c.T == 0) return hipSuccess;
  const int runs = (a.c.T + PREP_TC - 1) / PREP_TC;
  const dim3 grid((unsigned)((a.c.D / 8 + 255) / 256), runs, a.c.B);
  switch (a.c.K) {
#define X(k) \
  case k: hipLaunchKernelGGL(deltanet_conv_prep_kernel<k>, grid, dim3(256), 0, st, a); break;
    VM_CONV_K_CASES(X)
#undef X
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_conv1d_sequence(const Conv1dArgs& a, hipStream_t st) {
  if (a.B == 0 || a.T == 0) return hipSuccess;
  const int runs = (a.T + CONV_TC - 1) / CONV_TC;
  const dim3 grid((unsigned)((a.D / 8 + 255) / 256), runs, a.B);
  switch (a.K) {
#define X(k) \
  case k: hipLaunchKernelGGL(conv1d_sequence_kernel<k>, grid, dim3(256), 0, st, a); break;
    VM_CONV_K_CASES(X)
#undef X
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace vm
