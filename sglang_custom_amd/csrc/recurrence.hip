// Linear recurrences with one fp32 matrix per (sequence, head); the plain one:
//     S_t = diag(a_t) S_{t-1} + k_t v_t^T        S [dk, dv]
//     o_t = S_t^T (q_t * q_scale)
// a_t either per key channel and token, a = exp(logsigmoid(z + b) / tau) from gate logits z (fp32), or one number per head,
// or (state-space form) one number per head and token from a step size: dt = softplus(z_t[h] + dt_bias[h]),
// a_t = exp(-exp(rate_log[h]) dt), the write scaled by the same step, S_t = a_t S_{t-1} + dt k_t v_t^T, and a skip term
// skip[h] v_t added to the read-out.  q and k may have fewer heads than v (head h reads q / k head h / (heads / qk_heads)).
//
// One workgroup per (sequence of the step, head, block of 32 value columns): it loads the block's dk x 32 part of the
// sequence's matrix (zero at position 0), runs the step's tokens of that sequence through it in order, and stores it
// back.  A lane owns ONE column and R consecutive key channels of it in registers (8 lanes share a column, a wave holds 8
// columns, the 4 waves 32); per token it does R (mul, fma, fma) and the 8 partial dot products of a column meet over
// three lane exchanges.  q, k and the decays of the next TC tokens are staged in LDS (all fp32 from there on).  A decode
// step is the same launch with one token per sequence; what bounds it then is the matrix's trip through HBM, which each
// workgroup makes in whole 128-byte rows.
#include "common.cuh"

namespace mi355 {
namespace {

constexpr int RC_COLS = 32;   // value columns per workgroup
constexpr int RC_RG = 8;      // lanes that share a column
constexpr int RC_TC = 16;     // tokens staged at a time

__device__ __forceinline__ float log_sigmoid_f(float z) {
  // log(1 / (1 + exp(-z))) without overflow on either side
  return fminf(z, 0.f) - log1pf(expf(-fabsf(z)));
}

__device__ __forceinline__ float softplus_f(float z) { return z > 20.f ? z : log1pf(expf(z)); }

template <typename QT, typename VT, int R>
__global__ __launch_bounds__(256) void linear_recurrence_kernel(
    float* __restrict__ out, float* __restrict__ state, const QT* __restrict__ q, const QT* __restrict__ k,
    const VT* __restrict__ v, const float* __restrict__ gate_logits, const VT* __restrict__ gate_bias,
    const float* __restrict__ head_decay, const int32_t* __restrict__ req_to_state, const int64_t* __restrict__ req_pool_indices,
    const int32_t* __restrict__ seg_start, const int32_t* __restrict__ seg_len, const int64_t* __restrict__ positions, int heads,
    int dk, int dv, int64_t q_token_stride, int64_t k_token_stride, int64_t v_token_stride, int64_t gate_token_stride,
    float q_scale, float inv_tau, int qk_heads, const float* __restrict__ dt_logits, int64_t dt_token_stride,
    const float* __restrict__ dt_bias, const float* __restrict__ rate_log, const float* __restrict__ skip) {
  constexpr int DKP = R * RC_RG;     // key channels with padding
  __shared__ float dts[RC_TC], das[RC_TC];
  __shared__ __attribute__((aligned(16))) float qs[RC_TC][DKP];
  __shared__ __attribute__((aligned(16))) float ks[RC_TC][DKP];
  __shared__ __attribute__((aligned(16))) float as[RC_TC][DKP];
  __shared__ float vs[RC_TC][RC_COLS];
  const int b = blockIdx.z, h = blockIdx.y, c0 = blockIdx.x * RC_COLS;
  const int tid = threadIdx.x;
  const int rg = tid & (RC_RG - 1), cl = tid >> 3;       // lane = column * 8 + row group
  const int col = c0 + cl;
  const int64_t t0 = seg_start != nullptr ? seg_start[b] : b;
  const int n = seg_len != nullptr ? seg_len[b] : 1;
  if (n <= 0) return;
  const int64_t slot = req_to_state[req_pool_indices[b]];
  float* sp = state + ((slot * heads + h) * (int64_t)dk) * dv;
  float S[R];
  const bool fresh = positions[t0] == 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = rg * R + r;
    S[r] = (!fresh && i < dk && col < dv) ? sp[(int64_t)i * dv + col] : 0.f;
  }
  const float hd = head_decay != nullptr ? head_decay[h] : 1.f;
  const int hq = h / (heads / qk_heads);
  const float rate = dt_logits != nullptr ? expf(rate_log[h]) : 0.f;
  const float skip_h = skip != nullptr ? skip[h] : 0.f;
  for (int base = 0; base < n; base += RC_TC) {
    const int m = min(RC_TC, n - base);
    __syncthreads();
    if (dt_logits != nullptr) {
      if (tid < m) {
        const float dt = softplus_f(dt_logits[(t0 + base + tid) * dt_token_stride + h] + dt_bias[h]);
        dts[tid] = dt;
        das[tid] = expf(-rate * dt);
      }
      __syncthreads();
    }
    for (int e = tid; e < m * DKP; e += 256) {
      const int tt = e / DKP, i = e - tt * DKP;
      const int64_t t = t0 + base + tt;
      float qv = 0.f, kv = 0.f, av = 1.f;
      if (i < dk) {
        qv = to_f32(q[t * q_token_stride + (int64_t)hq * dk + i]) * q_scale;
        kv = to_f32(k[t * k_token_stride + (int64_t)hq * dk + i]);
        if (dt_logits != nullptr) {
          kv *= dts[tt];
          av = das[tt];
        } else if (gate_logits != nullptr) {
          float z = gate_logits[t * gate_token_stride + (int64_t)h * dk + i];
          if (gate_bias != nullptr) z += to_f32(gate_bias[(int64_t)h * dk + i]);
          av = expf(log_sigmoid_f(z) * inv_tau);
        } else {
          av = hd;
        }
      }
      qs[tt][i] = qv;
      ks[tt][i] = kv;
      as[tt][i] = av;
    }
    for (int e = tid; e < m * RC_COLS; e += 256) {
      const int tt = e / RC_COLS, c = e - tt * RC_COLS;
      vs[tt][c] = (c0 + c < dv) ? to_f32(v[(t0 + base + tt) * v_token_stride + (int64_t)h * dv + c0 + c]) : 0.f;
    }
    __syncthreads();
    for (int tt = 0; tt < m; ++tt) {
      const float vj = vs[tt][cl];
      float acc = 0.f;
#pragma unroll
      for (int r4 = 0; r4 < R; r4 += 4) {
        const float4 a4 = *reinterpret_cast<const float4*>(&as[tt][rg * R + r4]);
        const float4 k4 = *reinterpret_cast<const float4*>(&ks[tt][rg * R + r4]);
        const float4 q4 = *reinterpret_cast<const float4*>(&qs[tt][rg * R + r4]);
        S[r4 + 0] = fmaf(a4.x, S[r4 + 0], k4.x * vj);
        S[r4 + 1] = fmaf(a4.y, S[r4 + 1], k4.y * vj);
        S[r4 + 2] = fmaf(a4.z, S[r4 + 2], k4.z * vj);
        S[r4 + 3] = fmaf(a4.w, S[r4 + 3], k4.w * vj);
        acc = fmaf(S[r4 + 0], q4.x, acc);
        acc = fmaf(S[r4 + 1], q4.y, acc);
        acc = fmaf(S[r4 + 2], q4.z, acc);
        acc = fmaf(S[r4 + 3], q4.w, acc);
      }
      acc = group_sum<8>(acc);
      if (rg == 0 && col < dv) out[((t0 + base + tt) * heads + h) * (int64_t)dv + col] = fmaf(skip_h, vj, acc);
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = rg * R + r;
    if (i < dk && col < dv) sp[(int64_t)i * dv + col] = S[r];
  }
}

// ---- the recurrences with one decay per head and token over a step's many tokens, 64 of them at a time ------------------
// Inside a chunk the decays multiply out: with L_t the sum of their logarithms from the chunk's start to token t, the state at
// its start S0 and w_s = 1 (or the step size dt_s),
//     out_t = e^(L_t) S0^T q_t + sum_{s <= t} e^(L_t - L_s) (q_t . k_s) w_s u_s,     S <- e^(L_end) S0 + sum_s e^(L_end - L_s) w_s k_s u_s^T
// where u_s = v_s for the state-space form, and for the delta rule the solution of the unit lower triangular system
//     u_t + beta_t sum_{s < t} e^(L_t - L_s) (k_t . k_s) u_s = beta_t (v_t - e^(L_t) S0^T k_t).
// All of it is matrix products: the weights q . k and k . k and the state's update on the double matrix instruction, rounded once
// (their errors are the results' where decays are strong), everything else on the fp32 one; the triangular system is solved in
// blocks of 16 tokens with their inverses.  L is summed in double and
// kept as two floats, so that differences of long sums lose nothing.  Exponents are never positive.
// One workgroup of 8 waves per (sequence, head, 32 value columns), chunk after chunk; the next chunk's rows are on their way
// while one is multiplied, and where it pays what needs no state comes from a launch in front.  A token by token launch is a chain of LDS reads, multiply-adds and lane exchanges of 1000 (plain) and
// 1400 (delta) cycles a token, on one wave per SIMD: 4 x 1900 tokens, 16 heads of 64 x 128 took 800 and 1105 us; this took
// 214 and 342 in one launch (161 and 265 with every product in fp32, whose errors were 1.4 and 1.7 times the token by token form's at
// strong decays; now they are 0.6 to 1.0 times), takes 195 and 317 with the system solved in registers and the state in two buffers, and 148
// and 206 with the launch in front.  A chunk then takes its workgroup 4.0 and 5.2 us: 1.4 of them double products, 1.1 the outputs' products,
// the rest the rows' way through LDS and one or three barriers.
// What a later token of a chunk holds is multiplied by zero for an earlier one, which an infinity or a NaN survives.  They stay in
// the state, to the end: a sequence that ends with one in its state is done again token by token, so that non-finite
// inputs reach their own token's outputs and later ones only.  (The second run's code costs the delta rule's chunks 3 % through
// the compiler's schedule, 4 x 1000 tokens 178 -> 184 us; told that two waves a SIMD are all there will be, it costs the plain
// ones nothing.)
constexpr int CK = 64;               // tokens of a chunk, and key channels (padded)
constexpr int CLD = CK + 4;          // LDS row: the 16 rows of a 16-byte fragment read fall into different banks
constexpr int CK_THREADS = 512;

__device__ __forceinline__ f32x4 f4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ void mma4(f32x4& acc, const f32x4& a, const f32x4& b) {
#pragma unroll
  for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], acc, 0, 0, 0);
}
// sum_k A[i][k] B[j][k] over 64 of k; a, b: this lane's row li at k = 4 lg.  Four sums of 16 that meet in pairs: a chain of 64
// roundings shows in results that are little more than one such product.
__device__ __forceinline__ f32x4 tile_mma(const float* a, const float* b) {
  f32x4 p[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) p[k] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int k = 0; k < 4; ++k)
      p[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(f4(a + 16 * k)[j], f4(b + 16 * k)[j], p[k], 0, 0, 0);
  return (p[0] + p[1]) + (p[2] + p[3]);
}

// The same for weights, whose errors a strong decay leaves as the results': summed in double, rounded once.  The double instruction
// hands row 4 r + lg of its 16 to register r, so row i of A is loaded from row 4 (i & 3) + (i >> 2) of the tile: lane lg then holds
// rows 4 lg + r as in the fp32 layout.  a: the tile's first row, b: this lane's row, both at k = 0.
typedef double f64x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f32x4 tile_mma_exact(const float* a, const float* b, int li, int lg) {
  const float* ar = a + (4 * (li & 3) + (li >> 2)) * CLD + 4 * lg;
  const float* br = b + 4 * lg;
  f64x4 p = f64x4{0., 0., 0., 0.}, o = p;
#pragma unroll
  for (int k = 0; k < 4; k += 2) {
    const f32x4 a0 = f4(ar + 16 * k), b0 = f4(br + 16 * k), a1 = f4(ar + 16 * k + 16), b1 = f4(br + 16 * k + 16);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      p = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a0[j], (double)b0[j], p, 0, 0, 0);
      o = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a1[j], (double)b1[j], o, 0, 0, 0);
    }
  }
  p += o;
  return f32x4{(float)p[0], (float)p[1], (float)p[2], (float)p[3]};
}

struct ChunkArgs {
  float* out;
  float* state;
  const void* q;
  const void* k;
  const void* v;
  const float* logits;        // [tokens][heads] step-size (plain) or decay (delta) logits
  const float* bias;          // [heads]
  const float* rate_log;      // [heads]
  const float* skip;          // plain: [heads] or null
  const void* beta_logits;    // delta: [tokens][heads]
  const int32_t* req_to_state;
  const int64_t* req_pool_indices;
  const int32_t* seg_start;
  const int32_t* seg_len;
  const int64_t* positions;
  int64_t q_stride, k_stride, v_stride, logit_stride, beta_stride;
  int heads, qk_heads, dk, dv, beta_f32;
  float q_scale;
};

// A workgroup's sequence, head and columns token by token, 16 lanes a column, four channels each: for the rare sequences that the
// chunks do not serve.
typedef const ChunkArgs __attribute__((address_space(4))) ChunkArgsInMemory;
template <typename QT, typename VT, bool DELTA>
__device__ __forceinline__ void token_recurrence(ChunkArgsInMemory& p) {
  const int b = blockIdx.z, h = blockIdx.y, c = threadIdx.x >> 4, d0 = 4 * (threadIdx.x & 15), col = blockIdx.x * RC_COLS + c;
  const int hq = h / (p.heads / p.qk_heads);
  const int64_t t0 = p.seg_start[b], t1 = t0 + p.seg_len[b], slot = p.req_to_state[p.req_pool_indices[b]];
  float* const sp = p.state + ((slot * p.heads + h) * (int64_t)p.dk + d0) * p.dv + col;
  const float rate = expf(p.rate_log[h]), bias = p.bias[h], skip = !DELTA && p.skip != nullptr ? p.skip[h] : 0.f;
  const bool fresh = p.positions[t0] == 0, in_v = col < p.dv;
  float S[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) S[r] = !fresh && d0 + r < p.dk && in_v ? sp[(int64_t)r * p.dv] : 0.f;
  for (int64_t t = t0; t < t1; ++t) {
    const float v = in_v ? to_f32(((const VT*)p.v)[t * p.v_stride + (int64_t)h * p.dv + col]) : 0.f;
    const float dt = softplus_f(p.logits[t * p.logit_stride + h] + bias), decay = expf(-rate * dt);
    float k[4], y = 0.f, u = dt * v;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      k[r] = d0 + r < p.dk ? to_f32(((const QT*)p.k)[t * p.k_stride + (int64_t)hq * p.dk + d0 + r]) : 0.f;
      S[r] *= decay;
      y = fmaf(k[r], S[r], y);
    }
    if constexpr (DELTA) {
      y = group_sum<16>(y);
      const float z = p.beta_f32 ? static_cast<const float*>(p.beta_logits)[t * p.beta_stride + h]
                                 : to_f32(static_cast<const VT*>(p.beta_logits)[t * p.beta_stride + h]);
      u = (v - y) / (1.0f + expf(-z));
    }
    y = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (d0 + r < p.dk) {
        S[r] = fmaf(k[r], u, S[r]);
        y = fmaf(to_f32(((const QT*)p.q)[t * p.q_stride + (int64_t)hq * p.dk + d0 + r]) * p.q_scale, S[r], y);
      }
    y = group_sum<16>(y);
    if (d0 == 0 && in_v) p.out[(t * p.heads + h) * (int64_t)p.dv + col] = DELTA ? y : fmaf(skip, v, y);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (d0 + r < p.dk && in_v) sp[(int64_t)r * p.dv] = S[r];
}

// What a chunk's products take from its own tokens alone, in front of the serial launch: one record per (chunk, head), fragments as the
// lanes of a product hold them.  Floats: e^(L_t) [64], the state's weights e^(L_end - L_s) w_s [64], beta [64], 64 unused, ten tiles of M,
// and for the delta rule the system's six tiles under the diagonal ones and those ones' four inverses, tiles of [64 lanes][4].
constexpr int CK_M = 4 * CK, CK_A = CK_M + 10 * 256, CK_INV = CK_A + 6 * 256;
constexpr int chunk_record(bool delta) { return delta ? CK_INV + 4 * 256 : CK_A; }

// 64 tokens' decays, by one wave, a token a lane: L in two floats (null: not kept), e^L, the weights in the state, w
template <bool DELTA>
__device__ __forceinline__ void chunk_decays(float z, float beta_logit, float rate, float bias, int m, int lane, float* L0, float* L1, float* EL,
                                             float* WS, float* W) {
  const float sp_ = softplus_f(z + bias);
  float la = -rate * sp_;
  la = la < -1e4f ? -1e4f : la;      // e^-10000 is zero as well, and differences of sums stay finite
  if (lane >= m) la = 0.f;
  double sum = (double)la;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double up = __shfl_up(sum, o, 64);
    if (lane >= o) sum += up;
  }
  const double end = __shfl(sum, 63, 64);
  const float hi = (float)sum;
  L0[lane] = hi;
  L1[lane] = (float)(sum - (double)hi);
  EL[lane] = expf(hi);
  const float w = DELTA ? 1.0f / (1.0f + expf(-beta_logit)) : sp_;
  W[lane] = lane < m ? w : 0.f;
  WS[lane] = expf((float)(end - sum)) * (DELTA ? 1.f : lane < m ? w : 0.f);
}

// tile (ts, tt) of the weights, on or under the diagonal; lane holds s = 16 ts + 4 lg + r of token t = 16 tt + li: of u_s in out_t and
// (delta) of the system, its diagonal left out
template <bool DELTA>
__device__ __forceinline__ void chunk_weights(const float* Q, const float* K, const float* L0, const float* L1, const float* W, int tt, int ts, int li,
                                              int lg, f32x4& o, f32x4& sys) {
  const int t = tt * 16 + li, s = ts * 16 + 4 * lg;
  const f32x4 qk = tile_mma_exact(K + ts * 16 * CLD, Q + t * CLD, li, lg);
  const f32x4 l0 = f4(L0 + s), l1 = f4(L1 + s), w = f4(W + s);
  const float lt0 = L0[t], lt1 = L1[t];
  f32x4 a;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    a[r] = expf(fminf((lt0 - l0[r]) + (lt1 - l1[r]), 0.f));
    o[r] = s + r <= t ? qk[r] * a[r] * (DELTA ? 1.f : w[r]) : 0.f;
  }
  if constexpr (DELTA) {
    const f32x4 kk = tile_mma_exact(K + ts * 16 * CLD, K + t * CLD, li, lg);
    const float beta = W[t];
#pragma unroll
    for (int r = 0; r < 4; ++r) sys[r] = s + r < t ? kk[r] * a[r] * beta : 0.f;
  }
}

// the inverse of a unit lower triangular block of 16, a [16][ld] its strictly lower part: lane j < 16 has column j; to inv [16][20]
__device__ __forceinline__ void block_inverse(const float* a, int ld, float* inv, int lane) {
  float x[16];
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    float acc = lane == t ? 1.f : 0.f;
#pragma unroll
    for (int s4 = 0; s4 < t; s4 += 4) {
      const f32x4 av = f4(a + t * ld + s4);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (s4 + r < t) acc = fmaf(-av[r], x[s4 + r], acc);
    }
    x[t] = acc;
    inv[t * 20 + lane] = acc;
  }
}

__device__ __forceinline__ int chunks_of(int n) { return n > 0 ? (n + CK - 1) / CK : 0; }

// The records, a workgroup each, in no order: a column block's own workgroups of the serial launch each did this again, chunk after chunk.
// 1952 of them (4 x 1900 tokens, 16 heads, fp32 q and k) take 28 us, with the delta rule's system 47: 84 and 104 MB, and 10 (20) tiles of
// double products.
constexpr int CW_THREADS = 256;
template <typename QT, typename VT, bool DELTA>
__global__ __launch_bounds__(CW_THREADS) void chunk_weights_kernel(ChunkArgs p, float* records, int batch) {
  __shared__ __attribute__((aligned(16))) float Q[CK * CLD], K[CK * CLD], L0[CK], L1[CK], HEAD[3 * CK];
  __shared__ __attribute__((aligned(16))) float AD[DELTA ? 4 * 16 * 20 : 4], INV[DELTA ? 4 * 16 * 20 : 4];
  const int h = blockIdx.y, hq = h / (p.heads / p.qk_heads);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lg = lane >> 4;
  // the sequence that this chunk of the step belongs to: chunks are numbered through the sequences
  int64_t chunk = blockIdx.x;
  int b = -1, n = 0;
  for (int i0 = 0; i0 < batch; i0 += 64) {
    const int len = i0 + lane < batch ? p.seg_len[i0 + lane] : 0;
    int end = chunks_of(len);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int up = __shfl_up(end, o, 64);
      if (lane >= o) end += up;
    }
    const unsigned long long behind = __ballot((int64_t)end > chunk);
    if (behind != 0) {
      const int first = __ffsll(behind) - 1;
      b = i0 + first;
      n = __shfl(len, first, 64);
      chunk -= __shfl(end, first, 64) - chunks_of(n);
      break;
    }
    chunk -= __shfl(end, 63, 64);
  }
  if (b < 0) return;
  const int64_t t0 = p.seg_start[b] + chunk * CK;
  const int m = (int)min((int64_t)CK, n - chunk * CK);
  float* const rec = records + ((int64_t)blockIdx.x * p.heads + h) * chunk_record(DELTA);
  const QT* const qg = (const QT*)p.q;
  const QT* const kg = (const QT*)p.k;
  QT qr[16], kr[16];
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const int e = tid + CW_THREADS * u, t = min(e >> 6, m - 1), i = min(e & 63, p.dk - 1);
    qr[u] = qg[(t0 + t) * p.q_stride + (int64_t)hq * p.dk + i];
    kr[u] = kg[(t0 + t) * p.k_stride + (int64_t)hq * p.dk + i];
  }
  if (wave == 0) {
    const int64_t t = t0 + min(lane, m - 1);
    const float z = p.logits[t * p.logit_stride + h];
    float beta = 0.f;
    if (DELTA)
      beta = p.beta_f32 ? static_cast<const float*>(p.beta_logits)[t * p.beta_stride + h]
                        : to_f32(static_cast<const VT*>(p.beta_logits)[t * p.beta_stride + h]);
    chunk_decays<DELTA>(z, beta, expf(p.rate_log[h]), p.bias[h], m, lane, L0, L1, HEAD, HEAD + CK, HEAD + 2 * CK);
  }
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const int e = tid + CW_THREADS * u, t = e >> 6, i = e & 63;
    const bool in = t < m && i < p.dk;
    Q[t * CLD + i] = in ? to_f32(qr[u]) * p.q_scale : 0.f;
    K[t * CLD + i] = in ? to_f32(kr[u]) : 0.f;
  }
  __syncthreads();
  if (tid < 3 * CK) rec[tid] = HEAD[tid];
  for (int x = wave; x < 10; x += CW_THREADS / 64) {
    const int tt = x < 1 ? 0 : x < 3 ? 1 : x < 6 ? 2 : 3, ts = x - tt * (tt + 1) / 2;
    f32x4 o, sys;
    chunk_weights<DELTA>(Q, K, L0, L1, HEAD + 2 * CK, tt, ts, li, lg, o, sys);
    *reinterpret_cast<f32x4*>(rec + CK_M + x * 256 + 4 * lane) = o;
    if constexpr (DELTA) {
      if (tt == ts) *reinterpret_cast<f32x4*>(AD + (tt * 16 + li) * 20 + 4 * lg) = sys;
      else *reinterpret_cast<f32x4*>(rec + CK_A + (tt * (tt - 1) / 2 + ts) * 256 + 4 * lane) = sys;
    }
  }
  if constexpr (DELTA) {
    __syncthreads();
    if (lane < 16) block_inverse(AD + wave * 16 * 20, 20, INV + wave * 16 * 20, lane);
    __syncthreads();
    *reinterpret_cast<f32x4*>(rec + CK_INV + wave * 256 + 4 * lane) = f4(INV + (wave * 16 + li) * 20 + 4 * lg);
  }
}

// PREP: with chunk_weights_kernel's records for `chunks` of the step's chunks (a sequence that has more goes token by token)
template <typename QT, typename VT, bool DELTA, bool PREP>
__global__ __launch_bounds__(CK_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void chunk_recurrence_kernel(ChunkArgs p, const float* records, int64_t chunks) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr int REC = chunk_record(DELTA), RV = (REC / 4 + CK_THREADS - 1) / CK_THREADS;
  constexpr int BUF = 2 * CK * CLD + RC_COLS * CLD + REC;                 // PREP: a chunk's rows and record, twice
  float* const ST = lds;                                                  // [2][c][d] state
  float* Q = ST + 2 * RC_COLS * CLD;                                      // [t][d]
  float* K = Q + CK * CLD;                                                // [t][d]
  float* U = K + CK * CLD;                                                // [c][t] v, then the right-hand side, then u
  float* R = U + RC_COLS * CLD;                                           // PREP: the record, else its first three rows
  float* const L0 = R + 3 * CK;                                           // [t] L, upper part
  float* const L1 = L0 + CK;                                              // [t] lower part
  float* const M = L1 + CK;                                               // [t][s] weights of u_s in out_t
  float* const A = M + CK * CLD;                                          // delta: [t][s] strictly lower part of the system
  float* const INV = A + CK * CLD;                                        // delta: [4][16][20] inverses of its diagonal blocks
  __shared__ int not_finite;
  const int b = blockIdx.z, h = blockIdx.y, c0 = blockIdx.x * RC_COLS;
  const int hq = h / (p.heads / p.qk_heads);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lg = lane >> 4;
  const int64_t t0 = p.seg_start[b];
  const int n = p.seg_len[b];
  if (n <= 0) return;
  const float* rec = nullptr;
  bool served = true;
  if constexpr (PREP) {
    int before = 0;
    for (int i = lane; i < b; i += 64) before += chunks_of(p.seg_len[i]);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) before += __shfl_xor(before, o, 64);
    served = (int64_t)before + chunks_of(n) <= chunks;
    rec = records + ((int64_t)before * p.heads + h) * REC;
  }
  const int64_t slot = p.req_to_state[p.req_pool_indices[b]];
  float* const sp = p.state + ((slot * p.heads + h) * (int64_t)p.dk) * p.dv;
  const bool fresh = p.positions[t0] == 0;
  const float rate = expf(p.rate_log[h]), bias = p.bias[h];
  const float skip = !DELTA && p.skip != nullptr ? p.skip[h] : 0.f;
  const QT* const qg = (const QT*)p.q;
  const QT* const kg = (const QT*)p.k;
  const VT* const vg = (const VT*)p.v;

#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int e = tid + CK_THREADS * u, i = e >> 5, c = e & 31;
    ST[c * CLD + i] = (!fresh && i < p.dk && c0 + c < p.dv) ? sp[(int64_t)i * p.dv + c0 + c] : 0.f;
  }
  if (tid == 0) not_finite = !served;
  // this wave's tile of the state: d = 16 (wave >> 1) + 4 lg + r, column 16 (wave & 1) + li
  const int sd = (wave >> 1) * 16, sc = (wave & 1) * 16;

  // the next chunk's elements: tokens 8 wave + u of q and of k, channel lane; 4 of v, tokens 4 (tid >> 5) + u; one logit (or two)
  QT qr[8], kr[8];
  VT vr[4];
  float zr = 0.f, br = 0.f;
  f32x4 rr[RV];
  auto request = [&](int base) {
    const int m = n - base;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int t = min(8 * wave + u, m - 1), i = min(lane, p.dk - 1);
      qr[u] = qg[(t0 + base + t) * p.q_stride + (int64_t)hq * p.dk + i];
      kr[u] = kg[(t0 + base + t) * p.k_stride + (int64_t)hq * p.dk + i];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = min(4 * (tid >> 5) + u, m - 1), c = min(c0 + (tid & 31), p.dv - 1);
      vr[u] = vg[(t0 + base + t) * p.v_stride + (int64_t)h * p.dv + c];
    }
    if constexpr (PREP) {
      const float* const src = rec + (int64_t)(base / CK) * p.heads * REC;
#pragma unroll
      for (int u = 0; u < RV; ++u) rr[u] = f4(src + 4 * min(tid + CK_THREADS * u, REC / 4 - 1));
    } else if (tid < 64) {
      const int64_t t = t0 + base + min(tid, m - 1);
      zr = p.logits[t * p.logit_stride + h];
      if (DELTA)
        br = p.beta_f32 ? static_cast<const float*>(p.beta_logits)[t * p.beta_stride + h]
                        : to_f32(static_cast<const VT*>(p.beta_logits)[t * p.beta_stride + h]);
    }
  };
  auto stage = [&](int base) {
    const int m = n - base;
    f32x4 v4;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int t = 8 * wave + u;
      const bool in = t < m && lane < p.dk;
      Q[t * CLD + lane] = in ? to_f32(qr[u]) * p.q_scale : 0.f;
      K[t * CLD + lane] = in ? to_f32(kr[u]) : 0.f;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) v4[u] = 4 * (tid >> 5) + u < m && c0 + (tid & 31) < p.dv ? to_f32(vr[u]) : 0.f;
    *reinterpret_cast<f32x4*>(U + (tid & 31) * CLD + 4 * (tid >> 5)) = v4;
    if constexpr (PREP) {
#pragma unroll
      for (int u = 0; u < RV; ++u)
        if (tid + CK_THREADS * u < REC / 4) *reinterpret_cast<f32x4*>(R + 4 * (tid + CK_THREADS * u)) = rr[u];
    } else if (tid < 64) {
      chunk_decays<DELTA>(zr, br, rate, bias, m, lane, L0, L1, R, R + CK, R + 2 * CK);
    }
  };
  auto other_buffer = [&](int cur) { Q += cur ? -BUF : BUF, K += cur ? -BUF : BUF, U += cur ? -BUF : BUF, R += cur ? -BUF : BUF; };
  const int last_base = (n - 1) / CK * CK;
  if (served) {
    request(0);
    stage(0);
    request(min(CK, last_base));
  }
  __syncthreads();

  int cur = 0;
  for (int base = 0; served && base < n; base += CK, cur ^= 1) {
    const int m = min(CK, n - base);
    const float* const EL = R;                    // [t] e^(L_t)
    const float* const WS = EL + CK;              // [s] e^(L_end - L_s) w_s
    const float* const W = WS + CK;               // [s] w_s (plain) or beta_t (delta)
    const float* const S0 = ST + cur * RC_COLS * CLD;
    const float el_end = EL[CK - 1];

    if constexpr (!PREP) {
      for (int x = wave; x < 10; x += 8) {
        const int tt = x < 1 ? 0 : x < 3 ? 1 : x < 6 ? 2 : 3, ts = x - tt * (tt + 1) / 2;
        f32x4 o, sys;
        chunk_weights<DELTA>(Q, K, L0, L1, W, tt, ts, li, lg, o, sys);
        *reinterpret_cast<f32x4*>(M + (tt * 16 + li) * CLD + ts * 16 + 4 * lg) = o;
        if constexpr (DELTA) *reinterpret_cast<f32x4*>(A + (tt * 16 + li) * CLD + ts * 16 + 4 * lg) = sys;
      }
    }
    auto weights = [&](int tt, int s) { return PREP ? f4(R + CK_M + (tt * (tt + 1) / 2 + s) * 256 + 4 * lane) : f4(M + (tt * 16 + li) * CLD + s * 16 + 4 * lg); };
    // what the state's start has in the outputs: wave takes column tile wave & 1 of token tile wave >> 1; lane holds columns 4 lg + r of
    // token li of the tile.  (The six waves that solve nothing take it while the other two do.)
    f32x4 from_state;
    auto start_of_out = [&] { from_state = tile_mma(S0 + (sc + li) * CLD + 4 * lg, Q + (sd + li) * CLD + 4 * lg) * EL[sd + li]; };
    if (!DELTA || wave < 2) start_of_out();
    if constexpr (DELTA) {
      // right-hand side: lane holds tokens t = 16 (wave >> 1) + 4 lg + r of column 16 (wave & 1) + li
      const f32x4 y = tile_mma(K + (sd + li) * CLD + 4 * lg, S0 + (sc + li) * CLD + 4 * lg);
      float* const up = U + (sc + li) * CLD + sd + 4 * lg;
      const f32x4 vv = f4(up), el = f4(EL + sd + 4 * lg), be = f4(W + sd + 4 * lg);
      f32x4 o;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = be[r] * (vv[r] - el[r] * y[r]);
      *reinterpret_cast<f32x4*>(up) = o;
      __syncthreads();
      if constexpr (!PREP) {
        // inverses of the four diagonal blocks
        if (wave < 4 && lane < 16) block_inverse(A + (wave * 16) * CLD + wave * 16, CLD, INV + wave * 16 * 20, lane);
        __syncthreads();
      }
      // two waves, 16 columns each: block by block, what the earlier blocks take off and the diagonal block's inverse.  lane: tokens
      // 16 blk + 4 lg + r of column li, which is also a B row's k, so that a solved block goes on from the registers
      if (wave < 2) {
        float* const uc = U + (wave * 16 + li) * CLD + 4 * lg;
        f32x4 off[4], rhs[4], inv[4], a[6];
#pragma unroll
        for (int blk = 0; blk < 4; ++blk) {
          off[blk] = f32x4{0.f, 0.f, 0.f, 0.f};
          rhs[blk] = f4(uc + blk * 16);
          inv[blk] = PREP ? f4(R + CK_INV + blk * 256 + 4 * lane) : f4(INV + (blk * 16 + li) * 20 + 4 * lg);
#pragma unroll
          for (int s = 0; s < blk; ++s)
            a[blk * (blk - 1) / 2 + s] = PREP ? f4(R + CK_A + (blk * (blk - 1) / 2 + s) * 256 + 4 * lane) : f4(A + (blk * 16 + li) * CLD + s * 16 + 4 * lg);
        }
#pragma unroll
        for (int blk = 0; blk < 4; ++blk) {
          f32x4 x = f32x4{0.f, 0.f, 0.f, 0.f};
          mma4(x, inv[blk], rhs[blk] - off[blk]);
          *reinterpret_cast<f32x4*>(uc + blk * 16) = x;
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int to = blk + 1; to < 4; ++to)
              off[to] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[to * (to - 1) / 2 + blk][j], x[j], off[to], 0, 0, 0);
        }
      } else {
        start_of_out();
      }
    }
    if (DELTA || !PREP) __syncthreads();
    f32x4 us[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) us[s] = f4(U + (sc + li) * CLD + s * 16 + 4 * lg);
    // state, in double like the weights: the sum over 64 tokens rounds once
    f64x4 p64 = f64x4{0., 0., 0., 0.}, q64 = p64;
    const float* const kt = K + 4 * lg * CLD + sd + 4 * (li & 3) + (li >> 2);
#pragma unroll
    for (int s = 0; s < 4; s += 2) {
      f32x4 k0, k1;
#pragma unroll
      for (int j = 0; j < 4; ++j) k0[j] = kt[(s * 16 + j) * CLD], k1[j] = kt[(s * 16 + 16 + j) * CLD];
      const f32x4 w0 = f4(WS + s * 16 + 4 * lg), w1 = f4(WS + s * 16 + 16 + 4 * lg);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        p64 = __builtin_amdgcn_mfma_f64_16x16x4f64((double)k0[j], (double)us[s][j] * (double)w0[j], p64, 0, 0, 0);
        q64 = __builtin_amdgcn_mfma_f64_16x16x4f64((double)k1[j], (double)us[s + 1][j] * (double)w1[j], q64, 0, 0, 0);
      }
    }
    f32x4 S = f4(S0 + (sc + li) * CLD + sd + 4 * lg);
#pragma unroll
    for (int r = 0; r < 4; ++r) S[r] = (float)((double)S[r] * (double)el_end + (p64[r] + q64[r]));
    *reinterpret_cast<f32x4*>(ST + (cur ^ 1) * RC_COLS * CLD + (sc + li) * CLD + sd + 4 * lg) = S;
    // outputs
    const int t = sd + li;
    f32x4 acc = from_state;
    auto add = [&](auto tiles) {
      constexpr int N = decltype(tiles)::value;
      f32x4 part[N], ws[N];
#pragma unroll
      for (int s = 0; s < N; ++s) {
        part[s] = f32x4{0.f, 0.f, 0.f, 0.f};
        ws[s] = weights(N - 1, s);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int s = 0; s < N; ++s) part[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(us[s][j], ws[s][j], part[s], 0, 0, 0);
#pragma unroll
      for (int s = 0; s < N; ++s) acc += part[s];
    };
    switch (wave >> 1) {
      case 0: add(std::integral_constant<int, 1>{}); break;
      case 1: add(std::integral_constant<int, 2>{}); break;
      case 2: add(std::integral_constant<int, 3>{}); break;
      default: add(std::integral_constant<int, 4>{});
    }
    if constexpr (!DELTA) {
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] = fmaf(skip, U[(sc + 4 * lg + r) * CLD + t], acc[r]);
    }
    if constexpr (PREP) {
      // the next chunk's rows into the other buffer, the ones behind it from memory (at the end the last ones again: no branch).  In front of
      // the stores, for whose end a use of those rows would wait as well
      other_buffer(cur);
      stage(base + CK);
      request(min(base + 2 * CK, last_base));
    }
    if (t < m) {
      float* const o = p.out + ((t0 + base + t) * p.heads + h) * (int64_t)p.dv + c0 + sc + 4 * lg;
      if (p.dv % 4 == 0 && c0 + sc + 4 * lg + 4 <= p.dv) {
        *reinterpret_cast<f32x4*>(o) = acc;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (c0 + sc + 4 * lg + r < p.dv) o[r] = acc[r];
      }
    }
    if (!PREP && base + CK < n) {
      __syncthreads();
      stage(base + CK);
      request(min(base + 2 * CK, last_base));
    }
    __syncthreads();
  }
  float last[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int e = tid + CK_THREADS * u, i = e >> 5, c = e & 31;
    last[u] = ST[cur * RC_COLS * CLD + c * CLD + i];
    if (!isfinite(last[u])) not_finite = 1;
  }
  __syncthreads();
  if (!not_finite) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = tid + CK_THREADS * u, i = e >> 5, c = e & 31;
      if (i < p.dk && c0 + c < p.dv) sp[(int64_t)i * p.dv + c0 + c] = last[u];
    }
    return;
  }
  // (this workgroup's part of the state in memory is still the one that it began with.  The arguments are read afresh: kept in
  // registers through the chunks they would make those slower)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // every output above is written before the ones of the second run
  __syncthreads();
  ChunkArgsInMemory* args = (ChunkArgsInMemory*)__builtin_amdgcn_kernarg_segment_ptr();
  asm("" : "+s"(args));
  token_recurrence<QT, VT, DELTA>(*args);
}

// Which launches take the chunks: one decay per head and token, at most 64 key channels (what the LDS tiles hold), a step whose
// sequences have segments, of known lengths (tokens in all, the longest one), and less time by the two forms' models, which fit what
// was measured within 15 % (16 heads of 64 x 128, in us).  A token of the token-by-token form takes a chain of 0.40 (delta 0.55)
// or, from some 1000 workgroups on, its share of the chip, 0.43 (0.60) per 1000 of them; a chunk takes its workgroup 6.7 (10.6), one
// workgroup to a CU, and about 3 more before the first.  That is the price of chunks in one launch as they first were: with the state in two
// buffers they take a tenth less, behind records 4.0 (5.2), so where the rule takes chunks they are ahead by more, and many middling prompts
// that it leaves token by token (64 x 500) may be faster in chunks behind records; the lines have not been measured again.  Measured, token
// by token / chunks in that first form:
//   plain  1 x 16   9.8 / 10.4   1 x 64   27 / 11     8 x 65   32 / 35    16 x 64    42 / 42    64 x 4    27 / 149   64 x 500   813 / 905
//   delta  1 x 16  12.4 / 14.9   1 x 64   38 / 16     8 x 65   43 / 51    16 x 64    54 / 58    64 x 4    27 / 213   64 x 500  1096 / 1409
//   plain  4 x 2000   827 / 223   16 x 1000   464 / 440   16 x 2000   1010 / 865;   delta   1130 / 348   667 / 691   1369 / 1372
inline bool chunks_pay(bool delta, int64_t batch, int heads, int dk, int dv, int64_t tokens, int64_t longest) {
  if (dk > CK || tokens <= 0 || longest <= 0 || batch <= 0) return false;
  const double blocks = (double)heads * cdiv(dv, RC_COLS);                  // workgroups of a sequence
  const double narrow = dk <= 32 ? 0.8 : 1.0;                               // (a token's cost follows its channels, a chunk's does not)
  const double chain = narrow * (delta ? 0.55 : 0.40), share = narrow * (delta ? 0.60e-3 : 0.43e-3), chunk = delta ? 10.6 : 6.7;
  const double by_token = 5 + std::max(chain * longest, share * tokens * blocks);
  const double most = (double)cdiv(longest, CK);
  const double chunks = std::min(batch * most, tokens / (double)CK + batch);   // of one head's columns, over all sequences
  const double rounds = std::ceil(batch * blocks / 256);
  return 3 + std::max(chunk * most + 3, rounds * (chunk * chunks / batch + 3)) < 0.97 * by_token;
}

inline bool chunks_serve(bool delta, int64_t batch, int heads, int dk, int dv, int64_t tokens, int64_t longest, const int32_t* seg_len,
                         const float* out) {
  return seg_len != nullptr && (dv % 4 != 0 || aligned16(out)) && chunks_pay(delta, batch, heads, dk, dv, tokens, longest);
}

// Which of them have records made in front: a chunk behind that costs its workgroup 2.6 us less (delta 5.2), the launch and the first record
// 8 (10), and 1000 records 14 (24).  Measured, without / with (16 heads of 64 x 128):
//   plain  1 x 130  23 / 24   1 x 256  30 / 28   4 x 256  32 / 34   1 x 1000  104 / 74   4 x 1900  195 / 148
//   delta  1 x 130  37 / 32   4 x 130  37 / 35   4 x 256  49 / 46   1 x 1000  174 / 97   4 x 1900  317 / 206
inline int64_t chunk_records_bytes(bool delta, int64_t batch, int heads, int dk, int dv, int64_t tokens, int64_t longest) {
  if (!chunks_pay(delta, batch, heads, dk, dv, tokens, longest)) return 0;
  const double most = (double)cdiv(longest, CK), chunks = std::min(batch * most, tokens / (double)CK + batch);
  const double rounds = std::ceil(batch * (double)heads * cdiv(dv, RC_COLS) / 256);
  if ((delta ? 5.2 : 2.6) * std::max(most, rounds * chunks / batch) < (delta ? 10 : 8) + (delta ? 0.024 : 0.014) * chunks * heads) return 0;
  const int64_t bytes = (tokens / CK + batch) * heads * (int64_t)sizeof(float) * chunk_record(delta);
  return bytes <= ((int64_t)1 << 30) ? bytes : 0;
}

template <typename QT, typename VT, bool DELTA>
int launch_chunks(const ChunkArgs& p, int64_t batch, int64_t tokens, int64_t longest, float* records, int64_t bytes, hipStream_t st) {
  const dim3 grid((unsigned)cdiv(p.dv, RC_COLS), (unsigned)p.heads, (unsigned)batch);
  const int64_t need = chunk_records_bytes(DELTA, batch, p.heads, p.dk, p.dv, tokens, longest), chunks = tokens / CK + batch;
  if (records != nullptr && need > 0 && bytes >= need && aligned16(records)) {
    constexpr size_t lds = sizeof(float) * (2 * RC_COLS * CLD + 2 * (2 * CK * CLD + RC_COLS * CLD + chunk_record(DELTA)));
    auto kern = chunk_recurrence_kernel<QT, VT, DELTA, true>;
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL((chunk_weights_kernel<QT, VT, DELTA>), dim3((unsigned)chunks, (unsigned)p.heads), dim3(CW_THREADS), 0, st, p, records, (int)batch);
    hipLaunchKernelGGL(kern, grid, dim3(CK_THREADS), lds, st, p, records, chunks);
    return MI355_OK;
  }
  constexpr size_t lds = sizeof(float) * (3 * RC_COLS * CLD + 3 * CK * CLD + 5 * CK + (DELTA ? CK * CLD + 4 * 16 * 20 : 0));
  auto kern = chunk_recurrence_kernel<QT, VT, DELTA, false>;
  (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL(kern, grid, dim3(CK_THREADS), lds, st, p, (const float*)nullptr, (int64_t)0);
  return MI355_OK;
}

template <typename QT, typename VT>
int launch_recurrence(float* out, float* state, const void* q, const void* k, const void* v, const float* gate_logits,
                      const void* gate_bias, const float* head_decay, const int32_t* req_to_state, const int64_t* req_pool_indices,
                      const int32_t* seg_start, const int32_t* seg_len, const int64_t* positions, int64_t batch, int heads, int dk,
                      int dv, int64_t qs, int64_t ks, int64_t vs, int64_t gs, float q_scale, float tau, int qk_heads, const float* dt_logits,
                      int64_t dts, const float* dt_bias, const float* rate_log, const float* skip, int64_t tokens, int64_t longest,
                      float* records, int64_t record_bytes, hipStream_t stream) {
  if (dt_logits != nullptr && chunks_serve(false, batch, heads, dk, dv, tokens, longest, seg_len, out)) {
    const ChunkArgs p{out, state, q, k, v, dt_logits, dt_bias, rate_log, skip, nullptr, req_to_state, req_pool_indices, seg_start, seg_len,
                      positions, qs, ks, vs, dts, 0, heads, qk_heads, dk, dv, 0, q_scale};
    return launch_chunks<QT, VT, false>(p, batch, tokens, longest, records, record_bytes, stream);
  }
  const dim3 grid((unsigned)cdiv(dv, RC_COLS), (unsigned)heads, (unsigned)batch);
#define MI355_RC_LAUNCH(R)                                                                                                     \
  hipLaunchKernelGGL((linear_recurrence_kernel<QT, VT, R>), grid, dim3(256), 0, stream, out, state, (const QT*)q, (const QT*)k, \
                     (const VT*)v, gate_logits, (const VT*)gate_bias, head_decay, req_to_state, req_pool_indices, seg_start,   \
                     seg_len, positions, heads, dk, dv, qs, ks, vs, gs, q_scale, 1.0f / tau, qk_heads, dt_logits, dts, dt_bias,  \
                     rate_log, skip)
  if (dk <= 32) MI355_RC_LAUNCH(4);
  else if (dk <= 64) MI355_RC_LAUNCH(8);
  else if (dk <= 128) MI355_RC_LAUNCH(16);
  else MI355_RC_LAUNCH(32);
#undef MI355_RC_LAUNCH
  return MI355_OK;
}


// Gated delta rule on the same layout: per token
//     S <- diag(a_t) S;   u = beta_t (v_t - S^T k_t);   S <- S + k_t u^T;   o_t = S^T (q_t * q_scale)
// with a_t[i] = exp(-exp(rate_log[h]) * softplus(z_t[h, i] + rate_bias[h, i])) from fp32 logits z and beta_t = sigmoid of a
// logit per head.  With gate_per_head the decay is one number per head and token: z_t[h], rate_bias[h].  beta logits come
// in v's type or (beta_f32) in fp32.  q and k may have fewer heads than v (head h reads q / k head h / (heads / qk_heads)).  A column's
// S^T k and S^T q are each a sum over its eight lanes, so a token costs two rounds of lane exchanges.
template <typename QT, typename VT, int R>
__global__ __launch_bounds__(256) void gated_delta_rule_kernel(
    float* __restrict__ out, float* __restrict__ state, const QT* __restrict__ q, const QT* __restrict__ k,
    const VT* __restrict__ v, const VT* __restrict__ beta_logits, const float* __restrict__ gate_logits,
    const float* __restrict__ rate_bias, const float* __restrict__ rate_log, const int32_t* __restrict__ req_to_state,
    const int64_t* __restrict__ req_pool_indices, const int32_t* __restrict__ seg_start, const int32_t* __restrict__ seg_len,
    const int64_t* __restrict__ positions, int heads, int qk_heads, int dk, int dv, int64_t q_token_stride, int64_t k_token_stride,
    int64_t v_token_stride, int64_t beta_token_stride, int64_t gate_token_stride, float q_scale, int gate_per_head, int beta_f32) {
  constexpr int DKP = R * RC_RG;
  __shared__ __attribute__((aligned(16))) float qs[RC_TC][DKP];
  __shared__ __attribute__((aligned(16))) float ks[RC_TC][DKP];
  __shared__ __attribute__((aligned(16))) float as[RC_TC][DKP];
  __shared__ float vs[RC_TC][RC_COLS];
  __shared__ float bs[RC_TC];
  const int b = blockIdx.z, h = blockIdx.y, c0 = blockIdx.x * RC_COLS;
  const int hq = h / (heads / qk_heads);
  const int tid = threadIdx.x;
  const int rg = tid & (RC_RG - 1), cl = tid >> 3;
  const int col = c0 + cl;
  const int64_t t0 = seg_start != nullptr ? seg_start[b] : b;
  const int n = seg_len != nullptr ? seg_len[b] : 1;
  if (n <= 0) return;
  const int64_t slot = req_to_state[req_pool_indices[b]];
  float* sp = state + ((slot * heads + h) * (int64_t)dk) * dv;
  float S[R];
  const bool fresh = positions[t0] == 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = rg * R + r;
    S[r] = (!fresh && i < dk && col < dv) ? sp[(int64_t)i * dv + col] : 0.f;
  }
  const float rate = expf(rate_log[h]);
  for (int base = 0; base < n; base += RC_TC) {
    const int m = min(RC_TC, n - base);
    __syncthreads();
    for (int e = tid; e < m * DKP; e += 256) {
      const int tt = e / DKP, i = e - tt * DKP;
      const int64_t t = t0 + base + tt;
      float qv = 0.f, kv = 0.f, av = 1.f;
      if (i < dk) {
        qv = to_f32(q[t * q_token_stride + (int64_t)hq * dk + i]) * q_scale;
        kv = to_f32(k[t * k_token_stride + (int64_t)hq * dk + i]);
        const int64_t gi = gate_per_head ? h : (int64_t)h * dk + i;
        const float z = gate_logits[t * gate_token_stride + gi] + rate_bias[gi];
        av = expf(-rate * softplus_f(z));
      }
      qs[tt][i] = qv;
      ks[tt][i] = kv;
      as[tt][i] = av;
    }
    for (int e = tid; e < m * RC_COLS; e += 256) {
      const int tt = e / RC_COLS, c = e - tt * RC_COLS;
      vs[tt][c] = (c0 + c < dv) ? to_f32(v[(t0 + base + tt) * v_token_stride + (int64_t)h * dv + c0 + c]) : 0.f;
    }
    if (tid < m) {
      const int64_t bi = (t0 + base + tid) * beta_token_stride + h;
      const float bl = beta_f32 ? reinterpret_cast<const float*>(beta_logits)[bi] : to_f32(beta_logits[bi]);
      bs[tid] = 1.0f / (1.0f + expf(-bl));
    }
    __syncthreads();
    for (int tt = 0; tt < m; ++tt) {
      float dot = 0.f;
#pragma unroll
      for (int r4 = 0; r4 < R; r4 += 4) {
        const float4 a4 = *reinterpret_cast<const float4*>(&as[tt][rg * R + r4]);
        const float4 k4 = *reinterpret_cast<const float4*>(&ks[tt][rg * R + r4]);
        S[r4 + 0] *= a4.x;
        S[r4 + 1] *= a4.y;
        S[r4 + 2] *= a4.z;
        S[r4 + 3] *= a4.w;
        dot = fmaf(S[r4 + 0], k4.x, dot);
        dot = fmaf(S[r4 + 1], k4.y, dot);
        dot = fmaf(S[r4 + 2], k4.z, dot);
        dot = fmaf(S[r4 + 3], k4.w, dot);
      }
      dot = group_sum<8>(dot);
      const float u = bs[tt] * (vs[tt][cl] - dot);
      float acc = 0.f;
#pragma unroll
      for (int r4 = 0; r4 < R; r4 += 4) {
        const float4 k4 = *reinterpret_cast<const float4*>(&ks[tt][rg * R + r4]);
        const float4 q4 = *reinterpret_cast<const float4*>(&qs[tt][rg * R + r4]);
        S[r4 + 0] = fmaf(k4.x, u, S[r4 + 0]);
        S[r4 + 1] = fmaf(k4.y, u, S[r4 + 1]);
        S[r4 + 2] = fmaf(k4.z, u, S[r4 + 2]);
        S[r4 + 3] = fmaf(k4.w, u, S[r4 + 3]);
        acc = fmaf(S[r4 + 0], q4.x, acc);
        acc = fmaf(S[r4 + 1], q4.y, acc);
        acc = fmaf(S[r4 + 2], q4.z, acc);
        acc = fmaf(S[r4 + 3], q4.w, acc);
      }
      acc = group_sum<8>(acc);
      if (rg == 0 && col < dv) out[((t0 + base + tt) * heads + h) * (int64_t)dv + col] = acc;
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = rg * R + r;
    if (i < dk && col < dv) sp[(int64_t)i * dv + col] = S[r];
  }
}

template <typename QT, typename VT>
int launch_delta(float* out, float* state, const void* q, const void* k, const void* v, const void* beta_logits,
                 const float* gate_logits, const float* rate_bias, const float* rate_log, const int32_t* req_to_state,
                 const int64_t* req_pool_indices, const int32_t* seg_start, const int32_t* seg_len, const int64_t* positions,
                 int64_t batch, int heads, int qk_heads, int dk, int dv, int64_t qs, int64_t ks, int64_t vs, int64_t bs, int64_t gs,
                 float q_scale, int gate_per_head, int beta_f32, int64_t tokens, int64_t longest, float* records, int64_t record_bytes,
                 hipStream_t stream) {
  if (gate_per_head && chunks_serve(true, batch, heads, dk, dv, tokens, longest, seg_len, out)) {
    const ChunkArgs p{out, state, q, k, v, gate_logits, rate_bias, rate_log, nullptr, beta_logits, req_to_state, req_pool_indices, seg_start,
                      seg_len, positions, qs, ks, vs, gs, bs, heads, qk_heads, dk, dv, beta_f32, q_scale};
    return launch_chunks<QT, VT, true>(p, batch, tokens, longest, records, record_bytes, stream);
  }
  const dim3 grid((unsigned)cdiv(dv, RC_COLS), (unsigned)heads, (unsigned)batch);
#define MI355_GD_LAUNCH(R)                                                                                                     \
  hipLaunchKernelGGL((gated_delta_rule_kernel<QT, VT, R>), grid, dim3(256), 0, stream, out, state, (const QT*)q, (const QT*)k,  \
                     (const VT*)v, (const VT*)beta_logits, gate_logits, rate_bias, rate_log, req_to_state, req_pool_indices,   \
                     seg_start, seg_len, positions, heads, qk_heads, dk, dv, qs, ks, vs, bs, gs, q_scale, gate_per_head, beta_f32)
  if (dk <= 32) MI355_GD_LAUNCH(4);
  else if (dk <= 64) MI355_GD_LAUNCH(8);
  else if (dk <= 128) MI355_GD_LAUNCH(16);
  else MI355_GD_LAUNCH(32);
#undef MI355_GD_LAUNCH
  return MI355_OK;
}

// Matrix memory with exponential gates.  Per head and token, from two fp32 logits: the log input gate
// i = cap tanh((zi + bi) / cap), the log forget gate f = logsigmoid(cap tanh((zf + bf) / cap)), and
//     m' = max(f + m, i);   S <- e^(f + m - m') S + e^(i - m') k v^T;   n <- e^(f + m - m') n + e^(i - m') k;   m <- m'
//     o = S^T q / (max(|n . q|, e^-m) + 1e-6)            (q times q_scale; S, n and m start at zero)
// Same layout as above for S.  The normaliser n is one more column of S whose value is always 1: a fifth wave carries it
// (64 lanes share its dk channels) beside the four that carry the block's 32 columns, and the division happens when a stage's
// read-outs leave LDS in whole rows.  Every block of value columns keeps a copy of (n, m) of its own in norm_state
// [slots, heads, blocks, dk + 1] (m last): a block that starts late must not find what another one has already advanced.
constexpr int MM_THREADS = 320;

template <typename VT, int R>
__global__ __launch_bounds__(MM_THREADS) void matrix_memory_kernel(
    float* __restrict__ out, float* __restrict__ state, float* __restrict__ norm_state, const VT* __restrict__ q,
    const VT* __restrict__ k, const VT* __restrict__ v, const float* __restrict__ in_logits, const float* __restrict__ forget_logits,
    const float* __restrict__ in_bias, const float* __restrict__ forget_bias, const int32_t* __restrict__ req_to_state,
    const int64_t* __restrict__ req_pool_indices, const int32_t* __restrict__ seg_start, const int32_t* __restrict__ seg_len,
    const int64_t* __restrict__ positions, int heads, int dk, int dv, int64_t q_token_stride, int64_t k_token_stride,
    int64_t v_token_stride, int64_t gate_token_stride, float q_scale, float cap) {
  constexpr int DKP = R * RC_RG;
  constexpr int RN = DKP > 64 ? DKP / 64 : 1;       // channels of n per lane of the fifth wave
  __shared__ __attribute__((aligned(16))) float qs[RC_TC][DKP];
  __shared__ __attribute__((aligned(16))) float ks[RC_TC][DKP];
  __shared__ float vs[RC_TC][RC_COLS];
  __shared__ float os[RC_TC][RC_COLS + 1];
  __shared__ float li[RC_TC], lf[RC_TC], keep[RC_TC], write[RC_TC], floor_[RC_TC], inv_den[RC_TC];
  __shared__ float m_sh[2];
  const int b = blockIdx.z, h = blockIdx.y, c0 = blockIdx.x * RC_COLS;
  const int tid = threadIdx.x;
  const int rg = tid & (RC_RG - 1), cl = tid >> 3;
  const int col = c0 + cl;
  const bool column_wave = tid < 256;
  const int nl = tid & 63;
  const int64_t t0 = seg_start != nullptr ? seg_start[b] : b;
  const int n_tok = seg_len != nullptr ? seg_len[b] : 1;
  if (n_tok <= 0) return;
  const int64_t slot = req_to_state[req_pool_indices[b]];
  float* sp = state + ((slot * heads + h) * (int64_t)dk) * dv;
  float* np = norm_state + ((slot * heads + h) * (int64_t)gridDim.x + blockIdx.x) * (dk + 1);
  const bool fresh = positions[t0] == 0;
  float S[R], nv[RN];
  if (column_wave) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = rg * R + r;
      S[r] = (!fresh && i < dk && col < dv) ? sp[(int64_t)i * dv + col] : 0.f;
    }
  } else {
#pragma unroll
    for (int r = 0; r < RN; ++r) {
      const int i = nl * RN + r;
      nv[r] = (!fresh && i < dk) ? np[i] : 0.f;
    }
    if (nl == 0) m_sh[0] = fresh ? 0.f : np[dk];
  }
  const float bi = in_bias[h], bf = forget_bias[h];
  int par = 0;
  for (int base = 0; base < n_tok; base += RC_TC, par ^= 1) {
    const int m = min(RC_TC, n_tok - base);
    if (tid < m) {
      const int64_t g = (t0 + base + tid) * gate_token_stride + h;
      li[tid] = cap * tanhf((in_logits[g] + bi) / cap);
      lf[tid] = log_sigmoid_f(cap * tanhf((forget_logits[g] + bf) / cap));
    }
    __syncthreads();
    if (tid < m) {
      // the running maximum up to this token, by the same operations in the same order wherever the step was cut
      float prev = m_sh[par], cur = prev;
      for (int j = 0; j <= tid; ++j) {
        prev = cur;
        cur = fmaxf(lf[j] + prev, li[j]);
      }
      keep[tid] = expf(lf[tid] + prev - cur);
      write[tid] = expf(li[tid] - cur);
      floor_[tid] = expf(-cur);
      if (tid == m - 1) m_sh[par ^ 1] = cur;
    }
    for (int e = tid; e < m * RC_COLS; e += MM_THREADS) {
      const int tt = e / RC_COLS, c = e - tt * RC_COLS;
      vs[tt][c] = (c0 + c < dv) ? to_f32(v[(t0 + base + tt) * v_token_stride + (int64_t)h * dv + c0 + c]) : 0.f;
    }
    for (int e = tid; e < m * DKP; e += MM_THREADS) {
      const int tt = e / DKP, i = e - tt * DKP;
      const int64_t t = t0 + base + tt;
      qs[tt][i] = i < dk ? to_f32(q[t * q_token_stride + (int64_t)h * dk + i]) * q_scale : 0.f;
      ks[tt][i] = i < dk ? to_f32(k[t * k_token_stride + (int64_t)h * dk + i]) : 0.f;
    }
    __syncthreads();
    if (column_wave) {
      for (int tt = 0; tt < m; ++tt) {
        const float wv = write[tt] * vs[tt][cl], a = keep[tt];
        float acc = 0.f;
#pragma unroll
        for (int r4 = 0; r4 < R; r4 += 4) {
          const float4 k4 = *reinterpret_cast<const float4*>(&ks[tt][rg * R + r4]);
          const float4 q4 = *reinterpret_cast<const float4*>(&qs[tt][rg * R + r4]);
          S[r4 + 0] = fmaf(a, S[r4 + 0], k4.x * wv);
          S[r4 + 1] = fmaf(a, S[r4 + 1], k4.y * wv);
          S[r4 + 2] = fmaf(a, S[r4 + 2], k4.z * wv);
          S[r4 + 3] = fmaf(a, S[r4 + 3], k4.w * wv);
          acc = fmaf(S[r4 + 0], q4.x, acc);
          acc = fmaf(S[r4 + 1], q4.y, acc);
          acc = fmaf(S[r4 + 2], q4.z, acc);
          acc = fmaf(S[r4 + 3], q4.w, acc);
        }
        acc = group_sum<8>(acc);
        if (rg == 0) os[tt][cl] = acc;
      }
    } else {
      for (int tt = 0; tt < m; ++tt) {
        const float a = keep[tt], w = write[tt];
        float dot = 0.f;
#pragma unroll
        for (int r = 0; r < RN; ++r) {
          const int i = nl * RN + r;
          if (DKP >= 64 || i < DKP) {
            nv[r] = fmaf(a, nv[r], ks[tt][i] * w);
            dot = fmaf(nv[r], qs[tt][i], dot);
          }
        }
        dot = wave_sum(dot);
        if (nl == 0) inv_den[tt] = 1.0f / (fmaxf(fabsf(dot), floor_[tt]) + 1e-6f);
      }
    }
    __syncthreads();
    for (int e = tid; e < m * RC_COLS; e += MM_THREADS) {
      const int tt = e / RC_COLS, c = e - tt * RC_COLS;
      if (c0 + c < dv) out[((t0 + base + tt) * heads + h) * (int64_t)dv + c0 + c] = os[tt][c] * inv_den[tt];
    }
  }
  if (column_wave) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = rg * R + r;
      if (i < dk && col < dv) sp[(int64_t)i * dv + col] = S[r];
    }
  } else {
#pragma unroll
    for (int r = 0; r < RN; ++r) {
      const int i = nl * RN + r;
      if (i < dk) np[i] = nv[r];
    }
    if (nl == 0) np[dk] = m_sh[par];
  }
}

template <typename VT>
int launch_matrix_memory(float* out, float* state, float* norm_state, const void* q, const void* k, const void* v,
                         const float* in_logits, const float* forget_logits, const float* in_bias, const float* forget_bias,
                         const int32_t* req_to_state, const int64_t* req_pool_indices, const int32_t* seg_start, const int32_t* seg_len,
                         const int64_t* positions, int64_t batch, int heads, int dk, int dv, int64_t qs, int64_t ks, int64_t vs,
                         int64_t gs, float q_scale, float cap, hipStream_t stream) {
  const dim3 grid((unsigned)cdiv(dv, RC_COLS), (unsigned)heads, (unsigned)batch);
#define MI355_MM_LAUNCH(R)                                                                                                       \
  hipLaunchKernelGGL((matrix_memory_kernel<VT, R>), grid, dim3(MM_THREADS), 0, stream, out, state, norm_state, (const VT*)q,     \
                     (const VT*)k, (const VT*)v, in_logits, forget_logits, in_bias, forget_bias, req_to_state, req_pool_indices, \
                     seg_start, seg_len, positions, heads, dk, dv, qs, ks, vs, gs, q_scale, cap)
  if (dk <= 32) MI355_MM_LAUNCH(4);
  else if (dk <= 64) MI355_MM_LAUNCH(8);
  else if (dk <= 128) MI355_MM_LAUNCH(16);
  else MI355_MM_LAUNCH(32);
#undef MI355_MM_LAUNCH
  return MI355_OK;
}

}  // namespace
}  // namespace mi355

using namespace mi355;

int mi355_recurrence_takes_chunks(int delta, int64_t batch, int heads, int key_dim, int value_dim, int64_t tokens, int64_t longest) {
  return heads > 0 && key_dim > 0 && value_dim > 0 && chunks_pay(delta != 0, batch, heads, key_dim, value_dim, tokens, longest);
}

int64_t mi355_recurrence_workspace_bytes(int delta, int64_t batch, int heads, int key_dim, int value_dim, int64_t tokens, int64_t longest) {
  return heads > 0 && key_dim > 0 && value_dim > 0 ? chunk_records_bytes(delta != 0, batch, heads, key_dim, value_dim, tokens, longest) : 0;
}

int mi355_linear_recurrence(float* out, float* state, const void* q, const void* k, const void* v, const float* gate_logits,
                            const void* gate_bias, const float* head_decay, const int32_t* req_to_state,
                            const int64_t* req_pool_indices, const int32_t* seg_start, const int32_t* seg_len,
                            const int64_t* positions, int64_t batch, int heads, int key_dim, int value_dim, int64_t q_token_stride,
                            int64_t k_token_stride, int64_t v_token_stride, int64_t gate_token_stride, float q_scale, float tau,
                            int qk_dtype, int v_dtype, void* stream) {
  MI355_REQUIRE((gate_logits != nullptr) != (head_decay != nullptr), MI355_ERR_INVALID,
                "linear_recurrence: the decay is either gate logits per channel or one number per head");
  return mi355_linear_recurrence_ssm(out, state, q, k, v, gate_logits, gate_bias, head_decay, nullptr, 0, nullptr, nullptr, nullptr,
                                     req_to_state, req_pool_indices, seg_start, seg_len, positions, batch, heads, heads, key_dim,
                                     value_dim, q_token_stride, k_token_stride, v_token_stride, gate_token_stride, q_scale, tau,
                                     qk_dtype, v_dtype, stream);
}

int mi355_linear_recurrence_ssm(float* out, float* state, const void* q, const void* k, const void* v, const float* gate_logits,
                                const void* gate_bias, const float* head_decay, const float* dt_logits, int64_t dt_token_stride,
                                const float* dt_bias, const float* rate_log, const float* skip, const int32_t* req_to_state,
                                const int64_t* req_pool_indices, const int32_t* seg_start, const int32_t* seg_len,
                                const int64_t* positions, int64_t batch, int heads, int qk_heads, int key_dim, int value_dim,
                                int64_t q_token_stride, int64_t k_token_stride, int64_t v_token_stride, int64_t gate_token_stride,
                                float q_scale, float tau, int qk_dtype, int v_dtype, void* stream) {
  return mi355_linear_recurrence_ssm_sized(out, state, q, k, v, gate_logits, gate_bias, head_decay, dt_logits, dt_token_stride, dt_bias,
                                           rate_log, skip, req_to_state, req_pool_indices, seg_start, seg_len, positions, batch, heads,
                                           qk_heads, key_dim, value_dim, q_token_stride, k_token_stride, v_token_stride,
                                           gate_token_stride, q_scale, tau, qk_dtype, v_dtype, 0, 0, stream);
}

int mi355_linear_recurrence_ssm_sized(float* out, float* state, const void* q, const void* k, const void* v, const float* gate_logits,
                                const void* gate_bias, const float* head_decay, const float* dt_logits, int64_t dt_token_stride,
                                const float* dt_bias, const float* rate_log, const float* skip, const int32_t* req_to_state,
                                const int64_t* req_pool_indices, const int32_t* seg_start, const int32_t* seg_len,
                                const int64_t* positions, int64_t batch, int heads, int qk_heads, int key_dim, int value_dim,
                                int64_t q_token_stride, int64_t k_token_stride, int64_t v_token_stride, int64_t gate_token_stride,
                                float q_scale, float tau, int qk_dtype, int v_dtype, int64_t tokens, int64_t longest, void* stream) {
  return mi355_linear_recurrence_ssm_ws(out, state, q, k, v, gate_logits, gate_bias, head_decay, dt_logits, dt_token_stride, dt_bias, rate_log, skip,
                                        req_to_state, req_pool_indices, seg_start, seg_len, positions, batch, heads, qk_heads, key_dim,
                                        value_dim, q_token_stride, k_token_stride, v_token_stride, gate_token_stride, q_scale, tau,
                                        qk_dtype, v_dtype, tokens, longest, nullptr, 0, stream);
}

int mi355_linear_recurrence_ssm_ws(float* out, float* state, const void* q, const void* k, const void* v, const float* gate_logits,
                                const void* gate_bias, const float* head_decay, const float* dt_logits, int64_t dt_token_stride,
                                const float* dt_bias, const float* rate_log, const float* skip, const int32_t* req_to_state,
                                const int64_t* req_pool_indices, const int32_t* seg_start, const int32_t* seg_len,
                                const int64_t* positions, int64_t batch, int heads, int qk_heads, int key_dim, int value_dim,
                                int64_t q_token_stride, int64_t k_token_stride, int64_t v_token_stride, int64_t gate_token_stride,
                                float q_scale, float tau, int qk_dtype, int v_dtype, int64_t tokens, int64_t longest, void* workspace,
                              int64_t workspace_bytes, void* stream) {
  MI355_REQUIRE(out && state && q && k && v && req_to_state && req_pool_indices && positions, MI355_ERR_INVALID,
                "linear_recurrence: null pointer");
  MI355_REQUIRE((gate_logits != nullptr) + (head_decay != nullptr) + (dt_logits != nullptr) == 1, MI355_ERR_INVALID,
                "linear_recurrence: the decay is gate logits per channel, one number per head, or a step size per head and token");
  MI355_REQUIRE(dt_logits == nullptr || (dt_bias && rate_log && dt_token_stride >= heads), MI355_ERR_INVALID,
                "linear_recurrence: step sizes come with their bias and the heads' rates");
  MI355_REQUIRE((seg_start == nullptr) == (seg_len == nullptr), MI355_ERR_INVALID,
                "linear_recurrence: seg_start and seg_len come together");
  MI355_REQUIRE(batch >= 0 && batch <= 65535 && heads > 0 && heads <= 65535 && key_dim > 0 && value_dim > 0 && tau > 0.f &&
                    qk_heads > 0 && heads % qk_heads == 0, MI355_ERR_INVALID, "linear_recurrence: bad shape");
  MI355_REQUIRE(key_dim <= 256, MI355_ERR_UNSUPPORTED, "linear_recurrence: key width %d above 256", key_dim);
  MI355_REQUIRE(qk_dtype == v_dtype || qk_dtype == MI355_F32, MI355_ERR_UNSUPPORTED,
                "linear_recurrence: q and k come in the type of v or in fp32");
  if (batch == 0) return MI355_OK;
  int rc = MI355_OK;
  MI355_DISPATCH_DTYPE(v_dtype, "linear_recurrence", {
    if (qk_dtype == v_dtype)
      rc = launch_recurrence<T, T>(out, state, q, k, v, gate_logits, gate_bias, head_decay, req_to_state, req_pool_indices,
                                   seg_start, seg_len, positions, batch, heads, key_dim, value_dim, q_token_stride, k_token_stride,
                                   v_token_stride, gate_token_stride, q_scale, tau, qk_heads, dt_logits, dt_token_stride, dt_bias,
                                   rate_log, skip, tokens, longest, (float*)workspace, workspace_bytes, (hipStream_t)stream);
    else
      rc = launch_recurrence<float, T>(out, state, q, k, v, gate_logits, gate_bias, head_decay, req_to_state, req_pool_indices,
                                       seg_start, seg_len, positions, batch, heads, key_dim, value_dim, q_token_stride,
                                       k_token_stride, v_token_stride, gate_token_stride, q_scale, tau, qk_heads, dt_logits,
                                       dt_token_stride, dt_bias, rate_log, skip, tokens, longest, (float*)workspace, workspace_bytes, (hipStream_t)stream);
  });
  if (rc != MI355_OK) return rc;
  MI355_CHECK_LAUNCH("linear_recurrence");
  return MI355_OK;
}

int mi355_gated_delta_rule(float* out, float* state, const void* q, const void* k, const void* v, const void* beta_logits,
                           const float* gate_logits, const float* rate_bias, const float* rate_log, const int32_t* req_to_state,
                           const int64_t* req_pool_indices, const int32_t* seg_start, const int32_t* seg_len,
                           const int64_t* positions, int64_t batch, int heads, int qk_heads, int key_dim, int value_dim,
                           int64_t q_token_stride, int64_t k_token_stride, int64_t v_token_stride, int64_t beta_token_stride,
                           int64_t gate_token_stride, float q_scale, int qk_dtype, int v_dtype, void* stream) {
  return mi355_gated_delta_rule_ex(out, state, q, k, v, beta_logits, gate_logits, rate_bias, rate_log, req_to_state, req_pool_indices,
                                   seg_start, seg_len, positions, batch, heads, qk_heads, key_dim, value_dim, q_token_stride,
                                   k_token_stride, v_token_stride, beta_token_stride, gate_token_stride, q_scale, 0, 0, qk_dtype,
                                   v_dtype, stream);
}

int mi355_gated_delta_rule_ex(float* out, float* state, const void* q, const void* k, const void* v, const void* beta_logits,
                              const float* gate_logits, const float* rate_bias, const float* rate_log, const int32_t* req_to_state,
                              const int64_t* req_pool_indices, const int32_t* seg_start, const int32_t* seg_len,
                              const int64_t* positions, int64_t batch, int heads, int qk_heads, int key_dim, int value_dim,
                              int64_t q_token_stride, int64_t k_token_stride, int64_t v_token_stride, int64_t beta_token_stride,
                              int64_t gate_token_stride, float q_scale, int gate_per_head, int beta_f32, int qk_dtype, int v_dtype,
                              void* stream) {
  return mi355_gated_delta_rule_sized(out, state, q, k, v, beta_logits, gate_logits, rate_bias, rate_log, req_to_state, req_pool_indices,
                                      seg_start, seg_len, positions, batch, heads, qk_heads, key_dim, value_dim, q_token_stride,
                                      k_token_stride, v_token_stride, beta_token_stride, gate_token_stride, q_scale, gate_per_head,
                                      beta_f32, qk_dtype, v_dtype, 0, 0, stream);
}

int mi355_gated_delta_rule_sized(float* out, float* state, const void* q, const void* k, const void* v, const void* beta_logits,
                              const float* gate_logits, const float* rate_bias, const float* rate_log, const int32_t* req_to_state,
                              const int64_t* req_pool_indices, const int32_t* seg_start, const int32_t* seg_len,
                              const int64_t* positions, int64_t batch, int heads, int qk_heads, int key_dim, int value_dim,
                              int64_t q_token_stride, int64_t k_token_stride, int64_t v_token_stride, int64_t beta_token_stride,
                              int64_t gate_token_stride, float q_scale, int gate_per_head, int beta_f32, int qk_dtype, int v_dtype,
                              int64_t tokens, int64_t longest, void* stream) {
  return mi355_gated_delta_rule_ws(out, state, q, k, v, beta_logits, gate_logits, rate_bias, rate_log, req_to_state, req_pool_indices, seg_start,
                                   seg_len, positions, batch, heads, qk_heads, key_dim, value_dim, q_token_stride, k_token_stride,
                                   v_token_stride, beta_token_stride, gate_token_stride, q_scale, gate_per_head, beta_f32, qk_dtype,
                                   v_dtype, tokens, longest, nullptr, 0, stream);
}

int mi355_gated_delta_rule_ws(float* out, float* state, const void* q, const void* k, const void* v, const void* beta_logits,
                              const float* gate_logits, const float* rate_bias, const float* rate_log, const int32_t* req_to_state,
                              const int64_t* req_pool_indices, const int32_t* seg_start, const int32_t* seg_len,
                              const int64_t* positions, int64_t batch, int heads, int qk_heads, int key_dim, int value_dim,
                              int64_t q_token_stride, int64_t k_token_stride, int64_t v_token_stride, int64_t beta_token_stride,
                              int64_t gate_token_stride, float q_scale, int gate_per_head, int beta_f32, int qk_dtype, int v_dtype,
                              int64_t tokens, int64_t longest, void* workspace,
                              int64_t workspace_bytes, void* stream) {
  MI355_REQUIRE(out && state && q && k && v && beta_logits && gate_logits && rate_bias && rate_log && req_to_state &&
                    req_pool_indices && positions, MI355_ERR_INVALID, "gated_delta_rule: null pointer");
  MI355_REQUIRE((seg_start == nullptr) == (seg_len == nullptr), MI355_ERR_INVALID,
                "gated_delta_rule: seg_start and seg_len come together");
  MI355_REQUIRE(batch >= 0 && batch <= 65535 && heads > 0 && heads <= 65535 && qk_heads > 0 && heads % qk_heads == 0 &&
                    key_dim > 0 && value_dim > 0, MI355_ERR_INVALID, "gated_delta_rule: bad shape");
  MI355_REQUIRE(key_dim <= 256, MI355_ERR_UNSUPPORTED, "gated_delta_rule: key width %d above 256", key_dim);
  MI355_REQUIRE(qk_dtype == v_dtype || qk_dtype == MI355_F32, MI355_ERR_UNSUPPORTED,
                "gated_delta_rule: q and k come in the type of v or in fp32");
  if (batch == 0) return MI355_OK;
  int rc = MI355_OK;
  MI355_DISPATCH_DTYPE(v_dtype, "gated_delta_rule", {
    if (qk_dtype == v_dtype)
      rc = launch_delta<T, T>(out, state, q, k, v, beta_logits, gate_logits, rate_bias, rate_log, req_to_state, req_pool_indices,
                              seg_start, seg_len, positions, batch, heads, qk_heads, key_dim, value_dim, q_token_stride,
                              k_token_stride, v_token_stride, beta_token_stride, gate_token_stride, q_scale, gate_per_head, beta_f32,
                              tokens, longest, (float*)workspace, workspace_bytes, (hipStream_t)stream);
    else
      rc = launch_delta<float, T>(out, state, q, k, v, beta_logits, gate_logits, rate_bias, rate_log, req_to_state,
                                  req_pool_indices, seg_start, seg_len, positions, batch, heads, qk_heads, key_dim, value_dim,
                                  q_token_stride, k_token_stride, v_token_stride, beta_token_stride, gate_token_stride, q_scale,
                                  gate_per_head, beta_f32, tokens, longest, (float*)workspace, workspace_bytes, (hipStream_t)stream);
  });
  if (rc != MI355_OK) return rc;
  MI355_CHECK_LAUNCH("gated_delta_rule");
  return MI355_OK;
}

int mi355_matrix_memory_value_block(void) { return RC_COLS; }

int mi355_matrix_memory(float* out, float* state, float* norm_state, const void* q, const void* k, const void* v,
                        const float* in_logits, const float* forget_logits, const float* in_bias, const float* forget_bias,
                        const int32_t* req_to_state, const int64_t* req_pool_indices, const int32_t* seg_start, const int32_t* seg_len,
                        const int64_t* positions, int64_t batch, int heads, int key_dim, int value_dim, int norm_blocks,
                        int64_t q_token_stride, int64_t k_token_stride, int64_t v_token_stride, int64_t gate_token_stride,
                        float q_scale, float gate_cap, int dtype, void* stream) {
  MI355_REQUIRE(out && state && norm_state && q && k && v && in_logits && forget_logits && in_bias && forget_bias && req_to_state &&
                    req_pool_indices && positions, MI355_ERR_INVALID, "matrix_memory: null pointer");
  MI355_REQUIRE((seg_start == nullptr) == (seg_len == nullptr), MI355_ERR_INVALID, "matrix_memory: seg_start and seg_len come together");
  MI355_REQUIRE(batch >= 0 && batch <= 65535 && heads > 0 && heads <= 65535 && key_dim > 0 && value_dim > 0 && gate_cap > 0.f &&
                    gate_token_stride >= heads, MI355_ERR_INVALID, "matrix_memory: bad shape");
  MI355_REQUIRE(norm_blocks == cdiv(value_dim, RC_COLS), MI355_ERR_INVALID,
                "matrix_memory: %d copies of the normaliser for %d value columns (one per %d)", norm_blocks, value_dim, RC_COLS);
  MI355_REQUIRE(key_dim <= 256, MI355_ERR_UNSUPPORTED, "matrix_memory: key width %d above 256", key_dim);
  if (batch == 0) return MI355_OK;
  int rc = MI355_OK;
  MI355_DISPATCH_DTYPE(dtype, "matrix_memory", {
    rc = launch_matrix_memory<T>(out, state, norm_state, q, k, v, in_logits, forget_logits, in_bias, forget_bias, req_to_state,
                                 req_pool_indices, seg_start, seg_len, positions, batch, heads, key_dim, value_dim, q_token_stride,
                                 k_token_stride, v_token_stride, gate_token_stride, q_scale, gate_cap, (hipStream_t)stream);
  });
  if (rc != MI355_OK) return rc;
  MI355_CHECK_LAUNCH("matrix_memory");
  return MI355_OK;
}
