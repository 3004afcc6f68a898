// Extend / prefill attention: new tokens attend to (1) their sequence's cached prefix, gathered
// through kv_indices from the paged KV cache, and (2) the new tokens themselves (causal
// triangle), with one online softmax across both phases.
//
// Structure of the general kernel: a workgroup (4 waves) owns a tile of 64 "rows" = TM query tokens x Gc query heads
// that share one kv head, so every K/V tile staged in LDS is reused by all heads of the group.
// K/V tiles of BN keys are gathered with 16-byte loads into padded LDS rows (bank-conflict free
// for the access patterns below).  Scores and P.V are register-blocked fp32 VALU FMAs (each lane
// a 4 x KJ score block, then a 4 x DPL output block), which keeps exact-fp32 accumulation for
// every dtype -- this is also the fp32 parity path.  Row max uses xor-shuffles across the 16
// lanes that share a row; the row sum is reduced once at the end.
#include "common.cuh"
#include <algorithm>
#include <type_traits>
#include <math.h>

namespace mi355 {

static constexpr float kLog2eE = 1.4426950408889634f;

struct ExtendParams {
  const int32_t* qo_indptr;
  const int32_t* kv_indptr;
  const int32_t* kv_indices;
  const uint8_t* custom_mask;
  const int64_t* mask_indptr;
  int64_t q_stride, k_stride, v_stride;
  int is_causal, skip_prefix_custom_mask, hq, hkv, D, Dv, sliding_window;
  float sm_scale, logit_cap;
  // the cache buffers: elements between consecutive slots / consecutive kv heads ([slots, hkv, d] or head-major)
  int64_t kb_slot, kb_head, vb_slot, vb_head;
  uint32_t near_slots;   // DIRECT: slots below this one lie within the 32-bit offsets of a buffer
  int kv8;   // the cache holds e4m3fn bytes behind the element pointers (strides count bytes); read by the VALU kernel
  // latent form (extend_attn_latent_kernel): whole sequences, tokens seg_start[b] .. + seg_len[b]
  const int32_t* seg_start;
  const int32_t* seg_len;
  const int64_t* positions;   // [tokens]
  const float* inv_freq;      // [rot_dims / 2]
  const void* k_rope;         // [tokens, 64] rotated key part that the heads share, rows k_rope_stride apart
  int64_t k_rope_stride;
  int kv_head;                // elements between consecutive heads of k / v
  int rot_dims, interleaved;  // of the query's rope part: features 2 i with 2 i + 1, or (rot_dims 64) i with i + 32
  float rot_mag;
  // splits of the keys (grid y): unnormalised sums part [splits, rows, hq, Dv] and (maximum, weights' sum) part_ml [splits, rows, hq]
  float* part;
  float2* part_ml;
  int64_t rows;
};

// DP: padded head dim (>= D, Dv; multiple of 64). BN: keys per tile. VEC: 16-B global loads.
template <typename T, int DP, int BN, bool VEC>
__global__ __launch_bounds__(256, 2) void extend_attn_kernel(const T* __restrict__ q_ext,
                                                          const T* __restrict__ k_ext,
                                                          const T* __restrict__ v_ext,
                                                          T* __restrict__ o_ext,
                                                          const T* __restrict__ kbuf,
                                                          const T* __restrict__ vbuf,
                                                          ExtendParams p) {
  constexpr int VE = V16<T>::n;
  constexpr int LROW = DP + VE;          // padded LDS row (elements): +16 B
  constexpr int KJ = BN / 16;            // keys per lane in the score block
  constexpr int DPL = DP / 16;           // output features per lane
  constexpr int PROW = BN + 4;           // padded P row (floats)
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  T* qs = reinterpret_cast<T*>(smem_raw);            // [64][LROW]
  T* ks = qs + 64 * LROW;                            // [BN][LROW]
  T* vs = ks + BN * LROW;                            // [BN][LROW]
  float* ps = reinterpret_cast<float*>(vs + BN * LROW);  // [64][PROW]

  const int gtotal = p.hq / p.hkv;
  const int Gc = gtotal < 64 ? gtotal : 64;
  const int chunks_per_kv = gtotal / Gc;
  const int TM = 64 / Gc;
  const int kvh = blockIdx.y / chunks_per_kv;
  const int head0 = kvh * gtotal + (blockIdx.y % chunks_per_kv) * Gc;
  const int b = blockIdx.z;
  const int q_start = p.qo_indptr[b];
  const int ext_len = p.qo_indptr[b + 1] - q_start;
  const int t0 = blockIdx.x * TM;
  if (t0 >= ext_len) return;
  const int kv_start = p.kv_indptr[b];
  const int prefix_len = p.kv_indptr[b + 1] - kv_start;
  const int seq_len = prefix_len + ext_len;
  const int D = p.D, Dv = p.Dv;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c16 = lane & 15, rg = lane >> 4;  // c16: key / feature column group; rg: row group

  // rows of this lane: r_i = 16*wave + rg + 4*i
  int row_tok[4], row_head[4];
  bool row_ok[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 16 * wave + rg + 4 * i;
    row_tok[i] = r / Gc;
    row_head[i] = r - row_tok[i] * Gc;
    row_ok[i] = row_tok[i] < TM && t0 + row_tok[i] < ext_len;
  }

  // ---- stage Q (zero padded to DP, rows beyond the tile zero) ----
  for (int pidx = threadIdx.x; pidx < 64 * (DP / VE); pidx += 256) {
    const int r = pidx / (DP / VE), c = (pidx % (DP / VE)) * VE;
    const int tq = r / Gc, g = r - tq * Gc;
    Vec<T, VE> val;
#pragma unroll
    for (int j = 0; j < VE; ++j) val.v[j] = (T)0.f;
    if (tq < TM && t0 + tq < ext_len) {
      const T* src = q_ext + (int64_t)(q_start + t0 + tq) * p.q_stride + (int64_t)(head0 + g) * D;
      if (VEC && c + VE <= D) {
        val = ldvec<T, VE>(src + c);
      } else {
#pragma unroll
        for (int j = 0; j < VE; ++j)
          if (c + j < D) val.v[j] = src[c + j];
      }
    }
    stvec<T, VE>(qs + r * LROW + c, val);
  }

  float m[4], l[4], acc[4][DPL];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    m[i] = -INFINITY;
    l[i] = 0.f;
#pragma unroll
    for (int d = 0; d < DPL; ++d) acc[i][d] = 0.f;
  }

  const bool cap = p.logit_cap > 0.f;
  // keys of phase 2 this tile needs: causal -> up to its last token
  const int tile_last_tok = (t0 + TM < ext_len ? t0 + TM : ext_len) - 1;
  const int ext_keys = p.is_causal ? tile_last_tok + 1 : ext_len;

  for (int phase = 0; phase < 2; ++phase) {
    const int nkeys = phase == 0 ? prefix_len : ext_keys;
    for (int kb = 0; kb < nkeys; kb += BN) {
      __syncthreads();  // previous tile fully consumed (also covers the Q staging)
      // ---- stage K and V tiles ----
      for (int pidx = threadIdx.x; pidx < BN * (DP / VE); pidx += 256) {
        const int kr = pidx / (DP / VE), c = (pidx % (DP / VE)) * VE;
        const int key = kb + kr;
        Vec<T, VE> kval, vval;
#pragma unroll
        for (int j = 0; j < VE; ++j) {
          kval.v[j] = (T)0.f;
          vval.v[j] = (T)0.f;
        }
        if (key < nkeys) {
          const T *ksrc, *vsrc;
          if (phase == 0) {
            const int64_t slot = p.kv_indices[kv_start + key];
            ksrc = kbuf + slot * p.kb_slot + kvh * p.kb_head;
            vsrc = vbuf + slot * p.vb_slot + kvh * p.vb_head;
          } else {
            ksrc = k_ext + (int64_t)(q_start + key) * p.k_stride + (int64_t)kvh * D;
            vsrc = v_ext + (int64_t)(q_start + key) * p.v_stride + (int64_t)kvh * Dv;
          }
          if (phase == 0 && p.kv8) {   // e4m3fn prefix rows, widened exactly
            const int64_t slot = p.kv_indices[kv_start + key];
            const uint8_t* k8 = reinterpret_cast<const uint8_t*>(kbuf) + slot * p.kb_slot + kvh * p.kb_head;
            const uint8_t* v8 = reinterpret_cast<const uint8_t*>(vbuf) + slot * p.vb_slot + kvh * p.vb_head;
#pragma unroll
            for (int j = 0; j < VE; ++j) {
              if (c + j < D) kval.v[j] = from_f32<T>(__builtin_amdgcn_cvt_f32_fp8((int)k8[c + j], 0));
              if (c + j < Dv) vval.v[j] = from_f32<T>(__builtin_amdgcn_cvt_f32_fp8((int)v8[c + j], 0));
            }
          } else {
          if (VEC && c + VE <= D) {
            kval = ldvec<T, VE>(ksrc + c);
          } else {
#pragma unroll
            for (int j = 0; j < VE; ++j)
              if (c + j < D) kval.v[j] = ksrc[c + j];
          }
          if (VEC && c + VE <= Dv) {
            vval = ldvec<T, VE>(vsrc + c);
          } else {
#pragma unroll
            for (int j = 0; j < VE; ++j)
              if (c + j < Dv) vval.v[j] = vsrc[c + j];
          }
          }
        }
        stvec<T, VE>(ks + kr * LROW + c, kval);
        stvec<T, VE>(vs + kr * LROW + c, vval);
      }
      __syncthreads();

      // ---- scores: s[i][j] = q[row_i] . k[key c16 + 16 j] ----
      float s[4][KJ];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < KJ; ++j) s[i][j] = 0.f;
      const T* qrow = qs + (16 * wave + rg) * LROW;
      const T* krow = ks + c16 * LROW;
#pragma unroll 1
      for (int c = 0; c < DP; c += VE) {
        float qf[4][VE], kf[KJ][VE];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          Vec<T, VE> t = ldvec<T, VE>(qrow + 4 * i * LROW + c);
#pragma unroll
          for (int e = 0; e < VE; ++e) qf[i][e] = to_f32(t.v[e]);
        }
#pragma unroll
        for (int j = 0; j < KJ; ++j) {
          Vec<T, VE> t = ldvec<T, VE>(krow + 16 * j * LROW + c);
#pragma unroll
          for (int e = 0; e < VE; ++e) kf[j][e] = to_f32(t.v[e]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < KJ; ++j)
#pragma unroll
            for (int e = 0; e < VE; ++e) s[i][j] = fmaf(qf[i][e], kf[j][e], s[i][j]);
      }

      // ---- scale, cap, mask; online softmax ----
      float alpha[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int tq = t0 + row_tok[i];  // extend-local query index
        float mx = -INFINITY;
#pragma unroll
        for (int j = 0; j < KJ; ++j) {
          const int key = kb + c16 + 16 * j;
          float x = s[i][j] * p.sm_scale;
          if (cap) x = p.logit_cap * tanhf(x / p.logit_cap);
          x *= kLog2eE;
          bool keep = row_ok[i] && key < nkeys;
          if (phase == 0) {
            if (p.custom_mask && !p.skip_prefix_custom_mask && keep)
              keep = p.custom_mask[p.mask_indptr[b] + (int64_t)tq * seq_len + key] != 0;
            if (p.sliding_window > 0) keep = keep && tq <= key + p.sliding_window;
          } else {
            if (p.custom_mask) {
              if (keep)
                keep = p.custom_mask[p.mask_indptr[b] + (int64_t)tq * seq_len + prefix_len + key] != 0;
            } else if (p.is_causal) {
              keep = keep && key <= tq;
            }
          }
          x = keep ? x : -INFINITY;
          s[i][j] = x;
          mx = fmaxf(mx, x);
        }
        mx = row16_max(mx);
        const float mnew = fmaxf(m[i], mx);
        const float ms = mnew == -INFINITY ? 0.f : mnew;
        alpha[i] = exp2f(m[i] - ms);
        m[i] = mnew;
        float psum = 0.f;
        float* prow = ps + (16 * wave + rg + 4 * i) * PROW;
#pragma unroll
        for (int j = 0; j < KJ; ++j) {
          const float pe = exp2f(s[i][j] - ms);
          psum += pe;
          prow[c16 + 16 * j] = pe;
        }
        l[i] = l[i] * alpha[i] + psum;
      }
      __syncthreads();  // P visible (only same-wave rows are read, barrier keeps it simple)

      // ---- acc[i][d] = acc*alpha + sum_key P[row_i][key] * V[key][c16*DPL + d] ----
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int d = 0; d < DPL; ++d) acc[i][d] *= alpha[i];
      const float* pbase = ps + (16 * wave + rg) * PROW;
      const T* vcol = vs + c16 * DPL;
#pragma unroll 1
      for (int k4 = 0; k4 < BN; k4 += 4) {
        float pf[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float4 t = *reinterpret_cast<const float4*>(pbase + 4 * i * PROW + k4);
          pf[i][0] = t.x; pf[i][1] = t.y; pf[i][2] = t.z; pf[i][3] = t.w;
        }
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
          float vf[DPL];
          if constexpr (DPL >= VE) {
#pragma unroll
            for (int d0 = 0; d0 < DPL; d0 += VE) {
              Vec<T, VE> t = ldvec<T, VE>(vcol + (k4 + kk) * LROW + d0);
#pragma unroll
              for (int e = 0; e < VE; ++e) vf[d0 + e] = to_f32(t.v[e]);
            }
          } else {
            Vec<T, DPL> t = ldvec<T, DPL>(vcol + (k4 + kk) * LROW);
#pragma unroll
            for (int e = 0; e < DPL; ++e) vf[e] = to_f32(t.v[e]);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int d = 0; d < DPL; ++d) acc[i][d] = fmaf(pf[i][kk], vf[d], acc[i][d]);
        }
      }
    }
  }

  // ---- finish: reduce row sums over the 16 lanes of a row, normalise, store ----
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float lt = l[i];
    lt = row16_sum(lt);
    if (!row_ok[i]) continue;
    const float inv = lt > 0.f ? 1.0f / lt : 0.f;
    T* dst = o_ext + ((int64_t)(q_start + t0 + row_tok[i]) * p.hq + head0 + row_head[i]) * Dv +
             c16 * DPL;
    if (VEC && c16 * DPL + DPL <= Dv) {
      Vec<T, DPL> out;
#pragma unroll
      for (int d = 0; d < DPL; ++d) out.v[d] = from_f32<T>(acc[i][d] * inv);
      stvec<T, DPL>(dst, out);
    } else {
#pragma unroll
      for (int d = 0; d < DPL; ++d)
        if (c16 * DPL + d < Dv) dst[d] = from_f32<T>(acc[i][d] * inv);
    }
  }
}

// ------------------------------------------------------------------------------------------
// MFMA flash-attention tile for the common prefill case: head_dim = v_head_dim = 128, 16-bit,
// causal or full, no custom mask / sliding window / logit cap.
//
// grid (q blocks of 64 rows, longest first; Hq; B), block 256 = 4 waves x 16 query rows.
// Per 64-key tile (K and V rows staged once in LDS for the 4 waves, next tile prefetched into
// registers while this one is computed):
//   S^T = K . Q^T   : A = K rows from LDS (ds_read_b128), B = Q^T kept in registers.  With the keys
//                     on the MFMA row axis, lane (query j = l & 15, c = l >> 4) owns the scores of
//                     ITS query for keys 16t + 4c + r: the softmax is lane-local apart from two
//                     cross-row maxima, and the probabilities are ALREADY the B operand of the
//                     next product (k index (c, e) <-> key 16 (e >> 2) + 4c + (e & 3)).
//   O^T += V^T . P^T: A = V^T fetched from the row-major V tile with ds_read_b64_tr_b16 (hardware
//                     transpose: 4 key rows x 16 features per 16 lanes), in the same key order.
// The output accumulator holds O^T[d = 16 dt + 4c + r][query j] and is rescaled per lane.
// ------------------------------------------------------------------------------------------
constexpr int XK_ROW = 128 + 16;   // K tile row (elements): 288 B.  Measured: SQ_LDS_BANK_CONFLICT is zero with 288-B rows and
                                   // 24 % of the LDS-active cycles with 272-B rows for the ds_read_b128 fragment reads
constexpr int XV_ROW = 128 + 16;   // V tile row: 288 B -> conflict-free transposed reads

// Three waves per SIMD (168 registers): the phases of a tile (LDS reads, MFMAs, softmax arithmetic,
// transposed reads, MFMAs) run back to back within a wave, so it is the number of resident waves that
// overlaps them: 2.17 -> 1.75 ms per layer against two waves.  To fit, the K fragments of a k-step
// are read right before their MFMAs (no second fragment buffer: the other waves cover that latency).
// KV8: the prefix lives in an e4m3fn cache (kbuf / vbuf are byte buffers); its rows are widened to T
// while they are staged.  The extend part (k_ext / v_ext) is always T.
// v_exp_f32 as is: the library exp2f wraps it in range scaling so that results below 2^-126 come out
// as denormals instead of zero (five instructions per call, and this kernel is bound by instruction
// issue).  A softmax weight that small contributes nothing at 16-bit output precision.
__device__ __forceinline__ float raw_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

template <typename T, bool KV8 = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void extend_attn_mfma_kernel(const T* __restrict__ q_ext,
                                                               const T* __restrict__ k_ext,
                                                               const T* __restrict__ v_ext,
                                                               T* __restrict__ o_ext,
                                                               const T* __restrict__ kbuf,
                                                               const T* __restrict__ vbuf,
                                                               ExtendParams p) {
  constexpr int D = 128;
  using frag = typename Mfma<T>::frag;
  __shared__ __attribute__((aligned(16))) T ks[64 * XK_ROW];
  __shared__ __attribute__((aligned(16))) T vs[64 * XV_ROW];

  const int qb = gridDim.x - 1 - blockIdx.x;   // long (late) blocks first
  const int h = blockIdx.y, b = blockIdx.z;
  const int kvh = h / (p.hq / p.hkv);
  const int q_start = p.qo_indptr[b];
  const int ext = p.qo_indptr[b + 1] - q_start;
  const int kv_start = p.kv_indptr[b];
  const int prefix = p.kv_indptr[b + 1] - kv_start;
  const int r0 = qb * 64;
  if (r0 >= ext) return;   // whole workgroup: EXEC stays full for the transposed reads below

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int j16 = lane & 15, c4 = lane >> 4;
  const int qrow = r0 + wave * 16 + j16;                  // this lane's query (row of the extend part)
  const int qrow_c = qrow < ext ? qrow : ext - 1;
  const float qmul = p.sm_scale * kLog2eE;

  // B operand of S^T: Q[qrow][32 s + 8 c + 0..7]
  frag qf[4];
  {
    const T* qp = q_ext + (int64_t)(q_start + qrow_c) * p.q_stride + (int64_t)h * D + 8 * c4;
#pragma unroll
    for (int s = 0; s < 4; ++s) qf[s] = *reinterpret_cast<const frag*>(qp + 32 * s);
  }

  // keys this workgroup needs: [0, total) in the logical order prefix | extend
  const int last_row = min(r0 + 63, ext - 1);
  const int total = p.is_causal ? prefix + last_row + 1 : prefix + ext;
  const int n_tiles = (total + 63) / 64;
  const int my_limit = p.is_causal ? prefix + qrow_c : prefix + ext - 1;   // last visible key of this lane's query
  const int wave_min_limit = p.is_causal ? prefix + min(r0 + wave * 16, ext - 1) : prefix + ext - 1;

  // tile staging: thread -> rows (threadIdx.x >> 4) + 16 i, 16-B chunk (threadIdx.x & 15)
  const int srow = threadIdx.x >> 4, sch = threadIdx.x & 15;
  Vec<T, 8> kreg[4], vreg[4];
  // rows of the extend part are a fixed stride apart: one base pointer per staged row, no index math
  const T* k_lin = k_ext + (int64_t)(q_start - prefix + srow) * p.k_stride + (int64_t)kvh * D + sch * 8;
  const T* v_lin = v_ext + (int64_t)(q_start - prefix + srow) * p.v_stride + (int64_t)kvh * D + sch * 8;
  auto load_tile = [&](int kt) {
    if (kt * 64 >= prefix && kt * 64 + 63 < total) {   // whole tile in the extend part (workgroup-uniform)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t key = kt * 64 + 16 * i;
        kreg[i] = ldvec<T, 8>(k_lin + key * p.k_stride);
        vreg[i] = ldvec<T, 8>(v_lin + key * p.v_stride);
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int key = kt * 64 + srow + 16 * i;
      key = key < total ? key : total - 1;
      if (KV8 && key < prefix) {
        const int64_t slot = p.kv_indices[kv_start + key];
        const uint8_t* kp8 = reinterpret_cast<const uint8_t*>(kbuf) + slot * p.kb_slot + kvh * p.kb_head + sch * 8;
        const uint8_t* vp8 = reinterpret_cast<const uint8_t*>(vbuf) + slot * p.vb_slot + kvh * p.vb_head + sch * 8;
        kreg[i] = cvt8_from_fp8<T>(*reinterpret_cast<const uint2*>(kp8));
        vreg[i] = cvt8_from_fp8<T>(*reinterpret_cast<const uint2*>(vp8));
        continue;
      }
      const T *kp, *vp;
      if (key < prefix) {
        const int64_t slot = p.kv_indices[kv_start + key];
        kp = kbuf + slot * p.kb_slot + kvh * p.kb_head;
        vp = vbuf + slot * p.vb_slot + kvh * p.vb_head;
      } else {
        const int64_t tok = q_start + key - prefix;
        kp = k_ext + tok * p.k_stride + (int64_t)kvh * D;
        vp = v_ext + tok * p.v_stride + (int64_t)kvh * D;
      }
      kreg[i] = ldvec<T, 8>(kp + sch * 8);
      vreg[i] = ldvec<T, 8>(vp + sch * 8);
    }
  };
  auto store_tile = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      stvec<T, 8>(ks + (srow + 16 * i) * XK_ROW + sch * 8, kreg[i]);
      stvec<T, 8>(vs + (srow + 16 * i) * XV_ROW + sch * 8, vreg[i]);
    }
  };

  f32x4 ot[8];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) ot[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, lsum = 0.f;

  // LDS read bases
  const T* k_rd = ks + j16 * XK_ROW + 8 * c4;                          // + (16 t) rows, + 32 s
  // transposed read: lane 16 c + 4 q + pp supplies row (4 c + q), columns 4 pp .. 4 pp + 3
  const T* v_rd = vs + (4 * c4 + (j16 >> 2)) * XV_ROW + 4 * (j16 & 3);  // + (32 ks2 + 16 half) rows, + 16 dt

  load_tile(0);
  for (int kt = 0; kt < n_tiles; ++kt) {
    __syncthreads();            // previous tile fully consumed
    store_tile();
    __syncthreads();
    if (kt + 1 < n_tiles) load_tile(kt + 1);

    // S^T tile: st[t][r] = score of key 64 kt + 16 t + 4 c + r for this lane's query;
    // k-step major with the four key sub-tiles as independent accumulators
    f32x4 st[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) st[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      frag kf[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) kf[t] = *reinterpret_cast<const frag*>(k_rd + (16 * t) * XK_ROW + 32 * s);
#pragma unroll
      for (int t = 0; t < 4; ++t) st[t] = Mfma<T>::run(kf[t], qf[s], st[t]);
    }
    const bool need_mask = kt * 64 + 63 > wave_min_limit;   // wave-uniform
    float mloc = -INFINITY;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float x = st[t][r] * qmul;
        if (need_mask && kt * 64 + 16 * t + 4 * c4 + r > my_limit) x = -INFINITY;
        st[t][r] = x;
        mloc = fmaxf(mloc, x);
      }
    mloc = max_xor<32>(max_xor<16>(mloc));
    const float mnew = fmaxf(m, mloc);
    const float ms = mnew == -INFINITY ? 0.f : mnew;
    const float alpha = raw_exp2(m - ms);
    m = mnew;
    float psum = 0.f;
    frag pb[2];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float pe = raw_exp2(st[t][r] - ms);
        // the denominator sums the fp32 weights; only the P.V operand is rounded to the value dtype
        // (as the reference's kernel: deno += sum(p), acc += dot(p.to(v.dtype), v),
        // triton_ops/extend_attention.py:190,200-201 and 271,281-282)
        psum += pe;
        pb[t >> 1][(t & 1) * 4 + r] = (T)pe;
      }
    lsum = lsum * alpha + psum;
    // multiplying by exactly 1 changes nothing: rescale only when some lane's maximum moved
    if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0) {
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) ot[dt] *= alpha;
    }

#pragma unroll
    for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        const auto lo = TrRead<T>::run(v_rd + (32 * k2) * XV_ROW + 16 * dt);
        const auto hi = TrRead<T>::run(v_rd + (32 * k2 + 16) * XV_ROW + 16 * dt);
        frag va;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          va[e] = lo[e];
          va[4 + e] = hi[e];
        }
        ot[dt] = Mfma<T>::run(va, pb[k2], ot[dt]);
      }
  }

  lsum = sum_xor<32>(sum_xor<16>(lsum));
  if (qrow < ext) {
    const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
    T* op = o_ext + ((int64_t)(q_start + qrow) * p.hq + h) * D + 4 * c4;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      Vec<T, 4> w;
#pragma unroll
      for (int r = 0; r < 4; ++r) w.v[r] = from_f32<T>(ot[dt][r] * inv);
      stvec<T, 4>(op + 16 * dt, w);
    }
  }
}

// ------------------------------------------------------------------------------------------
// The same prefill case on v_mfma_f32_32x32x16: a wave owns 32 query rows, a workgroup 128 rows of
// one query head (4 waves).  Why: with the 16x16x32 tile above every MFMA needs a fresh 1-KiB A
// fragment from LDS (K rows for the scores, V^T for the outputs), and twelve waves' fragment reads
// take as many LDS cycles as their MFMAs take matrix-core cycles; a 32x32x16 MFMA does twice the
// work on a fragment of the same size, and the loop issues half as many MFMA + LDS instructions.
//   S^T = K . Q^T    : A = 32 key rows (ds_read_b128), B = the wave's 32 queries, kept in registers
//                      (8 k-steps of 16 features).  Lane (query j = l & 31, h = l >> 5) then owns the
//                      scores of ITS query for keys 8 (i >> 2) + 4 h + (i & 3) of each 32-key half.
//   O^T += V^T . P^T : registers 8 u' .. 8 u' + 7 of a score tile, rounded to T, ARE the B fragment of
//                      the 16-key step u (element e <-> key 16 u + 8 (e >> 2) + 4 h + (e & 3)); the A
//                      fragment (V^T in that key order) comes from two transposed reads of the
//                      row-major V tile.
// K and V tiles are plain 256-byte rows with the chunk index XOR-ed by ((row & 3) << 2 | (row >> 2) & 3):
// conflict-free for the 32-row fragment reads and for the transposed reads.
// Workgroup -> work mapping: a 1-D grid; consecutive workgroups go round-robin over the 8 XCDs, so
// workgroup L serves the (sequence, kv head) pair number (L & 7) + 8 * ((L >> 3) / per_pair): every
// query block and every query head of a pair runs on ONE XCD and finds the pair's K/V in that XCD's
// L2 after the first touch (the 2-D grid fetched each K/V row from HBM 2.8 times).
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ int xor_image_off(int row, int ch) {   // bytes; ch = 16-byte chunk 0..15 of a 256-byte row
  return 256 * row + 16 * (ch ^ (((row & 3) << 2) | ((row >> 2) & 3)));
}

// DQ: query / key head dimension, 128 or 192 (the multi-head form of MLA prefill: 128 nope + 64 rope features
// against 128-wide values).  Features 128 .. 191 of the K tile are a second 256-byte-row image (half of each row
// used) with the same chunk XOR, so the fragment reads of score steps 8 .. 11 are as conflict-free as the others.
// LATENT: no cached prefix; the heads' keys (features 0 .. 127) and values come interleaved per token and head out of one
// projection of the latent, the keys' features 128 .. 191 from one row per token that the heads share, and the queries'
// features 128 .. 191 are rotated here, in fp32 and rounded to T, as the absorbed kernels do it.
// D: value head dimension.  At 64 the rows of the tile images are half used (the XOR spreads their eight chunks over the whole
// 256 bytes), and P.V takes each weight as the sum of three 16-bit numbers, for the vector-ALU kernel that serves other forms of this size
// multiplies by fp32 weights: in bf16 they hold all 24 bits of a weight, in fp16, where the weights are scaled to 2^15 so that the terms of
// small ones are no subnormals, all down to 2^-16 and what lies above 2^-40 further down.
// MASK: a custom mask instead of the causal rule (and of a prefix without conditions, unless skip_prefix_custom_mask): a row
// [prefix + new tokens] of bytes per query.  The arithmetic is the causal launch's, so that a triangle for a mask gives its bits.
// careful (D = 64): value rows may hold infinities and NaN, which no product with a weight of zero may meet (keys that the query does not
// see) nor with a weight's lower terms.  The images then hold the rows without them, and beside them, in the half that is free, the rows
// as they are, from which they are added for the queries that see their key.  Returns (the same in all threads) whether a result is no number.
// DIRECT: the load unit writes the K/V images itself (buffer loads to LDS), the next tile's into a second stage while this one is worked on: one
// barrier a tile, and no registers, addresses of 64 bits or LDS stores for it.  A quarter of a launch was the tile's way through
// registers (1 x 4000 tokens, 32 / 8 heads: 168 us, 127 without any loads after the first tile; 4 x 490 on 1750 cached 90 and 63).  Rows of a tile are
// addressed with 32 bits: from the head's first cached row, or from the tile's own first row of this launch.  (global_load_lds would do without
// that, but the compiler takes it for a flat access and then waits for every LDS read behind it to the last one: 173 us.)
// us a launch, 16-bit rows: registers | DIRECT | and the weights of a k-step made beside the MFMAs of the one before, MFMAs at a raised wave
// priority: 5 x 1100 ragged 49.5 | 45.5 | 43.5; 4 x 515 on 1999 ragged 93.7 | 81.4 | 79.0; 192-wide latents of 4 x 2048
// tokens, 32 heads 238 | 213 | 204, 16 heads 131 | 114 | 108; 1 x 4000 179 | 163 | 155 (a slower card than the one of the figures above; on a third one
// 1 x 4000 167 | 146, 4 x 490 on 1750 95 | 82, 8 x 200 on 3000 134 | 109, registers | now).
// SPLIT: gridDim.y workgroups share the block's key tiles, in runs of at least SPLIT_TILES; extend_split_merge_kernel adds their sums.
constexpr int SPLIT_TILES = 4;
template <int DQ> constexpr int direct_stage_bytes() { return 2 * 64 * 256 + (DQ > 128 ? 64 * 128 : 0); }
// A buffer of 4 GiB from p on, and 16 bytes a lane of it to LDS (l and the lanes behind it)
__device__ __forceinline__ auto wide_rsrc(const void* p) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, -1, 0x00020000); }
__device__ __forceinline__ void buffer_to_lds16(__amdgpu_buffer_rsrc_t r, char* l, unsigned off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)l, 16, (int)off, 0, 0, 0);
}
template <typename T, bool KV8, int DQ, bool LATENT = false, int D = 128, bool MASK = false, bool SPLIT = false, bool DIRECT = false>
__device__ __forceinline__ bool extend_attn_mfma32_body(
    const T* __restrict__ q_ext, const T* __restrict__ k_ext, const T* __restrict__ v_ext, T* __restrict__ o_ext,
    const T* __restrict__ kbuf, const T* __restrict__ vbuf, const ExtendParams& p, int nqb, int npairs, bool careful = false) {
  constexpr int NS = DQ / 16;     // score k-steps
  constexpr bool WIDE = DQ > 128;
  constexpr bool TERMS = D == 64;
  constexpr float P_UP = TERMS && std::is_same<T, f16_t>::value ? 0x1p15f : 1.f;   // weights up to 2^15: terms of small ones stay normal
  constexpr int CH = D / 8, SR = 256 / CH, NI = 64 / SR;   // 16-byte chunks of a row; rows staged at once, and how often
  constexpr int ND = D / 32;      // 32-feature tiles of the output
  static_assert((D == 128 && (DQ == 128 || (DQ == 192 && !KV8))) || (D == 64 && DQ == 64), "64, 128, or 192 + 128 over a 16-bit cache");
  using frag = typename Mfma32<T>::frag;
  static_assert(!DIRECT || (D == 128 && !KV8 && (DQ == 128 || LATENT)), "16-bit rows, from the cache or of this launch");
  constexpr int STAGE = direct_stage_bytes<DQ>();
  extern __shared__ __attribute__((aligned(16))) char sm_direct[];
  __shared__ __attribute__((aligned(16))) char sm_images[DIRECT ? 16 : (WIDE ? 3 : 2) * 64 * 256 + 16];
  char* const ks = DIRECT ? sm_direct : sm_images;
  char* const vs = ks + 64 * 256;
  char* const ks2 = vs + 64 * 256;

  int tid = (int)threadIdx.x;
  if (careful) asm volatile("" : "+v"(tid));    // (addresses of its own: the first pass's would be kept for it in scratch memory)
  const int G = p.hq / p.hkv;
  const int per_pair = G * nqb;
  const int slot = blockIdx.x >> 3;
  const int pair = (blockIdx.x & 7) + 8 * (slot / per_pair);
  if (pair >= npairs) return false;
  const int t_in_pair = slot % per_pair;
  const int qb = nqb - 1 - t_in_pair / G;          // long (late) blocks first
  const int b = pair / p.hkv, kvh = pair % p.hkv, h = kvh * G + t_in_pair % G;
  const int q_start = LATENT ? p.seg_start[b] : p.qo_indptr[b];
  const int ext = LATENT ? p.seg_len[b] : p.qo_indptr[b + 1] - q_start;
  const int kv_start = LATENT ? 0 : p.kv_indptr[b];
  const int prefix = LATENT ? 0 : p.kv_indptr[b + 1] - kv_start;
  const int r0 = qb * 128;
  if (r0 >= ext) return false;   // whole workgroup: EXEC stays full for the transposed reads below

  const int lane = tid & 63, wave = tid >> 6;
  const int j32 = lane & 31, hh = lane >> 5;
  const int qrow = r0 + wave * 32 + j32;                  // this lane's query (row of the extend part)
  const int qrow_c = qrow < ext ? qrow : ext - 1;
  const float qmul = p.sm_scale * kLog2eE;

  // B operand of S^T: Q[qrow][16 s + 8 h + 0..7]
  frag qf[NS];
  {
    const T* qp = q_ext + (int64_t)(q_start + qrow_c) * p.q_stride + (int64_t)h * DQ + 8 * hh;
#pragma unroll
    for (int s = 0; s < NS; ++s) qf[s] = *reinterpret_cast<const frag*>(qp + 16 * s);
  }
  if constexpr (LATENT) {
    // lane's features 16 (s - 8) + 8 hh + 0 .. 7 of the rope part: pairs of neighbours lie in one fragment, pairs (i, i + 32)
    // in fragments s and s + 2
    const float pos = (float)p.positions[q_start + qrow_c];
    auto turn = [&](int i, T& a, T& c) {
      float sn, cs;
      sincosf(pos * p.inv_freq[i], &sn, &cs);
      sn *= p.rot_mag;
      cs *= p.rot_mag;
      const float u = to_f32(a), w = to_f32(c);
      a = from_f32<T>(u * cs - w * sn);
      c = from_f32<T>(w * cs + u * sn);
    };
    if (p.interleaved) {
#pragma unroll
      for (int s = 8; s < NS; ++s)
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          const int i = (16 * (s - 8) + 8 * hh + e) >> 1;
          if (2 * i < p.rot_dims) {
            T a = qf[s][e], c = qf[s][e + 1];
            turn(i, a, c);
            qf[s][e] = a;
            qf[s][e + 1] = c;
          }
        }
    } else if (p.rot_dims == 64) {
#pragma unroll
      for (int s = 8; s < 10; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          T a = qf[s][e], c = qf[s + 2][e];
          turn(16 * (s - 8) + 8 * hh + e, a, c);
          qf[s][e] = a;
          qf[s + 2][e] = c;
        }
    }
  }

  const int last_row = min(r0 + 127, ext - 1);
  const bool causal = LATENT || (!MASK && p.is_causal);
  const int total = causal ? prefix + last_row + 1 : prefix + ext;
  int n_tiles = (total + 63) / 64, first_tile = 0;
  if constexpr (SPLIT) {
    const int run = max((n_tiles + (int)gridDim.y - 1) / (int)gridDim.y, SPLIT_TILES);
    first_tile = run * (int)blockIdx.y;
    if (first_tile >= n_tiles) {   // (workgroup-uniform) no weights: the merge reads no sums
      if (hh == 0 && qrow < ext) p.part_ml[((int64_t)blockIdx.y * p.rows + q_start + qrow) * p.hq + h] = make_float2(-INFINITY, 0.f);
      return false;
    }
    n_tiles = min(n_tiles, first_tile + run);
  }
  const int my_limit = causal ? prefix + qrow_c : prefix + ext - 1;   // last visible key of this lane's query
  const int wave_min_limit = causal ? prefix + min(r0 + wave * 32, ext - 1) : prefix + ext - 1;
  const int wave_max_limit = causal ? prefix + min(r0 + wave * 32 + 31, ext - 1) : prefix + ext - 1;
  const bool no_rows = r0 + __builtin_amdgcn_readfirstlane(wave) * 32 >= ext;
  const uint8_t* mask_row = MASK ? p.custom_mask + p.mask_indptr[b] + (int64_t)qrow_c * (prefix + ext) : nullptr;

  // tile staging: thread -> rows tid / CH + SR i, 16-B chunk tid % CH
  const int srow = tid / CH, sch = tid % CH;
  // kreg2: chunk sch2 of features 128 and up of two of kreg's four rows, so that a paged row's slot is read once and every thread
  // has a part.  16 requests x 64 tokens on 2000 cached, 16 heads, 133 us, 2048 tokens on none 60; with rows of another deal,
  // whose slots are read again, 169 and 67; in the threads with sch < 8 alone 152 and 76.  LATENT, where these features are
  // rows of their own: eight neighbours a load (a whole step of Silatar 1 % less than in the first deal).
  Vec<T, 8> kreg[NI], vreg[NI], kreg2[WIDE ? 2 : 1];
  const int odd2 = sch >> 3, sch2 = sch & 7, srow2 = LATENT ? tid >> 3 : srow + 16 * odd2;   // rows srow2 + 32 j
  const T* k_lin = k_ext + (int64_t)(q_start - prefix + srow) * p.k_stride + (int64_t)kvh * (LATENT ? p.kv_head : DQ) + sch * 8;
  const T* v_lin = v_ext + (int64_t)(q_start - prefix + srow) * p.v_stride + (int64_t)kvh * (LATENT ? p.kv_head : D) + sch * 8;
  const T* r_lin = LATENT ? (const T*)p.k_rope + (int64_t)(q_start + srow2) * p.k_rope_stride + sch2 * 8
                          : k_ext + (int64_t)(q_start - prefix + srow2) * p.k_stride + (int64_t)kvh * DQ + 128 + sch2 * 8;
  const int64_t r_stride = LATENT ? p.k_rope_stride : p.k_stride;
  // Cache slots of the thread's rows of the next tile, read a tile ahead: otherwise every wave stands at the head of its tile for the
  // slots before it can request the rows behind them.  32 / 8 heads, us a launch: 4 x 490 tokens on 1750 cached 165 -> 131, 6 x 500
  // on 2900 278 -> 209, 1 x 65 on 3000 106 -> 82; without a prefix as before.
  int32_t next_slot[NI];
  auto load_slots = [&](int kt) {
    if (kt * 64 >= prefix) return;   // (workgroup-uniform)
#pragma unroll
    for (int i = 0; i < NI; ++i) next_slot[i] = p.kv_indices[kv_start + min(kt * 64 + srow + SR * i, prefix - 1)];
  };
  auto load_tile = [&](int kt) {
    if (kt * 64 >= prefix && kt * 64 + 63 < total) {   // whole tile in the extend part (workgroup-uniform)
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int64_t key = kt * 64 + SR * i;
        kreg[i] = ldvec<T, 8>(k_lin + key * p.k_stride);
        vreg[i] = ldvec<T, 8>(v_lin + key * p.v_stride);
      }
      if constexpr (WIDE) {
#pragma unroll
        for (int j = 0; j < 2; ++j) kreg2[j] = ldvec<T, 8>(r_lin + (int64_t)(kt * 64 + 32 * j) * r_stride);
      }
      return;
    }
    if constexpr (LATENT) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t key = min(kt * 64 + srow + 16 * i, total - 1) - srow;
        kreg[i] = ldvec<T, 8>(k_lin + key * p.k_stride);
        vreg[i] = ldvec<T, 8>(v_lin + key * p.v_stride);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) kreg2[j] = ldvec<T, 8>(r_lin + (int64_t)(min(kt * 64 + srow2 + 32 * j, total - 1) - srow2) * r_stride);
      return;
    }
    const T* row2[WIDE ? 4 : 1];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      int key = kt * 64 + srow + SR * i;
      key = key < total ? key : total - 1;
      if (KV8 && key < prefix) {
        const int64_t slot_ = next_slot[i];
        const uint8_t* kp8 = reinterpret_cast<const uint8_t*>(kbuf) + slot_ * p.kb_slot + kvh * p.kb_head + sch * 8;
        const uint8_t* vp8 = reinterpret_cast<const uint8_t*>(vbuf) + slot_ * p.vb_slot + kvh * p.vb_head + sch * 8;
        kreg[i] = cvt8_from_fp8<T>(*reinterpret_cast<const uint2*>(kp8));
        vreg[i] = cvt8_from_fp8<T>(*reinterpret_cast<const uint2*>(vp8));
        continue;
      }
      const T *kp, *vp;
      if (key < prefix) {
        const int64_t slot_ = next_slot[i];
        kp = kbuf + slot_ * p.kb_slot + kvh * p.kb_head;
        vp = vbuf + slot_ * p.vb_slot + kvh * p.vb_head;
      } else {
        const int64_t tok = q_start + key - prefix;
        kp = k_ext + tok * p.k_stride + (int64_t)kvh * DQ;
        vp = v_ext + tok * p.v_stride + (int64_t)kvh * D;
      }
      kreg[i] = ldvec<T, 8>(kp + sch * 8);
      vreg[i] = ldvec<T, 8>(vp + sch * 8);
      if constexpr (WIDE) row2[i] = kp;
    }
    if constexpr (WIDE) {
#pragma unroll
      for (int j = 0; j < 2; ++j) kreg2[j] = ldvec<T, 8>((odd2 ? row2[2 * j + 1] : row2[2 * j]) + 128 + sch2 * 8);
    }
  };
  auto store_tile = [&]() {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int off = xor_image_off(srow + SR * i, sch);
      *reinterpret_cast<Vec<T, 8>*>(ks + off) = kreg[i];
      if (TERMS && careful) {
        *reinterpret_cast<Vec<T, 8>*>(vs + xor_image_off(srow + SR * i, sch + 8)) = vreg[i];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (!(fabsf(to_f32(vreg[i].v[j])) < INFINITY)) vreg[i].v[j] = from_f32<T>(0.f);
      }
      *reinterpret_cast<Vec<T, 8>*>(vs + off) = vreg[i];
    }
    if constexpr (WIDE) {
#pragma unroll
      for (int j = 0; j < 2; ++j) *reinterpret_cast<Vec<T, 8>*>(ks2 + xor_image_off(srow2 + 32 * j, sch2)) = kreg2[j];
    }
  };

  // DIRECT: rows srow + 16 i of a tile go to the image's rows 4 wave + 16 i .. + 3 (1 KiB a wave, in the lanes' order); lane sch of a row fetches the
  // chunk that belongs there.  Rows of this launch: the tile's first row is the buffer's base; cached ones: the head's first.  A wave that has a
  // slot further away than the offsets reach (the launcher goes by the slots that the caller says there are) takes its rows through registers.
  [[maybe_unused]] const unsigned gch = (sch ^ (((srow & 3) << 2) | ((srow >> 2) & 3))) * 16u, gch2 = (sch2 ^ ((srow2 >> 1) & 7)) * 16u;
  [[maybe_unused]] const int wave_u = __builtin_amdgcn_readfirstlane(tid >> 6);
  [[maybe_unused]] auto direct_tile = [&](int kt, int stage) {
    char* const dst = sm_direct + stage * STAGE + 1024 * wave_u;
    const int64_t tok = (int64_t)q_start - prefix + kt * 64;
    const int left = total - kt * 64;      // rows of the tile that exist
    if (LATENT || kt * 64 >= prefix) {
      const auto rk = wide_rsrc(k_ext + tok * p.k_stride + (int64_t)kvh * (LATENT ? p.kv_head : DQ));
      const auto rv = wide_rsrc(v_ext + tok * p.v_stride + (int64_t)kvh * (LATENT ? p.kv_head : D));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = min(srow + 16 * i, left - 1);
        buffer_to_lds16(rk, dst + 4096 * i, row * (unsigned)p.k_stride * 2 + gch);
        buffer_to_lds16(rv, dst + 16384 + 4096 * i, row * (unsigned)p.v_stride * 2 + gch);
      }
      if constexpr (LATENT) {
        const auto rr = wide_rsrc((const T*)p.k_rope + tok * p.k_rope_stride);
#pragma unroll
        for (int j = 0; j < 2; ++j) buffer_to_lds16(rr, dst + 32768 + 4096 * j, min(srow2 + 32 * j, left - 1) * (unsigned)p.k_rope_stride * 2 + gch2);
      }
    } else if (kt * 64 + 64 <= prefix &&
               __builtin_amdgcn_ballot_w64(max(max((uint32_t)next_slot[0], (uint32_t)next_slot[1]), max((uint32_t)next_slot[2], (uint32_t)next_slot[3])) >=
                                           p.near_slots) == 0) {
      const auto rk = wide_rsrc(kbuf + kvh * p.kb_head), rv = wide_rsrc(vbuf + kvh * p.vb_head);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        buffer_to_lds16(rk, dst + 4096 * i, next_slot[i] * (unsigned)(p.kb_slot * 2) + gch);
        buffer_to_lds16(rv, dst + 16384 + 4096 * i, next_slot[i] * (unsigned)(p.vb_slot * 2) + gch);
      }
    } else {   // the tile that holds the prefix's last rows and the first new ones, or rows far away: through registers
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = min(kt * 64 + srow + 16 * i, total - 1);
        const bool old = key < prefix;
        const T* kp = old ? kbuf + (int64_t)next_slot[i] * p.kb_slot + kvh * p.kb_head : k_ext + (int64_t)(q_start + key - prefix) * p.k_stride + (int64_t)kvh * DQ;
        const T* vp = old ? vbuf + (int64_t)next_slot[i] * p.vb_slot + kvh * p.vb_head : v_ext + (int64_t)(q_start + key - prefix) * p.v_stride + (int64_t)kvh * D;
        const Vec<T, 8> kx = ldvec<T, 8>(kp + gch / 2), vx = ldvec<T, 8>(vp + gch / 2);
        *reinterpret_cast<Vec<T, 8>*>(dst + 4096 * i + 16 * lane) = kx;
        *reinterpret_cast<Vec<T, 8>*>(dst + 16384 + 4096 * i + 16 * lane) = vx;
      }
    }
  };

  f32x16 ot[ND];
#pragma unroll
  for (int dt = 0; dt < ND; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) ot[dt][i] = 0.f;
  float m = -INFINITY, lsum = 0.f;

  // K fragment of (32-key half hf, k-step s): row 32 hf + j32, chunk 2 s + h.  The XOR term depends on
  // (row & 15) only, i.e. on the lane: chunk ^ fx = (2 s) ^ (h ^ fx).
  const int fx = ((j32 & 3) << 2) | ((j32 >> 2) & 3);
  const int kcx = hh ^ fx;
  int cur = 0;                                              // DIRECT: the tile's stage
  const char* k_rd = ks + 256 * j32;                        // + 8192 hf + 16 * ((2 s) ^ kcx)
  const char* k_rd2 = ks2 + (DIRECT ? 128 : 256) * j32;     // steps 8 .. : chunk 2 (s - 8) + h of the second image
  auto k_frag = [&](int s_, int hf) -> frag {
    if (DIRECT && WIDE && s_ >= 8) return *reinterpret_cast<const frag*>(k_rd2 + cur + 4096 * hf + 16 * ((2 * (s_ & 7)) ^ (hh ^ ((j32 >> 1) & 7))));
    const char* base = ((WIDE && s_ >= 8) ? k_rd2 : k_rd) + cur;
    return *reinterpret_cast<const frag*>(base + 8192 * hf + 16 * ((2 * (s_ & 7)) ^ kcx));
  };
  // V^T fragment of (d tile dt, 16-key step u): lane group (l >> 4) = 2 h + dhalf serves features
  // 32 dt + 16 dhalf + 0..15; lane 4 q + pp of the group supplies row 16 u (+ 8) + 4 h + q, features 4 pp..4 pp + 3
  const int l16 = lane & 15, dhalf = (lane >> 4) & 1, tq = l16 >> 2, tpp = l16 & 3;
  const int vrow = 4 * hh + tq;                             // + 16 u (+ 8): (row & 3) = tq, (row >> 2) & 3 = (h + 2 hi) & 3
  const int vf_lo = (tq << 2) | (hh & 3), vf_hi = (tq << 2) | ((hh + 2) & 3);
  const int vch = 2 * dhalf + (tpp >> 1);                   // + 4 dt
  const char* v_rd = vs + 256 * vrow + 8 * (tpp & 1);

  // careful: the tile's values that are no numbers, for the queries that see their keys
  auto add_odd_values = [&](int kt) {
    bool odd = false;      // in row `lane` of the tile
#pragma unroll
    for (int ch = 8; ch < 16; ++ch) {
      const Vec<T, 8> x = *reinterpret_cast<const Vec<T, 8>*>(vs + xor_image_off(lane, ch));
#pragma unroll
      for (int j = 0; j < 8; ++j) odd |= !(fabsf(to_f32(x.v[j])) < INFINITY);
    }
    for (uint64_t rows = __builtin_amdgcn_ballot_w64(odd); rows != 0; rows &= rows - 1) {
      const int row = __builtin_ctzll(rows), key = kt * 64 + row;
      const bool seen = key <= my_limit && (!MASK || mask_row[min(key, my_limit)] != 0 || (key < prefix && p.skip_prefix_custom_mask));
#pragma unroll
      for (int dt = 0; dt < ND; ++dt)
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) {      // the lane's features, as they are stored below
          const Vec<T, 4> x = *reinterpret_cast<const Vec<T, 4>*>(vs + xor_image_off(row, 8 + 4 * dt + rq) + 8 * hh);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float v = to_f32(x.v[r]);
            ot[dt][4 * rq + r] += seen && !(fabsf(v) < INFINITY) ? v : 0.f;
          }
        }
    }
  };

  if constexpr (DIRECT) {
    if (!LATENT) load_slots(first_tile);
    direct_tile(first_tile, 0);
    if (!LATENT) load_slots(first_tile + 1);
  } else if (!careful) {
    if (!LATENT) load_slots(first_tile);
    load_tile(first_tile);
    if (!LATENT) load_slots(first_tile + 1);
  }
  for (int kt = first_tile; kt < n_tiles; ++kt) {
    if constexpr (DIRECT) {
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0x0070);   // vmcnt(0) lgkmcnt(0): this wave's part of the tile and the next one's slots are there
      __builtin_amdgcn_s_barrier();         // everybody's part is, and the other stage has been read
      __builtin_amdgcn_sched_barrier(0);
      const int stage = (kt - first_tile) & 1;
      cur = stage * STAGE;
      if (kt + 1 < n_tiles) direct_tile(kt + 1, stage ^ 1);
      if (!LATENT) load_slots(kt + 2);
      __builtin_amdgcn_sched_barrier(0);
    } else {
      __syncthreads();            // previous tile fully consumed
      if (careful) {              // (nothing ahead: no registers spilled for a rare path)
        load_slots(kt);
        load_tile(kt);
      }
      store_tile();
      __syncthreads();
      if (!careful) {
        if (kt + 1 < n_tiles) load_tile(kt + 1);
        if (!LATENT) load_slots(kt + 2);
      }
    }
    if (kt * 64 > wave_max_limit || no_rows) continue;   // nothing of the tile counts for any query of this wave (wave-uniform)

    f32x16 st[2];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int i = 0; i < 16; ++i) st[hf][i] = 0.f;
    // LDS fragment reads run AHEAD of the MFMAs that use them (register rings, fenced): written
    // read-MFMA-read-MFMA, hipcc keeps that order and every MFMA waits a full LDS round trip
    // (>= 64 cycles against the MFMA's 32).
    frag kr[3][2];   // K fragments of k-steps s, s + 1, s + 2
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      kr[s][0] = k_frag(s, 0);
      kr[s][1] = k_frag(s, 1);
    }
    // the first V^T fragments too: the tile is already in LDS, and the softmax below covers their latency
    typename TrRead<T>::v4 vlo[4], vhi[4];   // ring of four (u, dt) fragments
    auto v_read = [&](int i, int slot_) {
      const int u = i / ND, dt = i % ND;
      const int ch = 4 * dt + vch;
      vlo[slot_] = TrRead<T>::run(reinterpret_cast<const T*>(v_rd + cur + 256 * (16 * u) + 16 * (ch ^ vf_lo)));
      vhi[slot_] = TrRead<T>::run(reinterpret_cast<const T*>(v_rd + cur + 256 * (16 * u + 8) + 16 * (ch ^ vf_hi)));
    };
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if (s + 2 < NS) {
        kr[(s + 2) % 3][0] = k_frag(s + 2, 0);
        kr[(s + 2) % 3][1] = k_frag(s + 2, 1);
      } else if (s == NS - 2) {
        v_read(0, 0);
        v_read(1, 1);
      } else {
        v_read(2, 2);
        v_read(3, 3);
      }
      __builtin_amdgcn_sched_barrier(0);
      st[0] = Mfma32<T>::run(kr[s % 3][0], qf[s], st[0]);
      st[1] = Mfma32<T>::run(kr[s % 3][1], qf[s], st[1]);
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(0);
    // Softmax on the raw scores: the scale (sm_scale * log2 e > 0, checked by the launcher) commutes with
    // the maximum and folds into the exponent's multiply-add.  Only tiles that cross the wave's diagonal
    // pay for masking (two instructions per score: the key offsets within a tile are compile-time
    // constants, the lane's limit is one subtraction per tile); the branch is wave-uniform.
    float mloc = -INFINITY, least = INFINITY;
    if constexpr (TERMS) {
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int i = 0; i < 16; ++i) least = fminf(least, st[hf][i]);
    }
    if constexpr (MASK) {
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = kt * 64 + 4 * hh + 32 * hf + 8 * (i >> 2) + (i & 3);
          const bool seen = mask_row[min(key, my_limit)] != 0 || (key < prefix && p.skip_prefix_custom_mask);
          const float x = key > my_limit || !seen ? -INFINITY : st[hf][i];
          st[hf][i] = x;
          mloc = fmaxf(mloc, x);
        }
    } else if (kt * 64 + 63 > wave_min_limit) {
      const int lim = my_limit - kt * 64 - 4 * hh;
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float x = (32 * hf + 8 * (i >> 2) + (i & 3)) > lim ? -INFINITY : st[hf][i];
          st[hf][i] = x;
          mloc = fmaxf(mloc, x);
        }
    } else {
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int i = 0; i < 16; ++i) mloc = fmaxf(mloc, st[hf][i]);
    }
    mloc = max_xor<32>(mloc);
    const float mnew = fmaxf(m, mloc * qmul);
    const float ms = mnew == -INFINITY ? 0.f : mnew;
    const float alpha = TERMS ? exp2f(m - ms) : raw_exp2(m - ms);
    m = mnew;
    float psum = 0.f;
    frag pb[TERMS ? 3 : 4];
    // the lane's weights 2 j and 2 j + 1 of k-step u
    [[maybe_unused]] auto weights2 = [&](int u, int j) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float pe = raw_exp2(__builtin_fmaf(st[u >> 1][8 * (u & 1) + 2 * j + e], qmul, -ms));
        psum += pe;                          // fp32 weights in the denominator, T-rounded weights in P.V
        pb[u][2 * j + e] = (T)pe;
      }
    };
    if constexpr (!TERMS) {
#pragma unroll
      for (int j = 0; j < 4; ++j) weights2(0, j);
    }
    // TERMS: the lane's eight weights of k-step u.  Those below 2^-126 count: exp2f, in a tile that may have one (wave-uniform); the bare
    // instruction makes them zero.
    const bool deep = TERMS && __builtin_amdgcn_ballot_w64(__builtin_fmaf(least, qmul, -ms) < -126.f) != 0;
    auto terms = [&](int u) {
      float pe[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) pe[i] = __builtin_fmaf(st[u >> 1][8 * (u & 1) + i], qmul, -ms);
      if (deep) {
#pragma unroll
        for (int i = 0; i < 8; ++i) pe[i] = exp2f(pe[i]);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) pe[i] = raw_exp2(pe[i]);
      }
      unsigned w[3][4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float a = pe[2 * i], c = pe[2 * i + 1];
        psum += a;
        psum += c;
        a *= P_UP;
        c *= P_UP;
        w[0][i] = Pair16<T>::pack(a, c);
        a -= Pair16<T>::first(w[0][i]);
        c -= Pair16<T>::second(w[0][i]);
        w[1][i] = Pair16<T>::pack(a, c);
        w[2][i] = Pair16<T>::pack(a - Pair16<T>::first(w[1][i]), c - Pair16<T>::second(w[1][i]));
      }
#pragma unroll
      for (int t = 0; t < 3; ++t) pb[t] = __builtin_bit_cast(frag, w[t]);
    };
    if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0) {
#pragma unroll
      for (int dt = 0; dt < ND; ++dt) ot[dt] *= alpha;
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = 0; i < 4 * ND; ++i) {   // (u, dt) = (i / ND, i % ND); fragment i + 4 is requested right behind MFMA i
      frag va;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        va[e] = vlo[i & 3][e];
        va[4 + e] = vhi[i & 3][e];
      }
      if constexpr (TERMS) {
        if (i % ND == 0) terms(i / ND);
#pragma unroll
        for (int t = 0; t < 3; ++t) ot[i % ND] = Mfma32<T>::run(va, pb[t], ot[i % ND]);
      } else {
        ot[i % ND] = Mfma32<T>::run(va, pb[i / ND], ot[i % ND]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (i + 4 < 4 * ND) {
        v_read(i + 4, i & 3);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (!TERMS) {
        if (i / ND < 3) {
          weights2(i / ND + 1, i % ND);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    __builtin_amdgcn_s_setprio(0);
    if constexpr (!TERMS) lsum = lsum * alpha + psum;
    if constexpr (TERMS) {
      lsum = lsum * alpha + psum;
      if (careful) add_odd_values(kt);
    }
  }

  lsum = sum_xor<32>(lsum);
  bool odd = false;
  if (TERMS && !careful) {
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) odd |= !(fabsf(ot[dt][i]) < INFINITY);
    int* flags = reinterpret_cast<int*>(ks2);      // (unused otherwise)
    odd = __builtin_amdgcn_ballot_w64(odd) != 0;
    if (lane == 0) flags[wave] = odd;
    __syncthreads();
    odd = (flags[0] | flags[1] | flags[2] | flags[3]) != 0;
  }
  if (SPLIT) {
    if (qrow < ext) {
      const int64_t at = ((int64_t)blockIdx.y * p.rows + q_start + qrow) * p.hq + h;
      if (hh == 0) p.part_ml[at] = make_float2(m, lsum * P_UP);
      float* op = p.part + at * D + 4 * hh;
#pragma unroll
      for (int dt = 0; dt < ND; ++dt)
#pragma unroll
        for (int rq = 0; rq < 4; ++rq)
          *reinterpret_cast<float4*>(op + 32 * dt + 8 * rq) =
              make_float4(ot[dt][4 * rq], ot[dt][4 * rq + 1], ot[dt][4 * rq + 2], ot[dt][4 * rq + 3]);
    }
  } else if (qrow < ext) {
    const float inv = lsum > 0.f ? 1.f / (lsum * P_UP) : 0.f;
    T* op = o_ext + ((int64_t)(q_start + qrow) * p.hq + h) * D + 4 * hh;
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        Vec<T, 4> w;
#pragma unroll
        for (int r = 0; r < 4; ++r) w.v[r] = from_f32<T>(ot[dt][4 * rq + r] * inv);
        stvec<T, 4>(op + 32 * dt + 8 * rq, w);
      }
  }
  return odd;
}

// Two workgroups per CU (256 registers per lane) at head dimension 128; the 192-wide variant over a paged prefix needs
// ~270 registers and runs one workgroup per CU instead of spilling (measured at 4 x 4096 tokens x 16 heads: 470 TFLOP/s
// against 412 with 24 spilled registers at two workgroups per CU; issuing the next tile's loads behind the score phase
// spills more).
template <typename T, bool KV8, bool SPLIT, bool DIRECT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void extend_attn_mfma32_kernel(
    const T* __restrict__ q_ext, const T* __restrict__ k_ext, const T* __restrict__ v_ext, T* __restrict__ o_ext,
    const T* __restrict__ kbuf, const T* __restrict__ vbuf, ExtendParams p, int nqb, int npairs) {
  extend_attn_mfma32_body<T, KV8, 128, false, 128, false, SPLIT, DIRECT>(q_ext, k_ext, v_ext, o_ext, kbuf, vbuf, p, nqb, npairs);
}
// Head dimension 64 needs 190 registers: two workgroups per CU (three, with a few registers in scratch memory, took longer: 4 x 340 tokens on 1180
// cached 80 us).  Bound by the softmax's instructions (about fifteen per score, five of them the weights' three terms, beside an MFMA
// cycle).  32 / 8 heads in bf16, us a launch, vector-ALU kernel -> this one (two terms, no weight below 2^-126): 4 x 340 tokens on 1180
// cached 378 -> 68 (54), 704 + 430 tokens on none 121 -> 24 (20), 4000 on none 1493 -> 170 (136), 65 on 3000 510 -> 84 (73), 70 on none 24 -> 9
// (9); fp8 cache, 3 x 197 on 1614 478 -> 61 (53).  The heads of a group packed into the rows (less of the triangle's edge in vain) was
// no faster.
template <typename T, bool KV8, bool MASK, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void extend_attn_mfma32_d64_kernel(
    const T* __restrict__ q_ext, const T* __restrict__ k_ext, const T* __restrict__ v_ext, T* __restrict__ o_ext,
    const T* __restrict__ kbuf, const T* __restrict__ vbuf, ExtendParams p, int nqb, int npairs) {
  if (extend_attn_mfma32_body<T, KV8, 64, false, 64, MASK, SPLIT>(q_ext, k_ext, v_ext, o_ext, kbuf, vbuf, p, nqb, npairs)) {
    __syncthreads();
    extend_attn_mfma32_body<T, KV8, 64, false, 64, MASK, SPLIT>(q_ext, k_ext, v_ext, o_ext, kbuf, vbuf, p, nqb, npairs, true);
  }
}

// Adds the splits' sums: D / 4 lanes a (row, head), the sums of four splits in flight.
template <typename T, int D>
__global__ __launch_bounds__(256) void extend_split_merge_kernel(T* __restrict__ o, const float* __restrict__ part,
                                                                 const float2* __restrict__ ml, const int32_t* __restrict__ qo_indptr, int64_t bs,
                                                                 int64_t items, int hq, int splits) {
  constexpr int L = D / 4;
  const int64_t at = (int64_t)blockIdx.x * (256 / L) + threadIdx.x / L;
  if (at >= items || at < (int64_t)qo_indptr[0] * hq || at >= (int64_t)qo_indptr[bs] * hq) return;   // rows of no sequence stay as they are
  const int c = 4 * (threadIdx.x % L);
  float top = -INFINITY;
  for (int s = 0; s < splits; ++s) top = fmaxf(top, ml[s * items + at].x);
  const float ms = top == -INFINITY ? 0.f : top;
  float l = 0.f, acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < splits; s0 += 4) {
    float4 v[4];
    float w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int s = min(s0 + j, splits - 1);
      const float2 a = ml[s * items + at];
      const bool some = s0 + j < splits && a.y != 0.f;   // a split without weights has written no sums
      w[j] = some ? exp2f(a.x - ms) : 0.f;
      if (some) l = fmaf(a.y, w[j], l);
      v[j] = some ? *reinterpret_cast<const float4*>(part + (s * items + at) * D + c) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc[0] = fmaf(v[j].x, w[j], acc[0]);
      acc[1] = fmaf(v[j].y, w[j], acc[1]);
      acc[2] = fmaf(v[j].z, w[j], acc[2]);
      acc[3] = fmaf(v[j].w, w[j], acc[3]);
    }
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  Vec<T, 4> r;
#pragma unroll
  for (int j = 0; j < 4; ++j) r.v[j] = from_f32<T>(acc[j] * inv);
  stvec<T, 4>(o + at * D + c, r);
}

template <typename T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void extend_attn_mfma32_wide_kernel(
    const T* __restrict__ q_ext, const T* __restrict__ k_ext, const T* __restrict__ v_ext, T* __restrict__ o_ext,
    const T* __restrict__ kbuf, const T* __restrict__ vbuf, ExtendParams p, int nqb, int npairs) {
  extend_attn_mfma32_body<T, false, 192>(q_ext, k_ext, v_ext, o_ext, kbuf, vbuf, p, nqb, npairs);
}

// Whole prompts over a latent cache (rank 512 + 64) in expanded form: per visible pair and head 2 (128 + 64 + 128) flops
// instead of the absorbed form's 2 (512 + 64 + 512), for one projection of every latent to its heads' keys and values (4 x 1900
// tokens x 16 heads: 154 us, and about 70 for that projection; the absorbed launch with its two per-head products took 1570 us).
// Without a prefix to address, and with the rope part's rows dealt to all threads (two pieces each instead of four to half of
// them), the body fits 256 registers: two workgroups per CU, one's softmax beside the other's MFMAs.  At one per CU: 226 us; 32
// heads 404 -> 238.  DIRECT: for rows that 32-bit offsets reach.
template <typename T, bool DIRECT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void extend_attn_latent_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, T* __restrict__ o, ExtendParams p, int nqb, int npairs) {
  extend_attn_mfma32_body<T, false, 192, true, 128, false, false, DIRECT>(q, k, v, o, nullptr, nullptr, p, nqb, npairs);
}

template <typename T, int DP, int BN>
static int launch_extend_cfg(const void* q, const void* k, const void* v, void* o, const void* kb,
                             const void* vb, const ExtendParams& p, int64_t bs,
                             int64_t max_len_extend, bool vec, hipStream_t st) {
  constexpr int VE = V16<T>::n;
  const int gtotal = p.hq / p.hkv;
  const int Gc = gtotal < 64 ? gtotal : 64;
  const int TM = 64 / Gc;
  const dim3 grid((unsigned)((max_len_extend + TM - 1) / TM), (unsigned)(p.hkv * (gtotal / Gc)),
                  (unsigned)bs);
  const size_t lds = (size_t)(64 + 2 * BN) * (DP + VE) * sizeof(T) + (size_t)64 * (BN + 4) * 4;
  if (vec) {
    auto kern = extend_attn_kernel<T, DP, BN, true>;
    if (lds > 48 * 1024)
      (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(kern, grid, dim3(256), lds, st, (const T*)q, (const T*)k, (const T*)v, (T*)o,
                       (const T*)kb, (const T*)vb, p);
  } else {
    auto kern = extend_attn_kernel<T, DP, BN, false>;
    if (lds > 48 * 1024)
      (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(kern, grid, dim3(256), lds, st, (const T*)q, (const T*)k, (const T*)v, (T*)o,
                       (const T*)kb, (const T*)vb, p);
  }
  return MI355_OK;
}

// 0 = 32x32x16 tile (product), 1 = the 16x16x32 tile above (ablation; development build, mi355_debug_set key 8)
#ifdef MI355_DEV_BUILD
int g_extend_variant = 0;
#else
static constexpr int g_extend_variant = 0;
#endif

// Which of the 32 x 32 kernels serves the call; the maximum is taken of unscaled scores.
static bool mfma32_serves(int D, int Dv, bool kv8, bool mask, int sliding_window, float logit_cap, float sm_scale) {
  return ((D == 128 && Dv == 128) || (D == 192 && Dv == 128 && !kv8) || (D == 64 && Dv == 64)) && (!mask || D == 64) && sliding_window <= 0 &&
         logit_cap <= 0.f && sm_scale > 0.f && g_extend_variant == 0;
}

template <typename T, int D>
static int launch_mfma32(const void* q, const void* k, const void* v, void* o, const void* kb, const void* vb, ExtendParams p,
                         int64_t bs, int nqb, int64_t npairs, int64_t wgs, int splits, bool kv8, int64_t num_slots, hipStream_t st) {
  using Kernel = void (*)(const T*, const T*, const T*, T*, const T*, const T*, ExtendParams, int, int);
  Kernel kernel;
  int lds = 0;
  if constexpr (D == 64) {
    if (splits > 1)
      kernel = p.custom_mask ? (kv8 ? extend_attn_mfma32_d64_kernel<T, true, true, true> : extend_attn_mfma32_d64_kernel<T, false, true, true>)
                             : (kv8 ? extend_attn_mfma32_d64_kernel<T, true, false, true> : extend_attn_mfma32_d64_kernel<T, false, false, true>);
    else
      kernel = p.custom_mask ? (kv8 ? extend_attn_mfma32_d64_kernel<T, true, true, false> : extend_attn_mfma32_d64_kernel<T, false, true, false>)
                             : (kv8 ? extend_attn_mfma32_d64_kernel<T, true, false, false> : extend_attn_mfma32_d64_kernel<T, false, false, false>);
  } else {
    // (32-bit offsets: the cache of 4 GiB a layer and side, new rows of 16 MiB)
    const int64_t near = 0xffff0000ll / (2 * std::max(p.kb_slot, p.vb_slot));
    const bool direct = !kv8 && num_slots > 0 && num_slots <= near && p.k_stride < (1 << 23) && p.v_stride < (1 << 23);
    p.near_slots = (uint32_t)near;
    if (direct) kernel = splits > 1 ? extend_attn_mfma32_kernel<T, false, true, true> : extend_attn_mfma32_kernel<T, false, false, true>;
    else if (kv8) kernel = splits > 1 ? extend_attn_mfma32_kernel<T, true, true, false> : extend_attn_mfma32_kernel<T, true, false, false>;
    else kernel = splits > 1 ? extend_attn_mfma32_kernel<T, false, true, false> : extend_attn_mfma32_kernel<T, false, false, false>;
    if (direct) lds = 2 * direct_stage_bytes<128>();
  }
  if (lds != 0) (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  hipLaunchKernelGGL(kernel, dim3((unsigned)wgs, (unsigned)splits), dim3(256), lds, st, (const T*)q, (const T*)k, (const T*)v, (T*)o, (const T*)kb,
                     (const T*)vb, p, nqb, (int)npairs);
  if (splits > 1) {
    const int64_t items = p.rows * p.hq;
    hipLaunchKernelGGL((extend_split_merge_kernel<T, D>), dim3((unsigned)((items + 1024 / D - 1) / (1024 / D))), dim3(256), 0, st, (T*)o, p.part,
                       p.part_ml, p.qo_indptr, bs, items, p.hq, splits);
  }
  return MI355_OK;
}

template <typename T>
static int launch_extend(const void* q, const void* k, const void* v, void* o, const void* kb,
                         const void* vb, const ExtendParams& p, int64_t bs, int64_t max_len_extend,
                         bool kv8, int splits, int64_t num_slots, hipStream_t st) {   // kv8: the KV cache holds e4m3fn bytes
  constexpr int VE = V16<T>::n;
  const int dmax = p.D > p.Dv ? p.D : p.Dv;
  const bool vec = p.D % VE == 0 && p.Dv % VE == 0 && p.q_stride % VE == 0 &&
                   p.k_stride % VE == 0 && p.v_stride % VE == 0 && aligned16(q) && aligned16(k) &&
                   aligned16(v) && aligned16(o) && aligned16(kb) && aligned16(vb);
  if constexpr (!std::is_same<T, float>::value) {
    if (vec && mfma32_serves(p.D, p.Dv, kv8, p.custom_mask != nullptr, p.sliding_window, p.logit_cap, p.sm_scale)) {
      // 128 query rows of one head per workgroup; (sequence, kv head) pairs dealt round-robin to the XCDs
      const int nqb = (int)((max_len_extend + 127) / 128);
      const int64_t npairs = bs * p.hkv;
      const int64_t wgs = 8 * ((npairs + 7) / 8) * (p.hq / p.hkv) * nqb;
      if (wgs < (int64_t)1 << 31) {
        if (p.D == 64) return launch_mfma32<T, 64>(q, k, v, o, kb, vb, p, bs, nqb, npairs, wgs, splits, kv8, num_slots, st);
        if (p.D == 128) return launch_mfma32<T, 128>(q, k, v, o, kb, vb, p, bs, nqb, npairs, wgs, splits, kv8, num_slots, st);
        hipLaunchKernelGGL((extend_attn_mfma32_wide_kernel<T>), dim3((unsigned)wgs), dim3(256), 0, st, (const T*)q, (const T*)k,
                           (const T*)v, (T*)o, (const T*)kb, (const T*)vb, p, nqb, (int)npairs);
        return MI355_OK;
      }
    }
    if (vec && p.D == 128 && p.Dv == 128 && !p.custom_mask && p.sliding_window <= 0 && p.logit_cap <= 0.f) {
      const dim3 grid((unsigned)((max_len_extend + 63) / 64), (unsigned)p.hq, (unsigned)bs);
      if (kv8)
        hipLaunchKernelGGL((extend_attn_mfma_kernel<T, true>), grid, dim3(256), 0, st, (const T*)q, (const T*)k,
                           (const T*)v, (T*)o, (const T*)kb, (const T*)vb, p);
      else
        hipLaunchKernelGGL((extend_attn_mfma_kernel<T, false>), grid, dim3(256), 0, st, (const T*)q, (const T*)k,
                           (const T*)v, (T*)o, (const T*)kb, (const T*)vb, p);
      return MI355_OK;
    }
  }
  if (dmax <= 64) return launch_extend_cfg<T, 64, 64>(q, k, v, o, kb, vb, p, bs, max_len_extend, vec, st);
  if (dmax <= 128) return launch_extend_cfg<T, 128, 64>(q, k, v, o, kb, vb, p, bs, max_len_extend, vec, st);
  if (dmax <= 256) {
    if (sizeof(T) == 4)
      return launch_extend_cfg<T, 256, 32>(q, k, v, o, kb, vb, p, bs, max_len_extend, vec, st);
    return launch_extend_cfg<T, 256, 64>(q, k, v, o, kb, vb, p, bs, max_len_extend, vec, st);
  }
  set_error("extend_attention: head_dim %d / v_head_dim %d > 256 not supported", p.D, p.Dv);
  return MI355_ERR_UNSUPPORTED;
}

}  // namespace mi355

using namespace mi355;

extern "C" {

// The kernel holds two workgroups a CU, 512 in all; fewer leave CUs idle while each walks its keys alone.  Their number is estimated:
// rows / 128 blocks of queries and half a block of each sequence, at most the longest's for all, times the heads.  `tiles` of 64 keys
// a block on average, 4 or more a split.  us a launch out of cold caches, unsplit | split (32 / 8 heads): head_dim 128, fp8 cache 83 rows on 1933 cached
// 111 | 29 (in a step), 97 x 6 on 2663 212 | 124 (2), 152 x 3 on 2411 189 | 75 (4), bf16 99 on 572 28 | 23 (2); head_dim 64, 3 x 121 on
// 1513 50 | 35 (3), fp8 86 on 816 42 | 31 (2), 2 x 244 on 2141 97 | 49 (4).  Left whole: fewer than 512 cached tokens a sequence (1148 on
// none, head_dim 64, 37 | 42 in two; 3 x 993, 128, 51 | 80; and a whole prompt's first rows are then a shorter one's, bit for bit), 512 workgroups (4 x 490 on 1750 83 | 100), few tiles (400 new on 300, seven, 22 | 26).
int mi355_extend_attention_splits(int64_t rows, int64_t bs, int64_t max_len_extend, int64_t prefix_tokens, int has_mask, int hq, int head_dim,
                                  int v_head_dim, float sm_scale, float logit_cap, int sliding_window_size, int dtype) {
  const bool kv8 = (dtype & MI355_KV_FP8) != 0;
  if ((dtype & 0xff) == MI355_F32 || rows < 1 || bs < 1 || max_len_extend < 1 || hq < 1 || rows > (1 << 24) || hq > 4096 ||
      !mfma32_serves(head_dim, v_head_dim, kv8, has_mask != 0, sliding_window_size, logit_cap, sm_scale) || head_dim > 128 ||
      prefix_tokens < 512 * bs)
    return 1;
  const int64_t wgs = std::min(bs * ((max_len_extend + 127) / 128), rows / 128 + bs / 2 + 1) * hq;
  const int64_t tiles = (prefix_tokens + rows / 2) / bs / 64;
  return (int)std::max<int64_t>(1, std::min<int64_t>({512 / wgs, (tiles - 2) / SPLIT_TILES, 8}));
}

int64_t mi355_extend_attention_workspace_bytes(int64_t rows, int hq, int v_head_dim, int splits) {
  return splits > 1 ? (int64_t)splits * rows * hq * (v_head_dim + 2) * 4 : 0;
}

int mi355_extend_attention(const void* q_extend, const void* k_extend, const void* v_extend,
                           void* o_extend, const void* k_buffer, const void* v_buffer,
                           const int32_t* qo_indptr, const int32_t* kv_indptr,
                           const int32_t* kv_indices, const uint8_t* custom_mask,
                           const int64_t* mask_indptr, int is_causal, int skip_prefix_custom_mask,
                           int64_t bs, int64_t max_len_extend, int hq, int hkv, int head_dim,
                           int v_head_dim, int64_t q_stride, int64_t k_stride, int64_t v_stride,
                           int64_t num_slots, float sm_scale, float logit_cap,
                           int sliding_window_size, int dtype, void* stream) {
  return mi355_extend_attention_ws(q_extend, k_extend, v_extend, o_extend, k_buffer, v_buffer, qo_indptr, kv_indptr, kv_indices, custom_mask,
                                   mask_indptr, is_causal, skip_prefix_custom_mask, bs, max_len_extend, hq, hkv, head_dim, v_head_dim,
                                   q_stride, k_stride, v_stride, num_slots, sm_scale, logit_cap, sliding_window_size, dtype, 0, 1, nullptr,
                                   0, stream);
}

int mi355_extend_attention_ws(const void* q_extend, const void* k_extend, const void* v_extend,
                              void* o_extend, const void* k_buffer, const void* v_buffer,
                              const int32_t* qo_indptr, const int32_t* kv_indptr,
                              const int32_t* kv_indices, const uint8_t* custom_mask,
                              const int64_t* mask_indptr, int is_causal, int skip_prefix_custom_mask,
                              int64_t bs, int64_t max_len_extend, int hq, int hkv, int head_dim,
                              int v_head_dim, int64_t q_stride, int64_t k_stride, int64_t v_stride,
                              int64_t num_slots, float sm_scale, float logit_cap,
                              int sliding_window_size, int dtype, int64_t rows, int splits, void* workspace,
                              int64_t workspace_bytes, void* stream) {
  MI355_REQUIRE(q_extend && k_extend && v_extend && o_extend && qo_indptr && kv_indptr,
                MI355_ERR_INVALID, "extend_attention: null pointer");
  MI355_REQUIRE(k_buffer && v_buffer && kv_indices, MI355_ERR_INVALID,
                "extend_attention: k_buffer/v_buffer/kv_indices must be valid pointers (may be "
                "unused when every prefix is empty, but must not be null)");
  MI355_REQUIRE(!custom_mask || mask_indptr, MI355_ERR_INVALID,
                "extend_attention: custom_mask needs mask_indptr");
  MI355_REQUIRE(bs >= 0 && max_len_extend >= 0 && hq > 0 && hkv > 0 && hq % hkv == 0 &&
                    head_dim > 0 && v_head_dim > 0,
                MI355_ERR_INVALID, "extend_attention: bad shape");
  const int gtotal = hq / hkv;
  MI355_REQUIRE(gtotal <= 64 ? true : gtotal % 64 == 0, MI355_ERR_UNSUPPORTED,
                "extend_attention: q heads per kv head (%d) must be <= 64 or a multiple of 64",
                gtotal);
  MI355_REQUIRE(q_stride >= (int64_t)hq * head_dim && k_stride >= (int64_t)hkv * head_dim &&
                    v_stride >= (int64_t)hkv * v_head_dim,
                MI355_ERR_INVALID, "extend_attention: row strides smaller than rows");
  MI355_REQUIRE(bs <= 65535, MI355_ERR_UNSUPPORTED, "extend_attention: batch > 65535");
  if (bs == 0 || max_len_extend == 0) return MI355_OK;
  ExtendParams p = {};
  p.qo_indptr = qo_indptr;
  p.kv_indptr = kv_indptr;
  p.kv_indices = kv_indices;
  p.custom_mask = custom_mask;
  p.mask_indptr = mask_indptr;
  p.q_stride = q_stride;
  p.k_stride = k_stride;
  p.v_stride = v_stride;
  p.is_causal = is_causal;
  p.skip_prefix_custom_mask = skip_prefix_custom_mask;
  p.hq = hq;
  p.hkv = hkv;
  p.D = head_dim;
  p.Dv = v_head_dim;
  p.sliding_window = sliding_window_size;
  p.sm_scale = sm_scale;
  p.logit_cap = logit_cap;
  MI355_REQUIRE(!(dtype & MI355_KV_INTERLEAVED) || ((dtype & MI355_KV_HEAD_MAJOR) && head_dim == v_head_dim), MI355_ERR_INVALID,
                "extend_attention: an interleaved cache is head-major with head_dim == v_head_dim");
  kv_strides(dtype, num_slots, hkv, head_dim, p.kb_slot, p.kb_head);
  kv_strides(dtype, num_slots, hkv, v_head_dim, p.vb_slot, p.vb_head);
  int rc = MI355_OK;
  const bool kv8 = (dtype & MI355_KV_FP8) != 0;
  p.kv8 = kv8 ? 1 : 0;
  dtype &= 0xff;
  if (splits > 1) {
    MI355_REQUIRE(splits <= 65535 && rows > 0 && workspace && aligned16(workspace) &&
                      workspace_bytes >= mi355_extend_attention_workspace_bytes(rows, hq, v_head_dim, splits),
                  MI355_ERR_INVALID, "extend_attention: workspace of %ld bytes for %ld rows x %d splits", (long)workspace_bytes, (long)rows, splits);
    p.rows = rows;
    p.part = (float*)workspace;
    p.part_ml = (float2*)(p.part + (int64_t)splits * rows * hq * v_head_dim);
  }
  MI355_DISPATCH_DTYPE(dtype, "extend_attention",
                       rc = launch_extend<T>(q_extend, k_extend, v_extend, o_extend, k_buffer,
                                             v_buffer, p, bs, max_len_extend, kv8, splits > 1 ? splits : 1, num_slots, (hipStream_t)stream));
  if (rc != MI355_OK) return rc;
  MI355_CHECK_LAUNCH("extend_attention");
  return MI355_OK;
}

int mi355_latent_prefill_attention_supported(int nope_dim, int rope_dim, int v_dim, int rot_dims, int interleaved, int dtype) {
  return (dtype == MI355_BF16 || dtype == MI355_F16) && nope_dim == 128 && rope_dim == 64 && v_dim == 128 && rot_dims >= 0 &&
         rot_dims <= 64 && rot_dims % 2 == 0 && (interleaved || rot_dims == 0 || rot_dims == 64);
}

int mi355_latent_prefill_attention(void* out, const void* q, int64_t q_stride, const void* kv, int64_t kv_stride, const void* k_rope,
                                   int64_t k_rope_stride, const int32_t* seg_start, const int32_t* seg_len, const int64_t* positions,
                                   const float* inv_freq, int rot_dims, int interleaved, float rot_mag, int64_t bs, int64_t max_len,
                                   int heads, int nope_dim, int rope_dim, int v_dim, float scale, int dtype, void* stream) {
  MI355_REQUIRE(out && q && kv && k_rope && seg_start && seg_len && positions && (inv_freq || rot_dims == 0), MI355_ERR_INVALID,
                "latent_prefill_attention: null pointer");
  MI355_REQUIRE(mi355_latent_prefill_attention_supported(nope_dim, rope_dim, v_dim, rot_dims, interleaved, dtype), MI355_ERR_UNSUPPORTED,
                "latent_prefill_attention: 16-bit heads of 128 + 64 key and 128 value features (nope=%d rope=%d v=%d rot=%d dtype=%d)",
                nope_dim, rope_dim, v_dim, rot_dims, dtype);
  MI355_REQUIRE(bs >= 0 && max_len >= 0 && heads > 0 && scale > 0.f, MI355_ERR_INVALID, "latent_prefill_attention: bad shape");
  MI355_REQUIRE(q_stride >= (int64_t)heads * 192 && q_stride % 8 == 0 && kv_stride >= (int64_t)heads * 256 && kv_stride % 8 == 0 &&
                    k_rope_stride >= 64 && k_rope_stride % 8 == 0 && aligned16(q) && aligned16(kv) && aligned16(k_rope) && aligned16(out),
                MI355_ERR_INVALID, "latent_prefill_attention: rows must be 16-byte aligned and hold every head");
  if (bs == 0 || max_len == 0) return MI355_OK;
  ExtendParams p = {};
  p.seg_start = seg_start; p.seg_len = seg_len; p.positions = positions; p.inv_freq = inv_freq;
  p.rot_dims = rot_dims; p.interleaved = interleaved; p.rot_mag = rot_mag;
  p.q_stride = q_stride; p.k_stride = p.v_stride = kv_stride; p.kv_head = 256;
  p.k_rope = k_rope; p.k_rope_stride = k_rope_stride;
  p.is_causal = 1; p.hq = p.hkv = heads; p.D = 192; p.Dv = 128; p.sm_scale = scale;
  const int nqb = (int)((max_len + 127) / 128);
  const int64_t npairs = bs * heads, wgs = 8 * ((npairs + 7) / 8) * nqb;
  MI355_REQUIRE(wgs < (int64_t)1 << 31, MI355_ERR_UNSUPPORTED, "latent_prefill_attention: too many query blocks");
  // 80 KiB: two workgroups a CU (rows of 2^23 elements and more apart: through registers, as before there were buffer loads)
  const bool direct = kv_stride < (1 << 23) && k_rope_stride < (1 << 23);
  const int lds = direct ? 2 * direct_stage_bytes<192>() : 0;
#define MI355_LP(T)                                                                                                            \
  auto kernel = direct ? extend_attn_latent_kernel<T, true> : extend_attn_latent_kernel<T, false>;                             \
  if (lds != 0) (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);               \
  hipLaunchKernelGGL(kernel, dim3((unsigned)wgs), dim3(256), lds, (hipStream_t)stream, (const T*)q, (const T*)kv, (const T*)kv + 128, (T*)out, p, \
                     nqb, (int)npairs)
  if (dtype == MI355_BF16) { MI355_LP(bf16_t); }
  else { MI355_LP(f16_t); }
#undef MI355_LP
  MI355_CHECK_LAUNCH("latent_prefill_attention");
  return MI355_OK;
}

}  // extern "C"
