// Softmax attention over a sliding window with an optional sink in the denominator, grouped key heads, no rotation:
//     s_j = (q[t, h] . K[j, g]) * scale               for keys j with 0 <= pos(t) - j < window   (window <= 0: every j <= pos)
//     out[t, h] = sum_j exp(s_j) V[j, g] / (exp(sink_h) + sum_j exp(s_j)),        g = h / (H / G)
// over per-layer key / value buffers [slots, G, d] / [slots, G, dv] reached through the request table.  sink null: no such
// term; a sink of 0 adds one to the denominator.  Scores, weights and sums are fp32.
//
// A workgroup takes one run of consecutive tokens of one sequence, one kv head and the query heads that share it as rows of
// one tile, walks the key tiles that any of its rows can see (from the window's lower edge of the run's first token to the
// run's last token) and keeps the running (max, sum) pair per row, started at (sink, 1) -- or (-huge, 0) without a sink.
//   * 16-bit dtypes, d a multiple of 32 and dv of 16: matrix cores, 64 rows per workgroup (S^T = K Q^T and O^T = V^T P^T on
//     16x16x32 MFMA, a wave per 16 rows, the weights in the activation dtype),
//   * everything else (fp32, odd widths): vector ALU, 16 rows per workgroup, all fp32.
// Prefill portions, decode steps and mixed batches are the same launch, told apart only by the list of runs.  A launch of
// single tokens (a decode step) may cut each token's keys into num_splits ranges: every range leaves its unnormalised sum,
// running maximum and running sum in fp32 scratch (the sink belongs to the first range), and a second launch merges them.
//
// Averaged blocks (pool > 0, window > 0): beside the window's tokens, token i sees one key / value row for every block b of
// `pool` positions whose last position precedes its window, b pool + pool - 1 <= i - window; the rows are the means of the
// block's cached keys and values, kept in pooled buffers at row slot(b pool + pool - 1) / pool_div (mi355_pool_kv_blocks
// writes them when a block's last token enters the cache).  The walk then starts with the tiles of the pooled rows that the
// run's last token sees, masked per row, and goes on with the window's tiles; blocks and tokens share the running (max, sum).
// A gate per head (head_gate, logits) multiplies head h's result by its sigmoid.
#include "common.cuh"

#include <algorithm>
#include <type_traits>

namespace mi355 {
namespace {

constexpr int WA_ROWS = 16;
constexpr int WA_KT = 32;
constexpr float WA_NEG = -1.0e30f;

struct WaArgs {
  void* out;
  const void* q;
  const void* k_cache;
  const void* v_cache;
  const int32_t* req_to_token;
  const int64_t* req_pool_indices;
  const int32_t* tok_req;
  const int64_t* positions;
  const int32_t* blocks;
  const float* sink;
  const void* pooled_k;
  const void* pooled_v;
  const void* gate;        // [token][head] logits of the result's gate, or null
  int64_t gate_token_stride;
  int pool, pool_div;
  float* partial;          // num_splits > 1: [split][token][head][dv + 2] = unnormalised result | running max | running sum
  int64_t q_token_stride, q_head_stride, out_token_stride, out_head_stride, req_to_token_stride, tokens;
  int heads, kv_heads, d, dv, heads_per_tile, window, num_splits;
  float scale;
};

// 16 lanes that hold one row (a DPP row): max and sum over them, every lane gets the result.  Lane exchanges inside quads,
// then across the halves of a half row, then across the row's halves.
template <int CTRL> __device__ __forceinline__ float wa_dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float row16_max(float x) {
  x = fmaxf(x, wa_dpp<0xB1>(x));      // quad_perm [1,0,3,2]
  x = fmaxf(x, wa_dpp<0x4E>(x));      // quad_perm [2,3,0,1]
  x = fmaxf(x, wa_dpp<0x141>(x));     // row_half_mirror
  return fmaxf(x, wa_dpp<0x140>(x));  // row_mirror
}
__device__ __forceinline__ float row16_sum(float x) {
  x += wa_dpp<0xB1>(x);
  x += wa_dpp<0x4E>(x);
  x += wa_dpp<0x141>(x);
  return x + wa_dpp<0x140>(x);
}

__device__ __forceinline__ float wa_sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }

// Vector-ALU kernel.  sm: Qs [16][d] | Ks [KT][d + 1] | Vs [KT][dv] | Ps [16][KT]
template <typename T>
__global__ __launch_bounds__(256) void window_attention_valu_kernel(WaArgs a) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int d = a.d, dv = a.dv;
  float* Qs = sm;
  float* Ks = Qs + WA_ROWS * d;
  float* Vs = Ks + WA_KT * (d + 1);
  float* Ps = Vs + WA_KT * dv;
  __shared__ int row_pos[WA_ROWS];
  const int rep = a.heads / a.kv_heads;
  const int chunks = (rep + a.heads_per_tile - 1) / a.heads_per_tile;
  const int g = blockIdx.y / chunks, hc = blockIdx.y - g * chunks;
  const unsigned bx = gridDim.x - 1 - blockIdx.x;
  const int64_t t0 = a.blocks != nullptr ? a.blocks[2 * bx] : bx;
  const int nt = a.blocks != nullptr ? a.blocks[2 * bx + 1] : 1;
  const int b = a.tok_req != nullptr ? a.tok_req[t0] : (int)t0;
  const int32_t* table = a.req_to_token + a.req_pool_indices[b] * a.req_to_token_stride;
  const int h0 = g * rep + hc * a.heads_per_tile;
  const int nh = min(a.heads_per_tile, rep - hc * a.heads_per_tile);
  const int tid = threadIdx.x;
  const T* q = (const T*)a.q;
  for (int e = tid; e < WA_ROWS * d; e += 256) {
    const int r = e / d, i = e - r * d;
    const int tl = r / a.heads_per_tile, hl = r - tl * a.heads_per_tile;
    Qs[e] = (tl < nt && hl < nh) ? to_f32(q[(t0 + tl) * a.q_token_stride + (int64_t)(h0 + hl) * a.q_head_stride + i]) : 0.f;
  }
  if (tid < WA_ROWS) {
    const int tl = tid / a.heads_per_tile, hl = tid - tl * a.heads_per_tile;
    row_pos[tid] = (tl < nt && hl < nh) ? (int)a.positions[t0 + tl] : -1;
  }
  const int first = (int)a.positions[t0];
  const int last = first + nt - 1;                      // the run's tokens are consecutive
  const int lowest = a.window > 0 ? max(0, first - a.window + 1) : 0;
  const int split = blockIdx.z;
  const int all_lo = lowest / WA_KT, all_hi = last / WA_KT + 1;
  // pooled rows that the run's last token sees come first on the walk: ptiles tiles of them, then the window's tiles
  const int nb_run = (a.pool > 0 && a.window > 0 && last - a.window + 1 >= a.pool) ? (last - a.window + 1) / a.pool : 0;
  const int ptiles = (nb_run + WA_KT - 1) / WA_KT;
  const int ntiles = ptiles + all_hi - all_lo;
  const int per = (ntiles + a.num_splits - 1) / a.num_splits;
  const int tile_lo = split * per, tile_hi = min(ntiles, tile_lo + per);
  const int r = tid >> 4, cx = tid & 15;
  const int hl_r = r % a.heads_per_tile;
  float run_m = WA_NEG, run_l = 0.f;
  if (a.sink != nullptr && split == 0) { run_m = a.sink[h0 + min(hl_r, nh - 1)]; run_l = 1.f; }
  float acc[16];
#pragma unroll
  for (int m = 0; m < 16; ++m) acc[m] = 0.f;
  for (int tile = tile_lo; tile < tile_hi; ++tile) {
    const bool ptile = tile < ptiles;
    const int j0 = (ptile ? tile : all_lo + tile - ptiles) * WA_KT;
    const T* kc = (const T*)(ptile ? a.pooled_k : a.k_cache);
    const T* vc = (const T*)(ptile ? a.pooled_v : a.v_cache);
    __syncthreads();
    for (int e = tid; e < WA_KT * (d + dv); e += 256) {
      const bool isk = e < WA_KT * d;
      const int e2 = isk ? e : e - WA_KT * d;
      const int w = isk ? d : dv;
      const int kk = e2 / w, i = e2 - kk * w;
      const int j = j0 + kk;
      float val = 0.f;
      if (ptile ? j < nb_run : (j >= lowest && j <= last)) {
        const int64_t row = ptile ? table[j * a.pool + a.pool - 1] / a.pool_div : table[j];
        val = to_f32((isk ? kc : vc)[(row * a.kv_heads + g) * w + i]);
      }
      if (isk) Ks[kk * (d + 1) + i] = val;
      else Vs[e2] = val;
    }
    __syncthreads();
    const int rp = row_pos[r];
    float sc[WA_KT / 16];
    float tmax = WA_NEG;
#pragma unroll
    for (int u = 0; u < WA_KT / 16; ++u) {
      const int kk = cx + 16 * u;
      float s = 0.f;
      for (int i = 0; i < d; ++i) s = fmaf(Qs[r * d + i], Ks[kk * (d + 1) + i], s);
      const int j = j0 + kk;
      const bool seen = ptile ? (rp >= 0 && j * a.pool + a.pool - 1 <= rp - a.window) : (j <= rp && (a.window <= 0 || rp - j < a.window));
      sc[u] = seen ? s * a.scale : WA_NEG;
      tmax = fmaxf(tmax, sc[u]);
    }
    tmax = row16_max(tmax);
    const float new_m = fmaxf(run_m, tmax);
    const float alpha = expf(run_m - new_m);          // 1 when nothing changed, also for rows that have seen nothing yet
    float psum = 0.f;
#pragma unroll
    for (int u = 0; u < WA_KT / 16; ++u) {
      const float p = sc[u] > 0.5f * WA_NEG ? expf(sc[u] - new_m) : 0.f;
      Ps[r * WA_KT + cx + 16 * u] = p;
      psum += p;
    }
    psum = row16_sum(psum);
    run_l = run_l * alpha + psum;
    run_m = new_m;
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 16; ++m) acc[m] *= alpha;
    for (int kk = 0; kk < WA_KT; ++kk) {
      const float p = Ps[r * WA_KT + kk];
#pragma unroll
      for (int m = 0; m < 16; ++m) {
        const int c = cx + 16 * m;
        if (c < dv) acc[m] = fmaf(p, Vs[kk * dv + c], acc[m]);
      }
    }
  }
  const int tl = r / a.heads_per_tile, hl = r - tl * a.heads_per_tile;
  if (tl < nt && hl < nh) {
    if (a.num_splits > 1) {
      float* part = a.partial + (((int64_t)split * a.tokens + t0 + tl) * a.heads + h0 + hl) * (dv + 2);
#pragma unroll
      for (int m = 0; m < 16; ++m) {
        const int c = cx + 16 * m;
        if (c < dv) part[c] = acc[m];
      }
      if (cx == 0) { part[dv] = run_m; part[dv + 1] = run_l; }
      return;
    }
    float inv = run_l > 0.f ? 1.0f / run_l : 0.f;
    if (a.gate != nullptr) inv *= wa_sigmoid(to_f32(((const T*)a.gate)[(t0 + tl) * a.gate_token_stride + h0 + hl]));
#pragma unroll
    for (int m = 0; m < 16; ++m) {
      const int c = cx + 16 * m;
      if (c >= dv) continue;
      ((T*)a.out)[(t0 + tl) * a.out_token_stride + (int64_t)(h0 + hl) * a.out_head_stride + c] = from_f32<T>(acc[m] * inv);
    }
  }
}

// out[t, h] = sum_s acc_s e^(m_s - M) / sum_s l_s e^(m_s - M), M = max_s m_s, over the key ranges in order.  One workgroup per
// (token, head).
template <typename T>
__global__ __launch_bounds__(256) void window_attention_merge_kernel(T* __restrict__ out, const float* __restrict__ partial,
                                                                     int64_t tokens, int heads, int dv, int num_splits,
                                                                     int64_t out_token_stride, int64_t out_head_stride,
                                                                     const T* __restrict__ gate, int64_t gate_token_stride) {
  const int lane = threadIdx.x & 63;
  const int64_t idx = blockIdx.x, t = idx / heads;
  const int h = (int)(idx - t * heads);
  const int64_t stride = tokens * heads * (int64_t)(dv + 2);
  const float* p0 = partial + idx * (dv + 2);
  const bool has = lane < num_splits;      // lane k has split k's weight (at most 64 of them)
  const float m = has ? p0[lane * stride + dv] : WA_NEG, l = has ? p0[lane * stride + dv + 1] : 0.f;
  const float M = wave_max(m), w = has ? expf(m - M) : 0.f, L = wave_sum(l * w);   // (the lanes without a split have WA_NEG)
  float inv = L > 0.f ? 1.0f / L : 0.f;
  if (gate != nullptr) inv *= wa_sigmoid(to_f32(gate[t * gate_token_stride + h]));
  for (int c0 = 0; c0 < dv; c0 += 256) {
    const int c = c0 + (int)threadIdx.x;
    float s[1] = {0.f};
    const int64_t col[1] = {min(c, dv - 1)};
    fold_splits(s, p0, stride, num_splits, col, [&](int k) { return lane_value(w, k); }, [](float f, float v, float x) { return x + v * f; });
    if (c < dv) out[t * out_token_stride + (int64_t)h * out_head_stride + c] = from_f32<T>(s[0] * inv);
  }
}

// Matrix-core kernel for 16-bit dtypes, d % 32 == 0, dv % 16 == 0.  Four waves of 16 (token, head) rows.  Per key tile of 32 a
// wave computes S^T = K Q^T for its rows with 2 * d / 32 MFMA 16x16x32 (A = K rows from LDS, B = Q rows, held in registers):
// a lane then holds eight scores of ONE row, so that masks, maximum, sum and rescale factor are the lane's own but for two
// exchanges over registers, and its weights are, rounded to T, the B operand of O^T += V^T P^T as they stand (one MFMA
// 16x16x32 per 16 result columns, V read transposed).  Nothing travels between waves; the tiles of K and V take turns in two
// LDS buffers, one barrier each, the next tile's rows on their way from memory meanwhile.
// What bounds it: the vector ALU (about 90 operations per lane and tile beside 16 MFMAs at d = dv = 128; half of them in a tile
// that every row of the run sees whole, which has no masks).  FULL: d and dv are 64 CK and 64 CT, so that no condition stands
// between a tile's reads and MFMAs and the compiler requests the reads ahead; the other widths keep the general loops.  us a launch over
// 7381 prefill tokens of 16 heads over 4, masks on every tile and the general loops | now, at window 512 with averaged blocks of 64, window
// 64, window 16 (no tile is whole) and no window: d = dv = 128 122 | 104, 52.3 | 51.6, 45.0 | 44.9, 220 | 170; 64 72 | 57, 26.8 | 26.8, 23.1 | 23.2,
// 151 | 104; 96 100 | 90, 41.3 | 41.4, 34.0 | 34.8, 203 | 170; 192 and 128 151 | 136, 62.4 | 62.0, 48.0 | 48.6, 287 | 245; 64 and 256 170 | 154,
// 74.9 | 74.8, 62.0 | 62.6, 306 | 263; 256 263 | 241, 99.0 | 99.7, 77.7 | 79.4, 485 | 425.  A form with S = Q K^T, where a row's scores lay in
// 16 lanes, its weights and factor went through LDS and the waves shared the result columns (three barriers), took 2.35 times the time.
// Single tokens of 4 heads a key head are one live wave, whose chain is shorter too: 1 / 64 / 256 tokens x 2000 keys, same heads and
// window, 22 / 31 / 66 us against 31 / 41 / 131.
// Widths in (64, 128] by the general loops are held to 128 registers, four waves a SIMD (three spilled in front of the loop): at 131 and three
// waves 96 wide took 103, 44.6, 36.4 and 182 us of the above.
// sm: 2 x (Ks [32][d + 8] | Vs [32][dv + 8])   (all T)
constexpr int WAM_ROWS = 64;
constexpr int WAM_MAX = 256;     // d and dv

template <typename T, int CT, int CK, bool FULL>
__global__ __launch_bounds__(256, CT == 2 && CK == 2 && !FULL ? 4 : 1) void window_attention_mfma_kernel(WaArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smraw[];
  const int d = FULL ? 64 * CK : a.d, dv = FULL ? 64 * CT : a.dv;
  const int qld = d + 8, vld = dv + 8;
  const int buf_elems = WA_KT * (qld + vld);     // one tile's keys and values; two tiles in turn
  const int rep = a.heads / a.kv_heads;
  const int HR = a.heads_per_tile;
  const int chunks = (rep + HR - 1) / HR;
  const int g = blockIdx.y / chunks, hc = blockIdx.y - g * chunks;
  const unsigned bx = gridDim.x - 1 - blockIdx.x;
  const int64_t t0 = a.blocks != nullptr ? a.blocks[2 * bx] : bx;
  const int nt = a.blocks != nullptr ? a.blocks[2 * bx + 1] : 1;
  const int b = a.tok_req != nullptr ? a.tok_req[t0] : (int)t0;
  const int32_t* table = a.req_to_token + a.req_pool_indices[b] * a.req_to_token_stride;
  const int h0 = g * rep + hc * HR;
  const int nh = min(HR, rep - hc * HR);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int dch = d / 8, vch = dv / 8;           // 16-byte chunks per row
  const int live_rows = nt * HR;                 // rows at or past this hold no (token, head)
  using Frag = typename Mfma<T>::frag;
  // this lane's row (the column of its score and result tiles): query li of the wave's sixteen, features 32 c + 8 lg .. + 7
  const int row = 16 * wv + li;
  const int tl = row / HR, hl = row - tl * HR;
  const bool row_ok = tl < nt && hl < nh;
  const int rp = row_ok ? (int)a.positions[t0 + tl] : -1;
  Frag qf[2 * CK];
  {
    const T* q = (const T*)a.q + (t0 + (row_ok ? tl : 0)) * a.q_token_stride + (int64_t)(h0 + (row_ok ? hl : 0)) * a.q_head_stride + 8 * lg;
#pragma unroll
    for (int c = 0; c < 2 * CK; ++c) {
      Vec<T, 8> val;
#pragma unroll
      for (int x = 0; x < 8; ++x) val.v[x] = from_f32<T>(0.f);
      if (32 * c < d && row_ok) val = ldvec<T, 8>(q + 32 * c);
      qf[c] = __builtin_bit_cast(Frag, val);
    }
  }
  const int first = (int)a.positions[t0];
  const int last = first + nt - 1;
  const int lowest = a.window > 0 ? max(0, first - a.window + 1) : 0;
  const int split = blockIdx.z;
  const int all_lo = lowest / WA_KT, all_hi = last / WA_KT + 1;
  // pooled rows that the run's last token sees come first on the walk: ptiles tiles of them, then the window's tiles
  const int nb_run = (a.pool > 0 && a.window > 0 && last - a.window + 1 >= a.pool) ? (last - a.window + 1) / a.pool : 0;
  const int ptiles = (nb_run + WA_KT - 1) / WA_KT;
  const int ntiles = ptiles + all_hi - all_lo;
  const int per = (ntiles + a.num_splits - 1) / a.num_splits;
  const int tile_lo = split * per, tile_hi = min(ntiles, tile_lo + per);
  const int nblk = dv / 16;
  // running maximum of the row (the same in its four lanes) and this lane's share of the running sum
  float run_m = WA_NEG, run_l = 0.f;
  if (a.sink != nullptr && split == 0) { run_m = a.sink[h0 + min(hl, nh - 1)]; run_l = lg == 0 ? 1.f : 0.f; }
  f32x4 acc[4 * CT];
#pragma unroll
  for (int c = 0; c < 4 * CT; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  const T* kc = (const T*)a.k_cache;
  const T* vc = (const T*)a.v_cache;
  Vec<T, 8> kreg[CK], vreg[CT];
  int64_t ksrc[CK], vsrc[CT];
  int kkey[CK], kch[CK], vkey[CT], vchk[CT];     // (key, chunk) of this thread's pieces of a tile; past the last one: the last
#pragma unroll
  for (int u = 0; u < CK; ++u) { const int e = min(tid + 256 * u, WA_KT * dch - 1); kkey[u] = e / dch; kch[u] = 8 * (e - kkey[u] * dch); }
#pragma unroll
  for (int u = 0; u < CT; ++u) { const int e = min(tid + 256 * u, WA_KT * vch - 1); vkey[u] = e / vch; vchk[u] = 8 * (e - vkey[u] * vch); }
  // every load is unconditional: a piece past the tile's last one is the last one again (and never stored), keys outside
  // [0, last] (pooled rows past the last one the run sees) are clamped to a valid row (and masked below)
  auto load_slots = [&](int tile) {
    const bool ptile = tile < ptiles;
    const int j0 = (ptile ? tile : all_lo + tile - ptiles) * WA_KT;
    kc = (const T*)(ptile ? a.pooled_k : a.k_cache);
    vc = (const T*)(ptile ? a.pooled_v : a.v_cache);
    auto slot = [&](int j) -> int64_t { return ptile ? table[min(j, nb_run - 1) * a.pool + a.pool - 1] / a.pool_div : table[min(j, last)]; };
#pragma unroll
    for (int u = 0; u < CK; ++u) ksrc[u] = (slot(j0 + kkey[u]) * a.kv_heads + g) * d + kch[u];
#pragma unroll
    for (int u = 0; u < CT; ++u) vsrc[u] = (slot(j0 + vkey[u]) * a.kv_heads + g) * dv + vchk[u];
  };
  auto request = [&]() {
#pragma unroll
    for (int u = 0; u < CK; ++u) kreg[u] = ldvec<T, 8>(kc + ksrc[u]);
#pragma unroll
    for (int u = 0; u < CT; ++u) vreg[u] = ldvec<T, 8>(vc + vsrc[u]);
  };
  if (tile_lo < tile_hi) {
    load_slots(tile_lo);
    request();
    load_slots(min(tile_lo + 1, tile_hi - 1));
  }
  for (int tile = tile_lo; tile < tile_hi; ++tile) {
    const bool ptile = tile < ptiles;
    const int j0 = (ptile ? tile : all_lo + tile - ptiles) * WA_KT;
    T* Ks = reinterpret_cast<T*>(smraw) + (tile & 1) * buf_elems;   // (its readers, two tiles back, passed the last barrier)
    T* Vs = Ks + WA_KT * qld;
#pragma unroll
    for (int u = 0; u < CK; ++u)
      if (tid + 256 * u < WA_KT * dch) lds_store16(Ks + kkey[u] * qld + kch[u], kreg[u]);
#pragma unroll
    for (int u = 0; u < CT; ++u)
      if (tid + 256 * u < WA_KT * vch) lds_store16(Vs + vkey[u] * vld + vchk[u], vreg[u]);
    __syncthreads();
    if (tile + 1 < tile_hi) {                    // in flight during this tile's products
      request();
      load_slots(min(tile + 2, tile_hi - 1));
    }
    if (16 * wv >= live_rows) continue;
    f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int c = 0; c < 2 * CK; ++c) {
      if (32 * c < d) {
        s[0] = Mfma<T>::run(lds_load16<Frag>(Ks + li * qld + 32 * c + 8 * lg), qf[c], s[0]);
        s[1] = Mfma<T>::run(lds_load16<Frag>(Ks + (16 + li) * qld + 32 * c + 8 * lg), qf[c], s[1]);
      }
    }
    // the lane holds eight scores of its row: keys 4 lg + x of both halves of the tile
    float alpha, sum = 0.f;
    Vec<T, 8> p8;      // key slots 8 lg + i of the product with V: the keys above, in that order
    // A score is rounded where it is scaled, in both forms: a row's weights do not depend on which rows share its tiles.
    auto weigh = [&](auto whole) {
#pragma clang fp contract(off)
      bool seen[8];
      float x8[8], mx = run_m;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int j = j0 + 16 * (i >> 2) + 4 * lg + (i & 3);
        seen[i] = whole.value || (ptile ? (rp >= 0 && j * a.pool + a.pool - 1 <= rp - a.window)
                                        : (j <= rp && (a.window <= 0 || rp - j < a.window)));
        x8[i] = seen[i] ? s[i >> 2][i & 3] * a.scale : WA_NEG;
        mx = fmaxf(mx, x8[i]);
      }
      mx = max_xor<16>(mx);
      mx = max_xor<32>(mx);
      alpha = __expf(run_m - mx);
      run_m = mx;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float pe = seen[i] ? __expf(x8[i] - mx) : 0.f;
        sum += pe;
        p8.v[i] = from_f32<T>(pe);
      }
    };
    // every row of the run sees every key of the tile (rows without a token compute what nobody stores)
    if (ptile ? (j0 + WA_KT) * a.pool - 1 <= first - a.window
              : j0 + WA_KT - 1 <= first && (a.window <= 0 || last - j0 < a.window))
      weigh(std::true_type());
    else
      weigh(std::false_type());
    run_l = run_l * alpha + sum;
    if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0) {
#pragma unroll
      for (int c = 0; c < 4 * CT; ++c) acc[c] *= alpha;
    }
    const Frag pf = __builtin_bit_cast(Frag, p8);
    const T* vrow = Vs + (4 * lg + (li >> 2)) * vld + 4 * (li & 3);
#pragma unroll
    for (int c = 0; c < 4 * CT; ++c) {
      if (c < nblk) {
        typename TrRead<T>::v4 both[2] = {TrRead<T>::run(vrow + 16 * c), TrRead<T>::run(vrow + 16 * vld + 16 * c)};
        acc[c] = Mfma<T>::run(__builtin_bit_cast(Frag, both), pf, acc[c]);
      }
    }
  }
  run_l = sum_xor<32>(sum_xor<16>(run_l));
  if (!row_ok) return;
  // the lane holds features 16 c + 4 lg + x of its row
  if (a.num_splits > 1) {
    float* part = a.partial + (((int64_t)split * a.tokens + t0 + tl) * a.heads + h0 + hl) * (dv + 2);
#pragma unroll
    for (int c = 0; c < 4 * CT; ++c)
      if (c < nblk)
#pragma unroll
        for (int x = 0; x < 4; ++x) part[16 * c + 4 * lg + x] = acc[c][x];
    if (lg == 0) { part[dv] = run_m; part[dv + 1] = run_l; }
    return;
  }
  float mul = run_l > 0.f ? 1.f : 0.f;
  const float den = run_l > 0.f ? run_l : 1.f;
  if (a.gate != nullptr) mul *= wa_sigmoid(to_f32(((const T*)a.gate)[(t0 + tl) * a.gate_token_stride + h0 + hl]));
  T* out = (T*)a.out + (t0 + tl) * a.out_token_stride + (int64_t)(h0 + hl) * a.out_head_stride + 4 * lg;
  const bool four = (reinterpret_cast<uintptr_t>(a.out) & 7) == 0 && ((a.out_token_stride | a.out_head_stride) & 3) == 0;
#pragma unroll
  for (int c = 0; c < 4 * CT; ++c) {
    if (c >= nblk) continue;
    Vec<T, 4> w;
#pragma unroll
    for (int x = 0; x < 4; ++x) w.v[x] = from_f32<T>(acc[c][x] / den * mul);
    if (four) {
      stvec<T, 4>(out + 16 * c, w);
    } else {
#pragma unroll
      for (int x = 0; x < 4; ++x) out[16 * c + x] = w.v[x];
    }
  }
}

// One workgroup per token of the step; only a token whose position ends a block of `pool` does anything: it averages the
// block's cached rows into the pooled buffers' row for the block.  A row is kw key features followed (in another buffer) by
// vw value features, taken V at a time (16 bytes when the shapes allow, else one); the workgroup's threads form R lanes of
// rows x C columns of such vectors, lane r sums rows r, r + R, ... in fp32, the lanes' sums meet in LDS in lane order, one
// multiplication by 1 / pool.  The order of the additions depends on the shapes alone, never on how a prompt was cut.
template <typename T, int V>
__global__ __launch_bounds__(256) void pool_kv_blocks_kernel(T* __restrict__ pk, T* __restrict__ pv, const T* __restrict__ kc,
                                                             const T* __restrict__ vc, const int32_t* __restrict__ req_to_token,
                                                             const int64_t* __restrict__ req_pool_indices,
                                                             const int32_t* __restrict__ tok_req,
                                                             const int64_t* __restrict__ positions, int64_t req_to_token_stride,
                                                             int kw, int vw, int pool, int pool_div) {
  __shared__ float part[256 * V];
  const int64_t t = blockIdx.x;
  const int pos = (int)positions[t];
  if ((pos + 1) % pool != 0) return;
  const int b = tok_req != nullptr ? tok_req[t] : (int)t;
  const int32_t* table = req_to_token + req_pool_indices[b] * req_to_token_stride + (pos - pool + 1);
  const int64_t dst = table[pool - 1] / pool_div;
  const float inv = 1.0f / (float)pool;
  const int nk = kw / V, nv = (kw + vw) / V;           // vectors per row: keys first, then values
  const int C = min(nv, 256);                          // columns handled at a time
  int R = 256 / C;                                     // lanes of rows
  R = min(R, pool);
  const int tid = threadIdx.x;
  const int col = tid % C, lane = tid / C;
  for (int c0 = 0; c0 < nv; c0 += C) {
    const int c = c0 + col;
    const bool live = lane < R && c < nv;
    const bool isk = c < nk;
    const T* src = isk ? kc : vc;
    const int w = isk ? kw : vw;
    const int off = (isk ? c : c - nk) * V;
    float acc[V];
#pragma unroll
    for (int k = 0; k < V; ++k) acc[k] = 0.f;
    if (live) {
      int j = lane;
      for (; j + 3 * R < pool; j += 4 * R) {           // four rows in flight
        const Vec<T, V> a0 = ldvec<T, V>(src + (int64_t)table[j] * w + off);
        const Vec<T, V> a1 = ldvec<T, V>(src + (int64_t)table[j + R] * w + off);
        const Vec<T, V> a2 = ldvec<T, V>(src + (int64_t)table[j + 2 * R] * w + off);
        const Vec<T, V> a3 = ldvec<T, V>(src + (int64_t)table[j + 3 * R] * w + off);
#pragma unroll
        for (int k = 0; k < V; ++k) acc[k] = ((acc[k] + to_f32(a0.v[k])) + to_f32(a1.v[k])) + (to_f32(a2.v[k]) + to_f32(a3.v[k]));
      }
      for (; j < pool; j += R) {
        const Vec<T, V> a0 = ldvec<T, V>(src + (int64_t)table[j] * w + off);
#pragma unroll
        for (int k = 0; k < V; ++k) acc[k] += to_f32(a0.v[k]);
      }
    }
    __syncthreads();                                   // the last pass's readers are done
    if (live) {
#pragma unroll
      for (int k = 0; k < V; ++k) part[(lane * C + col) * V + k] = acc[k];
    }
    __syncthreads();
    if (live && lane == 0) {
      Vec<T, V> out;
#pragma unroll
      for (int k = 0; k < V; ++k) {
        float sum = part[col * V + k];
        for (int r = 1; r < R; ++r) sum += part[(r * C + col) * V + k];
        out.v[k] = from_f32<T>(sum * inv);
      }
      stvec<T, V>((isk ? pk : pv) + dst * w + off, out);
    }
  }
}

inline bool wa_mfma_shape(int dtype, int d, int dv) {
  return dtype != MI355_F32 && d % 32 == 0 && dv % 16 == 0 && d <= WAM_MAX && dv <= WAM_MAX;
}

template <typename T> int launch_window(const WaArgs& a, dim3 grid, bool mfma, hipStream_t stream) {
  if constexpr (!std::is_same<T, float>::value) {
    if (mfma) {
      const size_t lds = 2 * (size_t)WA_KT * (a.d + 8 + a.dv + 8) * sizeof(T);
#define MI355_WA_LAUNCH(CT, CK, FULL)                                                                                          \
  do {                                                                                                                         \
    if (lds > 64 * 1024) {                                                                                                     \
      hipError_t e = hipFuncSetAttribute((const void*)window_attention_mfma_kernel<T, CT, CK, FULL>,                           \
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                                \
      MI355_REQUIRE(e == hipSuccess, MI355_ERR_LAUNCH, "window_attention: %zu bytes of LDS refused", lds);                     \
    }                                                                                                                          \
    hipLaunchKernelGGL((window_attention_mfma_kernel<T, CT, CK, FULL>), grid, dim3(256), lds, stream, a);                      \
  } while (0)
#define MI355_WA_KEYS(CT)                                                                                                      \
  do {                                                                                                                         \
    if (a.d <= 64) MI355_WA_LAUNCH(CT, 1, false);                                                                              \
    else if (a.d <= 128) MI355_WA_LAUNCH(CT, 2, false);                                                                        \
    else MI355_WA_LAUNCH(CT, 4, false);                                                                                        \
  } while (0)
      if (a.d == 64 && a.dv == 64) MI355_WA_LAUNCH(1, 1, true);
      else if (a.d == 128 && a.dv == 128) MI355_WA_LAUNCH(2, 2, true);
      else if (a.dv <= 64) MI355_WA_KEYS(1);
      else if (a.dv <= 128) MI355_WA_KEYS(2);
      else MI355_WA_KEYS(4);
#undef MI355_WA_KEYS
#undef MI355_WA_LAUNCH
      return MI355_OK;
    }
  }
  const size_t lds = ((size_t)WA_ROWS * a.d + (size_t)WA_KT * (a.d + 1) + (size_t)WA_KT * a.dv + WA_ROWS * WA_KT) * sizeof(float);
  if (lds > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)window_attention_valu_kernel<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    MI355_REQUIRE(e == hipSuccess, MI355_ERR_LAUNCH, "window_attention: %zu bytes of LDS refused", lds);
  }
  hipLaunchKernelGGL((window_attention_valu_kernel<T>), grid, dim3(256), lds, stream, a);
  return MI355_OK;
}

inline int wa_heads_per_tile(int heads, int kv_heads, int rows) { return std::min(heads / kv_heads, rows); }

}  // namespace
}  // namespace mi355

using namespace mi355;

int mi355_window_attention_block_tokens(int heads, int kv_heads, int head_dim, int v_head_dim, int dtype) {
  if (heads <= 0 || kv_heads <= 0 || heads % kv_heads) return 0;
  const int rows = wa_mfma_shape(dtype, head_dim, v_head_dim) ? WAM_ROWS : WA_ROWS;
  return std::max(1, rows / wa_heads_per_tile(heads, kv_heads, rows));
}

int mi355_window_attention(void* out, const void* q, const void* k_cache, const void* v_cache, const int32_t* req_to_token,
                           const int64_t* req_pool_indices, const int32_t* tok_req, const int64_t* positions,
                           const int32_t* blocks, int64_t num_blocks, const float* sink, int64_t q_token_stride,
                           int64_t q_head_stride, int64_t out_token_stride, int64_t out_head_stride, int64_t req_to_token_stride,
                           int heads, int kv_heads, int head_dim, int v_head_dim, int window, float scale, int num_splits,
                           float* split_scratch, int64_t tokens, int max_run, int dtype, void* stream) {
  return mi355_window_attention_pooled(out, q, k_cache, v_cache, nullptr, nullptr, req_to_token, req_pool_indices, tok_req, positions,
                                       blocks, num_blocks, sink, nullptr, 0, q_token_stride, q_head_stride, out_token_stride,
                                       out_head_stride, req_to_token_stride, heads, kv_heads, head_dim, v_head_dim, window, 0, 1,
                                       scale, num_splits, split_scratch, tokens, max_run, dtype, stream);
}

int mi355_window_attention_pooled(void* out, const void* q, const void* k_cache, const void* v_cache, const void* pooled_k,
                                  const void* pooled_v, const int32_t* req_to_token, const int64_t* req_pool_indices,
                                  const int32_t* tok_req, const int64_t* positions, const int32_t* blocks, int64_t num_blocks,
                                  const float* sink, const void* head_gate, int64_t gate_token_stride, int64_t q_token_stride,
                                  int64_t q_head_stride, int64_t out_token_stride, int64_t out_head_stride,
                                  int64_t req_to_token_stride, int heads, int kv_heads, int head_dim, int v_head_dim, int window,
                                  int pool, int pool_div, float scale, int num_splits, float* split_scratch, int64_t tokens,
                                  int max_run, int dtype, void* stream) {
  MI355_REQUIRE(pool >= 0 && pool_div >= 1 && (pool == 0 || (pooled_k && pooled_v && window > 0)), MI355_ERR_INVALID,
                "window_attention: averaged blocks need their buffers and a window");
  MI355_REQUIRE(head_gate == nullptr || gate_token_stride >= heads, MI355_ERR_INVALID, "window_attention: bad gate stride");
  MI355_REQUIRE(num_splits >= 1 && num_splits <= 64 && (num_splits == 1 || (split_scratch && blocks == nullptr)), MI355_ERR_INVALID,
                "window_attention: key splits serve launches of one token per run and need scratch");
  MI355_REQUIRE(out && q && k_cache && v_cache && req_to_token && req_pool_indices && positions, MI355_ERR_INVALID,
                "window_attention: null pointer");
  MI355_REQUIRE(heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && head_dim > 0 && v_head_dim > 0 && tokens >= 0 &&
                    num_blocks >= 0, MI355_ERR_INVALID, "window_attention: bad shape");
  MI355_REQUIRE(head_dim <= 512 && v_head_dim <= 256, MI355_ERR_UNSUPPORTED, "window_attention: head width %d / %d not served",
                head_dim, v_head_dim);
  MI355_REQUIRE(blocks != nullptr || num_blocks == tokens, MI355_ERR_INVALID, "window_attention: without runs, one block per token");
  if (num_blocks == 0) return MI355_OK;
  WaArgs a;
  a.out = out; a.q = q; a.k_cache = k_cache; a.v_cache = v_cache; a.req_to_token = req_to_token;
  a.req_pool_indices = req_pool_indices; a.tok_req = tok_req; a.positions = positions; a.blocks = blocks; a.sink = sink;
  a.pooled_k = pooled_k; a.pooled_v = pooled_v; a.gate = head_gate; a.gate_token_stride = gate_token_stride; a.pool = pool;
  a.pool_div = pool_div;
  a.q_token_stride = q_token_stride; a.q_head_stride = q_head_stride; a.out_token_stride = out_token_stride;
  a.out_head_stride = out_head_stride; a.req_to_token_stride = req_to_token_stride; a.tokens = tokens; a.heads = heads;
  // the matrix-core kernel needs 16-byte rows everywhere; a caller whose q is laid out otherwise gets the vector-ALU kernel,
  // whose runs are shorter: max_run says how long the caller's runs may be, and a launch that cannot take them is refused
  const bool mfma = wa_mfma_shape(dtype, head_dim, v_head_dim) && q_token_stride % 8 == 0 && q_head_stride % 8 == 0 &&
                    aligned16(q) && aligned16(k_cache) && aligned16(v_cache) && (pool == 0 || (aligned16(pooled_k) && aligned16(pooled_v)));
  const int rows = mfma ? WAM_ROWS : WA_ROWS;
  a.kv_heads = kv_heads; a.d = head_dim; a.dv = v_head_dim; a.heads_per_tile = wa_heads_per_tile(heads, kv_heads, rows);
  a.window = window; a.scale = scale; a.num_splits = num_splits; a.partial = split_scratch;
  const int tokens_per_tile = std::max(1, rows / a.heads_per_tile);
  MI355_REQUIRE(max_run >= 1 && max_run <= tokens_per_tile, MI355_ERR_UNSUPPORTED,
                "window_attention: runs of up to %d tokens, this launch takes %d", max_run, tokens_per_tile);
  const int rep = heads / kv_heads;
  const int chunks = (rep + a.heads_per_tile - 1) / a.heads_per_tile;
  const dim3 grid((unsigned)num_blocks, (unsigned)(kv_heads * chunks), (unsigned)num_splits);
  MI355_REQUIRE(kv_heads * chunks <= 65535, MI355_ERR_UNSUPPORTED, "window_attention: too many heads");
  int rc = MI355_OK;
  MI355_DISPATCH_DTYPE(dtype, "window_attention", { rc = launch_window<T>(a, grid, mfma, (hipStream_t)stream); });
  if (rc != MI355_OK) return rc;
  MI355_CHECK_LAUNCH("window_attention");
  if (num_splits > 1) {
    const unsigned g2 = (unsigned)(tokens * heads);
    MI355_DISPATCH_DTYPE(dtype, "window_attention", {
      hipLaunchKernelGGL((window_attention_merge_kernel<T>), dim3(g2), dim3(256), 0, (hipStream_t)stream, (T*)out, split_scratch, tokens,
                         heads, v_head_dim, num_splits, out_token_stride, out_head_stride, (const T*)head_gate, gate_token_stride);
    });
    MI355_CHECK_LAUNCH("window_attention(merge)");
  }
  return MI355_OK;
}

int mi355_pool_kv_blocks(void* pooled_k, void* pooled_v, const void* k_cache, const void* v_cache, const int32_t* req_to_token,
                         const int64_t* req_pool_indices, const int32_t* tok_req, const int64_t* positions, int64_t tokens,
                         int64_t req_to_token_stride, int kv_heads, int head_dim, int v_head_dim, int pool, int pool_div, int dtype,
                         void* stream) {
  MI355_REQUIRE(pooled_k && pooled_v && k_cache && v_cache && req_to_token && req_pool_indices && positions, MI355_ERR_INVALID,
                "pool_kv_blocks: null pointer");
  MI355_REQUIRE(tokens >= 0 && tokens <= 0x7fffffff && kv_heads > 0 && head_dim > 0 && v_head_dim > 0 && pool >= 1 && pool_div >= 1,
                MI355_ERR_INVALID, "pool_kv_blocks: bad shape");
  if (tokens == 0) return MI355_OK;
  const int kw = kv_heads * head_dim, vw = kv_heads * v_head_dim;
  const int vecw = dtype == MI355_F32 ? 4 : 8;
  const bool vec = kw % vecw == 0 && vw % vecw == 0 && aligned16(pooled_k) && aligned16(pooled_v) && aligned16(k_cache) && aligned16(v_cache);
  MI355_DISPATCH_DTYPE(dtype, "pool_kv_blocks", {
    constexpr int V = 16 / sizeof(T);
    if (vec)
      hipLaunchKernelGGL((pool_kv_blocks_kernel<T, V>), dim3((unsigned)tokens), dim3(256), 0, (hipStream_t)stream, (T*)pooled_k,
                         (T*)pooled_v, (const T*)k_cache, (const T*)v_cache, req_to_token, req_pool_indices, tok_req, positions,
                         req_to_token_stride, kw, vw, pool, pool_div);
    else
      hipLaunchKernelGGL((pool_kv_blocks_kernel<T, 1>), dim3((unsigned)tokens), dim3(256), 0, (hipStream_t)stream, (T*)pooled_k,
                         (T*)pooled_v, (const T*)k_cache, (const T*)v_cache, req_to_token, req_pool_indices, tok_req, positions,
                         req_to_token_stride, kw, vw, pool, pool_div);
  });
  MI355_CHECK_LAUNCH("pool_kv_blocks");
  return MI355_OK;
}
