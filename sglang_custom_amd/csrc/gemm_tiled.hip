// Large-M projection GEMM  y[M, N] = x[M, K] @ W[N, K]^T  for gfx950, fp32 accumulation on the matrix
// cores: the prefill side of UnquantizedLinearMethod.apply
// (python/sglang/srt/layers/quantization/unquant.py:110-122) for 16-bit operands and of
// apply_fp8_linear (layers/quantization/fp8_utils.py:676-749) for fp8 W8A8 operands with per-token /
// per-channel scales, with the MLP's SiLU-and-mul (python/sglang/srt/models/llama.py:94-98,
// layers/activation.py:55-65) optionally applied in the epilogue.  The decode side (M <= 64) is the
// weight-streaming kernel in gemm.hip.
//
// Structure (one 512-thread workgroup per CU, 128 KiB of LDS, one 256 x 256 output tile):
//   * K is walked in tiles of 128 BYTES per row (64 16-bit or 128 fp8 elements); a tile's operands
//     live in LDS as four HALF-TILES of 128 rows x 128 bytes (x rows 0..127, x rows 128..255, W rows
//     0..127, W rows 128..255), two tiles resident;
//   * the load unit writes LDS itself (16 bytes a lane, 8 rows x 128 B per wave-instruction: whole cache
//     lines; buffer loads, in the grouped kernel global ones);
//   * the eight waves form two groups of four (group = row half of the tile, wave-in-group = 64
//     output columns).  A wave alternates a READ slot (its 8 load requests, then 24 ds_read_b128: its A
//     and B fragments of a whole K tile) with a MATRIX slot (nothing but 64 x v_mfma_f32_16x16x32 on
//     16-bit operands, or 32 x v_mfma_scale_f32_16x16x128_f8f6f4 with unit block scales on fp8
//     operands: twice the 16-bit rate per byte staged); the groups run one slot apart, so on every
//     SIMD one wave's matrix work covers the other wave's LDS reads and load issue (a load-to-LDS
//     holds the issuing wave for ~40 cycles: anywhere in a matrix slot that time is lost to the
//     matrix pipe).  One s_barrier per slot;
//   * a half-tile is requested by the group that owns it, one to two tiles ahead, as soon as its LDS
//     region is free, and is waited for (vmcnt(0)) by the requesting waves at the end of their next
//     MATRIX slot: at least one slot in flight, one barrier before its first reader;
//   * LDS rows are 128 bytes; the 16-byte chunk index is XOR-ed with a function of the row on the
//     SOURCE address of the load (the load unit writes lane-linear) and again on the fragment read:
//     conflict-free ds_read_b128 for 16-byte (16-bit) and 32-byte (fp8) fragments.
//   * W rows are assigned to MFMA row slots so that a lane ends up with two runs of 8 consecutive output
//     columns, 32 apart (or, for SiLU-and-mul, 8 gate columns and the 8 matching up columns): a 16-byte store
//     of a wave writes 64 bytes in a row of each of its 16 rows, and needs no cross-lane traffic (16 columns in a row for a
//     lane leave every second 16 bytes of a line to the next store: 4096 x 4096, K 2048, one tile a CU, 56.2 us instead of 53.2);
//   * workgroup -> tile: consecutive workgroups round-robin over the 8 XCDs, so workgroups b and
//     b + 8 share an L2; each XCD works through 8 x 4 blocks of tiles (32 CUs = one block);
//   * a workgroup stays on its CU and takes tile after tile: the K tiles of all its output tiles are one stream of requests, so
//     the next tile's operands are on their way while the last one's results are written (a group writes its results in front of
//     its first READ slot of the next tile, next to the other group's last MATRIX slot; with RoPE both write at once, see there);
//   * tiles beyond whole rounds of 256 may be split over K, their sums added by a second launch that also runs the epilogue.
// A tile that ends costs what its K tiles do not: with a workgroup per tile 10.6 us (7725 x 8192 columns, K 2048: 200 us of which the K
// tiles take 160), as it is 6.5.  us, a workgroup per tile -> now: 7725 x 8192 x K 2048 200.2 -> 187.5, K 4096 361 -> 346; 4605 x 6144 x K
// 4096 169 -> 163; 2 x 14336 x K 4096 with SiLU-and-mul 771 -> 751; 4096 x K 14336 511 -> 500.  (Waiting for the next tile's requests and
// not for the stores behind them gained nothing more; four waves of 128 x 128, a third fewer LDS reads, 2 to 9 % slower: a K tile with x = 0
// takes 1.03 us instead of 0.945, for nothing covers a wave's own LDS reads and requests but its MFMAs.)  That the walk through the tiles is fixed
// costs nothing over many rounds: 65536 rows, a workgroup per tile -> now, ms, 2 x 14336 columns 10.56 -> 10.29, 4096 x K 14336 5.19 -> 5.06, 4096
// x K 4096 1.50 -> 1.43; the first token of 64 x 1024 682 -> 661.
// What bounds it: the card's power.  The MFMAs of a K tile take 2048 of its 2320 cycles (88 %), but with random operands the
// clock falls to 1.7 GHz (4096 x 4096 x 4096: 98 us; with x = 0 2.17 GHz and 77).  So the order of a matrix slot's MFMAs counts: W fragments
// go forth in one row of x fragments and back in the next, one operand of every MFMA the last one's (a loop of MFMAs alone 2045 ->
// 2085 TFLOP/s, with the LDS reads 1797 -> 1829; 32 x 32 x 16 MFMAs 1795 and 1595).  A Llama-3-8B
// prefill of 4605 tokens 54.84 -> 54.00 ms.
#include "common.cuh"

namespace mi355 {
namespace {

constexpr int GT_HALF = 128 * 128;      // bytes of one half-tile
constexpr int GT_STAGE = 4 * GT_HALF;   // one K tile: x (2 halves) + W (2 halves)
constexpr int GT_LDS = 2 * GT_STAGE;    // 131072
constexpr int64_t GT_MAX_STRIDE = (1 << 23) - 8;   // elements between rows of x and W up to which 128 rows are addressed with 31 bits
constexpr int64_t GT_MAX_ROW = (1ll << 31) - 128;  // bytes of a row, counted with 31 bits

struct GemmTiledParams {
  const void* x;
  const void* w;
  const void* bias;
  void* y;
  const float* x_scale;   // fp8: per-token scales [M]
  const float* w_scale;   // fp8: per-channel scales [N]
  int M, N, K;      // N = rows of W
  int64_t ldx;      // elements between rows of x
  int ldy;          // elements between rows of y
  int mt, nt;       // output tiles along M and N
  int snt, nsuper;  // 8 x 4 blocks of tiles: count along N, total
  // tail tiles whose K is split over `splits` workgroups each (0: none): tiles at .. `full` - 1 in tile order are computed whole
  int full, tail, splits;
  float* part;      // [splits, tail, 8 waves, 8 row groups, 4 column groups, 64 lanes, 4] sums of the splits
  // EPI 2 (qkv projection + RoPE + KV-cache write)
  const int64_t* positions;   // [M]
  const void* cos_sin;        // [max_pos, 128]: cos | sin, fp32 or the tensor dtype
  int cs_f32;
  int hq, hkv;                // local query / kv heads (head_dim 128)
  void* k_buffer;             // [slots, hkv, 128], or head-major [hkv, slots, 128]
  void* v_buffer;
  int64_t kv_slot, kv_head;   // elements between consecutive slots / kv heads of the two buffers
  const void* loc;            // [M] cache slot of each row, int64 or int32
  int loc_i32;
  // EPI 3 (grouped: every 256-row tile of x multiplies the weight matrix of the tile's own expert)
  const int32_t* row_map;      // [M] source row of x for output row m; negative: a padding row.  Null: none is
  int gather;                  // whether row m reads row row_map[m] of x, or row m itself
  const int32_t* tile_expert;  // [mt] which of the stacked weight matrices tile tm uses
  const int32_t* tiles_used;   // device scalar: tiles at or past it are not computed
  int64_t w_expert_stride;     // elements between consecutive weight matrices
  int act;                     // on the result: 1 erf-GELU, 2 the square of relu
};

__device__ __forceinline__ void glds16(const void* g, char* l) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                   (__attribute__((address_space(3))) void*)l, 16, 0, 0);
}

typedef int i32x8 __attribute__((ext_vector_type(8)));

// XOR applied to the 16-byte chunk index of LDS row r (depends on r & 15 only).  16-bit fragments
// are one chunk per lane (chunk 4 kk + (lane >> 4)), fp8 fragments two (chunks 2 (lane >> 4) + {0, 1}):
// each needs its own function for the 16-lane service groups of ds_read_b128 to hit 16 distinct
// 16-byte bank groups.
template <bool FP8> __device__ __forceinline__ int gt_swz(int r) {
  return FP8 ? (((r >> 1) & 1) | (((r >> 3) & 1) << 2)) : ((r >> 1) & 7);
}

// T: output dtype and, for 16-bit GEMMs, the operand dtype.  FP8: operands are OCP e4m3fn bytes.
// EPI 0: y = T(acc (+ bias)); EPI 1: W = [gate; up] (N = 2 I rows), y[m, j] = silu_mul(T(gate_j), T(up_j));
// EPI 4: y = T(gelu_erf(T(acc))); EPI 5: as EPI 1 with y[m, j] = T(gelu_tanh(T(gate_j)) T(up_j)).  fp8: acc is first scaled, (acc * x_scale[m]) * w_scale[n].
// Epilogue of the qkv projection (EPI 2): neox RoPE over the whole 128-wide head on the q and k heads with
// the rounding points of mi355_rope_inplace (cos / sin -> T; every product and sum rounds to T on its own, so
// no contraction here); rotated q / k and plain v go to y, the k and v rows also to the KV cache.
// The lane holds, for each of its 8 rows, columns d0 .. d0 + 7 of one head (acc[mi][0..1]) and their rotation
// partners d0 + 64 .. d0 + 71 (acc[mi][2..3]).  Bound by the latency of its loads (positions, and the cos / sin rows that they name): all
// positions are requested first, cos / sin, cache slots and scales two or three rows ahead of the row that is worked on, and both groups of waves are
// here at once (TOGETHER in the kernel), or the second's chain would begin where the first's ends.  6144 columns, K 4096, us at 4605, 7725
// and 16384 rows of bf16: the groups one behind the other, two rows' loads at a time and 14 registers in scratch memory 192.6, 297, 609; no register
// there (see the kernel) 191, 297, 605; the groups together 188.6, 290, 590; rows ahead 185, 289, 583 (a workgroup per tile 191.7, 297, 598).
// fp8 at 4605 and 7725: 111, 170; 108, 166; 106, 161; 105, 159 (105.6, 165).
template <typename T, bool FP8, bool CSF32, int NM>
__device__ __forceinline__ void qkv_rope_epilogue(const GemmTiledParams& p, f32x4 (&acc)[NM][4], int mbase, int tn, int wc, int q4) {
#pragma clang fp contract(off)
  T* yg = (T*)p.y;
  const int head = 2 * tn + (wc >> 1), d0 = (wc & 1) * 32 + q4 * 8;
  const int col0 = head * 128 + d0;
  const bool rot = head < p.hq + p.hkv;
  T* cache_dst = nullptr;
  if (head >= p.hq + p.hkv) cache_dst = (T*)p.v_buffer + (int64_t)(head - p.hq - p.hkv) * p.kv_head + d0;
  else if (head >= p.hq) cache_dst = (T*)p.k_buffer + (int64_t)(head - p.hq) * p.kv_head + d0;
  float slo[8], shi[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    slo[j] = FP8 ? p.w_scale[col0 + j] : 1.f;
    shi[j] = FP8 ? p.w_scale[col0 + 64 + j] : 1.f;
  }
  // R - 1 rows' cos / sin, slots and scales are on their way in front of the row that is worked on (register budget)
  constexpr int R = CSF32 ? 3 : 4;
  auto row_of = [&](int mi) { return min(mbase + mi * 16, p.M - 1); };
  int posv[NM], slotv[R];   // positions and slot numbers fit 31 bits (the host checks the slot count)
  using CS = std::conditional_t<CSF32, float, T>;
  Vec<CS, 8> c[R], sn[R];
  float sxm[R];
#pragma unroll
  for (int mi = 0; mi < NM; ++mi) posv[mi] = (int)p.positions[row_of(mi)];
  auto request = [&](int mi) {   // (v heads read cos / sin too and ignore them: the branch below is wave-uniform)
    const int i = mi % R, m = row_of(mi);
    const int64_t pos = posv[mi];
    const CS* cs = (const CS*)p.cos_sin + pos * 128 + d0;
#pragma unroll
    for (int at = 0; at < 8; at += V16<CS>::n) {
      const auto cv = ldvec<CS, V16<CS>::n>(cs + at), sv = ldvec<CS, V16<CS>::n>(cs + 64 + at);
#pragma unroll
      for (int j = 0; j < V16<CS>::n; ++j) { c[i].v[at + j] = cv.v[j]; sn[i].v[at + j] = sv.v[j]; }
    }
    slotv[i] = cache_dst == nullptr ? 0 : p.loc_i32 ? ((const int32_t*)p.loc)[m] : (int)((const int64_t*)p.loc)[m];
    sxm[i] = FP8 ? p.x_scale[m] : 1.f;
  };
#pragma unroll
  for (int mi = 0; mi < min(R - 1, NM); ++mi) request(mi);
#pragma unroll
  for (int mi = 0; mi < NM; ++mi) {
    if (mi + R - 1 < NM) request(mi + R - 1);
    const int i = mi % R, m = mbase + mi * 16;
    float x1[8], x2[8];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float lo = acc[mi][h][r], hi = acc[mi][2 + h][r];
        if (FP8) { lo = (lo * sxm[i]) * slo[h * 4 + r]; hi = (hi * sxm[i]) * shi[h * 4 + r]; }
        round2_to<T>(lo, hi, x1[h * 4 + r], x2[h * 4 + r]);   // the projection's own result, rounded to T
      }
    Vec<T, 8> o1, o2;
    if (rot) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float cj = to_f32(c[i].v[j]), sj = to_f32(sn[i].v[j]);
        if constexpr (CSF32) round2_to<T>(cj, sj, cj, sj);   // a table of dtype T holds rounded values already
        float a1, a2, b1, b2;
        round2_to<T>(x1[j] * cj, x2[j] * sj, a1, a2);
        round2_to<T>(x2[j] * cj, x1[j] * sj, b1, b2);
        o1.v[j] = from_f32<T>(a1 - a2);
        o2.v[j] = from_f32<T>(b1 + b2);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) { o1.v[j] = from_f32<T>(x1[j]); o2.v[j] = from_f32<T>(x2[j]); }
    }
    if (m < p.M) {
      stvec<T, 8>(yg + (int64_t)m * p.ldy + col0, o1);
      stvec<T, 8>(yg + (int64_t)m * p.ldy + col0 + 64, o2);
      if (cache_dst != nullptr) {
        T* dst = cache_dst + (int64_t)slotv[i] * p.kv_slot;
        stvec<T, 8>(dst, o1);
        stvec<T, 8>(dst + 64, o2);
      }
    }
  }
  // (an end of its own for each kind of table: else the compiler joins the two forms' last stores and cuts one of them into pieces of 2 to 8 bytes)
  if constexpr (CSF32) asm volatile("; table in fp32" ::: "memory");
  else asm volatile("; table in the results' type" ::: "memory");
}

// Tile number `at` of the tile order: bands of 8 rows of tiles, blocks of 4 columns inside.
__device__ __forceinline__ void tile_of(const GemmTiledParams& p, int at, int& tm, int& tn) {
  const int band = at / (8 * p.nt), in = at - band * 8 * p.nt;
  const int rows = min(8, p.mt - 8 * band), col = in / (4 * rows), r = in - col * 4 * rows;
  tm = band * 8 + r % rows;
  tn = col * 4 + r / rows;
}

// erf-GELU for a 16-bit result: z Phi(z) with Phi(-u) = exp(-u^2 / 2) P(t), t = 1 / (1 + 0.42 u / sqrt 2), P the polynomial of degree 8 that is
// nearest to exp(x^2) erfc(x) / 2 over x in [0, 14] (fitted here to the least relative error, 1.1e-7); above zero z - z Phi(-z).  In fp32 its largest error
// is half of 0.5 z (1 + erff(z / sqrt 2))'s over [-8, 8] (2.4e-7; below -3, where 1 + erf cancels, it stays at 3e-6 of the result),
// rounded to 16 bits they have the same error to six digits.  Fifteen instructions and two of a quarter rate for erff's forty, which nothing
// covers in an epilogue: 32 experts' first product of 3000 x 4 rows, 2048 x 2048, 140 -> 131 us (113 without it); a dense one of 7725 x 8192
// columns, K 2048, about 45 us longer with it, for a launch of 61 to 67 of its own (4 TB/s).
__device__ __forceinline__ float gelu_erf(float z) {
  const float u = fabsf(z), t = __builtin_amdgcn_rcpf(fmaf(0.29698484809834996f, u, 1.0f));
  float p = 3.71014210e-02f;
  p = fmaf(p, t, -1.69227410e-01f);
  p = fmaf(p, t, 2.379644505e-01f);
  p = fmaf(p, t, -8.4074170e-02f);
  p = fmaf(p, t, 1.46434853e-01f);
  p = fmaf(p, t, 9.26121825e-02f);
  p = fmaf(p, t, 1.20913181e-01f);
  p = fmaf(p, t, 1.182676335e-01f);
  p = fmaf(p, t, 7.8031321e-06f);
  const float h = p * __builtin_amdgcn_exp2f(z * z * -0.72134752044448170f);
  return z > 0.f ? fmaf(-fminf(z, 30.f), h, z) : z * h;     // (infinity: itself; minus infinity and NaN: NaN, as by the formula)
}

// z / 2 (1 + tanh(sqrt(2 / pi) (z + 0.044715 z^3))) as z / (1 + e^(-2 ..)): nothing cancels below zero, and two instructions of a quarter rate for
// tanhf's thirty.  In the product's epilogue for a launch and two passes over the columns: a prompt of 4 x 1800 tokens through four layers of
// 2 x 5632 columns 3625 -> 3455 us in all, 3 x 360 1065 -> 991.
__device__ __forceinline__ float gelu_tanh_logistic(float z) {
  return z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-2.3022081985f * fmaf(0.044715f * z * z, z, z)));
}

constexpr bool gt_pairs(int epi) { return epi == 1 || epi == 5; }   // W = [gate; up]

// The results of NM groups of 16 rows (row mbase + 16 mi + r16 is lane (q4, r16)'s in group mi; mbase: the first group's first row).
// acc[mi][ni][r]: W slot 16 ni + 4 q4 + r of the wave's 64, which the load mapping made output column 32 (ni >> 1) + 8 q4 + 4 (ni & 1) + r
// (plain) or column 8 q4 + 4 (ni & 1) + r of gate (ni < 2) or up.  EPI 3: `live` rows of the tile are no padding.  BIAS: if there is one.  (With
// a form for each case in a small kernel the compiler joins their last stores, and cuts them into pieces of 2 to 8 bytes: the sums of 128 tail tiles
// 13.5 -> 16.0 us.)
template <typename T, int EPI, bool FP8, int NM, bool BIAS>
__device__ __forceinline__ void tile_epilogue(const GemmTiledParams& p, f32x4 (&acc)[NM][4], int m0, int tm, int tn, int wc, int q4, int r16,
                                              int live) {
  const int ncols = gt_pairs(EPI) ? (p.N >> 1) : p.N;   // output columns
  const int mbase = m0 + r16;
  T* yg = (T*)p.y;
  [[maybe_unused]] const T* bias = (const T*)p.bias;
  [[maybe_unused]] float sxm[NM];
#pragma unroll
  for (int mi = 0; mi < NM; ++mi) {
    const int m = mbase + mi * 16;
    sxm[mi] = FP8 && EPI != 2 ? p.x_scale[m < p.M ? m : p.M - 1] : 1.f;
  }
  if constexpr (EPI == 2) {
    if (p.cs_f32) qkv_rope_epilogue<T, FP8, true, NM>(p, acc, mbase, tn, wc, q4);
    else qkv_rope_epilogue<T, FP8, false, NM>(p, acc, mbase, tn, wc, q4);
  } else if (gt_pairs(EPI)) {
    const int j0 = tn * 128 + wc * 32 + q4 * 8;
    if (j0 < ncols) {
      float sg[8], su[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        sg[j] = FP8 ? p.w_scale[j0 + j] : 1.f;
        su[j] = FP8 ? p.w_scale[ncols + j0 + j] : 1.f;
      }
#pragma unroll
      for (int mi = 0; mi < NM; ++mi) {
        const int m = mbase + mi * 16;
        Vec<T, 8> o;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float gv = acc[mi][h][r], uv = acc[mi][2 + h][r];
            if (FP8) { gv = (gv * sxm[mi]) * sg[h * 4 + r]; uv = (uv * sxm[mi]) * su[h * 4 + r]; }
            o.v[h * 4 + r] = EPI == 5 ? from_f32<T>(gelu_tanh_logistic(round_to<T>(gv)) * round_to<T>(uv)) : silu_mul_one<T>(from_f32<T>(gv), from_f32<T>(uv));
          }
        if (m < p.M) stvec<T, 8>(yg + (int64_t)m * p.ldy + j0, o);
      }
    }
  } else {
    const int n0 = tn * 256 + wc * 64 + q4 * 8, n1 = n0 + 32;
    if (n0 < p.N) {
      float bv[16], sw[16];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        sw[j] = FP8 ? p.w_scale[n0 + j] : 1.f;
        sw[8 + j] = FP8 ? p.w_scale[min(n1, p.N - 8) + j] : 1.f;
      }
      if constexpr (BIAS) {
#pragma unroll
        for (int j = 0; j < 16; ++j) bv[j] = 0.f;
        if (bias != nullptr) {
          const Vec<T, 8> b0 = ldvec<T, 8>(bias + n0), b1 = ldvec<T, 8>(bias + min(n1, p.N - 8));
#pragma unroll
          for (int j = 0; j < 8; ++j) { bv[j] = to_f32(b0.v[j]); bv[8 + j] = to_f32(b1.v[j]); }
        }
      }
#pragma unroll
      for (int mi = 0; mi < NM; ++mi) {
        if (EPI == 3 && m0 - tm * 256 + mi * 16 >= live) break;   // (wave-uniform: no row of these groups is stored)
        const int m = mbase + mi * 16;
        Vec<T, 8> o0, o1;
#pragma unroll
        for (int ni = 0; ni < 2; ++ni)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float v0 = acc[mi][ni][r], v1 = acc[mi][2 + ni][r];
            if (FP8) { v0 = (v0 * sxm[mi]) * sw[ni * 4 + r]; v1 = (v1 * sxm[mi]) * sw[8 + ni * 4 + r]; }
            if constexpr (EPI == 4) {
              v0 = gelu_erf(round_to<T>(v0));
              v1 = gelu_erf(round_to<T>(v1));
            }
            if constexpr (EPI == 3) {
              if (p.act == 1) {
                v0 = gelu_erf(v0);
                v1 = gelu_erf(v1);
              } else if (p.act == 2) {
                v0 = fmaxf(v0, 0.f); v0 *= v0;
                v1 = fmaxf(v1, 0.f); v1 *= v1;
              }
            }
            if constexpr (BIAS) {
              v0 += bv[ni * 4 + r];
              v1 += bv[8 + ni * 4 + r];
            }
            o0.v[ni * 4 + r] = from_f32<T>(v0);
            o1.v[ni * 4 + r] = from_f32<T>(v1);
          }
        if (EPI == 3 ? m - tm * 256 < live : m < p.M) {
          stvec<T, 8>(yg + (int64_t)m * p.ldy + n0, o0);
          if (n1 < p.N) stvec<T, 8>(yg + (int64_t)m * p.ldy + n1, o1);
        }
      }
    }
  }
}

// The buffer that holds half h of a group's operand in tile (tm, tn), from its first row on: W for group 0 (waves of pairs: their gate or up
// rows), x for group 1.  Rows past the matrix read as zeros (of a gate, they are up rows); their results are not stored.
// WIDE: rows that lie further apart than a buffer's offsets reach: their address, and how many there are from it on (none: less than
// one; row `left` - 1 is the matrix's last one whatever its sign, and stands for those past it).
struct GtRows { const char* p; int64_t ld; int left; };
template <int EPI, int ES, bool WIDE>
__device__ __forceinline__ auto gt_half(const GemmTiledParams& p, int tm, int tn, int g, int wc, int h) {
  constexpr int NR = gt_pairs(EPI) ? 64 : 128;
  const int64_t row = g == 0 ? (int64_t)tn * (2 * NR) + h * NR + (gt_pairs(EPI) && (wc & 1) ? p.N >> 1 : 0) : (int64_t)tm * 256 + h * 128;
  const int64_t rows = g == 0 ? p.N : p.M, ld = (g == 0 ? (int64_t)p.K : p.ldx) * ES;
  if constexpr (WIDE) {
    return GtRows{(const char*)(g == 0 ? p.w : p.x) + row * ld, ld, (int)(rows - row)};
  } else {
    const int64_t bytes = row < rows ? min((rows - 1 - row) * ld + (int64_t)p.K * ES, (int64_t)0x7fffffff) : 0;
    return __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)(g == 0 ? p.w : p.x) + row * ld), 0, (int)bytes, 0x00020000);
  }
}
// 16 bytes a lane to LDS.  voff: bytes behind the half's first row (WIDE: 128 times the row, plus bytes), soff: bytes along the rows
__device__ __forceinline__ void gt_load(__amdgpu_buffer_rsrc_t r, char* l, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)l, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ void gt_load(const GtRows& r, char* l, int voff, int soff) {
  glds16(r.p + min(voff >> 7, r.left - 1) * r.ld + (voff & 127) + soff, l);
}

// What a workgroup works on: an output tile, or a split of a tail tile (K tiles t0 .. t0 + T - 1, sums to `part`).
struct GtItem { int tm, tn, t0, T; float* part; bool valid; };

// Item i of this workgroup.  Consecutive workgroups go to the eight XCDs in turn, and every XCD gets an equal run of the tiles in block
// order (bands of 8 rows, blocks of 4 columns inside): whole blocks in turn left some XCDs a round more than others where the last band is
// short -- 18 x 24 tiles: 72 on two XCDs and 40 on four, of 32 CUs each.  M = 4605, K = 4096: N = 6144 267 -> 190 us, N = 28672 846 -> 792;
// 7381 x 2048 -> 2 x 5632 302 -> 280.  Splits of tail tiles come last (whole tiles are a multiple of 256 then, an equal number for
// every workgroup); every XCD takes neighbouring ones, one stretch of K of all the tail's operands.
__device__ __forceinline__ GtItem gt_item(const GemmTiledParams& p, int i, int kt) {
  GtItem it{0, 0, 0, kt, nullptr, false};
  const int xcd = blockIdx.x & 7, li = blockIdx.x >> 3, wide = gridDim.x >> 3;
  const int whole = p.splits == 0 ? p.mt * p.nt : p.full, per = (whole + 7) >> 3, j = li + i * wide;
  if (j < per) {
    const int at = xcd * per + j;
    it.valid = at < whole;
    if (it.valid) tile_of(p, at, it.tm, it.tn);
  } else if (p.splits != 0 && j - per < wide) {
    int mine = li;
    asm volatile("" : "+s"(mine));    // (else the split is worked out in front of the tiles, and kept for all of them)
    const int tper = (p.tail * p.splits + 7) >> 3, u = xcd * tper + mine;
    it.valid = mine < tper && u < p.tail * p.splits;
    if (it.valid) {
      const int k = u / p.tail, t = u - k * p.tail;
      tile_of(p, p.full + t, it.tm, it.tn);
      it.part = p.part + ((int64_t)k * p.tail + t) * 65536;
      it.t0 = kt * k / p.splits;
      it.T = kt * (k + 1) / p.splits - it.t0;
    }
  }
  return it;
}

#define GT_SLOT_END()                                                                        \
  do {                                                                                       \
    __builtin_amdgcn_sched_barrier(0);                                                       \
    __builtin_amdgcn_s_barrier();                                                            \
    __builtin_amdgcn_sched_barrier(0);                                                       \
  } while (0)

template <typename T, int EPI, bool FP8, bool WIDE>
__global__ __launch_bounds__(512) void gemm_tiled_kernel(GemmTiledParams p) {
  extern __shared__ __attribute__((aligned(16))) char sm[];
  using frag = typename Mfma<T>::frag;
  constexpr int ES = FP8 ? 1 : 2;   // operand element bytes
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = wave >> 2, wc = wave & 3;
  const int kt = (p.K * ES) >> 7;   // K tiles of 128 bytes per row

  GtItem cur = gt_item(p, 0, kt);
  if (!cur.valid) return;

  // ---- the eight load instructions a wave issues per K tile -----------------------------------
  // A wave requests data only in its READ slot (a load-to-LDS holds the issuing wave ~40 cycles: in
  // front of or between the MFMAs of a matrix slot that time is lost to the matrix pipe, next to the
  // LDS reads of a READ slot it is covered by the other group's MFMAs).  Group 0 (READ slot 2t) requests
  // W of tile t + 1, both halves; group 1 (READ slot 2t + 1) requests x rows 128..255 of tile t + 1 and
  // x rows 0..127 of tile t + 2: each is free when requested (its last reader finished a slot earlier)
  // and is waited for -- by the waves that requested it, at the end of their MATRIX slot -- before
  // the barrier in front of the first slot that reads it.  A half-tile is 16 pieces of 8 rows x 128
  // bytes; wave wc of the group requests pieces 4 wc .. 4 wc + 3 of its group's two half-tiles:
  //   ldA: group 0 W rows 0..127 (tile t + 1), group 1 x rows 128..255 (tile t + 1)
  //   ldB: group 0 W rows 128..255 (tile t + 1), group 1 x rows 0..127 (tile t + 2)
  // A lane's offsets inside a half-tile's buffer are the same for every tile.
  int voff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int rr = (wc * 4 + i) * 8 + (lane >> 3);             // row inside the half-tile
    const int c = (lane & 7) ^ gt_swz<FP8>(rr);                // logical 16-byte chunk this lane fetches
    const int ni = (rr & 63) >> 4, ii = rr & 15, at8 = (ii >> 2) * 8 + (ni & 1) * 4 + (ii & 3);
    // EPI 2: a tile is two heads; wave wcb serves head 2 tn + (wcb >> 1), rotation pairs d and d + 64 with
    // d = 32 (wcb & 1) + at8: a lane ends with 8 d's and their partners.  Pairs: gt_half knows gate (ni < 2) from up.
    const int n = gt_pairs(EPI) ? (rr >> 6) * 32 + at8 : EPI == 2 ? (rr >> 6) * 32 + at8 + (ni >> 1) * 64 : (rr >> 6) * 64 + at8 + (ni >> 1) * 32;
    voff[i] = (WIDE ? (g == 0 ? n : rr) * 128 : (g == 0 ? n * p.K : rr * (int)p.ldx) * ES) + c * 16;
  }
  const int hA = g == 0 ? 0 : 1, hB = g == 0 ? 1 : 0;
  auto rA = gt_half<EPI, ES, WIDE>(p, cur.tm, cur.tn, g, wc, hA), rB = gt_half<EPI, ES, WIDE>(p, cur.tm, cur.tn, g, wc, hB);
  // LDS image of a K tile: x rows 0..255 (two halves), then W rows 0..255 (two halves)
  constexpr int LX0 = 0, LX1 = GT_HALF, LW0 = 2 * GT_HALF, LW1 = 3 * GT_HALF;
  char* const lds_w = sm + wc * 4096;   // this wave's four 1-KiB pieces inside a half-tile
  const int ldA_l = g == 0 ? LW0 : LX1, ldB_l = g == 0 ? LW1 : LX0;
  const int ldB_d = g == 0 ? 1 : 2;     // tile distance of the second request (the first is always t + 1)
// four 1-KiB pieces of one half-tile: bytes `koff` .. of the rows of buffer r, to stage `stage` (a running number's parity)
#define GT_REQUEST(r, koff, stage, ldso)                                                     \
  _Pragma("unroll") for (int i = 0; i < 4; ++i)                                              \
      gt_load(r, lds_w + (((stage) & 1) ? GT_STAGE : 0) + (ldso) + i * 1024, voff[i], koff)

  // ---- prologue: all of tile 0 and x rows 0..127 of tile 1 ------------------------------------
  int koff = cur.t0 * 128;    // of K tile t
  GT_REQUEST(rA, koff, 0, ldA_l);            // W0(0) | x1(0)
  GT_REQUEST(rB, koff, 0, ldB_l);            // W1(0) | x0(0)
  if (g == 1) GT_REQUEST(rB, koff + 128, 1, ldB_l);   // x0(1)

  // ---- fragment read addresses ----------------------------------------------------------------
  // 16-bit: fragment of k-step kk = chunk 4 kk + q4 (k-step 1 is rd0 ^ 64); fp8: the fragment of the
  // whole 128-deep tile = chunks 2 q4 and 2 q4 + 1 (rd0 and rd0 ^ 16)
  const int r16 = lane & 15, q4 = lane >> 4;
  const int rd0 = r16 * 128 + (((FP8 ? 2 * q4 : q4) ^ gt_swz<FP8>(r16)) << 4);
  const int a_off = g * GT_HALF, b_off = 2 * GT_HALF + wc * 8192;

  // EPI 2 waits for loads: both groups at once
  constexpr bool TOGETHER = EPI == 2;
  f32x4 acc[8][4];
  // two 16-byte registers per fragment slot: k-steps 0 / 1 (16-bit) or the two halves of the 32-byte
  // fp8 fragment
  i32x4 af[2][8], bf[2][4];
  int s = 0;                  // running number of the K tile: which stage it lies in
#define GT_TILE(FIRST, REQUESTS)                                                             \
  do {                                                                                       \
    const int cur_ = (s & 1) ? GT_STAGE : 0;                                                 \
    /* READ slot: request the group's two half-tiles, read the fragments of the whole K tile */ \
    REQUESTS                                                                                 \
    _Pragma("unroll") for (int kk = 0; kk < 2; ++kk) {                                       \
      const int ro_ = rd0 ^ (FP8 ? (kk << 4) : (kk << 6));                                   \
      const char* ab_ = sm + cur_ + a_off + ro_;                                             \
      const char* bb_ = sm + cur_ + b_off + ro_;                                             \
      _Pragma("unroll") for (int ni = 0; ni < 4; ++ni)                                       \
          bf[kk][ni] = *reinterpret_cast<const i32x4*>(bb_ + ni * 2048);                     \
      _Pragma("unroll") for (int mi = 0; mi < 8; ++mi)                                       \
          af[kk][mi] = *reinterpret_cast<const i32x4*>(ab_ + mi * 2048);                     \
    }                                                                                        \
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                                       \
    GT_SLOT_END();                                                                           \
    /* MATRIX slot: nothing but MFMAs, then the wave's requests of its READ slot must have landed */ \
    __builtin_amdgcn_s_setprio(1);                                                           \
    if constexpr (FP8) {                                                                     \
      _Pragma("unroll") for (int mi = 0; mi < 8; ++mi)                                       \
        _Pragma("unroll") for (int nj = 0; nj < 4; ++nj) {                                   \
          const int ni = (mi & 1) ? 3 - nj : nj;                                             \
          const i32x8 a8_ = __builtin_shufflevector(bf[0][ni], bf[1][ni], 0, 1, 2, 3, 4, 5, 6, 7);\
          const i32x8 b8_ = __builtin_shufflevector(af[0][mi], af[1][mi], 0, 1, 2, 3, 4, 5, 6, 7);\
          acc[mi][ni] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(                    \
              a8_, b8_, (FIRST) ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[mi][ni], 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f); \
        }                                                                                    \
    } else {                                                                                 \
      _Pragma("unroll") for (int kk = 0; kk < 2; ++kk)                                       \
        _Pragma("unroll") for (int mi = 0; mi < 8; ++mi)                                     \
          _Pragma("unroll") for (int nj = 0; nj < 4; ++nj) {                                 \
              const int ni = (mi & 1) ? 3 - nj : nj;                                         \
              acc[mi][ni] = Mfma<T>::run(__builtin_bit_cast(frag, bf[kk][ni]), __builtin_bit_cast(frag, af[kk][mi]), \
                                         (FIRST) && kk == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[mi][ni]); \
          }                                                                                  \
    }                                                                                        \
    __builtin_amdgcn_s_setprio(0);                                                           \
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                                         \
    GT_SLOT_END();                                                                           \
    ++s; koff += 128;                                                                        \
  } while (0)
#define GT_REQUESTS_INSIDE { GT_REQUEST(rA, koff + 128, s + 1, ldA_l); GT_REQUEST(rB, koff + 128 * ldB_d, s + ldB_d, ldB_l); }

  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // tile 0 (and x rows 0..127 of tile 1) have landed
  GT_SLOT_END();
  if (g == 1) GT_SLOT_END();   // the second group runs one slot behind the first
  for (int item = 1;; ++item) {
    const GtItem nxt = gt_item(p, item, kt);
    const auto nA = gt_half<EPI, ES, WIDE>(p, nxt.tm, nxt.tn, g, wc, hA), nB = gt_half<EPI, ES, WIDE>(p, nxt.tm, nxt.tn, g, wc, hB);
    const int nk = nxt.t0 * 128;
    int t = 0;
    if (!FP8 && cur.T > 2) {   // (sums that start in the MFMAs)
      GT_TILE(true, GT_REQUESTS_INSIDE);
      t = 1;
    } else {
#pragma unroll
      for (int mi = 0; mi < 8; ++mi)
#pragma unroll
        for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    for (; t + 2 < cur.T; ++t) GT_TILE(false, GT_REQUESTS_INSIDE);
    // The last two K tiles: x rows 0..127 and then everything is the next item's.  fp8 in a loop: as straight code the compiler moves
    // those MFMAs behind the barriers, into the epilogue, with 480 bytes of spilled registers.
    if constexpr (FP8) {
#pragma unroll 1
      for (; t < cur.T; ++t) {
        const bool last = t + 1 == cur.T;
        GT_TILE(false, {
          if (!last) { GT_REQUEST(rA, koff + 128, s + 1, ldA_l); }
          else if (nxt.valid) { GT_REQUEST(nA, nk, s + 1, ldA_l); }
          if (!last && g == 0) { GT_REQUEST(rB, koff + 128, s + 1, ldB_l); }
          else if (nxt.valid) { GT_REQUEST(nB, last && g == 1 ? nk + 128 : nk, last ? s + ldB_d : s, ldB_l); }
        });
      }
    } else {
      GT_TILE(false, {
        GT_REQUEST(rA, koff + 128, s + 1, ldA_l);
        if (g == 0) { GT_REQUEST(rB, koff + 128, s + 1, ldB_l); }
        else if (nxt.valid) { GT_REQUEST(nB, nk, s, ldB_l); }
      });
      GT_TILE(false, {
        if (nxt.valid) {
          GT_REQUEST(nA, nk, s + 1, ldA_l);
          GT_REQUEST(nB, nk + 128 * (ldB_d - 1), s + ldB_d, ldB_l);
        }
      });
    }
    if ((TOGETHER || !nxt.valid) && g == 0) __builtin_amdgcn_s_barrier();   // (the other group is one slot behind)
    // The lane's number and the arguments (the kernel's only one, so that they lie first) again: otherwise the compiler works out the epilogue's addresses in front of all tiles and keeps
    // them, with every argument, in scratch memory and in lanes of a register.  2 x 14336 columns with SiLU-and-mul, 65536 rows: 10.70 ms so,
    // 10.22 this way (a workgroup per tile 10.45).
    int zero = 0;
    asm volatile("" : "+v"(zero));
    const int el = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, zero));
    auto args = (const __attribute__((address_space(4))) GemmTiledParams*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    const GemmTiledParams& pe = *(const GemmTiledParams*)args;
    if (cur.part != nullptr) {   // a split of a tail tile: its sums as they lie in the registers
#pragma unroll
      for (int mi = 0; mi < 8; ++mi)
        if (cur.tm * 256 + g * 128 + mi * 16 < pe.M)
#pragma unroll
          for (int ni = 0; ni < 4; ++ni) *reinterpret_cast<f32x4*>(cur.part + ((wave * 8 + mi) * 4 + ni) * 256 + el * 4) = acc[mi][ni];
    } else if (EPI == 0 && pe.bias != nullptr) {
      tile_epilogue<T, EPI, FP8, 8, true>(pe, acc, cur.tm * 256 + g * 128, cur.tm, cur.tn, wc, el >> 4, el & 15, 256);
    } else {
      tile_epilogue<T, EPI, FP8, 8, false>(pe, acc, cur.tm * 256 + g * 128, cur.tm, cur.tn, wc, el >> 4, el & 15, 256);
    }
    if (!nxt.valid) break;
    if (TOGETHER && g == 1) GT_SLOT_END();   // and is again
    cur = nxt;
    rA = nA;
    rB = nB;
    koff = nk;
  }
#undef GT_REQUEST
#undef GT_REQUESTS_INSIDE
#undef GT_TILE
}

// The grouped products: a workgroup per tile, in blocks of 8 x 4 tiles (only the device knows how many tiles there are).
// MIXED: tiles without padding are as likely as tiles with; a wave whose rows are all there then takes a loop without the
// conditions that leave padding out.  Those cost a full tile 5 %, the second loop a mostly empty one 3 to 6 (32 experts of 2048 x
// 2048, 4 per token, both products: 8192 tokens 663 -> 624 us with it, 3000 297 -> 288, 1024 193 -> 197; 256 of 2048 x 512, 8 per
// token, 64 tokens 304 -> 322).
template <typename T, bool MIXED>
__global__ __launch_bounds__(512) void gemm_grouped_kernel(GemmTiledParams p) {
  extern __shared__ __attribute__((aligned(16))) char sm[];
  using frag = typename Mfma<T>::frag;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = wave >> 2, wc = wave & 3;

  // ---- workgroup -> output tile ------------------------------------------------------------
  // Consecutive workgroups go to the eight XCDs in turn: blocks of 8 x 4 tiles in turn.
  const int b = blockIdx.x, li = b >> 3;
  int tm, tn;
  const int T_ = p.K >> 6;     // K tiles of 128 bytes per row
  {
    const int st = (li >> 5) * 8 + (b & 7), within = li & 31;
    if (st >= p.nsuper) return;
    const int sup_m = st / p.snt, sup_n = st - sup_m * p.snt;
    // An expert's last tile is the one with padding.  The block's others go first, so that the short ones fill up where long ones end: 32
    // experts of 2048 x 2048, 4 per token, 1000 tokens 279 -> 263 us the layer (3000 313 either way), of 4096 x 4096, 1871 tokens 695 -> 667.
    const int used = min(*p.tiles_used, p.mt), rank = within >> 2;
    unsigned last = 0;     // of the block's eight tiles
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int t = sup_m * 8 + i;
      last |= (t + 1 >= used || p.tile_expert[max(min(t, used - 1), 0)] != p.tile_expert[max(min(t + 1, used - 1), 0)]) ? 1u << i : 0u;
    }
    const int whole = 8 - __popc(last);
    unsigned of = rank < whole ? ~last & 255u : last;
    for (int i = rank < whole ? rank : rank - whole; i > 0; --i) of &= of - 1;
    tm = sup_m * 8 + __builtin_ctz(of);
    tn = sup_n * 4 + (within & 3);
    if (tm >= used || tn >= p.nt) return;
  }
  // Rows of the tile up to the last one that is no padding (a plan's padding lies behind them; between them it reads row 0).
  // Padding rows are neither loaded, multiplied nor stored, 8, 16 and 1 at a time: an expert's last tile is as long as its rows.  64 tokens x 4 of 32 experts (2048 x 2048):
  // 88 us with padding worked on, 55 without (268 MB of weights); 1024 tokens: 85 and 72; 3000 tokens: 148 and 145.
  int live = 256;
  if (p.row_map != nullptr) {
    live = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned long long there = __ballot(p.row_map[tm * 256 + i * 64 + lane] >= 0);
      live = there != 0 ? 64 * i + 64 - __clzll(there) : live;
    }
    live = __builtin_amdgcn_readfirstlane(live);
  }
  const int live_mi = min(max((live - g * 128 + 15) >> 4, 0), 8);

  const char* xg = (const char*)p.x;
  const char* wg = (const char*)p.w + (int64_t)p.tile_expert[tm] * p.w_expert_stride * 2;

  // ---- per-lane source pointers of the eight load instructions a wave issues per K tile -----
  // A wave requests data only in its READ slot (a load-to-LDS holds the issuing wave ~40 cycles: in
  // front of or between the MFMAs of a matrix slot that time is lost to the matrix pipe, next to the
  // LDS reads of a READ slot it is covered by the other group's MFMAs).  Group 0 (READ slot 2t) requests
  // W of tile t + 1, both halves; group 1 (READ slot 2t + 1) requests x rows 128..255 of tile t + 1 and
  // x rows 0..127 of tile t + 2: each is free when requested (its last reader finished a slot earlier)
  // and is waited for -- by the waves that requested it, at the end of their MATRIX slot -- before
  // the barrier in front of the first slot that reads it.  A half-tile is 16 pieces of 8 rows x 128
  // bytes; wave wc of the group requests pieces 4 wc .. 4 wc + 3 of its group's two half-tiles:
  //   ldA: group 0 W rows 0..127 (tile t + 1), group 1 x rows 128..255 (tile t + 1)
  //   ldB: group 0 W rows 128..255 (tile t + 1), group 1 x rows 0..127 (tile t + 2)
  const char* ldA[4];
  const char* ldB[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int rr = (wc * 4 + i) * 8 + (lane >> 3);             // row inside the half-tile
    const int c = (lane & 7) ^ gt_swz<false>(rr);                // logical 16-byte chunk this lane fetches
    const char* xs[2];
    const char* ws[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      int m = tm * 256 + h * 128 + rr;
      m = m < p.M ? m : p.M - 1;
      // gathered rows; a padding row reads row 0 (its products are not stored)
      if (p.gather) m = max(p.row_map[m], 0);
      xs[h] = xg + ((int64_t)m * p.ldx) * 2 + c * 16;
      const int rb = h * 128 + rr, wcb = rb >> 6, sl = rb & 63, ni = sl >> 4, ii = sl & 15;
      int n = tn * 256 + wcb * 64 + (ni >> 1) * 32 + (ii >> 2) * 8 + (ni & 1) * 4 + (ii & 3);
      n = n < p.N ? n : p.N - 1;
      ws[h] = wg + ((int64_t)n * p.K) * 2 + c * 16;
    }
    ldA[i] = g == 0 ? ws[0] : xs[1];
    ldB[i] = g == 0 ? ws[1] : xs[0];
  }
  // LDS image of a K tile: x rows 0..255 (two halves), then W rows 0..255 (two halves)
  constexpr int LX0 = 0, LX1 = GT_HALF, LW0 = 2 * GT_HALF, LW1 = 3 * GT_HALF;
  char* const lds_w = sm + wc * 4096;   // this wave's four 1-KiB pieces inside a half-tile
  const int ldA_l = g == 0 ? LW0 : LX1, ldB_l = g == 0 ? LW1 : LX0;
  const int ldB_d = g == 0 ? 1 : 2;     // tile distance of the second request (the first is always t + 1)

  // Every expert's K is walked from another tile on and round the end.  Rows of operands lie 4 KB or more apart, so workgroups in
  // step ask for the same 128-byte column of all the weights and with it for few memory channels.  A layer of 32 experts of 2048 x 2048, 4
  // per token, us with K from its start -> staggered: 16 tokens 154 -> 131, 131 tokens 187 -> 144 (one product 75 -> 53: 268 MB at 5.1 TB/s),
  // 1000 309 -> 279, 3000 325 -> 310; by column of tiles as well 147 at 131, by that alone 167.  A dense product's rows and columns have one order
  // of K each, whichever tile they are in and whatever is fused behind it.
  const int rot = p.tile_expert[tm] % T_;
#define GT_AT(tl) ((int64_t)((tl) + rot >= T_ ? (tl) + rot - T_ : (tl) + rot) * 128)

  // ---- prologue: all of tile 0 and x rows 0..127 of tile 1 ------------------------------------
#pragma unroll
  for (int i = 0; i < 4; ++i) glds16(ldA[i] + GT_AT(0), lds_w + ldA_l + i * 1024);            // W0(0) | x1(0)
#pragma unroll
  for (int i = 0; i < 4; ++i) glds16(ldB[i] + GT_AT(0), lds_w + ldB_l + i * 1024);            // W1(0) | x0(0)
  if (g == 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) glds16(ldB[i] + GT_AT(1), lds_w + GT_STAGE + ldB_l + i * 1024);   // x0(1)
  }

  // ---- fragment read addresses ----------------------------------------------------------------
  // fragment of k-step kk = chunk 4 kk + q4 (k-step 1 is rd0 ^ 64)
  const int r16 = lane & 15, q4 = lane >> 4;
  const int rd0 = r16 * 128 + ((q4 ^ gt_swz<false>(r16)) << 4);
  const int a_off = g * GT_HALF, b_off = 2 * GT_HALF + wc * 8192;

  f32x4 acc[8][4];
#pragma unroll
  for (int mi = 0; mi < 8; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = f32x4{0.f, 0.f, 0.f, 0.f};
  i32x4 af[2][8], bf[2][4];

  // how many of the wave's four pieces of x rows 128..255 (ldA of group 1) and 0..127 (ldB) hold rows that are no padding
  const int nA = g == 1 ? min(max((live - 128 - wc * 32 + 7) >> 3, 0), 4) : 4;
  const int nB = g == 1 ? min(max((live - wc * 32 + 7) >> 3, 0), 4) : 4;
// four 1-KiB pieces of one half-tile of tile `tl`; TAIL: nothing past the last tile
#define GT_LOAD4(ptr, ldso, tl, TAIL, PART, COUNT)                                           \
  do {                                                                                       \
    if (!(TAIL) || (tl) < T_) {                                                              \
      char* d_ = lds_w + (((tl) & 1) ? GT_STAGE : 0) + (ldso);                               \
      _Pragma("unroll") for (int i = 0; i < 4; ++i)                                          \
          if (!(PART) || i < (COUNT)) glds16(ptr[i] + GT_AT(tl), d_ + i * 1024);   \
    }                                                                                        \
  } while (0)
#define GT_TILE(t, TAIL, PART)                                                               \
  do {                                                                                       \
    const int cur_ = ((t) & 1) ? GT_STAGE : 0;                                               \
    /* READ slot: request the group's two half-tiles, read the fragments of the whole K tile t */ \
    GT_LOAD4(ldA, ldA_l, (t) + 1, TAIL, PART, nA);                                           \
    GT_LOAD4(ldB, ldB_l, (t) + ldB_d, TAIL, PART, nB);                                       \
    _Pragma("unroll") for (int kk = 0; kk < 2; ++kk) {                                       \
      const int ro_ = rd0 ^ (kk << 6);                                                        \
      const char* ab_ = sm + cur_ + a_off + ro_;                                             \
      const char* bb_ = sm + cur_ + b_off + ro_;                                             \
      _Pragma("unroll") for (int ni = 0; ni < 4; ++ni)                                       \
          bf[kk][ni] = *reinterpret_cast<const i32x4*>(bb_ + ni * 2048);                     \
      _Pragma("unroll") for (int mi = 0; mi < 8; ++mi)                                       \
          if (!(PART) || mi < live_mi) af[kk][mi] = *reinterpret_cast<const i32x4*>(ab_ + mi * 2048); \
    }                                                                                        \
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                                       \
    GT_SLOT_END();                                                                           \
    /* MATRIX slot: nothing but MFMAs, then the wave's requests of its READ slot must have landed */ \
    __builtin_amdgcn_s_setprio(1);                                                           \
    _Pragma("unroll") for (int kk = 0; kk < 2; ++kk)                                         \
      _Pragma("unroll") for (int mi = 0; mi < 8; ++mi)                                       \
        if (!(PART) || mi < live_mi)                                                         \
        _Pragma("unroll") for (int nj = 0; nj < 4; ++nj) {                                   \
            const int ni = (mi & 1) ? 3 - nj : nj;                                           \
            acc[mi][ni] = Mfma<T>::run(__builtin_bit_cast(frag, bf[kk][ni]),                 \
                                       __builtin_bit_cast(frag, af[kk][mi]), acc[mi][ni]);   \
        }                                                                                    \
    __builtin_amdgcn_s_setprio(0);                                                           \
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                                         \
    GT_SLOT_END();                                                                           \
  } while (0)

  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // tile 0 (and x rows 0..127 of tile 1) have landed
  GT_SLOT_END();
  if (g == 1) GT_SLOT_END();   // the second group runs one slot behind the first
  int t = 0;
  if (!MIXED || live_mi < 8 || nA < 4 || nB < 4) {   // (per wave; the barriers are as many either way)
    for (; t + 2 < T_; ++t) GT_TILE(t, false, true);
    for (; t < T_; ++t) GT_TILE(t, true, true);
  } else {
    for (; t + 2 < T_; ++t) GT_TILE(t, false, false);   // every request exists: no conditions in the loop
    for (; t < T_; ++t) GT_TILE(t, true, false);
  }
  if (g == 0) __builtin_amdgcn_s_barrier();
#undef GT_LOAD4
#undef GT_TILE
#undef GT_AT

  tile_epilogue<T, 3, false, 8, false>(p, acc, tm * 256 + g * 128, tm, tn, wc, q4, r16, live);
}
#undef GT_SLOT_END

// Sums the splits of the tail tiles in their order and finishes the tiles: a wave takes one 16-row group of one of the tile's waves,
// its lanes' values in the order in which they were left (whole 1-KiB lines).
template <typename T, int EPI, bool FP8>
__global__ __launch_bounds__(256) void gemm_tiled_tail_kernel(GemmTiledParams p) {
  const int lane = threadIdx.x & 63, r16 = lane & 15, q4 = lane >> 4;
  const int task = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int t = task >> 6, wave = (task >> 3) & 7, mi = task & 7, g = wave >> 2, wc = wave & 3;
  int tm, tn;
  tile_of(p, p.full + t, tm, tn);
  const int m0 = tm * 256 + g * 128 + mi * 16;
  if (m0 >= p.M) return;
  f32x4 acc[1][4];
#pragma unroll
  for (int ni = 0; ni < 4; ++ni) acc[0][ni] = f32x4{0.f, 0.f, 0.f, 0.f};
  const float* src = p.part + (int64_t)t * 65536 + ((wave * 8 + mi) * 4) * 256 + lane * 4;
#pragma unroll 4
  for (int k = 0; k < p.splits; ++k) {
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) acc[0][ni] += *reinterpret_cast<const f32x4*>(src + (int64_t)k * p.tail * 65536 + ni * 256);
  }
  tile_epilogue<T, EPI, FP8, 1, EPI == 0>(p, acc, m0, tm, tn, wc, q4, r16, 256);
}

template <typename T, int EPI, bool FP8>
int launch_gemm_tiled(const GemmTiledParams& p, hipStream_t st) {
  auto kern = std::max<int64_t>(p.ldx, p.K) > GT_MAX_STRIDE ? gemm_tiled_kernel<T, EPI, FP8, true> : gemm_tiled_kernel<T, EPI, FP8, false>;
  (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, GT_LDS);
  // workgroups that stay: as many as there are CUs, in equal numbers for every XCD (with whole tiles in front of a tail: all of them)
  const int per = p.splits == 0 ? (int)cdiv((int64_t)p.mt * p.nt, 8) : std::max(p.full / 8, (int)cdiv((int64_t)p.tail * p.splits, 8));
  hipLaunchKernelGGL(kern, dim3((unsigned)(std::min(per, 32) * 8)), dim3(512), GT_LDS, st, p);
  if (p.splits != 0) hipLaunchKernelGGL((gemm_tiled_tail_kernel<T, EPI, FP8>), dim3((unsigned)p.tail * 16), dim3(256), 0, st, p);
  MI355_CHECK_LAUNCH(EPI == 2 ? "mi355_qkv_proj_rope_tiled" : FP8 ? "mi355_fp8_scaled_mm_tiled" : "mi355_linear_tiled");
  return MI355_OK;
}

template <typename T, bool MIXED>
int launch_gemm_grouped(const GemmTiledParams& p, hipStream_t st) {
  auto kern = gemm_grouped_kernel<T, MIXED>;
  (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, GT_LDS);
  hipLaunchKernelGGL(kern, dim3((unsigned)((p.nsuper + 7) / 8 * 32 * 8)), dim3(512), GT_LDS, st, p);   // 8 x 4 blocks in equal numbers for every XCD
  MI355_CHECK_LAUNCH("mi355_moe_grouped_linear_tiled");
  return MI355_OK;
}

bool pairs(int epilogue) { return epilogue == 1 || epilogue == 3; }   // of an entry point: W = [gate; up]

void fill_tiles(GemmTiledParams& p, int64_t m, int64_t n, int epilogue) {
  p.positions = nullptr; p.cos_sin = nullptr; p.cs_f32 = 0; p.hq = p.hkv = 0;
  p.k_buffer = p.v_buffer = nullptr; p.loc = nullptr; p.loc_i32 = 0; p.kv_slot = p.kv_head = 0;
  p.row_map = p.tile_expert = p.tiles_used = nullptr; p.gather = 0; p.w_expert_stride = 0; p.act = 0;
  p.full = p.tail = p.splits = 0; p.part = nullptr;
  const int ncols = pairs(epilogue) ? (int)(n / 2) : (int)n;
  p.ldy = ncols;
  p.mt = cdiv(m, 256);
  p.nt = pairs(epilogue) ? cdiv(ncols, 128) : cdiv(ncols, 256);
  p.snt = cdiv(p.nt, 4);
  p.nsuper = cdiv(p.mt, 8) * p.snt;
}

// One workgroup is one CU, so tiles beyond whole rounds of 256 keep few CUs busy for as long as a round takes: those are split over K
// where that pays.  Measured costs, in us: a K tile 1.2 (1.14 since workgroups stay), a split of a tile (256 KiB of sums, written and read again)
// 0.075, the launch that sums them 3.  bf16, us, whole tiles -> split: 4605 x 4096 x K 4096 (32 tail tiles, 5 splits) 157 -> 123, K 14336 (8) 523 -> 372;
// 2 x 14336 columns, K 4096, 520 rows (80, 3) 158 -> 128, 1134 (48, 5) 255 -> 219, 1962 (128, 2) 360 -> 351.  Past half a round
// (1353 rows of the last: 160 tiles) there is nobody to share with; 128 tiles of K 2048 (42 us whole) gain less than the sums cost.
int plan_tail(int64_t m, int64_t n, int64_t kbytes, int epilogue) {
  const int64_t tiles = cdiv(m, 256) * (pairs(epilogue) ? cdiv(n / 2, 128) : cdiv(n, 256));
  const int64_t kt = kbytes >> 7, tail = tiles % 256;
  if (tail == 0) return 0;
  int best = 0;
  float cost = 1.2f * kt;
  for (int64_t s = 2; s <= 256 / tail && s <= kt / 4; ++s) {
    const float c = 1.2f * cdiv(kt, s) + 0.075f * (tail * s) + 3.f;
    if (c < cost) { cost = c; best = (int)s; }
  }
  return best;
}

// workspace null: no tile is split
int set_tail(GemmTiledParams& p, int splits, void* workspace, int64_t workspace_bytes, const char* what) {
  if (workspace == nullptr || splits == 0) return MI355_OK;
  const int tail = p.mt * p.nt % 256;
  MI355_REQUIRE(aligned16(workspace) && workspace_bytes >= (int64_t)tail * splits * 65536 * 4, MI355_ERR_INVALID,
                "%s: workspace of %ld bytes for %d tiles x %d splits", what, (long)workspace_bytes, tail, splits);
  p.tail = tail; p.full = p.mt * p.nt - tail; p.splits = splits; p.part = (float*)workspace;
  return MI355_OK;
}

// ---- few rows -------------------------------------------------------------------------------------
// A prompt or chunk of a few hundred rows is bound by the weights' way to the LDS: the 256 x 256 tile leaves most CUs without work.  Here a
// workgroup has a ring of NS K tiles (128 bytes per row) in LDS, NS - 1 of them in flight, one barrier per tile, and (WM x WN waves)
// tiles of 16 NM x 64 outputs a wave.  KS groups of waves take K tiles in turn, each with a ring of its own, and add their sums
// through LDS: two groups are two times as many bytes in flight where there are fewer tiles than CUs.  Tiles may be split over K further,
// with sums in `part` as they lie in the registers (gemm_few_tail_kernel adds them).  K starts at another tile in every
// column of tiles and goes round the end (see gemm_grouped_kernel on why): a row's result depends on its own values alone.
template <typename T, int EPI, bool FP8, int NM, int WM, int WN, int KS, int NS>
__global__ __launch_bounds__(64 * WM * WN * KS) void gemm_few_kernel(GemmTiledParams p) {
  extern __shared__ __attribute__((aligned(16))) char sm[];
  using frag = typename Mfma<T>::frag;
  constexpr int ES = FP8 ? 1 : 2, BM = 16 * NM * WM, BN = 64 * WN, NW = WM * WN;
  constexpr int STAGE = (BM + BN) * 128, PP = (BM + BN) / 8 / NW;   // bytes of a K tile; 1-KiB pieces of it that a wave requests
  static_assert((BM + BN) / 8 % NW == 0 && NS >= 3 && (NS - 2) * PP < 64, "whole pieces a wave, counted waits");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kg = wave / NW, w = wave % NW, wm = w / WN, wn = w % WN;

  // every XCD takes a run of tiles, rows fastest: the weights of a column of tiles come into one L2
  const int splits = max(p.splits, 1), at = (blockIdx.x & 7) * (int)(gridDim.x >> 3) + (blockIdx.x >> 3);
  if (at >= p.mt * p.nt * splits) return;
  const int tm = at % p.mt, tn = at / p.mt / splits, split = at / p.mt % splits;
  const int all = (p.K * ES) >> 7, t0 = all * split / splits, T_ = all * (split + 1) / splits - t0;
  const int its = (T_ + KS - 1) / KS, rot = tn % T_;
  const int ncols = EPI == 1 ? (p.N >> 1) : p.N;

  const char* src[PP];
#pragma unroll
  for (int i = 0; i < PP; ++i) {
    const int row = (w * PP + i) * 8 + (lane >> 3), c = (lane & 7) ^ gt_swz<FP8>(row);
    if (row < BM) {
      const int m = min(tm * BM + row, p.M - 1);
      src[i] = (const char*)p.x + (int64_t)m * p.ldx * ES + c * 16;
    } else {
      const int r = row - BM, G = tn * WN + (r >> 6), ni = (r & 63) >> 4, ii = r & 15;   // the wave's 64 columns, as tile_epilogue has them
      int n;
      if (EPI == 1) n = min(G * 32 + (ii >> 2) * 8 + (ni & 1) * 4 + (ii & 3), ncols - 1) + (ni >> 1) * ncols;
      else n = min(G * 64 + (ni >> 1) * 32 + (ii >> 2) * 8 + (ni & 1) * 4 + (ii & 3), p.N - 1);
      src[i] = (const char*)p.w + (int64_t)n * p.K * ES + c * 16;
    }
    src[i] += (int64_t)t0 * 128;
  }
  char* const ring = sm + kg * NS * STAGE;
  char* const dst = ring + w * PP * 1024;
  auto request = [&](int it) {      // (a group without a tile in the last turn requests its last one again: the waits count requests)
    int tl = min(it * KS + kg, T_ - 1) + rot;
    tl = tl < T_ ? tl : tl - T_;
    char* d = dst + it % NS * STAGE;
#pragma unroll
    for (int i = 0; i < PP; ++i) glds16(src[i] + (int64_t)tl * 128, d + i * 1024);
  };
  const int r16 = lane & 15, q4 = lane >> 4;
  const int rd0 = r16 * 128 + (((FP8 ? 2 * q4 : q4) ^ gt_swz<FP8>(r16)) << 4);

  f32x4 acc[NM][4];
#pragma unroll
  for (int mi = 0; mi < NM; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int i = 0; i < NS - 1; ++i)
    if (i < its) request(i);
  for (int it = 0; it < its; ++it) {
    // this wave's part of tile `it` has landed; NS - 2 tiles behind it may be on their way
    if (it + NS - 2 < its) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * PP) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();      // every wave's part has, and every wave is done with tile it - 1
    __builtin_amdgcn_sched_barrier(0);
    if (it + NS - 1 < its) request(it + NS - 1);
    const char* stage = ring + it % NS * STAGE;
    i32x4 af[2][NM], bf[2][4];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int ro = rd0 ^ (FP8 ? (kk << 4) : (kk << 6));
      const char* ab = stage + wm * (NM * 2048) + ro;
      const char* bb = stage + BM * 128 + wn * 8192 + ro;
#pragma unroll
      for (int ni = 0; ni < 4; ++ni) bf[kk][ni] = *reinterpret_cast<const i32x4*>(bb + ni * 2048);
#pragma unroll
      for (int mi = 0; mi < NM; ++mi) af[kk][mi] = *reinterpret_cast<const i32x4*>(ab + mi * 2048);
    }
    if (KS == 1 || it * KS + kg < T_) {
      if constexpr (FP8) {
#pragma unroll
        for (int mi = 0; mi < NM; ++mi)
#pragma unroll
          for (int ni = 0; ni < 4; ++ni)
            acc[mi][ni] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                __builtin_shufflevector(bf[0][ni], bf[1][ni], 0, 1, 2, 3, 4, 5, 6, 7),
                __builtin_shufflevector(af[0][mi], af[1][mi], 0, 1, 2, 3, 4, 5, 6, 7), acc[mi][ni], 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
      } else {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int mi = 0; mi < NM; ++mi)
#pragma unroll
            for (int ni = 0; ni < 4; ++ni)
              acc[mi][ni] = Mfma<T>::run(__builtin_bit_cast(frag, bf[kk][ni]), __builtin_bit_cast(frag, af[kk][mi]), acc[mi][ni]);
      }
    }
  }
  if constexpr (KS > 1) {   // the groups' sums, in their order
    constexpr int PART = NM * 4 * 1024;
    static_assert((KS - 1) * NW * PART <= KS * NS * STAGE, "the sums lie where the rings were");
    __syncthreads();
    if (kg > 0) {
#pragma unroll
      for (int mi = 0; mi < NM; ++mi)
#pragma unroll
        for (int ni = 0; ni < 4; ++ni)
          *reinterpret_cast<f32x4*>(sm + ((kg - 1) * NW + w) * PART + (mi * 4 + ni) * 1024 + lane * 16) = acc[mi][ni];
    }
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int g = 1; g < KS; ++g)
#pragma unroll
      for (int mi = 0; mi < NM; ++mi)
#pragma unroll
        for (int ni = 0; ni < 4; ++ni)
          acc[mi][ni] += *reinterpret_cast<const f32x4*>(sm + ((g - 1) * NW + w) * PART + (mi * 4 + ni) * 1024 + lane * 16);
  }
  const int G = tn * WN + wn, m0 = tm * BM + wm * 16 * NM;
  if (p.splits > 1) {
    // [split][64 columns][16 rows][4][64 lanes][4], whole 1-KiB lines
    float* part = p.part + (((int64_t)split * p.nt * WN + G) * ((p.M + 15) >> 4) + (m0 >> 4)) * 1024 + lane * 4;
#pragma unroll
    for (int mi = 0; mi < NM; ++mi)
      if (m0 + mi * 16 < p.M)
#pragma unroll
        for (int ni = 0; ni < 4; ++ni) *reinterpret_cast<f32x4*>(part + mi * 1024 + ni * 256) = acc[mi][ni];
    return;
  }
  tile_epilogue<T, EPI, FP8, NM, EPI == 0>(p, acc, m0, 0, G >> 2, G & 3, q4, r16, 256);
}

// A wave adds the splits' sums of 16 rows x 64 columns (W rows) in their order and finishes them.
template <typename T, int EPI, bool FP8>
__global__ __launch_bounds__(256) void gemm_few_tail_kernel(GemmTiledParams p, int groups) {
  const int lane = threadIdx.x & 63, r16 = lane & 15, q4 = lane >> 4, rows16 = (p.M + 15) >> 4;
  const int task = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int G = task / rows16, m0 = (task - G * rows16) * 16;
  if (G >= groups) return;
  f32x4 acc[1][4];
#pragma unroll
  for (int ni = 0; ni < 4; ++ni) acc[0][ni] = f32x4{0.f, 0.f, 0.f, 0.f};
  const float* src = p.part + ((int64_t)G * rows16 + (m0 >> 4)) * 1024 + lane * 4;
#pragma unroll 4
  for (int k = 0; k < p.splits; ++k) {
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) acc[0][ni] += *reinterpret_cast<const f32x4*>(src + (int64_t)k * groups * rows16 * 1024 + ni * 256);
  }
  tile_epilogue<T, EPI, FP8, 1, EPI == 0>(p, acc, m0, 0, G >> 2, G & 3, q4, r16, 256);
}

template <typename T, int EPI, bool FP8, int NM, int WM, int WN, int KS, int NS>
int launch_few_config(GemmTiledParams p, int splits, hipStream_t st) {
  constexpr int BM = 16 * NM * WM, BN = 64 * WN, LDS = KS * NS * (BM + BN) * 128;
  p.mt = cdiv(p.M, BM);
  p.nt = cdiv(p.N, BN);      // (W rows: a group of 64 is 32 gate and 32 up columns with SiLU-and-mul)
  p.splits = splits;
  auto kern = gemm_few_kernel<T, EPI, FP8, NM, WM, WN, KS, NS>;
  (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  hipLaunchKernelGGL(kern, dim3((unsigned)(cdiv((int64_t)p.mt * p.nt * splits, 8) * 8)), dim3(64 * WM * WN * KS), LDS, st, p);
  if (splits > 1) {
    const int groups = p.nt * WN;
    hipLaunchKernelGGL((gemm_few_tail_kernel<T, EPI, FP8>), dim3((unsigned)cdiv((int64_t)groups * cdiv(p.M, 16), 4)), dim3(256), 0, st, p, groups);
  }
  MI355_CHECK_LAUNCH("mi355_linear_few");
  return MI355_OK;
}

// The workgroups that the kernel comes in: tile, K tiles a turn, and us: fixed and for a turn, alone on a CU (c0's 0.535: 32 KB at 60 GB/s, a
// load-to-LDS instruction of 1 KB every 35 cycles)
struct FewShape { int bm, bn, ks; float fixed, turn; };
constexpr FewShape FEW[] = {{128, 128, 1, 3.0f, 0.535f}, {64, 64, 2, 2.8f, 0.51f}, {128, 64, 2, 2.4f, 0.69f}};
struct FewPlan { int shape, splits; };

// The fastest of them in one round of workgroups (shape -1: none is), by what a launch was measured to take: the longer of its turns and
// of the weights at 4.6 TB/s; splits: a second launch and their sums written and read.  From a second round on the 256 x 256 tile or a
// library is ahead (2 x 14336 columns, K 4096, 207 rows: 448 tiles, 89 us, library 71), and from 256 rows in 16 bits, 512 in fp8.  us, library
// (with the activation behind it) | here: bf16 3072 x 2048 70 rows 11.9 | 11.5, 207 12.9 | 11.7; 2 x 8192 x 2048 207 31 | 25; 2048 x
// 8192 128 21 | 17, 207 28 | 21; 4096 x 4096 128 25 | 17, 207 22 | 20; 6144 x 4096 70 22 | 19, 207 26 | 27; 4096 x 14336 128 75 | 33 (256 x
// 256 tiles 43), 2 x 14336 x 4096 70 56 | 50; fp8 6144 x 4096 330 25 | 21, 2 x 14336 x 4096 70 37 | 29, 4096 x 14336 207 34 | 27.
FewPlan plan_few(int64_t m, int64_t n, int64_t k, bool fp8) {
  const int64_t kt = (fp8 ? k : k * 2) >> 7;
  FewPlan best = {-1, 1};
  float cost = 1e30f;
  if (m > (fp8 ? 512 : 256)) return best;
  for (int c = 0; c < 3; ++c) {
    const FewShape& f = FEW[c];
    const int64_t tiles = (int64_t)cdiv(m, f.bm) * cdiv(n, f.bn);
    for (int s = 1; s <= 8 && tiles * s <= 256; ++s) {
      if (s > 1 && kt / s < 4 * f.ks) break;
      const float turns = f.fixed + f.turn * cdiv(cdiv(kt, s), f.ks), stream = 2.f + 128e-6f / 4.6f * ((float)n * kt);
      const float c1 = std::max(turns, stream) + (s > 1 ? 2.6f + 1.7e-6f * ((float)s * m * n) : 0.f);
      if (c1 < cost) { cost = c1; best = {c, s}; }
    }
  }
  return best;
}

template <typename T, int EPI, bool FP8>
int launch_few(const GemmTiledParams& p, const FewPlan& plan, hipStream_t st) {
  switch (plan.shape) {
    case 0: return launch_few_config<T, EPI, FP8, 2, 4, 2, 1, 4>(p, plan.splits, st);
    case 1: return launch_few_config<T, EPI, FP8, 2, 2, 1, 2, 4>(p, plan.splits, st);
    default: return launch_few_config<T, EPI, FP8, 2, 4, 1, 2, 3>(p, plan.splits, st);
  }
}

}  // namespace
}  // namespace mi355

using namespace mi355;


extern "C" int mi355_tiled_tail_splits(int64_t m, int64_t n, int64_t k, int fp8, int epilogue) {
  if (m < 1 || n < 1 || k < 1 || m > (1 << 24) || n > (1 << 24)) return 0;
  return plan_tail(m, n, fp8 ? k : k * 2, epilogue);
}

extern "C" int64_t mi355_tiled_tail_workspace_bytes(int64_t m, int64_t n, int64_t k, int fp8, int epilogue) {
  const int64_t tail = (cdiv(m, 256) * (pairs(epilogue) ? cdiv(n / 2, 128) : cdiv(n, 256))) % 256;
  return mi355_tiled_tail_splits(m, n, k, fp8, epilogue) * tail * 65536 * 4;
}

extern "C" int mi355_linear_tiled_supported(int64_t m, int64_t n, int64_t k, int dtype, int epilogue) {
  if (dtype != MI355_BF16 && dtype != MI355_F16) return 0;
  if (m < 1 || n < 16 || k < 128 || (k & 63) != 0 || m > (1 << 24) || n > (1 << 24) || k * 2 > GT_MAX_ROW) return 0;
  return (epilogue >= 0 && epilogue <= 3 && n % 16 == 0) ? 1 : 0;   // silu-mul: 8 gate + 8 up columns per lane
}

extern "C" int mi355_linear_tiled(void* y, const void* x, const void* w, const void* bias, int64_t m,
                                  int64_t n, int64_t k, int64_t x_stride, int dtype, int epilogue,
                                  void* stream) {
  return mi355_linear_tiled_ws(y, x, w, bias, m, n, k, x_stride, dtype, epilogue, nullptr, 0, stream);
}

extern "C" int mi355_linear_tiled_ws(void* y, const void* x, const void* w, const void* bias, int64_t m,
                                     int64_t n, int64_t k, int64_t x_stride, int dtype, int epilogue,
                                     void* workspace, int64_t workspace_bytes, void* stream) {
  MI355_REQUIRE(y && x && w, MI355_ERR_INVALID, "mi355_linear_tiled: null pointer");
  MI355_REQUIRE(mi355_linear_tiled_supported(m, n, k, dtype, epilogue), MI355_ERR_UNSUPPORTED,
                "mi355_linear_tiled: needs a 16-bit dtype, K %% 64 == 0, K >= 128, N %% 16 == 0 (m=%ld n=%ld k=%ld "
                "dtype=%d epilogue=%d)", (long)m, (long)n, (long)k, dtype, epilogue);
  MI355_REQUIRE(x_stride >= k && x_stride % 8 == 0, MI355_ERR_INVALID,
                "mi355_linear_tiled: x_stride must be >= K and a multiple of 8 elements");
  MI355_REQUIRE(aligned16(x) && aligned16(w) && aligned16(y) && (bias == nullptr || aligned16(bias)),
                MI355_ERR_INVALID, "mi355_linear_tiled: pointers must be 16-byte aligned");
  MI355_REQUIRE(epilogue == 0 || bias == nullptr, MI355_ERR_UNSUPPORTED,
                "mi355_linear_tiled: no bias with an activation in the epilogue");
  GemmTiledParams p;
  p.x = x; p.w = w; p.bias = bias; p.y = y;
  p.x_scale = nullptr; p.w_scale = nullptr;
  p.M = (int)m; p.N = (int)n; p.K = (int)k;
  p.ldx = x_stride;
  fill_tiles(p, m, n, epilogue);
  if (const int rc = set_tail(p, plan_tail(m, n, k * 2, epilogue), workspace, workspace_bytes, "mi355_linear_tiled_ws")) return rc;
  hipStream_t st = (hipStream_t)stream;
  if (epilogue == 3) return dtype == MI355_BF16 ? launch_gemm_tiled<bf16_t, 5, false>(p, st) : launch_gemm_tiled<f16_t, 5, false>(p, st);
  if (epilogue == 2) return dtype == MI355_BF16 ? launch_gemm_tiled<bf16_t, 4, false>(p, st) : launch_gemm_tiled<f16_t, 4, false>(p, st);
  if (dtype == MI355_BF16)
    return epilogue == 1 ? launch_gemm_tiled<bf16_t, 1, false>(p, st) : launch_gemm_tiled<bf16_t, 0, false>(p, st);
  return epilogue == 1 ? launch_gemm_tiled<f16_t, 1, false>(p, st) : launch_gemm_tiled<f16_t, 0, false>(p, st);
}

extern "C" int mi355_fp8_scaled_mm_tiled_supported(int64_t m, int64_t n, int64_t k, int out_dtype, int epilogue);

extern "C" int mi355_linear_few_supported(int64_t m, int64_t n, int64_t k, int fp8, int out_dtype, int epilogue) {
  if (epilogue > 1 || !(fp8 ? mi355_fp8_scaled_mm_tiled_supported(m, n, k, out_dtype, epilogue) : mi355_linear_tiled_supported(m, n, k, out_dtype, epilogue))) return 0;
  return plan_few(m, n, k, fp8 != 0).shape >= 0 ? 1 : 0;
}

extern "C" int64_t mi355_linear_few_workspace_bytes(int64_t m, int64_t n, int64_t k, int fp8) {
  const FewPlan plan = plan_few(m, n, k, fp8 != 0);
  if (plan.shape < 0 || plan.splits == 1) return 0;
  return (int64_t)plan.splits * cdiv(n, FEW[plan.shape].bn) * (FEW[plan.shape].bn / 64) * cdiv(m, 16) * 4096;
}

extern "C" int mi355_linear_few(void* y, const void* x, const void* w, const float* x_scale, const float* w_scale, const void* bias, int64_t m,
                                int64_t n, int64_t k, int64_t x_stride, int out_dtype, int epilogue, void* workspace, int64_t workspace_bytes,
                                void* stream) {
  const bool fp8 = x_scale != nullptr;
  MI355_REQUIRE(y && x && w && (!fp8 || w_scale), MI355_ERR_INVALID, "mi355_linear_few: null pointer");
  MI355_REQUIRE(mi355_linear_few_supported(m, n, k, fp8, out_dtype, epilogue), MI355_ERR_UNSUPPORTED,
                "mi355_linear_few: needs a 16-bit result, K %% 64 == 0, K >= 128 (fp8: %% 128, 256), N %% 16 == 0 and one round of workgroups (m=%ld n=%ld "
                "k=%ld dtype=%d epilogue=%d)", (long)m, (long)n, (long)k, out_dtype, epilogue);
  MI355_REQUIRE(fp8 ? x_stride == k : (x_stride >= k && x_stride % 8 == 0), MI355_ERR_INVALID, "mi355_linear_few: bad x_stride");
  MI355_REQUIRE(aligned16(x) && aligned16(w) && aligned16(y) && (bias == nullptr || aligned16(bias)), MI355_ERR_INVALID,
                "mi355_linear_few: pointers must be 16-byte aligned");
  MI355_REQUIRE(epilogue == 0 || bias == nullptr, MI355_ERR_UNSUPPORTED, "mi355_linear_few: no bias with the SiLU-and-mul epilogue");
  const int64_t need = mi355_linear_few_workspace_bytes(m, n, k, fp8);
  MI355_REQUIRE(need == 0 || (workspace && aligned16(workspace) && workspace_bytes >= need), MI355_ERR_INVALID,
                "mi355_linear_few: workspace of %ld bytes, %ld needed", (long)workspace_bytes, (long)need);
  GemmTiledParams p;
  p.x = x; p.w = w; p.bias = bias; p.y = y;
  p.x_scale = x_scale; p.w_scale = w_scale;
  p.M = (int)m; p.N = (int)n; p.K = (int)k;
  p.ldx = x_stride;
  fill_tiles(p, m, n, epilogue);
  p.part = (float*)workspace;
  const FewPlan plan = plan_few(m, n, k, fp8);
  hipStream_t st = (hipStream_t)stream;
  if (fp8) {
    if (out_dtype == MI355_BF16) return epilogue == 1 ? launch_few<bf16_t, 1, true>(p, plan, st) : launch_few<bf16_t, 0, true>(p, plan, st);
    return epilogue == 1 ? launch_few<f16_t, 1, true>(p, plan, st) : launch_few<f16_t, 0, true>(p, plan, st);
  }
  if (out_dtype == MI355_BF16) return epilogue == 1 ? launch_few<bf16_t, 1, false>(p, plan, st) : launch_few<bf16_t, 0, false>(p, plan, st);
  return epilogue == 1 ? launch_few<f16_t, 1, false>(p, plan, st) : launch_few<f16_t, 0, false>(p, plan, st);
}

namespace mi355 {
// row_map says which rows are padding, and where the others come from if `gather` is set; `mixed`: see the kernel
int moe_grouped_linear_tiled(void* y, const void* x, int64_t x_stride, const void* w, const int32_t* row_map, int gather,
                             const int32_t* tile_expert, const int32_t* tiles_used, int act, int64_t rows, int64_t n, int64_t k,
                             int dtype, bool mixed, void* stream) {
  MI355_REQUIRE(y && x && w && tile_expert && tiles_used, MI355_ERR_INVALID, "mi355_moe_grouped_linear_tiled: null pointer");
  MI355_REQUIRE(rows > 0 && rows % 256 == 0 && mi355_linear_tiled_supported(rows, n, k, dtype, 0), MI355_ERR_UNSUPPORTED,
                "mi355_moe_grouped_linear_tiled: needs whole 256-row tiles, a 16-bit dtype, K %% 64 == 0, K >= 128, N %% 16 == 0 "
                "(rows=%ld n=%ld k=%ld dtype=%d)", (long)rows, (long)n, (long)k, dtype);
  MI355_REQUIRE(x_stride >= k && x_stride % 8 == 0 && aligned16(x) && aligned16(w) && aligned16(y), MI355_ERR_INVALID,
                "mi355_moe_grouped_linear_tiled: rows of x and the pointers must be 16-byte aligned");
  GemmTiledParams p;
  p.x = x; p.w = w; p.bias = nullptr; p.y = y;
  p.x_scale = nullptr; p.w_scale = nullptr;
  p.M = (int)rows; p.N = (int)n; p.K = (int)k;
  p.ldx = x_stride;
  fill_tiles(p, rows, n, 0);
  p.row_map = row_map; p.gather = gather; p.tile_expert = tile_expert; p.tiles_used = tiles_used; p.w_expert_stride = n * k; p.act = act;
  hipStream_t st = (hipStream_t)stream;
  if (mixed) return dtype == MI355_BF16 ? launch_gemm_grouped<bf16_t, true>(p, st) : launch_gemm_grouped<f16_t, true>(p, st);
  return dtype == MI355_BF16 ? launch_gemm_grouped<bf16_t, false>(p, st) : launch_gemm_grouped<f16_t, false>(p, st);
}
}  // namespace mi355

extern "C" int mi355_moe_grouped_linear_tiled(void* y, const void* x, int64_t x_stride, const void* w, const int32_t* row_map,
                                              const int32_t* tile_expert, const int32_t* tiles_used, int act, int64_t rows,
                                              int64_t n, int64_t k, int dtype, void* stream) {
  return moe_grouped_linear_tiled(y, x, x_stride, w, row_map, row_map != nullptr, tile_expert, tiles_used, act, rows, n, k, dtype, true,
                                  stream);
}

extern "C" int mi355_fp8_scaled_mm_tiled_supported(int64_t m, int64_t n, int64_t k, int out_dtype, int epilogue) {
  if (out_dtype != MI355_BF16 && out_dtype != MI355_F16) return 0;
  if (m < 1 || n < 16 || k < 256 || (k & 127) != 0 || m > (1 << 24) || n > (1 << 24) || k > GT_MAX_ROW) return 0;
  return ((epilogue == 0 || epilogue == 1) && n % 16 == 0) ? 1 : 0;
}

extern "C" int mi355_fp8_scaled_mm_tiled(void* y, const uint8_t* xq, const uint8_t* wq, const float* x_scale,
                                         const float* w_scale, const void* bias, int64_t m, int64_t n,
                                         int64_t k, int out_dtype, int epilogue, void* stream) {
  return mi355_fp8_scaled_mm_tiled_ws(y, xq, wq, x_scale, w_scale, bias, m, n, k, out_dtype, epilogue, nullptr, 0, stream);
}

extern "C" int mi355_fp8_scaled_mm_tiled_ws(void* y, const uint8_t* xq, const uint8_t* wq, const float* x_scale,
                                            const float* w_scale, const void* bias, int64_t m, int64_t n,
                                            int64_t k, int out_dtype, int epilogue, void* workspace,
                                            int64_t workspace_bytes, void* stream) {
  MI355_REQUIRE(y && xq && wq && x_scale && w_scale, MI355_ERR_INVALID, "mi355_fp8_scaled_mm_tiled: null pointer");
  MI355_REQUIRE(mi355_fp8_scaled_mm_tiled_supported(m, n, k, out_dtype, epilogue), MI355_ERR_UNSUPPORTED,
                "mi355_fp8_scaled_mm_tiled: needs a 16-bit output dtype, K %% 128 == 0, K >= 256, N %% 16 == 0 "
                "(m=%ld n=%ld k=%ld out_dtype=%d epilogue=%d)", (long)m, (long)n, (long)k, out_dtype, epilogue);
  MI355_REQUIRE(aligned16(xq) && aligned16(wq) && aligned16(y) && (bias == nullptr || aligned16(bias)),
                MI355_ERR_INVALID, "mi355_fp8_scaled_mm_tiled: pointers must be 16-byte aligned");
  MI355_REQUIRE(epilogue == 0 || bias == nullptr, MI355_ERR_UNSUPPORTED,
                "mi355_fp8_scaled_mm_tiled: no bias with the SiLU-and-mul epilogue");
  GemmTiledParams p;
  p.x = xq; p.w = wq; p.bias = bias; p.y = y;
  p.x_scale = x_scale; p.w_scale = w_scale;
  p.M = (int)m; p.N = (int)n; p.K = (int)k;
  p.ldx = k;
  fill_tiles(p, m, n, epilogue);
  if (const int rc = set_tail(p, plan_tail(m, n, k, epilogue), workspace, workspace_bytes, "mi355_fp8_scaled_mm_tiled_ws")) return rc;
  hipStream_t st = (hipStream_t)stream;
  if (out_dtype == MI355_BF16)
    return epilogue == 1 ? launch_gemm_tiled<bf16_t, 1, true>(p, st) : launch_gemm_tiled<bf16_t, 0, true>(p, st);
  return epilogue == 1 ? launch_gemm_tiled<f16_t, 1, true>(p, st) : launch_gemm_tiled<f16_t, 0, true>(p, st);
}

extern "C" int mi355_qkv_proj_rope_tiled_supported(int64_t m, int64_t k, int hq, int hkv, int head_dim,
                                                   int rotary_dim, int is_neox, int dtype, int fp8) {
  if (dtype != MI355_BF16 && dtype != MI355_F16) return 0;
  if (head_dim != 128 || rotary_dim != 128 || !is_neox || hq < 1 || hkv < 1 || ((hq + 2 * hkv) & 1)) return 0;
  if (m < 1 || m > (1 << 24) || (fp8 ? k : k * 2) > GT_MAX_ROW) return 0;
  return fp8 ? (k >= 256 && (k & 127) == 0) : (k >= 128 && (k & 63) == 0);
}

extern "C" int mi355_qkv_proj_rope_tiled(void* qkv, const void* x, const void* w, const float* x_scale,
                                         const float* w_scale, int64_t m, int64_t k, int64_t x_stride,
                                         int hq, int hkv, int head_dim, const int64_t* positions,
                                         const void* cos_sin_cache, int cache_dtype, int rotary_dim, int is_neox,
                                         void* k_buffer, void* v_buffer, const void* loc, int loc_itype,
                                         int64_t num_slots, int dtype, void* stream) {
  return mi355_qkv_proj_rope_tiled_ws(qkv, x, w, x_scale, w_scale, m, k, x_stride, hq, hkv, head_dim, positions, cos_sin_cache,
                                      cache_dtype, rotary_dim, is_neox, k_buffer, v_buffer, loc, loc_itype, num_slots, dtype, nullptr, 0,
                                      stream);
}

extern "C" int mi355_qkv_proj_rope_tiled_ws(void* qkv, const void* x, const void* w, const float* x_scale,
                                            const float* w_scale, int64_t m, int64_t k, int64_t x_stride,
                                            int hq, int hkv, int head_dim, const int64_t* positions,
                                            const void* cos_sin_cache, int cache_dtype, int rotary_dim, int is_neox,
                                            void* k_buffer, void* v_buffer, const void* loc, int loc_itype,
                                            int64_t num_slots, int dtype, void* workspace, int64_t workspace_bytes,
                                            void* stream) {
  const bool fp8 = x_scale != nullptr;
  const int kv_flags = dtype;
  dtype &= ~(MI355_KV_HEAD_MAJOR | MI355_KV_INTERLEAVED);
  MI355_REQUIRE(qkv && x && w && positions && cos_sin_cache && k_buffer && v_buffer && loc, MI355_ERR_INVALID,
                "mi355_qkv_proj_rope_tiled: null pointer");
  MI355_REQUIRE(!fp8 || w_scale, MI355_ERR_INVALID, "mi355_qkv_proj_rope_tiled: x_scale without w_scale");
  MI355_REQUIRE(mi355_qkv_proj_rope_tiled_supported(m, k, hq, hkv, head_dim, rotary_dim, is_neox, dtype, fp8),
                MI355_ERR_UNSUPPORTED,
                "mi355_qkv_proj_rope_tiled: needs a 16-bit dtype, head_dim = rotary_dim = 128, neox style, an even "
                "number of heads, K %% 64 == 0 (fp8: %% 128) (m=%ld k=%ld hq=%d hkv=%d head_dim=%d rotary_dim=%d)",
                (long)m, (long)k, hq, hkv, head_dim, rotary_dim);
  MI355_REQUIRE(cache_dtype == MI355_F32 || cache_dtype == dtype, MI355_ERR_UNSUPPORTED,
                "mi355_qkv_proj_rope_tiled: cos_sin_cache must be fp32 or the tensor dtype");
  MI355_REQUIRE(loc_itype == MI355_I32 || loc_itype == MI355_I64, MI355_ERR_INVALID,
                "mi355_qkv_proj_rope_tiled: loc must be int32 or int64");
  MI355_REQUIRE(fp8 ? x_stride == k : (x_stride >= k && x_stride % 8 == 0), MI355_ERR_INVALID,
                "mi355_qkv_proj_rope_tiled: bad x_stride");
  MI355_REQUIRE(aligned16(x) && aligned16(w) && aligned16(qkv) && aligned16(cos_sin_cache) && aligned16(k_buffer) &&
                    aligned16(v_buffer) && num_slots > 0 && num_slots < (1ll << 31),
                MI355_ERR_INVALID, "mi355_qkv_proj_rope_tiled: pointers must be 16-byte aligned");
  const int64_t n = (int64_t)(hq + 2 * hkv) * 128;
  GemmTiledParams p;
  p.x = x; p.w = w; p.bias = nullptr; p.y = qkv;
  p.x_scale = x_scale; p.w_scale = w_scale;
  p.M = (int)m; p.N = (int)n; p.K = (int)k;
  p.ldx = x_stride;
  fill_tiles(p, m, n, 0);
  p.positions = positions; p.cos_sin = cos_sin_cache; p.cs_f32 = cache_dtype == MI355_F32;
  p.hq = hq; p.hkv = hkv; p.k_buffer = k_buffer; p.v_buffer = v_buffer; p.loc = loc;
  kv_strides(kv_flags, num_slots, hkv, 128, p.kv_slot, p.kv_head);
  p.loc_i32 = loc_itype == MI355_I32;
  if (const int rc = set_tail(p, plan_tail(m, n, fp8 ? k : k * 2, 0), workspace, workspace_bytes, "mi355_qkv_proj_rope_tiled_ws")) return rc;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == MI355_BF16)
    return fp8 ? launch_gemm_tiled<bf16_t, 2, true>(p, st) : launch_gemm_tiled<bf16_t, 2, false>(p, st);
  return fp8 ? launch_gemm_tiled<f16_t, 2, true>(p, st) : launch_gemm_tiled<f16_t, 2, false>(p, st);
}
