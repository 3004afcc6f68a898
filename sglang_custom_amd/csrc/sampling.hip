// Sampling tail of the step: greedy arg-max, temperature softmax, and sort-free joint
// top-k / top-p / min-p sampling over fp32 [rows, vocab] logits.  Rows are 0.5 MB at vocab 128256, so
// every pass after the first is served from L2 / Infinity Cache.  What reads every entry is cut into
// chunks of a row, one workgroup each (row_chunks); without a workspace, and for short rows, one
// workgroup of 1024 threads does a whole row.
#include "common.cuh"
#include <math.h>
#include <algorithm>

namespace mi355 {

constexpr int SAMP_THREADS = 1024;

// ---- argmax: first index of the maximum (torch.argmax tie rule) --------------------------
// (maximum, first index) of elements [4 v0, 4 v1) of `row` -- plus the row's tail past the last whole
// float4 when `with_tail` -- reduced over the workgroup; valid in thread 0.  vec = the 16-byte path.
__device__ __forceinline__ void argmax_scan(const float* __restrict__ row, int64_t vocab, bool vec, int64_t v0, int64_t v1,
                                            bool with_tail, float& best_out, int& bidx_out) {
  __shared__ float sv[SAMP_THREADS / 64];
  __shared__ int si[SAMP_THREADS / 64];
  float best = -INFINITY;
  int bidx = 0x7fffffff;
  if (vec) {
    const int64_t nv = v1;
    auto take = [&](const float4& v, int64_t i) {
      const float a[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (a[j] > best || (a[j] == best && (int)(i * 4 + j) < bidx)) {
          best = a[j];
          bidx = (int)(i * 4 + j);
        }
    };
    // A lane meets its elements in rising index order, so "strictly greater" alone keeps the first
    // maximum: three branch-free instructions per element.  It cannot pick among elements equal to
    // the initial -inf; a lane that ends with nothing selected repeats the pass with the full rule.
    auto take_gt = [&](const float4& v, int64_t i) {
      const float a[4] = {v.x, v.y, v.z, v.w};
      const int base = (int)i * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool gt = a[j] > best;
        best = gt ? a[j] : best;
        bidx = gt ? base + j : bidx;
      }
    };
    // sixteen loads in flight per lane before the first comparison: 64 rows are 64 workgroups, so
    // a row is read at the latency of its load rounds (two for a 128k vocabulary), not at bandwidth
    constexpr int U = 16;
    auto scan = [&](auto&& pick) {
      for (int64_t i = v0 + threadIdx.x; i < nv; i += U * SAMP_THREADS) {
        float4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (i + u * SAMP_THREADS < nv) v[u] = *reinterpret_cast<const float4*>(row + (i + u * SAMP_THREADS) * 4);
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (i + u * SAMP_THREADS < nv) pick(v[u], i + u * SAMP_THREADS);
      }
    };
    scan(take_gt);
    if (bidx == 0x7fffffff) scan(take);
    if (with_tail)
      for (int64_t i = (vocab / 4) * 4 + threadIdx.x; i < vocab; i += SAMP_THREADS)
        if (row[i] > best || (row[i] == best && (int)i < bidx)) {
          best = row[i];
          bidx = (int)i;
        }
  } else {
    for (int64_t i = 4 * v0 + threadIdx.x; i < (with_tail ? vocab : 4 * v1); i += SAMP_THREADS)
      if (row[i] > best || (row[i] == best && (int)i < bidx)) {
        best = row[i];
        bidx = (int)i;
      }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(best, o, 64);
    const int oi = __shfl_xor(bidx, o, 64);
    if (ov > best || (ov == best && oi < bidx)) {
      best = ov;
      bidx = oi;
    }
  }
  if ((threadIdx.x & 63) == 0) {
    sv[threadIdx.x >> 6] = best;
    si[threadIdx.x >> 6] = bidx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < SAMP_THREADS / 64; ++w)
      if (sv[w] > best || (sv[w] == best && si[w] < bidx)) {
        best = sv[w];
        bidx = si[w];
      }
    best_out = best;
    bidx_out = bidx;
  }
}

__global__ __launch_bounds__(SAMP_THREADS) void argmax_kernel(int64_t* __restrict__ ids,
                                                             const float* __restrict__ logits,
                                                             int64_t vocab, int64_t row_stride) {
  const float* row = logits + (int64_t)blockIdx.x * row_stride;
  const bool vec = (row_stride % 4 == 0) && aligned16(logits);
  float best;
  int bidx;
  argmax_scan(row, vocab, vec, 0, vocab / 4, true, best, bidx);
  // a row without any finite-or-greater element (all NaN / -inf): index 0 like torch on -inf
  if (threadIdx.x == 0) ids[blockIdx.x] = bidx == 0x7fffffff ? 0 : bidx;
}

// A few rows (a decode batch) are a few workgroups: one workgroup reads its 0.5-MB row at what ONE CU can
// draw.  Here a row is cut into gridDim.y chunks; every chunk's (maximum, first index) is folded into the
// row's 64-bit cell with an atomic max -- key = (order-preserving image of the float) << 32 | ~index, so a
// larger key is a larger value or, among equal values, a smaller index: the same winner in any arrival
// order -- and the chunk that draws the row's last ticket decodes the cell into ids[row] and hands cell and
// ticket counter back zeroed.  All traffic on cells and counters is returning agent-scope atomics (each is
// complete before the next is issued), so nothing depends on cache write-back.
// grid (rows, chunks); cells: rows x uint64, tickets: rows x uint32, both zero between launches.
__global__ __launch_bounds__(SAMP_THREADS) void argmax_chunk_kernel(int64_t* __restrict__ ids,
                                                                   const float* __restrict__ logits, int64_t vocab,
                                                                   int64_t row_stride,
                                                                   unsigned long long* __restrict__ cells,
                                                                   unsigned* __restrict__ tickets) {
  const int r = blockIdx.x, c = blockIdx.y, chunks = gridDim.y;
  const float* row = logits + (int64_t)r * row_stride;
  const bool vec = (row_stride % 4 == 0) && aligned16(logits);
  const int64_t nv = vocab / 4, per = (nv + chunks - 1) / chunks;
  const int64_t v0 = c * per < nv ? c * per : nv, v1 = v0 + per < nv ? v0 + per : nv;
  float best;
  int bidx;
  argmax_scan(row, vocab, vec, v0, v1, c == chunks - 1, best, bidx);
  if (threadIdx.x != 0) return;
  unsigned u = __builtin_bit_cast(unsigned, best + 0.f);   // (-0 + 0 = +0: the two zeros are one value, as in a float compare)
  u = (u >> 31) ? ~u : (u | 0x80000000u);
  const unsigned long long key = ((unsigned long long)u << 32) | (unsigned long long)(0xffffffffu - (unsigned)bidx);
  (void)__hip_atomic_fetch_max(&cells[r], key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the maximum is in before the ticket is drawn
  const unsigned t = __hip_atomic_fetch_add(&tickets[r], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (t != (unsigned)(chunks - 1)) return;
  // every chunk's maximum is in (each was complete before its ticket was drawn): read the cell at the
  // point the atomics work at, then put cell and counter back to zero (nothing waits for those stores)
  const unsigned long long win = __hip_atomic_load(&cells[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&cells[r], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&tickets[r], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const unsigned idx = 0xffffffffu - (unsigned)(win & 0xffffffffu);
  ids[r] = idx == 0x7fffffffu ? 0 : (int64_t)idx;
}

// ---- softmax(logits / temperature), in place ----------------------------------------------
// Over the 16 waves of a workgroup: every lane takes one wave's value, four exchanges do the rest (sixteen LDS reads one behind
// the other are 0.4 us).
__device__ __forceinline__ float block_reduce_max(float x, float* red) {
  static_assert(SAMP_THREADS == 1024, "16 waves");
  x = wave_max(x);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  float t = red[threadIdx.x & 15];
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) t = fmaxf(t, __shfl_xor(t, o, 64));
  return t;
}
__device__ __forceinline__ float block_reduce_sum(float x, float* red) {
  x = wave_sum(x);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  float t = red[threadIdx.x & 15];
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
  return t;
}

__global__ __launch_bounds__(SAMP_THREADS) void softmax_temperature_kernel(
    float* __restrict__ logits, const float* __restrict__ temperatures, int64_t vocab,
    int64_t row_stride) {
  __shared__ float red[SAMP_THREADS / 64];
  float* row = logits + (int64_t)blockIdx.x * row_stride;
  const float t = temperatures[blockIdx.x];
  float mx = -INFINITY;
  for (int64_t i = threadIdx.x; i < vocab; i += SAMP_THREADS) mx = fmaxf(mx, row[i] / t);
  mx = block_reduce_max(mx, red);
  float sum = 0.f;
  for (int64_t i = threadIdx.x; i < vocab; i += SAMP_THREADS) sum += expf(row[i] / t - mx);
  sum = block_sum(sum, red);
  for (int64_t i = threadIdx.x; i < vocab; i += SAMP_THREADS) row[i] = expf(row[i] / t - mx) / sum;
}

// The same over chunks of a row, in two launches: every chunk leaves its maximum and its sum of exponentials, then
// every chunk normalises itself with what all of them left.  (A chunk without a number in it has no maximum to take off: its
// -inf entries count zero and a NaN makes its sum NaN, and with it the row, as one pass over the row has it.)  One workgroup per
// row reads its 0.5 MB three times with 4 bytes a lane in flight and has one CU's exponentials: 64 rows of 128256 took 146 us (64 CUs at work); this takes
// 11 + 10 us (33 MB read twice, the second time from L2, then read and written; 16 + 16 with a precise division per entry in
// both), bound by the exponentials and by the latency of a chunk's one round of loads.
constexpr int MAX_CHUNKS = 16;
struct ChunkSpan {
  int64_t v0, v1;   // first and one past the last of its groups of four elements
  bool tail;        // whether the row's last vocab % 4 elements belong to it
};
__device__ __forceinline__ ChunkSpan chunk_span(int64_t vocab, int c, int chunks) {
  const int64_t nv = vocab / 4, per = (nv + chunks - 1) / chunks;
  ChunkSpan s;
  s.v0 = min((int64_t)c * per, nv);
  s.v1 = min(s.v0 + per, nv);
  s.tail = c == chunks - 1;
  return s;
}
// f(value) of every element of the span; vec: rows start at 16-byte boundaries
template <typename F>
__device__ __forceinline__ void span_each(const float* __restrict__ row, int64_t vocab, const ChunkSpan& sp, bool vec, F&& f) {
  constexpr int U = 4;
  int64_t i = sp.v0 + threadIdx.x;
  for (; i + (U - 1) * SAMP_THREADS < sp.v1; i += U * SAMP_THREADS) {
    Vec<float, 4> v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float* p = row + (i + u * SAMP_THREADS) * 4;
      if (vec) v[u] = ldvec<float, 4>(p);
      else
#pragma unroll
        for (int j = 0; j < 4; ++j) v[u].v[j] = p[j];
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) f(v[u].v[j]);
  }
  for (; i < sp.v1; i += SAMP_THREADS)
#pragma unroll
    for (int j = 0; j < 4; ++j) f(row[i * 4 + j]);
  if (sp.tail) {
    const int64_t k = vocab / 4 * 4 + threadIdx.x;
    if (k < vocab) f(row[k]);
  }
}

// How a row's exponents are formed.  A temperature that is an ordinary positive number divides once: (x - max x) * (1 / t), where x / t
// takes a precise division per entry in both launches, and no further from float64 (the difference is exact near the maximum, where the mass is).
// Any other temperature (zero, negative, NaN, past 1e30 either way) keeps x / t - max(x / t).
// Which of the two is decided once for a launch's row, in front of its loops: as a choice inside them it had both sides computed for every
// entry, and the division's dozen instructions were a third of what there was (64 rows x 128256: 13.4 and 21.6 us so, 11.5 and 19.2
// this way; 200 rows, whose chunks are not held, 53 and 52 against 38 and 50).
template <bool PLAIN> struct RowScale {
  float t, inv;
  __device__ __forceinline__ explicit RowScale(float t_) : t(t_), inv(1.0f / t_) {}
  __device__ __forceinline__ float key(float x) const { return PLAIN ? x : x / t; }                 // what the maximum is taken of
  __device__ __forceinline__ float power(float k, float mx) const { return expf(PLAIN ? (k - mx) * inv : k - mx); }
};
template <typename F> __device__ __forceinline__ void with_row_scale(float t, F&& f) {
  if (t >= 1e-30f && t <= 1e30f) f(RowScale<true>(t));
  else f(RowScale<false>(t));
}

constexpr int KEEP = 8;   // 16-byte pieces of a chunk that a thread holds: chunks up to 32 K entries, every vocabulary up to 512 K at few rows

// The thread's pieces of a chunk, all requested before anything is used (a piece past the end repeats the last one).
__device__ __forceinline__ void chunk_load(Vec<float, 4> (&v)[KEEP], const float* __restrict__ row, const ChunkSpan& sp) {
#pragma unroll
  for (int u = 0; u < KEEP; ++u) {
    const int64_t i = sp.v0 + threadIdx.x + u * SAMP_THREADS;
    v[u] = ldvec<float, 4>(row + 4 * (i < sp.v1 ? i : sp.v1 - 1));
  }
}

__global__ __launch_bounds__(SAMP_THREADS) void softmax_partials_kernel(
    float2* __restrict__ partials, const float* __restrict__ logits, const float* __restrict__ temperatures, int64_t vocab,
    int64_t row_stride) {
  __shared__ float red[SAMP_THREADS / 64];
  const int r = blockIdx.x, c = blockIdx.y, chunks = gridDim.y;
  const float* row = logits + (int64_t)r * row_stride;
  const bool vec = (row_stride % 4 == 0) && aligned16(logits);
  const ChunkSpan sp = chunk_span(vocab, c, chunks);
  const float t = temperatures[r];
  float mx = -INFINITY, sum = 0.f;
  // More rows have fewer and longer chunks (row_chunks), which go through span_each twice: both launches at 128256 entries, 64 rows
  // (4 chunks) 41 us, 86 (3) 73, 200 (2) 116; a whole row a workgroup 157, 163, 182 (all with a division per entry: 200 rows are 82 without).
  if (vec && sp.v1 - sp.v0 <= KEEP * SAMP_THREADS && sp.v0 < sp.v1) {
    // The chunk is read once, into registers.
    Vec<float, 4> v[KEEP];
    chunk_load(v, row, sp);
    const int64_t k = vocab / 4 * 4 + threadIdx.x;
    const bool one = sp.tail && k < vocab;
    float last = one ? row[k] : -INFINITY;
    with_row_scale(t, [&](auto rs) {
      if (one) last = rs.key(last);
#pragma unroll
      for (int u = 0; u < KEEP; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[u].v[j] = rs.key(v[u].v[j]);
          mx = fmaxf(mx, v[u].v[j]);   // (a piece past the end repeats the last one: the maximum does not mind)
        }
      mx = block_reduce_max(fmaxf(mx, last), red);
      const float ref = mx == -INFINITY ? 0.f : mx;
#pragma unroll
      for (int u = 0; u < KEEP; ++u)
        if (sp.v0 + threadIdx.x + u * SAMP_THREADS < sp.v1)
#pragma unroll
          for (int j = 0; j < 4; ++j) sum += rs.power(v[u].v[j], ref);
      if (one) sum += rs.power(last, ref);
    });
  } else {
    with_row_scale(t, [&](auto rs) {
      span_each(row, vocab, sp, vec, [&](float x) { mx = fmaxf(mx, rs.key(x)); });
      mx = block_reduce_max(mx, red);
      const float ref = mx == -INFINITY ? 0.f : mx;
      span_each(row, vocab, sp, vec, [&](float x) { sum += rs.power(rs.key(x), ref); });
    });
  }
  sum = block_reduce_sum(sum, red);
  if (threadIdx.x == 0) partials[(int64_t)r * chunks + c] = float2{mx, sum};
}

// The row's maximum and sum from what its chunks left, and the entries' probabilities.  p: the lane's chunk (a lane per chunk).
__device__ __forceinline__ float2 chunk_partial(const float2* __restrict__ partials, int chunks) {
  const int i = threadIdx.x & (MAX_CHUNKS - 1);
  return i < chunks ? partials[i] : float2{-INFINITY, 0.f};
}
template <typename SCALE> struct RowNorm {
  SCALE rs;
  float mx, sum, inv_sum;
  __device__ __forceinline__ RowNorm(SCALE rs_, float2 p, int chunks) : rs(rs_) {
    mx = p.x;
#pragma unroll
    for (int o = MAX_CHUNKS / 2; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    sum = (int)(threadIdx.x & (MAX_CHUNKS - 1)) < chunks ? p.y * rs.power(p.x, mx) : 0.f;
#pragma unroll
    for (int o = MAX_CHUNKS / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
    inv_sum = 1.0f / sum;
  }
  // e / sum with sum in [1, vocab] (or NaN): the quotient by the reciprocal and one correction, in four operations
  __device__ __forceinline__ float prob(float x) const {
    const float e = rs.power(rs.key(x), mx), q = e * inv_sum;
    return fmaf(fmaf(-q, sum, e), inv_sum, q);
  }
};

// ---- joint top-k / top-p / min-p filter + inverse-CDF draw --------------------------------
// The kept set is {p >= tau}: tau is the smallest probability value v such that fewer than k
// entries are strictly larger than v and the mass strictly above v is <= top_p.  It is found
// by a 4-level radix select on the float bit pattern (non-negative floats order like their
// bits) with 256-bin count/mass histograms in LDS, i.e. 4 passes over the row instead of a
// sort.  min_p raises tau to min_p * pmax.  The draw walks the kept entries in index order.
struct SampleRow {
  const float* row;
  int64_t k;
  float top_p, min_p, uniform;
};
__device__ __forceinline__ SampleRow sample_row(const float* probs, const int32_t* top_ks, const float* top_ps,
                                                const float* min_ps, const float* uniform, int64_t row_stride) {
  SampleRow r;
  r.row = probs + (int64_t)blockIdx.x * row_stride;
  r.k = top_ks ? (int64_t)top_ks[blockIdx.x] : (int64_t)1 << 30;
  r.top_p = top_ps ? top_ps[blockIdx.x] : 1.0f;
  if (r.top_p >= 1.0f) r.top_p = INFINITY;  // disabled: no rounding artefacts at the tail
  r.min_p = min_ps ? min_ps[blockIdx.x] : 0.0f;
  r.uniform = uniform[blockIdx.x];
  return r;
}

// The routine's LDS comes from the kernel, which may have other uses for it.  Every piece starts at a 16-byte boundary and is
// an array of its own: the serial walks over them, what a short row spends its time on, then move four entries at a time (1 row
// of 1000 entries: 49 us; 56 as members of one structure without the boundaries).
struct SampleScratch {
  alignas(16) unsigned int hcount[256];
  alignas(16) float hmass[256];
  alignas(16) float scan[SAMP_THREADS];
  alignas(16) float red[SAMP_THREADS / 64];
};

__device__ __forceinline__ void sample_whole_row(int32_t* __restrict__ ids, const SampleRow& sr, int64_t vocab, unsigned int (&hcount)[256],
                                                 float (&hmass)[256], float (&s_scan)[SAMP_THREADS], float (&red)[SAMP_THREADS / 64]) {
  __shared__ unsigned int s_prefix;   // bits fixed so far (high bits of tau)
  __shared__ unsigned int s_count;    // entries strictly above the current bin range
  __shared__ float s_mass;            // mass strictly above the current bin range
  __shared__ int s_pick;
  const float* row = sr.row;
  const int64_t k = sr.k;
  const float top_p = sr.top_p, min_p = sr.min_p;

  if (threadIdx.x == 0) {
    s_prefix = 0;
    s_count = 0;
    s_mass = 0.f;
  }
  float pmax = 0.f;
  for (int64_t i = threadIdx.x; i < vocab; i += SAMP_THREADS) pmax = fmaxf(pmax, row[i]);
  pmax = block_reduce_max(pmax, red);

  for (int level = 0; level < 4; ++level) {
    const int shift = 24 - 8 * level;
    for (int i = threadIdx.x; i < 256; i += SAMP_THREADS) {
      hcount[i] = 0;
      hmass[i] = 0.f;
    }
    __syncthreads();
    const unsigned int prefix = s_prefix;
    const unsigned int himask = level == 0 ? 0u : (0xffffffffu << (shift + 8));
    for (int64_t i = threadIdx.x; i < vocab; i += SAMP_THREADS) {
      const float v = row[i];
      const unsigned int bits = __float_as_uint(v > 0.f ? v : 0.f);
      if ((bits & himask) == prefix) {
        const unsigned int bin = (bits >> shift) & 0xffu;
        atomicAdd(&hcount[bin], 1u);
        atomicAdd(&hmass[bin], v > 0.f ? v : 0.f);
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      unsigned int cnt = s_count;
      float mass = s_mass;
      int bin = 255;
      // walk down while every entry of the bin is certainly kept
      for (; bin > 0; --bin) {
        if (hcount[bin] == 0) continue;
        // the smallest entry of this bin sees at most cnt + hcount-1 larger entries and at
        // most mass + hmass (minus itself) above it; if the whole bin passes, keep going.
        const bool all_pass = (int64_t)cnt + hcount[bin] <= k && mass + hmass[bin] <= top_p;
        if (!all_pass) break;
        cnt += hcount[bin];
        mass += hmass[bin];
      }
      s_prefix = prefix | ((unsigned int)bin << shift);
      s_count = cnt;
      s_mass = mass;
    }
    __syncthreads();
  }
  // s_prefix is now a full 32-bit pattern v0.  Entries > v0 number s_count with mass s_mass;
  // entries == v0 are kept iff s_count < k and s_mass <= top_p (and v0 > 0).
  const unsigned int v0bits = s_prefix;
  const bool keep_v0 = (int64_t)s_count < k && s_mass <= top_p;
  float tau = __uint_as_float(keep_v0 ? v0bits : v0bits + 1u);  // next float up excludes v0
  tau = fmaxf(tau, min_p * pmax);
  if (!(tau > 0.f)) tau = __uint_as_float(1u);  // never keep zero-probability entries

  // total kept mass
  const int64_t per = (vocab + SAMP_THREADS - 1) / SAMP_THREADS;
  const int64_t lo = threadIdx.x * per, hi = lo + per < vocab ? lo + per : vocab;
  float part = 0.f;
  for (int64_t i = lo; i < hi; ++i) {
    const float v = row[i];
    if (v >= tau) part += v;
  }
  s_scan[threadIdx.x] = part;
  if (threadIdx.x == 0) s_pick = -1;
  __syncthreads();
  if (threadIdx.x == 0) {
    // serial exclusive scan of 1024 partials: tiny, deterministic
    float run = 0.f;
    for (int i = 0; i < SAMP_THREADS; ++i) {
      const float t = s_scan[i];
      s_scan[i] = run;
      run += t;
    }
    red[0] = run;
  }
  __syncthreads();
  const float total = red[0];
  const float target = sr.uniform * total;
  // the chunk containing the target: exclusive prefix <= target < prefix + part
  const float before = s_scan[threadIdx.x];
  if (part > 0.f && before <= target && (target < before + part)) {
    float run = before;
    int pick = -1;
    for (int64_t i = lo; i < hi; ++i) {
      const float v = row[i];
      if (v >= tau) {
        run += v;
        pick = (int)i;
        if (run > target) break;
      }
    }
    atomicMax(&s_pick, pick);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int pick = s_pick;
    if (pick < 0) {
      // rounding at the very end of the CDF: fall back to the last kept entry
      for (int64_t i = vocab - 1; i >= 0; --i)
        if (row[i] >= tau) {
          pick = (int)i;
          break;
        }
      if (pick < 0) pick = 0;
    }
    ids[blockIdx.x] = pick;
  }
}

__global__ __launch_bounds__(SAMP_THREADS) void topk_topp_minp_sample_kernel(
    int32_t* __restrict__ ids, const float* __restrict__ probs, const int32_t* __restrict__ top_ks,
    const float* __restrict__ top_ps, const float* __restrict__ min_ps,
    const float* __restrict__ uniform, int64_t vocab, int64_t row_stride) {
  __shared__ __attribute__((aligned(16))) unsigned int hcount[256];
  __shared__ __attribute__((aligned(16))) float hmass[256];
  __shared__ __attribute__((aligned(16))) float scan[SAMP_THREADS];
  __shared__ __attribute__((aligned(16))) float red[SAMP_THREADS / 64];
  sample_whole_row(ids, sample_row(probs, top_ks, top_ps, min_ps, uniform, row_stride), vocab, hcount, hmass, scan, red);
}

// ---- the same draw over chunks of a row -------------------------------------------------------
// Launch 1, a workgroup per chunk: the chunk's positive entries in 2048 bins of 1/16 binade (the upper 13 bits of the
// pattern), its maximum, and the entries of its highest bins as a list.  Entries of a bin share exponent and upper mantissa, so their
// count (upper 24 bits) and the sum of their 19 lower bits (lower 40) in one integer are their mass exactly, for one LDS atomic each; a
// count and a float atomic took 47 us where this takes 10.  With the softmax in front the launch is that one's second (softmax_sample).
// Launch 2, a workgroup per row: the first bin from the top that is not kept whole holds tau, and its entries are searched bit by bit.
// Where the chunks' lists reach down to that bin -- top_k, top_p or min_p of common size -- they are all that is read: four entries a
// thread, in registers, tau and the draw from them.  Otherwise (thousands kept, chunks that are not held in registers) the chunks' bins
// give the cut, its entries are collected in LDS by one pass over the row, and the draw is made among them if they and the larger ones
// are few, else a second pass sums what is kept per tile of 256 entries, and the tile the draw falls into is walked.  More entries in
// that bin than the list holds (an almost flat row) are searched in the row itself, a pass per step.  A row whose tau lies above 1.9
// (no probability does) takes sample_whole_row.
// The one-workgroup routine meets each of its four levels' 128256 entries in 256 bins of two binades, a handful of which
// take nearly all of them: 64 rows of 128256 with top_k 50, top_p 0.9 took 451 us, bound by those LDS atomics.  Launch 1 beside the
// softmax takes 19 us for that (apart 10 + 14), bound by LDS atomics, exponentials and 66 MB read and written; launch 2 takes 12 from the
// lists, a chain of some twenty barriers (28 from the row, one CU's pass over 0.5 MB; 58 when thousands are kept).
constexpr int SB_BINS = 2048, SB_SHIFT = 19, SB_LIST = 8192, SB_SHORT = 512, SB_TILE = 256, SB_MAX_TILES = 4096;
constexpr int SB_SUM_BITS = 40;
constexpr int64_t SB_MAX_VOCAB = (int64_t)SB_TILE * SB_MAX_TILES;   // 2^20: counts fit 24 bits, sums of 19 bits fit 40
typedef unsigned long long u64_t;

// The mass of x = (entries << SB_SUM_BITS) + the sum of their lower bits, where `bits` is the pattern they share above those.
__device__ __forceinline__ float bin_mass(unsigned bits, u64_t x) {
  const unsigned e = bits >> 23;                                                        // exponent field
  const double base = (double)((bits & ((1u << 23) - 1)) + (e ? 1u << 23 : 0u));        // an entry's mantissa without its lower bits
  return (float)ldexp((double)(x >> SB_SUM_BITS) * base + (double)(x & (((u64_t)1 << SB_SUM_BITS) - 1)), (int)(e ? e : 1u) - 150);
}

// What a chunk leaves beside its bins: the entries of its highest bins, in index order -- whole bins until there are more than top_k
// entries (the row's cut cannot lie below the bin that has the chunk's own top_k-th), but at most 1 / chunks of SB_TOP.  Those are nearly
// always all that a draw can take (top_p and min_p cut from below too), so that launch 2 reads them instead of the row.
constexpr int SB_TOP = 4096;
struct ChunkTop {
  int count;      // entries listed; -1: none are (a chunk that its workgroup does not hold in registers)
  int bin;        // the lowest bin listed
  float mx;       // the chunk's maximum
  int pad;
};
struct BinScratch {
  u64_t hist[SB_BINS];
  float red[SAMP_THREADS / 64];
  int waves[SAMP_THREADS / 64];
  int pieces[(KEEP + 1) * (SAMP_THREADS / 64)];
  int passing, listed;
};
__device__ __forceinline__ unsigned sb_bin(float v) { return min(__float_as_uint(v) >> SB_SHIFT, (unsigned)(SB_BINS - 1)); }
__device__ __forceinline__ void sb_count(u64_t* hist, float v) {
  if (v > 0.f) atomicAdd(&hist[sb_bin(v)], ((u64_t)1 << SB_SUM_BITS) + (__float_as_uint(v) & ((1u << SB_SHIFT) - 1)));
}

// Over a wave, all 64 lanes at it, in registers (rows of 16, then a row's last lane onto the next and the first half's onto the second);
// whole numbers, so that the order leaves no trace.  Inclusive sum, and largest value (of numbers >= 0).  The thirty exchanges of a chunk's
// list through the LDS crossbar, each waiting for the last, took 1 us of a launch: 8 rows x 128256 10.9 us for bins and lists so, 9.9 this way.
template <int CTRL, int ROWS> __device__ __forceinline__ int lanes_moved(int x) { return __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xF, false); }
__device__ __forceinline__ int wave_scan(int x) {
  x += lanes_moved<0x111, 0xF>(x);   // row_shr:1, 2, 4, 8
  x += lanes_moved<0x112, 0xF>(x);
  x += lanes_moved<0x114, 0xF>(x);
  x += lanes_moved<0x118, 0xF>(x);
  x += lanes_moved<0x142, 0xA>(x);   // row_bcast:15 onto rows 1 and 3
  return x + lanes_moved<0x143, 0xC>(x);   // row_bcast:31 onto rows 2 and 3
}
__device__ __forceinline__ int wave_largest(int x) {
  x = max(x, lanes_moved<0x111, 0xF>(x));
  x = max(x, lanes_moved<0x112, 0xF>(x));
  x = max(x, lanes_moved<0x114, 0xF>(x));
  x = max(x, lanes_moved<0x118, 0xF>(x));
  x = max(x, lanes_moved<0x142, 0xA>(x));
  return __builtin_amdgcn_readlane(max(x, lanes_moved<0x143, 0xC>(x)), 63);
}

// A chunk in registers (v as chunk_load lays it out, `last`: the thread's entry of the row's tail or 0): its list.  sm.hist is complete.
__device__ __forceinline__ void chunk_list(const Vec<float, 4> (&v)[KEEP], float last, const ChunkSpan& sp, int64_t vocab, int most,
                                           int want, BinScratch& sm, uint2* __restrict__ list, int& count, int& lowest) {
  constexpr int W = SAMP_THREADS / 64;
  const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // entries in this thread's two bins and all above
  const int c1 = (int)(sm.hist[SB_BINS - 1 - 2 * tid] >> SB_SUM_BITS), c0 = (int)(sm.hist[SB_BINS - 2 - 2 * tid] >> SB_SUM_BITS);
  const int incl = wave_scan(c0 + c1);
  if (lane == 63) sm.waves[wave] = incl;
  if (tid == 0) sm.passing = sm.listed = 0;
  __syncthreads();
  int above = incl;
#pragma unroll
  for (int w = 0; w < W; ++w) above += w < wave ? sm.waves[w] : 0;
  // A bin is listed if it and those above hold at most `most` entries, and those above it no more than `want` (counts grow on the way
  // down: the bins that pass are the highest ones).
  const int upper = above - c0, before_both = upper - c1;
  const bool high = upper <= most && before_both <= want, low = above <= most && upper <= want;
  const int pass = __popcll(__ballot(high)) + __popcll(__ballot(low));
  const int got = wave_largest(low ? above : high ? upper : 0);
  if (lane == 0) {
    atomicAdd(&sm.passing, pass);
    atomicMax(&sm.listed, got);
  }
  __syncthreads();
  lowest = SB_BINS - sm.passing;
  count = sm.listed;
  // the smallest value listed; nothing compares with NaN
  const float from = lowest == SB_BINS ? NAN : __uint_as_float(max((unsigned)lowest << SB_SHIFT, 1u));
  // places in index order: pieces, waves in a piece, lanes in a wave, four entries of a lane
  int at[KEEP + 1];
#pragma unroll
  for (int u = 0; u <= KEEP; ++u) {
    const bool there = u == KEEP || sp.v0 + tid + u * SAMP_THREADS < sp.v1;
    const Vec<float, 4> x = u == KEEP ? Vec<float, 4>{{last, 0.f, 0.f, 0.f}} : v[u < KEEP ? u : 0];
    int before = 0, total = 0, own = 0;
    if (__any(there && (x.v[0] >= from || x.v[1] >= from || x.v[2] >= from || x.v[3] >= from)))
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool in = there && x.v[j] >= from;
        const u64_t m = __ballot(in);
        before += __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
        total += __popcll(m);
        own |= in ? 1 << j : 0;
      }
    at[u] = own ? before << 4 | own : 0;
    if (lane == 0) sm.pieces[u * W + wave] = total;
  }
  __syncthreads();
  if (wave == 0) {
    int run = 0;
#pragma unroll
    for (int i = 0; i < (KEEP + 1) * W; i += 64) {
      const int n = i + lane < (KEEP + 1) * W ? sm.pieces[i + lane] : 0;
      const int x = wave_scan(n);
      if (i + lane < (KEEP + 1) * W) sm.pieces[i + lane] = run + x - n;
      run += __builtin_amdgcn_readlane(x, 63);
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u <= KEEP; ++u)
    if (at[u] != 0) {
      int to = sm.pieces[u * W + wave] + (at[u] >> 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (u == KEEP && j > 0) break;
        if (at[u] >> j & 1) {
          const float x = u == KEEP ? last : v[u < KEEP ? u : 0].v[j];
          const int64_t index = u == KEEP ? vocab / 4 * 4 + tid : (sp.v0 + tid + u * SAMP_THREADS) * 4 + j;
          list[to++] = uint2{__float_as_uint(x), (unsigned)index};
        }
      }
    }
}

// NORM: `data` holds logits, which become probabilities on the way (launch 2 of softmax_temperature); BINS: bins and lists of the
// probabilities.  Both at once: 64 rows x 128256 19 us, apart 10 + 14.
template <bool NORM, bool BINS>
__global__ __launch_bounds__(SAMP_THREADS) void sample_chunk_kernel(float* __restrict__ data, const float2* __restrict__ partials,
                                                                    const float* __restrict__ temperatures, const int32_t* __restrict__ top_ks,
                                                                    const float* __restrict__ top_ps, u64_t* __restrict__ bins, uint2* __restrict__ lists, ChunkTop* __restrict__ tops, int64_t vocab,
                                                                    int64_t row_stride) {
  __shared__ BinScratch sm;
  const int r = blockIdx.x, c = blockIdx.y, chunks = gridDim.y, tid = (int)threadIdx.x;
  float* row = data + (int64_t)r * row_stride;
  const bool vec = (row_stride % 4 == 0) && aligned16(data);
  const ChunkSpan sp = chunk_span(vocab, c, chunks);
  // A row that neither top_k nor top_p cuts short draws from entries that no list has, and without a list or a softmax nothing is gained by
  // holding the chunk either (300 rows x 32768: 30 us with lists, 14 with the chunk held, 10.5 so).
  const int want = BINS && top_ks != nullptr ? max(top_ks[r], 0) : 0x7fffffff;
  const bool listed = BINS && (want <= SB_TOP || (top_ps != nullptr && top_ps[r] < 1.0f));
  const bool held = (NORM || listed) && vec && sp.v1 - sp.v0 <= KEEP * SAMP_THREADS && sp.v0 < sp.v1;
  const float temperature = NORM ? temperatures[r] : 1.0f;
  const float2 partial = NORM ? chunk_partial(partials + (int64_t)r * chunks, chunks) : float2{0.f, 0.f};
  const int64_t k = vocab / 4 * 4 + tid;
  const bool one = sp.tail && k < vocab;
  float mx = 0.f, last = one ? row[k] : 0.f;
  int count = -1, lowest = SB_BINS;
  auto clear = [&] {
    if constexpr (BINS) {
      for (int i = tid; i < SB_BINS; i += SAMP_THREADS) sm.hist[i] = 0;
      __syncthreads();
    }
  };
  // f(prob), prob: of a logit, or the probability that it is already; the row's tail entry is taken here
  auto with_prob = [&](auto&& f) {
    auto go = [&](auto prob) {
      if (one) {
        last = prob(last);
        if (NORM) row[k] = last;
        mx = fmaxf(mx, last);
        if (BINS) sb_count(sm.hist, last);
      }
      f(prob);
    };
    if constexpr (NORM)
      with_row_scale(temperature, [&](auto rs) {
        const RowNorm<decltype(rs)> norm(rs, partial, chunks);
        go([&](float x) { return norm.prob(x); });
      });
    else
      go([](float x) { return x; });
  };
  if (held) {
    Vec<float, 4> v[KEEP];
    chunk_load(v, row, sp);
    clear();
    with_prob([&](auto prob) {
#pragma unroll
      for (int u = 0; u < KEEP; ++u) {
        const int64_t i = sp.v0 + tid + u * SAMP_THREADS;
        if (i < sp.v1) {
          if constexpr (NORM) {
            Vec<float, 4> w;
#pragma unroll
            for (int j = 0; j < 4; ++j) w.v[j] = prob(v[u].v[j]);
            stvec<float, 4>(row + i * 4, w);
            if (BINS) v[u] = w;
          }
          if constexpr (BINS)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              mx = fmaxf(mx, v[u].v[j]);
              sb_count(sm.hist, v[u].v[j]);
            }
        }
      }
    });
    if constexpr (BINS) {
      __syncthreads();
      const int most = SB_TOP / chunks;
      if (listed) chunk_list(v, last, sp, vocab, most, want, sm, lists + (int64_t)r * SB_TOP + c * most, count, lowest);
    }
  } else {
    clear();
    with_prob([&](auto prob) {
      auto load = [&](int64_t i) {
        Vec<float, 4> w;
        if (vec) w = ldvec<float, 4>(row + i * 4);
        else
#pragma unroll
          for (int j = 0; j < 4; ++j) w.v[j] = row[i * 4 + j];
        return w;
      };
      auto take = [&](Vec<float, 4> w, int64_t i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (NORM) w.v[j] = prob(w.v[j]);
          mx = fmaxf(mx, w.v[j]);
          if (BINS) sb_count(sm.hist, w.v[j]);
        }
        if (NORM) {
          if (vec) stvec<float, 4>(row + i * 4, w);
          else
#pragma unroll
            for (int j = 0; j < 4; ++j) row[i * 4 + j] = w.v[j];
        }
      };
      int64_t i = sp.v0 + tid;
      if constexpr (!NORM) {     // four loads in flight (beside the exponentials they gain nothing: 200 rows x 128256 166 us the batch, 173 so)
        for (; i + 3 * SAMP_THREADS < sp.v1; i += 4 * SAMP_THREADS) {
          Vec<float, 4> w[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) w[u] = load(i + u * SAMP_THREADS);
#pragma unroll
          for (int u = 0; u < 4; ++u) take(w[u], i + u * SAMP_THREADS);
        }
      }
      for (; i < sp.v1; i += SAMP_THREADS) take(load(i), i);
    });
  }
  if constexpr (BINS) {
    mx = block_reduce_max(mx, sm.red);
    u64_t* out = bins + ((int64_t)r * chunks + c) * SB_BINS;
    for (int i = tid; i < SB_BINS; i += SAMP_THREADS) out[i] = sm.hist[i];
    if (tid == 0) tops[(int64_t)r * chunks + c] = ChunkTop{count, lowest, mx, 0};
  }
}

// Of N bins (counts and masses in LDS), going down from the top: the first bin that is not kept whole, with the count and
// mass above it; bin -1 if there is none.  Counts and masses grow on the way down, so from that bin on none is.  Empty
// bins are passed over.  Every thread returns the same; begins and ends with a barrier.
struct BinCut {
  int bin;
  unsigned count;
  float mass;
};
struct CutScratch {
  unsigned wc[SAMP_THREADS / 64];
  float wm[SAMP_THREADS / 64];
  BinCut cut;
};
template <int N>
__device__ __forceinline__ BinCut cut_bins(const unsigned* hcount, const float* hmass, int64_t k, float top_p, unsigned count0,
                                           float mass0, CutScratch& sm) {
  constexpr int PER = (N + SAMP_THREADS - 1) / SAMP_THREADS;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int top = N - 1 - (int)threadIdx.x * PER;     // this thread's bins: top, top - 1, .. (PER of them)
  __syncthreads();
  unsigned c[PER], ci = 0;
  float m[PER], mi = 0.f;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    c[j] = top - j >= 0 ? hcount[top - j] : 0u;
    m[j] = top - j >= 0 ? hmass[top - j] : 0.f;
    ci += c[j];
    mi += m[j];
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned oc = __shfl_up(ci, o, 64);
    const float om = __shfl_up(mi, o, 64);
    if (lane >= o) {
      ci += oc;
      mi += om;
    }
  }
  if (lane == 63) {
    sm.wc[wave] = ci;
    sm.wm[wave] = mi;
  }
  if (threadIdx.x == 0) sm.cut = BinCut{-1, 0u, 0.f};
  const unsigned cx = __shfl_up(ci, 1, 64);            // what the lanes before this one have
  const float mx = __shfl_up(mi, 1, 64);
  __syncthreads();
  unsigned above = count0;
  float mass = mass0;
#pragma unroll
  for (int w = 0; w < SAMP_THREADS / 64; ++w) {
    const unsigned wc = sm.wc[w];
    const float wm = sm.wm[w];
    above += w < wave ? wc : 0u;
    mass += w < wave ? wm : 0.f;
  }
  if (lane > 0) {
    above += cx;
    mass += mx;
  }
  BinCut mine{-1, 0u, 0.f};
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    if (mine.bin < 0 && c[j] != 0) {
      if ((int64_t)above + c[j] <= k && mass + m[j] <= top_p) {
        above += c[j];
        mass += m[j];
      } else {
        mine = BinCut{top - j, above, mass};
      }
    }
  }
  if (mine.bin >= 0) atomicMax(&sm.cut.bin, mine.bin);
  __syncthreads();
  if (mine.bin >= 0 && mine.bin == sm.cut.bin) {
    sm.cut.count = mine.count;
    sm.cut.mass = mine.mass;
  }
  __syncthreads();
  return sm.cut;
}

// Four elements of a row from group i on (groups of 4; vec: one 16-byte load), zeros past the end.
__device__ __forceinline__ Vec<float, 4> row4(const float* __restrict__ row, int64_t vocab, int64_t i, bool vec) {
  Vec<float, 4> v;
  if (vec && i * 4 + 4 <= vocab) return ldvec<float, 4>(row + i * 4);
#pragma unroll
  for (int j = 0; j < 4; ++j) v.v[j] = i * 4 + j < vocab ? row[i * 4 + j] : 0.f;
  return v;
}

__global__ __launch_bounds__(SAMP_THREADS) void sample_pick_kernel(
    int32_t* __restrict__ ids, const u64_t* __restrict__ bins, const uint2* __restrict__ lists, const ChunkTop* __restrict__ tops, int chunks,
    const float* __restrict__ probs, const int32_t* __restrict__ top_ks, const float* __restrict__ top_ps,
    const float* __restrict__ min_ps, const float* __restrict__ uniform, int64_t vocab, int64_t row_stride) {
  // 2048 bins as counts and masses, or as the integers that both come from
  __shared__ alignas(16) u64_t hist[SB_BINS];
  unsigned* const hcount = reinterpret_cast<unsigned*>(hist);
  float* const hmass = reinterpret_cast<float*>(hist + SB_BINS / 2);
  __shared__ alignas(16) u64_t cells[1024];      // counts and sums of the cut bin's parts
  __shared__ union {
    unsigned list[SB_LIST];        // the cut bin's entries where the chunks' lists do not reach it, until tau is known
    float tile[SB_MAX_TILES];      // kept mass per tile of 256 entries, afterwards
    SampleScratch whole;
  } sm;
  __shared__ CutScratch cs;
  __shared__ double sums[SAMP_THREADS / 64];
  __shared__ unsigned n_list;
  __shared__ int s_tile, s_last, s_pick;
  __shared__ float s_before;
  const SampleRow sr = sample_row(probs, top_ks, top_ps, min_ps, uniform, row_stride);
  const float* row = sr.row;
  const bool vec = (row_stride % 4 == 0) && aligned16(probs);
  const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const ChunkTop* top = tops + (int64_t)blockIdx.x * chunks;
  const int most = SB_TOP / chunks;
  if (tid == 0) {
    n_list = 0;
    s_tile = SB_MAX_TILES;
    s_last = -1;
    s_pick = 0x7fffffff;
  }
  // The chunks' lists, four neighbouring slots a thread (an empty one is 0.0: not an entry); if all chunks have one they are complete
  // from bin `floor` on.  A lane per chunk.
  constexpr int SLOTS = SB_TOP / SAMP_THREADS;
  uint2 slot[SLOTS];
#pragma unroll
  for (int j = 0; j < SLOTS; ++j) {
    const int at = tid * SLOTS + j;
    slot[j] = lists[(int64_t)blockIdx.x * SB_TOP + min(at, most * chunks - 1)];
  }
  const int ci = tid & (MAX_CHUNKS - 1);
  const ChunkTop mine = top[min(ci, chunks - 1)];
  float pmax = mine.mx;
  int floor = mine.bin;
  bool lists_hold = __ballot(mine.count < 0) == 0;
#pragma unroll
  for (int o = MAX_CHUNKS / 2; o > 0; o >>= 1) {
    pmax = fmaxf(pmax, __shfl_xor(pmax, o, 64));
    floor = max(floor, __shfl_xor(floor, o, 64));
  }
#pragma unroll
  for (int j = 0; j < SLOTS; ++j) {
    const int at = tid * SLOTS + j, c = min(at / most, chunks - 1);
    const bool there = at - c * most < __shfl(mine.count, c, 64);
    if (!there) slot[j].x = 0u;
  }
  auto split = [&](int i, u64_t v) {     // (between two barriers)
    hcount[i] = (unsigned)(v >> SB_SUM_BITS);
    hmass[i] = bin_mass((unsigned)i << SB_SHIFT, v);
  };
  BinCut cut{-1, 0u, 0.f};
  if (lists_hold) {
    hist[tid] = hist[tid + SAMP_THREADS] = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < SLOTS; ++j)
      if ((int)sb_bin(__uint_as_float(slot[j].x)) >= floor) sb_count(hist, __uint_as_float(slot[j].x));
    __syncthreads();
    const u64_t lo = hist[tid], hi = hist[tid + SAMP_THREADS];
    __syncthreads();
    split(tid, lo);
    split(tid + SAMP_THREADS, hi);
    cut = cut_bins<SB_BINS>(hcount, hmass, sr.k, sr.top_p, 0u, 0.f, cs);
    lists_hold = cut.bin >= 0 || floor == 0;     // (everything above zero is listed and kept, or the cut lies below)
  }
  if (!lists_hold) {
    const u64_t* rb = bins + (int64_t)blockIdx.x * chunks * SB_BINS;
    u64_t lo = 0, hi = 0;
    for (int c = 0; c < chunks; ++c) {
      lo += rb[(int64_t)c * SB_BINS + tid];
      hi += rb[(int64_t)c * SB_BINS + tid + SAMP_THREADS];
    }
    __syncthreads();
    split(tid, lo);
    split(tid + SAMP_THREADS, hi);
    cut = cut_bins<SB_BINS>(hcount, hmass, sr.k, sr.top_p, 0u, 0.f, cs);
  }
  float tau = 0.f;
  bool few = false;
  if (cut.bin >= 0) {
    unsigned size = hcount[cut.bin];
    if (cut.bin == SB_BINS - 1) {
      __syncthreads();
      sample_whole_row(ids, sr, vocab, sm.whole.hcount, sm.whole.hmass, sm.whole.scan, sm.whole.red);
      return;
    }
    few = !lists_hold && cut.count + size <= (unsigned)SB_SHORT;
    // the cut bin's entries; with the larger ones and everybody's index if they are few
    const unsigned lowest = (unsigned)cut.bin << SB_SHIFT, bound = few ? 0x7f800001u : lowest + (1u << SB_SHIFT);   // (few: up to infinity, which the bins have counted)
    const bool listed = few || size <= (unsigned)SB_LIST;
    // f(bits, index) of every entry of the row in [lo, hi) patterns
    auto row_each = [&](unsigned lo, unsigned hi, auto&& f) {
      constexpr int U = 8;
      const int64_t groups = (vocab + 3) / 4;
      for (int64_t i0 = threadIdx.x; i0 < groups; i0 += U * SAMP_THREADS) {
        Vec<float, 4> v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int64_t i = i0 + u * SAMP_THREADS;
          if (i < groups) v[u] = row4(row, vocab, i, vec);
          else v[u] = Vec<float, 4>{{0.f, 0.f, 0.f, 0.f}};
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const unsigned bits = __float_as_uint(v[u].v[j]);
            if (v[u].v[j] > 0.f && bits >= lo && bits < hi) f(bits, (unsigned)((i0 + u * SAMP_THREADS) * 4 + j));
          }
      }
    };
    if (listed && !lists_hold)
      row_each(lowest, bound, [&](unsigned bits, unsigned index) {
        const unsigned at = atomicAdd(&n_list, 1u);
        if (at < (unsigned)SB_LIST) sm.list[at] = bits;
        if (few && at < (unsigned)SB_SHORT) sm.list[SB_SHORT + at] = index;
      });
    if (few) size += cut.count;
    // its 19 lower bits, ten and then nine of them
    unsigned prefix = (unsigned)cut.bin;
    unsigned himask = ~0u << SB_SHIFT;
    const int shifts[2] = {9, 0};
#pragma unroll
    for (int level = 0; level < 2; ++level) {
      const int nb = level == 0 ? 1024 : 512, shift = shifts[level];
      const unsigned want = prefix << (level == 0 ? SB_SHIFT : 9);
      __syncthreads();
      cells[tid] = 0;
      __syncthreads();
      auto part = [&](unsigned bits) {
        atomicAdd(&cells[(bits >> shift) & (unsigned)(nb - 1)], ((u64_t)1 << SB_SUM_BITS) + (bits & ((1u << shift) - 1)));
      };
      if (lists_hold) {
#pragma unroll
        for (int j = 0; j < SLOTS; ++j)
          if (slot[j].x != 0u && (slot[j].x & himask) == want) part(slot[j].x);
      } else if (listed) {
        for (unsigned i = threadIdx.x; i < size; i += SAMP_THREADS)
          if ((sm.list[i] & himask) == want) part(sm.list[i]);
      } else {
        row_each(want, want - himask, [&](unsigned bits, unsigned) { part(bits); });
      }
      __syncthreads();
      hcount[tid] = (unsigned)(cells[tid] >> SB_SUM_BITS);
      hmass[tid] = bin_mass(want + ((unsigned)tid << shift), cells[tid]);     // (parts past nb: none)
      const BinCut next = cut_bins<1024>(hcount, hmass, sr.k, sr.top_p, cut.count, cut.mass, cs);
      // the coarser bin was not kept whole, but its parts' rounded masses may add up to less: then its lowest part is taken
      cut = next.bin >= 0 ? next : BinCut{0, cut.count, cut.mass};
      prefix = (prefix << (level == 0 ? 10 : 9)) | (unsigned)cut.bin;
      himask = ~0u << shift;
    }
    // entries above the pattern number cut.count with mass cut.mass; those equal to it are kept iff the rule still holds
    const bool keep = (int64_t)cut.count < sr.k && cut.mass <= sr.top_p;
    tau = __uint_as_float(keep ? prefix : prefix + 1u);
  }
  tau = fmaxf(tau, sr.min_p * pmax);
  if (!(tau > 0.f)) tau = __uint_as_float(1u);   // never keep zero-probability entries
  if (lists_hold) {
    // the draw among the chunks' lists, four neighbouring entries a thread; sums in double
    double upto[SLOTS], run = 0.0;
    bool in[SLOTS];
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) {
      const float p = __uint_as_float(slot[j].x);
      in[j] = slot[j].x != 0u && p >= tau;
      run += in[j] ? (double)p : 0.0;
      upto[j] = run;
    }
    double incl = run;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const double up = __shfl_up(incl, o, 64);
      if (lane >= o) incl += up;
    }
    if (lane == 63) sums[wave] = incl;
    const double left = __shfl_up(incl, 1, 64);
    __syncthreads();
    double base = 0.0, total = 0.0;
#pragma unroll
    for (int w = 0; w < SAMP_THREADS / 64; ++w) {
      const double x = sums[w];
      base += w < wave ? x : 0.0;
      total += x;
    }
    if (lane > 0) base += left;
    // Slots are in index order: a wave's first entry past the draw and its last entry at all speak for it (an LDS atomic for every entry, on
    // one address, took 3 us where thousands are kept).
    int pick = -1, kept = -1;
#pragma unroll
    for (int j = SLOTS - 1; j >= 0; --j)
      if (in[j]) {
        if (kept < 0) kept = (int)slot[j].y;
        if (base + upto[j] > (double)sr.uniform * total) pick = (int)slot[j].y;
      }
    const u64_t picks = __ballot(pick >= 0), keeps = __ballot(kept >= 0);
    if (picks != 0 && lane == __ffsll((unsigned long long)picks) - 1) atomicMin(&s_pick, pick);
    if (keeps != 0 && lane == 63 - __clzll((long long)keeps)) atomicMax(&s_last, kept);
    __syncthreads();
    if (tid == 0) ids[blockIdx.x] = s_pick != 0x7fffffff ? s_pick : max(s_last, 0);
    return;
  }
  if (few) {
    // the draw among the listed entries, in index order; sums in double, so that the list's order leaves no trace
    __syncthreads();
    const int n = (int)min(n_list, (unsigned)SB_SHORT), me = (int)threadIdx.x;
    const bool in = me < n && __uint_as_float(sm.list[me]) >= tau;
    const unsigned own = in ? sm.list[SB_SHORT + me] : 0u;
    double upto = 0.0, total = 0.0;
    if (wave * 64 < n)
      for (int j = 0; j < n; ++j) {
        const float p = __uint_as_float(sm.list[j]);
        const double q = p >= tau ? (double)p : 0.0;
        total += q;
        upto += sm.list[SB_SHORT + j] <= own ? q : 0.0;
      }
    if (in) {
      atomicMax(&s_last, (int)own);
      if (upto > (double)sr.uniform * total) atomicMin(&s_pick, (int)own);
    }
    __syncthreads();
    if (threadIdx.x == 0) ids[blockIdx.x] = s_pick != 0x7fffffff ? s_pick : max(s_last, 0);
    return;
  }
  __syncthreads();

  // kept mass per tile of 256 entries (one wave's load)
  const int tiles = (int)((vocab + SB_TILE - 1) / SB_TILE);
  for (int t0 = wave; t0 < tiles; t0 += 8 * (SAMP_THREADS / 64)) {
    Vec<float, 4> v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int t = t0 + u * (SAMP_THREADS / 64);
      if (t < tiles) v[u] = row4(row, vocab, (int64_t)t * 64 + lane, vec);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int t = t0 + u * (SAMP_THREADS / 64);
      if (t < tiles) {
        float part = 0.f;
        bool any = false;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          any |= v[u].v[j] >= tau;
          part += v[u].v[j] >= tau ? v[u].v[j] : 0.f;
        }
        if (__any(any)) part = wave_sum(part);
        if (lane == 0) sm.tile[t] = part;
      }
    }
  }
  __syncthreads();
  // exclusive sums over tiles, four tiles a thread
  float part[4], before[4], run = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int t = (int)threadIdx.x * 4 + j;
    part[j] = t < tiles ? sm.tile[t] : 0.f;
    before[j] = run;
    run += part[j];
  }
  float incl = run;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float up = __shfl_up(incl, o, 64);
    if (lane >= o) incl += up;
  }
  if (lane == 63) cs.wm[wave] = incl;
  const float left = __shfl_up(incl, 1, 64);
  __syncthreads();
  float base = 0.f, total = 0.f;
  for (int w = 0; w < SAMP_THREADS / 64; ++w) {
    if (w < wave) base += cs.wm[w];
    total += cs.wm[w];
  }
  if (lane > 0) base += left;
  const float target = sr.uniform * total;
  // the first tile whose running mass passes the target, and the last one with anything in it
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int t = (int)threadIdx.x * 4 + j;
    if (part[j] > 0.f) {
      atomicMax(&s_last, t);
      if (base + before[j] + part[j] > target) atomicMin(&s_tile, t);
    }
  }
  __syncthreads();
  const int hit = s_tile < SB_MAX_TILES ? s_tile : s_last;   // rounding at the very end of the CDF: the last kept entry
  if (hit >= 0 && (int)threadIdx.x == hit / 4) s_before = base + before[hit % 4];
  __syncthreads();
  if (wave != 0) return;
  if (hit < 0) {
    if (lane == 0) ids[blockIdx.x] = 0;
    return;
  }
  const Vec<float, 4> v = row4(row, vocab, (int64_t)hit * 64 + lane, vec);
  float own = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) own += v.v[j] >= tau ? v.v[j] : 0.f;
  float sum = own;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float up = __shfl_up(sum, o, 64);
    if (lane >= o) sum += up;
  }
  const float upto = __shfl_up(sum, 1, 64);
  float at = s_before + (lane > 0 ? upto : 0.f);
  int pick = 0x7fffffff, kept = -1;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (v.v[j] >= tau) {
      at += v.v[j];
      kept = hit * SB_TILE + lane * 4 + j;
      if (pick == 0x7fffffff && at > target) pick = kept;
    }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    pick = min(pick, __shfl_xor(pick, o, 64));
    kept = max(kept, __shfl_xor(kept, o, 64));
  }
  if (lane == 0) ids[blockIdx.x] = pick != 0x7fffffff ? pick : kept;
}

// Chunks of a row for `rows` rows: enough workgroups for every CU, at least 8 K entries each (below that a launch is all
// latency), at most 16.
static int row_chunks(int64_t rows, int64_t vocab) {
  const int64_t want = (256 + rows - 1) / rows;
  return (int)std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(want, MAX_CHUNKS), vocab / 8192));
}

}  // namespace mi355

using namespace mi355;



extern "C" {

int mi355_argmax(int64_t* ids, const float* logits, int64_t rows, int64_t vocab,
                 int64_t row_stride, void* stream) {
  MI355_REQUIRE(ids && logits, MI355_ERR_INVALID, "argmax: null pointer");
  MI355_REQUIRE(rows >= 0 && vocab > 0 && vocab < (1LL << 31) && row_stride >= vocab,
                MI355_ERR_INVALID, "argmax: bad shape");
  if (rows == 0) return MI355_OK;
  hipLaunchKernelGGL(argmax_kernel, dim3((unsigned)rows), dim3(SAMP_THREADS), 0,
                     (hipStream_t)stream, ids, logits, vocab, row_stride);
  MI355_CHECK_LAUNCH("argmax");
  return MI355_OK;
}

int64_t mi355_argmax_workspace_bytes(int64_t rows) { return rows > 0 ? rows * 16 : 0; }

int mi355_argmax_chunked(int64_t* ids, const float* logits, int64_t rows, int64_t vocab, int64_t row_stride,
                         void* workspace, int64_t workspace_bytes, void* stream) {
  MI355_REQUIRE(ids && logits, MI355_ERR_INVALID, "argmax_chunked: null pointer");
  MI355_REQUIRE(rows >= 0 && rows <= 65535 && vocab > 0 && vocab < (1LL << 31) - 1 && row_stride >= vocab, MI355_ERR_INVALID,
                "argmax_chunked: bad shape");
  if (rows == 0) return MI355_OK;
  // enough workgroups for every CU; a chunk keeps at least 16 K elements
  int64_t chunks = (256 + rows - 1) / rows;
  chunks = std::min<int64_t>(chunks, std::max<int64_t>(1, vocab / 16384));
  chunks = std::min<int64_t>(chunks, 16);
  if (chunks <= 1 || !workspace) {
    hipLaunchKernelGGL(argmax_kernel, dim3((unsigned)rows), dim3(SAMP_THREADS), 0, (hipStream_t)stream, ids, logits, vocab,
                       row_stride);
  } else {
    MI355_REQUIRE(workspace_bytes >= mi355_argmax_workspace_bytes(rows) && (reinterpret_cast<uintptr_t>(workspace) & 7) == 0,
                  MI355_ERR_INVALID, "argmax_chunked: workspace of %lld bytes (8-byte aligned, zeroed) required",
                  (long long)mi355_argmax_workspace_bytes(rows));
    unsigned long long* cells = static_cast<unsigned long long*>(workspace);
    unsigned* tickets = reinterpret_cast<unsigned*>(cells + rows);
    hipLaunchKernelGGL(argmax_chunk_kernel, dim3((unsigned)rows, (unsigned)chunks), dim3(SAMP_THREADS), 0,
                       (hipStream_t)stream, ids, logits, vocab, row_stride, cells, tickets);
  }
  MI355_CHECK_LAUNCH("argmax_chunked");
  return MI355_OK;
}

int mi355_softmax_temperature(float* logits, const float* temperatures, int64_t rows,
                              int64_t vocab, int64_t row_stride, void* stream) {
  MI355_REQUIRE(logits && temperatures, MI355_ERR_INVALID, "softmax_temperature: null pointer");
  MI355_REQUIRE(rows >= 0 && vocab > 0 && row_stride >= vocab, MI355_ERR_INVALID,
                "softmax_temperature: bad shape");
  if (rows == 0) return MI355_OK;
  hipLaunchKernelGGL(softmax_temperature_kernel, dim3((unsigned)rows), dim3(SAMP_THREADS), 0,
                     (hipStream_t)stream, logits, temperatures, vocab, row_stride);
  MI355_CHECK_LAUNCH("softmax_temperature");
  return MI355_OK;
}

int64_t mi355_sampling_workspace_bytes(int64_t rows, int64_t vocab) {
  if (rows <= 0 || vocab <= 0) return 0;
  return rows * row_chunks(rows, vocab) * (SB_BINS * (int64_t)sizeof(u64_t) + (int64_t)(sizeof(ChunkTop) + sizeof(float2))) +
         rows * SB_TOP * (int64_t)sizeof(uint2);
}

int mi355_softmax_temperature_split(float* logits, const float* temperatures, int64_t rows, int64_t vocab, int64_t row_stride,
                                    void* workspace, int64_t workspace_bytes, void* stream) {
  MI355_REQUIRE(logits && temperatures, MI355_ERR_INVALID, "softmax_temperature_split: null pointer");
  MI355_REQUIRE(rows >= 0 && vocab > 0 && row_stride >= vocab, MI355_ERR_INVALID, "softmax_temperature_split: bad shape");
  const int chunks = rows > 0 ? row_chunks(rows, vocab) : 1;
  if (chunks <= 1 || !workspace) return mi355_softmax_temperature(logits, temperatures, rows, vocab, row_stride, stream);
  MI355_REQUIRE(workspace_bytes >= rows * chunks * (int64_t)sizeof(float2) && (reinterpret_cast<uintptr_t>(workspace) & 7) == 0,
                MI355_ERR_INVALID, "softmax_temperature_split: workspace of %lld bytes (8-byte aligned) required",
                (long long)mi355_sampling_workspace_bytes(rows, vocab));
  float2* partials = static_cast<float2*>(workspace);
  hipLaunchKernelGGL(softmax_partials_kernel, dim3((unsigned)rows, chunks), dim3(SAMP_THREADS), 0, (hipStream_t)stream, partials,
                     logits, temperatures, vocab, row_stride);
  hipLaunchKernelGGL((sample_chunk_kernel<true, false>), dim3((unsigned)rows, chunks), dim3(SAMP_THREADS), 0, (hipStream_t)stream, logits,
                     partials, temperatures, (const int32_t*)nullptr, (const float*)nullptr, (u64_t*)nullptr, (uint2*)nullptr, (ChunkTop*)nullptr, vocab, row_stride);
  MI355_CHECK_LAUNCH("softmax_temperature_split");
  return MI355_OK;
}

int mi355_top_k_top_p_min_p_sample(int32_t* ids, const float* probs, const int32_t* top_ks,
                                   const float* top_ps, const float* min_ps, const float* uniform,
                                   int64_t rows, int64_t vocab, int64_t row_stride, void* stream) {
  MI355_REQUIRE(ids && probs && uniform, MI355_ERR_INVALID, "top_k_top_p_min_p_sample: null pointer");
  MI355_REQUIRE(rows >= 0 && vocab > 0 && vocab < (1LL << 31) && row_stride >= vocab,
                MI355_ERR_INVALID, "top_k_top_p_min_p_sample: bad shape");
  if (rows == 0) return MI355_OK;
  hipLaunchKernelGGL(topk_topp_minp_sample_kernel, dim3((unsigned)rows), dim3(SAMP_THREADS), 0,
                     (hipStream_t)stream, ids, probs, top_ks, top_ps, min_ps, uniform, vocab,
                     row_stride);
  MI355_CHECK_LAUNCH("top_k_top_p_min_p_sample");
  return MI355_OK;
}

// Launches 1 (unless `fused`: with softmax_temperature's second one) and 2 of the draw over chunks.
static int sample_launches(int32_t* ids, float* data, const float* temperatures, const int32_t* top_ks, const float* top_ps, const float* min_ps,
                           const float* uniform, int64_t rows, int64_t vocab, int64_t row_stride, bool fused, void* workspace,
                           hipStream_t stream) {
  const int chunks = row_chunks(rows, vocab);
  const int64_t parts = rows * chunks;
  u64_t* bins = static_cast<u64_t*>(workspace);
  uint2* lists = reinterpret_cast<uint2*>(bins + parts * SB_BINS);
  ChunkTop* tops = reinterpret_cast<ChunkTop*>(lists + rows * SB_TOP);
  float2* partials = reinterpret_cast<float2*>(tops + parts);
  const dim3 grid((unsigned)rows, chunks), block(SAMP_THREADS);
  if (fused) {
    hipLaunchKernelGGL(softmax_partials_kernel, grid, block, 0, stream, partials, data, temperatures, vocab, row_stride);
    hipLaunchKernelGGL((sample_chunk_kernel<true, true>), grid, block, 0, stream, data, partials, temperatures, top_ks, top_ps, bins, lists, tops, vocab,
                       row_stride);
  } else {
    hipLaunchKernelGGL((sample_chunk_kernel<false, true>), grid, block, 0, stream, data, (const float2*)nullptr, (const float*)nullptr, top_ks, top_ps,
                       bins, lists, tops, vocab, row_stride);
  }
  hipLaunchKernelGGL(sample_pick_kernel, dim3((unsigned)rows), block, 0, stream, ids, bins, lists, tops, chunks, data, top_ks, top_ps, min_ps,
                     uniform, vocab, row_stride);
  MI355_CHECK_LAUNCH("top_k_top_p_min_p_sample_split");
  return MI355_OK;
}

int mi355_top_k_top_p_min_p_sample_split(int32_t* ids, const float* probs, const int32_t* top_ks, const float* top_ps,
                                         const float* min_ps, const float* uniform, int64_t rows, int64_t vocab,
                                         int64_t row_stride, void* workspace, int64_t workspace_bytes, void* stream) {
  // a short row is two launches' latency for nothing; a vocabulary past the tiles' table does not exist
  if (!workspace || rows <= 0 || vocab < 4096 || vocab > SB_MAX_VOCAB)
    return mi355_top_k_top_p_min_p_sample(ids, probs, top_ks, top_ps, min_ps, uniform, rows, vocab, row_stride, stream);
  MI355_REQUIRE(ids && probs && uniform, MI355_ERR_INVALID, "top_k_top_p_min_p_sample_split: null pointer");
  MI355_REQUIRE(row_stride >= vocab, MI355_ERR_INVALID, "top_k_top_p_min_p_sample_split: bad shape");
  const int64_t need = mi355_sampling_workspace_bytes(rows, vocab);
  MI355_REQUIRE(workspace_bytes >= need && (reinterpret_cast<uintptr_t>(workspace) & 7) == 0, MI355_ERR_INVALID,
                "top_k_top_p_min_p_sample_split: workspace of %lld bytes (8-byte aligned) required", (long long)need);
  return sample_launches(ids, const_cast<float*>(probs), nullptr, top_ks, top_ps, min_ps, uniform, rows, vocab, row_stride, false, workspace,
                         (hipStream_t)stream);
}

int mi355_softmax_sample_split(int32_t* ids, float* logits, const float* temperatures, const int32_t* top_ks, const float* top_ps,
                               const float* min_ps, const float* uniform, int64_t rows, int64_t vocab, int64_t row_stride, void* workspace,
                               int64_t workspace_bytes, void* stream) {
  MI355_REQUIRE(ids && logits && temperatures && uniform, MI355_ERR_INVALID, "softmax_sample_split: null pointer");
  MI355_REQUIRE(rows >= 0 && vocab > 0 && row_stride >= vocab, MI355_ERR_INVALID, "softmax_sample_split: bad shape");
  if (!workspace || rows == 0 || vocab < 4096 || vocab > SB_MAX_VOCAB || row_chunks(rows, vocab) <= 1) {
    const int rc = mi355_softmax_temperature_split(logits, temperatures, rows, vocab, row_stride, workspace, workspace_bytes, stream);
    if (rc != MI355_OK) return rc;
    return mi355_top_k_top_p_min_p_sample_split(ids, logits, top_ks, top_ps, min_ps, uniform, rows, vocab, row_stride, workspace,
                                                workspace_bytes, stream);
  }
  const int64_t need = mi355_sampling_workspace_bytes(rows, vocab);
  MI355_REQUIRE(workspace_bytes >= need && (reinterpret_cast<uintptr_t>(workspace) & 7) == 0, MI355_ERR_INVALID,
                "softmax_sample_split: workspace of %lld bytes (8-byte aligned) required", (long long)need);
  return sample_launches(ids, logits, temperatures, top_ks, top_ps, min_ps, uniform, rows, vocab, row_stride, true, workspace,
                         (hipStream_t)stream);
}

}  // extern "C"
