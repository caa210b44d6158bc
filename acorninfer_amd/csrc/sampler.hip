// Token sampler: temperature -> top-k -> top-p -> draw. Long rows (a language
// model's vocabulary) are split over kSplitG workgroups in four launches
// (sample_*_kernel below); short and very long rows, calls without a workspace and
// rows whose maximum / T overflows run as one workgroup per row (sample_row).
//
// Semantics follow acorninfer/sampler.py:38-68 (HF warper order):
//   x = logits / T                                   (fp32)
//   top-k: remove x < kth-largest(x)                 (ties with the kth are kept)
//   top-p: over the kept x sorted ascending (stable), cum = cumsum(softmax);
//          remove where cum <= 1 - p, always keep the largest
//   draw : token with probability softmax(x)[kept] (inverse CDF of a given
//          uniform u over the kept tokens in vocabulary order); logprob is the
//          log-softmax of the processed logits at the token.
// temperature == 0 means greedy (argmax, logprob 0), as Executor._sample
// routes it (engine/executor.py:128-138).
//
// One workgroup per row: the row is never sorted. Keys are the order-preserving uint32 image
// of fp32. top-k is a 4-pass radix select (8-bit digits, MSB first) with
// count histograms; top-p is the same descent over the softmax mass, with
// masses accumulated as 2^-40 fixed-point integers so that the LDS atomics
// are order independent (deterministic). The tie group at the top-p boundary
// is resolved in the stable ascending order HF sorts in: among equal values
// the higher vocabulary index is nearer the top.
#include <algorithm>

#include "common.h"

using namespace acorn;

namespace {

constexpr int kNT = 1024;
constexpr double kFix = 1099511627776.0;  // 2^40

typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
typedef uint16_t u16x2v __attribute__((ext_vector_type(2)));

// Element e of a 16-byte vector of T as float.
template <typename T> __device__ __forceinline__ float word_elem(const u32x4v& w, int e);
template <> __device__ __forceinline__ float word_elem<__bf16>(const u32x4v& w, int e) {
  return (e & 1) ? bf16_hi(w[e / 2]) : bf16_lo(w[e / 2]);
}
template <> __device__ __forceinline__ float word_elem<_Float16>(const u32x4v& w, int e) {
  const uint32_t v = w[e / 2];
  return (float)__builtin_bit_cast(_Float16, (uint16_t)((e & 1) ? v >> 16 : v & 0xffffu));
}
template <> __device__ __forceinline__ float word_elem<float>(const u32x4v& w, int e) {
  return __uint_as_float(w[e]);
}

// Exponent fields of a 16-byte vector folded into a running unsigned max
// (per 16-bit half for the half types): a field of all ones, i.e. an inf or
// NaN somewhere, survives as the maximum.
template <typename T> struct ExpBits;
template <> struct ExpBits<__bf16> { static constexpr uint32_t kMask = 0x7F807F80u; };
template <> struct ExpBits<_Float16> { static constexpr uint32_t kMask = 0x7C007C00u; };
template <> struct ExpBits<float> { static constexpr uint32_t kMask = 0x7F800000u; };
template <typename T> __device__ __forceinline__ uint32_t fold_exp(uint32_t acc, const u32x4v& w) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t x = w[i] & ExpBits<T>::kMask;
    if constexpr (sizeof(T) == 2)
      acc = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(
                                             __builtin_bit_cast(u16x2v, acc),
                                             __builtin_bit_cast(u16x2v, x)));
    else
      acc = max(acc, x);
  }
  return acc;
}
template <typename T> __device__ __forceinline__ bool exp_all_ones(uint32_t acc) {
  constexpr uint32_t m = ExpBits<T>::kMask;
  if constexpr (sizeof(T) == 2)
    return (acc & 0xffffu) == (m & 0xffffu) || (acc >> 16) == (m >> 16);
  else
    return acc == m;
}

__device__ __forceinline__ uint32_t okey(float x) {
  const uint32_t u = __float_as_uint(x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Block-wide exclusive scan of one float per thread (fixed order).
__device__ float block_exclusive_scan(float v, float* buf, float* total) {
  buf[threadIdx.x] = v;
  __syncthreads();
  for (int off = 1; off < kNT; off <<= 1) {
    const float add = threadIdx.x >= off ? buf[threadIdx.x - off] : 0.f;
    __syncthreads();
    buf[threadIdx.x] += add;
    __syncthreads();
  }
  const float incl = buf[threadIdx.x];
  *total = buf[kNT - 1];
  __syncthreads();
  return incl - v;
}

__device__ uint32_t block_exclusive_scan_u32(uint32_t v, uint32_t* buf, uint32_t* total) {
  buf[threadIdx.x] = v;
  __syncthreads();
  for (int off = 1; off < kNT; off <<= 1) {
    const uint32_t add = threadIdx.x >= off ? buf[threadIdx.x - off] : 0u;
    __syncthreads();
    buf[threadIdx.x] += add;
    __syncthreads();
  }
  const uint32_t incl = buf[threadIdx.x];
  *total = buf[kNT - 1];
  __syncthreads();
  return incl - v;
}

// This thread's share of a scan of p[0, n): its maximum `bv` (first index `bi`
// on ties) and whether it saw a NaN or an infinity. 16-byte vectors, kUnroll
// of them in flight per thread (for one workgroup a 151936-entry bf16 row is
// two rounds of requests); a scalar tail. Vector indices past the end re-read
// the last vector (unconditional loads keep the wait counts static) and are
// not visited.
// The per-element work is what bounds a workgroup that reads a whole row: per
// vector only its maximum is compared with the running one (the vector index
// of the first strict improvement is kept) and the exponent fields are folded
// into an integer max for the finiteness test. After the loop the kept vector
// is read again and its first element equal to the maximum taken: the
// thread's first maximum in index order, as an element-by-element scan would
// find.
template <typename T, int NT, int kUnroll>
__device__ __forceinline__ void scan_max(const T* p, int64_t n, float& bv, int64_t& bi,
                                         bool& bad) {
  const int tid = threadIdx.x;
  bv = -INFINITY;
  bi = INT64_MAX;
  bad = false;
  auto visit = [&](float l, int64_t i) {
    if (!(l == l) || l == INFINITY || l == -INFINITY) bad = true;
    if (l > bv || (l == bv && i < bi)) {
      bv = l;
      bi = i;
    }
  };
  constexpr int E = 16 / sizeof(T);                 // elements per vector
  const bool aligned = ((uintptr_t)p % 16) == 0;
  const int64_t nvec = aligned ? n / E : 0;
  const u32x4v* rv = (const u32x4v*)p;
  float vbest = -INFINITY;
  int64_t jbest = -1;
  uint32_t emax = 0;
  for (int64_t j0 = tid; j0 < nvec; j0 += (int64_t)NT * kUnroll) {
    u32x4v buf[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) buf[u] = rv[min(j0 + (int64_t)u * NT, nvec - 1)];
    // (the empty asm keeps every load ahead of the guarded uses below;
    // a load sunk into a guarded block is waited for on its own)
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) asm volatile("" ::"v"(buf[u]));
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int64_t j = j0 + (int64_t)u * NT;
      if (j < nvec) {
        float vm = word_elem<T>(buf[u], 0);
#pragma unroll
        for (int e = 1; e < E; ++e) vm = fmaxf(vm, word_elem<T>(buf[u], e));
        emax = fold_exp<T>(emax, buf[u]);
        if (vm > vbest) {
          vbest = vm;
          jbest = j;
        }
      }
    }
  }
  if (exp_all_ones<T>(emax)) bad = true;
  if (jbest >= 0) {
    const u32x4v w = rv[jbest];
    int ebest = E - 1;
#pragma unroll
    for (int e = E - 2; e >= 0; --e) ebest = word_elem<T>(w, e) == vbest ? e : ebest;
    bv = vbest;
    bi = jbest * E + ebest;
  }
  for (int64_t i = nvec * E + tid; i < n; i += NT) visit(to_f32(p[i]), i);
}

// The wave's first maximum in every lane.
__device__ __forceinline__ void wave_first_max(float& bv, int64_t& bi) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(bv, o);
    const int64_t oi = __shfl_xor(bi, o);
    if (ov > bv || (ov == bv && oi < bi)) {
      bv = ov;
      bi = oi;
    }
  }
}

// exp(x - M) as 2^-40 fixed point (sums of it do not depend on their order).
__device__ __forceinline__ unsigned long long mass_fix(float x, float M) {
  return (unsigned long long)((double)exp2f((x - M) * 1.4426950408889634f) * kFix);
}

// One row on one workgroup of kNT threads.
template <typename T>
__device__ void sample_row(
    const int64_t r, const T* __restrict__ logits, int64_t V,
    const float* __restrict__ temperature, const int32_t* __restrict__ top_k,
    const float* __restrict__ top_p, const float* __restrict__ uniform,
    int64_t* __restrict__ token, float* __restrict__ logprob, float* __restrict__ processed,
    int32_t* __restrict__ status) {
  __shared__ uint32_t hcnt[256];
  __shared__ unsigned long long hmass[256];
  __shared__ float sbuf[kNT];
  __shared__ uint32_t ubuf[kNT];
  __shared__ float red_f[kNT / kWave];
  __shared__ int64_t red_i[kNT / kWave];
  __shared__ uint32_t sh_u32[8];
  __shared__ unsigned long long sh_u64[4];
  __shared__ float sh_f[4];
  __shared__ int sh_bad;

  const T* row = logits + r * V;
  const float Tm = temperature[r];
  const int tid = threadIdx.x, lane = tid % kWave, wid = tid / kWave;
  if (tid == 0) sh_bad = 0;
  __syncthreads();

  // ---- pass 1: max (first index on ties), finiteness --------------------
  float bv;
  int64_t bi;
  bool bad;
  scan_max<T, kNT, 10>(row, V, bv, bi, bad);
  if (bad) sh_bad = 1;  // benign race: every writer stores 1
  wave_first_max(bv, bi);
  if (lane == 0) {
    red_f[wid] = bv;
    red_i[wid] = bi;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < kNT / kWave; ++w)
      if (red_f[w] > bv || (red_f[w] == bv && red_i[w] < bi)) {
        bv = red_f[w];
        bi = red_i[w];
      }
    red_f[0] = bv;
    red_i[0] = bi;
  }
  __syncthreads();
  const float lmax = red_f[0];
  const int64_t imax = red_i[0];
  if (sh_bad) {
    if (tid == 0) {
      status[r] = 1;
      token[r] = imax == INT64_MAX ? 0 : imax;
      logprob[r] = NAN;
    }
    return;
  }
  if (!(Tm > 0.f)) {  // greedy
    if (tid == 0) {
      status[r] = 0;
      token[r] = imax;
      logprob[r] = 0.f;
    }
    if (processed)
      for (int64_t i = tid; i < V; i += kNT) processed[r * V + i] = to_f32(row[i]);
    return;
  }
  const float M = lmax / Tm;  // max of x (division is monotone for T > 0)

  // ---- top-k: kth largest key by radix select on counts -------------------
  const int64_t kk = top_k[r];
  uint32_t kkey = 0;  // keep key >= kkey
  if (kk > 0 && kk < V) {
    uint32_t prefix = 0, pmask = 0;
    uint32_t remaining = (uint32_t)kk;
    for (int shift = 24; shift >= 0; shift -= 8) {
      for (int b = tid; b < 256; b += kNT) hcnt[b] = 0;
      __syncthreads();
      for (int64_t i = tid; i < V; i += kNT) {
        const uint32_t key = okey(to_f32(row[i]) / Tm);
        if ((key & pmask) == prefix) atomicAdd(&hcnt[(key >> shift) & 255u], 1u);
      }
      __syncthreads();
      if (tid == 0) {
        uint32_t acc = 0;
        int d = 255;
        for (; d > 0; --d) {
          if (acc + hcnt[d] >= remaining) break;
          acc += hcnt[d];
        }
        sh_u32[0] = (uint32_t)d;
        sh_u32[1] = remaining - acc;
      }
      __syncthreads();
      prefix |= sh_u32[0] << shift;
      pmask |= 255u << shift;
      remaining = sh_u32[1];
      __syncthreads();
    }
    kkey = prefix;
  }

  // ---- mass of the top-k set: Z = sum exp(x - M) over key >= kkey ---------
  // (fixed-point, order independent)
  auto wfix = [&](float x) { return mass_fix(x, M); };
  unsigned long long zl = 0;
  for (int64_t i = tid; i < V; i += kNT) {
    const float x = to_f32(row[i]) / Tm;
    if (okey(x) >= kkey) zl += wfix(x);
  }
  if (tid == 0) sh_u64[0] = 0;
  __syncthreads();
  atomicAdd(&sh_u64[0], zl);
  __syncthreads();
  const unsigned long long Zk = sh_u64[0];

  // ---- top-p: descend on mass to the boundary key --------------------------
  const float pp = top_p[r];
  uint32_t pkey = kkey;           // keep key > pkey, plus n_keep of the ties at pkey
  uint32_t tie_keep = 0xffffffffu;  // all ties kept unless reduced below
  bool ptie = false;
  if (pp < 1.0f) {
    const unsigned long long target = (unsigned long long)((double)pp * (double)Zk);
    uint32_t prefix = 0, pmask = 0;
    unsigned long long above = 0;
    uint32_t tie_cnt = 0;
    unsigned long long tie_mass = 0;
    for (int shift = 24; shift >= 0; shift -= 8) {
      for (int b = tid; b < 256; b += kNT) {
        hmass[b] = 0;
        hcnt[b] = 0;
      }
      __syncthreads();
      for (int64_t i = tid; i < V; i += kNT) {
        const float x = to_f32(row[i]) / Tm;
        const uint32_t key = okey(x);
        if (key >= kkey && (key & pmask) == prefix) {
          atomicAdd(&hmass[(key >> shift) & 255u], wfix(x));
          atomicAdd(&hcnt[(key >> shift) & 255u], 1u);
        }
      }
      __syncthreads();
      if (tid == 0) {
        unsigned long long acc = above;
        int d = 255;
        for (; d > 0; --d) {
          if (hcnt[d] && acc + hmass[d] >= target) break;
          acc += hmass[d];
        }
        // d == 0 is the last candidate bin
        sh_u32[0] = (uint32_t)d;
        sh_u64[1] = acc;
        sh_u32[2] = hcnt[d];
        sh_u64[2] = hmass[d];
      }
      __syncthreads();
      prefix |= sh_u32[0] << shift;
      pmask |= 255u << shift;
      above = sh_u64[1];
      tie_cnt = sh_u32[2];
      tie_mass = sh_u64[2];
      __syncthreads();
    }
    // tokens strictly above `prefix` hold mass `above` < target; the tie
    // group at `prefix` (tie_cnt tokens, equal mass q each) is kept while
    // above + r*q < target, r counted from the highest index down.
    pkey = prefix;
    if (tie_cnt > 0) {
      const double q = (double)tie_mass / (double)tie_cnt;
      uint32_t nk = 1;
      if (q > 0.0) {
        const double t = ((double)target - (double)above) / q;
        nk = (uint32_t)std::min<double>((double)tie_cnt, std::max(1.0, ceil(t)));
      } else {
        nk = tie_cnt;
      }
      if (nk < tie_cnt) {
        tie_keep = nk;
        ptie = true;
      }
    }
  }

  // ---- final keep rule, per contiguous segment (vocabulary order) -------
  const int64_t seg = (V + kNT - 1) / kNT;
  const int64_t s0 = std::min<int64_t>((int64_t)tid * seg, V);
  const int64_t s1 = std::min<int64_t>(s0 + seg, V);
  // ties at pkey: rank from the highest index (only needed when partially kept)
  uint32_t ties_after = 0;
  if (ptie) {
    uint32_t mine = 0;
    for (int64_t i = s0; i < s1; ++i)
      if (okey(to_f32(row[i]) / Tm) == pkey) ++mine;
    // exclusive scan from the end: ties in segments after mine
    uint32_t tot;
    const uint32_t before = block_exclusive_scan_u32(mine, ubuf, &tot);
    ties_after = tot - before - mine;
  }
  const bool use_p = pp < 1.0f;
  auto kept_at = [&](float x, uint32_t& tie_rank_from_end) -> bool {
    const uint32_t key = okey(x);
    if (key < kkey) return false;
    if (!use_p) return true;
    if (key > pkey) return true;
    if (key < pkey) return false;
    if (!ptie) return true;
    return tie_rank_from_end < tie_keep;
  };

  // segment mass (fp32, vocabulary order) for the inverse CDF
  float segm = 0.f;
  {
    uint32_t rank = ties_after;
    // walk backward to know each tie's rank from the end
    for (int64_t i = s1 - 1; i >= s0; --i) {
      const float x = to_f32(row[i]) / Tm;
      uint32_t rk = rank;
      const bool tie = okey(x) == pkey;
      if (kept_at(x, rk)) segm += exp2f((x - M) * 1.4426950408889634f);
      if (tie) ++rank;
    }
  }
  float Zf;
  const float before = block_exclusive_scan(segm, sbuf, &Zf);
  const float target = uniform[r] * Zf;
  // the segment where the running mass first exceeds the target
  if (tid == 0) {
    sh_u32[3] = 0xffffffffu;
    sh_f[0] = 0.f;
  }
  __syncthreads();
  if (segm > 0.f && before <= target && target < before + segm) atomicMin(&sh_u32[3], (uint32_t)tid);
  __syncthreads();
  uint32_t owner = sh_u32[3];
  if (owner == 0xffffffffu) {
    // rounding put the target at the very end: the last segment with mass
    if (tid == 0) sh_u32[4] = 0;
    __syncthreads();
    if (segm > 0.f) atomicMax(&sh_u32[4], (uint32_t)tid);
    __syncthreads();
    owner = sh_u32[4];
  }
  if ((uint32_t)tid == owner) {
    // forward walk; tie ranks from the end need the segment's tie total
    uint32_t seg_ties = 0;
    if (ptie)
      for (int64_t i = s0; i < s1; ++i)
        if (okey(to_f32(row[i]) / Tm) == pkey) ++seg_ties;
    uint32_t ties_seen = 0;
    float run = before;
    int64_t pick = -1, last_kept = -1;
    for (int64_t i = s0; i < s1; ++i) {
      const float x = to_f32(row[i]) / Tm;
      const bool tie = okey(x) == pkey;
      uint32_t rk = ties_after + (seg_ties - ties_seen - (tie ? 1u : 0u));
      if (kept_at(x, rk)) {
        run += exp2f((x - M) * 1.4426950408889634f);
        last_kept = i;
        if (run > target) {
          pick = i;
          break;
        }
      }
      if (tie) ++ties_seen;
    }
    if (pick < 0) pick = last_kept;
    const float xt = to_f32(row[pick]) / Tm;
    token[r] = pick;
    logprob[r] = (xt - M) - logf(Zf);
    status[r] = 0;
  }
  if (processed) {
    uint32_t rank = ties_after;
    for (int64_t i = s1 - 1; i >= s0; --i) {
      const float x = to_f32(row[i]) / Tm;
      uint32_t rk = rank;
      const bool tie = okey(x) == pkey;
      processed[r * V + i] = kept_at(x, rk) ? x : -INFINITY;
      if (tie) ++rank;
    }
  }
}

// ---- long rows: kSplitG workgroups per row --------------------------------
//
// One workgroup per row leaves all but `rows` CUs idle and walks the row about
// ten times, an IEEE division and often an LDS atomic per element each time:
// 464 us for 8 rows of 151936 (2.4 MB) at T 0.6, top-k 20, top-p 0.95. Here a
// row is kSplitG chunks of consecutive elements and each launch reads a chunk
// once:
//   stats   chunk maxima and finiteness; clears the row's histogram
//   hist    histogram of the row over kSplitNB bins of 1/64 in x = logit / T
//           below the maximum: counts (top-k) or fixed-point mass (top-p);
//           with neither, the chunk's mass. Top-k also lists the chunk's own
//           first k elements, in vocabulary order. Greedy and non-finite rows
//           end here
//   gather  the boundary bin, from the histogram; the elements that may lie on
//           the boundary (top-p: those in it; top-k, only where some chunk's
//           first k overflowed its list: all down to it) listed per chunk, and
//           the chunk's mass above it
//   pick    one workgroup per row ranks the listed elements by counting, which
//           gives the kept set, finds the drawn chunk from the chunks' masses
//           and the token inside it
// The selection is sample_row's, bit for bit: the same keys and the same
// integer masses relative to the row's maximum. A bin is a monotone function
// of x, so bins respect the key order. The draw adds integer masses instead of
// fp32 ones. Where the boundary holds more elements than the lists (a large top-k,
// many ties, a flat row) pick goes down the keys instead (split_descend).
// Four launches of a few microseconds each, bound by their latency: 27.3 us.
constexpr int kSplitG = 32;          // workgroups (chunks) per row
constexpr int kSplitNT = 1024;       // their threads
constexpr int kSplitNB = 2048;       // histogram bins: 32 in x, the last takes the rest
constexpr float kSplitScale = 64.f;  // bins per unit of x
constexpr int kSplitCapC = 64;       // listed elements per chunk (one wave)
constexpr int kSplitCap = kNT;       // listed elements per row (one per thread of `pick`)
// shorter rows: one workgroup reads them in less than four launches take
constexpr int64_t kSplitMinV = 16384;
// More rows: the stats of several chunks per workgroup, so that they stay one round
// of workgroups (two per CU), and chunks of `hist` and `gather` on 256 threads, whose
// dispatch is a quarter of the time (rows with nothing left to do, the greedy ones,
// cost no more than that). us at 64 rows of 151936, 1024 threads and a chunk each /
// this, one workgroup per row: greedy 36 / 15.6, 11.0; T 1 68 / 39, 170; top-p 0.9
// 160 / 114, 555; top-k 20 + top-p 93 / 57, 579. At 8 rows greedy takes 11.5, 10.7 on
// one workgroup; 64 greedy rows of 16384 14.4, 7.9 there, sampled 26 to 67, 30 to 138.
constexpr int64_t kSplitWGs = 512;
constexpr int64_t kSplitWideRows = 8;
constexpr int kSplitFewNT = 256;
constexpr int64_t kSplitMaxRows = 4096;  // bounds the workspace (34 KB per row)
// masses of at most 2^40 each add up in 64 bits
constexpr int64_t kSplitMaxV = (int64_t)1 << 23;

enum { kRowDrawn = 0, kRowBad = 1, kRowGreedy = 2, kRowWhole = 3 };
enum { kModeTopK = 0, kModeTopP = 1, kModeAll = 2 };

struct alignas(64) SplitRow {
  unsigned long long hist[kSplitNB];  // counts (top-k) or masses (top-p)
  uint32_t ckey[kSplitG * kSplitCapC];
  uint32_t cidx[kSplitG * kSplitCapC];
  unsigned long long hard[kSplitG];   // mass of the chunk's elements above the boundary bin
  float cmax[kSplitG];
  uint32_t cimax[kSplitG];
  uint32_t cbad[kSplitG];
  uint32_t lcnt[kSplitG];             // top-k: listed by `hist` (up to kSplitCapC), and ...
  uint32_t ccnt[kSplitG];             // ... by `gather`
  unsigned long long zk, above;       // top-p: the row's mass, and that above the boundary bin
  uint32_t state, pkey, tie0;         // kept: key > pkey, or key == pkey and index >= tie0
};

struct SplitArgs {
  const void* logits;
  int64_t V;
  const float* temperature;
  const int32_t* top_k;
  const float* top_p;
  const float* uniform;
  int64_t* token;
  float* logprob;
  float* processed;
  int32_t* status;
  SplitRow* ws;
};

__device__ __forceinline__ int64_t split_chunk(int64_t V) {
  return ((V + kSplitG - 1) / kSplitG + 7) & ~(int64_t)7;
}
__device__ __forceinline__ int split_mode(const SplitArgs& a, int64_t r) {
  const int64_t kk = a.top_k[r];
  if (kk > 0 && kk < a.V) return kModeTopK;
  return a.top_p[r] < 1.0f ? kModeTopP : kModeAll;
}
__device__ __forceinline__ int split_bin(float x, float M) {
  return (int)fminf((M - x) * kSplitScale, (float)(kSplitNB - 1));
}
__device__ __forceinline__ float key_float(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? k & 0x7fffffffu : ~k);
}

// The row's maximum (first index) and finiteness from its chunks', in every lane.
__device__ __forceinline__ bool split_stats(const SplitRow& w, float& lmax, int64_t& imax) {
  const int c = threadIdx.x % kSplitG;
  lmax = w.cmax[c];
  imax = w.cimax[c] == 0xffffffffu ? INT64_MAX : (int64_t)w.cimax[c];
  const bool bad = __any(w.cbad[c] != 0);
  wave_first_max(lmax, imax);
  return bad;
}

// Elements i .. i + 7 of a row as floats (clamped to end - 1).
template <typename T>
__device__ __forceinline__ void load8(const T* row, int64_t i, int64_t end, bool aligned,
                                      float (&v)[8]) {
  if (aligned && i + 8 <= end) {
    constexpr int E = 16 / sizeof(T);
    u32x4v w[8 / E];
#pragma unroll
    for (int q = 0; q < 8 / E; ++q) w[q] = ((const u32x4v*)(row + i))[q];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = word_elem<T>(w[e / E], e % E);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = to_f32(row[min(i + e, end - 1)]);
  }
}

// Elements [c0, c1) of a row in groups of eight, U of a thread's groups requested
// together. Rows whose groups are whole and 16-byte aligned (V % 8 == 0) are read
// as vectors, clamped to the last one so that every load is unconditional; others
// element by element.
template <typename T, int U = 1>
struct Octets {
  static constexpr int E = 16 / sizeof(T), Q = 8 / E;
  const T* row;
  int64_t c0, c1, n;                    // the range and its groups
  bool fast;
  u32x4v w[U][Q];
  __device__ Octets(const T* row_, int64_t V, int64_t c0_, int64_t c1_)
      : row(row_), c0(c0_), c1(c1_), n((c1_ - c0_ + 7) / 8),
        fast(((uintptr_t)row_ % 16) == 0 && V % 8 == 0) {}
  // request groups j0, j0 + stride, ... (U of them)
  __device__ __forceinline__ void load(int64_t j0, int64_t stride) {
    if (!fast || n == 0) return;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < Q; ++q)
        w[u][q] = ((const u32x4v*)(row + c0 + min(j0 + u * stride, n - 1) * 8))[q];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < Q; ++q) asm volatile("" ::"v"(w[u][q]));
  }
  // f(index, value) of the groups j0, j0 + stride, ... < end; the first U have
  // been requested by load(j0, stride)
  template <typename F>
  __device__ __forceinline__ void each(int64_t j0, int64_t stride, int64_t end, F f) {
    for (int64_t j = j0; j < end; j += U * stride) {
      if (j != j0) load(j, stride);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t ju = j + u * stride;
        if (ju >= end) continue;
        const int64_t i = c0 + ju * 8;
        float v[8];
        if (fast) {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = word_elem<T>(w[u][e / E], e % E);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = to_f32(row[min(i + e, c1 - 1)]);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (i + e < c1) f(i + e, v[e]);
      }
    }
  }
};

// Inclusive scan over the wave.
template <typename V>
__device__ __forceinline__ V wave_scan(V v) {
  const int lane = threadIdx.x % kWave;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const V u = __shfl_up(v, o);
    if (lane >= o) v += u;
  }
  return v;
}
// Exclusive scan over NT threads; `part` holds NT / 64 values of LDS.
template <typename V, int NT>
__device__ __forceinline__ V block_scan(V v, V* part, V& total) {
  const int lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
  const V incl = wave_scan(v);
  __syncthreads();                       // part's last readers are done
  if (lane == kWave - 1) part[wid] = incl;
  __syncthreads();
  V before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < NT / kWave; ++w) {
    if (w < wid) before += part[w];
    total += part[w];
  }
  return before + incl - v;
}

// `span` chunks per workgroup (U == 1: one): their maximum stands at the first.
template <typename T, int U>
__global__ __launch_bounds__(kSplitNT) void sample_stats_kernel(SplitArgs a, int span_) {
  __shared__ float red_f[kSplitNT / kWave];
  __shared__ int64_t red_i[kSplitNT / kWave];
  __shared__ int red_b[kSplitNT / kWave];
  const int span = U == 1 ? 1 : span_, per = kSplitG / span;
  const int64_t r = blockIdx.x / per;
  const int c = blockIdx.x % per * span, tid = threadIdx.x;
  SplitRow& w = a.ws[r];
  constexpr int kShare = kSplitNB / kSplitG;
  for (int q = tid; q < span * kShare; q += kSplitNT) w.hist[c * kShare + q] = 0;
  const int64_t c0 = min(c * split_chunk(a.V), a.V);
  const int64_t c1 = min(c0 + span * split_chunk(a.V), a.V);
  float bv;
  int64_t bi;
  bool bad;
  scan_max<T, kSplitNT, U>((const T*)a.logits + r * a.V + c0, c1 - c0, bv, bi, bad);
  if (bi != INT64_MAX) bi += c0;
  wave_first_max(bv, bi);
  bad = __any(bad);
  if (tid % kWave == 0) {
    red_f[tid / kWave] = bv;
    red_i[tid / kWave] = bi;
    red_b[tid / kWave] = bad;
  }
  __syncthreads();
  if (tid == 0) {
    for (int q = 1; q < kSplitNT / kWave; ++q) {
      if (red_f[q] > bv || (red_f[q] == bv && red_i[q] < bi)) {
        bv = red_f[q];
        bi = red_i[q];
      }
      bad |= red_b[q] != 0;
    }
    w.cmax[c] = bv;
    w.cimax[c] = bi == INT64_MAX ? 0xffffffffu : (uint32_t)bi;
    w.cbad[c] = bad;
    for (int q = 1; q < span; ++q) {
      w.cmax[c + q] = -INFINITY;
      w.cimax[c + q] = 0xffffffffu;
      w.cbad[c + q] = 0;
    }
  }
}

template <typename T, int NT>
__global__ __launch_bounds__(NT) void sample_hist_kernel(SplitArgs a) {
  __shared__ unsigned long long lhist[kSplitNB];
  __shared__ unsigned long long part[NT / kWave];
  __shared__ uint32_t upart[NT / kWave];
  __shared__ int sh_bin;
  const int64_t r = blockIdx.x / kSplitG;
  const int c = blockIdx.x % kSplitG, tid = threadIdx.x;
  SplitRow& w = a.ws[r];
  const float Tm = a.temperature[r];
  if (!(Tm > 0.f) && c != 0) return;
  const T* row = (const T*)a.logits + r * a.V;
  const int64_t c0 = min(c * split_chunk(a.V), a.V), c1 = min(c0 + split_chunk(a.V), a.V);
  Octets<T> o(row, a.V, c0, c1);
  // consecutive elements per thread: thread order is vocabulary order
  const int64_t seg = (o.n + NT - 1) / NT, end = min((tid + 1) * seg, o.n);
  o.load(tid * seg, 1);                  // in flight with the chunk maxima
  float lmax;
  int64_t imax;
  const bool bad = split_stats(w, lmax, imax);
  const float M = lmax / Tm;
  if (bad || !(Tm > 0.f) || !(fabsf(M) < INFINITY)) {
    if (c == 0 && tid == 0) {
      if (bad) {
        a.status[r] = 1;
        a.token[r] = imax == INT64_MAX ? 0 : imax;
        a.logprob[r] = NAN;
      } else if (!(Tm > 0.f)) {
        a.status[r] = 0;
        a.token[r] = imax;
        a.logprob[r] = 0.f;
      }
      w.state = bad ? kRowBad : !(Tm > 0.f) ? kRowGreedy : kRowWhole;
    }
    return;
  }
  const int mode = split_mode(a, r);
  for (int b = tid; b < kSplitNB; b += NT) lhist[b] = 0;
  __syncthreads();
  unsigned long long sum = 0;
  o.each(tid * seg, 1, end, [&](int64_t, float l) {
    const float x = l / Tm;
    if (mode == kModeTopK)
      atomicAdd(&lhist[split_bin(x, M)], 1ull);
    else if (mode == kModeTopP)
      atomicAdd(&lhist[split_bin(x, M)], mass_fix(x, M));
    else
      sum += mass_fix(x, M);
  });
  if (mode == kModeAll) {
    unsigned long long total;
    block_scan<unsigned long long, NT>(sum, part, total);
    if (tid == 0) w.hard[c] = total;
    return;
  }
  __syncthreads();
  constexpr int kPer = kSplitNB / NT;
  if (mode == kModeTopP) {
    for (int q = tid; q < kSplitNB; q += NT)
      if (lhist[q]) atomicAdd(&w.hist[q], lhist[q]);
    return;
  }
  // top-k: what lies past the chunk's own k-th element cannot be among the
  // row's first k: neither those bins nor those elements are passed on
  unsigned long long mine = 0, total;
  for (int q = 0; q < kPer; ++q) mine += lhist[tid * kPer + q];
  unsigned long long run = block_scan<unsigned long long, NT>(mine, part, total);
  const unsigned long long kk = (unsigned long long)a.top_k[r];
  if (tid == 0 && total < kk) sh_bin = kSplitNB - 1;
  for (int q = 0; q < kPer; ++q) {
    const unsigned long long h = lhist[tid * kPer + q];
    if (h && run < kk) {
      atomicAdd(&w.hist[tid * kPer + q], h);
      if (run + h >= kk) sh_bin = tid * kPer + q;
    }
    run += h;
  }
  __syncthreads();
  const int bin = sh_bin;
  uint32_t mine_n = 0, listed;
  if (seg > 1) o.load(tid * seg, 1);
  o.each(tid * seg, 1, end, [&](int64_t, float l) { mine_n += split_bin(l / Tm, M) <= bin; });
  uint32_t pos = block_scan<uint32_t, NT>(mine_n, upart, listed);
  if (mine_n && pos < (uint32_t)kSplitCapC) {
    if (seg > 1) o.load(tid * seg, 1);
    o.each(tid * seg, 1, end, [&](int64_t i, float l) {
      const float x = l / Tm;
      if (split_bin(x, M) <= bin) {
        if (pos < (uint32_t)kSplitCapC) {
          w.ckey[c * kSplitCapC + pos] = okey(x);
          w.cidx[c * kSplitCapC + pos] = (uint32_t)i;
        }
        ++pos;
      }
    });
  }
  if (tid == 0) w.lcnt[c] = listed;
}

// The first bin (from the maximum down) at which the running count or mass
// reaches `goal`, in sh_bin, and that above it in sh_above; NT threads hold
// the histogram's bins in order, PER each.
template <int NT, int PER>
__device__ __forceinline__ void split_boundary(const unsigned long long (&h)[PER],
                                               unsigned long long run, unsigned long long mine,
                                               unsigned long long goal, int* sh_bin,
                                               unsigned long long* sh_above) {
  if (run < goal && goal <= run + mine) {
    bool found = false;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      if (!found && goal <= run + h[q]) {
        found = true;
        *sh_bin = threadIdx.x * PER + q;
        *sh_above = run;
      }
      run += h[q];
    }
  }
}

// The mass that top-p keeps at least, of the mass it chooses from.
__device__ __forceinline__ unsigned long long split_goal(float p, unsigned long long z) {
  return max(1ull, (unsigned long long)(fmax((double)p, 0.0) * (double)z));
}

// The lowest float that `ok`, a property of all floats from some one up to top, holds for.
template <typename F>
__device__ __forceinline__ float lowest_float(float top, F ok) {
  uint32_t lo = okey(-3.402823466e38f), hi = okey(top);   // ok(hi)
  while (lo < hi) {                                       // 64 candidates at a time
    const uint32_t step = (hi - lo) / kWave + 1;
    const uint64_t at = (uint64_t)lo + (threadIdx.x % kWave) * (uint64_t)step;
    const uint32_t mine = at < hi ? (uint32_t)at : hi;
    const uint64_t yes = __ballot(ok(key_float(mine)));
    const int first = __ffsll((unsigned long long)yes) - 1;
    if (first < 0) {
      lo = __shfl(mine, kWave - 1) + 1;
    } else {
      hi = __shfl(mine, first);
      if (first > 0) lo = __shfl(mine, first - 1) + 1;
      else lo = hi;
    }
  }
  return key_float(hi);
}

// A row whose boundary holds more elements than the lists: the kept set by radix
// descent over the keys (11, 11 and 10 bits), as in sample_row, but from the
// boundary bin the histogram has found: the elements outside it are told by one
// comparison of the logit, rows are read as vectors, several in flight, and equal
// neighbours (ties) are added once per wave. Returns (lowest kept key, first kept
// index among its ties) and leaves the chunks' kept masses in cm, which holds
// those above the bin (top-p) or 0. Bound by the VALU work per element of one CU per
// row: 8 bf16 rows of 151936 with a spread of 2 around 8 (top-p 0.9 then ends in one
// value of 1460 tokens) 179 us, on sample_row 612; top-k 5000 142, there 377.
template <typename T>
__device__ unsigned long long split_descend(const T* row, int64_t V, int64_t chunk, float Tm,
                                            float M, float lmax, int mode, unsigned long long kk,
                                            float pp, int bin, unsigned long long above,
                                            unsigned long long zk, unsigned long long* part,
                                            unsigned long long* cm) {
  __shared__ unsigned long long hsum[kSplitNB], sh_above;
  __shared__ uint32_t hcnt[kSplitNB], ties[kSplitG], sh_d, sh_tie0;
  static_assert(kSplitNB == 2 * kNT, "two digits per thread");
  const int tid = threadIdx.x, lane = tid % kWave, wid = tid / kWave;
  Octets<T, 4> o(row, V, 0, V);
  uint32_t key = 0, cnt = 0;                          // of the boundary
  unsigned long long below = 0;                       // count or mass above it
  // the key at which the running count (top-k) or mass from the highest key down
  // passes `goal`, of logits in [lo, hi) with keys from kmin; `start` lies above them
  auto descend = [&](float lo, float hi, uint32_t kmin, bool by_mass, unsigned long long goal,
                     unsigned long long start) {
    uint32_t prefix = 0, pmask = 0;
    below = start;
#pragma unroll 1
    for (int shift = 21; shift >= 0; shift = shift == 21 ? 10 : shift - 10) {
      const uint32_t digits = shift ? 2047u : 1023u;
      for (int q = tid; q < kSplitNB; q += kNT) {
        hsum[q] = 0;
        hcnt[q] = 0;
      }
      if (tid == 0) sh_d = 0;
      __syncthreads();
      o.load(tid, kNT);
      o.each(tid, kNT, o.n, [&](int64_t, float l) {
        if (!(l >= lo && l < hi)) return;
        const float x = l / Tm;
        const uint32_t k = okey(x);
        if (k < kmin || (k & pmask) != prefix) return;
        const unsigned long long m = by_mass ? mass_fix(x, M) : 1ull;
        const uint32_t k0 = __builtin_amdgcn_readfirstlane(k);
        const uint64_t same = __ballot(k == k0);
        const int d = (int)((k >> shift) & digits);
        if (k != k0 || lane == __ffsll((unsigned long long)same) - 1) {
          const uint32_t c = k == k0 ? (uint32_t)__popcll(same) : 1u;
          atomicAdd(&hsum[d], c * m);
          atomicAdd(&hcnt[d], c);
        }
      });
      __syncthreads();
      const int d1 = kSplitNB - 1 - 2 * tid;          // this thread's digits, highest first
      const unsigned long long v1 = hsum[d1], v0 = hsum[d1 - 1];
      unsigned long long total;
      const unsigned long long run =
          below + block_scan<unsigned long long, kNT>(v1 + v0, part, total);
      if (run < goal && goal <= run + v1 + v0) {
        sh_d = goal <= run + v1 ? d1 : d1 - 1;
        sh_above = goal <= run + v1 ? run : run + v1;
      }
      __syncthreads();
      prefix |= sh_d << shift;
      pmask |= digits << shift;
      below = sh_above;
      cnt = hcnt[sh_d];
      __syncthreads();
    }
    key = prefix;
  };
  auto in_bin = [&](int b) {
    return lowest_float(lmax, [&](float l) { return split_bin(l / Tm, M) <= b; });
  };
  float lo = in_bin(bin), hi = bin > 0 ? in_bin(bin - 1) : INFINITY;
  uint32_t keep = 0xffffffffu;                        // ties kept
  unsigned long long goal = 0;
  if (mode == kModeTopK) {
    descend(lo, hi, 0u, false, kk, above);
    const uint32_t kkey = key;
    lo = lowest_float(lmax, [&](float l) { return okey(l / Tm) >= kkey; });
    hi = INFINITY;
    if (pp < 1.0f) {
      unsigned long long sum = 0;
      o.load(tid, kNT);
      o.each(tid, kNT, o.n, [&](int64_t, float l) {
        if (l >= lo && okey(l / Tm) >= kkey) sum += mass_fix(l / Tm, M);
      });
      block_scan<unsigned long long, kNT>(sum, part, zk);
      goal = split_goal(pp, zk);
      descend(lo, hi, kkey, true, goal, 0);
    }
  } else {
    goal = split_goal(pp, zk);
    descend(lo, hi, 0u, true, goal, above);
  }
  const unsigned long long m = mass_fix(key_float(key), M);
  if (goal > 0 && m > 0) {
    const double need = ceil(((double)goal - (double)below) / (double)m);
    keep = (uint32_t)fmax(1.0, fmin(need, (double)cnt));
  }
  // per chunk, a wave each: its ties and the mass above them
  for (int c = wid; c < kSplitG; c += kNT / kWave) {
    const int64_t c0 = min(c * chunk, V), c1 = min(c0 + chunk, V);
    Octets<T, 4> oc(row, V, c0, c1);
    unsigned long long sum = 0;
    uint32_t n = 0;
    oc.load(lane, kWave);
    oc.each(lane, kWave, oc.n, [&](int64_t, float l) {
      if (!(l >= lo && l < hi)) return;
      const float x = l / Tm;
      const uint32_t k = okey(x);
      if (k > key) sum += mass_fix(x, M);
      n += k == key;
    });
    sum = wave_scan(sum);
    n = wave_scan(n);
    if (lane == kWave - 1) {
      cm[c] += sum;
      ties[c] = n;
    }
  }
  if (tid == 0) sh_tie0 = 0;
  __syncthreads();
  // ties are kept from the highest index down: `drop` of them are not, the last of
  // these in chunk `cut`
  const uint32_t mine = lane < kSplitG ? ties[lane] : 0u, upto = wave_scan(mine);
  const uint32_t all = __shfl(upto, kWave - 1), drop = keep < all ? all - keep : 0u;
  const int cut = drop ? __ffsll((unsigned long long)__ballot(upto > drop)) - 1 : -1;
  const uint32_t before = upto - mine;
  if (tid < kSplitG) {
    const uint32_t lost = drop > before ? min(drop - before, mine) : 0u;
    cm[lane] += (mine - lost) * m;
  }
  if (cut >= 0) {                                     // the first kept tie's index
    const uint32_t rank = drop - __shfl(before, cut);
    const int64_t c0 = min(cut * chunk, V), c1 = min(c0 + chunk, V);
    const bool aligned = ((uintptr_t)row % 16) == 0 && V % 8 == 0;
    uint32_t base = 0;
    for (int64_t t0 = c0; t0 < c1 && base <= rank; t0 += kNT * 8) {
      const int64_t i = t0 + tid * 8;
      float x[8];
      uint32_t n = 0, tot;
      if (i < c1) {
        load8(row, i, c1, aligned, x);
#pragma unroll
        for (int e = 0; e < 8; ++e) n += i + e < c1 && okey(x[e] / Tm) == key;
      }
      uint32_t at = base + block_scan<uint32_t, kNT>(n, (uint32_t*)part, tot);
      if (n && at <= rank && rank < at + n) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (i + e < c1 && okey(x[e] / Tm) == key && at++ == rank) sh_tie0 = (uint32_t)(i + e);
      }
      base += tot;
    }
  }
  __syncthreads();
  return (unsigned long long)key << 32 | sh_tie0;
}

template <typename T, int NT>
__global__ __launch_bounds__(NT) void sample_gather_kernel(SplitArgs a) {
  __shared__ unsigned long long part[NT / kWave];
  __shared__ uint32_t upart[NT / kWave];
  __shared__ int sh_bin;
  __shared__ unsigned long long sh_above;
  const int64_t r = blockIdx.x / kSplitG;
  const int c = blockIdx.x % kSplitG, tid = threadIdx.x;
  SplitRow& w = a.ws[r];
  const float Tm = a.temperature[r];
  const int mode = split_mode(a, r);
  if (!(Tm > 0.f) || mode == kModeAll) return;
  if (mode == kModeTopK && !__any(w.lcnt[tid % kSplitG] > (uint32_t)kSplitCapC)) return;
  // the chunk, the histogram and the chunk maxima in one round trip. A thread
  // holds consecutive elements, so that thread order is vocabulary order
  const T* row = (const T*)a.logits + r * a.V;
  const int64_t c0 = min(c * split_chunk(a.V), a.V), c1 = min(c0 + split_chunk(a.V), a.V);
  Octets<T> o(row, a.V, c0, c1);
  const int64_t seg = (o.n + NT - 1) / NT;
  o.load(tid * seg, 1);
  constexpr int kPer = kSplitNB / NT;
  unsigned long long h[kPer], mine = 0, total;
#pragma unroll
  for (int q = 0; q < kPer; ++q) h[q] = w.hist[tid * kPer + q];
#pragma unroll
  for (int q = 0; q < kPer; ++q) asm volatile("" ::"v"(h[q]));
  float lmax;
  int64_t imax;
  const bool bad = split_stats(w, lmax, imax);
  const float M = lmax / Tm;
  if (bad || !(fabsf(M) < INFINITY)) return;

#pragma unroll
  for (int q = 0; q < kPer; ++q) mine += h[q];
  const unsigned long long run = block_scan<unsigned long long, NT>(mine, part, total);
  const unsigned long long goal =
      mode == kModeTopK ? (unsigned long long)a.top_k[r] : split_goal(a.top_p[r], total);
  split_boundary<NT, kPer>(h, run, mine, goal, &sh_bin, &sh_above);
  __syncthreads();
  const int bin = sh_bin;

  unsigned long long hard = 0;
  uint32_t mine_n = 0, listed;
  const int64_t end = min((tid + 1) * seg, o.n);
  o.each(tid * seg, 1, end, [&](int64_t, float l) {
    const float x = l / Tm;
    const int b = split_bin(x, M);
    if (b == bin || (mode == kModeTopK && b < bin))
      ++mine_n;
    else if (b < bin)
      hard += mass_fix(x, M);
  });
  uint32_t pos = block_scan<uint32_t, NT>(mine_n, upart, listed);
  if (mine_n && pos < (uint32_t)kSplitCapC) {    // (few threads: the chunk is read again)
    o.load(tid * seg, 1);
    o.each(tid * seg, 1, end, [&](int64_t i, float l) {
      const float x = l / Tm;
      const int b = split_bin(x, M);
      if (b == bin || (mode == kModeTopK && b < bin)) {
        if (pos < (uint32_t)kSplitCapC) {
          w.ckey[c * kSplitCapC + pos] = okey(x);
          w.cidx[c * kSplitCapC + pos] = (uint32_t)i;
        }
        ++pos;
      }
    });
  }
  unsigned long long hsum;
  block_scan<unsigned long long, NT>(hard, part, hsum);
  if (tid == 0) {
    w.hard[c] = hsum;
    w.ccnt[c] = listed;
    if (c == 0) {
      w.zk = total;
      w.above = sh_above;
    }
  }
}

template <typename T>
__global__ __launch_bounds__(kNT) void sample_pick_kernel(SplitArgs a) {
  __shared__ uint32_t skey[kSplitCap], sidx[kSplitCap];
  __shared__ unsigned long long sw[kSplitCap];
  __shared__ unsigned long long part[kNT / kWave];
  __shared__ unsigned long long cm[kSplitG];          // kept mass per chunk
  __shared__ uint32_t cnt[kSplitG], off[kSplitG + 1];
  __shared__ unsigned long long sh_zk, sh_low, sh_z, sh_rem, sh_above;
  __shared__ int sh_over, sh_chunk, sh_bin;
  const int64_t r = blockIdx.x;
  const int tid = threadIdx.x, lane = tid % kWave;
  SplitRow& w = a.ws[r];
  const float Tm = a.temperature[r];
  if (!(Tm > 0.f)) return;                            // written by `hist`
  // every slot of the lists (the unused ones hold anything), the counts and
  // the chunk maxima in one round trip
  constexpr int kSlots = kSplitG * kSplitCapC / kNT;
  uint32_t lk[kSlots], li[kSlots];
#pragma unroll
  for (int u = 0; u < kSlots; ++u) {
    lk[u] = w.ckey[u * kNT + tid];
    li[u] = w.cidx[u * kNT + tid];
  }
  constexpr int kPer = kSplitNB / kNT;
  unsigned long long h[kPer];                         // (top-k: the boundary bin again)
#pragma unroll
  for (int q = 0; q < kPer; ++q) h[q] = w.hist[tid * kPer + q];
  const uint32_t llist = w.lcnt[lane % kSplitG];
  const uint32_t clist = w.ccnt[lane % kSplitG];
  const unsigned long long lhard = w.hard[lane % kSplitG];
#pragma unroll
  for (int u = 0; u < kSlots; ++u) asm volatile("" ::"v"(lk[u]), "v"(li[u]));
#pragma unroll
  for (int q = 0; q < kPer; ++q) asm volatile("" ::"v"(h[q]));
  asm volatile("" ::"v"(llist), "v"(clist), "v"(lhard));
  float lmax;
  int64_t imax;
  const bool bad = split_stats(w, lmax, imax);
  const float M = lmax / Tm;
  if (bad) return;                                    // written by `hist`
  const int mode = split_mode(a, r);
  const int64_t kk = a.top_k[r];
  const float pp = a.top_p[r];
  const int64_t chunk = split_chunk(a.V);
  const bool whole = !(fabsf(M) < INFINITY);

  // the lists' lengths: top-k, those of `hist` unless one overflowed
  const bool again = mode == kModeTopK && __any(llist > (uint32_t)kSplitCapC);
  const uint32_t lcnt = mode == kModeTopK && !again ? llist : clist;
  const bool over = mode != kModeAll && __any(lcnt > (uint32_t)kSplitCapC);
  int bin = kSplitNB;                                 // elements past it are not on the boundary
  if (mode == kModeTopK && !whole) {
    unsigned long long mine = 0, total;
#pragma unroll
    for (int q = 0; q < kPer; ++q) mine += h[q];
    const unsigned long long run = block_scan<unsigned long long, kNT>(mine, part, total);
    split_boundary<kNT, kPer>(h, run, mine, (unsigned long long)kk, &sh_bin, &sh_above);
    __syncthreads();
    bin = sh_bin;
  }
  // compacted in slot order, which is vocabulary order: a wave holds one
  // chunk's list (kSplitCapC slots) per round
  static_assert(kSplitCapC == kWave && kSlots * kNT == kSplitG * kSplitCapC, "a wave per list");
  uint64_t sel[kSlots];
#pragma unroll
  for (int u = 0; u < kSlots; ++u) {
    const int c = u * (kNT / kWave) + tid / kWave;
    sel[u] = __ballot(mode != kModeAll && !whole && (uint32_t)lane < __shfl(lcnt, c) &&
                      split_bin(key_float(lk[u]), M) <= bin);
    if (lane == 0) cnt[c] = (uint32_t)__popcll(sel[u]);
  }
  __syncthreads();
  if (tid < kWave) {                                  // wave 0: the lists' offsets
    const uint32_t n = lane < kSplitG ? cnt[lane] : 0u;
    const uint32_t incl = wave_scan(n);
    if (lane < kSplitG) {
      off[lane + 1] = incl;
      cm[lane] = mode == kModeTopK ? 0 : lhard;
    }
    if (lane == 0) {
      off[0] = 0;
      sh_zk = 0;
      sh_low = ~0ull;
    }
    if (lane == kSplitG - 1) sh_over = over || incl > (uint32_t)kSplitCap;
  }
  __syncthreads();
  if (whole) {                                        // (uniform over the workgroup)
    if (tid == 0) w.state = kRowWhole;
    sample_row<T>(r, (const T*)a.logits, a.V, a.temperature, a.top_k, a.top_p, a.uniform,
                  a.token, a.logprob, a.processed, a.status);
    return;
  }
  const bool longer = sh_over;
  if (longer) {
    unsigned long long zk = 0;
    if (mode == kModeTopP) {                          // the boundary bin, as in `gather`
      unsigned long long mine = 0;
#pragma unroll
      for (int q = 0; q < kPer; ++q) mine += h[q];
      const unsigned long long run = block_scan<unsigned long long, kNT>(mine, part, zk);
      split_boundary<kNT, kPer>(h, run, mine, split_goal(pp, zk), &sh_bin, &sh_above);
      __syncthreads();
      bin = sh_bin;
    }
    const unsigned long long low = split_descend<T>(
        (const T*)a.logits + r * a.V, a.V, chunk, Tm, M, lmax, mode, (unsigned long long)kk, pp,
        bin, sh_above, zk, part, cm);
    if (tid == 0) sh_low = low;
  } else {
    const int n = (int)off[kSplitG];
#pragma unroll
    for (int u = 0; u < kSlots; ++u) {
      const int c = u * (kNT / kWave) + tid / kWave;
      if (sel[u] >> lane & 1) {
        const uint32_t at = off[c] + __popcll(sel[u] & (((uint64_t)1 << lane) - 1));
        skey[at] = lk[u];
        sidx[at] = li[u];
      }
    }
    __syncthreads();
    uint32_t key = 0, idx = 0;
    unsigned long long m = 0;
    if (tid < n) {
      key = skey[tid];
      idx = sidx[tid];
      m = mass_fix(key_float(key), M);
      sw[tid] = m;
    }
    __syncthreads();
    // rank by counting: elements above mine, their mass, ties and those after me
    uint32_t higher = 0, ties = 0, after = 0;
    unsigned long long above = 0;
    if ((tid & ~(kWave - 1)) < n) {
      for (int j = 0; j < n; ++j) {
        const uint32_t kj = skey[j];
        const unsigned long long mj = sw[j];
        if (kj > key) {
          ++higher;
          above += mj;
        }
        if (kj == key) {
          ++ties;
          after += j > tid;
        }
      }
    }
    bool keep = tid < n && (mode != kModeTopK || (int64_t)higher < kk);
    if (mode == kModeTopK && keep) atomicAdd(&sh_zk, m);
    __syncthreads();
    if (pp < 1.0f && mode != kModeAll) {
      const unsigned long long zk = mode == kModeTopK ? sh_zk : w.zk;
      if (mode == kModeTopP) above += w.above;
      const unsigned long long target = split_goal(pp, zk);
      // a group of equal values is kept while the mass above it is below the
      // target; of the last one, as many as reach it, from the highest index down
      keep = keep && above < target;
      if (keep && m > 0) {
        const double need = ceil(((double)target - (double)above) / (double)m);
        keep = (double)after < fmax(1.0, fmin(need, (double)ties));
      }
    }
    if (keep) {
      atomicAdd(&cm[idx / (uint32_t)chunk], m);
      atomicMin(&sh_low, ((unsigned long long)key << 32) | idx);
    }
    if (tid < n) sw[tid] = keep ? m : 0;
  }
  __syncthreads();
  const uint32_t pkey = mode == kModeAll ? 0u : (uint32_t)(sh_low >> 32);
  const uint32_t tie0 = mode == kModeAll ? 0u : (uint32_t)sh_low;
  if (tid < kWave) {                                  // wave 0: the drawn chunk
    const unsigned long long mc = lane < kSplitG ? cm[lane] : 0;
    const unsigned long long incl = wave_scan(mc);
    const unsigned long long Z = __shfl(incl, kWave - 1);
    const unsigned long long t = min(
        (unsigned long long)(fmax((double)a.uniform[r], 0.0) * (double)Z), Z - 1);
    const int c = __ffsll((unsigned long long)__ballot(incl > t)) - 1;
    if (lane == c) {
      sh_chunk = c;
      sh_rem = t - (incl - mc);
    }
    if (lane == 0) {
      sh_z = Z;
      w.state = kRowDrawn;
      w.pkey = pkey;
      w.tie0 = tie0;
    }
  }
  __syncthreads();
  const int c = sh_chunk;
  const unsigned long long rem = sh_rem;
  auto draw = [&](int64_t i, float x) {
    a.token[r] = i;
    a.logprob[r] = (x - M) - logf((float)((double)sh_z / kFix));
    a.status[r] = 0;
  };
  if (mode == kModeTopK && !longer) {                 // inside the chunk's list
    if (tid >= kWave) return;
    const int j = (int)off[c] + lane;
    const unsigned long long mj = j < (int)off[c + 1] ? sw[j] : 0;
    const int pick = __ffsll((unsigned long long)__ballot(wave_scan(mj) > rem)) - 1;
    if (lane == pick) draw(sidx[j], key_float(skey[j]));
    return;
  }
  const T* row = (const T*)a.logits + r * a.V;
  const bool aligned = ((uintptr_t)row % 16) == 0;
  const int64_t c0 = min(c * chunk, a.V), c1 = min(c0 + chunk, a.V);
  unsigned long long base = 0;
  for (int64_t t0 = c0; t0 < c1 && base <= rem; t0 += kNT * 8) {
    const int64_t i = t0 + tid * 8;
    float x[8];
    unsigned long long me[8], mine = 0, total;
    if (i < c1) load8(row, i, c1, aligned, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      me[e] = 0;
      if (i + e < c1) {
        x[e] = x[e] / Tm;
        const uint32_t k = okey(x[e]);
        if (k > pkey || (k == pkey && (uint64_t)(i + e) >= tie0)) me[e] = mass_fix(x[e], M);
      }
      mine += me[e];
    }
    unsigned long long run = base + block_scan<unsigned long long, kNT>(mine, part, total);
    if (run <= rem && rem < run + mine) {
      bool found = false;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        run += me[e];
        if (!found && rem < run) {
          found = true;
          draw(i + e, x[e]);
        }
      }
    }
    base += total;
  }
}

// The processed logits of the rows the split form drew (and of greedy ones).
template <typename T>
__global__ __launch_bounds__(kSplitNT) void sample_processed_kernel(SplitArgs a) {
  const int64_t r = blockIdx.x / kSplitG;
  const int c = blockIdx.x % kSplitG;
  const SplitRow& w = a.ws[r];
  const uint32_t state = w.state;
  if (state != kRowDrawn && state != kRowGreedy) return;
  const float Tm = a.temperature[r];
  const uint32_t pkey = w.pkey, tie0 = w.tie0;
  const T* row = (const T*)a.logits + r * a.V;
  const int64_t c0 = min(c * split_chunk(a.V), a.V), c1 = min(c0 + split_chunk(a.V), a.V);
  for (int64_t i = c0 + threadIdx.x; i < c1; i += kSplitNT) {
    const float l = to_f32(row[i]);
    const float x = l / Tm;
    const uint32_t k = okey(x);
    a.processed[r * a.V + i] =
        state == kRowGreedy ? l
                            : (k > pkey || (k == pkey && (uint64_t)i >= tie0)) ? x : -INFINITY;
  }
}

template <typename T>
__global__ __launch_bounds__(kNT) void sample_kernel(
    const T* __restrict__ logits, int64_t V, const float* __restrict__ temperature,
    const int32_t* __restrict__ top_k, const float* __restrict__ top_p,
    const float* __restrict__ uniform, int64_t* __restrict__ token, float* __restrict__ logprob,
    float* __restrict__ processed, int32_t* __restrict__ status) {
  sample_row<T>(blockIdx.x, logits, V, temperature, top_k, top_p, uniform, token, logprob,
                processed, status);
}

template <typename T, int NT>
void launch_split_chunks(const SplitArgs& a, int64_t rows, hipStream_t st) {
  const dim3 grid((unsigned)(rows * kSplitG));
  sample_hist_kernel<T, NT><<<grid, NT, 0, st>>>(a);
  sample_gather_kernel<T, NT><<<grid, NT, 0, st>>>(a);
}
template <typename T>
void launch_split(const SplitArgs& a, int64_t rows, hipStream_t st) {
  const dim3 grid((unsigned)(rows * kSplitG));
  int span = 1;
  while (span < kSplitG && rows * kSplitG / span > kSplitWGs) span *= 2;
  const dim3 stats((unsigned)(rows * (kSplitG / span)));
  if (span == 1)
    sample_stats_kernel<T, 1><<<stats, kSplitNT, 0, st>>>(a, span);
  else
    sample_stats_kernel<T, 4><<<stats, kSplitNT, 0, st>>>(a, span);
  if (rows <= kSplitWideRows)
    launch_split_chunks<T, kSplitNT>(a, rows, st);
  else
    launch_split_chunks<T, kSplitFewNT>(a, rows, st);
  sample_pick_kernel<T><<<(unsigned)rows, kNT, 0, st>>>(a);
  if (a.processed) sample_processed_kernel<T><<<grid, kSplitNT, 0, st>>>(a);
}

}  // namespace

extern "C" int acorn_sample_workspace(int64_t rows, int64_t vocab, int64_t* bytes) {
  if (rows < 0 || vocab <= 0 || !bytes) return ACORN_ERR_VALUE;
  *bytes = vocab >= kSplitMinV && vocab <= kSplitMaxV && rows <= kSplitMaxRows
               ? rows * (int64_t)sizeof(SplitRow)
               : 0;
  return ACORN_OK;
}

extern "C" int acorn_sample_split(const void* logits, int64_t rows, int64_t vocab, int dtype,
                                  const float* temperature, const int32_t* top_k,
                                  const float* top_p, const float* uniform, int64_t* token,
                                  float* logprob, float* processed, int32_t* status, void* ws,
                                  int64_t ws_bytes, void* stream) {
  int64_t need = 0;
  if (rows < 0 || vocab <= 0 || acorn_sample_workspace(rows, vocab, &need) != ACORN_OK)
    return ACORN_ERR_SHAPE;
  if (!ws || need == 0 || ws_bytes < need)
    return acorn_sample(logits, rows, vocab, dtype, temperature, top_k, top_p, uniform, token,
                        logprob, processed, status, stream);
  if (!logits || !temperature || !top_k || !top_p || !uniform || !token || !logprob || !status ||
      (uintptr_t)ws % alignof(SplitRow))
    return ACORN_ERR_VALUE;
  const SplitArgs a{logits, vocab,   temperature, top_k,     top_p,  uniform,
                    token,  logprob, processed,   status, (SplitRow*)ws};
  hipStream_t st = (hipStream_t)stream;
  switch (dtype) {
    case ACORN_F32: launch_split<float>(a, rows, st); break;
    case ACORN_F16: launch_split<_Float16>(a, rows, st); break;
    case ACORN_BF16: launch_split<__bf16>(a, rows, st); break;
    default: return ACORN_ERR_DTYPE;
  }
  ACORN_LAUNCH_CHECK();
  return ACORN_OK;
}

extern "C" int acorn_sample(const void* logits, int64_t rows, int64_t vocab, int dtype,
                            const float* temperature, const int32_t* top_k, const float* top_p,
                            const float* uniform, int64_t* token, float* logprob,
                            float* processed, int32_t* status, void* stream) {
  if (rows < 0 || vocab <= 0 || rows > 0x7fffffff || vocab > ((int64_t)1 << 31))
    return ACORN_ERR_SHAPE;
  if (rows == 0) return ACORN_OK;
  if (!logits || !temperature || !top_k || !top_p || !uniform || !token || !logprob || !status)
    return ACORN_ERR_VALUE;
  hipStream_t st = (hipStream_t)stream;
  dim3 grid((unsigned)rows), block(kNT);
  switch (dtype) {
    case ACORN_F32:
      sample_kernel<float><<<grid, block, 0, st>>>((const float*)logits, vocab, temperature, top_k, top_p, uniform, token, logprob, processed, status);
      break;
    case ACORN_F16:
      sample_kernel<_Float16><<<grid, block, 0, st>>>((const _Float16*)logits, vocab, temperature, top_k, top_p, uniform, token, logprob, processed, status);
      break;
    case ACORN_BF16:
      sample_kernel<__bf16><<<grid, block, 0, st>>>((const __bf16*)logits, vocab, temperature, top_k, top_p, uniform, token, logprob, processed, status);
      break;
    default:
      return ACORN_ERR_DTYPE;
  }
  ACORN_LAUNCH_CHECK();
  return ACORN_OK;
}
