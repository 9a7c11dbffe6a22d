// Per-sequence keep-set selection on CDNA4: segmented threshold select.
//
// A job is one (sequence, segment).  The segment's scores are mapped to
// order-preserving 32-bit keys; the exact key T of the K-th largest score and
// how many scores equal to T are still needed come from a histogram over value
// bins and an exact ranking inside one bin (binned again while a bin holds too
// many keys to rank).
// Emission keeps every key > T plus the first `need` keys == T (ties go to the
// lowest index), walking the segment in coalesced tiles: prefix sums of packed
// (greater, equal) counts give every key its output slot, so the output is
// sorted without a sort.
//
// Two launch shapes:
//  * kvc_select_keep: one 1024-thread workgroup per job.  Right for batches of
//    many sequences.
//  * kvc_select_keep_split: a job's segment is cut into chunks of >= 4096 keys,
//    one 256-thread workgroup each, in three launches (no workgroup waits for
//    another inside one): every chunk's histogram over value bins, the chunks'
//    keys of the bin that holds the threshold, and the emission, each chunk
//    starting from the counts of the chunks before it.  Right for a few long
//    sequences, which would otherwise run on a few CUs.
// Both produce the same indices.
//
// Segments follow select_keep_indices (tri/selection.py:108-196): the protected
// prefix [0, prefix) and recent window [n-recent, n) are always kept; policy
// GLOBAL keeps budget-prefix-recent of the middle; policy V3 cuts the middle
// into `segments` ranges [ms + M*k/S, ms + M*(k+1)/S) whose keep quota is
// len - (E*(stop-ms)/M - E*(start-ms)/M) with E = n - budget (integer floors).

#include "kvc_common.h"

namespace kvc {
namespace {

constexpr int kSelThreads = 1024;   // one workgroup per job
constexpr int kSplitThreads = 256;  // split path: one workgroup per chunk
constexpr int kSplitChunk = 4096;   // keys per chunk, at least
constexpr int kSplitMaxChunks = 32;
constexpr int kSelUnroll = 4;  // float4 words per thread in flight in a walk
constexpr int kEmitWords = 2;  // float4 words per thread per emission tile

struct SelectArgs {
  int n_seq, budget, prefix, recent, segments, policy;
  const int32_t* seq_lens;
  const int64_t* token_offsets;
  const float* scores;
  int64_t* keep;
  int64_t keep_stride;
  void* state;  // split path: [n_seq][segments] SplitState
};

struct Segment {
  int64_t start, stop, keep;
};

// floor(p / c) for p >= 0, c > 0 and a quotient below 2^31 (scores of one
// sequence): the double quotient is off by one at most, which the remainder
// shows.  The compiler's 64-bit division is some 150 instructions, five of
// them a job.
__device__ __forceinline__ int64_t div_floor(int64_t p, int64_t c) {
  int64_t q = static_cast<int64_t>(static_cast<double>(p) / static_cast<double>(c));
  const int64_t r = p - q * c;
  if (r < 0) --q;
  if (r >= c) ++q;
  return q;
}

__device__ __forceinline__ Segment v3_segment(int64_t ms, int64_t mc, int64_t evict, int k, int nseg) {
  Segment s;
  s.start = ms + div_floor(mc * k, nseg);
  s.stop = ms + div_floor(mc * (k + 1), nseg);
  const int64_t len = s.stop - s.start;
  if (len <= 0) {
    s.keep = 0;
    return s;
  }
  const int64_t before = evict * (s.start - ms) / mc;
  const int64_t after = evict * (s.stop - ms) / mc;
  const int64_t keep = len - (after - before);
  s.keep = keep > 0 ? keep : 0;
  return s;
}

// One (sequence, segment): its segment, first output slot and protected windows.
struct Job {
  int64_t n, prefix, recent, out_base;
  Segment s;
  bool exists;  // the segment index is in range for the policy
};

__device__ Job make_job(const SelectArgs& a, int b, int seg) {
  Job j;
  j.n = a.seq_lens[b];
  j.prefix = min(static_cast<int64_t>(a.prefix), j.n);
  j.recent = min(static_cast<int64_t>(a.recent), j.n - j.prefix);
  const int64_t ms = j.prefix;
  const int64_t mc = j.n - j.prefix - j.recent;
  const int nseg = (a.policy == KVC_POLICY_V3) ? a.segments : 1;
  j.exists = seg < nseg;
  j.out_base = j.prefix;
  j.s = Segment{ms, ms, 0};
  if (!j.exists) return j;
  if (a.policy == KVC_POLICY_V3) {
    if (mc <= 0) return j;
    const int64_t evict = j.n - a.budget;
    j.s = v3_segment(ms, mc, evict, seg, nseg);
    if (evict >= 0 && evict <= mc) {
      // Every quota is len - (after - before) >= 0 then, so the quotas before
      // this segment telescope (a chain of 64-bit divisions per segment cost
      // the eighth segment's workgroup 2 us before its first load).
      const int64_t before = j.s.start - ms;
      j.out_base += before - div_floor(evict * before, mc);
    } else {
      for (int k = 0; k < seg; ++k) j.out_base += v3_segment(ms, mc, evict, k, nseg).keep;
    }
  } else {
    j.s = Segment{ms, ms + mc, a.budget - j.prefix - j.recent};
  }
  return j;
}

// Protected windows (the workgroup of segment 0) and segments kept whole.
// Returns whether the job still needs a threshold.  Output rows are budget
// entries wide; the guards keep a caller that skipped validation (a sequence
// shorter than the budget) inside its row.
__device__ bool fill_fixed(const SelectArgs& a, const Job& j, int seg, int64_t* out, int tid, int nthreads) {
  if (seg == 0) {
    for (int64_t i = tid; i < j.prefix; i += nthreads) out[i] = i;
    for (int64_t i = tid; i < j.recent; i += nthreads) out[a.budget - j.recent + i] = j.n - j.recent + i;
  }
  const int64_t len = j.s.stop - j.s.start;
  if (!j.exists || j.s.keep <= 0 || len <= 0) return false;
  if (j.s.keep >= len) {
    for (int64_t i = tid; i < len && j.out_base + i < a.budget; i += nthreads) out[j.out_base + i] = j.s.start + i;
    return false;
  }
  return true;
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Calls f(score) for every score in [start, stop), spread over a workgroup of
// T threads: scalar head up to 16-byte alignment, float4 words U at a
// time (loads issued together), scalar tail.
template <int T, int U = kSelUnroll, typename F>
__device__ __forceinline__ void for_each_score(const float* sc, int64_t start, int64_t stop, F&& f) {
  const int tid = threadIdx.x;
  const int64_t misalign = (reinterpret_cast<uintptr_t>(sc + start) >> 2) & 3;
  int64_t head = (4 - misalign) & 3;
  if (head > stop - start) head = stop - start;
  for (int64_t i = start + tid; i < start + head; i += T) f(sc[i]);
  const int64_t body = start + head;
  const int64_t n4 = (stop - body) >> 2;
  const f32x4* v = reinterpret_cast<const f32x4*>(sc + body);
  for (int64_t w0 = tid; w0 < n4; w0 += static_cast<int64_t>(T) * U) {
    f32x4 x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t w = w0 + static_cast<int64_t>(u) * T;
      x[u] = v[w < n4 ? w : n4 - 1];  // in range; surplus words are ignored below
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t w = w0 + static_cast<int64_t>(u) * T;
      if (w < n4) {
#pragma unroll
        for (int e = 0; e < 4; ++e) f(x[u][e]);
      }
    }
  }
  for (int64_t i = body + 4 * n4 + tid; i < stop; i += T) f(sc[i]);
}

// The same for code that few calls run: one score a load and little code (the
// first pass over instructions costs more than the walk), except where 256
// threads walk a whole segment and wait for memory.
template <int T, typename F>
__device__ __forceinline__ void for_each_score_rarely(const float* sc, int64_t start, int64_t stop, F&& f) {
  if constexpr (T < kSelThreads) {
    for_each_score<T, 8>(sc, start, stop, f);
  } else {
#pragma unroll 1
    for (int64_t i0 = start + threadIdx.x; i0 < stop; i0 += kSelUnroll * T) {
      float x[kSelUnroll];
#pragma unroll
      for (int u = 0; u < kSelUnroll; ++u) x[u] = sc[min(i0 + u * T, stop - 1)];
#pragma unroll
      for (int u = 0; u < kSelUnroll; ++u)
        if (i0 + u * T < stop) f(x[u]);
    }
  }
}

// Exclusive prefix sum over a workgroup of T threads (thread order); *total
// gets the sum.  s_wave holds T/64 entries.
template <int T>
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* s_wave, uint32_t* total) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  uint32_t incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t u = __shfl_up(incl, off);
    if (lane >= off) incl += u;
  }
  if (lane == 63) s_wave[wave] = incl;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < T / 64; ++w) {
    const uint32_t t = s_wave[w];
    if (w < wave) before += t;
    all += t;
  }
  __syncthreads();  // s_wave is reused by the next scan
  *total = all;
  return before + incl - v;
}

// What the emission keeps: key k iff k > thresh, or k == thresh and fewer than
// need_eq ties precede it in the segment.  `all_ties`: every tie is kept (the
// usual case, one key at the threshold), so one comparison k >= thresh decides.
struct Keep {
  uint32_t thresh, need_eq;
  bool all_ties;
  int64_t* out;  // the row of kept indices; slots past `budget` are not written
  int out_base, budget;
};

__device__ __forceinline__ void emit_one(const Keep& kp, int64_t i, uint32_t k, uint32_t g, uint32_t e) {
  if (k > kp.thresh || (k == kp.thresh && e < kp.need_eq)) {
    const uint32_t slot = kp.out_base + g + min(e, kp.need_eq);
    if (slot < static_cast<uint32_t>(kp.budget)) kp.out[slot] = i;
  }
}

// Inclusive prefix sum over a wave's lanes: row shifts inside the rows of 16,
// then each row's last lane into the next row and row 1's into rows 2 and 3
// (VALU only; the same scan by lane exchanges is six LDS round trips).
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v) {
  int x = static_cast<int>(v);
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1, 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2, 3
  return static_cast<uint32_t>(x);
}

// One tile of the ordered emission by a workgroup of T threads: wave w holds
// words [64 words w, 64 words (w + 1)) of the tile, lane l of it words l,
// 64 + l, ... (coalesced, and wave, word, lane order is index order); words
// from n_words on are not part of the segment.  A word's count is packed
// (kept, ties apart unless all_ties); per word one scan over the lanes, and one
// total per wave through LDS.  first: index of the tile's first score.  g_run,
// e_run: keys > thresh and == thresh before the tile; with all_ties both kinds
// count in g_run.
template <int T, int K>
__device__ __forceinline__ void emit_tile(const Keep& kp, const f32x4 (&x)[K], int words, int n_words, int64_t first,
                                          uint32_t* s_wave, uint32_t* g_run, uint32_t* e_run) {
  static_assert(T * K * 4 < 65536, "a tile's counts fit 16 bits each");
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int w0 = wave * 64 * words + lane;
  const uint32_t tie = kp.all_ties ? 1u : 65536u;
  uint32_t before[K];  // packed counts of the wave's earlier words, this one's earlier lanes
  uint32_t mine = 0;
#pragma unroll
  for (int u = 0; u < K; ++u) {
    if (u < words) {
      uint32_t c = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t k = float_key(x[u][q]);
        c += k > kp.thresh ? 1u : (k == kp.thresh ? tie : 0u);
      }
      c = w0 + 64 * u < n_words ? c : 0u;
      const uint32_t incl = wave_inclusive_scan(c);
      before[u] = mine + incl - c;
      mine += __builtin_amdgcn_readlane(incl, 63);
    }
  }
  if (lane == 0) s_wave[wave] = mine;
  __syncthreads();
  uint32_t base = 0, all = 0;
#pragma unroll
  for (int w = 0; w < T / 64; ++w) {
    const uint32_t c = s_wave[w];
    if (w < wave) base += c;
    all += c;
  }
  if (kp.all_ties) {
    const uint32_t slot0 = kp.out_base + *g_run + base;
#pragma unroll
    for (int u = 0; u < K; ++u) {
      if (u < words && w0 + 64 * u < n_words) {
        uint32_t slot = slot0 + before[u];
        const int64_t i0 = first + 4 * static_cast<int64_t>(w0 + 64 * u);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const bool take = float_key(x[u][q]) >= kp.thresh;
          if (take && slot < static_cast<uint32_t>(kp.budget)) kp.out[slot] = i0 + q;
          slot += take;
        }
      }
    }
  } else {
#pragma unroll
    for (int u = 0; u < K; ++u) {
      if (u < words && w0 + 64 * u < n_words) {
        uint32_t g = *g_run + ((base + before[u]) & 0xFFFFu), e = *e_run + ((base + before[u]) >> 16);
        const int64_t i0 = first + 4 * static_cast<int64_t>(w0 + 64 * u);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t k = float_key(x[u][q]);
          emit_one(kp, i0 + q, k, g, e);
          g += k > kp.thresh;
          e += k == kp.thresh;
        }
      }
    }
  }
  *g_run += all & 0xFFFFu;
  *e_run += all >> 16;
}

// Counts `n` of three scores before or after the words and, in thread 0, emits them.
__device__ __forceinline__ void emit_ends(const Keep& kp, float x0, float x1, float x2, int n, int64_t first,
                                          uint32_t* g_run, uint32_t* e_run) {
  const float x[3] = {x0, x1, x2};
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    if (i < n) {
      const uint32_t k = float_key(x[i]);
      if (threadIdx.x == 0) emit_one(kp, first + i, k, *g_run, kp.all_ties ? 0u : *e_run);
      const bool eq = k == kp.thresh;
      *g_run += k > kp.thresh || (kp.all_ties && eq);
      if (!kp.all_ties) *e_run += eq;
    }
  }
}

// Ordered emission of [start, stop) by a workgroup of T threads, given the
// numbers g_run, e_run of keys > thresh and == thresh before `start` in the
// segment (all_ties: their sum in g_run), in tiles of T * kEmitWords float4
// words; the up to three scores before the first 16-byte boundary and after
// the last are counted by every thread and written by thread 0.
template <int T>
__device__ __forceinline__ void emit_range(const Keep& kp, const float* sc, int64_t start, int64_t stop, uint32_t g_run, uint32_t e_run,
                           uint32_t* s_wave) {
  const int64_t misalign = (reinterpret_cast<uintptr_t>(sc + start) >> 2) & 3;
  const int64_t head = min((4 - misalign) & 3, stop - start);
  const int64_t body = start + head;
  const int64_t n4 = (stop - body) >> 2;
  const int64_t tail0 = body + 4 * n4;
  float ends[6];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    ends[i] = sc[min(start + i, stop - 1)];
    ends[3 + i] = sc[min(tail0 + i, stop - 1)];
  }
  emit_ends(kp, ends[0], ends[1], ends[2], static_cast<int>(head), start, &g_run, &e_run);
  const f32x4* v = reinterpret_cast<const f32x4*>(sc + body);
  constexpr int64_t kTile = static_cast<int64_t>(T) * kEmitWords;
  const int w0 = (threadIdx.x >> 6) * 64 * kEmitWords + (threadIdx.x & 63);
  for (int64_t t0 = 0; t0 < n4; t0 += kTile) {
    f32x4 x[kEmitWords];
    const int left = static_cast<int>(min(n4 - t0, kTile));
#pragma unroll
    for (int u = 0; u < kEmitWords; ++u) x[u] = v[t0 + min(w0 + 64 * u, left - 1)];  // in range; surplus words are masked
    emit_tile<T, kEmitWords>(kp, x, kEmitWords, left, body + 4 * t0, s_wave, &g_run, &e_run);
    __syncthreads();  // s_wave is reused by the next tile
  }
  emit_ends(kp, ends[3], ends[4], ends[5], static_cast<int>(stop - tail0), tail0, &g_run, &e_run);
}

// ------------------------------------------------- one workgroup per job --

// Segments whose aligned body has at most kCacheWords float4 words a thread
// (16 384 scores at 1024 threads) are read once, into registers, in the
// emission's layout with as few words a thread as hold the segment.
constexpr int kCacheWords = 4;

// The threshold by value bins: a range of the scores is cut into kBins equal
// bins, one histogram of which names the bin that holds the K-th largest score;
// that bin's keys (a few dozen of 16 K aggregated scores) are gathered and
// ranked exactly against each other.  bin(x) = trunc(clamp((hi - x) * scale))
// is a composition of roundings that never increase, so bins keep the order of
// the keys, and any range is right: scores past it, infinities among them,
// count in the end bins.  One walk over scores that spread over many bins,
// where a radix pass on the sign and exponent sends most lanes of a wave to the
// same two counters, four times over.  Where the threshold's bin holds more than
// kMaxCand keys, it is ties of one key (tokens without a score among them) or
// is cut again (hard_threshold).  One workgroup's instructions per score bound
// this kernel (1024 threads on one CU), not its loads.
//
// Microseconds of one 4096-score sequence, 16 x 16384, one of 40000, against
// four radix passes: normal scores 7.8 / 11.3 / 23.4 (radix 11.1 / 19.8 / 39.8),
// with an outlier of 1e30 or one -inf 7.8 / 11.3 / 24, 70% -inf 11.4 / 13.6 / 30
// (12.2 / 19.8 / 39.7), Cauchy 8.2 / 15.6 / 29 (11 / 19.5 / 39), exp(3 normal)
// 10.7 / 18.7 / 33 (11 / 18.6 / 38), two values 11.3 / 17.9 / 36 (13 / 25 / 51),
// clipped at one standard deviation 7.7 / 11.6 / 33 (11 / 20 / 47); only zeros
// of both signs take longer, 18 / 31 / 59 (13 / 25 / 52).
constexpr int kBins = 2048;
constexpr int kBinBits = 11;
constexpr int kMaxCand = 1024;
constexpr int kRangeGroups = 16;  // of lanes, see select_segment
constexpr int kRangeWaves = kSelThreads / 64 / (64 / kRangeGroups);
static_assert(kBins == 1 << kBinBits && kBins == 2 * kSelThreads, "a thread owns two bins of the scan");
constexpr int kMaxCompared = 256;  // candidates compared with each other, see rank_candidates
static_assert(kMaxCompared <= kSplitThreads && kMaxCompared < kMaxCand, "a thread holds one of them");

constexpr uint32_t kMinusInf = 0xff800000u;  // bits; NaNs with the sign set are above

struct Picked {
  uint32_t thresh, need_eq, ties;  // key of the K-th largest score, its ties to keep, all its ties
};

__device__ __forceinline__ float key_float(uint32_t key) {
  return __uint_as_float((key & 0x80000000u) ? key ^ 0x80000000u : ~key);
}

__device__ __forceinline__ bool finite(float x) { return fabsf(x) <= 3.402823466e38f; }

// Smallest and largest key of a set of scores, smallest and largest finite one.
struct Range {
  uint32_t kl, kh;
  float lo, hi;
};

// The key with rank `need` from the top of the `count` <= kMaxCand keys of cand
// (in LDS, 16-byte aligned), written to `out`.  A few dozen keys, the usual
// number, are compared with each other.  More are held by one wave, 16 a lane
// at most, which sets the threshold's bits from the top by the number of keys
// at or above each trial: up to 4 us, where comparing 800 with each other took
// 25 of the whole workgroup.  Every thread calls it.
template <int T>
__device__ __forceinline__ void rank_candidates(uint32_t* cand, uint32_t count, uint32_t need, Picked* out) {
  constexpr int kWords = kMaxCand / 64;
  const uint32_t padded = (count + 3) & ~3u;  // with the smallest key, corrected below
  if (count <= kMaxCompared && threadIdx.x < padded - count) cand[count + threadIdx.x] = 0u;
  __syncthreads();  // the keys are written
  if (count <= kMaxCompared) {
    if (threadIdx.x < count) {
      const uint32_t mine = cand[threadIdx.x];
      uint32_t g = 0, e = mine == 0u ? count - padded : 0u;
      for (uint32_t k = 0; k < padded; k += 4) {
        const uint4 o = *reinterpret_cast<const uint4*>(cand + k);
        g += (o.x > mine) + (o.y > mine) + (o.z > mine) + (o.w > mine);
        e += (o.x == mine) + (o.y == mine) + (o.z == mine) + (o.w == mine);
      }
      if (g < need && need <= g + e) *out = Picked{mine, need - g, e};  // equal keys write the same
    }
  } else if (threadIdx.x < 64) {
    const uint32_t lane = threadIdx.x;
    const int words = static_cast<int>((count + 63) / 64);
    uint32_t key[kWords];
#pragma unroll
    for (int w = 0; w < kWords; ++w) key[w] = 64 * w + lane < count ? cand[64 * w + lane] : 0u;
    auto at_least = [&](uint32_t trial) {
      uint32_t n = 0;
#pragma unroll
      for (int w = 0; w < kWords; w += 4) {
        if (w >= words) break;
#pragma unroll
        for (int v = w; v < w + 4; ++v) n += static_cast<uint32_t>(__popcll(__ballot(key[v] >= trial)));
      }
      return n;
    };
    const uint32_t base = __builtin_amdgcn_readfirstlane(key[0]);
    uint32_t diff = 0;  // bits in which keys differ; those above are the threshold's
#pragma unroll
    for (int w = 0; w < kWords; ++w) diff |= 64 * w + lane < count ? key[w] ^ base : 0u;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) diff |= __shfl_xor(diff, off);
    diff = __builtin_amdgcn_readfirstlane(diff);
    uint32_t bit = diff ? 0x80000000u >> __clz(static_cast<int>(diff)) : 0u;
    uint32_t thresh = bit ? base & ~(2 * bit - 1) : base;
#pragma unroll 1
    for (; bit; bit >>= 1)
      if (at_least(thresh | bit) >= need) thresh |= bit;
    // Padding equals a threshold of zero only.
    const uint32_t more = diff == 0 || thresh == 0xffffffffu ? 0u : at_least(thresh + 1);
    const uint32_t from = diff == 0 || thresh == 0u ? count : at_least(thresh);
    if (lane == 0) *out = Picked{thresh, need - more, from - more};
  }
  __syncthreads();
}

// The union of the threads' ranges, by a workgroup of T threads.
template <int T>
__device__ __forceinline__ Range meet_ranges(Range r) {
  __shared__ Range waves[T / 64];
  auto meet = [&](int off) {
    r.kl = min(r.kl, __shfl_xor(r.kl, off));
    r.kh = max(r.kh, __shfl_xor(r.kh, off));
    r.lo = fminf(r.lo, __shfl_xor(r.lo, off));
    r.hi = fmaxf(r.hi, __shfl_xor(r.hi, off));
  };
#pragma unroll 1
  for (int off = 32; off >= 1; off >>= 1) meet(off);
  if ((threadIdx.x & 63) == 0) waves[threadIdx.x >> 6] = r;
  __syncthreads();
  r = waves[threadIdx.x & (T / 64 - 1)];
#pragma unroll 1
  for (int off = T / 128; off >= 1; off >>= 1) meet(off);
  __syncthreads();  // written again by the next call
  return r;
}

// The range of the scores that `member` accepts, by a workgroup of T threads.
template <int T, typename F>
__device__ __forceinline__ Range member_range(const float* sc, int64_t start, int64_t stop, F&& member) {
  Range r{0xffffffffu, 0u, INFINITY, -INFINITY};
  for_each_score_rarely<T>(sc, start, stop, [&](float x) {
    const uint32_t key = float_key(x);
    if (member(x, key)) {
      r.kl = min(r.kl, key);
      r.kh = max(r.kh, key);
      r.lo = fminf(r.lo, finite(x) ? x : INFINITY);
      r.hi = fmaxf(r.hi, finite(x) ? x : -INFINITY);
    }
  });
  return meet_ranges<T>(r);
}

// The bins of a workgroup of T threads, kBinCopies counters each: lane l counts
// in copy l % kBinCopies, so that lanes whose scores share a bin (ties, the
// crowded end of a skewed range) wait for each other in smaller groups.  One
// counter where chunks' workgroups share a CU, and its LDS.
template <int T>
constexpr int kBinCopies = T == kSelThreads ? 4 : 1;
template <int T>
__device__ __forceinline__ uint32_t* shared_bins() {
  __shared__ __attribute__((aligned(16))) uint32_t bins[kBins * kBinCopies<T>];
  return bins;
}
__device__ __forceinline__ uint32_t* shared_candidates() {
  __shared__ __attribute__((aligned(16))) uint32_t cand[kMaxCand];
  return cand;
}
template <int T>
__device__ __forceinline__ void clear_bins() {
  for (int i = threadIdx.x; i < kBins * kBinCopies<T> / 4; i += T)
    reinterpret_cast<uint4*>(shared_bins<T>())[i] = make_uint4(0, 0, 0, 0);
}
template <int T>
__device__ __forceinline__ void count_bin(int bin) {
  atomicAdd(&shared_bins<T>()[kBinCopies<T> * bin + (threadIdx.x & (kBinCopies<T> - 1))], 1u);
}
template <int T>
__device__ __forceinline__ uint32_t bin_total(int bin) {
  if constexpr (kBinCopies<T> == 1) return shared_bins<T>()[bin];
  static_assert(kBinCopies<T> == 1 || kBinCopies<T> == 4, "read as one word");
  const uint4 c = reinterpret_cast<const uint4*>(shared_bins<T>())[bin];
  return c.x + c.y + c.z + c.w;
}

// The need-th largest of the `count` scores of [start, stop) whose keys lie in
// [r.kl, r.kh], by a workgroup of T threads: that range is cut into kBins bins
// until at most kMaxCand keys share the threshold's bin, or it is one key.  Up
// to twice the bins are equal in value (the end bins hold what is not finite):
// what an outlier's bin holds spreads well.  Then they are equal in keys, which
// takes kBinBits bits off the range a turn.
template <int T>
__device__ __noinline__ Picked pick_in_range(const float* sc, int64_t start, int64_t stop, uint32_t need, Range r,
                                             uint32_t count) {
  constexpr int kOwn = kBins / T;  // bins a thread owns in the scan
  uint32_t* cand = shared_candidates();
  __shared__ uint32_t s_wave[T / 64];
  __shared__ uint32_t s_bin, s_need, s_count, s_filled;
  __shared__ Picked s_picked;
  const int tid = threadIdx.x;
  for (int turn = 0; r.kl != r.kh; ++turn) {
    const uint32_t kl = r.kl, span = r.kh - r.kl;
    const float lo = 0.5f * r.lo;  // halves: no range overflows
    const float scale = (kBins - 2 - 1.0f / 512.0f) / (0.5f * r.hi - lo);
    const bool values = turn < 2 && r.hi > r.lo && scale > 0.0f && scale < INFINITY;
    const int shift = max(32 - __clz(static_cast<int>(span)) - kBinBits, 0);
    auto bin_of = [&](float x, uint32_t key) -> int {
      if (!values) return static_cast<int>((key - kl) >> shift);
      if (!finite(x)) return (key >> 31) ? kBins - 1 : 0;
      return 1 + static_cast<int>((0.5f * x - lo) * scale);
    };
    clear_bins<T>();
    if (tid == 0) s_filled = 0;
    __syncthreads();
    for_each_score_rarely<T>(sc, start, stop, [&](float x) {
      const uint32_t key = float_key(x);
      if (key - kl <= span) count_bin<T>(bin_of(x, key));
    });
    __syncthreads();
    // Thread order is falling order of the bins.
    uint32_t c[kOwn], own = 0, total;
#pragma unroll
    for (int q = 0; q < kOwn; ++q) own += c[q] = bin_total<T>(kBins - 1 - kOwn * tid - q);
    uint32_t above = block_exclusive_scan<T>(own, s_wave, &total);
#pragma unroll
    for (int q = 0; q < kOwn; ++q) {
      if (above < need && need <= above + c[q]) {
        s_bin = static_cast<uint32_t>(kBins - 1 - kOwn * tid - q);
        s_need = need - above;
        s_count = c[q];
      }
      above += c[q];
    }
    __syncthreads();
    const int bin = static_cast<int>(s_bin);
    need = s_need;
    count = s_count;
    auto member = [&](float x, uint32_t key) { return key - kl <= span && bin_of(x, key) == bin; };
    if (count <= kMaxCand) {
      for_each_score_rarely<T>(sc, start, stop, [&](float x) {
        const uint32_t key = float_key(x);
        if (member(x, key)) cand[atomicAdd(&s_filled, 1u)] = key;
      });
      rank_candidates<T>(cand, count, need, &s_picked);
      return s_picked;
    }
    if (!values && shift == 0) return Picked{kl + static_cast<uint32_t>(bin), need, count};
    r = member_range<T>(sc, start, stop, member);
  }
  return Picked{r.kl, need, count};
}

// The first bins, from the largest scores down: a NaN counts in bin 0, where it
// belongs unless its sign is set.
__device__ __forceinline__ int value_bin(float x, float hi, float scale) {
  return static_cast<int>(__builtin_amdgcn_fmed3f((hi - x) * scale, 0.0f, static_cast<float>(kBins - 1)));
}

// The threshold of scores that the first set of bins did not separate: the
// need-th largest of the `count` scores with keys in [kl, kh], kl and kh among
// them, or (kl > kh) of all scores.  Out of line, as select_long below: what
// most calls run stays small in the instruction cache.
__device__ __noinline__ Picked hard_threshold(const float* sc, int64_t start, int64_t stop, uint32_t need, uint32_t count,
                                              uint32_t kl, uint32_t kh) {
  Range r{kl, kh, key_float(kl), key_float(kh)};
  if (kl > kh || !finite(r.lo) || !finite(r.hi))
    r = member_range<kSelThreads>(sc, start, stop, [&](float, uint32_t key) { return kl > kh || key - kl <= kh - kl; });
  return pick_in_range<kSelThreads>(sc, start, stop, need, r, count);
}

// Keeps the `keep` largest scores of [start, stop), their indices written from
// slot out_base on.  CACHED: at most kCacheWords words a thread.
template <bool CACHED>
__device__ __forceinline__ void select_segment(const float* sc, int64_t start, int64_t stop, uint32_t keep, int64_t* out,
                                               int out_base, int budget) {
  uint32_t* cand = shared_candidates();
  __shared__ uint32_t s_bin, s_need, s_count, s_filled, s_tie, s_sums[3];
  __shared__ Picked s_picked;
  __shared__ uint32_t s_wave[kSelThreads / 64];
  __shared__ bool s_odd[kSelThreads / 64];
  __shared__ float s_range[2][kSelThreads / 64][kRangeGroups];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int64_t misalign = (reinterpret_cast<uintptr_t>(sc + start) >> 2) & 3;
  const int64_t head = min((4 - misalign) & 3, stop - start);
  const int64_t body = start + head;
  const int64_t n4 = (stop - body) >> 2;
  const int64_t tail0 = body + 4 * n4;
  const f32x4* v = reinterpret_cast<const f32x4*>(sc + body);
  const int words = CACHED ? static_cast<int>((n4 + kSelThreads - 1) / kSelThreads) : 0;
  const int n_words = static_cast<int>(CACHED ? n4 : 0);
  const int w0 = wave * 64 * words + lane;
  f32x4 cx[kCacheWords];
  float ends[6];  // the up to three scores before the first and after the last 16-byte boundary
  if constexpr (CACHED) {
#pragma unroll
    for (int u = 0; u < kCacheWords; ++u)
      if (u < words) cx[u] = v[min(w0 + 64 * u, n_words - 1)];  // surplus words are masked
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      ends[e] = sc[min(start + e, stop - 1)];
      ends[3 + e] = sc[min(tail0 + e, stop - 1)];
    }
  }
  const int n_head = static_cast<int>(head), n_tail = static_cast<int>(stop - tail0);
  float my_end = 0.0f;  // lane e < 3 counts the head's score e, lane 3 + e the tail's
  if constexpr (CACHED) {
#pragma unroll
    for (int e = 0; e < 6; ++e) my_end = tid == e ? ends[e] : my_end;
  }
  // f(score) for every score of the segment, each by one thread.
  auto walk = [&](auto&& f) {
    if constexpr (!CACHED) {
      for_each_score<kSelThreads>(sc, start, stop, f);
    } else {
#pragma unroll
      for (int u = 0; u < kCacheWords; ++u)
        if (u < words && w0 + 64 * u < n_words) {
#pragma unroll
          for (int q = 0; q < 4; ++q) f(cx[u][q]);
        }
      if (tid < 6 && (tid < 3 ? tid < n_head : tid - 3 < n_tail)) f(my_end);
    }
  };

  // The bins' range, from the smallest and largest score of each of
  // kRangeGroups groups (every kRangeGroups-th lane): the largest of the
  // smallest to the smallest of the largest, so that a few outliers or
  // infinities do not stretch it.  odd: one of the scores is a NaN with its
  // sign set, which has no place among these bins.
  clear_bins<kSelThreads>();
  if (tid == 0) s_filled = s_sums[0] = s_sums[1] = s_sums[2] = 0;
  float lo = INFINITY, hi = -INFINITY;
  uint32_t bits = 0;
  walk([&](float x) {
    lo = fminf(lo, x);
    hi = fmaxf(hi, x);
    bits = max(bits, __float_as_uint(x));
  });
  bool odd = false;
  if (__any(bits >= kMinusInf)) {  // not from tokens without a score
    lo = INFINITY;
    walk([&](float x) { lo = fminf(lo, x == -INFINITY ? INFINITY : x); });
    odd = __any(bits > kMinusInf);
  }
#pragma unroll
  for (int off = 32; off >= kRangeGroups; off >>= 1) {
    lo = fminf(lo, __shfl_xor(lo, off));
    hi = fmaxf(hi, __shfl_xor(hi, off));
  }
  if (lane < kRangeGroups) {
    s_range[0][wave][lane] = lo;
    s_range[1][wave][lane] = hi;
  }
  if (lane == 0) s_odd[wave] = odd;
  __syncthreads();
  odd = __any(s_odd[lane & (kSelThreads / 64 - 1)]);
  {
    // Lane l: group l % kRangeGroups, a quarter of the waves.
    const int group = lane & (kRangeGroups - 1), w0 = (lane / kRangeGroups) * kRangeWaves;
    lo = s_range[0][w0][group], hi = s_range[1][w0][group];
#pragma unroll
    for (int w = 1; w < kRangeWaves; ++w) {
      lo = fminf(lo, s_range[0][w0 + w][group]);
      hi = fmaxf(hi, s_range[1][w0 + w][group]);
    }
  }
#pragma unroll
  for (int off = 32; off >= kRangeGroups; off >>= 1) {
    lo = fminf(lo, __shfl_xor(lo, off));
    hi = fmaxf(hi, __shfl_xor(hi, off));
  }
  if (lo > hi) lo = -INFINITY, hi = INFINITY;  // a group without scores
  static_assert(kRangeGroups == 16, "a row of lanes holds every group");
  lo = fmaxf(lo, dpp_quad_xor1(lo)), hi = fminf(hi, dpp_quad_xor1(hi));
  lo = fmaxf(lo, dpp_quad_xor2(lo)), hi = fminf(hi, dpp_quad_xor2(hi));
  lo = fmaxf(lo, dpp_row_half_mirror(lo)), hi = fminf(hi, dpp_row_half_mirror(hi));
  lo = fmaxf(lo, dpp_row_mirror(lo)), hi = fminf(hi, dpp_row_mirror(hi));
  if (lo > hi) {  // groups apart from each other
    const float t = lo;
    lo = hi;
    hi = t;
  }
  const float scale = static_cast<float>(kBins) / (hi - lo);
  auto bin_of = [&](float x) { return value_bin(x, hi, scale); };
  Picked picked{0u, 0u, 0u};
  // The same for every thread.  A range past float32 gives a scale of zero, one
  // of no width an infinity.
  bool found = !odd && hi > lo && scale > 0.0f && scale < INFINITY;
  // Where the bins leave off: the threshold's rank among `among` scores with
  // keys in [kl, kh] (all scores).
  uint32_t need = keep, among = static_cast<uint32_t>(stop - start), kl = 0xffffffffu, kh = 0;
  if (found) {
    walk([&](float x) { count_bin<kSelThreads>(bin_of(x)); });
    __syncthreads();
    // Thread t owns bins 2t and 2t + 1, in falling order of the scores.
    const uint32_t c0 = bin_total<kSelThreads>(2 * tid), c1 = bin_total<kSelThreads>(2 * tid + 1);
    uint32_t total;
    uint32_t above = block_exclusive_scan<kSelThreads>(c0 + c1, s_wave, &total);
    if (above < keep && keep <= above + c0 + c1) {
      const bool first = keep <= above + c0;
      if (!first) above += c0;
      s_bin = static_cast<uint32_t>(2 * tid + (first ? 0 : 1));
      s_need = keep - above;
      s_count = first ? c0 : c1;
    }
    __syncthreads();
    const int bin = static_cast<int>(s_bin);
    const uint32_t count = s_count, rank = s_need;
    if (count <= kMaxCand) {
      walk([&](float x) {
        if (bin_of(x) == bin) cand[atomicAdd(&s_filled, 1u)] = float_key(x);
      });
      rank_candidates<kSelThreads>(cand, count, rank, &s_picked);
      picked = s_picked;
    } else {
      // Tokens without a score (-inf) fill the bin, or ties of one key (probably
      // that of the member found first) beside a few others, or it has to be cut
      // again.
      walk([&](float x) {
        if (x != -INFINITY && bin_of(x) == bin) s_tie = float_key(x);
      });
      __syncthreads();
      const uint32_t tie = s_tie;
      uint32_t none = 0, equal = 0, higher = 0;
      walk([&](float x) {
        if (bin_of(x) == bin) {
          const uint32_t key = float_key(x);
          if (x == -INFINITY) {
            ++none;
          } else if (key == tie) {
            ++equal;
          } else {
            higher += key > tie;
            kl = min(kl, key);
            kh = max(kh, key);
          }
        }
      });
#pragma unroll 1
      for (int off = 32; off >= 1; off >>= 1) {
        none += __shfl_xor(none, off);
        equal += __shfl_xor(equal, off);
        higher += __shfl_xor(higher, off);
      }
      if (lane == 0) {
        atomicAdd(&s_sums[0], none);
        atomicAdd(&s_sums[1], equal);
        atomicAdd(&s_sums[2], higher);
      }
      const Range r = meet_ranges<kSelThreads>(Range{kl, kh, 0.0f, 0.0f});
      none = s_sums[0], equal = s_sums[1], higher = s_sums[2];
      need = rank;
      among = count - none;
      found = true;
      if (need > among) {
        picked = Picked{float_key(-INFINITY), need - among, none};
      } else if (higher < need && need <= higher + equal) {
        picked = Picked{tie, need - higher, equal};
      } else if (r.kl == r.kh) {  // the others are one key
        picked = Picked{r.kl, r.kl < tie ? need - equal : need, among - equal};
      } else {
        found = false;
        kl = min(r.kl, tie);
        kh = max(r.kh, tie);
      }
    }
  }
  if (!found) picked = hard_threshold(sc, start, stop, need, among, kl, kh);
  const Keep kp{picked.thresh, picked.need_eq, picked.ties == picked.need_eq, out, out_base, budget};
  if constexpr (CACHED) {
    uint32_t g_run = 0, e_run = 0;
    emit_ends(kp, ends[0], ends[1], ends[2], n_head, start, &g_run, &e_run);
    emit_tile<kSelThreads, kCacheWords>(kp, cx, words, n_words, body, s_wave, &g_run, &e_run);
    emit_ends(kp, ends[3], ends[4], ends[5], n_tail, tail0, &g_run, &e_run);
  } else {
    emit_range<kSelThreads>(kp, sc, start, stop, 0u, 0u, s_wave);
  }
}

// Longer segments re-read the scores in every walk.  Out of line: the short
// form's code then stays small in the instruction cache.
__device__ __noinline__ void select_long(const float* sc, int64_t start, int64_t stop, uint32_t keep, int64_t* out,
                                         int out_base, int budget) {
  select_segment<false>(sc, start, stop, keep, out, out_base, budget);
}

__global__ __launch_bounds__(kSelThreads) void select_kernel(SelectArgs a) {
  const int b = blockIdx.y;
  const int seg = blockIdx.x;
  const Job j = make_job(a, b, seg);
  int64_t* out = a.keep + static_cast<int64_t>(b) * a.keep_stride;
  if (!fill_fixed(a, j, seg, out, threadIdx.x, kSelThreads)) return;
  const float* sc = a.scores + a.token_offsets[b];
  const uint32_t keep = static_cast<uint32_t>(j.s.keep);
  const int out_base = static_cast<int>(j.out_base);
  if (j.s.stop - j.s.start <= 4 * kCacheWords * kSelThreads)
    select_segment<true>(sc, j.s.start, j.s.stop, keep, out, out_base, a.budget);
  else
    select_long(sc, j.s.start, j.s.stop, keep, out, out_base, a.budget);
}

// ------------------------------------------------------ split over chunks --

// The threshold of a long segment, in three launches (seven when four radix
// passes named it, a clear before and a count after: 4 x 130816 scores 37.7 us
// against 19.7 now).  Bins are equal cells of a range taken from a sample, so no
// launch has to find the range first: any range is right, since scores past it
// count in the last bins, and the bins only have to keep the order of the keys.  Every chunk stores a histogram of its own
// (no atomics, nothing to clear), every chunk of the second launch adds them
// all, and the threshold's bin holds some hundred keys, ranked exactly.  More
// than kSplitCand keys there are usually ties of one key and a few others: the
// second launch counts the keys equal to and above one of them.  Where that does
// not name the threshold, every chunk's workgroup bins the whole segment's keys
// of that bin again (ten times the usual time, so the bins' range is chosen to
// make it rare).
//
// Microseconds of 4 x 131072 scores, keep 4608 of each, against the seven
// launches: normal 20 (38.4), an outlier of 1e30 20 (38.5), 70% -inf 21 (38.5),
// Cauchy 19 (38.4), exp(3 normal) 19 (38.5), two values 25 (39), one value 26
// (39).  262144 scores of exp(3 normal) of which 100000 are kept, 8000 in the
// threshold's bin, take 270 (42).
constexpr int kSplitBins = 1024;
constexpr int kSplitCand = 4096;
constexpr int kSplitRanked = 1024;  // candidates ranked against each other; more are binned first
constexpr int kSplitSamples = 1024;
static_assert(kSplitRanked <= kMaxCand, "one wave ranks them");
static_assert(kSplitBins == 4 * kSplitThreads, "a thread owns four bins");

// Per-job scratch (in the caller's workspace), written before it is read by
// every call.
struct SplitState {
  float lo, scale;             // bin of x: (x - lo) * scale
  uint32_t rank, count;        // the threshold's rank from the top of its bin, keys in that bin
  // Where the bin is too full for cand: one of its keys (a sample's, probably the
  // ties'), and per chunk the keys equal to it and above it, and the smallest and
  // largest of the others.
  uint32_t tie, reserved[3];
  uint32_t equal[kSplitMaxChunks];
  uint32_t higher[kSplitMaxChunks];
  uint32_t least[kSplitMaxChunks];
  uint32_t most[kSplitMaxChunks];
  uint32_t above[kSplitMaxChunks];   // a chunk's keys in higher bins
  uint32_t before[kSplitMaxChunks];  // candidates of the chunks before
  uint32_t hist[kSplitMaxChunks][kSplitBins];
  float cand[kSplitCand];      // the bin's scores, chunk after chunk
};
static_assert(sizeof(SplitState) % 16 == 0, "jobs' states stay aligned");

__host__ __device__ inline int64_t split_chunk_len(int64_t len) {
  int64_t cs = (len + kSplitMaxChunks - 1) / kSplitMaxChunks;
  if (cs < kSplitChunk) cs = kSplitChunk;
  return (cs + 3) & ~int64_t(3);
}

__host__ __device__ inline int split_chunks(int64_t len) {
  return len <= 0 ? 0 : static_cast<int>((len + split_chunk_len(len) - 1) / split_chunk_len(len));
}

__device__ __forceinline__ SplitState* split_state(const SelectArgs& a, int b, int seg) {
  return static_cast<SplitState*>(a.state) + static_cast<int64_t>(b) * a.segments + seg;
}

// Place of sample i in a segment of len scores.
__device__ __forceinline__ int64_t sample_at(int64_t i, int64_t len) { return i * len / kSplitSamples; }

// Order-preserving bin of a score.  Infinities and NaNs have the end bins to
// themselves, by their sign (many tokens without a score are then one key); a
// scale of zero puts every finite score in bin 1.
__device__ __forceinline__ int split_bin(float x, float lo, float scale) {
  if (!finite(x)) return (float_key(x) >> 31) ? kSplitBins - 1 : 0;
  return static_cast<int>(fminf(fmaxf((x - lo) * scale, 1.0f), static_cast<float>(kSplitBins - 2)));
}

// The chunk of this workgroup (grid: chunks, segments, n_seq).
struct Chunk {
  Job j;
  int c;
  int chunks;
  int64_t start, stop;
  bool live;  // the job needs a threshold and the chunk exists
};

__device__ __forceinline__ Chunk make_chunk(const SelectArgs& a) {
  Chunk k;
  k.c = blockIdx.x;
  k.j = make_job(a, blockIdx.z, blockIdx.y);
  const int64_t len = k.j.s.stop - k.j.s.start;
  k.chunks = split_chunks(len);
  k.live = k.j.exists && k.j.s.keep > 0 && len > k.j.s.keep && k.c < k.chunks;
  const int64_t cs = split_chunk_len(len);
  k.start = k.j.s.start + k.c * cs;
  k.stop = min(k.j.s.stop, k.start + cs);
  return k;
}

// Launch 1: protected windows and segments kept whole (chunk 0), the bins'
// range, the chunk's histogram.
__global__ __launch_bounds__(kSplitThreads) void select_split_bins_kernel(SelectArgs a) {
  __shared__ __attribute__((aligned(16))) uint32_t bins[kSplitBins];
  __shared__ float s_range[2][kSplitThreads / 64][kRangeGroups];
  const int tid = threadIdx.x;
  const Chunk k = make_chunk(a);
  if (k.c == 0)
    fill_fixed(a, k.j, blockIdx.y, a.keep + static_cast<int64_t>(blockIdx.z) * a.keep_stride, tid, kSplitThreads);
  if (!k.live) return;  // the whole workgroup
  const float* sc = a.scores + a.token_offsets[blockIdx.z];
  const int64_t len = k.j.s.stop - k.j.s.start;
  for (int i = tid; i < kSplitBins; i += kSplitThreads) bins[i] = 0;
  float lo = INFINITY, hi = -INFINITY;
  float x[kSplitSamples / kSplitThreads];
#pragma unroll
  for (int u = 0; u < kSplitSamples / kSplitThreads; ++u)
    x[u] = sc[k.j.s.start + sample_at(tid + kSplitThreads * u, len)];
#pragma unroll
  for (int u = 0; u < kSplitSamples / kSplitThreads; ++u) {
    lo = fminf(lo, finite(x[u]) ? x[u] : INFINITY);
    hi = fmaxf(hi, finite(x[u]) ? x[u] : -INFINITY);
  }
  // Smallest and largest sample of each group of lanes l % kRangeGroups.
  lo = fminf(lo, __shfl_xor(lo, 32)), hi = fmaxf(hi, __shfl_xor(hi, 32));
  lo = fminf(lo, __shfl_xor(lo, 16)), hi = fmaxf(hi, __shfl_xor(hi, 16));
  const int group = tid & (kRangeGroups - 1);
  if ((tid & 63) < kRangeGroups) {
    s_range[0][tid >> 6][group] = lo;
    s_range[1][tid >> 6][group] = hi;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kSplitThreads / 64; ++w) {
    lo = fminf(lo, s_range[0][w][group]);
    hi = fmaxf(hi, s_range[1][w][group]);
  }
  if (lo > hi) lo = -INFINITY, hi = INFINITY;  // a group without scores
  // The largest of the groups' smallest to the smallest of their largest: a few
  // outliers do not stretch the range.  Of normal scores it ends at about 1.75
  // standard deviations.  The bins reach further, above all at the top, where
  // the threshold of a small budget lies.
  lo = fmaxf(lo, dpp_quad_xor1(lo)), hi = fminf(hi, dpp_quad_xor1(hi));
  lo = fmaxf(lo, dpp_quad_xor2(lo)), hi = fminf(hi, dpp_quad_xor2(hi));
  lo = fmaxf(lo, dpp_row_half_mirror(lo)), hi = fminf(hi, dpp_row_half_mirror(hi));
  lo = fmaxf(lo, dpp_row_mirror(lo)), hi = fminf(hi, dpp_row_mirror(hi));
  const float width = fabsf(hi - lo);  // groups apart from each other: hi < lo
  lo = fminf(lo, hi) - 0.25f * width;
  float scale = kSplitBins / (3.0f * width);
  if (!(width > 0.0f && scale > 0.0f && scale < INFINITY && fabsf(lo) < INFINITY)) {
    lo = 0.0f;
    scale = 0.0f;
  }
  for_each_score<kSplitThreads>(sc, k.start, k.stop, [&](float v) { atomicAdd(&bins[split_bin(v, lo, scale)], 1u); });
  __syncthreads();
  SplitState* st = split_state(a, blockIdx.z, blockIdx.y);
  reinterpret_cast<uint4*>(st->hist[k.c])[tid] = reinterpret_cast<const uint4*>(bins)[tid];
  if (k.c == 0 && tid == 0) {
    st->lo = lo;
    st->scale = scale;
  }
}

// Launch 2: the threshold's bin from all chunks' histograms; the chunk's keys
// of that bin and its number of keys in higher ones.
__global__ __launch_bounds__(kSplitThreads) void select_split_candidates_kernel(SelectArgs a) {
  __shared__ uint32_t s_wave[kSplitThreads / 64];
  __shared__ uint32_t s_bin, s_rank, s_count, s_before, s_filled, s_least, s_most, s_first, s_equal, s_higher;
  const int tid = threadIdx.x;
  const Chunk k = make_chunk(a);
  if (!k.live) return;
  if (tid == 0) {
    s_least = 0xffffffffu;
    s_most = 0;
    s_first = kSplitSamples;
    s_equal = 0;
    s_higher = 0;
  }
  SplitState* st = split_state(a, blockIdx.z, blockIdx.y);
  const uint32_t keep = static_cast<uint32_t>(k.j.s.keep);
  const float lo = st->lo, scale = st->scale;
  // Thread t owns bins top - 4t .. top - 4t - 3: thread order is falling order.
  const int word = kSplitThreads - 1 - tid;
  uint32_t all[4] = {0, 0, 0, 0}, pre[4] = {0, 0, 0, 0}, own[4] = {0, 0, 0, 0};
  uint4 h[kSplitMaxChunks];  // every load in flight at once
#pragma unroll
  for (int c = 0; c < kSplitMaxChunks; ++c) h[c] = reinterpret_cast<const uint4*>(st->hist[min(c, k.chunks - 1)])[word];
#pragma unroll
  for (int c = 0; c < kSplitMaxChunks; ++c) {
    const uint32_t v[4] = {h[c].w, h[c].z, h[c].y, h[c].x};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      all[q] += c < k.chunks ? v[q] : 0u;
      pre[q] += c < k.c ? v[q] : 0u;
      own[q] = c == k.c ? v[q] : own[q];
    }
  }
  if (tid == 0) s_filled = 0;
  uint32_t total;
  uint32_t above = block_exclusive_scan<kSplitThreads>(all[0] + all[1] + all[2] + all[3], s_wave, &total);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (above < keep && keep <= above + all[q]) {
      s_bin = static_cast<uint32_t>(kSplitBins - 1 - 4 * tid - q);
      s_rank = keep - above;
      s_count = all[q];
      s_before = pre[q];
    }
    above += all[q];
  }
  __syncthreads();
  const int bin = static_cast<int>(s_bin);
  const uint32_t count = s_count, before = s_before;
  uint32_t higher = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) higher += kSplitBins - 1 - 4 * tid - q > bin ? own[q] : 0u;
  uint32_t above_here;
  block_exclusive_scan<kSplitThreads>(higher, s_wave, &above_here);
  if (tid == 0) {
    st->above[k.c] = above_here;
    st->before[k.c] = before;
    if (k.c == 0) {
      st->rank = s_rank;
      st->count = count;
    }
  }
  const float* sc = a.scores + a.token_offsets[blockIdx.z];
  if (count <= kSplitCand) {
    for_each_score<kSplitThreads>(sc, k.start, k.stop, [&](float x) {
      if (split_bin(x, lo, scale) == bin) st->cand[before + atomicAdd(&s_filled, 1u)] = x;
    });
    return;
  }
  // The same sample for every chunk: the first in the bin.
  const int64_t len = k.j.s.stop - k.j.s.start;
  float x[kSplitSamples / kSplitThreads];
#pragma unroll
  for (int u = 0; u < kSplitSamples / kSplitThreads; ++u) x[u] = sc[k.j.s.start + sample_at(tid + kSplitThreads * u, len)];
#pragma unroll
  for (int u = kSplitSamples / kSplitThreads - 1; u >= 0; --u) {
    const uint64_t in = __ballot(split_bin(x[u], lo, scale) == bin);
    if (in && (tid & 63) == 0) atomicMin(&s_first, static_cast<uint32_t>(tid + kSplitThreads * u + __ffsll(static_cast<unsigned long long>(in)) - 1));
  }
  __syncthreads();
  const uint32_t tie = s_first < kSplitSamples ? float_key(sc[k.j.s.start + sample_at(s_first, len)]) : 0u;
  uint32_t least = 0xffffffffu, most = 0, equal = 0, above_tie = 0;
  for_each_score<kSplitThreads>(sc, k.start, k.stop, [&](float x) {
    if (split_bin(x, lo, scale) == bin) {
      const uint32_t key = float_key(x);
      if (key == tie) {
        ++equal;
      } else {
        above_tie += key > tie;
        least = min(least, key);
        most = max(most, key);
      }
    }
  });
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    least = min(least, __shfl_xor(least, off));
    most = max(most, __shfl_xor(most, off));
    equal += __shfl_xor(equal, off);
    above_tie += __shfl_xor(above_tie, off);
  }
  if ((tid & 63) == 0) {
    atomicMin(&s_least, least);
    atomicMax(&s_most, most);
    atomicAdd(&s_equal, equal);
    atomicAdd(&s_higher, above_tie);
  }
  __syncthreads();
  if (tid == 0) {
    st->least[k.c] = s_least;
    st->most[k.c] = s_most;
    st->equal[k.c] = s_equal;
    st->higher[k.c] = s_higher;
    if (k.c == 0) st->tie = tie;
  }
}

// Launch 3: the threshold among the candidates, and the chunk's ordered emission.
__global__ __launch_bounds__(kSplitThreads, 4) void select_split_emit_kernel(SelectArgs a) {
  __shared__ __attribute__((aligned(16))) float cand[kSplitCand];
  uint32_t* keys = shared_candidates();
  __shared__ uint32_t s_wave[kSplitThreads / 64];
  __shared__ Picked s_picked;
  const int tid = threadIdx.x;
  const Chunk k = make_chunk(a);
  if (!k.live) return;
  const SplitState* st = split_state(a, blockIdx.z, blockIdx.y);
  const float* sc = a.scores + a.token_offsets[blockIdx.z];
  const uint32_t count = st->count, rank = st->rank;
  Picked p;
  uint32_t g = 0, e = 0;  // this thread's share of the keys > and == the threshold before the chunk
  const uint32_t before = st->before[k.c];
  if (count <= kSplitCand) {
    for (uint32_t i = tid; i < count; i += kSplitThreads) cand[i] = st->cand[i];
    if (count <= kSplitRanked) {
      for (uint32_t i = tid; i < count; i += kSplitThreads) keys[i] = float_key(st->cand[i]);
      rank_candidates<kSplitThreads>(keys, count, rank, &s_picked);
      p = s_picked;
    } else {
      __syncthreads();
      const Range r = member_range<kSplitThreads>(cand, 0, count, [](float, uint32_t) { return true; });
      p = pick_in_range<kSplitThreads>(cand, 0, count, rank, r, count);
    }
    for (uint32_t i = tid; i < before; i += kSplitThreads) {
      const uint32_t key = float_key(cand[i]);
      g += key > p.thresh;
      e += key == p.thresh;
    }
    if (tid < k.c) g += st->above[tid];
  } else {
    const uint32_t tie = st->tie;
    uint32_t least = 0xffffffffu, most = 0, equal = 0, higher = 0, equal_before = 0, higher_before = 0;
    for (int c = 0; c < k.chunks; ++c) {
      if (c == k.c) equal_before = equal, higher_before = higher;
      least = min(least, st->least[c]);
      most = max(most, st->most[c]);
      equal += st->equal[c];
      higher += st->higher[c];
    }
    if (tid < k.c) g += st->above[tid];
    if (higher < rank && rank <= higher + equal) {  // the ties' key
      p = Picked{tie, rank - higher, equal};
      if (tid == 0) g += higher_before, e = equal_before;
    } else if (least == most) {  // the others are one key
      const bool below = least < tie;
      p = Picked{least, below ? rank - equal : rank, count - equal};
      if (tid == 0) g += below ? equal_before : 0u, e = before - equal_before;
    } else {
      least = min(least, equal > 0 ? tie : least);
      most = max(most, equal > 0 ? tie : most);
      const Range r{least, most, key_float(least), key_float(most)};
      p = pick_in_range<kSplitThreads>(sc, k.j.s.start, k.j.s.stop, rank, r, count);
      g = 0;
      if (k.c > 0)
        for_each_score_rarely<kSplitThreads>(sc, k.j.s.start, k.start, [&](float x) {
          const uint32_t key = float_key(x);
          g += key > p.thresh;
          e += key == p.thresh;
        });
    }
  }
  uint32_t g0, e0;
  block_exclusive_scan<kSplitThreads>(g, s_wave, &g0);
  block_exclusive_scan<kSplitThreads>(e, s_wave, &e0);
  int64_t* out = a.keep + static_cast<int64_t>(blockIdx.z) * a.keep_stride;
  const Keep kp{p.thresh, p.need_eq, p.ties == p.need_eq, out, static_cast<int>(k.j.out_base), a.budget};
  // With every tie kept, both kinds count in the first number.
  emit_range<kSplitThreads>(kp, sc, k.start, k.stop, kp.all_ties ? g0 + e0 : g0, kp.all_ties ? 0u : e0, s_wave);
}

int check_select_args(const char* who, int n_seq, int max_seq_len, const int32_t* seq_lens,
                      const int64_t* token_offsets, const float* scores, int budget, int protected_prefix,
                      int protected_recent, int segments, int policy, int64_t* keep, int64_t keep_stride) {
  if (n_seq <= 0 || n_seq > 65535) return fail(KVC_EINVAL, "%s: bad n_seq %d", who, n_seq);
  if (budget <= 0 || budget > max_seq_len) return fail(KVC_EINVAL, "%s: budget must be in [1, max_seq_len]", who);
  if (protected_prefix < 0 || protected_recent < 0)
    return fail(KVC_EINVAL, "%s: protected windows must be non-negative", who);
  if (static_cast<int64_t>(protected_prefix) + protected_recent > budget)
    return fail(KVC_EINVAL, "%s: protected windows cannot exceed the budget", who);
  if (segments <= 0) return fail(KVC_EINVAL, "%s: segments must be positive", who);
  if (policy != KVC_POLICY_GLOBAL && policy != KVC_POLICY_V3)
    return fail(KVC_EINVAL, "%s: unknown policy %d", who, policy);
  if (keep_stride < budget) return fail(KVC_EINVAL, "%s: keep_stride < budget", who);
  if (!seq_lens || !token_offsets || !scores || !keep) return fail(KVC_EINVAL, "%s: null pointer", who);
  return 0;
}

SelectArgs make_select_args(int n_seq, const int32_t* seq_lens, const int64_t* token_offsets, const float* scores,
                            int budget, int protected_prefix, int protected_recent, int segments, int policy,
                            int64_t* keep, int64_t keep_stride) {
  SelectArgs sa;
  sa.n_seq = n_seq;
  sa.budget = budget;
  sa.prefix = protected_prefix;
  sa.recent = protected_recent;
  sa.segments = policy == KVC_POLICY_V3 ? segments : 1;
  sa.policy = policy;
  sa.seq_lens = seq_lens;
  sa.token_offsets = token_offsets;
  sa.scores = scores;
  sa.keep = keep;
  sa.keep_stride = keep_stride;
  sa.state = nullptr;
  return sa;
}

}  // namespace
}  // namespace kvc

using namespace kvc;

extern "C" int kvc_select_keep(kvc_stream_t stream, int n_seq, int max_seq_len,
                               const int32_t* seq_lens, const int64_t* token_offsets,
                               const float* scores, int budget, int protected_prefix,
                               int protected_recent, int segments, int policy, int64_t* keep,
                               int64_t keep_stride) {
  if (int rc = check_select_args("kvc_select_keep", n_seq, max_seq_len, seq_lens, token_offsets, scores, budget,
                                 protected_prefix, protected_recent, segments, policy, keep, keep_stride))
    return rc;
  const SelectArgs sa = make_select_args(n_seq, seq_lens, token_offsets, scores, budget, protected_prefix,
                                         protected_recent, segments, policy, keep, keep_stride);
  dim3 grid(static_cast<unsigned>(sa.segments), static_cast<unsigned>(n_seq));
  select_kernel<<<grid, kSelThreads, 0, as_stream(stream)>>>(sa);
  return launch_status("kvc_select_keep");
}

extern "C" size_t kvc_select_workspace_bytes(int n_seq, int segments, int policy) {
  if (n_seq <= 0 || segments <= 0) return 0;
  const int nseg = policy == KVC_POLICY_V3 ? segments : 1;
  return static_cast<size_t>(n_seq) * nseg * sizeof(SplitState);
}

extern "C" int kvc_select_keep_split(kvc_stream_t stream, int n_seq, int max_seq_len,
                                     const int32_t* seq_lens, const int64_t* token_offsets,
                                     const float* scores, int budget, int protected_prefix,
                                     int protected_recent, int segments, int policy, int64_t* keep,
                                     int64_t keep_stride, void* workspace, size_t workspace_bytes) {
  if (int rc = check_select_args("kvc_select_keep_split", n_seq, max_seq_len, seq_lens, token_offsets, scores,
                                 budget, protected_prefix, protected_recent, segments, policy, keep, keep_stride))
    return rc;
  const size_t need = kvc_select_workspace_bytes(n_seq, segments, policy);
  if (!workspace || workspace_bytes < need || reinterpret_cast<uintptr_t>(workspace) % 16)
    return fail(KVC_EINVAL, "kvc_select_keep_split: a 16-byte aligned workspace of %zu bytes is needed", need);
  SelectArgs sa = make_select_args(n_seq, seq_lens, token_offsets, scores, budget, protected_prefix,
                                   protected_recent, segments, policy, keep, keep_stride);
  sa.state = workspace;
  // A segment is at most the whole sequence.
  const int chunks = split_chunks(max_seq_len);
  hipStream_t st = as_stream(stream);
  const dim3 grid(static_cast<unsigned>(chunks), static_cast<unsigned>(sa.segments), static_cast<unsigned>(n_seq));
  select_split_bins_kernel<<<grid, kSplitThreads, 0, st>>>(sa);
  if (int rc = launch_status("kvc_select_keep_split(bins)")) return rc;
  select_split_candidates_kernel<<<grid, kSplitThreads, 0, st>>>(sa);
  if (int rc = launch_status("kvc_select_keep_split(candidates)")) return rc;
  select_split_emit_kernel<<<grid, kSplitThreads, 0, st>>>(sa);
  return launch_status("kvc_select_keep_split(emit)");
}
