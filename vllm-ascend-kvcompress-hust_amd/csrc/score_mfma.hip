// TriAttention paged-K scoring on the matrix cores (v_mfma_f32_16x16x32_bf16 /
// v_mfma_f32_16x16x32_f16).
//
// The linear part of the score is a small GEMM per KV head: a 16-token x
// head_dim tile of bf16 keys times head_dim x 16 folded weights (query heads of
// the GQA group on the N axis, unused columns zero).  The keys are exact bf16
// A operands read straight from the paged cache; the float32 weights enter as a
// bf16 hi/lo pair (W = hi + lo to ~2^-16), so two MFMAs per 32-deep K step
// give the float32 dot product to well inside the parity tolerance.  The
// magnitude term sum_f W3_f |k_f| is a second GEMM over the F frequencies with
// |k| computed in the lane (hi/lo split as well; hi*hi + hi*lo + lo*hi).
//
// Operand layout of v_mfma_f32_16x16x32_bf16 (checked on the device): lane l
// holds A[l%16][8*(l/16) + e], B[8*(l/16) + e][l%16] and D[4*(l/16) + i][l%16].
// K step j of the linear part covers head dims 32j .. 32j+31, so lane l of
// step j reads dims 32j + 8*(l/16) .. +8 of token l%16: one 16-byte load.  With
// half-style RoPE and F a multiple of 32, the real parts (step j < F/32) and
// imaginary parts (step j + F/32) of frequencies 32j + 8*(l/16) + e sit in the
// same lane, so |k| needs no data exchange and lands exactly in the layout of
// the magnitude GEMM's A operand.
//
// Interleaved RoPE keeps (real, imaginary) of frequency f in dims (2f, 2f+1),
// so each 32-bit word of a lane's K chunk is one frequency: linear steps 2q and
// 2q+1 give the lane 4 + 4 magnitudes, frequencies 16(2q+h) + 4*(l/16) + i for
// h in {0,1}, i < 4, which fill magnitude step q (the fold lays the magnitude
// weights out in the same order), again without a data exchange.
//
// fp16 caches: the keys are exact fp16 A operands and the weights enter as
// fp16 hi/lo pairs (about 22 significant bits).  fp16's range is narrow, so
// each query head's weights (a B column) are first scaled by a power of two
// that brings the column's largest weight to [2^13, 2^14); the column of the
// product is scaled back on the float32 accumulator, both steps exact.  |k| is
// scaled by 1/4 before its fp16 split (|k| of fp16 keys can exceed 65504) and
// the magnitude weights by 4.
//
// Two words a weight drop 2^-17 of it.  The shapes that the vector scorer used
// to take, in float32, keep that: three words a weight and three of |k|, the
// six products that reach 2^-24.  Their K steps may be partly filled (F not a
// multiple of 32: 96 or 80 dims, 32 rotary of 128): the real parts, the
// imaginary parts and the pass dims each start a step of their own, and lanes
// past a kind's dims hold zero weights.  Scoring 8 sequences of 2048-16384
// tokens x 4 layers, 8 KV heads of 96 dims, took 150 us on the vector ALUs and
// 120 here (with its weight fold, which reads along the frequencies, 12 to 6);
// the vector instructions that split |k| bound it.
//
// Work split: a wave owns one KV head and walks 16-token tiles of its
// workgroup's 256-token span; a workgroup covers hpw KV heads (hpw in {1,2,4}
// dividing kv_heads) and 4/hpw interleaved tile streams per head.  The next
// tile's keys are loaded before the current tile's MFMAs.  Raw scores and the
// float64 per-tile partial sums have the same layout as the VALU scorer's, so
// kvc_head_stats and kvc_aggregate are shared.
//
// A tile costs 136 vector instructions at 128 dims (208 with masked keys,
// per-lane addresses, separate squares and sums of the scores in the loop), so
// the shapes of two words a weight are bound by memory: 16 x 16384 tokens x 6
// layers of 8 heads x 128 dims read 3.2 GB of keys, 523 us for a bare read in
// this access pattern, and write 0.25 GB of scores, which stretch the bare
// read and write to 655 us (the kernel: 668).

#include "mfma_common.h"


namespace kvc {
namespace {

constexpr int kMfmaMaxHeadsPerWg = 4;            // hpw

struct MfmaGeometry {
  int nk, nf, terms;  // linear / magnitude K steps of 32, words per weight
  int hpw, nsub;      // KV heads per workgroup, tile streams per head
  int head_groups;    // kv_heads / hpw
};

inline MfmaGeometry geometry(const ScoreShape& s) {
  MfmaGeometry g;
  const MfmaSteps m = mfma_steps(s);
  g.nk = m.nk;
  g.nf = m.nf;
  g.terms = m.terms;
  g.hpw = (s.kv_heads % 4 == 0) ? 4 : (s.kv_heads % 2 == 0) ? 2 : 1;
  g.nsub = 4 / g.hpw;
  g.head_groups = s.kv_heads / g.hpw;
  return g;
}

// ---------------------------------------------------------------- fold ------

// Fragments hold the eight 16-bit values of each lane of live query heads
// (g < qpk), packed as [fragment][kb][g]; the scorer zeroes the B columns of
// the other lanes, so a wave reads qpk/16 of a full fragment.  Weight for query head g
// (tri/scoring.py:70-81, 117-119 folded with the phase means):
//   real part of frequency f      : sqrt(fss) (qr c - qi s)
//   imaginary part of frequency f : sqrt(fss) (qi c + qr s)
//   pass dim p                    : q_pass[p]
// Magnitude weight of frequency f: sqrt(fss) * extra.  Fragment terms*j + k
// holds word k of K step j (linear steps, then magnitude steps): the rounding
// of what the words before it leave of the weight.
//
// Folded weight of K-step element (step, kb, e) for query head g of
// a (sequence, layer, KV head) whose phases are pc, ps.  Elements past the
// frequencies or the pass dims (dead lanes of a kind's last step) are zero.
__device__ __forceinline__ float folded_weight(const FoldArgs& a, const float* pc, const float* ps, int nk, int nf,
                                              int64_t row, int step, int kb, int e) {
  if (step < 2 * nf) {
    if (a.zero_rotary) return 0.0f;
    // Half style: steps 0 .. nf-1 real, nf .. 2nf-1 imaginary parts of 32
    // frequencies each; interleaved: 32 dims of (real, imaginary) pairs.
    const int i = 32 * step + 8 * kb + e;
    const bool real = a.interleaved ? (i & 1) == 0 : step < nf;
    const int f = a.interleaved ? i >> 1 : (step < nf ? i : i - 32 * nf);
    if (f >= a.freq) return 0.0f;
    const int64_t o = row * a.freq + f;
    const float qr = a.q_real[o], qi = a.q_imag[o], sc = a.scale[o];
    const float c = pc[f], sn = ps[f];
    return real ? sc * (qr * c - qi * sn) : sc * (qi * c + qr * sn);
  }
  if (step < nk) {
    const int p = 32 * (step - 2 * nf) + 8 * kb + e;
    return p < a.pass ? a.q_pass[row * a.pass + p] : 0.0f;
  }
  const int q = step - nk;
  const int f = a.interleaved ? 16 * (2 * q + (e >> 2)) + 4 * kb + (e & 3) : 32 * q + 8 * kb + e;
  if (f >= a.freq) return 0.0f;
  const int64_t o = row * a.freq + f;
  return a.scale[o] * a.extra[o];
}

// The 16-bit words of the eight weights w, word k to dst + k * stride (of three
// fp16 words each divided by kLowScale more than the one before).
template <bool F16>
__device__ __forceinline__ void store_words(float (&w)[8], int terms, uint16_t* dst, int64_t stride) {
  for (int k = 0; k < terms; ++k) {
    u32x4 out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t word = 0;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float& v = w[2 * i + h];
        uint32_t bits;
        if (F16) {
          bits = __builtin_bit_cast(uint16_t, static_cast<_Float16>(v));
          if (terms == 3 && k == 0) bits &= MfmaElem<true>::kLeadMask;
          v -= static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(bits)));
          if (terms == 3) v *= 1.0f / MfmaElem<true>::kLowScale;
        } else {
          bits = bf16_bits(v) & 0xffffu;
          v -= bf16_value(bits);
        }
        word |= bits << (16 * h);
      }
      out[i] = word;
    }
    *reinterpret_cast<u32x4*>(dst + k * stride) = out;
  }
}

// The fragments of `heads` KV heads of one (sequence b, layer) for `threads`
// threads starting at `first`, phases pc, ps.  bf16: a thread a live lane of a K step.  fp16: a wave
// a column (KV head, query head g); lane l < 4*(nk+nf) owns K step l/4, row
// block l%4: its eight weights (magnitude weights times 1/kMagScale), then the
// column's largest magnitude over the wave picks the power-of-two scale 2^s
// that brings it to [2^13, 2^14) (s in [-126, 126]; none when it is 0, inf or
// NaN), the words are those of 2^s w, and lane 0 writes 2^-s.
template <bool F16>
__device__ __forceinline__ void fold_layer(const FoldArgs& a, const float* pc, const float* ps, int b, int layer, int nk,
                                           int nf, int terms, uint16_t* frags, float* inv_scale, int head_begin, int heads,
                                           int first, int threads) {
  const int packed = 4 * a.qpk;  // live lanes per fragment
  const int steps = nk + nf;
  const int64_t head0 = (static_cast<int64_t>(b) * a.n_layers + layer) * a.kv_heads;
  const int items = F16 ? heads * a.qpk * 64 : heads * steps * packed;
  for (int idx = first; idx < items; idx += threads) {
    int head, g, step, kb;
    bool active = true;
    if (F16) {
      const int lane = idx & 63, col = idx >> 6;
      head = col / a.qpk;
      g = col - head * a.qpk;
      step = lane >> 2;
      kb = lane & 3;
      active = step < steps;
    } else {
      const int r = idx / packed, pl = idx - r * packed;
      head = r / steps;
      step = r - head * steps;
      kb = pl / a.qpk;
      g = pl - kb * a.qpk;
    }
    head += head_begin;
    const int64_t row = (static_cast<int64_t>(layer) * a.kv_heads + head) * a.qpk + g;
    float w[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) w[e] = active ? folded_weight(a, pc, ps, nk, nf, row, step, kb, e) : 0.0f;
    if (F16) {
      float big = 0.0f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (step >= nk) w[e] *= 1.0f / MfmaElem<true>::kMagScale;
        big = fmaxf(big, fabsf(w[e]));
      }
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) big = fmaxf(big, __shfl_xor(big, off));
      int sh = 0;
      if (big > 0.0f && big <= 3.4e38f) {
        int ex;
        (void)frexpf(big, &ex);  // big < 2^ex
        sh = 14 - ex;
        sh = sh < -126 ? -126 : (sh > 126 ? 126 : sh);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) w[e] = ldexpf(w[e], sh);
      if ((idx & 63) == 0) inv_scale[(head0 + head) * a.qpk + g] = ldexpf(1.0f, -sh);
    }
    if (active)
      store_words<F16>(w, terms, frags + (((head0 + head) * terms * steps + terms * step) * packed + kb * a.qpk + g) * 8,
                       packed * 8);
  }
}

// grid (blocks, layers, sequences): phases from the caller's tables.
constexpr int kFoldThreads = 256;
template <bool F16>
__global__ __launch_bounds__(kFoldThreads) void fold_mfma_kernel(FoldArgs a, int nk, int nf, int terms,
                                                                 uint16_t* __restrict__ frags,
                                                                 float* __restrict__ inv_scale) {
  const int layer = blockIdx.y, b = blockIdx.z;
  const int64_t at = b * a.phase_seq_stride + static_cast<int64_t>(layer) * a.freq;
  fold_layer<F16>(a, a.phase_cos + at, a.phase_sin + at, b, layer, nk, nf, terms, frags, inv_scale, 0,
                  a.kv_heads, blockIdx.x * kFoldThreads + threadIdx.x, gridDim.x * kFoldThreads);
}

// grid (layers, sequences, head splits): a workgroup forms its (sequence,
// layer)'s mean phases, which every head shares, in LDS (and split 0 in the
// caller's tables), and folds its KV heads' weights from them.  One workgroup's
// scattered loads of the statistics bound it, so the heads are split until some
// 512 workgroups share them, each forming the phases again.  As two launches this was
// 4.2 + 6.2 us for one sequence x 6 layers of 40 heads, and the gap between
// them; in one workgroup a layer 10.6, with the heads split 8.1.  16 sequences:
// 4.9 + 8.6 before, 12.9 now.
constexpr int kFoldPhaseThreads = 1024;
constexpr int kFoldMaxFreq = 128;
template <bool F16>
__global__ __launch_bounds__(kFoldPhaseThreads) void fold_phases_kernel(FoldArgs a, PhaseArgs ph, int width, int nk, int nf,
                                                                        int terms, uint16_t* __restrict__ frags,
                                                                        float* __restrict__ inv_scale) {
  __shared__ float s_cos[kFoldMaxFreq], s_sin[kFoldMaxFreq];
  const int layer = blockIdx.x, b = blockIdx.y;
  const float rs = static_cast<float>(ph.round_starts[b]);
  const int64_t at = (static_cast<int64_t>(b) * a.n_layers + layer) * a.freq;
  for (int i = threadIdx.x; i < a.freq * width; i += kFoldPhaseThreads) {  // whole lane groups
    const int f = i / width, lane = i & (width - 1);
    const float2 m = mean_phase(lane, width, rs, ph.omega[static_cast<int64_t>(layer) * a.freq + f], ph.offsets, ph.n_offsets);
    if (lane == 0) {
      s_cos[f] = m.x;
      s_sin[f] = m.y;
      if (blockIdx.z == 0) {
        ph.phase_cos[at + f] = m.x;
        ph.phase_sin[at + f] = m.y;
      }
    }
  }
  __syncthreads();
  const int per = (a.kv_heads + gridDim.z - 1) / gridDim.z;
  const int head = blockIdx.z * per;
  fold_layer<F16>(a, s_cos, s_sin, b, layer, nk, nf, terms, frags, inv_scale, head, min(per, a.kv_heads - head),
                  threadIdx.x, kFoldPhaseThreads);
}

// --------------------------------------------------------------- score ------

// The score of one key row for one query head in plain float32, weights folded
// in place.  Split words turn an infinity into a NaN (inf - inf, inf * 0), so
// the tokens whose products are not finite are scored again here.
template <bool F16>
__device__ __forceinline__ float plain_score(const FoldArgs& a, int b, int layer, int64_t row,
                                             KVC_GLOBAL const uint16_t* key) {
  auto at = [&](int d) { return F16 ? fp16_lo(key[d]) : bf16_lo(key[d]); };
  const float* pc = a.phase_cos + b * a.phase_seq_stride + static_cast<int64_t>(layer) * a.freq;
  const float* ps = a.phase_sin + b * a.phase_seq_stride + static_cast<int64_t>(layer) * a.freq;
  float v = 0.0f;
#pragma unroll 1
  for (int f = 0; f < a.freq; ++f) {
    const int64_t o = row * a.freq + f;
    const float qr = a.q_real[o], qi = a.q_imag[o], sc = a.scale[o], c = pc[f], sn = ps[f];
    const float re = at(a.interleaved ? 2 * f : f), im = at(a.interleaved ? 2 * f + 1 : a.freq + f);
    v = fmaf(sc * (qr * c - qi * sn), re, v);
    v = fmaf(sc * (qi * c + qr * sn), im, v);
    v = fmaf(sc * a.extra[o], __builtin_amdgcn_sqrtf(fmaf(im, im, re * re)), v);
  }
#pragma unroll 1
  for (int p = 0; p < a.pass; ++p) v = fmaf(a.q_pass[row * a.pass + p], at(a.rotary_dim + p), v);
  return v;
}

// 16-token tiles per prefetch group, and the waves per SIMD asked of the
// compiler: three words a weight in registers leave room for two waves up to
// nine K steps when a group is one tile from six steps on.
template <int NK, int NF, bool PART>
struct MfmaTiling {
  static constexpr int G = PART && NK >= 6 ? 1 : 2;
  static constexpr int kWavesPerSimd = PART && 12 * (NK + NF) + 8 * G * NK <= 232 ? 2 : 1;  // 1: no request
};

template <int NK, int NF, bool F16, bool IL, bool PART>
__global__ __launch_bounds__(kScoreThreads)
__attribute__((amdgpu_waves_per_eu(MfmaTiling<NK, NF, PART>::kWavesPerSimd))) void score_mfma_kernel(ScoreArgs a, FoldArgs fold, MfmaGeometry geo,
                                                                   int qpk, const u32x4* __restrict__ frags,
                                                                   const float* __restrict__ inv_scale) {
  typedef MfmaElem<F16> E;
  typedef typename E::vec vec_t;
  const int layer = blockIdx.z;
  const int b = blockIdx.y;
  const int tile = blockIdx.x / geo.head_groups;
  const int hg = blockIdx.x - tile * geo.head_groups;
  const int n = a.seq_lens[b];
  const int t0 = tile * kScoreTile;
  if (t0 >= n) return;  // whole workgroup leaves together
  const int t1 = min(n, t0 + kScoreTile);

  const int lane = threadIdx.x & 63;
  // The wave's number, and what follows from it (its head, its tiles and their
  // addresses), is kept in scalar registers.
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15;   // A row (token in tile) / D column (query head)
  const int kb = lane >> 4;  // K block of A/B, row block of D
  const int head = hg * geo.hpw + wave % geo.hpw;
  const int sub = wave / geo.hpw;

  // Folded weight fragments of (sequence, layer, head).
  constexpr int TERMS = PART ? 3 : 2;
  constexpr int kFrags = TERMS * (NK + NF);
  // Packed fragments [frag][kb][g < qpk]; lanes of query heads g >= qpk read
  // the kb group's first word (a line the live lanes read anyway) and zero it.
  const int packed = 4 * qpk;
  const bool live_col = r < qpk;
  const u32x4* fp = frags + (((static_cast<int64_t>(b) * a.n_layers + layer) * a.kv_heads + head) * kFrags) * packed +
                    kb * qpk + (live_col ? r : 0);
  auto frag_word = [&](int f) {
    const u32x4 v = fp[f * packed];
    return __builtin_bit_cast(vec_t, live_col ? v : u32x4{0, 0, 0, 0});
  };
  vec_t w[NK][TERMS], m[NF][TERMS];
  // fp16: the scale that takes this lane's output column back from the
  // scaled weights.
  const float col_scale =
      F16 ? inv_scale[((static_cast<int64_t>(b) * a.n_layers + layer) * a.kv_heads + head) * qpk + (live_col ? r : 0)]
          : 1.0f;
#pragma unroll
  for (int k = 0; k < TERMS; ++k) {
#pragma unroll
    for (int j = 0; j < NK; ++j) w[j][k] = frag_word(TERMS * j + k);
#pragma unroll
    for (int q = 0; q < NF; ++q) m[q][k] = frag_word(TERMS * (NK + q) + k);
  }

  KVC_GLOBAL const uint16_t* kbase = gptr_from_int<const uint16_t>(a.k_layer_ptrs[layer]);
  const int64_t* bt = a.block_ids + a.block_offsets[b];
  const int64_t n_blocks = a.block_offsets[b + 1] - a.block_offsets[b];
  const int64_t row_elems = static_cast<int64_t>(a.kv_heads) * a.head_dim;
  const int64_t head_off = static_cast<int64_t>(head) * a.head_dim;
  // Byte offset from a tile's first token to this lane's chunk of K step j.
  // With every step full it is 64*j past the lane's own.  PART: the steps of a
  // kind start at their own base, and a chunk of the kind's last step that lies
  // past its dims re-reads the row's first chunk (its weights are zero).
  const uint32_t row_off = static_cast<uint32_t>(r) * static_cast<uint32_t>(row_elems) * 2;
  uint32_t chunk[NK];
#pragma unroll
  for (int j = 0; j < NK; ++j) {
    int d = 32 * j + 8 * kb;
    if (PART) {
      int at, end;  // place inside the kind, its dims
      if (j >= 2 * NF) {
        at = 32 * (j - 2 * NF) + 8 * kb;
        end = a.head_dim - a.rotary_dim;
        d = a.rotary_dim + at;
      } else if (IL) {
        at = d;
        end = a.rotary_dim;
      } else {
        at = 32 * (j % NF) + 8 * kb;
        end = a.freq;
        d = (j < NF ? 0 : a.freq) + at;
      }
      if (at >= end) d = 0;
    }
    chunk[j] = row_off + 2 * static_cast<uint32_t>(d);
  }
  const int64_t tok_base = a.token_offsets[b];
  float* raw_out = a.raw + layer * a.raw_layer_stride;
  const int n_mt = (t1 - t0 + 15) / 16;  // 16-token tiles in the span
  const bool writer = r < qpk;
  const int hl_wave = wave % geo.hpw;  // KV head slot of this wave inside the workgroup

  // Score stage: [hpw][qpk][kStageStride] floats, rows padded by four floats
  // so the query-head rows of one wave start in different LDS banks.
  __shared__ __attribute__((aligned(16))) float stage[kMfmaMaxHeadsPerWg * kMfmaMaxQpk * kStageStride];
  float* stage_row = stage + (hl_wave * qpk + (writer ? r : 0)) * kStageStride;

  SpanPages pages;
  pages.resolve(kbase, bt, n_blocks, a.num_pages, a.page_stride, t0);

  auto load_tile = [&](int mt, u32x4 (&ka)[NK]) {
    // The loads are unconditional (loads under a branch would make the
    // compiler wait for every load in flight at the join) and always hit a row
    // inside the pool: tiles the prefetch reaches past the span re-read the
    // span's last tile, which this wave has just read (a cache hit, not HBM
    // traffic), unresolved pages read page 0 and rows past the sequence
    // whatever their page holds.  A token is a row of every product, so those
    // rows reach only scores that are set to zero or never stored, and the keys
    // need no masking; the tile's address is scalar.
    const int rel = min(mt, n_mt - 1) * 16;
    bool page_ok = false;
    KVC_GLOBAL const char* at = reinterpret_cast<KVC_GLOBAL const char*>(
        pages.page(rel, &page_ok) + static_cast<int64_t>(rel & (kBlockSize - 1)) * row_elems + head_off);
#pragma unroll
    for (int j = 0; j < NK; ++j) ka[j] = load_k(reinterpret_cast<KVC_GLOBAL const u32x4*>(at + chunk[j]));
  };

  auto score_tile = [&](int mt, const u32x4 (&ka)[NK]) {
    // Independent accumulation chains keep consecutive MFMAs apart.
    f32x4 acc0 = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 acc1 = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (PART) {
      // Three words a weight and three of |k|: the products that reach 2^-24.
      // Each step's leading products are a sum of their own and the sums meet
      // pairwise, so that they round at their own size.  fp16: acc0 holds
      // products one kLowScale up, acc1 two.
      constexpr int kChains = NK + NF;
      f32x4 lead[kChains];
#pragma unroll
      for (int c = 0; c < kChains; ++c) lead[c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      f32x4 low = {0.0f, 0.0f, 0.0f, 0.0f};  // bf16: products with the lower words of |k|
#pragma unroll
      for (int j = 0; j < NK; ++j) {
        const vec_t kv = __builtin_bit_cast(vec_t, ka[j]);
        lead[j] = E::mfma(kv, w[j][0], lead[j]);
        acc0 = E::mfma(kv, w[j][1], acc0);
        acc1 = E::mfma(kv, w[j][2], acc1);
      }
#pragma unroll
      for (int q = 0; q < NF; ++q) {
        vec_t k3[3];
        magnitude_words<F16, IL, NK, NF, 3>(ka, q, k3);
        lead[NK + q] = E::mfma(k3[0], m[q][0], lead[NK + q]);
        acc0 = E::mfma(k3[0], m[q][1], acc0);
        acc1 = E::mfma(k3[0], m[q][2], acc1);
        f32x4& once = F16 ? acc0 : low;
        f32x4& twice = F16 ? acc1 : low;
        once = E::mfma(k3[1], m[q][0], once);
        twice = E::mfma(k3[1], m[q][1], twice);
        twice = E::mfma(k3[2], m[q][0], twice);
      }
#pragma unroll
      for (int width = 1; width < kChains; width *= 2)
#pragma unroll
        for (int c = 0; c + width < kChains; c += 2 * width) lead[c] += lead[c + width];
      acc1 = F16 ? (acc1 * E::kLowScale + acc0) * E::kLowScale : acc1 + low + acc0;
      acc0 = lead[0];
    } else {
#pragma unroll
      for (int j = 0; j < NK; ++j) {
        const vec_t kv = __builtin_bit_cast(vec_t, ka[j]);
        if (j & 1) {
          acc1 = E::mfma(kv, w[j][0], acc1);
          acc1 = E::mfma(kv, w[j][1], acc1);
        } else {
          acc0 = E::mfma(kv, w[j][0], acc0);
          acc0 = E::mfma(kv, w[j][1], acc0);
        }
      }
#pragma unroll
      for (int q = 0; q < NF; ++q) {
        vec_t k2[2];
        magnitude_words<F16, IL, NK, NF, 2>(ka, q, k2);
        acc0 = E::mfma(k2[0], m[q][0], acc0);
        acc1 = E::mfma(k2[0], m[q][1], acc1);
        acc0 = E::mfma(k2[1], m[q][0], acc0);
      }
    }
    f32x4 acc = acc0 + acc1;
    if (F16) acc *= col_scale;
    bool page_ok = false;
    KVC_GLOBAL const uint16_t* tile_base = pages.page(mt * 16, &page_ok);
    if (!page_ok) acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (PART) {
      unsigned plain = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (writer && t0 + mt * 16 + 4 * kb + i < t1 && !(fabsf(acc[i]) <= 3.402823466e38f)) plain |= 1u << i;
      if (__any(plain != 0)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int in_page = (mt * 16 + 4 * kb + i) & (kBlockSize - 1);
          if (plain >> i & 1)
            acc[i] = plain_score<F16>(fold, b, layer, (static_cast<int64_t>(layer) * a.kv_heads + head) * qpk + r,
                                      tile_base + in_page * row_elems + head_off);
        }
      }
    }
    // D[4*kb + i][r]: token t0 + 16*mt + 4*kb + i, query head r of this KV head.
    // Scores go to the workgroup's LDS stage (four adjacent tokens per lane,
    // one 16-byte write); global stores and the head sums wait until the span
    // is done: the loop's waits then cover only K loads (vector memory
    // operations retire in issue order, and a store in the loop would hold up
    // the next tile), and the sums use every lane instead of qpk of 16.
    if (writer) *reinterpret_cast<f32x4*>(stage_row + mt * 16 + 4 * kb) = acc;
  };

  // Tiles sub, sub + nsub, ... in groups of G; the next group's
  // keys are in flight while the current group is scored.
  constexpr int G = MfmaTiling<NK, NF, PART>::G;
  u32x4 ka[G][NK], kb2[G][NK];
  const int step = geo.nsub;
  int mt = sub;
#pragma unroll
  for (int g = 0; g < G; ++g) load_tile(mt + g * step, ka[g]);
  for (; mt < n_mt; mt += 2 * G * step) {
#pragma unroll
    for (int g = 0; g < G; ++g) load_tile(mt + (G + g) * step, kb2[g]);
#pragma unroll
    for (int g = 0; g < G; ++g)
      if (mt + g * step < n_mt) score_tile(mt + g * step, ka[g]);
    if (mt + G * step >= n_mt) break;
#pragma unroll
    for (int g = 0; g < G; ++g) load_tile(mt + (2 * G + g) * step, ka[g]);
#pragma unroll
    for (int g = 0; g < G; ++g)
      if (mt + (G + g) * step < n_mt) score_tile(mt + (G + g) * step, kb2[g]);
  }

  __syncthreads();

  // Stage -> raw scores: row (hl, g) holds query head (hg*hpw + hl)*qpk + g
  // for the span's tokens.  Head-major scores are contiguous per row (a wave a
  // row, 16-byte stores where aligned); token-major ones are contiguous across
  // the rows.  Non-temporal 16-byte stores measured 1-2% faster scoring than
  // plain ones (the scores are read once more, by the aggregation pass).
  const int span = t1 - t0;
  const int rows = geo.hpw * qpk;
  const int q_first = hg * geo.hpw * qpk;
  if (a.raw_token_stride == 1) {
    static_assert(kScoreTile == 4 * 64, "a lane stores four tokens of a row");
    const int c = lane << 2;
    for (int row = wave; row < rows; row += kScoreThreads / 64) {
      const float* src = stage + row * kStageStride + c;
      float* dst = raw_out + (tok_base + t0 + c) + static_cast<int64_t>(q_first + row) * a.raw_head_stride;
      if (c + 3 < span && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
        __builtin_nontemporal_store(*reinterpret_cast<const f32x4*>(src), reinterpret_cast<f32x4*>(dst));
      } else {
        for (int i = 0; i < 4 && c + i < span; ++i) dst[i] = src[i];
      }
    }
  } else {
    int t = threadIdx.x / rows, row = threadIdx.x - t * rows;
    const int dt = kScoreThreads / rows, drow = kScoreThreads - dt * rows;
    while (t < span) {
      raw_out[(tok_base + t0 + t) * a.raw_token_stride + static_cast<int64_t>(q_first + row) * a.raw_head_stride] =
          stage[row * kStageStride + t];
      t += dt;
      row += drow;
      if (row >= rows) {
        row -= rows;
        ++t;
      }
    }
  }

  // Per query head, the float64 sums of the span's scores and their squares:
  // `per` threads a row take every per-th four tokens, then one adds them up.
  constexpr int kSumThreads = 16;
  __shared__ double red[2][kScoreThreads];
  const int per = min(kSumThreads, kScoreThreads / rows);
  {
    const int row = threadIdx.x / per, part = threadIdx.x - row * per;
    double sum = 0.0, sumsq = 0.0;
    if (row < rows) {
      for (int c = part * 4; c < span; c += per * 4) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(stage + row * kStageStride + c);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const double dv = static_cast<double>(c + i < span ? v[i] : 0.0f);
          sum += dv;
          sumsq = fma(dv, dv, sumsq);
        }
      }
    }
    red[0][threadIdx.x] = sum;
    red[1][threadIdx.x] = sumsq;
  }
  __syncthreads();
  if (static_cast<int>(threadIdx.x) < rows) {
    double s0 = 0.0, s1 = 0.0;
    for (int k = 0; k < per; ++k) {
      s0 += red[0][threadIdx.x * per + k];
      s1 += red[1][threadIdx.x * per + k];
    }
    const int n_heads = a.kv_heads * qpk;
    double* dst = a.partials +
                  (((static_cast<int64_t>(layer) * a.n_seq + b) * a.max_tiles + tile) * n_heads + q_first + threadIdx.x) * 2;
    dst[0] = s0;
    dst[1] = s1;
  }
}

using MfmaKernel = void (*)(ScoreArgs, FoldArgs, MfmaGeometry, int, const u32x4*, const float*);

template <bool F16, bool IL>
MfmaKernel pick_full(int nk, int nf) {
  switch (nk * 16 + nf) {
    case 2 * 16 + 1: return score_mfma_kernel<2, 1, F16, IL, false>;
    case 4 * 16 + 1: return score_mfma_kernel<4, 1, F16, IL, false>;
    case 4 * 16 + 2: return score_mfma_kernel<4, 2, F16, IL, false>;
    case 8 * 16 + 1: return score_mfma_kernel<8, 1, F16, IL, false>;
    case 8 * 16 + 2: return score_mfma_kernel<8, 2, F16, IL, false>;
    case 8 * 16 + 4: return score_mfma_kernel<8, 4, F16, IL, false>;
    default: return nullptr;
  }
}
// The other shapes: every (nf, pass steps) that up to 128 rotary of up to 256
// dims give.
template <bool F16, bool IL, int NF, int NP_MAX>
MfmaKernel pick_part_pass(int np) {
  if (np == NP_MAX) return score_mfma_kernel<2 * NF + NP_MAX, NF, F16, IL, true>;
  if constexpr (NP_MAX > 0) return pick_part_pass<F16, IL, NF, NP_MAX - 1>(np);
  return nullptr;
}
template <bool F16, bool IL>
MfmaKernel pick_part(int nk, int nf) {
  switch (nf) {
    case 1: return pick_part_pass<F16, IL, 1, 8>(nk - 2);
    case 2: return pick_part_pass<F16, IL, 2, 6>(nk - 4);
    default: return nullptr;
  }
}
template <bool F16, bool IL>
MfmaKernel pick_typed(const ScoreShape& s) {
  const MfmaSteps m = mfma_steps(s);
  return mfma_two_words(s) ? pick_full<F16, IL>(m.nk, m.nf) : pick_part<F16, IL>(m.nk, m.nf);
}
MfmaKernel pick(const ScoreShape& s, int dtype, int rope_style) {
  const bool il = rope_style == KVC_ROPE_INTERLEAVED;
  if (dtype == KVC_DTYPE_FP16) return il ? pick_typed<true, true>(s) : pick_typed<true, false>(s);
  return il ? pick_typed<false, true>(s) : pick_typed<false, false>(s);
}

}  // namespace

bool mfma_scorer_supported(const ScoreShape& s, int dtype, int rope_style) {
  if (dtype != KVC_DTYPE_BF16 && dtype != KVC_DTYPE_FP16) return false;
  if (rope_style != KVC_ROPE_HALF && rope_style != KVC_ROPE_INTERLEAVED) return false;
  if (!mfma_shape(s) || s.qpk > kMfmaMaxQpk) return false;
  return pick(s, dtype, rope_style) != nullptr;
}

namespace {
// Workgroups a (sequence, layer) is folded by.
unsigned fold_blocks(const ScoreShape& s, int dtype) {
  const MfmaGeometry geo = geometry(s);
  const int cols = s.kv_heads * s.qpk;
  return static_cast<unsigned>(ceil_div(dtype == KVC_DTYPE_FP16 ? cols * 64 : cols * 4 * (geo.nk + geo.nf), kFoldThreads));
}
}  // namespace

int64_t mfma_fold_items(const ScoreShape& s, int dtype) {
  return static_cast<int64_t>(fold_blocks(s, dtype)) * kFoldThreads * s.n_layers * s.n_seq;
}

// Workgroups a (sequence, layer) is folded by where they form its phases too.
static int64_t phase_fold_splits(const ScoreShape& s) {
  const int64_t splits = ceil_div(512, static_cast<int64_t>(s.n_layers) * s.n_seq);
  return splits < s.kv_heads ? splits : s.kv_heads;
}

int64_t mfma_phase_fold_items(const ScoreShape& s) {
  return static_cast<int64_t>(s.n_layers) * s.n_seq * phase_fold_splits(s) * kFoldPhaseThreads;
}

int launch_mfma_fold(hipStream_t stream, const ScoreShape& s, int dtype, const FoldArgs& fa, void* weights) {
  const MfmaGeometry geo = geometry(s);
  const int64_t items = mfma_fold_items(s, dtype);
  if (items > kMaxDispatchItems || s.n_seq > 65535 || s.n_layers > 65535)
    return fail(KVC_EINVAL, "kvc_score_paged: the weight fold's %lld work-items exceed one dispatch",
                static_cast<long long>(items));
  uint16_t* frags = static_cast<uint16_t*>(weights);
  float* inv_scale = reinterpret_cast<float*>(static_cast<char*>(weights) + mfma_fragment_only_bytes(s));
  const dim3 grid(fold_blocks(s, dtype), static_cast<unsigned>(s.n_layers), static_cast<unsigned>(s.n_seq));
  (dtype == KVC_DTYPE_FP16 ? fold_mfma_kernel<true> : fold_mfma_kernel<false>)<<<grid, kFoldThreads, 0, stream>>>(
      fa, geo.nk, geo.nf, geo.terms, frags, inv_scale);
  return launch_status("kvc_score_paged(fold)");
}

int launch_mfma_scorer(hipStream_t stream, const ScoreShape& s, int dtype, const PhaseArgs* phases, const FoldArgs& fa,
                       const ScoreArgs& sa, void* weights) {
  const MfmaGeometry geo = geometry(s);
  MfmaKernel kern = pick(s, dtype, fa.interleaved ? KVC_ROPE_INTERLEAVED : KVC_ROPE_HALF);
  if (!kern) return fail(KVC_EINVAL, "kvc_score_paged: no MFMA scorer for head_dim %d rotary_dim %d", s.head_dim, s.rotary_dim);
  if (s.n_seq > 65535 || s.n_layers > 65535)
    return fail(KVC_EINVAL, "kvc_score_paged: too many sequences or layers for one launch");
  if (phases) {
    uint16_t* out = static_cast<uint16_t*>(weights);
    float* scale = reinterpret_cast<float*>(static_cast<char*>(weights) + mfma_fragment_only_bytes(s));
    const dim3 grid(static_cast<unsigned>(s.n_layers), static_cast<unsigned>(s.n_seq),
                    static_cast<unsigned>(phase_fold_splits(s)));
    (dtype == KVC_DTYPE_FP16 ? fold_phases_kernel<true> : fold_phases_kernel<false>)<<<grid, kFoldPhaseThreads, 0, stream>>>(
        fa, *phases, phase_lanes(phases->n_offsets), geo.nk, geo.nf, geo.terms, out, scale);
    if (int rc = launch_status("kvc_score_paged(phases and fold)")) return rc;
  } else if (int rc = launch_mfma_fold(stream, s, dtype, fa, weights)) {
    return rc;
  }
  const uint16_t* frags = static_cast<const uint16_t*>(weights);
  const float* inv_scale = reinterpret_cast<const float*>(static_cast<const char*>(weights) + mfma_fragment_only_bytes(s));
  const int64_t gx = static_cast<int64_t>(s.max_tiles) * geo.head_groups;
  if (gx > 0x7fffffff) return fail(KVC_EINVAL, "kvc_score_paged: grid too large");
  dim3 grid(static_cast<unsigned>(gx), static_cast<unsigned>(s.n_seq), static_cast<unsigned>(s.n_layers));
  kern<<<grid, kScoreThreads, 0, stream>>>(sa, fa, geo, s.qpk, reinterpret_cast<const u32x4*>(frags), inv_scale);
  return launch_status("kvc_score_paged");
}

}  // namespace kvc
