// Sequences cut along T for the sequential passes: when there are too few (sequence, head) pairs for the 256 CUs, a
// pass over the chunks of a pair leaves most of the GPU idle (16 pairs x 4 V slices = 64 work-groups) and takes as
// long as its chain of chunks.  A sequence is then cut into segments:
//   1. every FINE segment (len1 chunks) is run from a zero state, all at once, for the state alone (no output): its
//      own contribution Q and, for the delta rule, the matrix P that carries an initial state to its end;
//   2. the segments of a pair are combined in order, S <- P S + Q (one small product per fine segment), which leaves
//      the initial state of every COARSE segment (len3 = a multiple of len1 chunks) in memory;
//   3. the ordinary pass runs over the coarse segments as if each were a sequence of its own.
// Backward likewise from the end, with P transposed.  Cuts lie on chunk boundaries and never show outside: every
// per-chunk buffer keeps its place.
#pragma once
#include "lmoe_seq.hpp"

namespace lmoe {

// What the kernels need to know; len1 = 0: not cut.
struct Split {
  int32_t len1;          // chunks per fine segment
  int32_t len3;          // chunks per coarse segment (a multiple of len1)
  int32_t n1, n3;        // segments of all sequences (packed input: upper bounds; a segment beyond the true count ends at once)
  bf16 *P, *PT;          // [n1][H][K][K]  transitions of the fine segments less their decay (delta rule; without a gate two
                         // such matrices, hi and lo), in operand order, and
                         // the same transposed (kept for the backward; NULL in a call that keeps nothing)
  float *D, *DT;         // [n1][H]        decays of the fine segments (beside P, PT); chunk_gla: [n1][H][K]
  float* Q;              // [n1][H][K][V]  their contributions
  float* S;              // [n3][H][K][V]  state (gradient) a coarse segment starts from
  float* Z;              // [n1][H][K]     contributions to the normaliser's column (chunk_simple_gla)
};

// Sequences of fewer chunks gain nothing (three kernels in place of one).  Above 32 768 tokens (packed: on average) they
// are left whole although they would gain (65 536 tokens, 16 heads, by the model of plan_split: 794 us in place of 1741):
// there a sequence gives the same bits alone and inside a packed batch that fills the CUs, which the ops are held to.
// Between the two limits it does not: what is cut depends on how many pairs a call has, and results differ by rounding.
constexpr int SPLIT_MIN_CHUNKS = 24, SPLIT_MAX_CHUNKS = 512;

__host__ __device__ inline int seg_count(int nchunks, int len) { return (nchunks + len - 1) / len; }

struct SegInfo {
  int n;          // sequence (-1: no such segment)
  int j;          // segment inside the sequence
  int nseg;       // segments of the sequence
};

// Segment number s (segments of all sequences in order) -> sequence and place inside it.  Packed input: every lane
// counts the segments of one sequence, a scan over the wave gives the first segment of each (64 sequences a round).
// All lanes of the wave must be active.
__device__ __forceinline__ SegInfo seg_find(const lmoe_args& a, int len, int s) {
  SegInfo r;
  if (!a.cu_seqlens) {
    // (uniform, said to the compiler: what derives from it stays in scalar registers)
    r.nseg = __builtin_amdgcn_readfirstlane(seg_count((a.T + CH - 1) / CH, len));
    r.n = __builtin_amdgcn_readfirstlane(s / r.nseg);
    r.j = s - r.n * r.nseg;
    if (r.n >= a.N) r.n = -1;
    return r;
  }
  const int l = lane_id();
  int base = 0;
  for (int n0 = 0; n0 < a.N; n0 += 64) {
    const int n = n0 + l;
    const int cnt = n < a.N ? seg_count(a.seq_chunk0[n + 1] - a.seq_chunk0[n], len) : 0;
    int incl = cnt;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_up(incl, d, 64);
      if (l >= d) incl += y;
    }
    const int total = __shfl(incl, 63, 64);
    if (s < base + total) {
      const unsigned long long m = __ballot(s < base + incl);
      const int w = __ffsll(m) - 1;                    // the first sequence whose segments reach past s
      r.n = __builtin_amdgcn_readfirstlane(n0 + w);
      r.nseg = __builtin_amdgcn_readlane(cnt, w);
      r.j = s - base - (__builtin_amdgcn_readlane(incl, w) - r.nseg);
      r.j = __builtin_amdgcn_readfirstlane(r.j);
      return r;
    }
    base += total;
  }
  r.n = -1; r.j = 0; r.nseg = 0;
  return r;
}
// number of the first segment of sequence n
__device__ __forceinline__ int seg_base(const lmoe_args& a, int len, int n) {
  if (!a.cu_seqlens) return n * seg_count((a.T + CH - 1) / CH, len);
  const int l = lane_id();
  int sum = 0;
  for (int m = l; m < n; m += 64) sum += seg_count(a.seq_chunk0[m + 1] - a.seq_chunk0[m], len);
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) sum += __shfl_xor(sum, d, 64);
  return __builtin_amdgcn_readfirstlane(sum);
}
// chunks [j len, (j + 1) len) of a sequence as a sequence of their own
__device__ __forceinline__ SeqInfo seg_cut(SeqInfo s, int j, int len) {
  s.tok0 += j * len * CH;
  s.len = min(s.len - j * len * CH, len * CH);
  s.chunk0 += j * len;
  s.nchunks = (s.len + CH - 1) / CH;
  return s;
}

// What a sequential pass works on: sequence number i of the call in the order of seq_at, or (CUT) coarse segment number i.
// CUT is a parameter of the passes: asked at run time whether the call is cut, the passes over whole sequences took
// 1.5 % longer (14 packed sequences of 5542 tokens, 32 heads, K = V = 64: 45.0 -> 45.7 us; 8 x 1181 tokens, 32 heads,
// K = 64, V = 128 with the normaliser: 68.7 -> 69.8).
struct PassItem {
  SeqInfo sq;
  int n;                 // sequence (-1: nothing to do)
  bool first, last;      // the item holds the first / the last chunk of its sequence
};
__device__ __forceinline__ PassItem whole_sequence(const lmoe_args& a, int i) {
  PassItem p;
  p.n = seq_at(a, i);
  p.sq = seq_info(a, p.n);
  p.first = p.last = true;
  return p;
}
template <bool CUT> __device__ __forceinline__ PassItem pass_item(const lmoe_args& a, const Split& sp, int i) {
  if constexpr (!CUT) return whole_sequence(a, i);
  PassItem p;
  const SegInfo g = seg_find(a, sp.len3, i);
  p.n = g.n;
  p.first = g.j == 0;
  p.last = g.j == g.nseg - 1;
  if (g.n >= 0) {
    p.sq = seg_cut(seq_info(a, g.n), g.j, sp.len3);
    p.sq.tok0 = __builtin_amdgcn_readfirstlane(p.sq.tok0);
    p.sq.len = __builtin_amdgcn_readfirstlane(p.sq.len);
    p.sq.chunk0 = __builtin_amdgcn_readfirstlane(p.sq.chunk0);
    p.sq.nchunks = __builtin_amdgcn_readfirstlane(p.sq.nchunks);
  }
  return p;
}
// the same where only dense input is ever cut
template <bool CUT> __device__ __forceinline__ PassItem pass_item_dense(const lmoe_args& a, const Split& sp, int i) {
  if constexpr (!CUT) return whole_sequence(a, i);
  PassItem p;
  const int nseg = seg_count((a.T + CH - 1) / CH, sp.len3), j = i - __builtin_amdgcn_readfirstlane(i / nseg) * nseg;
  p.n = __builtin_amdgcn_readfirstlane(i / nseg);
  p.sq = seg_cut(seq_info(a, p.n), j, sp.len3);
  p.first = j == 0;
  p.last = j == nseg - 1;
  return p;
}
// What the rules below expect of a cut, as a part of the whole call by their figures: 0.9, less at V = 128 where the pass over whole
// sequences takes slices of 16 columns (2-byte elements, a CU for each), which the figures do not know.  Every call that the lower
// limits leave whole was timed both ways, one call replayed as a graph, time cut : whole.
//   chunk_simple_gla, K = V = 128, 0.835: forward 0.99 to 1.29, forward and backward 1.05 to 1.29 (16 pairs of 20 chunks 28.6 : 25.0
//     and 81 : 69 us, 32 of 43 61 : 51 and 177 : 149); with the normaliser 0.94 (16 of 21) to 1.23 and 1.02 to 1.27.  Below, cuts win:
//     0.80 57.3 : 62.1 us forward (16 of 40), 0.83 22.2 : 22.9 (8 of 17; the training call of it loses, 58 : 53).
//   chunk_simple_gla, K = 64, 0.868: 0.91 (8 of 17) to 1.29 and 0.95 (24 of 38) to 1.24; normalised 0.95 to 1.34 and 0.94 to 1.24
//   delta rule, K = V = 128, 0.85: 0.98 (16 of 37) to 1.14 and 1.03 to 1.15
// The same lower limits at the other sizes lost: delta rule K = 64, V = 128 0.92 to 1.07 and 0.95 to 1.05, K = 128, V = 64 0.88 to 1.01
// and 0.94 to 1.05 (28 of 44 62 : 70 and 155 : 165 us), chunk_simple_gla K = 128, V = 64 0.79 to 1.06 and 0.94 to 1.07 (16 of 17 18.4 : 21.6
// and 57 : 58).  At K = V = 64 every cut up to 0.9 wins (by 1.08 to 2), and chunk_gla's do there and at K = V = 128.  Several packed sequences
// keep 0.9: the longest, which the average does not show, gains more.
inline float cut_limit(const lmoe_args& a, float at128, float at64) {
  const bool narrow = (!a.cu_seqlens || a.N == 1) && a.dtype == LMOE_BF16 && a.V == 128 && (int64_t)a.N * a.H * (a.V / 16) <= cu_count();
  return !narrow ? 0.9f : a.K == 128 ? at128 : at64;
}
// How a call is cut (pointers left open), or len1 = 0.  `slices` = work-groups of the ordinary pass per (sequence, head),
// which hold a CU each; the work-groups of step 1 carry all columns and hold a CU each too.  Chosen by what the three steps
// were measured to take (us, K = V = 128, delta rule; half of it per chunk at K = V = 64):
//   ordinary pass   1.7 per chunk up to 64 work-groups, 2.1 beyond, 2.2 on a full GPU
//   step 1          7 + 3.3 per chunk        step 2   4 + 0.65 per fine segment       step 3   1 + 2.2 per chunk
// These are the passes with two and three barriers per chunk the rule was fitted to; the forward pass now takes 1.35 to 1.6 per
// chunk, with slices of 16 columns less (cut_limit).  Where the kernels count (one pass replayed as a graph, whole -> cut, K = V = 128):
// training 16 pairs of 48 chunks 170 -> 158, 16 of 256 920 -> 615; forward 16 pairs of 47 chunks 80 -> 63, 8 of 32 48 -> 43.  A
// training call of up to 48 chunks that the
// host issues one by one is bound by the host, and the cut's launches show (8 pairs of 24 chunks 125 -> 140).
inline Split plan_split(const lmoe_args& a, int slices) {
  Split s = {};
  if (a.dtype != LMOE_BF16 || a.N < 1 || a.T < 1) return s;
  const int cus = cu_count(), slots = cus / (a.H * slices);       // coarse segments that fill the CUs, all sequences together
  // at least three coarse segments each: with two, the longest sequence that gained (256 chunks, 32 pairs) took 0.8 of
  // the time, most 0.9 and more
  if (slots < 3 * a.N) return s;
  // Packed: the lengths are not known here, as if they were equal.  T and N alone decide: NT is the chunk count where the
  // offsets lie on the host and a bound where they lie on the device, and a batch gives the same bits either way.
  // A sequence then has T / 64 / N chunks, or one more for the partial ones; cut if the model gains with either: it sees the
  // average, and the longest sequence decides what the pass takes in one piece (with the smaller count alone six sequences
  // of 20 229 tokens, 4 heads, K = V = 64 were left whole: 62 -> 215 us).
  const bool packed = a.cu_seqlens != nullptr;
  const int seqs = packed ? a.N : 1, chunks = seg_count(a.T, CH), least = seg_count(chunks, seqs);
  const float w = (a.K + a.V) / 256.f;
  // packed: sum over the sequences of ceil(chunks / len3) <= NT / len3 + N segments
  const int rmax = packed && a.N > 1 ? (slots - a.N) / a.N : slots / a.N;
  if (chunks > seqs * SPLIT_MAX_CHUNKS) return s;
  for (int nch = packed ? seg_count(chunks + seqs, seqs) : least; nch >= least && nch >= SPLIT_MIN_CHUNKS && !s.len1; --nch) {
    float best = cut_limit(a, 0.85f, 0.9f) * nch * w * (a.N * a.H * slices <= 64 ? 1.7f : 2.1f);
    for (int r = 3; r <= rmax && r <= 32; ++r)
      for (int f = 1; f <= 4; ++f) {
        const int len3 = seg_count(nch, r), len1 = seg_count(len3, f), nf = seg_count(nch, len1);
        const int rounds = seg_count(a.N * a.H * nf, cus);
        const float t = 12.f + 3.3f * w * len1 * rounds + 0.65f * w * (nf - f) + 2.2f * w * (len1 * f);
        if (t < best) { best = t; s.len1 = len1; s.len3 = len1 * f; }
      }
  }
  if (!s.len1) return s;
  s.n1 = packed ? a.NT / s.len1 + a.N : a.N * seg_count(chunks, s.len1);
  s.n3 = packed ? a.NT / s.len3 + a.N : a.N * seg_count(chunks, s.len3);
  return s;
}
// The cut of a dense call whose step 2 is a few loads at the start of the pass.  c3 us per chunk of the ordinary pass, b3
// more where every CU runs one, wg3 its work-groups; c1, wg1 the same of step 1, per fine segment.  A work-group of the
// pass takes 2.5 to start, and `pre` per fine segment it starts from: work-groups in several rounds pay that every time.
// Without these two terms 16 pairs of 49 chunks (K = V = 128, retention) were cut into 25 (1600 work-groups of two chunks,
// 82 us for the pass that takes 64 in one piece), 28 pairs of 110 chunks into 16 (123 against 138).
inline Split plan_cut(const lmoe_args& a, float limit, float c3, float b3, float c1, float pre, int64_t wg3, int64_t wg1) {
  Split s = {};
  const int cus = cu_count(), nch = (a.T + CH - 1) / CH;
  const float w = (a.K + a.V) / 256.f;
  auto rounds = [](int64_t n, int64_t per) { return (float)((n + per - 1) / per); };
  auto pass = [&](int64_t wg, int chunks) {             // (the last round may leave CUs idle)
    const int64_t full = wg / cus, rest = wg % cus;
    return 2.5f * rounds(wg, cus) + chunks * (full * (c3 + b3) + (rest ? c3 + b3 * rest / cus : 0.f));
  };
  float best = limit * pass(wg3, nch);
  for (int r = 2; r <= 32 && r <= nch; ++r) {
    const int len3 = seg_count(nch, r);
    if (seg_count(nch, len3) != r) continue;
    for (int f = 1; f <= 4; ++f) {
      if (len3 % f) continue;
      const int len1 = len3 / f, nf = seg_count(nch, len1);
      const int64_t segs = wg1 * (r - 1) * f;
      // step 1: two work-groups to a CU, and what they write; the pass: the last segment starts from all, the average
      // one from half of them
      const float t = 8.f + c1 * len1 * rounds(segs, 2 * cus) + 0.015f * w * segs + pass(wg3 * r, len3) +
                      pre * (r - 1) * f * fmaxf(1.f, 0.5f * rounds(wg3 * r, cus));
      if (t < best) { best = t; s.len1 = len1; s.len3 = len3; s.n1 = a.N * nf; s.n3 = a.N * r; }
    }
  }
  return s;
}
// The same for chunk_simple_gla, whose transitions are numbers: step 2 is a few loads at the start of the pass
// (seg_prefix), and a cut pays from a handful of chunks on.  Dense input only (the places of packed sequences are not
// known here).  Measured, us per chunk of the ordinary pass (V slices of 32, 4-byte elements 16): K = V = 64 0.88,
// 128 1.3; 4-byte elements 3.9, 6.0 (whatever the number of work-groups, up to one per CU).  us per call, not cut -> cut:
// forward K = V = 128, T = 4096, 16 pairs 82 -> 52, 4 pairs 80 -> 34; K = V = 64, T = 8192, 8 pairs 113 -> 32; 4-byte
// elements K = V = 64, 4 pairs, T = 512 33.8 -> 13.6 (kernels alone), T = 2048 124 -> 28; with the normaliser, forward +
// backward, K = V = 128, T = 8192, 8 pairs 383 -> 172.  64 pairs at K = V = 128 fill the CUs: never cut.
inline Split plan_split_scalar(const lmoe_args& a) {
  const Split s = {};
  if (a.N < 1 || a.T < 1 || a.cu_seqlens) return s;
  const bool f4 = a.dtype != LMOE_BF16;
  const int cus = cu_count(), nch = (a.T + CH - 1) / CH, pairs = a.N * a.H;
  if (!f4 && (int64_t)pairs * (a.V / 64) >= cus) return s;        // the pass takes wide slices there and fills the CUs
  // (2-byte elements: up to 16 chunks a cut saves 5 us at most; those and very long sequences are left whole and give the
  // same bits alone and in a batch that fills the CUs)
  if (nch < (f4 ? 3 : 17) || nch > SPLIT_MAX_CHUNKS) return s;
  const float w = (a.K + a.V) / 256.f;
  const int64_t wg3 = (int64_t)pairs * (a.V / (f4 ? 16 : 32));
  // (the passes of a normalised call ask for more per chunk: 128 work-groups of K = 64, V = 128 in two took 270 -> 297 for
  // forward and backward together, 384 of K = V = 128 759 -> 857)
  if (!f4 && a.normalize && 2 * wg3 >= cus) return s;
  const float c3 = f4 ? 1.9f + 4.1f * w : 0.45f + 0.85f * w, c1 = f4 ? 1.f + 2.f * w : 0.3f + 0.6f * w;
  return plan_cut(a, cut_limit(a, 0.835f, 0.868f), c3, f4 ? 0.f : 0.3f * w, c1, (f4 ? 0.25f : 0.5f) * w, wg3, (int64_t)pairs * (f4 ? a.V / 32 : 1));
}
// The same for chunk_gla (2-byte elements, dense; a transition is one decay per state row).  The pass fetches q, k and the
// intra-chunk matrix once per V slice of 32, so a chunk costs more the more CUs run one.  Measured, us per chunk with 64, 128,
// 256 work-groups: K = V = 64 0.8-1.0, 1.2, 1.6, K = V = 128 1.0, 1.2-1.7, 1.8-2.2; step 1 6-9 + 1.3 per chunk (128).
// us of pass + step 1, not cut -> cut: forward K = V = 128, T = 4096, 16 pairs 64 -> 40, T = 8192, 4 pairs 120 -> 41; K = 64,
// V = 128, T = 8192, 8 pairs 89 -> 33 (backward 65 -> 34).  32 pairs, T = 2048, K = V = 128 in two would take 39 -> 54: not cut.
inline Split plan_split_gla(const lmoe_args& a) {
  if (a.N < 1 || a.T < 1 || a.cu_seqlens || a.dtype != LMOE_BF16) return Split{};
  const int nch = (a.T + CH - 1) / CH, pairs = a.N * a.H;
  // wide slices fill the CUs; short and very long sequences are left whole, as above
  if ((int64_t)pairs * (a.V / 64) >= cu_count() || nch < 17 || nch > SPLIT_MAX_CHUNKS) return Split{};
  const float w = (a.K + a.V) / 256.f;
  return plan_cut(a, 0.9f, 0.35f + 0.4f * w, 0.6f + 0.4f * w, 0.4f + 0.8f * w, 0.5f * w, (int64_t)pairs * (a.V / 32), pairs);
}
// S <- D S + Q over the n fine segments in front of a coarse one, in order (step = -1: behind it, from the last on).
// q, d: Q (its column v0 + lane % 16, row krow0 + 4 (lane / 16)) and D of the first; four segments' loads at a time.
template <int K, int V, int MB, int NB>
__device__ __forceinline__ void seg_prefix(f32x4 (&S)[MB][NB], const float* q, const float* d, int H, int n, int step) {
  const int64_t qs = (int64_t)step * H * V * K, ds = (int64_t)step * H;
  for (int i0 = 0; i0 < n; i0 += 4) {
    f32x4 x[4][MB][NB];
    float dec[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = min(i0 + u, n - 1);
      dec[u] = d[i * ds];
#pragma unroll
      for (int mi = 0; mi < MB; ++mi)
#pragma unroll
        for (int ni = 0; ni < NB; ++ni) x[u][mi][ni] = *(const f32x4*)(q + i * qs + 16 * ni * K + 16 * mi);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (i0 + u < n) {
#pragma unroll
        for (int mi = 0; mi < MB; ++mi)
#pragma unroll
          for (int ni = 0; ni < NB; ++ni) S[mi][ni] = S[mi][ni] * dec[u] + x[u][mi][ni];
      }
    }
  }
}
// the same for the column of the normaliser (no decay: ungated calls)
template <int K, int MB> __device__ __forceinline__ void seg_prefix_z(f32x4 (&z)[MB], const float* p, int H, int n, int step) {
  const int64_t zs = (int64_t)step * H * K;
  for (int i = 0; i < n; ++i)
#pragma unroll
    for (int mi = 0; mi < MB; ++mi) z[mi] += *(const f32x4*)(p + i * zs + 16 * mi);
}
// chunk_gla: a decay per state row (d: D at row krow0 + 4 (lane / 16) of the first segment)
template <int K, int V, int MB, int NB>
__device__ __forceinline__ void seg_prefix_rows(f32x4 (&S)[MB][NB], const float* q, const float* d, int H, int n, int step) {
  const int64_t qs = (int64_t)step * H * V * K, ds = (int64_t)step * H * K;
  for (int i0 = 0; i0 < n; i0 += 4) {
    f32x4 x[4][MB][NB], dec[4][MB];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = min(i0 + u, n - 1);
#pragma unroll
      for (int mi = 0; mi < MB; ++mi) {
        dec[u][mi] = *(const f32x4*)(d + i * ds + 16 * mi);
#pragma unroll
        for (int ni = 0; ni < NB; ++ni) x[u][mi][ni] = *(const f32x4*)(q + i * qs + 16 * ni * K + 16 * mi);
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (i0 + u < n) {
#pragma unroll
        for (int mi = 0; mi < MB; ++mi)
#pragma unroll
          for (int ni = 0; ni < NB; ++ni) S[mi][ni] = S[mi][ni] * dec[u][mi] + x[u][mi][ni];
      }
    }
  }
}
inline int pass_items(const lmoe_args& a, const Split& sp) { return sp.len3 ? sp.n3 : a.N; }

}  // namespace lmoe
