// Gated delta rule: the fine segments of sequences that are cut along T (lmoe_split.hpp), run for their state alone.
//
//   forward  (k_gdn_seg_fwd): per chunk  X = k S;  Z = beta v - beta e^{b} X;  v_new = Tinv Z;  S <- e^{b_C} S + k^T (e_d v_new)
//     from S = 0 on the V columns of v (contribution Q) and from S = 1 on K columns with v = 0 (transition P).
//   backward (k_gdn_seg_bwd): per chunk from the end  dv_new = scale P^T do + e_d (k dS');  dZ = Tinv^T dv_new;
//     dS = e^{b_C} dS' + q^T (scale e_b do) - (k beta e^{b})^T dZ   from dS' = 0 (its transition is the transposed P).
//
// P is handed on as D 1 + R with D = the product of the chunk decays in fp32 and R in the 2-byte type, and applied as
// S <- D S + R S + Q with S rounded for the product R S only: what a chunk of the ordinary pass does to the state (the
// carry in fp32, the update through 2-byte operands).
// TWO (calls without a gate): nothing fades, and these two roundings per segment show beside those of the chunks: against
// float64 o, dq and dk were off by 1.04 times as much as behind the pass over whole sequences, the final state by up to
// 1.25 times where v falls to a hundredth half way.  R and the rounded S are then carried as two 2-byte terms each (hi hi +
// hi lo + lo hi): 0.94 to 1.00 of the whole pass's error.  16 heads, 3001 tokens, K = V = 128: 61 -> 66 us (whole 92).
// Gated calls stay at one term: 1.00 with the decays of a mixer (A in 1 .. 16), 0.96 at a decay of 0.002 per token.
//
// One work-group carries all columns of a segment: k, Tinv (q, the intra-chunk P) are fetched once per chunk for up to
// V + K (V) columns, where the slices of the ordinary pass fetch them once per 32.  Every wave owns all K rows of 32
// (backward: 16) columns in registers (accumulators of one product are operands of the next, an operand fragment from LDS serves two column blocks) and every wave loads: two LDS buffers, one barrier per
// chunk, the next chunk's loads in flight over the whole of this one.  2-byte elements only.
#pragma once
#include "lmoe_gdn_state_reg.hpp"
#include "lmoe_split.hpp"

namespace lmoe {

// A [64][COLS] tile moved by NT threads: registers <- memory (rows past the end re-read the last one), LDS <- registers.
template <int COLS, int NT> struct WideTile {
  static constexpr int VPR = COLS / 8, NVEC = CH * VPR, PASSES = (NVEC + NT - 1) / NT;
  struct Regs { bf16x8 v[PASSES]; };
  static __device__ __forceinline__ void coords(int p, int& row, int& col) {
    const int idx = min(p * NT + (int)threadIdx.x, NVEC - 1);     // (a thread past the tile repeats its last vector)
    row = idx / VPR; col = (idx % VPR) * 8;
  }
  static __device__ __forceinline__ void load(Regs& r, const bf16* __restrict__ src, int64_t stride, int len) {
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      int row, col; coords(p, row, col);
      r.v[p] = *(const bf16x8*)(src + (int64_t)min(row, len - 1) * stride + col);
    }
  }
  template <bool SILU = false>
  static __device__ __forceinline__ void store(Regs& r, bf16* tile, int ld, int len, bool act = false) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      int row, col; coords(p, row, col);
      if constexpr (SILU) {
        if (act) {
#pragma unroll
          for (int i = 0; i < 8; ++i) r.v[p][i] = (bf16)silu_of((float)r.v[p][i]);
        }
      }
      if (len < CH) {                                             // uniform: only the last chunk of a sequence
        u32x4 w = __builtin_bit_cast(u32x4, r.v[p]);
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = row < len ? w[i] : 0u;
        r.v[p] = __builtin_bit_cast(bf16x8, w);
      }
      *(bf16x8*)(tile + row * ld + col) = r.v[p];
    }
  }
};

// Row stride of a tile of D columns read row by row (16-byte fragments: 8 cycles of the LDS) and through the transposing
// reads of load_frag_t_state: 5.5 cycles at 80 or 48 words, 8 at 68 or 36 (measured, eight waves)
template <int D> constexpr int seg_ld = D + 32;
// Numbering of accumulator rows and operands as in lmoe_gdn_state_reg.hpp: element i of block m in lane group g is row
// 32 (m / 2) + 8 g + 4 (m % 2) + i, lane r of an A operand reads row 32 (m / 2) + 8 (r / 4) + 4 (m % 2) + r % 4
__device__ __forceinline__ int acc_row4(int m, int g) { return 32 * (m >> 1) + 8 * g + 4 * (m & 1); }
__device__ __forceinline__ int frag_row(int m, int fr) { return 32 * (m >> 1) + 4 * (m & 1) + 8 * (fr >> 2) + (fr & 3); }
__device__ __forceinline__ bf16x8 row_frag(const bf16* row, int ks, int g) { return *(const bf16x8*)(row + 32 * ks + 8 * g); }

template <int KT, int NCB>
__device__ __forceinline__ void load_state(f32x4 (&S)[KT][NCB], const float* __restrict__ p, int W, int col, int g) {
#pragma unroll
  for (int mi = 0; mi < KT; ++mi)
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[mi][cb][i] = p[(int64_t)(acc_row4(mi, g) + i) * W + col + 16 * cb];
}
// S[mi][cb] <- dec S + tile^T bv over the 64 tokens of a [64][K] tile (bv: two 32-token operands per column block).  A
// group of four fragments is requested, and the next four blocks of S scaled, while the products of the group before
// run (sched_mix); `first` = the group the caller has requested, whose blocks it has scaled.
struct Frags4 { bf16x8 f[4]; };
// instruction mix of a region of n products: behind each up to `valu` vector instructions and one LDS read (a wave
// issues in order: products in a row each wait for the matrix pipe, and so does whatever stands behind them)
template <int N, int VALU> __device__ __forceinline__ void sched_mix() {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, VALU, 0);
  }
}
__device__ __forceinline__ void state_frags(Frags4& x, const bf16* tile, int ld, int s, int m0, int l) {
#pragma unroll
  for (int m = 0; m < 4; ++m) x.f[m] = load_frag_t_state(tile, ld, 32 * s, m0 + m, l);
}
template <int KT, int NCB>
__device__ __forceinline__ void state_scale(f32x4 (&S)[KT][NCB], int m0, float dec) {
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) S[m0 + m][cb] *= dec;
}
template <int KT, int NCB, bool SCALE>
__device__ __forceinline__ void state_update(f32x4 (&S)[KT][NCB], const bf16* tile, int ld, const bf16x8 (&bv)[2][NCB], const Frags4& first, float dec, int l) {
  constexpr int NG = KT / 4;
  Frags4 x[2];
  x[0] = first;
#pragma unroll
  for (int i = 0; i < 2 * NG; ++i) {
    __builtin_amdgcn_sched_barrier(0);
    if (i + 1 < 2 * NG) state_frags(x[(i + 1) & 1], tile, ld, (i + 1) / NG, 4 * ((i + 1) % NG), l);
    if (SCALE && i + 1 < NG) state_scale<KT, NCB>(S, 4 * (i + 1), dec);
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) ET<bf16>::mma(S[4 * (i % NG) + m][cb], x[i & 1].f[m], bv[i / NG][cb]);
    sched_mix<4 * NCB, 2>();
  }
  __builtin_amdgcn_sched_barrier(0);
}
// X = tile S for the 64 rows of a [64][K] tile, likewise one step of fragments ahead; `tail` runs with the last products
// (the caller requests there what it reads next)
template <int KS, int NCB, typename F>
__device__ __forceinline__ void tile_times_state(f32x4 (&X)[4][NCB], const bf16* tile, int ld, const f32x4 (&S)[2 * KS][NCB], int fr, int g, F&& tail) {
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) X[t][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 fk[2][4], bS[2][NCB];
#pragma unroll
  for (int t = 0; t < 4; ++t) fk[0][t] = row_frag(tile + frag_row(t, fr) * ld, 0, g);
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) bS[0][cb] = frag_of_blocks(S[0][cb], S[1][cb]);
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    __builtin_amdgcn_sched_barrier(0);
    if (ks + 1 < KS) {
#pragma unroll
      for (int t = 0; t < 4; ++t) fk[(ks + 1) & 1][t] = row_frag(tile + frag_row(t, fr) * ld, ks + 1, g);
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) bS[(ks + 1) & 1][cb] = frag_of_blocks(S[2 * ks + 2][cb], S[2 * ks + 3][cb]);
    } else {
      tail();
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) ET<bf16>::mma(X[t][cb], fk[ks & 1][t], bS[ks & 1][cb]);
    sched_mix<4 * NCB, 2>();
  }
  __builtin_amdgcn_sched_barrier(0);
}

// A [K][K] matrix M in the order of A operands: for block row rb and contraction step ks, lane l = 16 g + r holds
// M[16 rb + r][32 ks + 8 g ..+7] at frag_slot + 8 l: every load of a wave is 1 KB in one piece.
template <int K> __host__ __device__ constexpr int frag_slot(int rb, int ks) { return (rb * (K / 32) + ks) * 512; }

// 2-byte terms a number of R is carried in
template <bool TWO> constexpr int split_terms = TWO ? 2 : 1;

constexpr int SEG_FWD_THREADS = 512;      // waves 0 .. 3: up to 128 columns of Q, waves 4 .. 7: of P; all eight load
// the part of one wave of fine segment s1 of head h: 32 of the W columns of Q (TRANS = false, W = V) or of P (W = K)
template <int K, int V, bool TRANS, bool TWO>
__device__ __forceinline__ void seg_fwd_columns(const lmoe_args& a, const Split& sp, int s1, int h, const SegInfo& sg,
                                                const SeqInfo& sq, bool busy, bool in_last3, char* s_mem, float (&s_g)[2][4 * CH]) {
  constexpr int NT = SEG_FWD_THREADS, LDK = seg_ld<K>, LDC = CH + LPAD, LDV = V + LPAD, NCB = 2;
  constexpr int KT = K / 16, KS = K / 32;
  bf16* const s_k = (bf16*)s_mem;
  bf16* const s_ti = s_k + 2 * CH * LDK;
  bf16* const s_v = s_ti + 2 * CH * LDC;
  const int l = lane_id(), fr = l & 15, g = l >> 4, wv = wave_id() & 3;
  const int col0 = 32 * wv;
  typedef WideTile<K, NT> TK;
  typedef WideTile<CH, NT> TC;
  typedef WideTile<V, NT> TV;
  struct Pre { typename TK::Regs k; typename TC::Regs t; typename TV::Regs v; float g; };
  Pre pre;
  auto issue = [&](int c) {
    c = min(c, sq.nchunks - 1);
    const int tok = sq.tok0 + c * CH;
    const int64_t ch = (int64_t)(sq.chunk0 + c) * a.H + h;
    TK::load(pre.k, row_ptr<bf16>(a.k, sq.b, tok, h), a.k.st, CH);
    TC::load(pre.t, (const bf16*)a.tinv + ch * CH * CH, CH, CH);
    TV::load(pre.v, row_ptr<bf16>(a.v, sq.b, tok, h), a.v.st, CH);
    pre.g = a.gcum[ch * GATE_ROWS * CH + (threadIdx.x & 255)];
  };
  auto stage = [&](int buf) {                                     // (every chunk here is full: a partial one ends its sequence)
    TK::store(pre.k, s_k + buf * CH * LDK, LDK, CH);
    TC::store(pre.t, s_ti + buf * CH * LDC, LDC, CH);
    TV::template store<true>(pre.v, s_v + buf * CH * LDV, LDV, CH, a.v_act != 0);
    s_g[buf][threadIdx.x & 255] = pre.g;                          // (waves 4 .. 7: the same bytes again)
  };
  issue(0);
  f32x4 S[KT][2];
  float D = 1.f;
#pragma unroll
  for (int mi = 0; mi < KT; ++mi)
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[mi][cb][i] = TRANS && (acc_row4(mi, g) + i) == col0 + 16 * cb + fr ? 1.f : 0.f;
  if (!TRANS && busy && sg.j == 0 && a.h0) load_state<KT, NCB>(S, a.h0 + ((int64_t)sg.n * a.H + h) * K * V, V, col0 + fr, g);
  stage(0);
  issue(1);
  lds_barrier();
  for (int c = 0; c < sq.nchunks; ++c) {
    const int cur = c & 1;
    const bf16 *tk = s_k + cur * CH * LDK, *ti = s_ti + cur * CH * LDC, *tv = s_v + cur * CH * LDV;
    const float* tg = s_g[cur];
    if (busy) {
      f32x4 X[4][2], be[4], ff[4], ed[4];
      bf16x8 fv[2][2], fti[6];
      tile_times_state<KS, NCB>(X, tk, LDK, S, fr, g, [&]() {
#pragma unroll
        for (int m = 0; m < 4; ++m) ff[m] = *(const f32x4*)&tg[3 * CH + acc_row4(m, g)];
        if constexpr (!TRANS) {
#pragma unroll
          for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int cb = 0; cb < 2; ++cb) fv[s][cb] = ET<bf16>::load_frag_t(tv, LDV, 32 * s, col0 + 16 * cb, l);
#pragma unroll
          for (int m = 0; m < 4; ++m) be[m] = *(const f32x4*)&tg[2 * CH + acc_row4(m, g)];
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) fti[t] = row_frag(ti + frag_row(t, fr) * LDC, 0, g);
        fti[4] = row_frag(ti + frag_row(2, fr) * LDC, 1, g);
        fti[5] = row_frag(ti + frag_row(3, fr) * LDC, 1, g);
      });
      bf16x8 Z[2][2];
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
          for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float x = ff[2 * s + e][i] * X[2 * s + e][cb][i];
              if constexpr (TRANS) Z[s][cb][4 * e + i] = (bf16)-x;
              else Z[s][cb][4 * e + i] = (bf16)__builtin_fmaf(be[2 * s + e][i], (float)fv[s][cb][4 * e + i], -x);
            }
      Frags4 first;
      state_frags(first, tk, LDK, 0, 0, l);
#pragma unroll
      for (int m = 0; m < 4; ++m) ed[m] = *(const f32x4*)&tg[CH + acc_row4(m, g)];
      const float dec = tg[CH - 1];
      __builtin_amdgcn_sched_barrier(0);
      f32x4 vn[4][2];                                             // v_new = Tinv Z (Tinv is lower triangular)
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
          vn[t][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
          ET<bf16>::mma(vn[t][cb], fti[t], Z[0][cb]);
        }
#pragma unroll
      for (int t = 2; t < 4; ++t)
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) ET<bf16>::mma(vn[t][cb], fti[2 + t], Z[1][cb]);
      state_scale<KT, NCB>(S, 0, dec);
      if constexpr (TRANS) D *= dec;
      __builtin_amdgcn_sched_barrier(0);
      bf16x8 bv[2][2];
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) bv[s][cb] = frag_of_blocks(vn[2 * s][cb] * ed[2 * s], vn[2 * s + 1][cb] * ed[2 * s + 1]);
      state_update<KT, NCB, true>(S, tk, LDK, bv, first, dec, l);
    }
    stage(1 - cur);
    issue(c + 2);
    lds_barrier();
  }
  const int64_t slot = (int64_t)s1 * a.H + h;
  if constexpr (!TRANS) {
    if (!busy) return;
    float* out = sp.Q + slot * K * V;
#pragma unroll
    for (int mi = 0; mi < KT; ++mi)
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int i = 0; i < 4; ++i) out[(int64_t)(acc_row4(mi, g) + i) * V + col0 + 16 * cb + fr] = S[mi][cb][i];
  } else {
    // R in the order in which the combination reads it as an operand (frag_slot): R^T as it lies in the accumulators,
    // R through LDS ([column][row], transposing reads)
    constexpr int LDP = K + LPAD, RK = split_terms<TWO> * K * K;
    bf16* const s_r = (bf16*)s_mem;
    if (busy) {
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
          for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (acc_row4(2 * ks + e, g) + i == col0 + 16 * cb + fr) S[2 * ks + e][cb][i] -= D;
          const bf16x8 x = frag_of_blocks(S[2 * ks][cb], S[2 * ks + 1][cb]);
          bf16* const pt = sp.PT + slot * RK + frag_slot<K>((col0 >> 4) + cb, ks) + 8 * l;
          bf16* const r = s_r + (col0 + 16 * cb + fr) * LDP + 32 * ks + 8 * g;
          if (sp.PT) *(bf16x8*)pt = x;
          *(bf16x8*)r = x;
          if constexpr (TWO) {
            bf16x8 y;
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] = (bf16)(S[2 * ks + (e >> 2)][cb][e & 3] - (float)x[e]);
            if (sp.PT) *(bf16x8*)(pt + K * K) = y;
            *(bf16x8*)(r + K * LDP) = y;
          }
        }
      if (wv == 0 && l == 0) {
        if (sp.PT) sp.DT[slot] = D;
        sp.D[slot] = D;
      }
    }
    if (in_last3 || sg.j == 0) return;                            // (the transitions of the last coarse segment serve the backward only)
    lds_barrier();
    for (int u = wv; u < (K / 16) * KS; u += 4) {
      const int rb = u / KS, ks = u % KS;
      bf16* const p = sp.P + slot * RK + frag_slot<K>(rb, ks) + 8 * l;
      *(bf16x8*)p = ET<bf16>::load_frag_t(s_r, LDP, 32 * ks, 16 * rb, l);
      if constexpr (TWO) *(bf16x8*)(p + K * K) = ET<bf16>::load_frag_t(s_r + K * LDP, LDP, 32 * ks, 16 * rb, l);
    }
  }
}

// grid: (fine segment, head)
template <int K, int V, bool TWO>
__global__ __launch_bounds__(SEG_FWD_THREADS) void k_gdn_seg_fwd(const lmoe_args a, const Split sp) {
  static_assert(V <= 128 && K <= 128, "a wave per 32 columns");
  constexpr int LDK = seg_ld<K>, LDC = CH + LPAD, LDV = V + LPAD;
  constexpr int TILES = 2 * (CH * LDK + CH * LDC + CH * LDV) * 2, RBYTES = split_terms<TWO> * K * (K + LPAD) * 2;
  __shared__ __attribute__((aligned(16))) char s_mem[TILES > RBYTES ? TILES : RBYTES];
  __shared__ __attribute__((aligned(16))) float s_g[2][4 * CH];   // e^b, e^{b_C - b}, beta, beta e^b
  const int h = blockIdx.x % a.H, s1 = blockIdx.x / a.H;
  const SegInfo sg = seg_find(a, sp.len1, s1);
  if (sg.n < 0 || sg.j == sg.nseg - 1) return;                    // (the last segment's end is nobody's start)
  const SeqInfo whole = seq_info(a, sg.n);
  // Q of what lies before the last coarse segment; P of every segment but the first (of those of the last coarse
  // segment for the backward, where there is one)
  const bool in_last3 = sg.j * sp.len1 / sp.len3 == (whole.nchunks - 1) / sp.len3;
  if (in_last3 && (whole.nchunks <= sp.len3 || !sp.PT)) return;
  const SeqInfo sq = seg_cut(whole, sg.j, sp.len1);
  const int wv = wave_id();
  if (wv >= 4) seg_fwd_columns<K, V, true, TWO>(a, sp, s1, h, sg, sq, sg.j > 0 && 32 * (wv - 4) < K, in_last3, s_mem, s_g);
  else seg_fwd_columns<K, V, false, TWO>(a, sp, s1, h, sg, sq, !in_last3 && 32 * wv < V, in_last3, s_mem, s_g);
}

constexpr int SEG_BWD_THREADS = 512;      // 16 of the V columns per wave

template <int K, int V>
__global__ __launch_bounds__(SEG_BWD_THREADS) void k_gdn_seg_bwd(const lmoe_args a, const Split sp) {
  constexpr int NT = SEG_BWD_THREADS, LDK = seg_ld<K>, LDC = CH + LPAD, LDV = V + LPAD;
  constexpr int KT = K / 16, KS = K / 32, NCB = 1;
  __shared__ __attribute__((aligned(16))) bf16 b_k[2][CH * LDK], b_q[2][CH * LDK], b_ti[2][CH * LDC], b_p[2][CH * LDC], b_do[2][CH * LDV];
  __shared__ __attribute__((aligned(16))) float b_g[2][4 * CH];   // e^b, e^{b_C - b}, beta, beta e^b
  const int h = blockIdx.x % a.H, s1 = blockIdx.x / a.H;
  const SegInfo sg = seg_find(a, sp.len1, s1);
  if (sg.n < 0 || sg.j * sp.len1 < sp.len3) return;               // (nothing precedes the first coarse segment)
  const int l = lane_id(), fr = l & 15, g = l >> 4, wv = wave_id();
  const int col0 = 16 * wv;
  const bool busy = col0 < V;
  const SeqInfo sq = seg_cut(seq_info(a, sg.n), sg.j, sp.len1);
  typedef WideTile<K, NT> TK;
  typedef WideTile<CH, NT> TC;
  typedef WideTile<V, NT> TV;
  struct Pre { typename TK::Regs k, q; typename TC::Regs t, p; typename TV::Regs d; float g; };
  Pre pre;
  auto clen = [&](int c) { return min(CH, sq.len - c * CH); };
  auto issue = [&](Pre& p, int c) {
    c = max(c, 0);
    const int tok = sq.tok0 + c * CH, len = clen(c);
    const int64_t ch = (int64_t)(sq.chunk0 + c) * a.H + h;
    TK::load(p.k, row_ptr<bf16>(a.k, sq.b, tok, h), a.k.st, len);
    TK::load(p.q, row_ptr<bf16>(a.q, sq.b, tok, h), a.q.st, len);
    TC::load(p.t, (const bf16*)a.tinv + ch * CH * CH, CH, CH);
    TC::load(p.p, (const bf16*)a.pmat + ch * CH * CH, CH, CH);
    TV::load(p.d, row_ptr<bf16>(a.d_o, sq.b, tok, h), a.d_o.st, len);
    p.g = a.gcum[ch * GATE_ROWS * CH + (threadIdx.x & 255)];
  };
  auto stage = [&](Pre& p, int c, int buf) {
    const int len = clen(max(c, 0));
    TK::store(p.k, b_k[buf], LDK, len);
    TK::store(p.q, b_q[buf], LDK, len);
    TC::store(p.t, b_ti[buf], LDC, CH);
    TC::store(p.p, b_p[buf], LDC, CH);
    TV::store(p.d, b_do[buf], LDV, len);
    b_g[buf][threadIdx.x & 255] = p.g;
  };
  issue(pre, sq.nchunks - 1);
  const float scale = a.scale;
  f32x4 S[KT][NCB];
#pragma unroll
  for (int mi = 0; mi < KT; ++mi)
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) S[mi][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (busy && sg.j == sg.nseg - 1 && a.dht) load_state<KT, NCB>(S, a.dht + ((int64_t)sg.n * a.H + h) * K * V, V, col0 + fr, g);
  stage(pre, sq.nchunks - 1, 0);
  issue(pre, sq.nchunks - 2);
  lds_barrier();
  for (int c = sq.nchunks - 1, cur = 0; c >= 0; --c, cur ^= 1) {
    const bf16 *s_k = b_k[cur], *s_q = b_q[cur], *s_ti = b_ti[cur], *s_p = b_p[cur], *s_do = b_do[cur];
    const float* s_g = b_g[cur];
    if (busy) {
    f32x4 X[4][NCB], ed[4], ff[4], eb[4];
    bf16x8 fd[2][NCB], fp[6], ft[6], dvn[2][NCB];
    tile_times_state<KS, NCB>(X, s_k, LDK, S, fr, g, [&]() {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) fd[s][cb] = ET<bf16>::load_frag_t(s_do, LDV, 32 * s, col0 + 16 * cb, l);
#pragma unroll
      for (int t = 0; t < 4; ++t) fp[t] = load_frag_t_state(s_p, LDC, 32, t, l);
      fp[4] = load_frag_t_state(s_p, LDC, 0, 0, l);
      fp[5] = load_frag_t_state(s_p, LDC, 0, 1, l);
#pragma unroll
      for (int m = 0; m < 4; ++m) ed[m] = *(const f32x4*)&s_g[CH + acc_row4(m, g)];
    });
#pragma unroll
    for (int t = 0; t < 4; ++t) ft[t] = load_frag_t_state(s_ti, LDC, 32, t, l);
    ft[4] = load_frag_t_state(s_ti, LDC, 0, 0, l);
    ft[5] = load_frag_t_state(s_ti, LDC, 0, 1, l);
#pragma unroll
    for (int m = 0; m < 4; ++m) { ff[m] = *(const f32x4*)&s_g[3 * CH + acc_row4(m, g)]; eb[m] = *(const f32x4*)&s_g[acc_row4(m, g)]; }
    __builtin_amdgcn_sched_barrier(0);
    f32x4 y[4][NCB];                                                // P^T do (P, Tinv are lower triangular)
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) {
        y[t][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
        ET<bf16>::mma(y[t][cb], fp[t], fd[1][cb]);
      }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) ET<bf16>::mma(y[t][cb], fp[4 + t], fd[0][cb]);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
        for (int i = 0; i < 4; ++i) dvn[t >> 1][cb][4 * (t & 1) + i] = (bf16)__builtin_fmaf(scale, y[t][cb][i], ed[t][i] * X[t][cb][i]);
    Frags4 first;
    state_frags(first, s_q, LDK, 0, 0, l);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 4; ++t)                                   // dZ = Tinv^T dv_new
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) {
        y[t][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
        ET<bf16>::mma(y[t][cb], ft[t], dvn[1][cb]);
      }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) ET<bf16>::mma(y[t][cb], ft[4 + t], dvn[0][cb]);
    const float dec = s_g[CH - 1];
    state_scale<KT, NCB>(S, 0, dec);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
        for (int i = 0; i < 8; ++i) fd[s][cb][i] = (bf16)((float)fd[s][cb][i] * (scale * eb[2 * s + (i >> 2)][i & 3]));
    __builtin_amdgcn_sched_barrier(0);
    state_update<KT, NCB, true>(S, s_q, LDK, fd, first, dec, l);
    bf16x8 bz[2][NCB];
    state_frags(first, s_k, LDK, 0, 0, l);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) bz[s][cb] = frag_of_blocks(-(y[2 * s][cb] * ff[2 * s]), -(y[2 * s + 1][cb] * ff[2 * s + 1]));
    state_update<KT, NCB, false>(S, s_k, LDK, bz, first, dec, l);
    }
    stage(pre, c - 1, cur ^ 1);
    issue(pre, c - 2);
    lds_barrier();
  }
  if (!busy) return;
  float* out = sp.Q + ((int64_t)s1 * a.H + h) * K * V;
#pragma unroll
  for (int mi = 0; mi < KT; ++mi)
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
      for (int i = 0; i < 4; ++i) out[(int64_t)(acc_row4(mi, g) + i) * V + col0 + 16 * cb + fr] = S[mi][cb][i];
}

// The segments of one (sequence, head) combined in order for 16 columns of the state: S <- D_s S + R_s S + Q_s
// (backward: R_s^T, from the end); wave w holds the rows 32 w ..  The operands of the next segment are requested before
// the products of this one.  Leaves the state every coarse segment starts from.  Bound by what a CU gets of R per step
// (K = 128: 32 KB in 0.9 us).
template <int K, bool BWD, bool TWO>
__global__ __launch_bounds__(2 * K) void k_split_combine(const lmoe_args a, const Split sp) {
  constexpr int LD = K + LPAD, KS = K / 32, TERMS = split_terms<TWO>;
  __shared__ __attribute__((aligned(16))) bf16 s_S[2][TERMS][16 * LD];
  const int V = a.V, ncb = V / 16;
  // the column blocks of a pair on one XCD: they read the same P at the same time
  const int jj = blockIdx.x >> 3, cb = jj % ncb, pair = jj / ncb * 8 + (blockIdx.x & 7), h = pair % a.H, n = pair / a.H;
  if (n >= a.N) return;
  const int l = lane_id(), fr = l & 15, g = l >> 4, row0 = 32 * wave_id(), col = 16 * cb + fr;
  const int nch = seq_info(a, n).nchunks;
  const int64_t plane = (int64_t)K * V;
  if (nch == 0) {                                    // no chunk: the state passes through (the ordinary pass has no item for it)
    const float* x = BWD ? a.dht : a.h0;
    float* y = BWD ? a.dh0 : a.ht;
    if (y)
      for (int i = threadIdx.x; i < K * 16; i += 2 * K) {
        const int64_t at = ((int64_t)n * a.H + h) * plane + (int64_t)(i / 16) * V + 16 * cb + i % 16;
        y[at] = x ? x[at] : 0.f;
      }
    return;
  }
  const int f = sp.len3 / sp.len1, nf = seg_count(nch, sp.len1), nc = seg_count(nch, sp.len3);
  if (nc < 2) return;
  const int base1 = seg_base(a, sp.len1, n), base3 = seg_base(a, sp.len3, n);
  const int first = BWD ? nf - 1 : 0, steps = BWD ? nf - 1 - f : (nc - 1) * f - 1;      // products that follow the first segment
  struct Pre { bf16x8 A[TERMS][2][KS]; f32x4 q[2]; float D; };
  Pre pre[2];
  auto load_q = [&](f32x4 (&q)[2], int s) {
    const float* p = sp.Q + ((int64_t)(base1 + s) * a.H + h) * plane + col;
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
      for (int i = 0; i < 4; ++i) q[mi][i] = p[(int64_t)(row0 + 16 * mi + 4 * g + i) * V];
  };
  auto issue = [&](Pre& x, int t) {
    t = max(min(t, steps), 1);
    const int s = BWD ? first - t : t;
    load_q(x.q, s);
    const int64_t slot = (int64_t)(base1 + s) * a.H + h;
    const bf16* R = (BWD ? sp.PT : sp.P) + slot * TERMS * K * K + 8 * l;
    x.D = (BWD ? sp.DT : sp.D)[slot];
#pragma unroll
    for (int u = 0; u < TERMS; ++u)
#pragma unroll
      for (int mi = 0; mi < 2; ++mi)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) x.A[u][mi][ks] = *(const bf16x8*)(R + u * K * K + frag_slot<K>(row0 / 16 + mi, ks));
  };
  f32x4 acc[2];
  load_q(acc, first);
  auto emit = [&](int t) {
    const int s = BWD ? first - t : t;
    if ((BWD ? s : s + 1) % f) return;
    float* p = sp.S + ((int64_t)(base3 + (BWD ? s / f - 1 : (s + 1) / f)) * a.H + h) * plane + col;
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
      for (int i = 0; i < 4; ++i) p[(int64_t)(row0 + 16 * mi + 4 * g + i) * V] = acc[mi][i];
  };
  emit(0);
  if (steps < 1) return;
  issue(pre[0], 1);
  ring_loop<2>(steps, [&](auto slot, const int t0) {
    constexpr int cur = decltype(slot)::value;
    issue(pre[1 - cur], t0 + 2);
#pragma unroll
    for (int mi = 0; mi < 2; ++mi) {
      f32x4 rest = acc[mi];
#pragma unroll
      for (int u = 0; u < TERMS; ++u) {
        bf16x4 x;
#pragma unroll
        for (int i = 0; i < 4; ++i) { x[i] = (bf16)rest[i]; rest[i] -= (float)x[i]; }
        *(bf16x4*)&s_S[cur][u][fr * LD + row0 + 16 * mi + 4 * g] = x;
      }
    }
    lds_barrier();
    bf16x8 b[TERMS][KS];
#pragma unroll
    for (int u = 0; u < TERMS; ++u)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) b[u][ks] = row_frag(&s_S[cur][u][fr * LD], ks, g);
#pragma unroll
    for (int mi = 0; mi < 2; ++mi) acc[mi] = acc[mi] * pre[cur].D + pre[cur].q[mi];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int mi = 0; mi < 2; ++mi) {
        ET<bf16>::mma(acc[mi], pre[cur].A[0][mi][ks], b[0][ks]);
        if constexpr (TWO) {
          ET<bf16>::mma(acc[mi], pre[cur].A[0][mi][ks], b[1][ks]);
          ET<bf16>::mma(acc[mi], pre[cur].A[1][mi][ks], b[0][ks]);
        }
      }
    emit(t0 + 1);
  });
}

}  // namespace lmoe
