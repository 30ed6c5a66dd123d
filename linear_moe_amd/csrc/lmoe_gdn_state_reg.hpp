// Gated delta rule, forward sequential pass for 2-byte elements with the state held in registers as an MFMA operand.
//
//   per chunk:  X = k S;   Z = beta (v - e^{b} X);   v_new = Tinv Z        ( = u - w S with u = Tinv (v beta), w = Tinv (k beta e^{b}) )
//               o = scale [ e^{b} (q S) + P v_new ];   S' = e^{b_C} S + k^T (e_d v_new)
//
// What bounds a sequential pass on this GPU is the rate at which ONE wave gets LDS reads served (about one wave-wide
// read instruction per 23 cycles, whatever its width; measured), not the matrix cores and not the number of barriers:
// the work of a chunk is therefore laid out so that every operand read from LDS is a single 16-byte read per MFMA, no
// operand is read that can stay in registers, and the reads are spread over four waves.
//   * Consumer wave j (waves 0, 1) owns ALL K rows of the 16 columns 16 j .. of the slice.  An accumulator block holds
//     four rows of one column per lane; two blocks give the 8 contraction elements an MFMA B operand wants, so the
//     state enters  k S  -- and v_new enters  k^T (e_d v_new)  -- straight from the registers the previous product left
//     it in.  For that to fit plain 16-byte row reads of the other operand, accumulator rows are NUMBERED accordingly:
//     block pair (2 s, 2 s + 1), lane group g, element i  <->  index 32 s + 8 g + 4 e + i  (e = block parity).  The row an A
//     operand lane reads (k, Tinv rows) and the columns a transposing read addresses (k^T) follow that numbering;
//     nothing is ever permuted in memory.  The same registers are 8 consecutive rows of a column: S^T and v_new^T go to
//     LDS as 16-byte writes.
//   * w and u are never formed: v_new = Tinv Z costs 6 products (Tinv is lower triangular) on top of X = k S.
//   * ONE barrier per chunk.  Every tile exists twice (156 KB of LDS at K = 128) and a window reads only what the window
//     before it completed, so no team waits for another inside a window:
//       consumers, window c:   v_new(c), S at the start of chunk c + 1
//       helpers, window c:     the output of chunk c - 1 (its q S is in their registers, v_new and P of it in LDS), then
//                              q S and P of chunk c
//       team 1, window c:      stores v_new(c - 1), P(c - 1), o(c - 2); stages k(c + 1) and requests the next
//       team 2, window c:      stores S at the start of chunk c; stages q, Tinv, v, gates of c + 1 and requests the next
//     (Two barriers per chunk, P formed by team 1 in front of the second one, which the consumers waited for: a window was 4600
//     cycles, of which the consumers worked 3700; now 3500, and 3300 of them are the consumers' reads.  B=2 H=16 T=2048 K=V=128
//     saving: 58 -> 49 us; forward-only B=4 T=8192: 232 -> 191; the saving call of that size 268 -> 255, now bound by
//     the 600 MB it writes.)
//   * Helper wave j (waves 2, 3) forms the output of the columns 16 j .. from S^T and v_new^T in LDS, transposed so that
//     a lane holds four consecutive columns of one token, and five of the ten blocks of the lower triangle of
//     P = (q k^T) . Gamma over the q rows it reads for q S anyway (two rows of k blocks are all that P adds to its reads; on the
//     loader waves P took 80 KB of reads per chunk).  P never passes through memory on its way to the output; a call
//     that saves for the backward stores it once: every V-slice work-group its share of the rows.
//   * Few (sequence, head) pairs (the rule: lmoe_gdn_state.hip) take slices of BV = 16 columns: one consumer wave, the
//     columns' output split over the helpers by token blocks, the second consumer's wave gone.
//   * The loaders' stores lie behind no branch (the first two windows are peeled off), so that a wait for a load never waits
//     for stores behind it.
#pragma once
#include <type_traits>
#include "lmoe_gdn_state.hpp"
#include "lmoe_split.hpp"

namespace lmoe {

// Time stamps of the traced instance (TRACE = true): every team's leading wave notes the shader clock when it
// enters the window of a chunk, when it arrives at and leaves the barrier at its end and at a few points in between, into LDS
// (a global store would stall the traced wave at the issue); the traced work-group copies them out when it ends.
// Slots: 0 consumer wave, 1 helper wave, 2 loader team 1, 3 loader team 2; marks per (slot, chunk): see
// lmoe_trace_gdn_state_fwd in include/lmoe.h.  The first TRACE_LDS_CHUNKS chunks are recorded (what the LDS has room for beside
// the tiles); the caller's buffer has TRACE_CHUNKS, zero where nothing was recorded.
constexpr int TRACE_CHUNKS = 128, TRACE_MARKS = 8, TRACE_SLOTS = 4, TRACE_LDS_CHUNKS = 48;

// A fragment of k^T for the state block mi (see the numbering above): contraction = tokens k0 + 8 g .. + 7 (rows of
// the tile), lane fr <-> state row  32 (mi / 2) + 8 (fr / 4) + 4 (mi % 2) + fr % 4  (columns of the tile)
__device__ __forceinline__ bf16x8 load_frag_t_state(const bf16* tile, int ld, int k0, int mi, int l) {
  const int s = l & 15;
  const bf16* p = tile + (k0 + 8 * (l >> 4) + (s >> 2)) * ld + 32 * (mi >> 1) + 8 * (s & 3) + 4 * (mi & 1);
  typedef __attribute__((address_space(3))) bf16x4 lds_b4;
  const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_b4*)p);
  const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_b4*)(p + 4 * ld));
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}
// (frag_of_blocks, lmoe_common.hpp: two accumulator blocks -> the 8 contraction elements of an operand)

// f(number, ti, tj) for the blocks (ti >= tj) of the lower triangle of a 4 x 4 arrangement with tj = TA or tj = TB = 3 - TA
template <int TA, int TB, int X = 0, int TI = TA, int TJ = TA, typename F>
__device__ __forceinline__ void static_for_blocks(F&& f) {
  if constexpr (TI < 4) {
    f(std::integral_constant<int, X>(), std::integral_constant<int, TI>(), std::integral_constant<int, TJ>());
    static_for_blocks<TA, TB, X + 1, TI + 1, TJ>(f);
  } else if constexpr (TJ == TA) {
    static_for_blocks<TA, TB, X, TB, TB>(f);
  }
}

template <int K, int V, bool SAVE, bool TRACE = false, bool CUT = false, int BV = 32>
__global__ __launch_bounds__(3 * NTHR) void k_gdn_state_fwd_reg(const lmoe_args a, const Split sp, long long* tr, int traced_wg) {
  typedef bf16 T;
  static_assert(BV == 32 || BV == 16, "a consumer wave per 16 columns");
  constexpr int LDK = K + LPAD, LDC = CH + LPAD, LDU = BV + LPAD;
  constexpr int KT = K / 16, KS = K / 32;
  constexpr int LPA = GdnStateCfg<T>::LPF, LPB = GdnStateCfg<T>::LPF;       // register sets per prefetch ring (3: no change)
  // every tile twice: buffer c & 1 belongs to chunk c (s_hT: the state at its start)
  __shared__ __attribute__((aligned(16))) T s_k[2][CH * LDK];       // k [64][K]
  __shared__ __attribute__((aligned(16))) T s_q[2][CH * LDK];       // q [64][K]
  __shared__ __attribute__((aligned(16))) T s_ti[2][CH * LDC];      // Tinv [64][64]
  __shared__ __attribute__((aligned(16))) T s_p[2][CH * LDC];       // P [64][64]
  __shared__ __attribute__((aligned(16))) T s_v[2][CH * LDU];       // v [64][BV]
  __shared__ __attribute__((aligned(16))) T s_hT[2][BV * LDK];      // S^T [BV][K]
  __shared__ __attribute__((aligned(16))) T s_vT[2][BV * LDC];      // v_new^T [BV][64]
  __shared__ __attribute__((aligned(16))) T s_o[2][CH * LDU];       // o [64][BV]
  __shared__ __attribute__((aligned(16))) float s_gt[2][GATE_ROWS][CH];     // e^b, e^{b_C - b}, beta, beta e^b, b
  __shared__ uint32_t s_tr[TRACE ? TRACE_SLOTS * TRACE_LDS_CHUNKS * TRACE_MARKS : 1];
  __shared__ long long s_tr0;
  auto TR = [&](int slot, int c, int mark) {
    if constexpr (TRACE) {
      if ((int)blockIdx.x == traced_wg && (threadIdx.x & 63) == 0 && c < TRACE_LDS_CHUNKS)
        s_tr[(slot * TRACE_LDS_CHUNKS + c) * TRACE_MARKS + mark] = (uint32_t)__builtin_readcyclecounter();
    }
  };
  if constexpr (TRACE) {
    for (int i = threadIdx.x; i < TRACE_SLOTS * TRACE_LDS_CHUNKS * TRACE_MARKS; i += 3 * NTHR) s_tr[i] = 0;
    if (threadIdx.x == 0) s_tr0 = __builtin_readcyclecounter();
    __syncthreads();
  }

  constexpr int NVS = V / BV;
  const int xcd = blockIdx.x & 7, jj = blockIdx.x >> 3;
  const int vsl = jj % NVS, pair = (jj / NVS) * 8 + xcd;
  if (pair >= (CUT ? sp.n3 : a.N) * a.H) return;
  const int v0 = vsl * BV, h = pair % a.H;
  const PassItem item = pass_item<CUT>(a, sp, pair / a.H);
  if (CUT && item.n < 0) return;
  const int n = item.n;
  const SeqInfo sq = item.sq;
  const int l = lane_id();
  const int team = threadIdx.x / NTHR;
  if (sq.nchunks == 0) {
    if (a.ht && team == 0) {
      for (int idx = threadIdx.x; idx < K * BV; idx += NTHR) {
        const int r = idx / BV, c = v0 + idx % BV;
        const int64_t o = ((int64_t)n * a.H + h) * K * V + (int64_t)r * V + c;
        a.ht[o] = a.h0 ? a.h0[o] : 0.f;
      }
    }
    return;
  }
  typedef TileIO<T, CH, K> IOK;
  typedef TileIO<T, CH, BV> IOV;
  typedef TileIO<T, CH, CH> IOP;
  typedef TileIO<T, BV, K> IOHT;

  auto store_state = [&](int c) {             // hs(c) <- S^T at the start of chunk c
    typename IOHT::Regs rh;
    IOHT::load_lds(rh, s_hT[c & 1], LDK);
    IOHT::template store_global<true>(rh, (T*)a.hs + (((int64_t)(sq.chunk0 + c) * a.H + h) * V + v0) * K, K, BV);
  };

  if (team == 1) {
    // ------------------------- loaders, ring A (k) and all stores -------------------------
    struct PreA { typename IOK::Regs rk; int len; };
    PreA pa[LPA];
    auto issue_a = [&](PreA& P, int c) {      // always issued, chunk index clamped (see k_gdn_state_fwd)
      c = min(c, sq.nchunks - 1);
      const int tok = sq.tok0 + c * CH;
      P.len = min(CH, sq.len - c * CH);
      IOK::load_nomask(P.rk, row_ptr<T>(a.k, sq.b, tok, h), a.k.st, P.len);
    };
    auto stage_a = [&](PreA& P, int c) {
      IOK::mask(P.rk, P.len);
      IOK::store_lds(P.rk, s_k[c & 1], LDK);
    };
    // this work-group's share of the rows of P (formed by the helpers, the whole matrix in s_p): 64 / NVS rows, the same
    // number of bytes from every thread (128 threads with 16 bytes each and 128 that repeated them, so that no store sat
    // behind a branch, wrote part of P twice: 33 MB more of the 604 written at B=4 T=8192 H=16, by the counters, and the writes bound a
    // saving call)
    constexpr int PROWS = CH / NVS, PVEC = CH * PROWS / NTHR;
    typedef T pvec __attribute__((ext_vector_type(PVEC)));
    const int pidx = threadIdx.x & (NTHR - 1);
    const int prow = vsl * PROWS + pidx * PVEC / CH, pcol = pidx * PVEC % CH;
    const int wt = wave_id() - 4;
    auto store_saved = [&](int c) {           // v_new(c) (back in [token][column] through transposing reads) and P(c)
      const pvec pv = *(const pvec*)(s_p[c & 1] + prow * LDC + pcol);
      // (BV = 16: a wave takes 32 tokens, waves 2, 3 the same again)
      const int vl = BV == 32 ? l : (l & 31), vt = BV == 32 ? 16 * wt : 32 * (wt & 1) + 16 * (l >> 5);
      const typename ET<T>::frag x = ET<T>::load_frag_t(s_vT[c & 1], LDC, 0, vt, vl);
      __builtin_nontemporal_store(pv, (pvec*)((T*)a.pmat + (((int64_t)(sq.chunk0 + c) * a.H + h) * CH + prow) * CH + pcol));
      // (all 64 rows: those past the end of a partial chunk are zero)
      __builtin_nontemporal_store(x, (typename ET<T>::vec*)(slice_ptr<T>(a.vnew, sq.chunk0 + c, h, a.H, V, v0) + (vt + (vl & 15)) * SLICE_COLS + 8 * (vl >> 4)));
    };
    auto store_out = [&](int c) {
      const int tok = sq.tok0 + c * CH;
      const int len = min(CH, sq.len - c * CH);
      typename IOV::Regs ro;
      IOV::load_lds_clamped(ro, s_o[c & 1], LDU, len);
      IOV::template store_global_clamped<false>(ro, row_ptr<T>(a.o, sq.b, tok, h) + v0, a.o.st, len);
    };
    // the blocks of P above the diagonal, which no helper writes, are cleared once
    {
      const int t = threadIdx.x & (NTHR - 1), r = t >> 4, cc = t & 15;
#pragma unroll
      for (int I = 0; I < 3; ++I)
#pragma unroll
        for (int J = I + 1; J < 4; ++J) s_p[0][(16 * I + r) * LDC + 16 * J + cc] = s_p[1][(16 * I + r) * LDC + 16 * J + cc] = (T)0.f;
    }
#pragma unroll
    for (int j = 0; j < LPA; ++j) issue_a(pa[j], j);
    wait_all_loads();
    stage_a(pa[0], 0);
    issue_a(pa[0], LPA);
    lds_barrier();
    auto window = [&](auto slot, const int c, auto stores) {
      constexpr int jn = (decltype(slot)::value + 1) % LPA;
      if (wave_id() == 4) TR(2, c, 0);
      stores(c);
      if (wave_id() == 4) TR(2, c, 1);
      stage_a(pa[jn], c + 1);               // (past the last chunk: a clamped copy of it, never used)
      if (wave_id() == 4) TR(2, c, 4);
      issue_a(pa[jn], c + 1 + LPA);
      if (wave_id() == 4) TR(2, c, 2);
      lds_barrier();
      if (wave_id() == 4) TR(2, c, 3);
    };
    // the first two windows have fewer results to store: outside of the loop, whose stores then lie behind no branch
    window(std::integral_constant<int, 0>(), 0, [](int) {});
    if (sq.nchunks > 1) {
      window(std::integral_constant<int, 1 % LPA>(), 1, [&](int c) { if constexpr (SAVE) store_saved(c - 1); });
      ring_loop<LPA>(sq.nchunks - 2, [&](auto slot, const int c2) {
        window(std::integral_constant<int, (decltype(slot)::value + 2) % LPA>(), c2 + 2, [&](int c) {
          if constexpr (SAVE) store_saved(c - 1);
          store_out(c - 2);
        });
      });
    }
    if constexpr (SAVE) store_saved(sq.nchunks - 1);
    if (sq.nchunks > 1) store_out(sq.nchunks - 2);
    lds_barrier();                                                                       // o of the last chunk
    store_out(sq.nchunks - 1);
    if constexpr (TRACE) {
      if ((int)blockIdx.x == traced_wg)
        for (int i = threadIdx.x & (NTHR - 1); i < TRACE_SLOTS * TRACE_CHUNKS * TRACE_MARKS; i += NTHR) {
          const int c = i / TRACE_MARKS % TRACE_CHUNKS, slot = i / (TRACE_MARKS * TRACE_CHUNKS);
          const uint32_t x = c < TRACE_LDS_CHUNKS ? s_tr[(slot * TRACE_LDS_CHUNKS + c) * TRACE_MARKS + i % TRACE_MARKS] : 0u;
          tr[i] = x ? s_tr0 + (long long)(uint32_t)(x - (uint32_t)s_tr0) : 0;
        }
    }
    return;
  }
  if (team == 2) {
    // ------------------------- loaders, ring B (q, Tinv, v, gates) ------------------------
    struct PreB { typename IOK::Regs rq; typename IOP::Regs rt; typename IOV::Regs rv; float gt, b; int len; };
    PreB pb[LPB];
    const int wt = wave_id() - 8;            // each wave carries one row of the gate table; b: the last row, every wave
    auto issue_b = [&](PreB& P, int c) {
      c = min(c, sq.nchunks - 1);
      const int tok = sq.tok0 + c * CH;
      P.len = min(CH, sq.len - c * CH);
      IOK::load_nomask(P.rq, row_ptr<T>(a.q, sq.b, tok, h), a.q.st, P.len);
      IOP::load_nomask(P.rt, (const T*)a.tinv + ((int64_t)(sq.chunk0 + c) * a.H + h) * CH * CH, CH, CH);
      IOV::load_nomask(P.rv, row_ptr<T>(a.v, sq.b, tok, h) + v0, a.v.st, P.len);
      const float* gc = a.gcum + ((int64_t)(sq.chunk0 + c) * a.H + h) * GATE_ROWS * CH;
      P.gt = gc[wt * CH + l];
      P.b = gc[4 * CH + l];
    };
    auto stage_b = [&](PreB& P, int buf) {
      IOK::mask(P.rq, P.len);                // (rows past the end: P is zero there as the backward expects it)
      IOK::store_lds(P.rq, s_q[buf], LDK);
      IOP::store_lds(P.rt, s_ti[buf], LDC);
      if (a.v_act) {                         // v = silu(v as given): the activation in front of the op, applied here
#pragma unroll
        for (int p = 0; p < IOV::PASSES; ++p)
#pragma unroll
          for (int i = 0; i < IOV::VEC; ++i) P.rv.v[p][i] = ET<T>::from_f(silu_of(ET<T>::to_f(P.rv.v[p][i])));
      }
      IOV::mask(P.rv, P.len);
      IOV::store_lds(P.rv, s_v[buf], LDU);
      s_gt[buf][wt][l] = P.gt;
      s_gt[buf][4][l] = P.b;                 // (the same from all four)
    };
#pragma unroll
    for (int j = 0; j < LPB; ++j) issue_b(pb[j], j);
    wait_all_loads();
    stage_b(pb[0], 0);
    issue_b(pb[0], LPB);
    lds_barrier();
    ring_loop<LPB>(sq.nchunks, [&](auto slot, const int c) {
      constexpr int jn = (decltype(slot)::value + 1) % LPB;
      if (wave_id() == 8) TR(3, c, 0);
      if constexpr (SAVE) store_state(c);
      if (wave_id() == 8) TR(3, c, 1);
      stage_b(pb[jn], (c + 1) & 1);         // (past the last chunk: a clamped copy of it, never used)
      if (wave_id() == 8) TR(3, c, 4);
      issue_b(pb[jn], c + 1 + LPB);
      if (wave_id() == 8) TR(3, c, 2);
      lds_barrier();
      if (wave_id() == 8) TR(3, c, 3);
    });
    lds_barrier();
    return;
  }

  const int wv = wave_id();
  const int fr = l & 15, g = l >> 4;
  const float scale = a.scale;
  if (wv >= 2) {
    // --------------------- helpers: P of the chunk and the output of its columns ---------------------
    __builtin_amdgcn_s_setprio(2);
    // helper J: output columns 16 J .. of the slice; blocks (ti, tj) of P with tj = J and tj = 3 - J (five each)
    auto help = [&](auto which) {
      constexpr int J = decltype(which)::value;
      constexpr int TA = J, TB = 3 - J;          // its two rows of k blocks
      // (q S)^T of a chunk: columns of the slice x tokens 16 t ..  BV = 16: helper J takes the token blocks t = 2 J, 2 J + 1
      constexpr int T0 = BV == 32 ? 0 : 2 * J, T1 = BV == 32 ? 4 : 2 * J + 2, C0 = BV == 32 ? 16 * J : 0;
      f32x4 oa[4];
      typename ET<T>::frag fv[2], fp[6];
      // o(c) = scale (e^b q S + P v_new), in the window behind the one that formed q S, P and v_new
      auto finish_fetch = [&](int c) {
        const T* s_pc = s_p[c & 1];
        const T* s_vc = s_vT[c & 1];
#pragma unroll
        for (int s = 0; s < 2; ++s) fv[s] = ET<T>::load_frag(s_vc + (C0 + fr) * LDC + 32 * s + 8 * g);
#pragma unroll
        for (int t = T0; t < T1; ++t) fp[t] = ET<T>::load_frag(s_pc + (16 * t + fr) * LDC + 8 * g);
        if constexpr (T1 == 4) {
          fp[4] = ET<T>::load_frag(s_pc + (32 + fr) * LDC + 32 + 8 * g);
          fp[5] = ET<T>::load_frag(s_pc + (48 + fr) * LDC + 32 + 8 * g);
        }
      };
      auto finish = [&](int c) {
#pragma unroll
        for (int t = T0; t < T1; ++t) ET<T>::mma(oa[t], fv[0], fp[t]);
        if constexpr (T1 == 4) {
          ET<T>::mma(oa[2], fv[1], fp[4]);
          ET<T>::mma(oa[3], fv[1], fp[5]);
        }
#pragma unroll
        for (int t = T0; t < T1; ++t) {
          oa[t] *= scale;
          acc_to_lds_t<T>(oa[t], s_o[c & 1], LDU, C0, 16 * t, l);                    // o [token][column]: 8-byte writes
        }
      };
      lds_barrier();
      for (int c = 0; c < sq.nchunks; ++c) {
        const int cur = c & 1;
        if (J == 0) TR(1, c, 0);
        const T *s_kc = s_k[cur], *s_qc = s_q[cur], *s_hc = s_hT[cur];
        typename ET<T>::frag fs[2], fq[2][4], fk[2][2];
        auto fetch = [&](int ks, int buf) {
          fs[buf] = ET<T>::load_frag(s_hc + (C0 + fr) * LDK + 32 * ks + 8 * g);
#pragma unroll
          for (int t = 0; t < 4; ++t) fq[buf][t] = ET<T>::load_frag(s_qc + (16 * t + fr) * LDK + 32 * ks + 8 * g);
          fk[buf][0] = ET<T>::load_frag(s_kc + (16 * TA + fr) * LDK + 32 * ks + 8 * g);
          fk[buf][1] = ET<T>::load_frag(s_kc + (16 * TB + fr) * LDK + 32 * ks + 8 * g);
        };
        if (c > 0) finish_fetch(c - 1);
        f32x4 bj[2];
        float bi[4], eb[4];
        bj[0] = *(const f32x4*)&s_gt[cur][4][16 * TA + 4 * g];
        bj[1] = *(const f32x4*)&s_gt[cur][4][16 * TB + 4 * g];
#pragma unroll
        for (int t = 0; t < 4; ++t) { bi[t] = s_gt[cur][4][16 * t + fr]; eb[t] = s_gt[cur][0][16 * t + fr]; }
        fetch(0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (c > 0) finish(c - 1);
        if (J == 0) TR(1, c, 1);
        // the decay factors of P, Gamma_ij = e^{b_i - b_j} for i >= j, while the fragments are on their way (rows past
        // the end of a partial chunk: q is zero there)
        f32x4 gm[5];
        static_for_blocks<TA, TB>([&](auto x, auto ti, auto tj) {
          constexpr int X = decltype(x)::value, TI = decltype(ti)::value, TJ = decltype(tj)::value;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float y = texp<T>(bi[TI] - bj[TJ == TA ? 0 : 1][e]);
            gm[X][e] = (TI > TJ || fr >= 4 * g + e) ? y : 0.f;
          }
        });
        // (q S)^T and, over the same q rows, its blocks of P = (q k^T) . Gamma, formed transposed (k rows as the A
        // operand) so that a lane holds four consecutive columns of one row (8-byte writes)
        f32x4 pc[5];
#pragma unroll
        for (int t = 0; t < 4; ++t) oa[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int x = 0; x < 5; ++x) pc[x] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const int bf = ks & 1;
          if (ks + 1 < KS) fetch(ks + 1, bf ^ 1);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int t = T0; t < T1; ++t) ET<T>::mma(oa[t], fs[bf], fq[bf][t]);
          static_for_blocks<TA, TB>([&](auto x, auto ti, auto tj) {
            constexpr int X = decltype(x)::value, TI = decltype(ti)::value, TJ = decltype(tj)::value;
            ET<T>::mma(pc[X], fk[bf][TJ == TA ? 0 : 1], fq[bf][TI]);
          });
          __builtin_amdgcn_sched_barrier(0);
        }
        static_for_blocks<TA, TB>([&](auto x, auto ti, auto tj) {
          constexpr int X = decltype(x)::value, TI = decltype(ti)::value, TJ = decltype(tj)::value;
          bf16x4 y;
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = (bf16)(pc[X][e] * gm[X][e]);
          *(bf16x4*)(s_p[cur] + (16 * TI + fr) * LDC + 16 * TJ + 4 * g) = y;
        });
#pragma unroll
        for (int t = T0; t < T1; ++t) oa[t] *= eb[t];
        if (J == 0) TR(1, c, 2);
        lds_barrier();
        if (J == 0) TR(1, c, 3);
      }
      finish_fetch(sq.nchunks - 1);
      finish(sq.nchunks - 1);
      lds_barrier();
    };
    if (wv == 2) help(std::integral_constant<int, 0>());
    else help(std::integral_constant<int, 1>());
    return;
  }

  if (BV == 16 && wv == 1) return;                   // (a wave that has ended is not waited for at a barrier)
  // --------------------------------- consumers: the chain ---------------------------------
  __builtin_amdgcn_s_setprio(3);
  const int j = wv;
  const int vc = v0 + 16 * j + fr;                   // the column of this lane
  // row of the state / token of a token-row block that accumulator element i of block m holds in this lane
  auto idx_of = [&](int m, int i) { return 32 * (m >> 1) + 8 * g + 4 * (m & 1) + i; };
  // row an A-operand lane reads for block m of a token-row product
  auto arow_of = [&](int m) { return 32 * (m >> 1) + 4 * (m & 1) + 8 * (fr >> 2) + (fr & 3); };
  f32x4 S[KT];
#pragma unroll
  for (int mi = 0; mi < KT; ++mi) S[mi] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (a.h0 || !item.first) {
    const float* h0 = item.first ? a.h0 + ((int64_t)n * a.H + h) * K * V : sp.S + (int64_t)pair * K * V;
#pragma unroll
    for (int mi = 0; mi < KT; ++mi)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[mi][i] = h0[(int64_t)idx_of(mi, i) * V + vc];
  }
  // the state as the operand of the next chunk and, the same registers, as S^T [column][K]: 8 consecutive rows per lane
  typename ET<T>::frag bS[KS];
  auto put_state = [&](int buf) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      bS[ks] = frag_of_blocks(S[2 * ks], S[2 * ks + 1]);
      *(bf16x8*)(s_hT[buf] + (16 * j + fr) * LDK + 32 * ks + 8 * g) = bS[ks];
    }
  };
  put_state(0);
  lds_barrier();
  for (int c = 0; c < sq.nchunks; ++c) {
    const int cur = c & 1;
    const T* s_kc = s_k[cur];
    if (wv == 0) TR(0, c, 0);
    // X = k S; beside it, off the chain, what does not depend on it: e^{b_C} S, beta v
    f32x4 X[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) X[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    typename ET<T>::frag fti[6];
    f32x4 bv[2][2], ff[2][2];
    {
      typename ET<T>::frag fk[2][4], fv[2];
      f32x4 be[2][2];
#pragma unroll
      for (int t = 0; t < 4; ++t) fk[0][t] = ET<T>::load_frag(s_kc + arow_of(t) * LDK + 8 * g);
      const float dec = s_gt[cur][0][CH - 1];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (ks + 1 < KS) {
#pragma unroll
          for (int t = 0; t < 4; ++t) fk[(ks + 1) & 1][t] = ET<T>::load_frag(s_kc + arow_of(t) * LDK + 32 * (ks + 1) + 8 * g);
        }
        if (ks == KS - 2) {
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            fv[s] = ET<T>::load_frag_t(s_v[cur], LDU, 32 * s, 16 * j, l);
            be[s][0] = *(const f32x4*)&s_gt[cur][2][32 * s + 8 * g]; be[s][1] = *(const f32x4*)&s_gt[cur][2][32 * s + 8 * g + 4];
          }
        }
        if (ks == KS - 1) {
#pragma unroll
          for (int s = 0; s < 2; ++s) { ff[s][0] = *(const f32x4*)&s_gt[cur][3][32 * s + 8 * g]; ff[s][1] = *(const f32x4*)&s_gt[cur][3][32 * s + 8 * g + 4]; }
#pragma unroll
          for (int t = 0; t < 4; ++t) fti[t] = ET<T>::load_frag(s_ti[cur] + arow_of(t) * LDC + 8 * g);
          fti[4] = ET<T>::load_frag(s_ti[cur] + arow_of(2) * LDC + 32 + 8 * g);
          fti[5] = ET<T>::load_frag(s_ti[cur] + arow_of(3) * LDC + 32 + 8 * g);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < 4; ++t) ET<T>::mma(X[t], fk[ks & 1][t], bS[ks]);
        if (ks == 0) {
#pragma unroll
          for (int mi = 0; mi < KT; ++mi) S[mi] *= dec;
        }
        if (ks == KS - 1) {
#pragma unroll
          for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
              for (int i = 0; i < 4; ++i) bv[s][e][i] = be[s][e][i] * (float)fv[s][4 * e + i];
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (wv == 0) TR(0, c, 1);
    // the k^T fragments of the first half of the update
    typename ET<T>::frag fkt[2][KT];
#pragma unroll
    for (int mi = 0; mi < KT; ++mi) fkt[0][mi] = load_frag_t_state(s_kc, LDK, 0, mi, l);
    // Z = beta v - (beta e^{b}) X  (8 tokens of this lane's column per 32-token step), then v_new = Tinv Z
    f32x4 vn[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) vn[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    typename ET<T>::frag Z[2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          Z[s][4 * e + i] = (bf16)__builtin_fmaf(-ff[s][e][i], X[2 * s + e][i], bv[s][e][i]);
    ET<T>::mma(vn[0], fti[0], Z[0]);
    ET<T>::mma(vn[1], fti[1], Z[0]);
    ET<T>::mma(vn[2], fti[2], Z[0]);
    ET<T>::mma(vn[3], fti[3], Z[0]);
    ET<T>::mma(vn[2], fti[4], Z[1]);
    ET<T>::mma(vn[3], fti[5], Z[1]);
    __builtin_amdgcn_sched_barrier(0);
    // (its factors and the fragments of the second half: Tinv's registers are free)
    f32x4 ed[2][2];
#pragma unroll
    for (int s = 0; s < 2; ++s) { ed[s][0] = *(const f32x4*)&s_gt[cur][1][32 * s + 8 * g]; ed[s][1] = *(const f32x4*)&s_gt[cur][1][32 * s + 8 * g + 4]; }
#pragma unroll
    for (int mi = 0; mi < KT; ++mi) fkt[1][mi] = load_frag_t_state(s_kc, LDK, 32, mi, l);
    __builtin_amdgcn_sched_barrier(0);
    if (wv == 0) TR(0, c, 5);
    // v_new rounded once to the storage type: the state update, the output and the backward see the same values
    typename ET<T>::frag vb[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      vb[s] = frag_of_blocks(vn[2 * s], vn[2 * s + 1]);
      typename ET<T>::frag bvd;
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int i = 0; i < 4; ++i) bvd[4 * e + i] = (bf16)((float)vb[s][4 * e + i] * ed[s][e][i]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int mi = 0; mi < KT; ++mi) ET<T>::mma(S[mi], fkt[s][mi], bvd);
      __builtin_amdgcn_sched_barrier(0);
    }
    // v_new^T [column][64]: 8 consecutive tokens per lane
#pragma unroll
    for (int s = 0; s < 2; ++s) *(bf16x8*)(s_vT[cur] + (16 * j + fr) * LDC + 32 * s + 8 * g) = vb[s];
    if (wv == 0) TR(0, c, 6);
    put_state(cur ^ 1);                               // the state at the start of the next chunk
    if (wv == 0) TR(0, c, 2);
    lds_barrier();
    if (wv == 0) TR(0, c, 3);
  }
  lds_barrier();
  if (a.ht && item.last) {
    float* ht = a.ht + ((int64_t)n * a.H + h) * K * V;
#pragma unroll
    for (int mi = 0; mi < KT; ++mi)
#pragma unroll
      for (int i = 0; i < 4; ++i) ht[(int64_t)idx_of(mi, i) * V + vc] = S[mi][i];
  }
}

}  // namespace lmoe
