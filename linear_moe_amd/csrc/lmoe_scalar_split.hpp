// Sequences of chunk_simple_gla cut along T: the state every fine segment adds, formed for all segments at once.
//   forward :  Q = sum_t e^{b_end - b_t} k_t^T v_t      backward:  Q = sum_t scale e^{b_t - b_start} q_t^T do_t
// (b the running log-decay, b_end / b_start at the segment's last / before its first token) and D = e^{b_end - b_start};
// the sequential pass then starts a coarse segment from the segments in front of it (behind it, in the backward),
// S <- D S + Q, one fine segment after the other (seg_prefix).
#pragma once
#include "lmoe_split.hpp"
#include "lmoe_scalar_fwd.hpp"

namespace lmoe {

// ------------------------------------------------------------------------- //
// Work-group of 256 threads = one (fine segment, head, V slice of BV columns); wave w owns state rows [w K/4, (w+1) K/4)
// in fp32 MFMA accumulators.  The next chunk travels in registers while the current one is multiplied out of LDS; two or
// more work-groups per CU hide the two barriers per chunk.  2-byte elements carry all V columns, so that k (q) is read
// once; 4-byte ones (matrix instructions of a sixteenth the rate) 32, for more work-groups.
// BWD: q, do in place of k, v, chunks from the last to the first.  NORM (2-byte elements, ungated): with the normaliser's
// column, Z = sum_t k_t forward, Z = sum_t q_t^T (scale dden_t) backward (NORM = 1: dden_t = -(do_t . o_t) / den_t and the
// rows of do over den; NORM = 2: dden given), as in k_state_fwd_b and k_state_bwd.
// ------------------------------------------------------------------------- //
template <typename T, int K, int V, int BV, bool BWD, int NORM>
__global__ __launch_bounds__(NTHR) void k_scalar_seg_state(const lmoe_args a, const Split sp, int seg0, int nsegs) {
  static_assert(!NORM || (sizeof(T) == 2 && BV == V), "the normaliser's column: 2-byte elements, whole rows");
  constexpr int LDK = K + LPAD, LDU = BV + LPAD, MB = K / 64, NB = BV / 16, NVS = V / BV;
  __shared__ __attribute__((aligned(16))) T s_k[CH * LDK];
  __shared__ __attribute__((aligned(16))) T s_u[CH * LDU];
  __shared__ __attribute__((aligned(16))) float s_f[64];                   // row factors of v / do
  __shared__ __attribute__((aligned(16))) float s_dd[NORM ? 64 : 4];
  __shared__ float s_dec;
  const int vsl = blockIdx.x % NVS, h = (blockIdx.x / NVS) % a.H, r = blockIdx.x / NVS / a.H;
  const int n = r / nsegs, i = seg0 + r % nsegs, v0 = vsl * BV;            // sequence, fine segment inside it
  const SeqInfo sq = seg_cut(seq_info(a, n), i, sp.len1);
  const int l = lane_id(), wv = wave_id(), krow0 = wv * (K / 4);
  typedef TileIO<T, CH, K> IOK;
  typedef TileIO<T, CH, BV> IOV;
  const lmoe_tensor &kt = BWD ? a.q : a.k, &ut = BWD ? a.d_o : a.v;
  const bool gated = a.gate != LMOE_GATE_NONE && a.g.ptr != nullptr;
  const void* gptr = gated ? a.g.ptr : a.k.ptr;
  constexpr bool DOT = BWD && NORM == 1, GIVEN = BWD && NORM == 2;
  struct Pre { typename IOK::Regs rk; typename IOV::Regs ru; uint32_t graw; };
  Pre P;
  typename IOV::Regs ro;                                                   // DOT: rows of the normalised output
  float rD[DOT ? IOV::PASSES : 1], dl = 0.f;
  auto chunk_at = [&](int j) { return BWD ? sq.nchunks - 1 - j : j; };
  auto issue = [&](int c) {
    const int tok = sq.tok0 + c * CH, len = min(CH, sq.len - c * CH);
    IOK::load_nomask(P.rk, row_ptr<T>(kt, sq.b, tok, h), kt.st, len);
    IOV::load_nomask(P.ru, row_ptr<T>(ut, sq.b, tok, h) + v0, ut.st, len);
    P.graw = load_scalar_raw(gptr, a.g_dtype, gated ? row_off(a.g, sq.b, tok + min(l, len - 1), h) : 0);
    if constexpr (DOT) {
      IOV::load_nomask(ro, row_ptr<T>(a.o, sq.b, tok, h) + v0, a.o.st, len);
      const float* den = (const float*)a.den.ptr;
#pragma unroll
      for (int p = 0; p < IOV::PASSES; ++p) {
        int row, col; IOV::coords(p, row, col);
        rD[p] = den[row_off(a.den, sq.b, tok + min(row, len - 1), h)];
      }
      dl = den[row_off(a.den, sq.b, tok + min(l, len - 1), h)];
    }
    if constexpr (GIVEN) dl = ((const float*)a.dden.ptr)[row_off(a.dden, sq.b, tok + min(l, len - 1), h)];
  };
  f32x4 S[MB][NB], Sz[NORM ? MB : 1];
  acc_zero(S);
#pragma unroll
  for (int mi = 0; mi < (NORM ? MB : 1); ++mi) Sz[mi] = f32x4{0.f, 0.f, 0.f, 0.f};
  float D = 1.f;
  issue(chunk_at(0));
  for (int j = 0; j < sq.nchunks; ++j) {
    const int len = min(CH, sq.len - chunk_at(j) * CH);
    if constexpr (DOT) {
#pragma unroll
      for (int p = 0; p < IOV::PASSES; ++p) {
        int row, col; IOV::coords(p, row, col);
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < IOV::VEC; ++e) sum += ET<T>::to_f(P.ru.v[p][e]) * ET<T>::to_f(ro.v[p][e]);
        sum = group_sum<IOV::VPR>(sum);
        if (col == 0) s_dd[row] = row < len ? -a.scale * sum / rD[p] : 0.f;
      }
    }
    IOK::mask(P.rk, len);
    IOV::mask(P.ru, len);
    IOK::store_lds(P.rk, s_k, LDK);
    IOV::store_lds(P.ru, s_u, LDU);
    if (wv == 0) {
      const float x = wave_incl_scan((gated && l < len) ? scalar_from_raw(P.graw, a.g_dtype) : 0.f);
      const float xl = __shfl(x, 63, 64);
      s_f[l] = DOT ? a.scale / dl : BWD ? a.scale * expf(x) : expf(xl - x);
      if constexpr (GIVEN) s_dd[l] = l < len ? a.scale * dl : 0.f;
      if (l == 0) s_dec = expf(xl);
    }
    issue(chunk_at(min(j + 1, sq.nchunks - 1)));      // (always: past the end the last chunk again, never used)
    lds_barrier();
    const float dec = s_dec;
    D *= dec;
#pragma unroll
    for (int mi = 0; mi < MB; ++mi)
#pragma unroll
      for (int ni = 0; ni < NB; ++ni) S[mi][ni] *= dec;
#pragma unroll
    for (int kk = 0; kk < CH; kk += 32) {
      typename ET<T>::frag af[MB];
#pragma unroll
      for (int mi = 0; mi < MB; ++mi) af[mi] = ET<T>::load_frag_t(s_k, LDK, kk, krow0 + 16 * mi);
#pragma unroll
      for (int ni = 0; ni < NB; ++ni) {
        typename ET<T>::frag bf = ET<T>::load_frag_t(s_u, LDU, kk, 16 * ni);
        scale_frag<T>(bf, &s_f[kk + 8 * (l >> 4)]);
#pragma unroll
        for (int mi = 0; mi < MB; ++mi) ET<T>::mma(S[mi][ni], af[mi], bf);
      }
      if constexpr (NORM != 0) {
        typename ET<T>::frag fz;
        if constexpr (BWD) {
          const f32x4 d0 = *(const f32x4*)&s_dd[kk + 8 * (l >> 4)], d1 = *(const f32x4*)&s_dd[kk + 8 * (l >> 4) + 4];
#pragma unroll
          for (int e = 0; e < 4; ++e) { fz[e] = (bf16)d0[e]; fz[e + 4] = (bf16)d1[e]; }
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) fz[e] = (bf16)1.f;
        }
#pragma unroll
        for (int mi = 0; mi < MB; ++mi) ET<T>::mma(Sz[mi], af[mi], fz);
      }
    }
    lds_barrier();
  }
  const int64_t o = (int64_t)(n * seg_count((a.T + CH - 1) / CH, sp.len1) + i) * a.H + h;
#pragma unroll
  for (int mi = 0; mi < MB; ++mi)
#pragma unroll
    for (int ni = 0; ni < NB; ++ni)
      *(f32x4*)(sp.Q + (o * V + v0 + acc_col(ni)) * K + krow0 + acc_row(mi, 0)) = S[mi][ni];
  if constexpr (NORM != 0) {
    if ((l & 15) == 0) {
#pragma unroll
      for (int mi = 0; mi < MB; ++mi) *(f32x4*)(sp.Z + o * K + krow0 + acc_row(mi, 0)) = Sz[mi];
    }
  }
  if (threadIdx.x == 0 && vsl == 0) sp.D[o] = D;
}

}  // namespace lmoe
