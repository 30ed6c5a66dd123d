// Sequences of chunk_gla cut along T: the state every fine segment adds, formed for all segments at once.
//   forward :  Q = sum_t (k_t e^{b_end - b_t})^T v_t      backward:  Q = sum_t scale (q_t e^{b_t - b_start})^T do_t
// and D = e^{b_end - b_start}, a decay per state row; the sequential pass then starts a coarse segment from the segments
// in front of it (behind it, in the backward), S <- diag(D) S + Q, one fine segment after the other (seg_prefix_rows).
#pragma once
#include "lmoe_gla.hpp"

namespace lmoe {

// ------------------------------------------------------------------------- //
// Work-group of 256 threads = one (fine segment, head), all V columns, so that the gated k (q) rows are read once; wave w
// owns state rows [w K/4, (w+1) K/4) in fp32 MFMA accumulators.  Operands as k_gla_intra_fwd stored them: no gate, no
// exponential.  Bound by the latency of a chunk's loads: the next chunk travels in registers while the current one is
// multiplied out of LDS, and two or more work-groups per CU cover the two barriers.
// BWD: q e^{b}, do in place of k e^{b_C - b}, v, chunks from the last to the first.
// ------------------------------------------------------------------------- //
template <typename T, int K, int V, bool BWD>
__global__ __launch_bounds__(NTHR) void k_gla_seg_state(const lmoe_args a, const Split sp, int seg0, int nsegs) {
  static_assert(sizeof(T) == 2, "2-byte elements");
  constexpr int LDK = K + LPAD, LDU = V + LPAD, MB = K / 64, NB = V / 16;
  __shared__ __attribute__((aligned(16))) T s_k[CH * LDK];
  __shared__ __attribute__((aligned(16))) T s_u[CH * LDU];
  const int h = blockIdx.x % a.H, r = blockIdx.x / a.H;
  const int n = r / nsegs, i = seg0 + r % nsegs;                           // sequence, fine segment inside it
  const SeqInfo sq = seg_cut(seq_info(a, n), i, sp.len1);
  const int krow0 = wave_id() * (K / 4);
  typedef TileIO<T, CH, K> IOK;
  typedef TileIO<T, CH, V> IOV;
  const lmoe_tensor& ut = BWD ? a.d_o : a.v;
  const T* kp = (const T*)(BWD ? a.qe : a.ke);
  typename IOK::Regs rk;
  typename IOV::Regs ru;
  f32x4 next[MB], D[MB], S[MB][NB];
  acc_zero(S);
#pragma unroll
  for (int mi = 0; mi < MB; ++mi) D[mi] = f32x4{1.f, 1.f, 1.f, 1.f};
  auto chunk_at = [&](int j) { return BWD ? sq.nchunks - 1 - j : j; };
  auto issue = [&](int c) {
    const int64_t item = (int64_t)(sq.chunk0 + c) * a.H + h;
    IOK::load_nomask(rk, kp + item * CH * K, K, CH);
    IOV::load_nomask(ru, row_ptr<T>(ut, sq.b, sq.tok0 + c * CH, h), ut.st, min(CH, sq.len - c * CH));
#pragma unroll
    for (int mi = 0; mi < MB; ++mi)
#pragma unroll
      for (int e = 0; e < 4; ++e) next[mi][e] = a.gcum[item * K + krow0 + acc_row(mi, e)];
  };
  issue(chunk_at(0));
  for (int j = 0; j < sq.nchunks; ++j) {
    IOV::mask(ru, min(CH, sq.len - chunk_at(j) * CH));
    IOK::store_lds(rk, s_k, LDK);
    IOV::store_lds(ru, s_u, LDU);
#pragma unroll
    for (int mi = 0; mi < MB; ++mi) {
      D[mi] *= next[mi];
#pragma unroll
      for (int ni = 0; ni < NB; ++ni) S[mi][ni] *= next[mi];
    }
    issue(chunk_at(min(j + 1, sq.nchunks - 1)));      // (always: past the end the last chunk again, never used)
    lds_barrier();
#pragma unroll
    for (int kk = 0; kk < CH; kk += 32) {
      typename ET<T>::frag af[MB];
#pragma unroll
      for (int mi = 0; mi < MB; ++mi) af[mi] = ET<T>::load_frag_t(s_k, LDK, kk, krow0 + 16 * mi);
#pragma unroll
      for (int ni = 0; ni < NB; ++ni) {
        const typename ET<T>::frag bf = ET<T>::load_frag_t(s_u, LDU, kk, 16 * ni);
#pragma unroll
        for (int mi = 0; mi < MB; ++mi) ET<T>::mma(S[mi][ni], af[mi], bf);
      }
    }
    lds_barrier();
  }
  const int64_t o = (int64_t)(n * seg_count((a.T + CH - 1) / CH, sp.len1) + i) * a.H + h;
  const float f = BWD ? a.scale : 1.f;
#pragma unroll
  for (int mi = 0; mi < MB; ++mi) {
    const int row = krow0 + acc_row(mi, 0);
#pragma unroll
    for (int ni = 0; ni < NB; ++ni) *(f32x4*)(sp.Q + (o * V + acc_col(ni)) * K + row) = S[mi][ni] * f;
    if ((lane_id() & 15) == 0) *(f32x4*)(sp.D + o * K + row) = D[mi];
  }
}

}  // namespace lmoe
