// Instantiation and launch of the forward kernel of chunk_simple_gla, plus the toolkit self-test.
#include <type_traits>
#include "lmoe_launch.hpp"
#include "lmoe_scalar_chunks.hpp"
#include "lmoe_scalar_split.hpp"

namespace lmoe {

// V-slice of the sequential state pass
template <typename T, int V> struct FwdTiles {
  static constexpr int BVS = sizeof(T) == 4 ? 16 : 32;
};

// How the sequences of a call are cut along T: not at all without a workspace for it.
inline Split scalar_split(const lmoe_args& a) {
  Split sp = {};
  if (!a.seg_ws) return sp;
  sp = plan_split_scalar(a);
  if (!sp.len1) return sp;
  const int64_t n1 = (int64_t)sp.n1 * a.H;
  sp.Q = a.seg_ws;
  sp.Z = sp.Q + n1 * a.K * a.V;
  sp.D = sp.Z + n1 * a.K;
  return sp;
}
// 4-byte elements: whether every chunk runs on its own (k_state_fwd_chunks).  Without and with it, us, K = V = 64 (two work-groups
// to a CU): 32 pairs of 8 chunks 34 and 20, 64 of 4 19 and 17, 64 of 8 35 and 39; K = V = 128 (one): 8 pairs of 8 chunks 26
// and 20, 16 of 8 38 and 38, 16 of 4 29 and 17, 32 of 4 30 and 32.  Up to two chunks there is next to nothing to form twice: 128
// pairs of 2 21 and 16.5, K = V = 128 68 and 59; but with a final state, one work-group more per sequence, 32 pairs of 1 12.9
// and 14.8, 8 of 1 11.5 and 9.2.  A chunk in front to a wave, eight at most: runs of two gave 4 pairs of 16 chunks 13.9 and
// 12.6 but 16 of 16 26 and 28, and every other call their loop.
inline bool fwd_by_chunks(const lmoe_args& a) {
  if (a.dtype == LMOE_BF16 || a.cu_seqlens) return false;
  const int nch = (a.T + CH - 1) / CH, per_cu = a.K == 64 ? 4 : 2;
  const int64_t wgs = (int64_t)a.N * a.H * (nch + (a.ht ? 1 : 0)) * (a.V / 16);
  return nch <= CHUNKS_PREFIX_WAVES && wgs <= (int64_t)cu_count() * (a.ht ? min(nch, per_cu) : nch <= 2 ? 8 : per_cu);
}
// (a forward call that runs by chunks needs no buffers; asked without either output, the larger of both directions)
int64_t scalar_split_floats(const lmoe_args& a) {
  if (a.o.ptr && !a.d_o.ptr && fwd_by_chunks(a)) return 0;
  const Split sp = plan_split_scalar(a);
  return (int64_t)sp.n1 * a.H * (a.K * a.V + a.K + 1);
}
// what the fine segments add (forward: but for those of the last coarse segment; backward: of the first)
template <bool BWD> struct ScalarSeg {
  template <typename T, int K, int V> struct F {
    template <int NORM> static void go(const lmoe_args& a, const Split& sp, hipStream_t st) {
      constexpr int BV = sizeof(T) == 4 ? 32 : V;
      const int n = sp.n1 / a.N, f = sp.len3 / sp.len1, r = sp.n3 / a.N;
      const int seg0 = BWD ? f : 0, nsegs = BWD ? n - f : (r - 1) * f;
      hipLaunchKernelGGL((k_scalar_seg_state<T, K, V, BV, BWD, NORM>), dim3(a.N * nsegs * a.H * (V / BV)), dim3(NTHR), 0, st,
                         a, sp, seg0, nsegs);
    }
    static void run(const lmoe_args& a, const Split& sp, hipStream_t st) {
      if constexpr (sizeof(T) == 2) {
        if (a.normalize && !BWD) return go<1>(a, sp, st);
        if (a.normalize == 1) return go<1>(a, sp, st);
        if (a.normalize == 2) return go<2>(a, sp, st);
      }
      go<0>(a, sp, st);
    }
  };
};
Split launch_scalar_seg(const lmoe_args& a, bool bwd, hipStream_t st) {
  const Split sp = scalar_split(a);
  if (sp.len1) {
    if (bwd) dispatch<ScalarSeg<true>::F>(a, st, sp);
    else dispatch<ScalarSeg<false>::F>(a, st, sp);
  }
  return sp;
}

// the pass for 2-byte elements on V slices of BV columns: saving or forward-only, plain or with the normalised output
template <typename T, int K, int V, int BV, bool CUT> void launch_fwd_b(const lmoe_args& a, const Split& sp, hipStream_t st) {
  const dim3 grid(((pass_items(a, sp) * a.H + 7) / 8) * 8 * (V / BV)), block(3 * NTHR);
  long long* const no_trace = nullptr;
  // Which loads (KEPT).  Without and with the kept offset, us.  It needs registers, which slices of 64 columns at K = 128 have
  // not, and gives a partial tile a path of its own, so it pays in the full ones:
  //   K = 128: 64 pairs of 64 chunks 97 and 90, 60 pairs of 400 tokens 13.9 and 13.6; but 16 pairs of 100 tokens 7.5 and 7.8, of
  //   30 tokens 6.3 and 6.8, of 64 5.9 and 5.7
  //   K = 64, half the loads per tile: the plain pass loses (V = 64, 64 pairs of 64 chunks 46.4 and 48.7, packed 8192 x 8 33.5 and
  //   35.0; only saving calls that write more than the memory-side cache holds gained, V = 128, 64 pairs of 64 chunks 73.5 and
  //   70.4).  The normalised one: 64 pairs of 64 chunks 64.9 and 60.0, 60 pairs of 250 tokens 8.3 and 8.4, of 192 7.3 and 7.0;
  //   saving 60 pairs of 1000 tokens 20.2 and 20.3, of 400 11.7 and 11.9, of 640 14.7 and 14.5
  const bool tail = a.cu_seqlens || a.T % CH;
  const int tokens = a.cu_seqlens ? a.T / max(a.N, 1) : a.T;                    // of a sequence, on average
  auto go = [&](auto save, auto norm) {
    constexpr bool SAVE = decltype(save)::value, NORM = decltype(norm)::value;
    if constexpr (!CUT && fwd_may_keep<NORM, K, BV>()) {
      if (tail && tokens < (K == 128 ? 128 : SAVE ? 1024 : 256)) {
        hipLaunchKernelGGL((k_state_fwd_b<T, K, V, BV, SAVE, false, NORM, CUT, false>), grid, block, 0, st, a, sp, no_trace, -1);
        return;
      }
    }
    hipLaunchKernelGGL((k_state_fwd_b<T, K, V, BV, SAVE, false, NORM, CUT>), grid, block, 0, st, a, sp, no_trace, -1);
  };
  typedef std::true_type yes;
  typedef std::false_type no;
  if (a.normalize) {
    if (a.hs) go(yes(), yes());
    else go(no(), yes());
  } else {
    if (a.hs) go(yes(), no());
    else go(no(), no());
  }
}
template <typename T, int K, int V> struct StateFwd {
  static void run(const lmoe_args& a, hipStream_t st) {
    constexpr int BV = FwdTiles<T, V>::BVS;
    if constexpr (sizeof(T) == 2) {
      // 64-wide slices where they still fill the chip: every V slice of a (sequence, head) fetches all of q and k and
      // forms all of P, so two wide slices cost less per output column than four narrow ones; the results do not
      // depend on the width (a state element and an output element are the same sums in either split)
      if constexpr (V >= 64) {
        if ((int64_t)a.N * a.H * (V / 64) >= cu_count()) {
          launch_fwd_b<T, K, V, 64, false>(a, Split{}, st);
          return;
        }
      }
      const Split sp = launch_scalar_seg(a, false, st);
      if (sp.len1) launch_fwd_b<T, K, V, BV, true>(a, sp, st);
      // slices of 16 columns where each finds a CU of its own (us, 32 and 16 columns; same bits): K = V = 128, 4 pairs of 8 chunks
      // 14.1 and 13.1, 32 of 16 25.1 and 23.8, normalised 27.8 and 25.9, 32 of 32 51.3 and 44.5, saving 50.0 and 44.3; K = V = 64,
      // 16 of 16 18.6 and 17.8; but 48 pairs of 16, K = V = 128, 26.0 and 42.8
      else if ((int64_t)a.N * a.H * (V / 16) <= cu_count()) launch_fwd_b<T, K, V, 16, false>(a, sp, st);
      else launch_fwd_b<T, K, V, BV, false>(a, sp, st);
    } else {
      if (fwd_by_chunks(a)) {
        const int nch = (a.T + CH - 1) / CH;
        hipLaunchKernelGGL((k_state_fwd_chunks<K, V>), dim3((nch + (a.ht ? 1 : 0)) * a.N * a.H * (V / 16)), dim3(3 * NTHR), 0, st, a);
        return;
      }
      const Split sp = launch_scalar_seg(a, false, st);
      const int grid = ((pass_items(a, sp) * a.H + 7) / 8) * 8 * (V / BV);
      if (sp.len1) {
        if (a.hs) hipLaunchKernelGGL((k_state_fwd<T, K, V, BV, true, true>), dim3(grid), dim3(3 * NTHR), 0, st, a, sp);
        else hipLaunchKernelGGL((k_state_fwd<T, K, V, BV, false, true>), dim3(grid), dim3(3 * NTHR), 0, st, a, sp);
      } else {
        if (a.hs) hipLaunchKernelGGL((k_state_fwd<T, K, V, BV, true, false>), dim3(grid), dim3(3 * NTHR), 0, st, a, sp);
        else hipLaunchKernelGGL((k_state_fwd<T, K, V, BV, false, false>), dim3(grid), dim3(3 * NTHR), 0, st, a, sp);
      }
    }
  }
};
void launch_state_fwd(const lmoe_args& a, hipStream_t st) { dispatch<StateFwd>(a, st); }
// the traced instance of the pass (2-byte elements, K = V = 128, forward-only call)
bool launch_state_fwd_trace(const lmoe_args& a, long long* tr, int work_group, hipStream_t st) {
  if (a.dtype != LMOE_BF16 || a.K != 128 || a.V != 128 || a.hs) return false;
  constexpr int BV = FwdTiles<bf16, 128>::BVS;
  const int grid = ((a.N * a.H + 7) / 8) * 8 * (128 / BV);
  if (work_group < 0 || work_group >= grid) return false;
  hipLaunchKernelGGL((k_state_fwd_b<bf16, 128, 128, BV, false, true>), dim3(grid), dim3(3 * NTHR), 0, st, a, Split{}, tr, work_group);
  return true;
}
// C = A B^T (64 x 64, contraction along the tile columns) and G = A^T B (KD x KD, contraction
// along the tile rows, i.e. the transposed-fragment path) over one pair of 64 x KD tiles,
// through the loaders / fragments / accumulator stores of the toolkit
template <typename T, int KD>
__global__ __launch_bounds__(NTHR) void k_selftest(const T* A, const T* B, float* C, float* G) {
  constexpr int LD = KD + LPAD, LDC = CH + LPAD;
  __shared__ __attribute__((aligned(16))) T s_a[CH * LD];
  __shared__ __attribute__((aligned(16))) T s_b[CH * LD];
  __shared__ __attribute__((aligned(16))) float s_c[CH * LDC];
  typedef TileIO<T, CH, KD> IO;
  typename IO::Regs ra, rb;
  IO::load(ra, A, KD, CH);
  IO::load(rb, B, KD, CH);
  IO::store_lds(ra, s_a, LD);
  IO::store_lds(rb, s_b, LD);
  __syncthreads();
  const int wv = wave_id(), l = lane_id();
  f32x4 acc[1][4];
  acc_zero(acc);
  gemm<T, 1, 4, false, false>(acc, s_a, LD, 16 * wv, s_b, LD, 0, 0, KD);
  for (int nj = 0; nj < 4; ++nj) acc_to_lds_t<float>(acc[0][nj], s_c, LDC, 16 * wv, 16 * nj);   // s_c = C^T
  __syncthreads();
  for (int idx = threadIdx.x; idx < CH * CH; idx += NTHR) {
    const int r = idx / CH, c = idx % CH;
    C[idx] = s_c[c * LDC + r];
  }
  // G rows [wv * KD/4, (wv+1) * KD/4)
  constexpr int MB = KD / 64, NB = KD / 16;
  f32x4 g[MB][NB];
  acc_zero(g);
  gemm<T, MB, NB, true, true>(g, s_a, LD, wv * (KD / 4), s_b, LD, 0, 0, CH);
  for (int mi = 0; mi < MB; ++mi)
    for (int ni = 0; ni < NB; ++ni)
      for (int i = 0; i < 4; ++i)
        G[(wv * (KD / 4) + 16 * mi + 4 * (l >> 4) + i) * KD + 16 * ni + (l & 15)] = g[mi][ni][i];
}

void launch_selftest(int dtype, int kd, const void* A, const void* B, float* C, float* G, hipStream_t st) {
  if (dtype == LMOE_BF16) {
    if (kd == 64) hipLaunchKernelGGL((k_selftest<bf16, 64>), dim3(1), dim3(NTHR), 0, st, (const bf16*)A, (const bf16*)B, C, G);
    else hipLaunchKernelGGL((k_selftest<bf16, 128>), dim3(1), dim3(NTHR), 0, st, (const bf16*)A, (const bf16*)B, C, G);
  } else {
    if (kd == 64) hipLaunchKernelGGL((k_selftest<float, 64>), dim3(1), dim3(NTHR), 0, st, (const float*)A, (const float*)B, C, G);
    else hipLaunchKernelGGL((k_selftest<float, 128>), dim3(1), dim3(NTHR), 0, st, (const float*)A, (const float*)B, C, G);
  }
}

}  // namespace lmoe
