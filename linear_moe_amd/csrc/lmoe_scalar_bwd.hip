// Instantiation and launch of the backward kernels of chunk_simple_gla.
#include "lmoe_launch.hpp"
#include "lmoe_scalar_bwd.hpp"

namespace lmoe {

template <typename T, int V> struct BwdTiles {
  static constexpr int BVS = sizeof(T) == 4 ? 16 : 32;                // V-slice of the sequential pass
  static constexpr int BVD = V == 128 ? 64 : V;                       // V-slice of k_bwd_dv (LDS for 2-3 work-groups per CU)
  static constexpr int BVH = sizeof(T) == 4 ? 32 : 64;                // V-slice loop of k_bwd_dqk
};

template <bool LOCAL> struct BwdDv {
  template <typename T, int K, int V> struct F {
    static void run(const lmoe_args& a, hipStream_t st) {
      constexpr int BV = BwdTiles<T, V>::BVD;
      hipLaunchKernelGGL((k_bwd_dv<T, K, V, BV, LOCAL>), dim3(a.NT, a.H, V / BV), dim3(NTHR), 0, st, a);
    }
  };
};
template <typename T, int K, int V> struct StateBwd {
  static void run(const lmoe_args& a, hipStream_t st) {
    constexpr int BV = BwdTiles<T, V>::BVS;
    // 64-wide slices where they still fill the chip (2-byte elements): every V slice of a (sequence, head) fetches all
    // of q and k, so two wide slices ask the memory system for less per output column than four narrow ones; a state
    // element is the same sum over the tokens in either split
    constexpr int BW = (sizeof(T) == 2 && V >= 64) ? 64 : BV;
    if (BW != BV && (int64_t)a.N * a.H * (V / BW) >= cu_count()) {
      launch<BW, false>(a, Split{}, st);
      return;
    }
    const Split sp = launch_scalar_seg(a, true, st);
    if (sp.len1) launch<BV, true>(a, sp, st);
    else {
      if constexpr (sizeof(T) == 2) {
        // slices of 16 columns where each finds a CU of its own: K = V = 128, 16 pairs of 16 chunks 19.4 -> 16.8 us, K = V = 64
        // 15.6 -> 13.6; same bits
        if (!a.normalize && (int64_t)a.N * a.H * (V / 16) <= cu_count()) return launch<16, false>(a, sp, st);
      }
      launch<BV, false>(a, sp, st);
    }
  }
  template <int BVX, bool CUT> static void launch(const lmoe_args& a, const Split& sp, hipStream_t st) {
    const dim3 grid(((pass_items(a, sp) * a.H + 7) / 8) * 8 * (V / BVX)), block(2 * NTHR);
    // Rows' places in registers (KEPT) are 10 to 17 of them, and with 4-byte elements and in the wide slices of the
    // normalised pass (K = 128) they cost a CU its last work-group: the second at K = 128, the third at K = 64 with 4-byte elements.
    // That matters where the launch has one, without and with them (us): K = 128, more work-groups than CUs: 4-byte, 64 pairs of
    // 32 chunks 95 and 121, 24 pairs of 128 chunks cut 161 and 180; normalised, 256 pairs of 16 chunks 67 and 74.  K = 64, 4-byte,
    // more than two per CU (whole backward): 96 pairs of 32 chunks, V = 128, 382 and 406, 384 of 16, V = 64, 459 and 466.
    // With fewer they gain, as they do elsewhere: K = 128, 4-byte, 32 pairs of 128 chunks 242 and 228; normalised, 128 pairs
    // of 32 chunks 76 and 72; K = 64, 4-byte, 128 pairs of 32 chunks, V = 64, 319 and 316.
    const bool last = grid.x > (unsigned)(cu_count() * (K == 128 ? 1 : 2));
    if constexpr (sizeof(T) == 2) {        // the pass behind the normalised output exists for 2-byte elements
      if (a.normalize == 1) {
        if constexpr (K == 128 && BVX == 64) {
          if (last) {
            hipLaunchKernelGGL((k_state_bwd<T, K, V, BVX, 1, CUT, false>), grid, block, 0, st, a, sp);
            return;
          }
        }
        hipLaunchKernelGGL((k_state_bwd<T, K, V, BVX, 1, CUT>), grid, block, 0, st, a, sp);
        return;
      }
      if (a.normalize == 2) {
        hipLaunchKernelGGL((k_state_bwd<T, K, V, BVX, 2, CUT>), grid, block, 0, st, a, sp);
        return;
      }
    }
    if constexpr (sizeof(T) == 4) {
      if (last) {
        hipLaunchKernelGGL((k_state_bwd<T, K, V, BVX, 0, CUT, false>), grid, block, 0, st, a, sp);
        return;
      }
    }
    hipLaunchKernelGGL((k_state_bwd<T, K, V, BVX, 0, CUT>), grid, block, 0, st, a, sp);
  }
};
template <typename T, int K, int V> struct BwdDqk {
  static void run(const lmoe_args& a, hipStream_t st) {
    constexpr int BVH = BwdTiles<T, V>::BVH;
    const int grid = persistent_grid(a.NT * a.H, 1);
    if constexpr (sizeof(T) == 2) {
      if (a.normalize == 1) hipLaunchKernelGGL((k_bwd_dqkv<T, K, V, BVH, 1>), dim3(grid), dim3(2 * NTHR), 0, st, a);
      else if (a.normalize == 2) hipLaunchKernelGGL((k_bwd_dqkv<T, K, V, BVH, 2>), dim3(grid), dim3(2 * NTHR), 0, st, a);
      else hipLaunchKernelGGL((k_bwd_dqkv<T, K, V, BVH>), dim3(grid), dim3(2 * NTHR), 0, st, a);
    } else {
      hipLaunchKernelGGL((k_bwd_dqk<T, K, V, BVH>), dim3(grid), dim3(2 * NTHR), 0, st, a);
    }
  }
};

void launch_bwd_dv(const lmoe_args& a, bool local, hipStream_t st) {
  if (local) dispatch<BwdDv<true>::F>(a, st); else dispatch<BwdDv<false>::F>(a, st);
}
void launch_state_bwd(const lmoe_args& a, hipStream_t st) { dispatch<StateBwd>(a, st); }
void launch_bwd_dqk(const lmoe_args& a, hipStream_t st) { dispatch<BwdDqk>(a, st); }

}  // namespace lmoe
