// Instantiation and launch of the sequential passes of the gated delta rule.
#include "lmoe_launch.hpp"
#include "lmoe_gdn_state.hpp"
#include "lmoe_gdn_state_reg.hpp"
#include "lmoe_gdn_split.hpp"

namespace lmoe {

// Width of the V-slice a work-group carries: the narrow slice gives more work-groups (a problem
// with few (sequence, head) pairs must still reach every CU); with enough pairs the wide slice
// halves the number of times k, w, q, P are read and stores whole 128-byte lines of o, v_new.
// (V = 256: not cut; 12 waves of a fine segment's work-group would leave each too few registers for its columns)
Split gdn_split_plan(const lmoe_args& a) { return a.V <= 128 ? plan_split(a, a.V / 32) : Split{}; }
template <typename T, int V> inline bool wide_slices(const lmoe_args& a) {
  constexpr int BW = GdnStateCfg<T>::BV_WIDE;
  return BW <= V && BW != GdnStateCfg<T>::BV && (int64_t)a.N * a.H * (V / BW) >= cu_count();
}
// whether `slices` work-groups per (sequence, head) have a CU each
inline bool pairs_on_cus(const lmoe_args& a, int slices) { return (int64_t)a.N * a.H * slices <= cu_count(); }
// The transitions of a call without a gate are carried in two terms (lmoe_gdn_split.hpp).
inline bool two_terms(const lmoe_args& a) { return a.gate == LMOE_GATE_NONE; }
// How the sequences of a call are cut: not at all without a workspace for it.
inline Split gdn_split(const lmoe_args& a, bool bwd) {
  Split sp = {};
  if (!a.seg_ws || ((bwd || a.hs) && !a.seg_p)) return sp;
  sp = gdn_split_plan(a);
  if (!sp.len1) return sp;
  const int64_t n1 = (int64_t)sp.n1 * a.H, n3 = (int64_t)sp.n3 * a.H, terms = two_terms(a) ? 2 : 1;
  sp.Q = a.seg_ws;
  sp.S = sp.Q + n1 * a.K * a.V;
  sp.P = (bf16*)(sp.S + n3 * a.K * a.V);
  sp.D = (float*)(sp.P + n1 * terms * a.K * a.K);
  if (bwd || a.hs) {
    sp.PT = (bf16*)a.seg_p;
    sp.DT = (float*)(sp.PT + n1 * terms * a.K * a.K);
  }
  return sp;
}
template <int K, int V> void combine(const lmoe_args& a, const Split& sp, bool bwd, hipStream_t st) {
  const dim3 grid((a.N * a.H + 7) / 8 * 8 * (V / 16)), block(2 * K);
  if (two_terms(a)) {
    if (bwd) hipLaunchKernelGGL((k_split_combine<K, true, true>), grid, block, 0, st, a, sp);
    else hipLaunchKernelGGL((k_split_combine<K, false, true>), grid, block, 0, st, a, sp);
  } else {
    if (bwd) hipLaunchKernelGGL((k_split_combine<K, true, false>), grid, block, 0, st, a, sp);
    else hipLaunchKernelGGL((k_split_combine<K, false, false>), grid, block, 0, st, a, sp);
  }
}
template <typename T, int K, int V, int BV> void launch_fwd(const lmoe_args& a, hipStream_t st) {
  const int grid = ((a.N * a.H + 7) / 8) * 8 * (V / BV);
  // w formed on the chip from Tinv where Tinv is there and LDS has room for a second k tile
  constexpr bool CAN_WT = sizeof(T) == 2;
  const bool wt = CAN_WT && a.tinv != nullptr;
  if constexpr (CAN_WT && BV == 32) {
    if (wt) {       // 2-byte elements with Tinv: the state stays in registers (lmoe_gdn_state_reg.hpp)
      if constexpr (V <= 128) {
        const Split sp = gdn_split(a, false);
        if (sp.len1) {
          if (two_terms(a)) hipLaunchKernelGGL((k_gdn_seg_fwd<K, V, true>), dim3(sp.n1 * a.H), dim3(SEG_FWD_THREADS), 0, st, a, sp);
          else hipLaunchKernelGGL((k_gdn_seg_fwd<K, V, false>), dim3(sp.n1 * a.H), dim3(SEG_FWD_THREADS), 0, st, a, sp);
          combine<K, V>(a, sp, false, st);
          const int items = ((sp.n3 * a.H + 7) / 8) * 8 * (V / BV);
          if (a.hs) hipLaunchKernelGGL((k_gdn_state_fwd_reg<K, V, true, false, true>), dim3(items), dim3(3 * NTHR), 0, st, a, sp, (long long*)nullptr, -1);
          else hipLaunchKernelGGL((k_gdn_state_fwd_reg<K, V, false, false, true>), dim3(items), dim3(3 * NTHR), 0, st, a, sp, (long long*)nullptr, -1);
          return;
        }
      }
      // Slices of 16 columns where they all find a CU of their own: a chunk is a chain on one wave either way, and half the
      // waves ask the LDS beside it.  us with the preparation in front, 32 and 16 columns: K = V = 128, 8 pairs of 16 chunks 31.4
      // and 28.7, 32 of 32 62.1 and 58.6 (saving 64.5 and 62.9), K = V = 64, 32 of 32 46.0 and 42.7; but 48 pairs, K = V = 128,
      // 67.9 and 99.9.  Same bits.
      if constexpr (V <= 128) {
        if (pairs_on_cus(a, V / 16)) {
          const dim3 narrow(((a.N * a.H + 7) / 8) * 8 * (V / 16));
          if (a.hs) hipLaunchKernelGGL((k_gdn_state_fwd_reg<K, V, true, false, false, 16>), narrow, dim3(3 * NTHR), 0, st, a, Split{}, (long long*)nullptr, -1);
          else hipLaunchKernelGGL((k_gdn_state_fwd_reg<K, V, false, false, false, 16>), narrow, dim3(3 * NTHR), 0, st, a, Split{}, (long long*)nullptr, -1);
          return;
        }
      }
      if (a.hs) hipLaunchKernelGGL((k_gdn_state_fwd_reg<K, V, true>), dim3(grid), dim3(3 * NTHR), 0, st, a, Split{}, (long long*)nullptr, -1);
      else hipLaunchKernelGGL((k_gdn_state_fwd_reg<K, V, false>), dim3(grid), dim3(3 * NTHR), 0, st, a, Split{}, (long long*)nullptr, -1);
      return;
    }
  }
  // (2-byte elements at V = 256 run with Tinv only, i.e. above: the entry points reject a call without it)
  if constexpr (!(CAN_WT && V > 128)) {
    if (a.hs) {
      if (wt) hipLaunchKernelGGL((k_gdn_state_fwd<T, K, V, BV, true, CAN_WT>), dim3(grid), dim3(3 * NTHR), 0, st, a);
      else hipLaunchKernelGGL((k_gdn_state_fwd<T, K, V, BV, true, false>), dim3(grid), dim3(3 * NTHR), 0, st, a);
    } else {
      if (wt) hipLaunchKernelGGL((k_gdn_state_fwd<T, K, V, BV, false, CAN_WT>), dim3(grid), dim3(3 * NTHR), 0, st, a);
      else hipLaunchKernelGGL((k_gdn_state_fwd<T, K, V, BV, false, false>), dim3(grid), dim3(3 * NTHR), 0, st, a);
    }
  }
}
template <typename T, int K, int V, int BV> void launch_bwd(const lmoe_args& a, hipStream_t st) {
  if constexpr (sizeof(T) == 2 && BV == 32 && V <= 128) {
    const Split sp = gdn_split(a, true);
    if (sp.len1) {
      hipLaunchKernelGGL((k_gdn_seg_bwd<K, V>), dim3(sp.n1 * a.H), dim3(SEG_BWD_THREADS), 0, st, a, sp);
      combine<K, V>(a, sp, true, st);
      hipLaunchKernelGGL((k_gdn_state_bwd<T, K, V, BV, true>), dim3(((sp.n3 * a.H + 7) / 8) * 8 * (V / BV)), dim3(3 * NTHR), 0, st, a, sp);
      return;
    }
  }
  if constexpr (sizeof(T) == 2 && V <= 128) {
    // slices of 16 columns where they all find a CU of their own: 32 pairs of 32 chunks, K = V = 128, 50.9 -> 44.3 us; same bits
    if (pairs_on_cus(a, V / 16)) {
      hipLaunchKernelGGL((k_gdn_state_bwd<T, K, V, 16>), dim3(((a.N * a.H + 7) / 8) * 8 * (V / 16)), dim3(3 * NTHR), 0, st, a, Split{});
      return;
    }
  }
  hipLaunchKernelGGL((k_gdn_state_bwd<T, K, V, BV>), dim3(((a.N * a.H + 7) / 8) * 8 * (V / BV)), dim3(3 * NTHR), 0, st, a, Split{});
}
template <typename T, int K, int V> struct GdnStateFwd {
  static void run(const lmoe_args& a, hipStream_t st) {
    constexpr int BW = GdnStateCfg<T>::BV_WIDE <= V ? GdnStateCfg<T>::BV_WIDE : GdnStateCfg<T>::BV;
    // the register-resident pass is bound by its products, not by latency: twice the columns take twice as long,
    // so it keeps the narrow slice (more work-groups) whatever the problem size
    const bool reg = sizeof(T) == 2 && a.tinv != nullptr;
    if (!reg && wide_slices<T, V>(a)) launch_fwd<T, K, V, BW>(a, st);
    else launch_fwd<T, K, V, GdnStateCfg<T>::BV>(a, st);
  }
};
template <typename T, int K, int V> struct GdnStateBwd {
  static void run(const lmoe_args& a, hipStream_t st) {
    constexpr int BW = GdnStateCfg<T>::BV_WIDE <= V ? GdnStateCfg<T>::BV_WIDE : GdnStateCfg<T>::BV;
    if (wide_slices<T, V>(a)) launch_bwd<T, K, V, BW>(a, st);
    else launch_bwd<T, K, V, GdnStateCfg<T>::BV>(a, st);
  }
};
void launch_gdn_state_fwd(const lmoe_args& a, hipStream_t st) { dispatch_gdn<GdnStateFwd>(a, st); }
// the traced instance of the register-resident forward pass (2-byte elements, K = V = 128, saving call)
bool launch_gdn_state_fwd_trace(const lmoe_args& a, long long* tr, int work_group, hipStream_t st) {
  if (a.dtype != LMOE_BF16 || a.K != 128 || a.V != 128 || !a.tinv || !a.hs) return false;
  const int grid = ((a.N * a.H + 7) / 8) * 8 * (128 / 32);
  if (work_group < 0 || work_group >= grid) return false;
  hipLaunchKernelGGL((k_gdn_state_fwd_reg<128, 128, true, true>), dim3(grid), dim3(3 * NTHR), 0, st, a, Split{}, tr, work_group);
  return true;
}
void split_lengths(const lmoe_args& a, int op, int32_t* fine, int32_t* coarse) {
  const Split sp = op == LMOE_OP_SIMPLE_GLA ? plan_split_scalar(a) : op == LMOE_OP_GLA ? plan_split_gla(a) : gdn_split_plan(a);
  *fine = sp.len1;
  *coarse = sp.len3;
}
int64_t split_floats(const lmoe_args& a, int op, int part) {
  if (op == LMOE_OP_SIMPLE_GLA && part == 1) return scalar_split_floats(a);
  if (op == LMOE_OP_GLA && part == 1) return gla_split_floats(a);
  if (op != LMOE_OP_GATED_DELTA_RULE) return 0;
  const Split sp = gdn_split_plan(a);
  // a matrix of one or two 2-byte terms and a decay per fine segment
  const int64_t trans = (int64_t)sp.n1 * a.H * (a.K * a.K / (two_terms(a) ? 1 : 2) + 1);
  return part == 0 ? trans : (int64_t)(sp.n1 + sp.n3) * a.H * a.K * a.V + trans;
}
void launch_gdn_state_bwd(const lmoe_args& a, hipStream_t st) { dispatch_gdn<GdnStateBwd>(a, st); }

}  // namespace lmoe
