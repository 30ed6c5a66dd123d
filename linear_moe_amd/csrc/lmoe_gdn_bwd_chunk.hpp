// Gated delta rule, chunk-parallel part of the backward: everything that follows the reverse
// state pass, for one (chunk, head) at a time, in one kernel.
//
// The WY form of a chunk is v_new = Tinv Z with Z = beta (v - e^{b} k S) and Tinv = (I + L)^{-1},
// L = strictlower((beta k k^T) . Gamma): v_new solves (I + L) v_new = Z.  Its backward needs no product
// with Tinv once dZ = Tinv^T dv_new is known (the reverse state pass writes dZ, not dv_new):
//     dv = beta dZ,   d(k beta e^{b}) = -dZ S^T,   dL = -strictlower(dZ v_new^T),   dS -= (k beta e^{b})^T dZ.
//
// Inputs per chunk: do, v' = v_new, dZ, S^T and dS'^T (hs, dhs: [V][K]), q, k, v, g, beta.  With
// b = cumulative gate inside the chunk, Gamma_ij = e^{b_i - b_j}, k_b = beta k, k_bg = k_b e^{b}:
//   stage 1 (loop over V-slices of width BVH, contraction over the slice's columns)
//     dP   += do v'^T            dq_i += do S^T         dk_d += v' dS'^T
//     dk_bg -= dZ S^T            dLf  += dZ v'^T
//     (loader waves, from the registers they stage:  dv = beta dZ, stored;  dbeta += <dZ, v>)
//   stage 2
//     G    = scale (dP . Gamma) [i >= j],     dM = -(dLf . Gamma) [i > j]       (L = M . Gamma_s, M = k_b k^T)
//     dq   = scale e_b dq_i + G k                       (stored)
//     dk   = e_d dk_d + G^T q                           (the part that does not pass through the WY form)
//     dk_b = dM k + dk_bg e^{b}
//     dk  += dM^T k_b + dk_b beta                       (stored);   dbeta += <dk_b, k>
//     db_i = q_i.dq_i - k_i.dk_i(first part) + k_b.(dM k) - k.(dM^T k_b) + dk_bg.k_bg
//            (+ on the last row  sum_j (e_d dk_d . k)_j + e^{b_C} <S, dS'>),   dg = reverse cumsum of db
// Nothing but the final gradients leaves the chip.
//
// persistent: grid = one work-group per CU, item = (chunk, head).  Work-group = 12 waves on one
// barrier script: 8 compute waves and 4 loader waves.
//   Compute wave w owns chunk rows 16 (w % 4) .. + 15 and column half w / 4 of every product (half
//   of K for the K-wide ones, 32 of the 64 columns for the chunk x chunk ones).  The compute waves
//   touch only LDS and the matrix cores, apart from the 64 floats of dbeta and dg per item.
//   The loader waves own all other global traffic: they keep the next slices, the next q and k and the
//   next item's g, beta in flight in registers (whole 128-byte lines per row), stage them into
//   LDS (slices into NBUF alternating buffers, q and k into tiles of their own; the three chunk x chunk
//   tiles of stage 2 lie over the last slice buffer), form dv and the value part of dbeta from the
//   registers on the way, and lift dq, dk out of LDS and store them.  They also form <S, dS'> from
//   the registers they hold and the gate cumsum of the chunk.
//   Script per item (NS = 4 slices), three slice buffers:   D0 D1 D2 A | b c d
//     window w: the compute team works on slice w (buffer w % 3); the loaders stage slice w + 2, then q
//     (window 2) and k (window 3), and slices 0, 1 of the next item during b .. d
//   one slice buffer:  [R(0)] D(0) R(1) D(1) .. D(NS-1) | A | b c d | R(0) of the next item
// What bounds it (8192 items, K = V = 128, 16 heads): with its loads served by the L2 and nothing stored 237 us, the compute
// waves alone 167, the loader waves alone 174; with memory, the loaders alone 347, and 304 (5.8 TB/s) with their arithmetic out.  So the loader waves: their
// work between two requests was cut to dot-product instructions for <dZ, v> and <S, dS'>, one set of divisions
// per item, and the compute waves' LDS traffic (reads and 2-byte accesses of stage 2) to a third.  370 -> 350 us; where
// memory binds less 50 -> 43 (2048 x 2 tokens), 97 -> 78 (K = V = 64, 4096 x 4).
#pragma once
#include <type_traits>
#include "lmoe_seq.hpp"

namespace lmoe {

// LDS bytes of k_gdn_bwd_chunk
template <typename T, int K, int BVH, int NBUF> struct GdnBwdChunkLds {
  static constexpr int LDV = BVH + LPAD, LDC = CH + LPAD, LDK = K + LPAD;
  static constexpr int A_END = 3 * CH * LDV + 2 * BVH * LDK;      // do, v_new, dZ; S^T, dS'^T of one slice
  static constexpr int T_END = 3 * CH * LDC;                      // G^T, dM^T, (beta dM)^T: over the last slice buffer
  static constexpr int S_END = (NBUF - 1) * A_END + (A_END > T_END ? A_END : T_END);   // slice buffers, the last one widened to hold the tiles
  static constexpr int NREG = S_END + 2 * CH * LDK;               // ..; q, k
  static constexpr int BYTES = NREG * (int)sizeof(T) + (13 * 64 + 16) * 4;
};

// compile-time loop: f(IC<0>()), .., f(IC<N - 1>())
template <int I> struct IC { static constexpr int value = I; };
template <int N, int I = 0, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(IC<I>());
    static_for<N, I + 1>(f);
  }
}

// Forces x to be computed here: without it the compiler moves a running sum's updates down to
// the sum's first use, and keeps every operand alive (spilled) until then.
__device__ __forceinline__ void pin(float& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void pin(float (&x)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) pin(x[i]);
}

// QKACT: q and k as given are l2norm(silu(.)) of rows of a projection that the caller holds (lmoe_args.q_raw, k_raw):
// dq and dk leave as the gradients with respect to those rows - the backward of the L2 norm and of SiLU is applied to
// the dq, dk tiles on their way from LDS to memory, by the loader threads that store them, from the raw rows, which
// are requested when stage 2 begins.  (What it costs is those rows: 32 KB more per item through a request path that is
// full; the arithmetic, spread over the first windows of the next item or not, is a tenth of it.)
template <typename T, int K, int V, int BVH, int NBUF, int DEPTH, bool QKACT = false>
__global__ __launch_bounds__(3 * NTHR) void k_gdn_bwd_chunk(const lmoe_args a) {
  static_assert(!QKACT || (sizeof(T) == 2 && NBUF == 3), "the activation backward exists for 2-byte elements");
  typedef GdnBwdChunkLds<T, K, BVH, NBUF> L;
  constexpr int LDV = L::LDV, LDC = L::LDC, LDK = L::LDK;
  constexpr int NS = V / BVH;
  constexpr int KH = K / 2, NBK = KH / 16;     // columns / 16-wide tiles of a K-wide product per compute wave
  static_assert(V % BVH == 0 && BVH == 32, "V-slices: the 8 compute waves split a 64 x 32 slice product 4 x 2");
  static_assert(NBUF == 1 || NBUF == 3, "one slice buffer, or three in rotation");
  // tiles of one V-slice
  constexpr int A_DO = 0, A_VN = A_DO + CH * LDV, A_DZ = A_VN + CH * LDV,
                A_H = A_DZ + CH * LDV, A_DH = A_H + BVH * LDK, A_END = L::A_END;
  // stage 2: q (later dq on its way out) and k (later dk) in tiles of their own; T0 = G^T, T1 = dM^T,
  // T2 = (diag(beta) dM)^T over the last slice buffer
  constexpr int B_T0 = (NBUF - 1) * A_END, B_T1 = B_T0 + CH * LDC, B_T2 = B_T1 + CH * LDC;
  constexpr int B_Q = L::S_END, B_K = B_Q + CH * LDK;
  __shared__ __attribute__((aligned(16))) T smem[L::NREG];
  // gate cumsum, its exponentials and beta: two copies, the loaders fill the next item's during stage 2
  __shared__ float s_gb[2][64], s_geb[2][64], s_ged[2][64], s_gbeta[2][64], s_db[2][64], s_dbeta[2][64], s_dbv[64], s_red[16];

  typedef TileIO<T, CH, BVH> IOV;
  typedef TileIO<T, BVH, K> IOH;
  typedef TileIO<T, CH, K> IOK;
  const int nitems = num_chunks(a) * a.H;
  if (nitems <= 0) return;                   // (a chunk count read on the device may be zero)
  const int stride = gridDim.x;

  if (threadIdx.x >= 2 * NTHR) {
    // --------------------------------- loaders -------------------------------------------
    const int l = lane_id();
    // thread index inside the team, refreshed per item: the per-thread tile offsets are then recomputed
    // where they are used instead of held (and spilled) for the whole kernel
    int tid = threadIdx.x & (NTHR - 1);
    const int lw = wave_id() - 8;            // wave of the loader team
    // The bulk input of an item is a sequence of NU units: the NS slices, then q, then k.  Units go
    // through DEPTH register sets in rotation (unit u uses set u % DEPTH; NU is a multiple of DEPTH):
    // staging unit u into LDS frees its set for unit u + DEPTH, so DEPTH - 1 .. DEPTH units are in
    // flight at any time.  Every load is issued unconditionally (item index clamped to the last item):
    // a load that is skipped on some path would make the compiler drain all outstanding loads at
    // every use.
    constexpr int NU = NS + 2;
    constexpr int PV = IOV::PASSES, PH = IOH::PASSES, PK = IOK::PASSES;
    constexpr int NVEC = (4 * PV + 2 * PH) > PK ? (4 * PV + 2 * PH) : PK;
    static_assert(NU % DEPTH == 0, "units per item and register sets");
    typedef typename ET<T>::vec vec;
    struct Unit { vec v[NVEC]; int len; };
    Unit U[DEPTH];
    uint32_t graw, braw;
    int glen;
    float hdh = 0.f;   // partial <S, dS'> of the item whose slices are being staged
    float dbv[PV];     // partial <dZ, v> of this thread's rows of that item
#pragma unroll
    for (int p = 0; p < PV; ++p) dbv[p] = 0.f;
    // Where an item's rows lie: worked out once per item, for its six units, its stores and (as the item after this one) its
    // first units.  (Per unit, the divisions by H and by the chunks of a sequence were a thousand scalar instructions
    // per item on the waves whose requests bound the kernel.  The row pointers are formed where they are used: kept as
    // well, they spill to vector lanes.)
    struct Item { int it, h, b, tok, len; };
    auto item_at = [&](int it) {
      Item I;
      I.it = __builtin_amdgcn_readfirstlane(min(it, nitems - 1));
      const int cid = I.it / a.H;
      I.h = I.it - cid * a.H;
      const ChunkInfo ci = chunk_info(a, cid);
      I.b = ci.b; I.tok = ci.tok; I.len = ci.len;
      return I;
    };
    auto rows = [&](const lmoe_tensor& x, const Item& I) { return row_ptr<T>(x, I.b, I.tok, I.h); };
    // unit u counted from the first unit of the item cur (u >= NU: units of the item after it, nxt)
    auto issue = [&](auto uc, const Item& cur, const Item& nxt) {
      constexpr int u = decltype(uc)::value, unit = u % NU;
      static_assert(u < 2 * NU, "units of this item and the next");
      const Item& I = u < NU ? cur : nxt;
      Unit& R = U[u % DEPTH];
      R.len = I.len;
      if constexpr (unit < NS) {
        constexpr int vv = unit * BVH;
        static_assert(BVH == SLICE_COLS, "a slice of this kernel is one block of vnew / dvnew");
        // do, v: the caller's rows; vnew, dvnew (= dZ): one contiguous block per (chunk, head, slice)
        const int64_t block = ((int64_t)I.it * NS + unit) * (CH * SLICE_COLS);
        const T* ts[4] = {rows(a.d_o, I) + vv, (const T*)a.vnew.ptr + block, (const T*)a.dvnew.ptr + block, rows(a.v, I) + vv};
        const int64_t st[4] = {a.d_o.st, SLICE_COLS, SLICE_COLS, a.v.st};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          typename IOV::Regs r;
          IOV::load_nomask(r, ts[t], st[t], I.len, tid);
#pragma unroll
          for (int p = 0; p < PV; ++p) R.v[t * PV + p] = r.v[p];
        }
        const T* hp[2] = {(const T*)a.hs, (const T*)a.dhs};
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          typename IOH::Regs r;
          IOH::load_nomask(r, hp[t] + ((int64_t)I.it * V + vv) * K, K, BVH, tid);       // it = cid * H + h
#pragma unroll
          for (int p = 0; p < PH; ++p) R.v[4 * PV + t * PH + p] = r.v[p];
        }
      } else {
        typename IOK::Regs r;
        const lmoe_tensor& x = unit == NS ? a.q : a.k;
        IOK::load_nomask(r, rows(x, I), x.st, I.len, tid);
#pragma unroll
        for (int p = 0; p < PK; ++p) R.v[p] = r.v[p];
      }
    };
    // dv of a slice on its way from the registers to memory
    struct DV { typename IOV::Regs r; };
    // unit u (u >= NU: of the next item) from its registers into LDS; slices go to buffer buf, and their dv = beta dZ
    // into d (gp = the copy of the gate arrays that holds the beta of the unit's item)
    auto stage = [&](auto uc, int buf, int gp, DV& d) {
      constexpr int u = decltype(uc)::value, unit = u % NU;
      Unit& R = U[u % DEPTH];
      if constexpr (unit < NS) {
        T* base = smem + buf * A_END;
        // dv and <dZ, v> first, from the registers as loaded: rows past the end of a partial chunk repeat its last row
        // there, which is what the branch-free store of dv rewrites
#pragma unroll
        for (int p = 0; p < PV; ++p) {
          int row, col; IOV::coords(p, row, col, tid);
          const float bt = s_gbeta[gp][min(row, R.len - 1)];
          const vec z = R.v[2 * PV + p], vv = R.v[3 * PV + p];
          vec o;
          float s = 0.f;
          if (sizeof(T) == 2 && a.v_act) {
            // v as given is the argument of a SiLU: the op runs on silu(v) (rounded to the element type, as the
            // forward pass staged it) and dv is the gradient with respect to the argument
#pragma unroll
            for (int i = 0; i < IOV::VEC; ++i) {
              const float zf = ET<T>::to_f(z[i]), vr = ET<T>::to_f(vv[i]);
              o[i] = ET<T>::from_f(zf * bt * silu_grad(vr));
              s += zf * ET<T>::to_f(ET<T>::from_f(silu_of(vr)));
            }
          } else {
#pragma unroll
            for (int i = 0; i < IOV::VEC; ++i) o[i] = ET<T>::from_f(ET<T>::to_f(z[i]) * bt);
            s = dot_vec(z, vv, 0.f);
          }
          d.r.v[p] = o;
          s = group_sum<IOV::VPR>(s);                   // the VPR lanes that hold one row are neighbours
          dbv[p] += row < R.len ? s : 0.f;
          pin(dbv[p]);
        }
        constexpr int off[3] = {A_DO, A_VN, A_DZ};
#pragma unroll
        for (int t = 0; t < 3; ++t) {
          typename IOV::Regs r;
#pragma unroll
          for (int p = 0; p < PV; ++p) r.v[p] = R.v[t * PV + p];
          IOV::mask(r, R.len, tid);
          IOV::store_lds(r, base + off[t], LDV, tid);
        }
        typename IOH::Regs rh, rdh;
#pragma unroll
        for (int p = 0; p < PH; ++p) { rh.v[p] = R.v[4 * PV + p]; rdh.v[p] = R.v[4 * PV + PH + p]; }
#pragma unroll
        for (int p = 0; p < PH; ++p) hdh = dot_vec(rh.v[p], rdh.v[p], hdh);
        pin(hdh);                                         // here, not where the item is closed (the tiles would stay live)
        IOH::store_lds(rh, base + A_H, LDK, tid);
        IOH::store_lds(rdh, base + A_DH, LDK, tid);
      } else {
        typename IOK::Regs r;
#pragma unroll
        for (int p = 0; p < PK; ++p) r.v[p] = R.v[p];
        IOK::mask(r, R.len, tid);
        IOK::store_lds(r, smem + (unit == NS ? B_Q : B_K), LDK, tid);
      }
    };
    auto store_dv = [&](const DV& d, const Item& I, int s) {
      IOV::template store_global_clamped<true>(d.r, rows(a.dv, I) + s * BVH, a.dv.st, I.len, tid);
    };
    // an item and the request of its gates
    auto issue_gates = [&](int it) {
      const Item I = item_at(it);
      glen = I.len;
      graw = gate_prefetch(a, I.b, I.tok, I.len, I.h);
      braw = load_scalar_raw(a.beta.ptr, a.beta_dtype, row_off(a.beta, I.b, I.tok + min(l, I.len - 1), I.h));
      return I;
    };
    // gate cumsum and beta of an item into copy par
    auto stage_gates = [&](int par) {
      gate_finish_wave(a, graw, glen, l, lw == 0, s_gb[par], s_geb[par], s_ged[par]);
      if (lw == 1) s_gbeta[par][l] = l < glen ? scalar_from_raw(braw, a.beta_dtype) : 0.f;
    };
    // the sums of an item whose slices have all been staged
    auto close_item = [&]() {
      hdh = wave_sum(hdh);
      if (l == 0) s_red[lw] = hdh;
      hdh = 0.f;
#pragma unroll
      for (int p = 0; p < PV; ++p) {
        int row, col; IOV::coords(p, row, col, tid);
        if (col == 0) s_dbv[row] = dbv[p];
        dbv[p] = 0.f;
      }
    };
    // QKACT: the raw rows behind q and k of an item, and the backward of y = l2norm(silu(x)) on a tile of dy:
    //   s = silu(x), r = (|s|^2 + eps)^-1/2, dx = silu'(x) (dy r - (dy . s) r^3 s)
    // with the sums of a row over the VPR neighbouring lanes that hold it (the arithmetic, step for step, of the row
    // kernel that does the same in front of the op: the results agree bit for bit)
    typename IOK::Regs XQ, XK;
    auto issue_raw = [&](const Item& I) __attribute__((always_inline)) {
      if constexpr (QKACT) {
        IOK::load_nomask(XQ, rows(a.q_raw, I), a.q_raw.st, I.len, tid);
        IOK::load_nomask(XK, rows(a.k_raw, I), a.k_raw.st, I.len, tid);
      }
    };
    auto act_backward = [&](typename IOK::Regs& r, const typename IOK::Regs& X) __attribute__((always_inline)) {
      if constexpr (QKACT) {
#pragma unroll
        for (int p = 0; p < PK; ++p) {
          float sv[IOK::VEC], gv[IOK::VEC], fv[IOK::VEC], ss = 0.f, c = 0.f;
#pragma unroll
          for (int i = 0; i < IOK::VEC; ++i) {
            const float x = ET<T>::to_f(X.v[p][i]), sg = sigmoid_fast(x);
            sv[i] = x * sg;
            gv[i] = sg * (1.0f + x * (1.0f - sg));
            ss += sv[i] * sv[i];
          }
#pragma unroll
          for (int i = 0; i < IOK::VEC; ++i) { fv[i] = ET<T>::to_f(r.v[p][i]); c += fv[i] * sv[i]; }
          ss = group_sum<IOK::VPR>(ss);
          c = group_sum<IOK::VPR>(c);
          const float rn = rsqrt_fast(ss + a.qk_eps);
          c = c * rn * rn * rn;
#pragma unroll
          for (int i = 0; i < IOK::VEC; ++i) r.v[p][i] = ET<T>::from_f((fv[i] * rn - c * sv[i]) * gv[i]);
        }
      }
    };
    // (a launch sized by an upper bound of the chunk count may hold work-groups without an item: they stage the last
    // item like every load past the end and skip the loop)
    const int it0 = min((int)blockIdx.x, nitems - 1);
    DV d0, d1;
    Item cur = issue_gates(it0);
    static_for<DEPTH>([&](auto jc) { issue(jc, cur, cur); });
    // the first loads may be ordered freely by the compiler; were they still pending at the loop
    // header, its wait-count analysis would carry that order into every iteration
    wait_all_loads();
    stage_gates(0);
    Item nxt = issue_gates(it0 + stride);
    lds_barrier();                                                                       // beta of the first item staged
    stage(IC<0>(), 0, 0, d0);
    issue(IC<DEPTH>(), cur, nxt);
    store_dv(d0, cur, 0);
    if constexpr (NBUF == 3) {
      stage(IC<1>(), 1, 0, d1);
      issue(IC<1 + DEPTH>(), cur, nxt);
      store_dv(d1, cur, 1);
    }
    int par = 0;
    lds_barrier();                                                                       // first slice staged
    for (int it = blockIdx.x; it < nitems; it += stride) {
      tid = fresh_index(tid) & (NTHR - 1);
      Item aft;                                                                          // two items ahead
      if constexpr (NBUF == 3) {
        // window w: the compute team works on slice w.  Slice s lives in buffer s % 3 and is staged two
        // windows ahead; q and k follow in windows 2 and 3.
        // In every window the loaders fill LDS first and meet the compute team at the barrier; the stores and the
        // requests that refill the freed registers follow the barrier.  Requests stall at the issue while the CU's
        // queue is full (32 KB take about a microsecond): issued before the barrier, that stall holds up the
        // compute team.
        static_for<NS>([&](auto wc) {
          constexpr int w = decltype(wc)::value, u = w + 2;    // u < NS: a slice (buffer u % 3), then q, then k
          stage(IC<u>(), u % 3, par, d0);
          if constexpr (w == NS - 1) close_item();
          lds_barrier();                                                                 // D(w); the last one is A
          if constexpr (u < NS) store_dv(d0, cur, u);
          if constexpr (w < NS - 1) issue(IC<u + DEPTH>(), cur, nxt);                       // q, k, slice 0 of the next item
        });
        issue_raw(cur);                                                                  // (QKACT) used behind d
        issue(IC<NS + 1 + DEPTH>(), cur, nxt);                                           // slice 1 of the next item
        stage_gates(par ^ 1);                                  // the next item's; its copy is idle since d of the last item
        aft = issue_gates(it + 2 * stride);
        lds_barrier();                                                                   // b
        stage(IC<NU>(), 0, par ^ 1, d0);                       // slice 0 of the next item (buffer 0: slice 3 is done)
        lds_barrier();                                                                   // c
        store_dv(d0, nxt, 0);
        issue(IC<NU + DEPTH>(), cur, nxt);                                               // slice 2 of the next item
        stage(IC<NU + 1>(), 1, par ^ 1, d1);                   // slice 1 of the next item
        lds_barrier();                                                                   // d: dq, dk lie in the q, k tiles
        store_dv(d1, nxt, 1);
        issue(IC<NU + 1 + DEPTH>(), cur, nxt);                                           // slice 3 of the next item
      } else {
        static_for<NS>([&](auto sc) {
          constexpr int s = decltype(sc)::value;
          if constexpr (s > 0) lds_barrier();                                            // R(s)
          lds_barrier();                                                                 // D(s)
          if constexpr (s + 1 < NS) {
            stage(IC<s + 1>(), 0, par, d0);
            issue(IC<s + 1 + DEPTH>(), cur, nxt);
            store_dv(d0, cur, s + 1);
          }
        });
        stage(IC<NS>(), 0, par, d0);                                                     // q
        issue(IC<NS + DEPTH>(), cur, nxt);
        stage(IC<NS + 1>(), 0, par, d0);                                                 // k
        issue(IC<NS + 1 + DEPTH>(), cur, nxt);
        close_item();
        lds_barrier();                                                                   // A
        stage_gates(par ^ 1);
        aft = issue_gates(it + 2 * stride);
        lds_barrier();                                                                   // b
        lds_barrier();                                                                   // c
        lds_barrier();                                                                   // d
      }
      {
        typename IOK::Regs r;
        IOK::load_lds_clamped(r, smem + B_Q, LDK, cur.len, tid);
        act_backward(r, XQ);
        IOK::template store_global_clamped<true>(r, rows(a.dq, cur), a.dq.st, cur.len, tid);
        if constexpr (sizeof(T) == 4) tid = fresh_index(tid) & (NTHR - 1);       // (one tile's addresses at a time: both spill)
        IOK::load_lds_clamped(r, smem + B_K, LDK, cur.len, tid);
        act_backward(r, XK);
        IOK::template store_global_clamped<true>(r, rows(a.dk, cur), a.dk.st, cur.len, tid);
      }
      if constexpr (NBUF == 1) {
        stage(IC<NU>(), 0, par ^ 1, d0);                       // slice 0 of the next item
        issue(IC<NU + DEPTH>(), cur, nxt);
        store_dv(d0, nxt, 0);
        lds_barrier();                                                                   // R(0) of the next item
      }
      par ^= 1;
      cur = nxt;
      nxt = aft;
    }
    return;
  }

  // --------------------------------- compute ---------------------------------------------
  __builtin_amdgcn_s_setprio(3);           // compute waves before the loader wave of their SIMD
  const int wv = wave_id();
  const int r0 = 16 * (wv & 3);            // rows of this wave
  const int ch = wv >> 2;                  // column half
  const int c0 = 32 * ch;                  // first column in a chunk x chunk product
  const int k0 = KH * ch;                  // first column in a K-wide product
  const float scale = a.scale;
  int par = 0;
  lds_barrier();                                                                         // beta of the first item staged
  lds_barrier();                                                                         // first slice staged
  for (int it = blockIdx.x; it < nitems; it += stride) {
    const float* s_b = s_gb[par]; const float* s_eb = s_geb[par]; const float* s_ed = s_ged[par];
    const float* s_beta = s_gbeta[par];
    // the lane index is refreshed per item: address arithmetic derived from it then stays inside
    // the iteration instead of living in registers for the whole kernel
    const int l = fresh_index(lane_id()) & 63;
    const int fr = l & 15, fg = 8 * (l >> 4);
    const int rb = r0 + 4 * (l >> 4);      // chunk x chunk products: element i is row rb + i, column (tile) + fr
    // K-wide products are formed transposed (the state, k or q as the A operand): element i is K column kc + 16 ni + i of
    // token r0 + fr, so that q, k are read and dq, dk written four columns (8 bytes) at a time and the factors of a token
    // are one value per lane.  (Token by row, the same accesses were 96 2-byte ones per wave and item.)
    const int tk = r0 + fr, kc = k0 + 4 * (l >> 4);
    f32x4 dP[1][2], dLf[1][2], dqi[NBK], dkd[NBK], dkbg[NBK];
    acc_zero(dP); acc_zero(dLf);
#pragma unroll
    for (int ni = 0; ni < NBK; ++ni) dqi[ni] = dkd[ni] = dkbg[ni] = f32x4{0.f, 0.f, 0.f, 0.f};
    // ---- stage 1 ----
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if constexpr (NBUF == 1) {
        if (s > 0) lds_barrier();                                                        // R(s)
      }
      const T* base = smem + (NBUF == 3 ? (s % 3) * A_END : 0);
      const T* DO = base + A_DO; const T* VN = base + A_VN; const T* DZ = base + A_DZ;
      const T* HT = base + A_H; const T* DHT = base + A_DH;
#pragma unroll
      for (int kk = 0; kk < BVH; kk += 32) {
        const typename ET<T>::frag aDO = ET<T>::load_frag(DO + (r0 + fr) * LDV + kk + fg);
        const typename ET<T>::frag aVN = ET<T>::load_frag(VN + (r0 + fr) * LDV + kk + fg);
        const typename ET<T>::frag aDZ = ET<T>::load_frag(DZ + (r0 + fr) * LDV + kk + fg);
#pragma unroll
        for (int nj = 0; nj < 2; ++nj) {
          const typename ET<T>::frag bVN = ET<T>::load_frag(VN + (c0 + 16 * nj + fr) * LDV + kk + fg);
          ET<T>::mma(dP[0][nj], aDO, bVN);
          ET<T>::mma(dLf[0][nj], aDZ, bVN);
        }
#pragma unroll
        for (int ni = 0; ni < NBK; ++ni) {
          const typename ET<T>::frag bH = ET<T>::load_frag_t(HT, LDK, kk, k0 + 16 * ni, l);
          ET<T>::mma(dqi[ni], bH, aDO);
          ET<T>::mma(dkbg[ni], bH, aDZ);                                                 // + dZ S^T: dk_bg is its negative
          ET<T>::mma(dkd[ni], ET<T>::load_frag_t(DHT, LDK, kk, k0 + 16 * ni, l), aVN);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      lds_barrier();                                                                     // D(s); with three buffers the last one is A
    }
    if constexpr (NBUF == 1) lds_barrier();                                              // A: q, k staged
    // ---- stage 2 ----
    T* Qt = smem + B_Q; T* Kt = smem + B_K; T* T0 = smem + B_T0; T* T1 = smem + B_T1; T* T2 = smem + B_T2;
    typedef typename ET<T>::vec4 vec4;
    typedef typename ET<T>::frag frag;
    constexpr int CS = CH / 32;
    // The k^T fragments serve three of the four products and are requested while G and dM are formed; the rows of q and k
    // that the sums need are read once.  (Every product with fragments of its own, each step waited for: 80 transposing
    // reads per wave and item where these are 32, and the LDS round trips of 8 steps behind barrier b.)
    // 2-byte elements only: a 4-byte fragment is eight registers, and kept they and the rows spill (81 registers at K = 128;
    // 1024 items, K = V = 128: 197 us, and 156 without).  Those instances read each where it is used, a step at a time.
    constexpr bool KEPT = sizeof(T) == 2;
    frag ft[KEPT ? CS : 1][NBK];
    vec4 k4[NBK], q4[NBK];
    auto keep = [&](const T* tile) {
      if constexpr (KEPT) {
#pragma unroll
        for (int ks = 0; ks < CS; ++ks)
#pragma unroll
          for (int ni = 0; ni < NBK; ++ni) ft[ks][ni] = ET<T>::load_frag_t(tile, LDK, 32 * ks, k0 + 16 * ni, l);
      }
    };
    // (4-byte: through an offset the compiler cannot see through, which would otherwise keep the values of the first reading)
    auto row4 = [&](const vec4& kept, const T* tile, int ni) -> vec4 {
      if constexpr (KEPT) return kept;
      else return *(const vec4*)(tile + fresh_index(tk * LDK + kc + 16 * ni));
    };
    keep(Kt);
#pragma unroll
    for (int nj = 0; nj < 2; ++nj) {
      f32x4 g, m, mb;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = rb + i, cc = c0 + 16 * nj + fr;
        const float e = (r >= cc) ? texp<T>(s_b[r] - s_b[cc]) : 0.f;
        g[i] = scale * dP[0][nj][i] * e;
        m[i] = (r > cc) ? -dLf[0][nj][i] * e : 0.f;
        mb[i] = m[i] * s_beta[r];
      }
      acc_to_lds_t<T>(g, T0, LDC, r0, c0 + 16 * nj, l);                                  // G^T [j][i]
      acc_to_lds_t<T>(m, T1, LDC, r0, c0 + 16 * nj, l);                                  // dM^T [j][i]
      acc_to_lds_t<T>(mb, T2, LDC, r0, c0 + 16 * nj, l);                                 // (diag(beta) dM)^T [j][i]
    }
    lds_barrier();                                                                       // b
    float dbp[4] = {0.f, 0.f, 0.f, 0.f};      // db of token tk (partial over elements, lanes and column halves)
    float dbt[4] = {0.f, 0.f, 0.f, 0.f};      // dbeta of token tk, the part through k_b
    float kk = 0.f;
    // acc += (tile^T's rows r0 .., or the tile's rows) times the operand x (q or k), which ft holds.  The tiles are triangular:
    // rows of the first half have no entries in the second half of the contraction, and the other way round for the
    // transposed tile
    auto products = [&](f32x4 (&acc)[NBK], const T* tile, auto transposed, const T* x) {
      constexpr bool TR = decltype(transposed)::value;
      auto tile_frag = [&](int ks) {
        return TR ? ET<T>::load_frag_t(tile, LDC, 32 * ks, r0, l) : ET<T>::load_frag(tile + tk * LDC + 32 * ks + fg);
      };
      frag fb[KEPT ? CS : 1];
      if constexpr (!KEPT) __builtin_amdgcn_sched_barrier(0);
      if constexpr (KEPT) {
#pragma unroll
        for (int ks = 0; ks < CS; ++ks) fb[ks] = tile_frag(ks);
      }
#pragma unroll
      for (int ni = 0; ni < NBK; ++ni) acc[ni] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < CS; ++ks) {
        if (TR ? (ks == 0 || r0 >= 32) : (ks == 1 || r0 < 32)) {
          if constexpr (KEPT) {
#pragma unroll
            for (int ni = 0; ni < NBK; ++ni) ET<T>::mma(acc[ni], ft[ks][ni], fb[ks]);
          } else {
            const frag y = tile_frag(ks);
#pragma unroll
            for (int ni = 0; ni < NBK; ++ni) ET<T>::mma(acc[ni], ET<T>::load_frag_t(x, LDK, 32 * ks, k0 + 16 * ni, l), y);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
    };
    if constexpr (KEPT) {
#pragma unroll
      for (int ni = 0; ni < NBK; ++ni) {
        q4[ni] = *(const vec4*)(Qt + tk * LDK + kc + 16 * ni);
        k4[ni] = *(const vec4*)(Kt + tk * LDK + kc + 16 * ni);
      }
    }
    const float ebt = s_eb[tk], edt = s_ed[tk], bt = s_beta[tk];
    f32x4 dq[NBK], dk[NBK], m[NBK];
    products(dq, T0, std::true_type(), Kt);                                              // (G k)^T
    if constexpr (KEPT) products(m, T1, std::true_type(), Kt);                           // (dM k)^T: closes dk_b
#pragma unroll
    for (int ni = 0; ni < NBK; ++ni) {
      const vec4 q_ = row4(q4[ni], Qt, ni);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float dqv = scale * ebt * dqi[ni][i] + dq[ni][i];
        dbp[i] += ET<T>::to_f(q_[i]) * dqv;
        dq[ni][i] = dqv;                                                                 // final dq
      }
    }
    pin(dbp);
    if constexpr (!KEPT) products(m, T1, std::true_type(), Kt);
#pragma unroll
    for (int ni = 0; ni < NBK; ++ni) {
      const vec4 k_ = row4(k4[ni], Kt, ni);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float kv = ET<T>::to_f(k_[i]);
        const float kbv = kv * bt;
        const float dkbgv = -dkbg[ni][i];
        const float dkb = m[ni][i] + dkbgv * ebt;
        dbt[i] += dkb * kv;
        dbp[i] += kbv * m[ni][i] + dkbgv * kbv * ebt;
        dk[ni][i] = dkb * bt;
      }
    }
    pin(dbp);
    pin(dbt);
    products(m, T2, std::false_type(), Kt);                                              // (dM^T k_b)^T
    keep(Qt);                                              // k^T is done with: q^T for the last product
#pragma unroll
    for (int ni = 0; ni < NBK; ++ni) {
      const vec4 k_ = row4(k4[ni], Kt, ni);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        dbp[i] -= ET<T>::to_f(k_[i]) * m[ni][i];
        dk[ni][i] += m[ni][i];
      }
    }
    pin(dbp);
    products(m, T0, std::false_type(), Qt);                                              // (G^T q)^T
#pragma unroll
    for (int ni = 0; ni < NBK; ++ni) {
      const vec4 k_ = row4(k4[ni], Kt, ni);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float kv = ET<T>::to_f(k_[i]);
        const float dkdv = edt * dkd[ni][i];
        const float dkv = dkdv + m[ni][i];                                               // the part of dk that does not pass through the WY form
        dbp[i] -= kv * dkv;
        kk += kv * dkdv;
        dk[ni][i] += dkv;                                                                // final dk
      }
    }
    // over the elements and the four lanes that hold a token
    float dbs = (dbp[0] + dbp[1]) + (dbp[2] + dbp[3]), dts = (dbt[0] + dbt[1]) + (dbt[2] + dbt[3]);
    dbs += __shfl_xor(dbs, 16, 64);
    dts += __shfl_xor(dts, 16, 64);
    dbs += __shfl_xor(dbs, 32, 64);
    dts += __shfl_xor(dts, 32, 64);
    kk = wave_sum(kk);
    lds_barrier();                                                                       // c: q, k, the chunk x chunk tiles read
#pragma unroll
    for (int ni = 0; ni < NBK; ++ni) {
      acc_to_lds_t<T>(dq[ni], Qt, LDK, k0 + 16 * ni, r0, l);                          // dq, dk on their way out
      acc_to_lds_t<T>(dk[ni], Kt, LDK, k0 + 16 * ni, r0, l);
    }
    if (l < 16) {
      s_db[ch][tk] = dbs;
      s_dbeta[ch][tk] = dts;
    }
    if (l == 0) s_red[4 + wv] = kk;
    lds_barrier();                                                                       // d
    if (threadIdx.x < 64) {
      const int cid = it / a.H, h = it % a.H;
      const ChunkInfo ci = chunk_info(a, cid);
      // refreshed: the LDS addresses derived from it are otherwise hoisted out of the item loop and spilled
      const int j = fresh_index(threadIdx.x) & 63;
      float x = 0.f;
      if (j < ci.len) {
        const float y = s_dbeta[0][j] + s_dbeta[1][j] + s_dbv[j];
        const int64_t at = row_off(a.dbeta, ci.b, ci.tok + j, h);
        if (a.dbeta_bf16) ((bf16*)a.dbeta.ptr)[at] = (bf16)y;
        else ((float*)a.dbeta.ptr)[at] = y;
        x = s_db[0][j] + s_db[1][j];
        // last-row term; rows past the end of a partial chunk carry zero q, k, so the term may sit
        // on the last valid row without changing the reverse cumulative sum
        if (j == ci.len - 1) {
          float skk = 0.f, shd = 0.f;
#pragma unroll
          for (int w = 0; w < 8; ++w) skk += s_red[4 + w];
#pragma unroll
          for (int w = 0; w < 4; ++w) shd += s_red[w];
          x += skk + expf(s_b[CH - 1]) * shd;
        }
      }
      x = wave_rev_scan(x);
      if (j < ci.len) ((float*)a.dg.ptr)[row_off(a.dg, ci.b, ci.tok + j, h)] = x;
    }
    if constexpr (NBUF == 1) lds_barrier();                                              // R(0) of the next item
    par ^= 1;
  }
}

}  // namespace lmoe
