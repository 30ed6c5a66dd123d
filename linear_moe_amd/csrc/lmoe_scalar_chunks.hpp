// chunk_simple_gla forward, 4-byte elements, short sequences: every chunk on its own.
//
// A pass over a sequence is a chain of chunks (4 us each at K = 64, 6 at K = 128) on few CUs, and cut into segments
// (lmoe_scalar_split.hpp) two launches.  Here every work-group takes one (sequence, head, chunk, 16-column slice of V), sums up
// the state its chunk starts from itself,  S = sum over the chunks in front of  (decay to their end)  k^T (e_d v),  and forms
// the chunk's output: no chain, one launch.  The sums over the tokens in front are formed again by every chunk, which with
// the waves of a work-group bounds how long a sequence may be: fwd_by_chunks (lmoe_scalar_fwd.hip).
#pragma once
#include "lmoe_seq.hpp"

namespace lmoe {

constexpr int CHUNKS_PREFIX_WAVES = 8;      // at most so many chunks in front of a work-group's own (or behind the last)

// Work-group of twelve waves.  Waves 0 .. 7 take one of the chunks in front of this one each, straight from memory into matrix
// operands; their sums meet in LDS and are folded in order, S <- D S + Q.  Waves 8 .. 11 meanwhile form
// (q k^T . Gamma) v  of 16 output rows each, also straight from memory, and add  e^b q S  when the state is there.  A matrix
// step of four tokens is numbered so that the lanes' loads are 16-byte ones: a lane's four values of a k row are one row of
// four blocks of the state, its four of a q row four steps of a contraction.  With a final state asked for, one more
// work-group per sequence stands behind the last chunk.
// Bound by its launch, the first loads and the matrix instructions of the last chunks' work-groups (a wave's share of a 64-token
// chunk: 64 of 32 cycles at K = 64).  us, replayed as a graph, segments and pass (T = 256, 64: the pass) -> this, B = 1, H = 4:
// K = V = 64, T = 512 12.4 -> 8.8, T = 256 18.4 -> 7.1, T = 64 7.05 -> 6.6; K = V = 128, T = 512 20.0 -> 13.8.  K = 64: loads of 8 steps
// in flight and 76 registers, for two work-groups per CU (16 steps, 146 registers and one: 32 pairs of 8 chunks 28.5 -> 22.1);
// K = 128, where that spills: one, 126 registers.  (A loop over a run of chunks per wave, for longer sequences: 148, K = V = 128 14.4.)
template <int K, int V>
__global__ __launch_bounds__(3 * NTHR, K == 64 ? 6 : 3) void k_state_fwd_chunks(const lmoe_args a) {
  constexpr int BV = 16, NVS = V / BV, NW = CHUNKS_PREFIX_WAVES, LD = K + 4, HB = K / 64, NK = K / 16, NS = K == 64 ? 4 : 8;
  __shared__ __attribute__((aligned(16))) float s_part[NW][BV * LD];       // S^T of a wave's run [column][K]
  __shared__ __attribute__((aligned(16))) float s_S[BV * LD];
  __shared__ __attribute__((aligned(16))) float s_f[NW + 4][CH];           // per wave: token factors, log-decays
  __shared__ float s_dec[NW];
  const int nch = (a.T + CH - 1) / CH, nit = nch + (a.ht ? 1 : 0), pairs = a.N * a.H;
  // the last chunks, which have most in front of them, first; the slices and chunks of a pair on one XCD where the pairs divide evenly
  int vsl, pair, c;
  if (pairs % 8 == 0) {
    const int j = blockIdx.x >> 3, r = j / NVS;
    vsl = j % NVS; pair = (r % (pairs / 8)) * 8 + (blockIdx.x & 7); c = nit - 1 - r / (pairs / 8);
  } else {
    const int r = blockIdx.x / NVS;
    vsl = blockIdx.x % NVS; pair = r % pairs; c = nit - 1 - r / pairs;
  }
  const int n = pair / a.H, h = pair % a.H, v0 = vsl * BV;
  const int l = lane_id(), fr = l & 15, g = l >> 4, wv = wave_id();
  const bool gated = a.gate != LMOE_GATE_NONE && a.g.ptr != nullptr;
  const float* const kp = row_ptr<float>(a.k, n, 0, h);
  const float* const vp = row_ptr<float>(a.v, n, 0, h) + v0 + fr;
  auto log_decay = [&](int tok, int len) {                                 // of this lane's token of a chunk
    return gated && l < len ? load_scalar(a.g.ptr, a.g_dtype, row_off(a.g, n, tok + min(l, len - 1), h)) : 0.f;
  };

  if (wv < NW) {
    // a thread's four state rows of one column, as they are folded
    const int t = threadIdx.x, col = t / (K / 4), kr = t % (K / 4) * 4;
    f32x4 S = {0.f, 0.f, 0.f, 0.f};
    if (col < BV && a.h0) {
      const float* h0 = a.h0 + ((int64_t)pair * K + kr) * V + v0 + col;
#pragma unroll
      for (int i = 0; i < 4; ++i) S[i] = h0[i * V];
    }
    if (wv < c) {
      f32x4 acc[HB][4];                      // [64-row group][m]: rows 64 hb + 16 g + 4 i + m of column fr
#pragma unroll
      for (int hb = 0; hb < HB; ++hb)
#pragma unroll
        for (int m = 0; m < 4; ++m) acc[hb][m] = f32x4{0.f, 0.f, 0.f, 0.f};
      const int tok = wv * CH, len = min(CH, a.T - tok);
      const float x = wave_incl_scan(log_decay(tok, len)), xl = __shfl(x, 63, 64);
      if (gated) {
        s_f[wv][l] = expf(xl - x);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
      // token 16 g + s of step s (rows past the end of the sequence re-read the last one and count as zero)
#pragma unroll 2
      for (int s0 = 0; s0 < 16; s0 += NS) {
        f32x4 kk[HB][NS];
        float vv[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          const int row = min(16 * g + s0 + s, len - 1);
#pragma unroll
          for (int hb = 0; hb < HB; ++hb) kk[hb][s] = *(const f32x4*)(kp + (int64_t)(tok + row) * a.k.st + 64 * hb + 4 * fr);
          vv[s] = vp[(int64_t)(tok + row) * a.v.st];
        }
        if (len < CH) {
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            const bool in = 16 * g + s0 + s < len;
#pragma unroll
            for (int hb = 0; hb < HB; ++hb)
#pragma unroll
              for (int m = 0; m < 4; ++m) kk[hb][s][m] = in ? kk[hb][s][m] : 0.f;
            vv[s] = in ? vv[s] : 0.f;
          }
        }
        if (gated) {
#pragma unroll
          for (int s = 0; s < NS; s += 4) {
            const f32x4 f = *(const f32x4*)&s_f[wv][16 * g + s0 + s];
#pragma unroll
            for (int i = 0; i < 4; ++i) vv[s + i] *= f[i];
          }
        }
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
          for (int hb = 0; hb < HB; ++hb)
#pragma unroll
            for (int m = 0; m < 4; ++m) acc[hb][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[hb][s][m], vv[s], acc[hb][m], 0, 0, 0);
      }
#pragma unroll
      for (int hb = 0; hb < HB; ++hb)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          *(f32x4*)&s_part[wv][fr * LD + 64 * hb + 16 * g + 4 * i] = f32x4{acc[hb][0][i], acc[hb][1][i], acc[hb][2][i], acc[hb][3][i]};
      if (l == 0) s_dec[wv] = gated ? expf(xl) : 1.f;
    }
    lds_barrier();
    if (col < BV) {
      for (int w = 0; w < c; ++w) S = S * s_dec[w] + *(const f32x4*)&s_part[w][col * LD + kr];
      if (c < nch) {
        *(f32x4*)&s_S[col * LD + kr] = S;
        if (a.hs) *(f32x4*)((float*)a.hs + (((int64_t)(n * nch + c) * a.H + h) * V + v0 + col) * K + kr) = S;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) a.ht[((int64_t)pair * K + kr + i) * V + v0 + col] = S[i];
      }
    }
    lds_barrier();
    return;
  }

  // ------------------------- output rows 16 w .. of the chunk -------------------------
  const int w = wv - NW, tok = c * CH, len = min(CH, a.T - tok);
  f32x4 o = {0.f, 0.f, 0.f, 0.f}, q4[NK];
  const bool busy = 16 * w < len;            // (behind the last chunk: len <= 0)
  if (busy) {
    const float* qr = row_ptr<float>(a.q, n, tok + min(16 * w + fr, len - 1), h) + 4 * g;
#pragma unroll
    for (int s = 0; s < NK; ++s) q4[s] = *(const f32x4*)(qr + 16 * s);
    struct Rows { f32x4 k[NK]; float v[4]; } rows[2];
    auto issue = [&](Rows& r, int tj) {
      const float* kr = kp + (int64_t)(tok + min(16 * tj + fr, len - 1)) * a.k.st + 4 * g;
#pragma unroll
      for (int s = 0; s < NK; ++s) r.k[s] = *(const f32x4*)(kr + 16 * s);
#pragma unroll
      for (int e = 0; e < 4; ++e) r.v[e] = vp[(int64_t)(tok + min(16 * tj + 4 * g + e, len - 1)) * a.v.st];
    };
    issue(rows[0], 0);
    const float b = wave_incl_scan(log_decay(tok, len));
    float bi = 0.f;
    if (gated) {
      s_f[wv][l] = b;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      bi = s_f[wv][16 * w + fr];
    }
    // P^T blocks (tokens 16 tj .. x rows 16 w ..): a lane holds P[row fr][16 tj + 4 g + e], which is the operand of P v.  The
    // rows of the next block are requested ahead of the products of this one
#pragma unroll
    for (int tj = 0; tj < 4; ++tj) {
      if (tj > w) break;
      const Rows& r = rows[tj & 1];
      if (tj < 3) issue(rows[(tj + 1) & 1], min(tj + 1, w));
      f32x4 p = {0.f, 0.f, 0.f, 0.f}, bj = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < NK; ++s)
#pragma unroll
        for (int e = 0; e < 4; ++e) p = __builtin_amdgcn_mfma_f32_16x16x4f32(r.k[s][e], q4[s][e], p, 0, 0, 0);
      if (gated) bj = *(const f32x4*)&s_f[wv][16 * tj + 4 * g];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int jt = 16 * tj + 4 * g + e;
        float x = gated ? p[e] * expf(bi - bj[e]) : p[e];
        x = 16 * w + fr >= jt ? x : 0.f;
        o = __builtin_amdgcn_mfma_f32_16x16x4f32(x, jt < len ? r.v[e] : 0.f, o, 0, 0, 0);
      }
    }
  }
  lds_barrier();
  lds_barrier();
  if (busy) {
    f32x4 oS = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NK; ++s) {
      const f32x4 S = *(const f32x4*)&s_S[fr * LD + 16 * s + 4 * g];
#pragma unroll
      for (int e = 0; e < 4; ++e) oS = __builtin_amdgcn_mfma_f32_16x16x4f32(q4[s][e], S[e], oS, 0, 0, 0);
    }
    f32x4 eb = {1.f, 1.f, 1.f, 1.f};
    if (gated) {
      const f32x4 b = *(const f32x4*)&s_f[wv][16 * w + 4 * g];
#pragma unroll
      for (int e = 0; e < 4; ++e) eb[e] = expf(b[e]);
    }
    float* op = row_ptr<float>(a.o, n, tok, h) + v0 + fr;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 16 * w + 4 * g + e;
      if (row < len) op[(int64_t)row * a.o.st] = a.scale * (eb[e] * oS[e] + o[e]);
    }
  }
}

}  // namespace lmoe
