// Index tables formed on the device in a few launches: the chunk tables of packed input, and the routing tables of a
// mixture-of-memories layer.  Both are small integer work between the products: what they cost is launches.
#include "lmoe_launch.hpp"
#include "lmoe_seq.hpp"

namespace lmoe {

__device__ __forceinline__ int64_t load_index(const void* p, int is64, int64_t i) {
  return is64 ? ((const int64_t*)p)[i] : (int64_t)((const int32_t*)p)[i];
}

// Exclusive prefix sums of x[0 .. n) in LDS, in place, x[n] = total: PER consecutive entries per thread, the thread
// totals scanned inside a wave and the wave totals by every thread for itself.  All threads of the work-group call it;
// it begins and ends with a barrier.
template <int NT_, int PER>
__device__ __forceinline__ void block_exclusive_scan(int* x, int n, int* s_wave) {
  constexpr int NW = NT_ / 64;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  __syncthreads();
  int own[PER], sum = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int j = t * PER + i;
    own[i] = j < n ? x[j] : 0;
    sum += own[i];
  }
  int incl = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int y = __shfl_up(incl, d, 64);
    if (lane >= d) incl += y;
  }
  if (lane == 63) s_wave[wv] = incl;
  __syncthreads();
  int base = incl - sum, total = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    if (w < wv) base += s_wave[w];
    total += s_wave[w];
  }
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int j = t * PER + i;
    if (j < n) x[j] = base;
    base += own[i];
  }
  if (t == 0) x[n] = total;
  __syncthreads();
}

// ------------------------------------------------------------------------- //
// Chunk tables of packed input.  One launch: every work-group forms the chunk counts of all sequences and their prefix
// sums in LDS for itself (N <= SEQ_TABLES_MAX entries out of the L2) and fills its share of the chunk map (the sequence
// of a chunk by bisection) and of the order of the sequences (rank = how many are longer, or as long and earlier).
// Bound by its launch: 4.6 us at N = 8, T = 8192, in place of about twenty small tensor operations per new batch of
// offsets (with the routing tables below 197 us of kernels, now 20; the step around both 880 -> 448 us).  Above SEQ_TABLES_MAX sequences (32 KB of LDS, N^2 comparisons) the caller sorts.
// ------------------------------------------------------------------------- //
__global__ __launch_bounds__(NTHR) void k_seq_tables(const void* __restrict__ offs, int is64, int N, int nt_max,
                                                     int32_t* __restrict__ cu, int32_t* __restrict__ chunk_map,
                                                     int32_t* __restrict__ seq_chunk0, int32_t* __restrict__ nt_dev,
                                                     int32_t* __restrict__ seq_order) {
  constexpr int PER = SEQ_TABLES_MAX / NTHR;
  __shared__ __attribute__((aligned(16))) int s_n[SEQ_TABLES_MAX];
  __shared__ int s_c0[SEQ_TABLES_MAX + 1];
  __shared__ int s_wave[NTHR / 64];
  const int t = threadIdx.x;
  for (int i = t; i < N; i += NTHR) {
    const int64_t len = load_index(offs, is64, i + 1) - load_index(offs, is64, i);
    const int n = len > 0 ? (int)((len + CH - 1) / CH) : 0;
    s_n[i] = n;
    s_c0[i] = n;
  }
  block_exclusive_scan<NTHR, PER>(s_c0, N, s_wave);
  const int gid = blockIdx.x * NTHR + t, gsize = gridDim.x * NTHR;
  for (int i = gid; i <= N; i += gsize) {
    cu[i] = (int32_t)load_index(offs, is64, i);
    seq_chunk0[i] = s_c0[i];
  }
  if (gid == 0) nt_dev[0] = s_c0[N];
  for (int c = gid; c < nt_max; c += gsize) {
    int lo = 0, hi = N;                       // the last entry of s_c0[0 .. N] that is <= c (rows past the count: N)
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (s_c0[mid] <= c) lo = mid; else hi = mid - 1;
    }
    chunk_map[2 * c] = lo;
    chunk_map[2 * c + 1] = c - s_c0[lo];
  }
  if (seq_order) {
    for (int i = gid; i < N; i += gsize) {
      const int own = s_n[i];
      int rank = 0;
      for (int j = 0; j < N; ++j) rank += (s_n[j] > own || (s_n[j] == own && j < i)) ? 1 : 0;
      seq_order[rank] = i;
    }
  }
}

void launch_seq_tables(const void* offs, int is64, int N, int nt_max, int32_t* cu, int32_t* chunk_map,
                       int32_t* seq_chunk0, int32_t* nt_dev, int32_t* seq_order, hipStream_t st) {
  const int want = ((nt_max > N ? nt_max : N) + NTHR) / NTHR;
  const int grid = want < 64 ? want : 64;
  hipLaunchKernelGGL(k_seq_tables, dim3(grid), dim3(NTHR), 0, st, offs, is64, N, nt_max, cu, chunk_map, seq_chunk0, nt_dev,
                     seq_order);
}

// ------------------------------------------------------------------------- //
// Routing tables of a mixture-of-memories layer: a stable counting sort of the choices (b, t, k) by (memory, batch row),
// in three launches (few choices: one, k_mom_route below).  The choices of a batch row are one contiguous range, cut into segments; counts[(e B + b)
// nseg + s] then lies in the order of the result, and its prefix sums are where every (memory, row, segment) begins.
//   count: choices per memory of a segment
//   scan:  prefix sums (one work-group), the capacity, offsets of the sequences; counts -> first row of a segment, less
//          the rows its sequence drops: a choice whose row then lies before the first row of its sequence is dropped
//   place: rows of the choices, in order: a wave walks a quarter of the segment 64 choices at a time, choices of the
//          same memory find each other by ballots over the bits of the memory index
// Bound by the launches and the serial scan: 2 x 2048 tokens, 4 memories, top 2: 3.4 + 7.2 + 4.6 us, in place of a
// stable radix sort and about 25 small tensor operations.
// Memory indices outside [0, E) are dropped; rows no choice fills (there are some only then, or with a capacity) get -1.
// ------------------------------------------------------------------------- //
// Choices of a batch row per work-group of count and place: the wave that ranks them takes them 64 at a time, so short
// segments first (512 against 2048 on 2 x 2048 tokens, top 2: 8 against 15 us of both); long ones where the table of counts
// would not fit the scan's work-group.
constexpr int MOM_SEG_SHORT = 512, MOM_SEG_LONG = 2048;
constexpr int MOM_SCAN_THR = 1024;
constexpr int MOM_SCAN_MAX = 8192;             // entries of counts (32 KB of LDS twice in the scan)
constexpr int MOM_E_MAX = 1024;

__device__ __forceinline__ int memory_of(const void* sel, int is64, int64_t i, int E) {
  const int64_t m = load_index(sel, is64, i);
  return m >= 0 && m < E ? (int)m : E;
}

// lanes of the wave that hold the same key (all 64 lanes call it)
__device__ __forceinline__ uint64_t same_key_lanes(int key, int bits) {
  uint64_t m = ~0ull;
  for (int b = 0; b < bits; ++b) {
    const uint64_t set = __ballot((key >> b) & 1);
    m &= ((key >> b) & 1) ? set : ~set;
  }
  return m;
}

__global__ __launch_bounds__(NTHR) void k_mom_count(const void* __restrict__ sel, int is64, int per_row, int E, int nseg, int seg,
                                                    int32_t* __restrict__ counts) {
  __shared__ int s_n[MOM_E_MAX + 1];
  const int s = blockIdx.x, b = blockIdx.y, B = gridDim.y;
  for (int e = threadIdx.x; e <= E; e += NTHR) s_n[e] = 0;
  __syncthreads();
  const int i1 = min((s + 1) * seg, per_row);
  for (int i = s * seg + threadIdx.x; i < i1; i += NTHR)
    atomicAdd(&s_n[memory_of(sel, is64, (int64_t)b * per_row + i, E)], 1);
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += NTHR) counts[((int64_t)e * B + b) * nseg + s] = s_n[e];
}

__global__ __launch_bounds__(MOM_SCAN_THR) void k_mom_scan(int B, int E, int nseg, int cap, int32_t* __restrict__ counts,
                                                           int32_t* __restrict__ cu, int64_t* __restrict__ max_len,
                                                           int64_t* __restrict__ mem_offsets) {
  constexpr int PER = MOM_SCAN_MAX / MOM_SCAN_THR;
  __shared__ int s_ex[MOM_SCAN_MAX + 1], s_cu[MOM_SCAN_MAX + 1], s_wave[MOM_SCAN_THR / 64], s_longest;
  const int t = threadIdx.x, NS = E * B, M = NS * nseg;
  for (int i = t; i < M; i += MOM_SCAN_THR) s_ex[i] = counts[i];
  if (t == 0) s_longest = 0;
  block_exclusive_scan<MOM_SCAN_THR, PER>(s_ex, M, s_wave);
  int longest = 0;
  for (int i = t; i < NS; i += MOM_SCAN_THR) longest = max(longest, s_ex[(i + 1) * nseg] - s_ex[i * nseg]);
  atomicMax(&s_longest, longest);
  __syncthreads();
  const int kept_max = cap < 0 ? s_longest : min(s_longest, cap);
  for (int i = t; i < NS; i += MOM_SCAN_THR) s_cu[i] = min(s_ex[(i + 1) * nseg] - s_ex[i * nseg], kept_max);
  block_exclusive_scan<MOM_SCAN_THR, PER>(s_cu, NS, s_wave);
  for (int i = t; i <= NS; i += MOM_SCAN_THR) {
    cu[i] = s_cu[i];
    if (i % B == 0) mem_offsets[i / B] = s_cu[i];
  }
  if (t == 0) max_len[0] = kept_max;
  for (int i = t; i < M; i += MOM_SCAN_THR) {
    const int q = i / nseg, len = s_ex[(q + 1) * nseg] - s_ex[q * nseg];
    counts[i] = s_cu[q] + (s_ex[i] - s_ex[q * nseg]) - (len - min(len, kept_max));
  }
}

__global__ __launch_bounds__(NTHR) void k_mom_place(const void* __restrict__ sel, int is64, int per_row, int topk, int E,
                                                    int nseg, int seg, int bits, const int32_t* __restrict__ first,
                                                    const int32_t* __restrict__ cu, int32_t* __restrict__ src_token,
                                                    int32_t* __restrict__ src_choice, int32_t* __restrict__ row_of) {
  constexpr int NW = NTHR / 64;
  __shared__ int s_run[NW][MOM_E_MAX + 1];     // per wave: choices of a memory (first walk), next row (second walk)
  const int s = blockIdx.x, b = blockIdx.y, B = gridDim.y;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (int i = threadIdx.x; i < NW * (MOM_E_MAX + 1); i += NTHR) (&s_run[0][0])[i] = 0;
  __syncthreads();
  const int64_t row0 = (int64_t)b * per_row;
  const int sub = seg / NW, i0 = s * seg + wv * sub, i1 = min(i0 + sub, per_row);
  for (int i = i0 + lane; i < i1; i += 64) atomicAdd(&s_run[wv][memory_of(sel, is64, row0 + i, E)], 1);
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += NTHR) {
    int at = first[((int64_t)e * B + b) * nseg + s];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const int n = s_run[w][e];
      s_run[w][e] = at;
      at += n;
    }
  }
  __syncthreads();
  volatile int* run = s_run[wv];
  for (int i = i0; i < i1; i += 64) {          // (uniform for the wave; lanes past the end carry the key "none")
    const bool valid = i + lane < i1;
    const int e = valid ? memory_of(sel, is64, row0 + i + lane, E) : E;
    const uint64_t same = same_key_lanes(e, bits);
    const int rank = __popcll(same & ((1ull << lane) - 1));
    const int base = run[e];
    __builtin_amdgcn_wave_barrier();
    if (e < E && rank == 0) run[e] = base + __popcll(same);
    __builtin_amdgcn_wave_barrier();
    if (valid) {
      const int64_t c = row0 + i + lane;
      int row = base + rank;
      if (e == E || row < cu[e * B + b]) row = -1;
      row_of[c] = row;
      if (row >= 0) {
        src_choice[row] = (int32_t)c;
        src_token[row] = (int32_t)(c / topk);
      }
    }
  }
  const int64_t n = (int64_t)B * per_row, step = (int64_t)gridDim.x * B * NTHR;
  for (int64_t r = cu[E * B] + ((int64_t)b * gridDim.x + s) * NTHR + threadIdx.x; r < n; r += step) {
    src_choice[r] = -1;
    src_token[r] = -1;
  }
}

// The three steps in one launch, for few choices and up to 16 memories (mom_route_takes): every work-group counts the choices of
// all segments for itself (out of the L2, a wave 64 at a time; lane e keeps the count of memory e from the ballots), its first
// wave forms the prefix sums, and it places its own segment, a wave per 64 choices.  Nothing is handed from one launch to the next.
// Bound by its launch, three round trips to memory and the counting, 64 choices in some 4 E + 16 instructions of a wave.
// 2 x 2048 tokens, 4 memories, top 2: 13.4 us in three launches -> 7.7 (replayed as a graph; traced 3.2 + 7.1 + 4.6 -> 9.5; with
// the prefix sums over the whole work-group, as in k_mom_scan, 12.0); 128 tokens, top 1: 12.0 -> 4.2.  Three launches take 13.4
// to 14.2 whatever the sizes: 8192 choices of 16 memories 12.8 here, 16384 of 8 15.3, 32768 of 4 19.9 and of 16 40.
constexpr int ROUTE_THR = 1024, ROUTE_SEG = 512, ROUTE_E = 16, ROUTE_MAX = 1024, ROUTE_WORK = 131072;
static bool mom_route_takes(int64_t B, int64_t per_row, int64_t E) {
  return E <= ROUTE_E && B * per_row * (E + 4) <= ROUTE_WORK && B * E * ((per_row + ROUTE_SEG - 1) / ROUTE_SEG) <= ROUTE_MAX;
}
// Exclusive prefix sums of x[0 .. n) in place, x[n] = total, by one wave: ROUTE_MAX / 64 consecutive entries per lane
__device__ __forceinline__ void wave_exclusive_scan(int* x, int n, int lane) {
  const int per = (n + 63) / 64, j0 = lane * per;
  int sum = 0;
  for (int i = j0; i < min(j0 + per, n); ++i) sum += x[i];
  int incl = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int y = __shfl_up(incl, d, 64);
    if (lane >= d) incl += y;
  }
  int base = incl - sum;
  for (int i = j0; i < min(j0 + per, n); ++i) {
    const int y = x[i];
    x[i] = base;
    base += y;
  }
  if (lane == 63) x[n] = incl;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__global__ __launch_bounds__(ROUTE_THR) void k_mom_route(const void* __restrict__ sel, int is64, int per_row, int topk, int E, int cap,
                                                         int32_t* __restrict__ cu, int64_t* __restrict__ max_len,
                                                         int64_t* __restrict__ mem_offsets, int32_t* __restrict__ src_token,
                                                         int32_t* __restrict__ src_choice, int32_t* __restrict__ row_of) {
  constexpr int NW = ROUTE_THR / 64, GROUPS = ROUTE_SEG / 64, STEP = NW / GROUPS, AHEAD = 4;
  __shared__ int s_ex[ROUTE_MAX + 1], s_cu[ROUTE_MAX + 1], s_grp[GROUPS][ROUTE_E], s_kept;
  const int s = blockIdx.x, b = blockIdx.y, nseg = gridDim.x, B = gridDim.y;
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6), NS = E * B, M = NS * nseg;
  // this wave's 64 choices of its own segment (waves beyond the segment's: none)
  const int i_own = s * ROUTE_SEG + wv * 64 + lane;
  const bool valid = wv < GROUPS && i_own < per_row;
  const int64_t c = (int64_t)b * per_row + i_own;
  const int e_own = valid ? memory_of(sel, is64, c, E) : E;
  for (int i = t; i < M; i += ROUTE_THR) s_ex[i] = 0;
  __syncthreads();
  // 64 choices, number wv % GROUPS, of every STEP-th segment (segments of all rows in order); a few segments' loads at a time
  int row = 0, seg = wv / GROUPS;
  while (row < B) {
    int key[AHEAD], at[AHEAD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      while (seg >= nseg) { seg -= nseg; ++row; }
      const int i = seg * ROUTE_SEG + (wv % GROUPS) * 64 + lane;
      at[u] = row < B ? row * nseg + seg : -1;
      key[u] = row < B && i < per_row ? memory_of(sel, is64, (int64_t)row * per_row + i, E) : E;
      seg += STEP;
    }
    while (seg >= nseg) { seg -= nseg; ++row; }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      if (at[u] < 0) break;
      int own = 0;
      for (int e = 0; e < E; ++e) {
        const int n = __popcll(__ballot(key[u] == e));
        own = lane == e ? n : own;
      }
      if (lane < E) {
        const int r = at[u] / nseg;
        if (own) atomicAdd(&s_ex[(lane * B + r) * nseg + at[u] - r * nseg], own);
        if (at[u] == b * nseg + s) s_grp[wv % GROUPS][lane] = own;
      }
    }
  }
  __syncthreads();
  // prefix sums and the capacity, as in k_mom_scan
  if (wv == 0) {
    wave_exclusive_scan(s_ex, M, lane);
    int kept = 0;
    for (int i = lane; i < NS; i += 64) kept = max(kept, s_ex[(i + 1) * nseg] - s_ex[i * nseg]);
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) kept = max(kept, __shfl_xor(kept, d, 64));
    if (cap >= 0) kept = min(kept, cap);
    for (int i = lane; i < NS; i += 64) s_cu[i] = min(s_ex[(i + 1) * nseg] - s_ex[i * nseg], kept);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    wave_exclusive_scan(s_cu, NS, lane);
    if (lane == 0) s_kept = kept;
  }
  __syncthreads();
  if (s == 0 && b == 0) {
    for (int i = t; i <= NS; i += ROUTE_THR) {
      cu[i] = s_cu[i];
      if (i % B == 0) mem_offsets[i / B] = s_cu[i];
    }
    if (t == 0) max_len[0] = s_kept;
  }
  if (wv < GROUPS) {
    int bits = 1;
    while ((E >> bits) != 0) ++bits;           // the keys are 0 .. E
    const int rank = __popcll(same_key_lanes(e_own, bits) & ((1ull << lane) - 1));
    int at = -1;
    if (e_own < E) {
      const int q = e_own * B + b, q0 = s_ex[q * nseg], len = s_ex[(q + 1) * nseg] - q0;
      at = s_cu[q] + (s_ex[q * nseg + s] - q0) - (len - min(len, s_kept)) + rank;
      for (int g = 0; g < wv; ++g) at += s_grp[g][e_own];
      if (at < s_cu[q]) at = -1;               // (dropped by the capacity)
    }
    if (valid) {
      row_of[c] = at;
      if (at >= 0) {
        src_choice[at] = (int32_t)c;
        src_token[at] = (int32_t)c / topk;
      }
    }
  }
  const int64_t n = (int64_t)B * per_row, step = (int64_t)nseg * B * ROUTE_THR;
  for (int64_t r = s_cu[NS] + ((int64_t)b * nseg + s) * ROUTE_THR + t; r < n; r += step) {
    src_choice[r] = -1;
    src_token[r] = -1;
  }
}

static int64_t mom_segments(int64_t per_row, int seg) { return (per_row + seg - 1) / seg; }
static int mom_seg(int64_t B, int64_t per_row, int64_t E) {
  return B * E * mom_segments(per_row, MOM_SEG_SHORT) <= MOM_SCAN_MAX ? MOM_SEG_SHORT : MOM_SEG_LONG;
}

int64_t mom_plan_ints(int64_t B, int64_t per_row, int64_t E) {
  if (B <= 0 || per_row <= 0 || E <= 0 || E > MOM_E_MAX || B > 65535) return 0;
  if (B * per_row > 0x7fffffff) return 0;
  const int64_t m = B * E * mom_segments(per_row, mom_seg(B, per_row, E));
  return m <= MOM_SCAN_MAX ? m : 0;
}

void launch_mom_plan(const void* sel, int is64, int B, int per_row, int topk, int E, int cap, int32_t* counts, int32_t* cu,
                     int64_t* max_len, int64_t* mem_offsets, int32_t* src_token, int32_t* src_choice, int32_t* row_of,
                     hipStream_t st) {
  if (mom_route_takes(B, per_row, E)) {
    hipLaunchKernelGGL(k_mom_route, dim3((int)mom_segments(per_row, ROUTE_SEG), B), dim3(ROUTE_THR), 0, st, sel, is64, per_row, topk, E, cap,
                       cu, max_len, mem_offsets, src_token, src_choice, row_of);
    return;
  }
  const int seg = mom_seg(B, per_row, E), nseg = (int)mom_segments(per_row, seg);
  int bits = 1;
  while ((E >> bits) != 0) ++bits;             // the keys are 0 .. E
  hipLaunchKernelGGL(k_mom_count, dim3(nseg, B), dim3(NTHR), 0, st, sel, is64, per_row, E, nseg, seg, counts);
  hipLaunchKernelGGL(k_mom_scan, dim3(1), dim3(MOM_SCAN_THR), 0, st, B, E, nseg, cap, counts, cu, max_len, mem_offsets);
  hipLaunchKernelGGL(k_mom_place, dim3(nseg, B), dim3(NTHR), 0, st, sel, is64, per_row, topk, E, nseg, seg, bits, counts, cu,
                     src_token, src_choice, row_of);
}

}  // namespace lmoe
