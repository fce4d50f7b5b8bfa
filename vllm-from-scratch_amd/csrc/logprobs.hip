// Speculative logprobs: for every output position of a verification step, the log-softmax
// (or the logits themselves) of the row that position was sampled from, its top-k and the
// sampled token's logprob and rank (minivllm/sample/rejection_sampler.py:229-300 with
// Sampler.compute_logprobs / gather_logprobs / batched_count_greater_than,
// minivllm/sample/sampler.py:313-349).
//
// Position (r, j) of request r (j <= max_spec_len) reads compact row start_r + j (clamped to
// the last row), where the compact rows are each request's K_r verify rows followed by its
// bonus row and start_r is the request's first compact row.  A verify row comes from `target`
// (through target_rows when given), a bonus row from `bonus`.  Placeholder ids (-1) read
// token 0.  Per row:
//   lp(x) = (x - M) - log(sum exp(x - M))   (log-softmax, fp32)   or   lp(x) = x  (logits mode)
//   out[0] = (token, lp(x_token)), out[1 .. k] = top-k of lp by (value desc, index asc),
//   rank = #{i : lp(x_i) >= lp(x_token)}.
//
// Two paths, the same results:
//   split     (a workspace, k <= 128, rows long enough for k): lp_scan_kernel reads each position's row once, split into
//             chunks over workgroups; lp_finish_kernel, one workgroup per position, combines the
//             chunks and finds the top-k in the few places that can hold it.
//   lists     (any k, no workspace): spec_logprobs_kernel, one 512-thread workgroup per position:
//             pass 1 reduces (M, S); pass 2 keeps per-thread lists of the KMAX largest
//             (value, index) keys, counts the rank, then merges the lists per wave and across
//             waves by rounds of key maxima.  For k > KMAX, pass 2 repeats over the keys below
//             the last one found, KMAX at a time (ceil(k / 32) passes for k > 8).
#include "logprobs.h"
#include "mvsd_device.h"

namespace mvsd {

constexpr int kLpThreads = 512;
constexpr int kLpWaves = kLpThreads / kWave;

__device__ inline uint64_t umax_key(uint64_t a, uint64_t b) { return a > b ? a : b; }

// ------------------------------------------------------------------ positions --------

// The row and the token of position n.
template <typename S>
struct Position {
  const S* row;
  int token;
};

__device__ inline int64_t token_at(const LogprobParams& p, int64_t i) {
  return p.tokens64 ? static_cast<const int64_t*>(p.tokens)[i]
                    : (int64_t) static_cast<const int32_t*>(p.tokens)[i];
}

__device__ inline int64_t row_inside(int64_t row, int64_t num_rows) {
  return num_rows > 0 ? min(max(row, (int64_t)0), num_rows - 1) : row;
}

template <typename S>
__device__ inline Position<S> position(const LogprobParams& p, int n) {
  Position<S> at;
  int64_t token;
  if (p.flat) {
    at.row = static_cast<const S*>(p.bonus) + (int64_t)n * p.bstride;
    token = token_at(p, n);
  } else {
    const int r = n / p.W, j = n - r * p.W;
    const int start = r == 0 ? 0 : p.cu_sampled[r - 1];
    token = token_at(p, (int64_t)r * p.tok_stride + j);
    const int c = min(start + j, p.P + p.B - 1);
    // request owning compact row c: r itself for its own rows, else (padding positions) the
    // first q with cu_sampled[q] > c
    int q = r;
    if (c >= p.cu_sampled[r]) {
      int lo = r, hi = p.B - 1;
      while (lo < hi) {
        const int mid = (lo + hi) / 2;
        if (p.cu_sampled[mid] > c) hi = mid;
        else lo = mid + 1;
      }
      q = lo;
    } else if (c < start) {  // the clamped row of a request past the last one
      int lo = 0, hi = r;
      while (lo < hi) {
        const int mid = (lo + hi) / 2;
        if (p.cu_sampled[mid] > c) hi = mid;
        else lo = mid + 1;
      }
      q = lo;
    }
    const int qstart = q == 0 ? 0 : p.cu_sampled[q - 1];
    const int kq = p.cu_sampled[q] - qstart - 1;  // verify rows of request q
    if (c - qstart < kq && p.P > 0) {
      // verify rows before c: c minus the bonus rows of requests < q (in bounds whatever
      // cu_sampled holds)
      const int vrow = min(max(c - q, 0), p.P - 1);
      const int64_t trow =
          row_inside(p.target_rows ? p.target_rows[vrow] : vrow, p.target_num_rows);
      at.row = static_cast<const S*>(p.target) + trow * p.tstride;
    } else {
      const int64_t brow = row_inside(p.bonus_rows ? p.bonus_rows[q] : q, p.bonus_num_rows);
      at.row = static_cast<const S*>(p.bonus) + brow * p.bstride;
    }
  }
  at.token = token == -1 ? 0 : (int)min(max(token, (int64_t)0), (int64_t)p.V - 1);
  return at;
}

__device__ inline void put_id(const LogprobParams& p, int64_t at, int id) {
  if (p.ids64) static_cast<int64_t*>(p.ids)[at] = id;
  else static_cast<int32_t*>(p.ids)[at] = id;
}

__device__ inline void put_rank(const LogprobParams& p, int64_t at, int rank) {
  if (p.ids64) static_cast<int64_t*>(p.ranks)[at] = rank;
  else static_cast<int32_t*>(p.ranks)[at] = rank;
}

// ------------------------------------------------------------------ lists ------------

template <int KMAX, int NW>
struct ListSmem {
  uint64_t cand[NW * KMAX];
  uint64_t bound;
};

// The k largest (value(i), i) of i in [0, V) by (value desc, index asc), as emit(slot, index)
// in that order; visit(v) is called once for every value.  Round t collects the next
// min(KMAX, k - done) largest keys strictly below the last key of round t - 1; keys are
// distinct (the index is in the low word), so the rounds partition the top-k exactly.
template <int KMAX, int NW, typename At, typename Visit, typename Emit>
__device__ inline void topk_by_lists(int V, int k, ListSmem<KMAX, NW>& sm, At&& value,
                                     Visit&& visit, Emit&& emit) {
  const int tid = threadIdx.x, lane = lane_id(), wid = wave_id();
  uint64_t bound = ~0ull;
  int done = 0;
  bool first_pass = true;
  while (first_pass || done < k) {
    const int need = min(KMAX, k - done);
    uint64_t key[KMAX];
#pragma unroll
    for (int i = 0; i < KMAX; ++i) key[i] = 0;
    for (int i = tid; i < V; i += NW * kWave) {
      const float v = value(i);
      if (first_pass) visit(v);
      uint64_t kk = argmax_key(v, i);
      if (kk < bound && kk > key[KMAX - 1]) {
        // insertion into the descending list (one compare-exchange step per slot)
#pragma unroll
        for (int s2 = 0; s2 < KMAX; ++s2) {
          const uint64_t a = key[s2];
          const bool sw = kk > a;
          key[s2] = sw ? kk : a;
          kk = sw ? a : kk;
        }
      }
    }
    // per-wave merge: `need` rounds, the lane holding the largest head pops it
    for (int round = 0; round < need; ++round) {
      const uint64_t best = wave_max_u64(key[0]);
      if (lane == 0) sm.cand[wid * KMAX + round] = best;
      if (key[0] == best && best != 0) {
#pragma unroll
        for (int s2 = 0; s2 + 1 < KMAX; ++s2) key[s2] = key[s2 + 1];
        key[KMAX - 1] = 0;
      }
    }
    __syncthreads();
    // block merge by wave 0: lanes hold the waves' sorted candidate lists
    if (wid == 0) {
      constexpr int PER = (NW * KMAX + kWave - 1) / kWave;
      uint64_t cand[PER];
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int ci = lane * PER + i;
        cand[i] = ci < NW * KMAX && (ci % KMAX) < need ? sm.cand[ci] : 0;
      }
      // sort each lane's few candidates (descending)
#pragma unroll
      for (int a = 0; a < PER; ++a)
#pragma unroll
        for (int b = a + 1; b < PER; ++b) {
          const uint64_t hi2 = umax_key(cand[a], cand[b]);
          const uint64_t lo2 = cand[a] ^ cand[b] ^ hi2;
          cand[a] = hi2;
          cand[b] = lo2;
        }
      uint64_t last = bound;
      for (int round = 0; round < need; ++round) {
        const uint64_t best = wave_max_u64(cand[0]);
        if (lane == 0) emit(done + round, min(max(key_index(best), 0), V - 1));
        last = best;
        if (cand[0] == best && best != 0) {
#pragma unroll
          for (int s2 = 0; s2 + 1 < PER; ++s2) cand[s2] = cand[s2 + 1];
          cand[PER - 1] = 0;
        }
      }
      if (lane == 0) sm.bound = last;
    }
    __syncthreads();
    bound = sm.bound;
    done += need;
    first_pass = false;
  }
}

template <int KMAX>
__global__ __launch_bounds__(kLpThreads) void spec_logprobs_kernel(LogprobParams p) {
#pragma clang fp contract(off)
  __shared__ float s_m[kLpWaves], s_s[kLpWaves];
  __shared__ ListSmem<KMAX, kLpWaves> s_list;
  __shared__ int s_rank;
  const int tid = threadIdx.x, lane = lane_id(), wid = wave_id();
  const int n = blockIdx.x;  // position r * W + j
  const Position<float> at = position<float>(p, n);
  const float* x = at.row;

  // ---- pass 1: row max and sum of exp(x - max) ----
  if (tid == 0) s_rank = 0;
  float lpm = 0.f, L = 0.f;
  if (!p.logits_mode) {
    float m = -INFINITY, s = 0.f;
    for (int i = tid; i < p.V; i += kLpThreads) {
      const float v = x[i];
      if (v > m) {
        s = s * expf(m - v);
        m = v;
      }
      if (v != -INFINITY) s += expf(v - m);  // masked entries add nothing (and no NaN)
    }
    const float wm = wave_max(m);
    const float ws = wave_sum(m == -INFINITY ? 0.f : s * expf(m - wm));
    if (lane == 0) {
      s_m[wid] = wm;
      s_s[wid] = ws;
    }
    __syncthreads();
    float M = -INFINITY;
    for (int w = 0; w < kLpWaves; ++w) M = fmaxf(M, s_m[w]);
    float S = 0.f;
    for (int w = 0; w < kLpWaves; ++w)
      if (s_m[w] != -INFINITY) S += s_s[w] * expf(s_m[w] - M);
    lpm = M;
    L = logf(S);
  }
  __syncthreads();
  auto lp = [&](float v) { return p.logits_mode ? v : (v - lpm) - L; };
  const float tlp = lp(x[at.token]);
  // the order the top-k and the rank use: the log-softmax, or the raw values
  auto ord = [&](float v) { return p.rank_raw ? v : lp(v); };
  const float tord = ord(x[at.token]);

  // ---- pass 2 (repeated): the top-k lists, and the rank count ----
  const int64_t out = (int64_t)n * (p.k + 1);
  int cnt = 0;
  topk_by_lists<KMAX, kLpWaves>(
      p.V, p.k, s_list, [&](int i) { return ord(x[i]); },
      [&](float v) { cnt += v >= tord ? 1 : 0; },
      [&](int slot, int idx) {
        // the value is recomputed from the index (the key's order bits merge -0.0 and +0.0)
        put_id(p, out + 1 + slot, idx);
        p.lps[out + 1 + slot] = lp(x[idx]);
      });
  for (int off = kWave / 2; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, kWave);
  if (lane == 0) atomicAdd(&s_rank, cnt);
  __syncthreads();
  if (tid == 0) {
    put_id(p, out, at.token);
    p.lps[out] = tlp;
    put_rank(p, n, s_rank);
  }
}

// ------------------------------------------------------------------ split ------------
// lp_scan_kernel, one 256-thread workgroup per (position, chunk of columns): every thread
// holds NV 16-byte vectors of the row, so the row is read once, with all of a workgroup's
// loads in flight together.  It leaves
//   stats[n, c]          the chunk's maximum, sum of exp(x - maximum), number of entries at or
//                        above the token's value, and largest entry below the token's value;
//   group_keys[n, c, g]  the ordered key of the largest entry of group g, the entries held by 16
//                        consecutive lanes (a chunk has 16 groups of 16 * NV * VEC entries).
// lp_finish_kernel, one 256-thread workgroup per position:
//   - M and S from the chunks, hence lp;
//   - the rank: the count of entries x >= x_token, plus, where lp merges values (the largest entry
//     below the token's value has the token's lp), those entries of the chunk counted again;
//   - theta, the k-th largest of the maxima of 256 disjoint unions of groups (64 for k <= 32, found
//     by one wave: a sixteenth of the compares, and a few more candidates): at least k entries
//     reach it, so the top-k are among the entries whose order value reaches theta's, and these lie in
//     the groups whose maximum does (about k of them).  Their entries are gathered into LDS (one
//     float compare passes over the positions where no lane holds a candidate) and ranked by
//     counting.
//   - More candidates than LDS holds: the entries strictly above theta, then as many entries equal
//     to it as are missing, lowest index first; or, if even those above do not fit, the lists.
// What bounds it: the scan is one read of the rows with about 12 VALU operations per entry
// (128 us for 1280 fp32 rows of 151936 columns under the profiler, 6.1 TB/s); the finish is a chain
// of a few small loads and barriers (21 us for those rows, 28 before the 64 unions and the compare;
// 8 us for 32).  The scan's exponentials are exp2 of the rounded product (x - max) log2(e), where the
// lists call expf: against 64 bits the values are as close (the mean error over 60 sets of rows
// 3.95e-8 and 4.38e-8).  The lists path spends about 40
// operations on every entry (64-bit keys, serial insertion) and reads rows twice with 4-byte
// loads: it took 2908 us for those 1280 rows with k = 20 (now 149 us in all), and 236 us for 24
// bf16 rows with k = 5 (now 17 us).

constexpr int kSplitMaxK = 128;       // theta is read off 256 keys
constexpr int kGroupsPerChunk = 16;   // of 16 lanes each
constexpr int kMaxGroups = 4096;      // LDS for the groups of one row
constexpr int kLpCap = 1024;          // gathered candidates
constexpr int kThetaWaveK = 32;       // largest k whose theta is read off 64 keys
constexpr float kLpLog2e = 1.44269504088896340736f;

// Columns per chunk: 8192, or 2048 where rows of 8192-column chunks would leave compute units
// idle (fewer than 4 workgroups each; fp32 rows, k = 20, short / long chunks: 64 rows of 151936 columns
// 19 / 21 us, 1000 rows 127 / 115; of 100000 16 / 18 and 85 / 79; of 50257 13 / 16 and 44 / 50) or give
// fewer than two groups per candidate wanted, so that theta is a poor bound or none: 1000 fp32 rows of 32000 columns took 90 us with long chunks and 45
// with short ones for k = 64 (64 long groups), 1488 and 53 for k = 128; of 65536 columns 70 and 62
// for k = 64 (128 groups, where the two meet).
constexpr int kChunkLong = 8192, kChunkShort = 2048;

// Groups of a row that hold entries (16-bit rows can have a few less in their last chunk).
static int64_t row_groups(int64_t V, int64_t chunk) {
  const int64_t rest = (V % chunk + 63) / 64;
  return V / chunk * kGroupsPerChunk + (rest < kGroupsPerChunk ? rest : kGroupsPerChunk);
}

static int split_chunk(int64_t positions, int64_t V, int64_t k) {
  const int64_t wgs = positions * ((V + kChunkLong - 1) / kChunkLong);
  const int64_t groups_short = (V + kChunkShort - 1) / kChunkShort * kGroupsPerChunk;
  const bool want_short = wgs < 1024 || row_groups(V, kChunkLong) < 2 * k;
  return want_short && groups_short <= kMaxGroups ? kChunkShort : kChunkLong;
}

// Rows too short to give theta (fewer groups than k, and more entries than the candidate buffer)
// end in the lists, by 256 threads after the scan, where the lists kernel has 512 and no scan.  Up
// to one workgroup per compute unit that kernel is the faster one, beyond it the slower (k = 128, V =
// 8000: 181 us against 276 for 256 rows, 349 against 302 for 320; V = 4096: 143 / 164 and 279 / 196).
// With as many groups as k = 128, theta is the least of the groups' maxima, which one row in 25 has
// more than 1024 entries above (V = 16384: 258 us against 522 for 128 rows; below 16 rows most calls
// meet none); a sixteenth more groups are enough (V = 17000: 261 against 37).
constexpr int64_t kListPositions = 256, kFewPositions = 16;
static bool lists_are_faster(int64_t positions, int64_t V, int64_t k) {
  const int64_t need = k <= 96 || positions < kFewPositions ? k : k + k / 16;
  return V > kLpCap && row_groups(V, kChunkShort) < need && positions <= kListPositions;
}

template <int DT, int NV>
__global__ __launch_bounds__(kThreads) void lp_scan_kernel(LogprobParams p) {
  using S = typename Elem<DT>::storage;
  constexpr int VEC = Elem<DT>::kVec;
  constexpr int CH = NV * kThreads * VEC;
  __shared__ float s_m[kWaves], s_s[kWaves], s_prev[kWaves];
  __shared__ int s_cnt[kWaves];
  const int n = blockIdx.x / p.nchunks, c = blockIdx.x - n * p.nchunks;
  const Position<S> at = position<S>(p, n);
  const int tid = threadIdx.x;
  const int c0 = c * CH + tid * VEC;
  float v[NV][VEC];
  const bool full = (c + 1) * CH <= p.V;
  u32x4 q[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j)
    q[j] = load_vec_inside<DT>(at.row, c0 + j * kThreads * VEC, p.V);
#pragma unroll
  for (int j = 0; j < NV; ++j)
#pragma unroll
    for (int e = 0; e < VEC; ++e) v[j][e] = vec_elem<DT>(q[j], e);
  if (!full) {
    // entries outside the vector's own columns (load_vec_inside) count as absent
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int col = c0 + j * kThreads * VEC;
#pragma unroll
      for (int e = 0; e < VEC; ++e)
        v[j][e] = inside_col<DT>(col, e, p.V) < 0 ? -INFINITY : v[j][e];
    }
  }
  const float t = Elem<DT>::cvt(at.row[at.token]);
  float m = -INFINITY, prev = -INFINITY;
  int cnt = 0;  // of the wave
#pragma unroll
  for (int j = 0; j < NV; ++j)
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      m = fmaxf(m, v[j][e]);
      bool ge = v[j][e] >= t;
      prev = fmaxf(prev, v[j][e] < t ? v[j][e] : -INFINITY);
      if (!full) ge = ge & (inside_col<DT>(c0 + j * kThreads * VEC, e, p.V) >= 0);
      cnt += __popcll(__ballot(ge));
    }
  float g = max16(m);
  const float wm = fmaxf(fmaxf(readlane_f32(g, 0), readlane_f32(g, 16)),
                         fmaxf(readlane_f32(g, 32), readlane_f32(g, 48)));
  // sum of exp(x - wave maximum); in logits mode the same sweep only looks for NaN
  float s = 0.f;
  if (p.logits_mode) {
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
      for (int e = 0; e < VEC; ++e) s += v[j][e] != v[j][e] ? NAN : 0.f;
  } else if (wm != -INFINITY) {
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
      for (int e = 0; e < VEC; ++e) s += __builtin_amdgcn_exp2f((v[j][e] - wm) * kLpLog2e);
  } else {  // every entry is -inf or NaN
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
      for (int e = 0; e < VEC; ++e) s += v[j][e] != v[j][e] ? NAN : 0.f;
  }
  s = wave_sum(s);
  uint32_t key = ordered_bits(g);
  if (s != s) {
    // a NaN (or +inf) in the wave: a group with a NaN has the NaN key
    float nan = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
      for (int e = 0; e < VEC; ++e) nan = v[j][e] != v[j][e] ? 1.f : nan;
    if (max16(nan) != 0.f) key = 0xffffffffu;
  }
  const float wprev = wave_max(prev);
  const int64_t slot = (int64_t)n * p.nchunks + c;
  if ((tid & 15) == 0) p.group_keys[slot * kGroupsPerChunk + tid / 16] = key;
  if (lane_id() == 0) {
    s_m[wave_id()] = wm;
    s_s[wave_id()] = s;
    s_prev[wave_id()] = wprev;
    s_cnt[wave_id()] = cnt;
  }
  __syncthreads();
  if (tid == 0) {
    float M = s_m[0], P = s_prev[0], sum = 0.f;
    int count = s_cnt[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) {
      M = fmaxf(M, s_m[w]);
      P = fmaxf(P, s_prev[w]);
      count += s_cnt[w];
    }
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
      sum += s_m[w] == -INFINITY ? s_s[w] : s_s[w] * __builtin_amdgcn_exp2f((s_m[w] - M) * kLpLog2e);
    p.stats[slot] = make_float4(M, sum, __int_as_float(count), P);
  }
}

struct FinishSmem {
  uint64_t cand[kLpCap];
  __align__(16) uint32_t tkey[kThreads];
  __align__(16) uint32_t theta_key[kWave];
  ListSmem<8, kWaves> lists;
  float red[kWaves];
  int wave_cnt[kWaves];
  int groups, count, rank, flagged;
  uint32_t theta;
};

template <int DT, int NV>
__global__ __launch_bounds__(kThreads) void lp_finish_kernel(LogprobParams p) {
#pragma clang fp contract(off)
  using S = typename Elem<DT>::storage;
  constexpr int VEC = Elem<DT>::kVec;
  constexpr int CH = NV * kThreads * VEC;
  __shared__ FinishSmem sm;
  // the row's group keys, then (as 16-bit numbers) the groups whose maximum reaches theta: sized
  // by the launch, so that rows of ordinary length leave room for eight workgroups per CU
  extern __shared__ uint32_t s_group[];
  const int tid = threadIdx.x, lane = lane_id(), wid = wave_id();
  const int n = blockIdx.x, nch = p.nchunks, V = p.V, k = p.k;
  const int ng = nch * kGroupsPerChunk;
  uint16_t* s_glist = reinterpret_cast<uint16_t*>(s_group + ng);
  const uint32_t* gk = p.group_keys + (int64_t)n * ng;
  float4 st = make_float4(-INFINITY, 0.f, 0.f, -INFINITY);
  if (tid < nch) st = p.stats[(int64_t)n * nch + tid];
  uint32_t top = 0;  // the largest of this thread's groups
  for (int g = tid; g < ng; g += kThreads) {
    const uint32_t key = gk[g];
    s_group[g] = key;
    top = max(top, key);
  }
  const Position<S> at = position<S>(p, n);
  const S* x = at.row;
  const float tval = Elem<DT>::cvt(x[at.token]);
  sm.tkey[tid] = top;
  if (tid == 0) {
    sm.groups = sm.count = sm.rank = sm.flagged = 0;
    sm.theta = 0xffffffffu;
  }

  // ---- M, S, the rank of entries at or above the token's value ----
  float lpm = 0.f, L = 0.f;
  if (!p.logits_mode) {
    float M[1] = {st.x};
    block_max<1>(M, sm.red);
    // a chunk of -inf and NaN alone has sum NaN
    float sum[1] = {st.x == -INFINITY ? st.y : st.y * expf(st.x - M[0])};
    block_sum<1>(sum, sm.red);
    lpm = M[0];
    L = logf(sum[0]);
  } else {
    __syncthreads();
  }
  auto lp = [&](float v) { return p.logits_mode ? v : (v - lpm) - L; };
  auto ord = [&](float v) { return p.rank_raw ? v : lp(v); };
  const float tlp = lp(tval), tord = ord(tval);
  {
    int cnt = __float_as_int(st.z);
    for (int off = kWave / 2; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, kWave);
    if (lane == 0) atomicAdd(&sm.rank, cnt);
  }
  // lp can merge values: an entry below the token's value counts when its lp is the token's
  if (!p.rank_raw && !p.logits_mode && st.w > -INFINITY && ord(st.w) >= tord)
    s_glist[atomicAdd(&sm.flagged, 1)] = (uint16_t)tid;
  __syncthreads();
  for (int f = 0; f < sm.flagged; ++f) {  // rare
    const int c = s_glist[f];
    int cnt = 0;
    for (int i = c * CH + tid; i < min(V, (c + 1) * CH); i += kThreads) {
      const float v = Elem<DT>::cvt(x[i]);
      cnt += (v < tval) & (ord(v) >= tord);
    }
    for (int off = kWave / 2; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, kWave);
    if (lane == 0) atomicAdd(&sm.rank, cnt);
  }
  __syncthreads();
  const int64_t out = (int64_t)n * (k + 1);
  if (tid == 0) {
    put_id(p, out, at.token);
    p.lps[out] = tlp;
    put_rank(p, n, tord != tord ? 0 : sm.rank);  // nothing compares >= NaN
  }
  if (k == 0) return;

  // ---- theta: the k-th largest of the 256 threads' keys, or of 64 maxima of four of them ----
  // (fewer than k keys are above the k-th largest, and it is the smallest such key)
  if (k <= kThetaWaveK) {  // block-uniform
    uint32_t own = 0;
    if (wid == 0) {
#pragma unroll
      for (int w = 0; w < kWaves; ++w) own = max(own, sm.tkey[w * kWave + lane]);
      sm.theta_key[lane] = own;
    }
    __syncthreads();
    if (wid == 0) {
      int above = 0;
      const uint4* keys = reinterpret_cast<const uint4*>(sm.theta_key);
#pragma unroll
      for (int j = 0; j < kWave / 4; ++j) {
        const uint4 o = keys[j];
        above += (o.x > own) + (o.y > own) + (o.z > own) + (o.w > own);
      }
      if (above < k) atomicMin(&sm.theta, own);
    }
  } else {
    int above = 0;
    const uint4* keys = reinterpret_cast<const uint4*>(sm.tkey);
#pragma unroll 8
    for (int j = 0; j < kThreads / 4; ++j) {
      const uint4 o = keys[j];
      above += (o.x > top) + (o.y > top) + (o.z > top) + (o.w > top);
    }
    if (above < k) atomicMin(&sm.theta, top);
  }
  __syncthreads();
  // ordered keys of the order values; key 0 (no entry) stays 0
  auto ord_key = [&](float v) { return ordered_bits(ord(v)); };
  auto ord_key_of = [&](uint32_t key) {
    return key == 0 ? 0u : key == 0xffffffffu ? 0xffffffffu : ord_key(key_float(key));
  };
  const uint32_t theta = ord_key_of(sm.theta);
  for (int g = tid; g < ng; g += kThreads)
    if (s_group[g] != 0 && ord_key_of(s_group[g]) >= theta)
      s_glist[atomicAdd(&sm.groups, 1)] = (uint16_t)g;
  __syncthreads();
  const int nl = sm.groups;

  // ---- the entries of those groups whose order value is at or above `floor` ----
  auto gather = [&](uint32_t floor) {
    const float floor_v = key_float(floor);
    for (int b = 0; b < nl; b += kThreads / 16) {
      const int li = b + tid / 16;
      const bool on = li < nl;
      const int g = on ? s_glist[li] : 0;
      // group g holds what lanes 16 (g % 16) .. of chunk g / 16 held in the scan
      const int c0 = (g / kGroupsPerChunk) * CH + ((g % kGroupsPerChunk) * 16 + (tid & 15)) * VEC;
      u32x4 q[NV];
#pragma unroll
      for (int j = 0; j < NV; ++j) q[j] = load_vec_inside<DT>(x, c0 + j * kThreads * VEC, V);
#pragma unroll
      for (int j = 0; j < NV; ++j) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          const float v = vec_elem<DT>(q[j], e);
          // most positions of the group hold no candidate (a NaN on either side goes on)
          if (__ballot(!(ord(v) < floor_v)) == 0) continue;
          const int col = inside_col<DT>(c0 + j * kThreads * VEC, e, V);
          const uint32_t key = ord_key(v);
          const bool take = on && col >= 0 && key >= floor;
          const uint64_t mask = __ballot(take);
          if (mask == 0) continue;
          const int leader = __ffsll((long long)mask) - 1;
          int base = 0;
          if (lane == leader) base = atomicAdd(&sm.count, __popcll(mask));
          base = __shfl(base, leader);
          const int pos = base + __popcll(mask & ((1ull << lane) - 1ull));
          if (take && pos < kLpCap)
            sm.cand[pos] = ((uint64_t)key << 32) | (uint64_t)(0xffffffffu - (uint32_t)col);
        }
      }
    }
    __syncthreads();
  };
  auto emit = [&](int slot, int idx) {
    // the value is recomputed from the index (the key's order bits merge -0.0 and +0.0)
    put_id(p, out + 1 + slot, idx);
    p.lps[out + 1 + slot] = lp(Elem<DT>::cvt(x[idx]));
  };
  // writes the gathered candidates of rank below k, counting the larger keys
  auto write_ranked = [&](int m) {
    for (int i = tid; i < m; i += kThreads) {
      const uint64_t mine = sm.cand[i];
      int rank = 0;
      for (int j = 0; j < m; ++j) rank += sm.cand[j] > mine;
      if (rank < k) emit(rank, key_index(mine));
    }
  };
  gather(theta);
  const int m = sm.count;
  if (m <= kLpCap) {
    write_ranked(m);
    return;
  }
  // Too many: runs of equal values at theta (masked rows), or large values side by side.
  __syncthreads();
  if (tid == 0) sm.count = 0;
  __syncthreads();
  if (theta != 0xffffffffu) gather(theta + 1);  // block-uniform
  const int above = sm.count;
  if (above > kLpCap) {
    __syncthreads();
    topk_by_lists<8, kWaves>(V, k, sm.lists, [&](int i) { return ord(Elem<DT>::cvt(x[i])); },
                             [](float) {}, emit);
    return;
  }
  write_ranked(above);
  int found = above;  // the rest: entries equal to theta, lowest index first
  for (int b = 0; b < V && found < k; b += kThreads) {
    const int i = b + tid;
    const bool eq = i < V && ord_key(Elem<DT>::cvt(x[i])) == theta;
    const uint64_t mask = __ballot(eq);
    __syncthreads();
    if (lane == 0) sm.wave_cnt[wid] = __popcll(mask);
    __syncthreads();
    int pos = found, total = 0;
    for (int w = 0; w < kWaves; ++w) {
      pos += w < wid ? sm.wave_cnt[w] : 0;
      total += sm.wave_cnt[w];
    }
    pos += __popcll(mask & ((1ull << lane) - 1ull));
    if (eq && pos < k) emit(pos, i);
    found += total;
  }
}

hipError_t launch_spec_logprobs(const LogprobParams& p, hipStream_t stream) {
  const int n = p.B * p.W;
  if (n <= 0) return hipSuccess;
  if (p.k <= 8)
    hipLaunchKernelGGL(spec_logprobs_kernel<8>, dim3(n), dim3(kLpThreads), 0, stream, p);
  else
    hipLaunchKernelGGL(spec_logprobs_kernel<32>, dim3(n), dim3(kLpThreads), 0, stream, p);
  return hipGetLastError();
}

int64_t split_logprobs_workspace_bytes(int64_t positions, int64_t V, int64_t k) {
  if (positions <= 0 || k > kSplitMaxK || lists_are_faster(positions, V, k)) return 0;
  const int64_t chunk = split_chunk(positions, V, k);
  const int64_t nch = (V + chunk - 1) / chunk;
  // a row's groups fit LDS; the scan's threads stay below 2^32
  if (nch * kGroupsPerChunk > kMaxGroups || positions * nch >= (1ll << 24)) return 0;
  return positions * nch * (int64_t)(sizeof(float4) + kGroupsPerChunk * sizeof(uint32_t));
}

template <int DT>
static void launch_split_dt(const LogprobParams& p, int chunk, hipStream_t stream) {
  constexpr int kLong = kChunkLong / (kThreads * Elem<DT>::kVec);
  constexpr int kShort = kChunkShort / (kThreads * Elem<DT>::kVec);
  const int n = p.B * p.W;
  const dim3 scan((unsigned)n * (unsigned)p.nchunks), finish((unsigned)n), block(kThreads);
  const unsigned lds = (unsigned)(p.nchunks * kGroupsPerChunk * 6);  // keys and 16-bit list
  if (chunk == kChunkLong) {
    hipLaunchKernelGGL((lp_scan_kernel<DT, kLong>), scan, block, 0, stream, p);
    hipLaunchKernelGGL((lp_finish_kernel<DT, kLong>), finish, block, lds, stream, p);
  } else {
    hipLaunchKernelGGL((lp_scan_kernel<DT, kShort>), scan, block, 0, stream, p);
    hipLaunchKernelGGL((lp_finish_kernel<DT, kShort>), finish, block, lds, stream, p);
  }
}

hipError_t launch_split_logprobs(LogprobParams p, int dtype, void* workspace, hipStream_t stream) {
  const int64_t n = (int64_t)p.B * p.W;
  if (n <= 0) return hipSuccess;
  const int chunk = split_chunk(n, p.V, p.k);
  p.nchunks = (p.V + chunk - 1) / chunk;
  p.stats = static_cast<float4*>(workspace);
  p.group_keys = reinterpret_cast<uint32_t*>(p.stats + n * p.nchunks);
  switch (dtype) {
    case MVSD_F32: launch_split_dt<MVSD_F32>(p, chunk, stream); break;
    case MVSD_BF16: launch_split_dt<MVSD_BF16>(p, chunk, stream); break;
    case MVSD_F16: launch_split_dt<MVSD_F16>(p, chunk, stream); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace mvsd
