// Sampling constraints of the verify rows (top-k / top-p per request) as per-row thresholds,
// for the verify kernel to apply while it streams the raw rows.
//
// Reference: apply_sampling_constraints (minivllm/sample/rejection_sampler.py:537-571) divides
// the gathered fp32 verify rows by the request temperature (greedy T = 0 -> 1; nothing at all
// when every request is greedy) and calls apply_top_k_top_p
// (minivllm/sample/ops/topk_topp_sampler.py:48-79): ascending sort; top-k masks the values
// below the k-th largest (:61-69); top-p masks the ascending prefix whose cumulative softmax
// mass is <= 1 - p and never the last entry (:71-77).  Equal values keep index order, as a
// stable sort keeps them.
//
// With v = fl(x / T), the masked entries of a row are a prefix of the order (v, index), so the
// first kept entry (v_f, i_f) describes them: entry i is masked iff v < v_f, or v == v_f and
// i < i_f.  Division by T > 0 is monotone, hence v < v_f iff x < A with
// A = min{x : fl(x / T) >= v_f}, and v <= v_f iff x < B with B = min{x : fl(x / T) > v_f}:
//     masked(x, i) = x < A || (x < B && i <= J),   J = i_f - 1,
// a test on the raw values that needs no division.  A row with only top-k has B = -inf.
//
// Per row (one 512-thread workgroup):
//   pass 1   the row maximum and every thread's own maximum;
//   top-k    for k <= 512 the k-th largest thread maximum bounds the k-th largest entry from
//            below, so the entries at or above it (about k of them) are gathered into LDS,
//            sorted by (v, index), and read off; otherwise (or if too many tie) a bisection
//            over the value keys counts entries per pass;
//   top-p    masses floor(2^40 * exp(v - v_max)) in 64-bit fixed point, so sums are exact and
//            independent of order.  With a top-k candidate set the prefix is found in LDS;
//            otherwise a histogram over 4096 logarithmic mass bins (96 per factor of two)
//            locates the bin of the first kept entry, whose entries are gathered, sorted and
//            scanned; an overfull bin falls back to bisection over (v, index).
// The limit floor((1 - p) * S) is computed exactly in integers.
#include <float.h>
#include <string.h>

#include <type_traits>

#include "mvsd_device.h"
#include "verify.h"

namespace mvsd {
namespace {

#ifndef MVSD_CONSTRAINT_BATCH
#define MVSD_CONSTRAINT_BATCH 3   // 16-byte vectors per thread per batch of a row walk
#endif

#ifndef MVSD_CONSTRAINT_THREADS
#define MVSD_CONSTRAINT_THREADS 512
#endif
#ifndef MVSD_CONSTRAINT_CAP
#define MVSD_CONSTRAINT_CAP 4096
#endif

constexpr int kCT = MVSD_CONSTRAINT_THREADS;  // threads per row
constexpr int kCW = kCT / kWave;
constexpr int kCap = MVSD_CONSTRAINT_CAP;     // candidates gathered in LDS
constexpr int kBins = 4096;              // top-p histogram bins
constexpr float kBinScale = 96.f * 1.44269504088896340736f;  // bins per unit of v_max - v
constexpr float kLog2e = 1.44269504088896340736f;
constexpr uint32_t kNanKey = 0xffffffffu;

struct ConstraintSmem {
  union {
    unsigned long long hist[kBins];
    unsigned long long cand[kCap];     // ordered_bits(v) << 32 | index, sorted ascending
  } u;
  unsigned long long part[kCT];        // scan partials
  unsigned long long red[kCW];
  unsigned long long bcast[4];
  int count;
};

// Calls g(vector index, 16-byte vector) for every vector of a row of nvec vectors: full
// batches of U vectors per thread, two batches in flight (each iteration issues one buffer's
// next loads before consuming the other, and the loads of a full batch are unconditional, the
// last one clamped to the last full batch, so each wait covers exactly one batch), then the
// remaining vectors one per thread and step.
template <typename P, typename G>
__device__ inline void for_each_vector(const P* xv, int nvec, G&& g) {
  constexpr int U = MVSD_CONSTRAINT_BATCH;
  constexpr int step = U * kCT;
  const int tid = threadIdx.x;
  const int nfull = nvec / step;
  auto load = [&](u32x4 (&buf)[U], int j) {
    const int base = min(j, nfull - 1) * step + tid;
#pragma unroll
    for (int u = 0; u < U; ++u) buf[u] = xv[base + u * kCT];
  };
  auto consume = [&](const u32x4 (&buf)[U], int j) {
#pragma unroll
    for (int u = 0; u < U; ++u) g(j * step + tid + u * kCT, buf[u]);
  };
  if (nfull > 0) {
    u32x4 a[U], b[U];
    load(a, 0);
    for (int j = 0;;) {
      load(b, j + 1);
      // a compiler barrier: the loads above stay issued ahead of the consumption below
      asm volatile("" ::: "memory");
      consume(a, j);
      if (++j == nfull) break;
      load(a, j + 1);
      asm volatile("" ::: "memory");
      consume(b, j);
      if (++j == nfull) break;
    }
  }
  for (int v = nfull * step + tid; v < nvec; v += kCT) g(v, xv[v]);
}

// Calls f(i0, v, n) for every group of consecutive entries: v[0, n) are entries i0, i0 + 1,
// ...; a group is one 16-byte vector (n = VEC), or one of the row's last entries that fill none
// (n = 1).  Per-group work lets a pass test a whole vector with one branch.  Rows of any alignment
// and length take the vector walk (a scalar walk for odd ones took 56 us instead of 39 on top-p
// rows of 50257 bf16 entries).
template <int DT, typename F>
__device__ inline void for_each_group(const typename Elem<DT>::storage* __restrict__ x, int V,
                                      F&& f) {
  constexpr int VEC = Elem<DT>::kVec;
  const int nvec = V / VEC;
  for_each_vector(reinterpret_cast<const Vec16<DT>*>(x), nvec, [&](int vi, const u32x4& r) {
    float v[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) v[j] = vec_elem<DT>(r, j);
    f(vi * VEC, v, VEC);
  });
  const int i = nvec * VEC + (int)threadIdx.x;
  if (i < V) {
    float v[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) v[j] = Elem<DT>::cvt(x[i]);
    f(i, v, 1);
  }
}

// Calls f(index, value) for every entry of the row.
template <int DT, typename F>
__device__ inline void for_each_entry(const typename Elem<DT>::storage* __restrict__ x, int V,
                                      F&& f) {
  constexpr int VEC = Elem<DT>::kVec;
  for_each_group<DT>(x, V, [&](int i0, const float (&v)[VEC], int n) {
#pragma unroll
    for (int j = 0; j < VEC; ++j)
      if (j < n) f(i0 + j, v[j]);
  });
}

// q[j] = x[j] / T for a group; one branch per group to the IEEE divide when any entry is
// outside the range of the corrected division.
template <int N>
__device__ inline void divide_group(const Divider& d, const float (&x)[N], float (&q)[N]) {
  float least = INFINITY, most = 0.f;  // a NaN leaves them: its quotient is NaN either way
#pragma unroll
  for (int j = 0; j < N; ++j) {
    least = fminf(least, fabsf(x[j]));
    most = fmaxf(most, fabsf(x[j]));
    const float q0 = x[j] * d.rt;
    q[j] = fmaf(fmaf(-q0, d.t, x[j]), d.rt, q0);
  }
  if (!(least >= d.lo && most <= d.hi)) {
#pragma unroll
    for (int j = 0; j < N; ++j) q[j] = x[j] / d.t;
  }
}

__device__ inline unsigned long long block_sum_u64(unsigned long long v, ConstraintSmem& sm) {
  v = wave_sum_u64(v);
  if (lane_id() == 0) sm.red[wave_id()] = v;
  __syncthreads();
  unsigned long long s = 0;
  for (int w = 0; w < kCW; ++w) s += sm.red[w];
  __syncthreads();
  return s;
}

__device__ inline uint32_t block_max_u32(uint32_t v, ConstraintSmem& sm) {
  v = wave_max_u32(v);
  if (lane_id() == 0) sm.red[wave_id()] = v;
  __syncthreads();
  uint32_t m = 0;
  for (int w = 0; w < kCW; ++w) m = max(m, (uint32_t)sm.red[w]);
  __syncthreads();
  return m;
}

// Inclusive scan of one value per thread in thread order: within each wave by shuffles, then the
// totals of the waves before.
__device__ inline unsigned long long block_scan_u64(unsigned long long v, ConstraintSmem& sm) {
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const unsigned long long add = __shfl_up(v, off);
    v += lane_id() >= off ? add : 0ull;
  }
  if (lane_id() == kWave - 1) sm.red[wave_id()] = v;
  __syncthreads();
  for (int w = 0; w < wave_id(); ++w) v += sm.red[w];
  __syncthreads();
  return v;
}

// exp(-d) for d = v_max - v >= 0 (or +inf), in [0, 1].
__device__ inline float mass_exp(float d) { return __builtin_amdgcn_exp2f(-d * kLog2e); }

// floor(2^40 * e): the 64-bit fixed-point mass.
__device__ inline unsigned long long mass_from_e(float e) {
  const float h = e * 256.f;  // e * 2^8, exact
  const float hi = floorf(h);
  const uint32_t lo = (uint32_t)((h - hi) * 4294967296.f);  // exact fraction * 2^32 < 2^32
  return ((unsigned long long)(uint32_t)hi << 32) | lo;
}

// Histogram bin of d = v_max - v: 96 bins per factor of two of mass, bin 0 at the maximum,
// clamped to the last bin past d = 29.6 (masses there are below 2^-40 of the maximum's, 0 in
// fixed point).  A non-decreasing function of d, computed with correctly rounded operations,
// so the entries of one bin are an interval of v, and of x.
__device__ inline int mass_bin(float d) {
  const float y = d * kBinScale;
  return y < (float)(kBins - 1) ? (y > 0.f ? (int)y : 0) : kBins - 1;
}

__device__ inline unsigned long long mass_of(float d) { return mass_from_e(mass_exp(d)); }

// floor(t * S) for fp32 t in (0, 1] and S < 2^64, exactly (t = mant * 2^(e - 24)).
__device__ inline unsigned long long scaled_floor(float t, unsigned long long S) {
  int e;
  const float fr = frexpf(t, &e);
  const unsigned long long mant = (unsigned long long)(fr * 16777216.0f);
  const int sh = 24 - e;
  const unsigned long long lo = mant * S;
  const unsigned long long hi = __umul64hi(mant, S);
  return sh >= 64 ? (hi >> (sh - 64)) : ((hi << (64 - sh)) | (lo >> sh));
}

// Smallest non-NaN float x with fl(x / T) >= v (v not NaN): within a few floats of v * T, where
// eight neighbouring keys are tried side by side (key order, in which fl(x / T) is monotone); a
// bisection over all keys where that window does not hold the step.
__device__ inline float min_x_reaching(float v, float T) {
  const float x0 = v * T;
  if (fabsf(x0) > 0x1p-100f && fabsf(x0) < 0x1p100f) {
    const uint32_t first = ordered_bits(x0) - 4u;  // keys of floats of x0's sign
    int below = 0;
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) below += key_float(first + j) / T >= v ? 0 : 1;
    if (below > 0 && below < 8) return key_float(first + (uint32_t)below);
  }
  uint32_t lo = ordered_bits(-INFINITY), hi = ordered_bits(INFINITY);  // pred(hi) holds
  if (key_float(lo) / T >= v) return -INFINITY;
  while (hi - lo > 1) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if (key_float(mid) / T >= v) hi = mid;
    else lo = mid;
  }
  return key_float(hi);
}

// Next float above v in the order where -0 == +0 (v finite).
__device__ inline float next_up(float v) {
  return v == 0.f ? __uint_as_float(1u) : key_float(ordered_bits(v) + 1u);
}

// Appends key to the LDS candidate list where pred holds (one LDS atomic per wave).
__device__ inline void append(bool pred, unsigned long long key, ConstraintSmem& sm) {
  const unsigned long long mask = __ballot(pred);
  if (mask == 0) return;
  const int leader = __ffsll((long long)mask) - 1;
  int base = 0;
  if (lane_id() == leader) base = atomicAdd(&sm.count, __popcll(mask));
  base = __shfl(base, leader);
  if (pred) {
    const int pos = base + __popcll(mask & ((1ull << lane_id()) - 1ull));
    if (pos < kCap) sm.u.cand[pos] = key;
  }
}

// Appends the keys of this lane's flagged entries (c[j]: key(j)) to the LDS candidate list:
// per-lane positions from the wave's ballots, one LDS atomic per wave.  Safe with inactive
// lanes (ballots count active lanes only).
__device__ inline int lanes_below(unsigned long long mask) {
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                        __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

template <int N, typename K>
__device__ inline void append_group(const bool (&c)[N], K&& key, ConstraintSmem& sm) {
  int total = 0, pos = 0;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const unsigned long long m = __ballot(c[j]);
    total += __popcll(m);
    pos += lanes_below(m);
  }
  if (total == 0) return;
  const int leader = __ffsll((long long)__ballot(true)) - 1;
  int base = 0;
  if (lane_id() == leader) base = atomicAdd(&sm.count, total);
  pos += __shfl(base, leader);
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if (c[j]) {
      if (pos < kCap) sm.u.cand[pos] = key(j);
      ++pos;
    }
  }
}

// Smallest non-NaN x whose bin mass_bin(vmax - fl(x / T)) is at most b: the bin of x falls as x
// grows, so the entries of bin b are exactly those with min_x_in_bins(b) <= x <
// min_x_in_bins(b - 1).  Bisection over the ordered keys with the histogram's own arithmetic.
__device__ inline float min_x_in_bins(float vmax, const Divider& dv, int b) {
  if (b < 0) return INFINITY;  // no x has a negative bin; +inf bounds every finite entry
  auto in = [&](uint32_t key) { return mass_bin(vmax - divide(dv, key_float(key))) <= b; };
  uint32_t lo = ordered_bits(-INFINITY), hi = ordered_bits(INFINITY);  // in(hi) holds
  if (in(lo)) return -INFINITY;
  while (hi - lo > 1) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if (in(mid)) hi = mid;
    else lo = mid;
  }
  return key_float(hi);
}

// The k-th largest (1 <= k <= kCT) of the block's keys, one per thread (`mine`), by radix
// selection: four rounds of an 8-bit digit, each counting the keys that share the digits found
// so far per next digit (LDS atomics on 256 counters), after which one wave picks the digit
// holding the k-th largest.  Every thread receives the key.  Uses sm.part and sm.bcast.
__device__ inline uint32_t kth_largest_key(uint32_t mine, int k, ConstraintSmem& sm) {
  int* cnt = reinterpret_cast<int*>(sm.part);  // 256 counters
  const int tid = threadIdx.x;
  uint32_t prefix = 0, pmask = 0;
  int need = k;  // rank of the wanted key among the keys matching the prefix
#pragma unroll 1
  for (int shift = 24; shift >= 0; shift -= 8) {
    for (int b = tid; b < 256; b += kCT) cnt[b] = 0;
    __syncthreads();
    if ((mine & pmask) == prefix) atomicAdd(&cnt[(mine >> shift) & 255u], 1);
    __syncthreads();
    if (tid < kWave) {
      // lane l holds digits 255 - 4l .. 252 - 4l, the largest first
      int c[4], own = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        c[j] = cnt[255 - 4 * tid - j];
        own += c[j];
      }
      int incl = own;
#pragma unroll
      for (int off = 1; off < kWave; off <<= 1) {
        const int t = __shfl_up(incl, off);
        if (tid >= off) incl += t;
      }
      const int above = incl - own;  // keys with a larger digit than this lane's
      if (above < need && need <= incl) {
        int run = above, j = 0;
        while (run + c[j] < need) run += c[j++];
        sm.bcast[0] = (unsigned long long)(255 - 4 * tid - j);
        sm.bcast[1] = (unsigned long long)(need - run);
      }
    }
    __syncthreads();
    prefix |= (uint32_t)sm.bcast[0] << shift;
    pmask |= 0xffu << shift;
    need = (int)sm.bcast[1];
    __syncthreads();
  }
  return prefix;
}

// Sorts cand[0, n), ascending; n <= kCap, keys distinct.  Up to one key per thread by counting
// the smaller ones (two barriers), more by a bitonic network (one barrier per step).
__device__ inline void sort_candidates(int n, ConstraintSmem& sm) {
  if (n <= kCT) {
    const unsigned long long mine = sm.u.cand[min((int)threadIdx.x, max(n - 1, 0))];
    int rank = 0;
#pragma unroll 4
    for (int j = 0; j < n; ++j) rank += sm.u.cand[j] < mine;
    __syncthreads();
    if ((int)threadIdx.x < n) sm.u.cand[rank] = mine;
    __syncthreads();
    return;
  }
  int N = 1;
  while (N < n) N <<= 1;
  for (int i = n + (int)threadIdx.x; i < N; i += kCT) sm.u.cand[i] = ~0ull;
  __syncthreads();
  for (int size = 2; size <= N; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = threadIdx.x; i < N / 2; i += kCT) {
        const int lo = 2 * i - (i & (stride - 1));
        const int hi = lo + stride;
        const bool up = (lo & size) == 0;
        const unsigned long long a = sm.u.cand[lo], b = sm.u.cand[hi];
        if ((a > b) == up) {
          sm.u.cand[lo] = b;
          sm.u.cand[hi] = a;
        }
      }
      __syncthreads();
    }
  }
}

// First position f in the sorted cand[s, e) where base + (mass of cand[s..f]) > limit, or
// e - 1 when there is none (the last entry is always kept).  mass(key) is a candidate's mass.
template <typename M>
__device__ inline int first_over(int s, int e, unsigned long long base, unsigned long long limit,
                                 ConstraintSmem& sm, M&& mass) {
  const int len = e - s;
  const int per = (len + kCT - 1) / kCT;
  const int b0 = s + (int)threadIdx.x * per, b1 = min(e, b0 + per);
  unsigned long long seg = 0;
  for (int i = b0; i < b1; ++i) seg += mass(sm.u.cand[i]);
  if (threadIdx.x == 0) sm.bcast[0] = (unsigned long long)(e - 1);
  const unsigned long long incl = block_scan_u64(seg, sm);
  unsigned long long run = base + (incl - seg);
  if (run <= limit && limit < base + incl) {
    for (int i = b0; i < b1; ++i) {
      run += mass(sm.u.cand[i]);
      if (run > limit) {
        sm.bcast[0] = (unsigned long long)i;
        break;
      }
    }
  }
  __syncthreads();
  const int f = (int)sm.bcast[0];
  __syncthreads();
  return f;
}

// Request of verify row `row` (the first r with cu[r] > row; -1 past the last request), or the
// row itself when there is no cu (one row per request).
__device__ inline int request_of(const VerifyParams& p, int row) {
  if (!p.cu) return row < p.B ? row : -1;
  if (p.B <= 0 || row >= p.cu[p.B - 1]) return -1;
  int lo = 0, hi = p.B - 1;
  while (lo < hi) {
    const int mid = (lo + hi) / 2;
    if (p.cu[mid] > row) hi = mid;
    else lo = mid + 1;
  }
  return lo;
}

// How much work the verify rows of request r take in the constraints kernel: 0 none (no
// constraint, or a greedy request with top-k only: see row_thresholds), 1 random with top-p
// (three passes per row), 2 random with top-k only (one pass), 3 greedy with top-p (one pass,
// more when a row's maximum is tied).
__device__ inline int request_class(const VerifyParams& p, int r) {
  if (p.all_greedy) return 0;
  const int64_t kk = p.top_k ? p.top_k[r] : (int64_t)p.V;
  const bool has_k = kk > 0 && kk < p.V;
  const bool has_p = p.top_p && 1.0f - p.top_p[r] > 0.f;
  const bool greedy = p.temperature != nullptr && p.temperature[r] == 0.f;
  if ((!has_k && !has_p) || (greedy && !has_p)) return 0;
  return greedy ? 3 : (has_p ? 1 : 2);
}

// The plan of a masked call (one 1024-thread workgroup, one request per thread at a time):
// the neutral mask for every row of class 0, and the other rows listed by class, as row + 1,
// so that the rows with the most passes start first.  The order inside a class does not
// matter: each row's mask depends on its own row only.
__global__ __launch_bounds__(1024) void constraint_plan_kernel(VerifyParams p) {
  __shared__ int cnt[4], base[4];
  const int tid = threadIdx.x;
  if (tid < 4) cnt[tid] = 0;
  __syncthreads();
  const float4 neutral = make_float4(-INFINITY, -INFINITY, __int_as_float(-1), 0.f);
  // rows past the last request belong to none
  for (int j = max(p.B > 0 ? p.cu[p.B - 1] : 0, 0) + tid; j < p.P; j += 1024) p.masks[j] = neutral;
  for (int r = tid; r < p.B; r += 1024) {
    const int begin = max(r == 0 ? 0 : p.cu[r - 1], 0), end = min(p.cu[r], p.P);
    const int c = request_class(p, r);
    if (c == 0) {
      for (int j = begin; j < end; ++j) p.masks[j] = neutral;
    } else if (end > begin) {
      atomicAdd(&cnt[c], end - begin);
    }
  }
  __syncthreads();
  if (tid == 0) {
    base[1] = 0;
    base[2] = cnt[1];
    base[3] = cnt[1] + cnt[2];
    cnt[1] = cnt[2] = cnt[3] = 0;
  }
  __syncthreads();
  for (int r = tid; r < p.B; r += 1024) {
    const int begin = max(r == 0 ? 0 : p.cu[r - 1], 0), end = min(p.cu[r], p.P);
    const int c = request_class(p, r);
    if (c != 0 && end > begin) {
      const int at = base[c] + atomicAdd(&cnt[c], end - begin);
      // (cumulative counts that decrease would list a row more than once: only P places)
      for (int j = begin; j < min(end, p.P - at + begin); ++j) p.order[at + (j - begin)] = j + 1;
    }
  }
}

// Top-p of a greedy row whose maximum is tied (ties >= 2 entries at raw key mkey), without
// top-k.  Only the row's argmax matters, and the temperature is 1, so v = x and the tied
// entries are exactly the entries at the maximum, each of mass mass_of(0) = 2^40.  The masked
// prefix of the order (v, index) reaches them only when the mass below the maximum is at most
// the limit; then it takes every entry below the maximum and the first m tied entries in index
// order, m = floor((limit - below) / 2^40) (at most ties - 1: the last entry is always kept).
// One pass sums the masses; a second gathers the tied entries' indices only when the prefix
// reaches them.  Returns 0 (no mask changes the argmax: the neutral mask), 1 (A, B, J set), or
// -1 (more tied entries than LDS holds: the general path).
template <int DT>
__device__ inline int greedy_tied_top_p(const typename Elem<DT>::storage* __restrict__ x, int V,
                                        const Divider& dv, float T, float t,
                                        uint32_t mkey, unsigned long long ties,
                                        ConstraintSmem& sm, float& A, float& Bv, int& J) {
  constexpr int VEC = Elem<DT>::kVec;
  const float vmax = divide(dv, key_float(mkey));
  if (vmax != vmax || fabsf(vmax) == INFINITY) return 0;
  unsigned long long s = 0;
  for_each_group<DT>(x, V, [&](int, const float (&v)[VEC], int n) {
    float q[VEC];
    divide_group(dv, v, q);
#pragma unroll
    for (int j = 0; j < VEC; ++j)
      if (j < n) s += mass_of(vmax - q[j]);
  });
  const unsigned long long total = block_sum_u64(s, sm);
  const unsigned long long limit = scaled_floor(fminf(t, 1.f), total);
  constexpr unsigned long long kUnit = 1ull << 40;  // mass_of(0)
  const unsigned long long below = total - ties * kUnit;
  if (limit < below + kUnit) return 0;  // the first maximum is kept
  if (ties > (unsigned long long)kCap) return -1;
  unsigned long long m = (limit - below) / kUnit;
  if (m > ties - 1) m = ties - 1;
  if (threadIdx.x == 0) sm.count = 0;
  __syncthreads();
  for_each_group<DT>(x, V, [&](int i0, const float (&v)[VEC], int n) {
    bool c[VEC], any = false;
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      c[j] = (j < n) && ordered_bits(v[j]) == mkey;
      any |= c[j];
    }
    if (__ballot(any) == 0) return;
#pragma unroll
    for (int j = 0; j < VEC; ++j)
      append(c[j], c[j] ? (((unsigned long long)mkey << 32) | (uint32_t)(i0 + j)) : 0ull, sm);
  });
  __syncthreads();
  const int n = sm.count;  // == ties
  sort_candidates(n, sm);
  const int i_f = (int)(uint32_t)sm.u.cand[min((int)m, n - 1)];
  A = min_x_reaching(vmax, T);
  Bv = min_x_reaching(next_up(vmax), T);
  J = i_f - 1;
  return 1;
}

// The mask (A, B, J) of target row xrow from request r's top-k / top-p (r < 0: none); false when
// nothing is masked.
template <int DT>
__device__ __forceinline__ bool row_thresholds(const VerifyParams& p, int r, int64_t xrow,
                                               ConstraintSmem& sm, float& A, float& Bv, int& J) {
  using S = typename Elem<DT>::storage;
  const int tid = threadIdx.x;
  A = -INFINITY;
  Bv = -INFINITY;
  J = -1;
  if (p.all_greedy || r < 0) return false;
  const int64_t kk = p.top_k ? p.top_k[r] : (int64_t)p.V;
  const float t = p.top_p ? 1.0f - p.top_p[r] : 0.f;
  const bool has_k = kk > 0 && kk < p.V;
  const bool has_p = t > 0.f;  // p >= 1 keeps every entry of non-zero probability
  if (!has_k && !has_p) return false;
  // A greedy row only needs its argmax (the first maximum, or the first NaN).  Top-k keeps
  // every entry at or above the k-th largest, so it never masks a maximum or a NaN; top-p
  // masks an ascending prefix that never includes the last entry of the order (v, index), so
  // it masks a maximum only when the maximum is tied (a NaN makes every mass NaN and masks
  // nothing).  Such a row gets no mask unless it has top-p and a tied maximum.  (The in-place
  // top-k / top-p of the sampler passes no temperatures: none of its rows is greedy.)
  const bool greedy_row = p.temperature != nullptr && p.temperature[r] == 0.f;
  if (greedy_row && !has_p) return false;
  const float T = req_temperature(p, r);
  const Divider dv = make_divider(T);
  const int V = p.V;
  const S* x = static_cast<const S*>(p.target) + xrow * p.target_stride;

  // ---- pass 1: row maximum and per-thread maxima (ordered keys of the raw values); rows with
  // top-k only also keep each thread's four largest keys ----
  const bool k_only = has_k && !has_p && kk <= kCT;
  uint32_t t0 = 0, t1 = 0, t2 = 0, t3 = 0;
  constexpr int VEC = Elem<DT>::kVec;
  if (k_only) {
    // The four largest values in floats (NaN read as -inf and flagged): max / min pairs.  A
    // row with a NaN, which ranks above every number, takes the key-based walk below.
    float f0 = -INFINITY, f1 = -INFINITY, f2 = -INFINITY, f3 = -INFINITY;
    int seen = 0;
    bool nan = false;
    for_each_group<DT>(x, V, [&](int, const float (&v)[VEC], int n) {
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        if (j < n) {
          nan |= v[j] != v[j];
          float c = v[j] == v[j] ? v[j] : -INFINITY, m;
          m = fmaxf(f0, c); c = fminf(f0, c); f0 = m;
          m = fmaxf(f1, c); c = fminf(f1, c); f1 = m;
          m = fmaxf(f2, c); c = fminf(f2, c); f2 = m;
          f3 = fmaxf(f3, c);
        }
      }
      seen += n;
    });
    // a slot no entry filled keeps key 0, below every entry's key
    t0 = seen > 0 ? ordered_bits(f0) : 0u;
    t1 = seen > 1 ? ordered_bits(f1) : 0u;
    t2 = seen > 2 ? ordered_bits(f2) : 0u;
    t3 = seen > 3 ? ordered_bits(f3) : 0u;
    if (__syncthreads_or(nan)) {
      t0 = t1 = t2 = t3 = 0;
      for_each_group<DT>(x, V, [&](int, const float (&v)[VEC], int n) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
          if (j < n) {
            uint32_t c = ordered_bits(v[j]), m;
            m = max(t0, c); c = min(t0, c); t0 = m;
            m = max(t1, c); c = min(t1, c); t1 = m;
            m = max(t2, c); c = min(t2, c); t2 = m;
            t3 = max(t3, c);
          }
        }
      });
    }
  } else {
    // The thread maximum in floats, the number of entries equal to it (for the greedy tie
    // test; -0 and +0 compare equal, as their keys do) and a NaN flag (NaN ranks above every
    // number, so the thread's key is then the NaN key).
    float fm = -INFINITY;
    uint32_t ties = 0;
    bool nan = false;
    for_each_group<DT>(x, V, [&](int, const float (&v)[VEC], int n) {
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        if (j < n) {
          nan |= v[j] != v[j];
          ties = v[j] > fm ? 1u : ties + (v[j] == fm);
          fm = fmaxf(fm, v[j]);
        }
      }
    });
    t0 = nan ? kNanKey : (ties > 0 ? ordered_bits(fm) : 0u);
    t1 = ties;
  }
  const uint32_t mkey = block_max_u32(t0, sm);
  if (greedy_row) {
    const unsigned long long ties = block_sum_u64(t0 == mkey ? t1 : 0u, sm);
    if (mkey == kNanKey || ties < 2) return false;
    if (!has_k) {
      const int g = greedy_tied_top_p<DT>(x, V, dv, T, t, mkey, ties, sm, A, Bv, J);
      if (g >= 0) return g == 1;
    }
  }

  // ---- top-k: v_k, the k-th largest v, and the entries with v >= v_k in LDS if they fit ----
  bool cand_ok = false;
  int n = 0, lo_k = 0;
  if (has_k) {
    const int k = (int)kk;
    uint32_t theta = 0;
    if (k <= kCT) {
      // theta: the k-th largest thread maximum; at least k entries are >= theta
      theta = kth_largest_key(t0, k, sm);
      if (tid == 0) sm.count = 0;
      __syncthreads();
    }
    bool k_done = false;
    uint32_t vk_key = 0;
    if (k_only && theta != 0) {
      // Every entry >= theta is among its thread's four largest unless that thread's fourth
      // largest is >= theta too; then the general path below runs instead.
      const int overflow = __syncthreads_or(t3 >= theta);
      if (!overflow) {
        uint32_t* ck = reinterpret_cast<uint32_t*>(sm.u.cand);
        auto put = [&](uint32_t key) {
          const bool c = key >= theta;
          const unsigned long long mask = __ballot(c);
          if (mask == 0) return;
          const int leader = __ffsll((long long)mask) - 1;
          int base = 0;
          if (lane_id() == leader) base = atomicAdd(&sm.count, __popcll(mask));
          base = __shfl(base, leader);
          if (c) ck[base + __popcll(mask & ((1ull << lane_id()) - 1ull))] = key;
        };
        put(t0);
        put(t1);
        put(t2);
        __syncthreads();
        const int nk = sm.count;  // <= 3 * kCT, and >= k
        // the k-th largest key: the entry with k - 1 entries above it (ties by position)
        for (int i = tid; i < nk; i += kCT) {
          const uint32_t mine = ck[i];
          int rank = 0;
          for (int j = 0; j < nk; ++j) {
            const uint32_t o = ck[j];
            rank += (o > mine) | ((o == mine) & (j < i));
          }
          if (rank == k - 1) sm.bcast[1] = mine;
        }
        __syncthreads();
        vk_key = ordered_bits(divide(dv, key_float((uint32_t)sm.bcast[1])));
        k_done = true;
      }
    }
    if (!k_done && k <= kCT) {
      // Gather every entry whose v reaches fl(theta / T) (x >= theta2): that includes every
      // entry with v >= v_k.  (theta = 0: fewer than k threads hold entries; NaN theta:
      // gather everything.)
      const float theta2 = theta == 0 ? -INFINITY
                           : (theta == kNanKey ? NAN : min_x_reaching(divide(dv, key_float(theta)), T));
      if (tid == 0) sm.count = 0;
      __syncthreads();
      for_each_group<DT>(x, V, [&](int i0, const float (&v)[VEC], int n) {
        bool c[VEC], any = false;
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
          c[j] = (j < n) && !(v[j] < theta2);
          any |= c[j];
        }
        if (__ballot(any) == 0) return;
#pragma unroll
        for (int j = 0; j < VEC; ++j)
          append(c[j], c[j] ? (((unsigned long long)ordered_bits(divide(dv, v[j])) << 32) | (uint32_t)(i0 + j)) : 0ull, sm);
      });
      __syncthreads();
      n = sm.count;
      cand_ok = n <= kCap;
    }
    if (k_done) {
      // v_k found from the per-thread keys
    } else if (cand_ok) {
      sort_candidates(n, sm);
      vk_key = (uint32_t)(sm.u.cand[max(n - k, 0)] >> 32);
      int below = 0;
      for (int i = tid; i < n; i += kCT) below += (uint32_t)(sm.u.cand[i] >> 32) < vk_key;
      lo_k = (int)block_sum_u64((unsigned long long)below, sm);
    } else {
      // largest raw key K with count(key(x) >= K) >= k, by bisection (one pass per step)
      uint64_t lo = 0, hi = 0x100000000ull;  // count(>= lo) >= k > count(>= hi)
      while (hi - lo > 1) {
        const uint64_t mid = (lo + hi) / 2;
        unsigned long long c = 0;
        for_each_entry<DT>(x, V, [&](int, float v) { c += ordered_bits(v) >= (uint32_t)mid; });
        if (block_sum_u64(c, sm) >= (unsigned long long)k) lo = mid;
        else hi = mid;
      }
      vk_key = ordered_bits(divide(dv, key_float((uint32_t)lo)));
    }
    // A NaN k-th value compares false with everything: the reference then masks nothing.
    if (vk_key != kNanKey) A = min_x_reaching(key_float(vk_key), T);
  }

  // ---- top-p over the entries top-k keeps (x >= A) ----
  // A NaN or infinite maximum makes every softmax value NaN in the reference, and then no
  // cumulative sum compares <= 1 - p.
  const float vmax = cand_ok ? key_float((uint32_t)(sm.u.cand[max(n - 1, 0)] >> 32))
                             : divide(dv, key_float(mkey));
  if (!has_p || mkey == kNanKey || vmax != vmax || fabsf(vmax) == INFINITY) return A != -INFINITY;
  const float tl = fminf(t, 1.f);
  unsigned long long fkey;  // ordered_bits(v_f) << 32 | i_f of the first kept entry
  if (cand_ok) {
    unsigned long long seg = 0;
    for (int i = lo_k + tid; i < n; i += kCT)
      seg += mass_of(vmax - key_float((uint32_t)(sm.u.cand[i] >> 32)));
    const unsigned long long total = block_sum_u64(seg, sm);
    fkey = sm.u.cand[max(first_over(lo_k, n, 0, scaled_floor(tl, total), sm,
                                    [&](unsigned long long key) {
                                      return mass_of(vmax - key_float((uint32_t)(key >> 32)));
                                    }), 0)];
  } else {
    for (int b = tid; b < kBins; b += kCT) sm.u.hist[b] = 0;
    __syncthreads();
    for_each_group<DT>(x, V, [&](int, const float (&v)[VEC], int n) {
      float q[VEC];
      divide_group(dv, v, q);
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        // one branch per entry: the mass is computed for every entry and cleared for a masked
        // entry or a lane past n
        const float d = vmax - q[j];
        const unsigned long long keep = 0ull - (unsigned long long)(j < n && !(v[j] < A));
        const unsigned long long m = mass_of(d) & keep;
        if (m) atomicAdd(&sm.u.hist[mass_bin(d)], m);
      }
    });
    __syncthreads();
    // Bins run from large v (bin 0) to small v, so the mass below a bin is a suffix sum.
    // Thread t owns bins [per t, per (t + 1)); the scan runs over reversed thread order.
    constexpr int per = kBins / kCT;
    unsigned long long s4 = 0;
    for (int j = 0; j < per; ++j) s4 += sm.u.hist[tid * per + j];
    const int rt = kCT - 1 - tid;
    sm.part[rt] = s4;
    __syncthreads();
    for (int off = 1; off < kCT; off <<= 1) {
      const unsigned long long add = rt >= off ? sm.part[rt - off] : 0ull;
      __syncthreads();
      sm.part[rt] += add;
      __syncthreads();
    }
    const unsigned long long incl = sm.part[rt];  // mass of bins >= per t
    const unsigned long long total = sm.part[kCT - 1];
    if (tid == 0) {
      sm.bcast[2] = 0;
      sm.bcast[3] = 0;
    }
    __syncthreads();
    const unsigned long long limit = scaled_floor(tl, total);
    if (limit >= total) {
      // every entry but the last of the order (v, index) is masked
      unsigned long long best = 0;
      for_each_entry<DT>(x, V, [&](int i, float v) {
        if (!(v < A)) {
          const unsigned long long key = ((unsigned long long)ordered_bits(divide(dv, v)) << 32) | (uint32_t)i;
          best = key > best ? key : best;
        }
      });
      best = wave_max_u64(best);
      if (lane_id() == 0) sm.red[wave_id()] = best;
      __syncthreads();
      for (int w = 0; w < kCW; ++w) best = sm.red[w] > best ? sm.red[w] : best;
      __syncthreads();
      fkey = best;
    } else {
      if (tid == 0) sm.count = 0;
      unsigned long long run = incl - s4;  // mass of bins >= per (t + 1)
      if (run <= limit && limit < incl) {
        for (int j = per - 1; j >= 0; --j) {
          const unsigned long long h = sm.u.hist[tid * per + j];
          if (run + h > limit) {
            sm.bcast[2] = (unsigned long long)(tid * per + j);
            sm.bcast[3] = run;
            break;
          }
          run += h;
        }
      }
      __syncthreads();
      const int bin = (int)sm.bcast[2];
      const unsigned long long base = sm.bcast[3];  // mass below the bin
      // the bin's entries as an interval of raw values (no divide or exp per entry), kept by
      // top-k too (x >= A)
      const float blo = fmaxf(min_x_in_bins(vmax, dv, bin), A);
      const float bhi = min_x_in_bins(vmax, dv, bin - 1);
      for_each_group<DT>(x, V, [&](int i0, const float (&v)[VEC], int n) {
        bool c[VEC];
#pragma unroll
        for (int j = 0; j < VEC; ++j) c[j] = (j < n) && v[j] >= blo && v[j] < bhi;
        append_group(c, [&](int j) {
          return ((unsigned long long)ordered_bits(divide(dv, v[j])) << 32) | (uint32_t)(i0 + j);
        }, sm);
      });
      __syncthreads();
      const int nb = sm.count;
      if (nb <= kCap) {
        sort_candidates(nb, sm);
        fkey = sm.u.cand[max(first_over(0, nb, base, limit, sm, [&](unsigned long long key) {
                               return mass_of(vmax - key_float((uint32_t)(key >> 32)));
                             }), 0)];
      } else {
        // Too many entries in one bin (long runs of equal values): bisection over the value
        // keys, then over the indices within the value, with exact sums per pass.
        const unsigned long long rem = limit - base;
        int64_t klo = -1, khi = 0xffffffffll;  // cum(klo) <= rem < cum(khi)
        unsigned long long cum_lo = 0;
        while (khi - klo > 1) {
          const int64_t mid = (klo + khi) / 2;
          unsigned long long c = 0;
          for_each_entry<DT>(x, V, [&](int, float v) {
            const float q = divide(dv, v);
            const float d = vmax - q;
            if (!(v < A) && mass_bin(d) == bin && ordered_bits(q) <= (uint32_t)mid) c += mass_of(d);
          });
          const unsigned long long cm = block_sum_u64(c, sm);
          if (cm > rem) {
            khi = mid;
          } else {
            klo = mid;
            cum_lo = cm;
          }
        }
        const uint32_t f_key = (uint32_t)khi;
        const unsigned long long mu = mass_of(vmax - key_float(f_key));
        const unsigned long long j = mu ? (rem - cum_lo) / mu : 0;  // entries of v_f masked
        int ilo = -1, ihi = V - 1;  // count(v_f, index <= ilo) <= j < count(v_f, index <= ihi)
        while (ihi - ilo > 1) {
          const int mid = (ilo + ihi) / 2;
          unsigned long long c = 0;
          for_each_entry<DT>(x, V, [&](int i, float v) {
            c += (i <= mid) & !(v < A) & (ordered_bits(divide(dv, v)) == f_key);
          });
          if (block_sum_u64(c, sm) > j) ihi = mid;
          else ilo = mid;
        }
        fkey = ((unsigned long long)f_key << 32) | (uint32_t)ihi;
      }
    }
  }
  const float vf = key_float((uint32_t)(fkey >> 32));
  A = min_x_reaching(vf, T);
  Bv = min_x_reaching(next_up(vf), T);
  J = (int)(uint32_t)fkey - 1;
  return true;
}

// WRITE = false: one row mask per verify row into p.masks.  WRITE = true (fp32 rows, no
// temperature): the masked entries of each row are set to -inf in place.
template <int DT, bool WRITE>
__global__ __launch_bounds__(kCT) void constraints_kernel(VerifyParams p) {
  __shared__ ConstraintSmem sm;
  __shared__ int s_row;
  int row = blockIdx.x;
  if (p.order) {
    // take this workgroup's entry of the plan, and clear it for the next call
    if (threadIdx.x == 0) {
      s_row = p.order[blockIdx.x] - 1;
      p.order[blockIdx.x] = 0;
    }
    __syncthreads();
    row = s_row;
    if (row < 0) return;
  }
  float A, Bv;
  int J;
  const bool any = row_thresholds<DT>(p, request_of(p, row), target_row(p, row), sm, A, Bv, J);
  if constexpr (!WRITE) {
    if (threadIdx.x == 0) p.masks[row] = make_float4(A, Bv, __int_as_float(J), 0.f);
  } else {
    if (!any) return;
    float* x = const_cast<float*>(static_cast<const float*>(p.target)) + target_row(p, row) * p.target_stride;
    const float4 m = make_float4(A, Bv, __int_as_float(J), 0.f);
    const int V = p.V;
    u32x4_align4* xv = reinterpret_cast<u32x4_align4*>(x);
    for_each_vector(xv, V / 4, [&](int vi, u32x4 r) {
      bool any_masked = false;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float v = __uint_as_float(r[j]);
        if (row_masked(m, v, vi * 4 + j) && v != -INFINITY) {
          r[j] = __float_as_uint(-INFINITY);
          any_masked = true;
        }
      }
      if (any_masked) xv[vi] = r;
    });
    const int i = V / 4 * 4 + (int)threadIdx.x;
    if (i < V && row_masked(m, x[i], i)) x[i] = -INFINITY;
  }
}

// ------------------------------------------------------------------ rows split over workgroups
// The same masks with each row's walks split over workgroups, for callers that bring scratch:
//   split_plan     one workgroup: lists the rows that need work (SplitRow) and writes the neutral
//                  mask of the others;
//   split_scan     one workgroup per (listed row, chunk of columns), the chunk in registers: the
//                  chunk's maximum (and, for greedy rows, how often it occurs), the largest entry of
//                  each group of 128, and for top-p rows a histogram of the masses over bins
//                  of 1/16 in v;
//   split_pick     one workgroup per listed row.  Rows with top-k: the k-th largest of the threads'
//                  largest groups bounds the k-th largest entry from below, so the entries that
//                  reach it (about k) are gathered from the groups whose maximum does, sorted, and
//                  top-k and top-p are read off them.  Rows with top-p alone: the merged histogram
//                  gives an interval of v that holds the first kept entry;
//   split_mass     one workgroup per (row, chunk) of the rows with top-p alone: the exact fixed-point
//                  mass of the chunk, of its entries below the interval, and the indices of those
//                  inside it;
//   split_finish   one workgroup per listed row: with the exact total, the first kept entry is
//                  found among the interval's entries.  The histogram only proposes the interval:
//                  the exact sums confirm that the crossing lies in it, and a row where it does
//                  not, or that does not fit (more than 4096 entries, k above 512), takes
//                  row_thresholds in this workgroup.
// (and split_apply where the rows themselves are masked in place).
// So a top-p row is read twice instead of three times, by as many workgroups as it has chunks.
// What bounds it: for a few rows the chain of five short kernels (8 bf16 rows of 151936 entries with
// top-p: 38 us a call, where the row kernel takes 71; the 32 rows of a step of 8 requests, half of
// them with top-k too, kernel by kernel under the profiler: plan 4 us, scan 8, pick 22, mass 12,
// finish 14); for many, the exponentials of scan and mass, about 30 VALU operations per entry each.

constexpr int kSplitThreads = 256;
constexpr int kSplitLong = 8192, kSplitShort = 2048;  // columns per chunk
constexpr int kSplitGroup = 128;                      // entries of a group
constexpr int kSplitMaxGroups = 4096;                 // of one row
constexpr int kSplitMaxChunks = 256;                  // of one row
constexpr int kSplitBins = 256;                       // 1/16 in v each, from the chunk's maximum down
constexpr float kSplitBinsPerUnit = 16.f;
constexpr int kSplitCopies = 4;                       // of a chunk's histogram, one per lane mod 4
constexpr int kSplitGrid = 2048;                      // workgroups of the scan and mass launches
constexpr int kSplitSub = kCT;                        // bins of the interval's entries

enum SplitMode : int { kSplitDone = 0, kSplitInterval = 1, kSplitTies = 2, kSplitGeneral = 3 };

struct SplitRow {
  int64_t xrow;   // row in the target tensor
  int row;        // mask written
  int k;          // top-k, or 0
  float t;        // 1 - top_p, or 0
  float T;        // temperature divisor
  int greedy;
  // from split_pick
  int mode;
  float x_lo, x_hi, vmax;
  uint32_t mkey;
  unsigned long long ties;
  int count;      // candidates listed by split_mass
  int req;        // request of the row
};
static_assert(sizeof(SplitRow) == 64, "row descriptor layout");

struct SplitHead {
  int rows;   // listed rows: first those with top-p alone
  int exact;  // rows with top-p alone
};

struct SplitParams {
  VerifyParams p;
  const int32_t* bonus_rows;  // [B] target row of each request's bonus row, mask P + r; or null
  int nch;
  SplitHead* head;
  SplitRow* rows;                // [P]
  float* cmax;                   // [P, nch]
  uint32_t* cties;               // [P, nch] greedy rows: entries at the chunk's maximum
  float* csum;                   // [P, nch] greedy rows: sum of exp(x - the chunk's maximum)
  uint32_t* gkeys;               // [P, nch, chunk / kSplitGroup]
  float* hist;                   // [P, nch, kSplitBins]
  unsigned long long* cmass;     // [P, nch, 2] total, below the interval
  uint32_t* cand;                // [P, kCap] column indices
};

// 0: the rows of request r need no work, 1: top-p alone, 2: top-k; with the request's parameters.
__device__ inline int split_class(const SplitParams& sp, int r, int& k, float& t, float& T,
                                  int& greedy) {
  const VerifyParams& p = sp.p;
  if (p.all_greedy) return 0;
  const int64_t kk = p.top_k ? p.top_k[r] : (int64_t)p.V;
  k = kk > 0 && kk < p.V ? (int)kk : 0;
  t = p.top_p ? fmaxf(1.0f - p.top_p[r], 0.f) : 0.f;  // p >= 1 (or NaN) keeps every entry
  const float temp = p.temperature ? p.temperature[r] : 1.f;
  greedy = p.temperature != nullptr && temp == 0.f;
  T = p.temperature && p.apply_temperature && !greedy ? temp : 1.f;
  if (k == 0 && !(t > 0.f)) return 0;
  if (greedy && !(t > 0.f)) return 0;
  return k > 0 ? 2 : 1;
}

__global__ __launch_bounds__(1024) void split_plan_kernel(SplitParams sp) {
  __shared__ int cnt[3];
  const VerifyParams& p = sp.p;
  const int tid = threadIdx.x;
  if (tid < 3) cnt[tid] = 0;
  __syncthreads();
  const float4 neutral = make_float4(-INFINITY, -INFINITY, __int_as_float(-1), 0.f);
  const int rows = p.cu ? (p.B > 0 ? min(max(p.cu[p.B - 1], 0), p.P) : 0) : min(p.B, p.P);
  for (int j = rows + tid; j < p.P; j += 1024) p.masks[j] = neutral;
  auto span = [&](int r, int& begin, int& end) {
    begin = p.cu ? max(r == 0 ? 0 : p.cu[r - 1], 0) : r;
    end = min(p.cu ? p.cu[r] : r + 1, p.P);
  };
  int k, greedy;
  float t, T;
  for (int r = tid; r < p.B; r += 1024) {
    int begin, end;
    span(r, begin, end);
    const int c = split_class(sp, r, k, t, T, greedy);
    const int n = max(end - begin, 0) + (sp.bonus_rows ? 1 : 0);
    if (c == 0) {
      for (int j = begin; j < end; ++j) p.masks[j] = neutral;
      if (sp.bonus_rows) p.masks[p.P + r] = neutral;
    } else if (n > 0) {
      atomicAdd(&cnt[c], n);
    }
  }
  __syncthreads();
  // the descriptors' room; cumulative counts that decrease would list a row more than once
  const int room = p.P + (sp.bonus_rows ? p.B : 0);
  const int exact = cnt[1];
  if (tid == 0) {
    sp.head->rows = min(exact + cnt[2], room);
    sp.head->exact = min(exact, room);
  }
  __syncthreads();
  if (tid < 3) cnt[tid] = tid == 2 ? exact : 0;
  __syncthreads();
  for (int r = tid; r < p.B; r += 1024) {
    int begin, end;
    span(r, begin, end);
    const int c = split_class(sp, r, k, t, T, greedy);
    const int n = max(end - begin, 0) + (sp.bonus_rows ? 1 : 0);
    if (c == 0 || n == 0) continue;
    const int at = atomicAdd(&cnt[c], n);
    for (int u = 0; u < n && at + u < room; ++u) {
      const int j = begin + u;
      SplitRow d{};
      d.row = j < end ? j : p.P + r;
      d.xrow = j < end ? target_row(p, j) : clamped_row(p, sp.bonus_rows[r]);
      d.req = r;
      d.k = k;
      d.t = t;
      d.T = T;
      d.greedy = greedy;
      sp.rows[at + u] = d;
    }
  }
}

// A chunk's entries in registers: columns c0 + j * kSplitThreads * VEC + e.  Entries past the row's
// end (in its last vectors, those that load_vec_inside moved back) hold `pad`; col(j, e) is -1.
template <int DT, int NV>
struct SplitChunk {
  static constexpr int VEC = Elem<DT>::kVec;
  static constexpr int CH = NV * kSplitThreads * VEC;
  // a group: the entries of this many consecutive lanes (4 or 16)
  static constexpr int kGroupLanes = kSplitGroup / (NV * VEC);
  static constexpr int kGroups = CH / kSplitGroup;
  float v[NV][VEC];
  int c0, V;
  __device__ inline void load(const typename Elem<DT>::storage* x, int c, int V_, float pad) {
    V = V_;
    c0 = c * CH + (int)threadIdx.x * VEC;
    u32x4 q[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j)
      q[j] = load_vec_inside<DT>(x, c0 + j * kSplitThreads * VEC, V);
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
      for (int e = 0; e < VEC; ++e) v[j][e] = vec_elem<DT>(q[j], e);
    if ((c + 1) * CH > V) {
#pragma unroll
      for (int j = 0; j < NV; ++j)
#pragma unroll
        for (int e = 0; e < VEC; ++e) v[j][e] = col(j, e) < 0 ? pad : v[j][e];
    }
  }
  __device__ inline int col(int j, int e) const {
    return inside_col<DT>(c0 + j * kSplitThreads * VEC, e, V);
  }
};

// The maximum over each group's lanes, in every one of them.
template <int LANES>
__device__ inline float group_max(float v) {
  static_assert(LANES == 4 || LANES == 16, "DPP quads or rows");
  v = fmaxf(v, dpp_f32<kDppXor1>(v));
  v = fmaxf(v, dpp_f32<kDppXor2>(v));
  if constexpr (LANES == 16) {
    v = fmaxf(v, dpp_f32<kDppHalfMirror>(v));
    v = fmaxf(v, dpp_f32<kDppMirror>(v));
  }
  return v;
}

template <int DT, int NV>
__global__ __launch_bounds__(kSplitThreads) void split_scan_kernel(SplitParams sp) {
  using S = typename Elem<DT>::storage;
  constexpr int VEC = Elem<DT>::kVec;
  constexpr int NW = kSplitThreads / kWave;
  __shared__ float s_max[NW];
  __shared__ uint32_t s_ties[NW];
  __shared__ float s_sum[NW];
  // 64-bit integer sums (ds_add_u64): LDS float atomics took about 4 cycles per lane, which made
  // this kernel 229 us long where a read of its rows takes 40.  The copies keep lanes of one wave
  // that meet in a bin from queueing.
  __shared__ __align__(16) unsigned long long s_hist[kSplitBins * kSplitCopies];
  const int items = sp.head->rows * sp.nch;
  // listed rows are few in most calls: a bounded grid, since 38,000 workgroups that find nothing
  // to do took 50 us to dispatch
  for (int item = blockIdx.x; item < items; item += gridDim.x) {
    const int i = item / sp.nch, c = item - i * sp.nch;
    const SplitRow& d = sp.rows[i];
    const int tid = threadIdx.x;
    const bool hist = d.k == 0 && !d.greedy;
    const S* x = static_cast<const S*>(sp.p.target) + d.xrow * sp.p.target_stride;
    SplitChunk<DT, NV> ch;
    ch.load(x, c, sp.p.V, -INFINITY);
    if (hist) {
#pragma unroll
      for (int u = 0; u < kSplitCopies; ++u) s_hist[u * kSplitThreads + tid] = 0;
    }
    float m = -INFINITY, odd = 0.f;  // NaN when an entry is NaN or infinite
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        m = fmaxf(m, ch.v[j][e]);
        odd = fmaf(ch.v[j][e], 0.f, odd);
      }
    using Chunk = SplitChunk<DT, NV>;
    const float g = group_max<Chunk::kGroupLanes>(m);
    uint32_t key = ordered_bits(g);
    if (__ballot(odd != odd) != 0) {  // a group with a NaN has the NaN key
      float nan = 0.f;
#pragma unroll
      for (int j = 0; j < NV; ++j)
#pragma unroll
        for (int e = 0; e < VEC; ++e) nan = ch.v[j][e] != ch.v[j][e] ? 1.f : nan;
      key = group_max<Chunk::kGroupLanes>(nan) != 0.f ? kNanKey : key;
    }
    const float wm = wave_max(m);
    if (lane_id() == 0) s_max[wave_id()] = wm;
    const int64_t slot = (int64_t)i * sp.nch + c;
    if (tid % Chunk::kGroupLanes == 0)
      sp.gkeys[slot * Chunk::kGroups + tid / Chunk::kGroupLanes] = key;
    __syncthreads();
    float M = s_max[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) M = fmaxf(M, s_max[w]);
    if (tid == 0) sp.cmax[slot] = M;
    if (d.greedy) {
      // greedy rows are not divided: T = 1
      uint32_t ties = 0;
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < NV; ++j)
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          ties += ch.v[j][e] == M;
          sum += __builtin_amdgcn_exp2f((ch.v[j][e] - M) * kLog2e);
        }
      sum = wave_sum(sum);
      for (int off = kWave / 2; off > 0; off >>= 1) ties += __shfl_xor(ties, off);
      if (lane_id() == 0) {
        s_ties[wave_id()] = ties;
        s_sum[wave_id()] = sum;
      }
      __syncthreads();
      if (tid == 0) {
        ties = 0;
        sum = 0.f;
        for (int w = 0; w < NW; ++w) {
          ties += s_ties[w];
          sum += s_sum[w];
        }
        sp.cties[slot] = ties;
        sp.csum[slot] = sum;
      }
    }
    if (hist) {
      if (M > -INFINITY && M < INFINITY) {
        const float c1 = kLog2e / d.T, per = kSplitBinsPerUnit / d.T;
        const float base = floorf(M * per);
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
          for (int e = 0; e < VEC; ++e) {
            const float w = __builtin_amdgcn_exp2f((ch.v[j][e] - M) * c1);
            const float b = fminf(base - floorf(ch.v[j][e] * per), (float)(kSplitBins - 1));
            const uint32_t mass = (uint32_t)fmaxf(w * 0x1p31f, 0.f);  // 0 for a NaN entry
            if (mass)
              atomicAdd(&s_hist[(int)b * kSplitCopies + (tid & (kSplitCopies - 1))],
                        (unsigned long long)mass);
          }
      }
      __syncthreads();
      unsigned long long sum = 0;
#pragma unroll
      for (int u = 0; u < kSplitCopies; ++u) sum += s_hist[tid * kSplitCopies + u];
      sp.hist[slot * kSplitBins + tid] = (float)sum * 0x1p-31f;
    }
    __syncthreads();  // the next item reuses the shared arrays
  }
}

struct SplitPickSmem {
  ConstraintSmem c;
  float hist[kSplitBins];
  float weight[kSplitMaxChunks];  // per chunk: exp(its maximum - the row's)
  int shift[kSplitMaxChunks];       // and its first bin in the row's bins
  __align__(16) uint32_t tkey[kCT];
  uint32_t theta;
  int groups;
};

// Top-k and, with t > 0, top-p over the gathered entries cand[0, n): every entry that can be among
// the k largest values, and all entries of each of its values.
__device__ inline bool candidate_thresholds(int n, int k, float t, float T, ConstraintSmem& sm,
                                            float& A, float& Bv, int& J) {
  const int tid = threadIdx.x;
  sort_candidates(n, sm);
  const uint32_t vk_key = (uint32_t)(sm.u.cand[max(n - k, 0)] >> 32);
  int below = 0;
  for (int i = tid; i < n; i += kCT) below += (uint32_t)(sm.u.cand[i] >> 32) < vk_key;
  const int lo_k = (int)block_sum_u64((unsigned long long)below, sm);
  // A NaN k-th value compares false with everything: the reference then masks nothing.
  if (vk_key != kNanKey) A = min_x_reaching(key_float(vk_key), T);
  const float vmax = key_float((uint32_t)(sm.u.cand[max(n - 1, 0)] >> 32));
  if (!(t > 0.f) || vmax != vmax || fabsf(vmax) == INFINITY) return A != -INFINITY;
  unsigned long long seg = 0;
  for (int i = lo_k + tid; i < n; i += kCT)
    seg += mass_of(vmax - key_float((uint32_t)(sm.u.cand[i] >> 32)));
  const unsigned long long total = block_sum_u64(seg, sm);
  const int f = first_over(lo_k, n, 0, scaled_floor(fminf(t, 1.f), total), sm,
                           [&](unsigned long long key) {
                             return mass_of(vmax - key_float((uint32_t)(key >> 32)));
                           });
  const unsigned long long fkey = sm.u.cand[max(f, 0)];
  const float vf = key_float((uint32_t)(fkey >> 32));
  A = min_x_reaching(vf, T);
  Bv = min_x_reaching(next_up(vf), T);
  J = (int)(uint32_t)fkey - 1;
  return true;
}

template <int DT, int NV>
__global__ __launch_bounds__(kCT) void split_pick_kernel(SplitParams sp) {
  using S = typename Elem<DT>::storage;
  constexpr int VEC = Elem<DT>::kVec;
  constexpr int CH = NV * kSplitThreads * VEC;
  __shared__ SplitPickSmem sm;
  extern __shared__ uint16_t s_glist[];  // [groups of a row]
  const int i = blockIdx.x;
  if (i >= sp.head->rows) return;
  SplitRow& d = sp.rows[i];
  const int tid = threadIdx.x, nch = sp.nch, V = sp.p.V;
  const int64_t slot0 = (int64_t)i * nch;
  const int k = d.k;
  const float t = d.t, T = d.T;
  const Divider dv = make_divider(T);
  const S* x = static_cast<const S*>(sp.p.target) + d.xrow * sp.p.target_stride;
  auto done = [&](float A, float Bv, int J) {
    if (tid == 0) {
      sp.p.masks[d.row] = make_float4(A, Bv, __int_as_float(J), 0.f);
      d.mode = kSplitDone;
    }
  };
  using Chunk = SplitChunk<DT, NV>;
  constexpr int GL = Chunk::kGroupLanes, kGroups = Chunk::kGroups;
  const int ng = nch * kGroups;
  constexpr int kPerThread = kSplitMaxGroups / kCT;
  uint32_t gk[kPerThread], top = 0;
#pragma unroll
  for (int u = 0; u < kPerThread; ++u) {
    gk[u] = u * kCT + tid < ng ? sp.gkeys[slot0 * kGroups + u * kCT + tid] : 0u;
    top = max(top, gk[u]);
  }
  if (tid == 0) {
    sm.theta = 0xffffffffu;
    sm.groups = sm.c.count = 0;
  }
  sm.tkey[tid] = top;
  const uint32_t mkey = block_max_u32(top, sm.c);
  const float cm = tid < nch ? sp.cmax[slot0 + tid] : -INFINITY;
  if (d.greedy) {
    // only the argmax matters (row_thresholds): a tied maximum that top-p can reach
    const float M = key_float(mkey);
    const unsigned long long ties = block_sum_u64(
        tid < nch && cm == M ? (unsigned long long)sp.cties[slot0 + tid] : 0ull, sm.c);
    const float vmax = divide(dv, M);
    if (mkey == kNanKey || ties < 2 || (k == 0 && fabsf(vmax) == INFINITY)) {
      done(-INFINITY, -INFINITY, -1);
      return;
    }
    if (k == 0) {
      // The first maximum stays when the mass up to and including it passes the limit
      // (split_finish decides that exactly).  The float sums settle it for most rows.  A sum of
      // positive terms is off by at most 1e-5 of itself (about 60 roundings of 2^-24 in a row,
      // and those of the exponents), so `below`, the sum less the ties, by 1e-5 of the sum: much of
      // it where nearly all of the mass is ties.  The fixed-point masses lose below 2^-40 each.
      float sum[1] = {tid < nch && cm > -INFINITY
                          ? sp.csum[slot0 + tid] * __builtin_amdgcn_exp2f((cm - M) * kLog2e)
                          : 0.f};
      block_sum<1, kCW>(sum, reinterpret_cast<float*>(sm.c.part));
      const float below = fmaxf(sum[0] - (float)ties - 1e-5f * sum[0], 0.f);
      if (t * sum[0] * 1.001f < below * 0.999f + 0.999f) {
        done(-INFINITY, -INFINITY, -1);
        return;
      }
      if (tid == 0) {
        d.x_lo = M;
        d.x_hi = INFINITY;
        d.vmax = vmax;
        d.mkey = mkey;
        d.ties = ties;
        d.mode = kSplitTies;
      }
      return;
    }
  }
  if (k > 0) {
    if (k > kCT) {
      if (tid == 0) d.mode = kSplitGeneral;
      return;
    }
    int above = 0;
    const uint4* keys = reinterpret_cast<const uint4*>(sm.tkey);
#pragma unroll 8
    for (int j = 0; j < kCT / 4; ++j) {
      const uint4 o = keys[j];
      above += (o.x > top) + (o.y > top) + (o.z > top) + (o.w > top);
    }
    if (above < k) atomicMin(&sm.theta, top);  // the k-th largest is the smallest such key
    __syncthreads();
    // every entry whose v reaches fl(theta / T) (x >= floor) is a candidate; theta 0: fewer than
    // k threads hold groups; a NaN theta: everything is
    const uint32_t theta = sm.theta;
    const float floor_x = theta == 0 ? -INFINITY
                          : theta == kNanKey ? NAN
                                             : min_x_reaching(divide(dv, key_float(theta)), T);
#pragma unroll
    for (int u = 0; u < kPerThread; ++u)
      if (u * kCT + tid < ng && (gk[u] == kNanKey || !(key_float(gk[u]) < floor_x)))
        s_glist[atomicAdd(&sm.groups, 1)] = (uint16_t)(u * kCT + tid);
    __syncthreads();
    const int nl = sm.groups;
    for (int b = 0; b < nl; b += kCT / GL) {
      const int li = b + tid / GL;
      const bool on = li < nl;
      const int g = on ? s_glist[li] : 0;
      // what the scan's lanes GL (g % kGroups) .. of chunk g / kGroups held
      const int c0 = (g / kGroups) * CH + ((g % kGroups) * GL + tid % GL) * VEC;
      u32x4 q[NV];
#pragma unroll
      for (int j = 0; j < NV; ++j) q[j] = load_vec_inside<DT>(x, c0 + j * kSplitThreads * VEC, V);
#pragma unroll
      for (int j = 0; j < NV; ++j) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          const int col = inside_col<DT>(c0 + j * kSplitThreads * VEC, e, V);
          const float v = vec_elem<DT>(q[j], e);
          const bool take = on && col >= 0 && !(v < floor_x);
          if (__ballot(take) == 0) continue;
          append(take, take ? (((unsigned long long)ordered_bits(divide(dv, v)) << 32) | (uint32_t)col)
                            : 0ull, sm.c);
        }
      }
    }
    __syncthreads();
    const int n = sm.c.count;
    if (n > kCap) {
      if (tid == 0) d.mode = kSplitGeneral;
      return;
    }
    float A = -INFINITY, Bv = -INFINITY;
    int J = -1;
    candidate_thresholds(n, k, mkey == kNanKey ? 0.f : t, T, sm.c, A, Bv, J);
    done(A, Bv, J);
    return;
  }
  // ---- top-p alone: the interval of v that holds the first kept entry ----
  const float M = key_float(mkey);
  const float vmax = divide(dv, M);
  if (mkey == kNanKey || vmax != vmax || fabsf(vmax) == INFINITY) {
    done(-INFINITY, -INFINITY, -1);
    return;
  }
  const float c1 = kLog2e / T, per = kSplitBinsPerUnit / T;
  const float base = floorf(M * per);
  {
    // merge the chunks' histograms: row bin b is chunk bin b - (base - the chunk's base); what
    // lies past the row's last bin counts there
    constexpr int U = 8, step = kCT / kSplitBins, last = kSplitBins - 1;
    if (tid < nch) {
      const bool on = cm > -INFINITY;
      sm.weight[tid] = on ? __builtin_amdgcn_exp2f((cm - M) * c1) : 0.f;
      sm.shift[tid] = on ? (int)fminf(base - floorf(cm * per), (float)kSplitBins) : kSplitBins;
    }
    __syncthreads();
    const int b = tid & last;
    float acc = 0.f, tail[1] = {0.f};
    for (int c0 = tid / kSplitBins; c0 < nch; c0 += U * step) {
      float h[U], own[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = c0 + u * step, cc = min(c, nch - 1), o = sm.shift[cc];
        const float* hc = sp.hist + (slot0 + cc) * kSplitBins;
        h[u] = hc[max(b - o, 0)];
        own[u] = hc[b];
        h[u] *= c < nch && b < last && b >= o ? sm.weight[cc] : 0.f;
        own[u] *= c < nch && b + o >= last ? sm.weight[cc] : 0.f;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        acc += h[u];
        tail[0] += own[u];
      }
    }
    float* half = reinterpret_cast<float*>(sm.tkey);
    half[tid] = acc;
    block_sum<1, kCW>(tail, reinterpret_cast<float*>(sm.c.part));
    if (tid < kSplitBins)
      sm.hist[tid] = tid == last ? tail[0] : half[tid] + half[tid + kSplitBins];
  }
  __syncthreads();
  if (tid < kWave) {
    // lane l holds bins 255 - 4 l .. 252 - 4 l, the smallest values first
    float h[4], own = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      h[j] = sm.hist[kSplitBins - 1 - 4 * tid - j];
      own += h[j];
    }
    float incl = own;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const float a = __shfl_up(incl, off);
      if (tid >= off) incl += a;
    }
    const float limit = fminf(t, 1.f) * readlane_f32(incl, kWave - 1);
    // the bins where the running mass passes the limit, less and more its rounding; none: bin 0
    auto bin_over = [&](float lim) {
      float run = incl - own;
      int at = -1;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        run += h[j];
        if (at < 0 && run > lim) at = kSplitBins - 1 - 4 * tid - j;
      }
      const unsigned long long mask = __ballot(at >= 0);
      return mask ? __shfl(at, __ffsll((long long)mask) - 1) : 0;
    };
    const int j_lo = bin_over(limit * (1.f - 1e-4f)), j_hi = bin_over(limit * (1.f + 1e-4f));
    // bin j holds v in [base - j, base - j + 1) / 16, up to the rounding of v
    auto edge = [&](float e, float sign) {
      const float v = e / kSplitBinsPerUnit;
      return v + sign * (fabsf(v) * 0x1p-20f + 0x1p-30f);
    };
    const float v_lo = edge(base - (float)j_lo, -1.f), v_hi = edge(base - (float)j_hi + 1.f, 1.f);
    // two bisections side by side
    const float r = min_x_reaching(tid == 0 ? v_lo : v_hi, T);
    const float x_lo = readlane_f32(r, 0), x_hi = readlane_f32(r, 1);
    if (tid == 0) {
      d.x_lo = j_lo == kSplitBins - 1 ? -INFINITY : x_lo;
      d.x_hi = j_hi == 0 ? INFINITY : x_hi;
      d.vmax = vmax;
      d.mkey = mkey;
      d.mode = kSplitInterval;
    }
  }
}

template <int DT, int NV>
__global__ __launch_bounds__(kSplitThreads) void split_mass_kernel(SplitParams sp) {
  using S = typename Elem<DT>::storage;
  constexpr int VEC = Elem<DT>::kVec;
  constexpr int NW = kSplitThreads / kWave;
  __shared__ unsigned long long s_total[NW], s_below[NW];
  __shared__ int s_n[NW], s_base;
  const int items = sp.head->exact * sp.nch;
  for (int item = blockIdx.x; item < items; item += gridDim.x) {
    const int i = item / sp.nch, c = item - i * sp.nch;
    SplitRow& d = sp.rows[i];
    const int mode = d.mode;
    if (mode != kSplitInterval && mode != kSplitTies) continue;
    __syncthreads();  // the item before is done with the shared arrays
    const int tid = threadIdx.x;
    const float x_lo = d.x_lo, x_hi = d.x_hi, vmax = d.vmax;
    const S* x = static_cast<const S*>(sp.p.target) + d.xrow * sp.p.target_stride;
    SplitChunk<DT, NV> ch;
    // a column past the row holds NaN: its mass is 0, and it is in no interval
    ch.load(x, c, sp.p.V, NAN);
    int n = 0;  // candidates of this lane
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
      for (int e = 0; e < VEC; ++e) n += (ch.v[j][e] >= x_lo) & (ch.v[j][e] < x_hi);
    const int mine = n;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const int a = __shfl_up(n, off);
      n += lane_id() >= off ? a : 0;
    }
    const int wid = wave_id();
    if (lane_id() == kWave - 1) s_n[wid] = n;
    __syncthreads();
    int base = 0, all = 0;
    for (int w = 0; w < NW; ++w) {
      base += w < wid ? s_n[w] : 0;
      all += s_n[w];
    }
    // the place in the row's list is asked for here and used after the masses
    int place = 0;
    if (tid == 0 && all > 0) place = atomicAdd(&d.count, all);
    const Divider dv = make_divider(d.T);
    unsigned long long total = 0, below = 0;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      float q[VEC];
      divide_group(dv, ch.v[j], q);
      float e40[VEC], top = 0.f;
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        e40[e] = mass_exp(vmax - q[e]) * 0x1p40f;
        top = fmaxf(top, e40[e]);
      }
      // entries more than 8 ln 2 below the maximum have masses below 2^32: the plain conversion
      if (__ballot(!(top < 0x1p32f)) == 0) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          const uint32_t m = (uint32_t)fmaxf(e40[e], 0.f);  // 0 for NaN
          total += m;
          below += ch.v[j][e] < x_lo ? m : 0u;
        }
      } else {
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          const unsigned long long m = e40[e] > 0.f ? mass_from_e(e40[e] * 0x1p-40f) : 0ull;
          total += m;
          below += ch.v[j][e] < x_lo ? m : 0ull;
        }
      }
    }
    total = wave_sum_u64(total);
    below = wave_sum_u64(below);
    if (lane_id() == 0) {
      s_total[wid] = total;
      s_below[wid] = below;
    }
    if (tid == 0) s_base = place;
    __syncthreads();
    if (tid == 0) {
      unsigned long long* out = sp.cmass + ((int64_t)i * sp.nch + c) * 2;
      total = below = 0;
      for (int w = 0; w < NW; ++w) {
        total += s_total[w];
        below += s_below[w];
      }
      out[0] = total;
      out[1] = below;
    }
    if (mine == 0) continue;  // this lane lists nothing
    int at = s_base + base + n - mine;
    uint32_t* cand = sp.cand + (int64_t)i * kCap;
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
      for (int e = 0; e < VEC; ++e)
        if (ch.v[j][e] >= x_lo && ch.v[j][e] < x_hi) {
          if (at < kCap) cand[at] = (uint32_t)ch.col(j, e);
          ++at;
        }
  }
}

template <int DT>
__global__ __launch_bounds__(kCT) void split_finish_kernel(SplitParams sp) {
  using S = typename Elem<DT>::storage;
  __shared__ ConstraintSmem sm;
  __shared__ unsigned long long s_sums[kCW][3];
  __shared__ uint32_t s_ends[kCW][2];
  const int i = blockIdx.x;
  if (i >= sp.head->rows) return;
  const SplitRow& d = sp.rows[i];
  const int mode = d.mode;
  if (mode == kSplitDone) return;
  const int tid = threadIdx.x;
  auto write = [&](float A, float Bv, int J) {
    if (tid == 0) sp.p.masks[d.row] = make_float4(A, Bv, __int_as_float(J), 0.f);
  };
  const int n = d.count;
  bool general = mode == kSplitGeneral || n > kCap;
  if (!general) {
    const float T = d.T, vmax = d.vmax;
    const Divider dv = make_divider(T);
    const S* x = static_cast<const S*>(sp.p.target) + d.xrow * sp.p.target_stride;
    unsigned long long total = 0, below = 0;
    for (int c = tid; c < sp.nch; c += kCT) {
      const unsigned long long* m = sp.cmass + ((int64_t)i * sp.nch + c) * 2;
      total += m[0];
      below += m[1];
    }
    // the interval's entries: at most kCap / kCT per thread
    constexpr int PER = kCap / kCT;
    uint32_t col[PER], key[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int at = u * kCT + tid;
      col[u] = at < n ? sp.cand[(int64_t)i * kCap + at] : 0u;
    }
#pragma unroll
    for (int u = 0; u < PER; ++u)
      key[u] = u * kCT + tid < n ? ordered_bits(divide(dv, Elem<DT>::cvt(x[col[u]]))) : 0u;
    unsigned long long inside = 0;
    uint32_t lo = 0xffffffffu, hi = 0;
#pragma unroll
    for (int u = 0; u < PER; ++u)
      if (u * kCT + tid < n) {
        inside += mass_of(vmax - key_float(key[u]));
        lo = min(lo, key[u]);
        hi = max(hi, key[u]);
      }
    // the sums over the block, behind one barrier
    total = wave_sum_u64(total);
    below = wave_sum_u64(below);
    inside = wave_sum_u64(inside);
    lo = ~wave_max_u32(~lo);
    hi = wave_max_u32(hi);
    if (lane_id() == 0) {
      s_sums[wave_id()][0] = total;
      s_sums[wave_id()][1] = below;
      s_sums[wave_id()][2] = inside;
      s_ends[wave_id()][0] = lo;
      s_ends[wave_id()][1] = hi;
    }
    for (int b = tid; b < kSplitSub; b += kCT) sm.u.hist[b] = 0;
    if (tid == 0) sm.count = 0;
    __syncthreads();
    total = below = inside = 0;
    for (int w = 0; w < kCW; ++w) {
      total += s_sums[w][0];
      below += s_sums[w][1];
      inside += s_sums[w][2];
      lo = min(lo, s_ends[w][0]);
      hi = max(hi, s_ends[w][1]);
    }
    const unsigned long long limit = scaled_floor(fminf(d.t, 1.f), total);
    if (mode == kSplitTies) {
      // greedy_tied_top_p: each tied entry has mass 2^40
      constexpr unsigned long long kUnit = 1ull << 40;
      if (limit < below + kUnit) {
        write(-INFINITY, -INFINITY, -1);
        return;
      }
      const unsigned long long m = min((limit - below) / kUnit, d.ties - 1);
      __syncthreads();
#pragma unroll
      for (int u = 0; u < PER; ++u)
        if (u * kCT + tid < n)
          sm.u.cand[u * kCT + tid] = ((unsigned long long)key[u] << 32) | col[u];
      __syncthreads();
      sort_candidates(n, sm);
      const int i_f = (int)(uint32_t)sm.u.cand[min((int)m, n - 1)];
      write(min_x_reaching(vmax, T), min_x_reaching(next_up(vmax), T), i_f - 1);
      return;
    }
    const bool last = limit >= total;  // every entry but the last of the order is masked
    general = n == 0 || (last ? d.x_hi != INFINITY : limit < below || limit >= below + inside);
    if (!general) {
      // equal parts of the interval's keys: their masses, then the part where the mass passes
      const float scale = (float)kSplitSub / ((float)(hi - lo) + 1.f);
      auto sub_of = [&](uint32_t kk) {
        return min((int)((float)(kk - lo) * scale), kSplitSub - 1);  // non-decreasing in kk
      };
      int sub[PER];
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        sub[u] = -1;
        if (u * kCT + tid < n) {
          sub[u] = sub_of(key[u]);
          atomicAdd(&sm.u.hist[sub[u]], mass_of(vmax - key_float(key[u])));
        }
      }
      __syncthreads();
      const unsigned long long h = sm.u.hist[tid];
      if (tid == 0) {
        sm.bcast[2] = (unsigned long long)sub_of(hi);  // last: the part of the largest key
        sm.bcast[3] = below;
      }
      const unsigned long long incl = below + block_scan_u64(h, sm);
      if (!last && incl - h <= limit && limit < incl) {
        sm.bcast[2] = (unsigned long long)tid;
        sm.bcast[3] = incl - h;
      }
      __syncthreads();
      const int part = (int)sm.bcast[2];
      const unsigned long long base = sm.bcast[3];
#pragma unroll
      for (int u = 0; u < PER; ++u)
        append(sub[u] == part, ((unsigned long long)key[u] << 32) | col[u], sm);
      __syncthreads();
      const int np = sm.count;
      sort_candidates(np, sm);
      const int f = last ? np - 1
                         : first_over(0, np, base, limit, sm, [&](unsigned long long kk) {
                             return mass_of(vmax - key_float((uint32_t)(kk >> 32)));
                           });
      const unsigned long long fkey = sm.u.cand[max(f, 0)];
      const float vf = key_float((uint32_t)(fkey >> 32));
      write(min_x_reaching(vf, T), min_x_reaching(next_up(vf), T), (int)(uint32_t)fkey - 1);
      return;
    }
  }
  float A, Bv;
  int J;
  __syncthreads();
  row_thresholds<DT>(sp.p, d.req, d.xrow, sm, A, Bv, J);
  write(A, Bv, J);
}

// The masked entries of fp32 rows become -inf, one workgroup per (row, chunk); rows without a mask
// are not touched.
__global__ __launch_bounds__(kSplitThreads) void split_apply_kernel(SplitParams sp) {
  constexpr int NV = kSplitLong / (kSplitThreads * 4);
  const int nch = (sp.p.V + kSplitLong - 1) / kSplitLong;
  const int i = blockIdx.x / nch, c = blockIdx.x - i * nch;
  if (i >= sp.head->rows) return;
  const SplitRow& d = sp.rows[i];
  const float4 m = sp.p.masks[d.row];
  if (m.x == -INFINITY && m.y == -INFINITY) return;
  float* x = const_cast<float*>(static_cast<const float*>(sp.p.target)) + d.xrow * sp.p.target_stride;
  SplitChunk<MVSD_F32, NV> ch;
  ch.load(x, c, sp.p.V, -INFINITY);
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    bool any = false;
    u32x4 out;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float v = ch.v[j][e];
      const bool mask = row_masked(m, v, ch.col(j, e)) && v != -INFINITY;
      any |= mask;
      out[e] = __float_as_uint(mask ? -INFINITY : v);
    }
    if (!any) continue;
    const int col = ch.c0 + j * kSplitThreads * 4;
    if (col + 4 <= sp.p.V) {
      *reinterpret_cast<u32x4_align4*>(x + col) = out;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (ch.col(j, e) >= 0) x[ch.col(j, e)] = __uint_as_float(out[e]);
    }
  }
}

int split_chunk(int64_t rows, int64_t V) {
  // 2048 columns while chunks of 8192 would be about one workgroup per compute unit.  Top-p bf16 rows
  // of 151936 entries, short / long chunks: 8 rows 38 / 35 us, 16 rows 44 / 40, 32 rows 56 / 42; of
  // 65536: 8 rows 28 / 31, 32 rows 33 / 32, 64 rows 41 / 35.  Half greedy, a quarter top-k, a quarter
  // top-p, of 151936: 40 / 45, 42 / 45, 46 / 46 and 64 rows 55 / 49; of 65536: 36 / 42, 36 / 43 (32
  // rows) and 39 / 43.
  return rows * ((V + kSplitLong - 1) / kSplitLong) < 300 &&
                 (V + kSplitShort - 1) / kSplitShort <= kSplitMaxChunks
             ? kSplitShort
             : kSplitLong;
}

struct SplitLayout {
  int chunk, nch;
  int64_t head, rows, cmax, cties, csum, gkeys, hist, cmass, cand, masks, total;
};

// Whether a call's rows are split: few of them and long ones, with their groups in LDS.  With many
// rows every compute unit has rows of its own, and the row kernel, which takes one exponential per
// entry instead of two, is as fast: top-p rows of 151936 bf16 entries took 71 us (row kernel)
// against 38 (split) for 8 rows, 75 / 49 for 64, 77 / 68 for 128, 78 / 82 for 192 and 112 / 165 for
// 512; half greedy, a quarter top-k, a quarter top-p: 75 / 60 for 128, 78 / 77 for 256.  On short
// rows the chain of launches is the longer one for batches of every class: those mixed rows took
// 42 / 37 us for 16 rows of 65536 entries and 42 / 43 for 64, but 36 / 36 and 37 / 45 of 50257 and 30 /
// 36 and 30 / 37 of 32000 (top-p rows alone still gain there for few rows: 37 / 30 for 16 of 50257, 30 /
// 28 of 32000).
constexpr int64_t kSplitRows = 128, kSplitMinV = 65536;
bool split_rows(int64_t P, int64_t V) {
  const int64_t chunk = split_chunk(P, V), nch = (V + chunk - 1) / chunk;
  return P <= kSplitRows && V >= kSplitMinV && nch * (chunk / kSplitGroup) <= kSplitMaxGroups;
}

SplitLayout split_layout(int64_t P, int64_t V) {
  SplitLayout l;
  l.chunk = split_chunk(P, V);
  l.nch = (int)((V + l.chunk - 1) / l.chunk);
  int64_t off = 0;
  const int64_t slots = P * l.nch;
  auto take = [&](int64_t bytes) {
    const int64_t at = off;
    off += (bytes + 255) / 256 * 256;
    return at;
  };
  l.head = take(sizeof(SplitHead));
  l.rows = take(P * (int64_t)sizeof(SplitRow));
  l.cmax = take(slots * 4);
  l.cties = take(slots * 4);
  l.csum = take(slots * 4);
  l.gkeys = take(slots * (l.chunk / kSplitGroup) * 4);
  l.hist = take(slots * kSplitBins * 4);
  l.cmass = take(slots * 16);
  l.cand = take(P * (int64_t)kCap * 4);
  l.masks = take(P * 16);
  l.total = off;
  return l;
}

template <int DT>
void launch_split_dt(const SplitParams& sp, int chunk, hipStream_t stream) {
  constexpr int kLong = kSplitLong / (kSplitThreads * Elem<DT>::kVec);
  constexpr int kShort = kSplitShort / (kSplitThreads * Elem<DT>::kVec);
  const int64_t n = sp.p.P + (sp.bonus_rows ? sp.p.B : 0), items = n * sp.nch;
  const dim3 rows((unsigned)n), slots((unsigned)(items < kSplitGrid ? items : kSplitGrid));
  const dim3 block(kSplitThreads), wide(kCT);
  const unsigned lds = (unsigned)sp.nch * (unsigned)(chunk / kSplitGroup) * 2;
  if (chunk == kSplitLong) {
    hipLaunchKernelGGL((split_scan_kernel<DT, kLong>), slots, block, 0, stream, sp);
    hipLaunchKernelGGL((split_pick_kernel<DT, kLong>), rows, wide, lds, stream, sp);
    hipLaunchKernelGGL((split_mass_kernel<DT, kLong>), slots, block, 0, stream, sp);
  } else {
    hipLaunchKernelGGL((split_scan_kernel<DT, kShort>), slots, block, 0, stream, sp);
    hipLaunchKernelGGL((split_pick_kernel<DT, kShort>), rows, wide, lds, stream, sp);
    hipLaunchKernelGGL((split_mass_kernel<DT, kShort>), slots, block, 0, stream, sp);
  }
  hipLaunchKernelGGL((split_finish_kernel<DT>), rows, wide, 0, stream, sp);
}

}  // namespace

int64_t split_constraints_bytes(int64_t rows, int64_t V) {
  return rows > 0 && V > 0 && split_rows(rows, V) ? split_layout(rows, V).total : 0;
}

hipError_t launch_split_constraints(const VerifyParams& params, int target_dtype,
                                    const int32_t* bonus_rows, bool apply, void* scratch,
                                    hipStream_t stream) {
  const int64_t n = params.P + (bonus_rows ? params.B : 0);
  if (n == 0) return hipSuccess;
  const SplitLayout l = split_layout(n, params.V);
  char* ws = static_cast<char*>(scratch);
  SplitParams sp;
  memset(&sp, 0, sizeof(sp));
  sp.p = params;
  sp.p.order = nullptr;
  if (!sp.p.masks) sp.p.masks = reinterpret_cast<float4*>(ws + l.masks);
  sp.bonus_rows = bonus_rows;
  sp.nch = l.nch;
  sp.head = reinterpret_cast<SplitHead*>(ws + l.head);
  sp.rows = reinterpret_cast<SplitRow*>(ws + l.rows);
  sp.cmax = reinterpret_cast<float*>(ws + l.cmax);
  sp.cties = reinterpret_cast<uint32_t*>(ws + l.cties);
  sp.csum = reinterpret_cast<float*>(ws + l.csum);
  sp.gkeys = reinterpret_cast<uint32_t*>(ws + l.gkeys);
  sp.hist = reinterpret_cast<float*>(ws + l.hist);
  sp.cmass = reinterpret_cast<unsigned long long*>(ws + l.cmass);
  sp.cand = reinterpret_cast<uint32_t*>(ws + l.cand);
  hipLaunchKernelGGL(split_plan_kernel, dim3(1), dim3(1024), 0, stream, sp);
  switch (target_dtype) {
    case MVSD_F32: launch_split_dt<MVSD_F32>(sp, l.chunk, stream); break;
    case MVSD_BF16: launch_split_dt<MVSD_BF16>(sp, l.chunk, stream); break;
    case MVSD_F16: launch_split_dt<MVSD_F16>(sp, l.chunk, stream); break;
    default: return hipErrorInvalidValue;
  }
  if (apply) {
    const int nch = (params.V + kSplitLong - 1) / kSplitLong;
    hipLaunchKernelGGL(split_apply_kernel, dim3((unsigned)params.P * (unsigned)nch),
                       dim3(kSplitThreads), 0, stream, sp);
  }
  return hipGetLastError();
}

hipError_t launch_constraints(const VerifyParams& params, int target_dtype, hipStream_t stream) {
  if (params.P == 0) return hipSuccess;
  if (params.order)
    hipLaunchKernelGGL(constraint_plan_kernel, dim3(1), dim3(1024), 0, stream, params);
  const dim3 grid((unsigned)params.P), block(kCT);
  switch (target_dtype) {
    case MVSD_F32: hipLaunchKernelGGL((constraints_kernel<MVSD_F32, false>), grid, block, 0, stream, params); break;
    case MVSD_BF16: hipLaunchKernelGGL((constraints_kernel<MVSD_BF16, false>), grid, block, 0, stream, params); break;
    case MVSD_F16: hipLaunchKernelGGL((constraints_kernel<MVSD_F16, false>), grid, block, 0, stream, params); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_topk_topp(float* logits, int64_t stride, const int64_t* top_k, const float* top_p,
                            int64_t num_rows, int64_t vocab_size, hipStream_t stream) {
  if (num_rows == 0) return hipSuccess;
  VerifyParams p;
  memset(&p, 0, sizeof(p));
  p.target = logits;
  p.target_stride = stride;
  p.target_num_rows = num_rows;
  p.B = (int)num_rows;
  p.P = (int)num_rows;
  p.V = (int)vocab_size;
  p.top_k = top_k;
  p.top_p = top_p;
  hipLaunchKernelGGL((constraints_kernel<MVSD_F32, true>), dim3((unsigned)num_rows), dim3(kCT), 0,
                     stream, p);
  return hipGetLastError();
}

}  // namespace mvsd
