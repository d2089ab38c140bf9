// The support of a temperature / top-k / top-p filtered row (aspec/models/ops/loss.py:57-80), for the
// filtered logits (sampling.hip) and the sampled L1 (sampled_l1.hip).
//
// Per row and side (draft: `draft_sampling`, teacher: `target_sampling`):
//   scaled = temperature != 1 ? (x - max x) * (1/T) : x            (fp32, x the bf16 logit)
//   order  = scaled descending, ties by token index (a stable sort)
//   keep   = rank < top_k (0 < top_k < V)  and  mass before the token <= top_p (top_p < 1),
//            the mass from softmax(scaled) over the full row
//   p      = softmax(scaled) over the kept tokens, 0 elsewhere.
//
// One 512-thread workgroup owns a row; the row lives in registers as packed bf16 (NV chunks of
// eight per thread, up to 98304 tokens; longer rows are read again from global memory on each
// pass) and nothing is sorted. A row takes three passes: the maximum; the total mass, with every
// token's mass and count added to a histogram of LDS bins, 1/32 nat of scaled logit each; and, the
// bin that holds the boundary found by a scan, the exact mass above that bin and the list of its
// tokens. One wave then finishes on the list: the boundary key (a binary search over the bin's few
// distinct bf16 values), its tie group in scaled values (a temperature can merge neighbouring bf16
// values into one fp32 value), the kept count within the group from its mass per token, and, when
// the group is cut, the index of the last kept token. A token is kept iff its scaled value is above
// the boundary's, or equal and its index <= last.
//
// The histogram's masses (fp32, any order) only propose a bin: it is taken when the exact mass above
// it is <= top_p of the total and the mass with it is not, else its neighbour is tried, and no
// further bin than that. Masses are fp32 per token, summed in fp64: over the row in a fixed order, and
// over a bin's list exactly (its masses lie within e^(1/32) of each other, so at most 2048 of them sum
// without rounding). A boundary in the last, open bin or in one of more than 2048 tokens (flat rows,
// few distinct values) is found in passes over the row's 16-bit keys instead (search_row), where sums
// in a fixed order decide as well. So the order of the atomics can show only where fp64 sums differ in
// their last digits.
#pragma once

#include <cmath>

#include "common.h"

namespace aspec {
namespace {

constexpr int kSampThreads = 512;
constexpr int kSampWaves = kSampThreads / 64;
constexpr float kLog2e = 1.4426950408889634f;
constexpr int kBins = 2048;        // bins of 1/32 nat below the maximum: 64 nats, the last one open
constexpr float kBinsPerNat = 32.f;
constexpr int kListCap = 2048;     // tokens of the boundary's bin that the list holds
constexpr int kBinTries = 2;       // bins looked at before the search over the whole row
constexpr uint32_t kNegInfBits = 0xff80u;  // bf16 -inf: the padding of a row's tail

// per-row, per-side record (8 words); the sampled-L1 row holds draft, teacher, then the masses
constexpr int kSideWords = 8;
constexpr int kL1Words = 24;
constexpr uint32_t kFlagTemp = 1, kFlagNaN = 2, kFlagAll = 4;

struct SideParams {
  float rcp_t;   // 1/T in fp32 (1 without a temperature)
  float top_p;   // fp32, as the reference compares its fp32 cumulative mass
  int64_t top_k;
  int temp, use_p, use_k;
};

struct SideStats {
  float m;        // row max of the logits
  float rcp_t;
  uint32_t okey;  // boundary key of the scaled values
  int32_t last;   // last kept token index among the boundary ties
  float zinv;     // 1 / sum over kept tokens of exp(scaled - max scaled)
  uint32_t flags;
  int32_t nmax;   // tokens equal to the max (the max's gradient is shared among them)
  uint32_t pad;
};

struct SampledArgs {
  const uint16_t* x;
  const uint16_t* y;
  const int64_t* yidx;
  int64_t trows, rows, V;
  SideParams px, py;
  float* out;          // sampling_logits: fp32 [rows][V]
  const float* gout;   // sampling_logits backward: fp32 [rows][V]
  float* l1;
  float* stats;
  const float* g_l1;
  uint16_t* dx;
  int32_t* flags;
};

__device__ __forceinline__ float bf16f(uint32_t h) { return __uint_as_float(h << 16); }

// ordered key of an fp32 value (-0 equals +0, as in a sort's comparisons)
__device__ __forceinline__ uint32_t ord_key(float o) {
  uint32_t b = __float_as_uint(o);
  if ((b << 1) == 0) b = 0;
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
// ordered 16-bit key of a bf16 value, and back
__device__ __forceinline__ uint32_t x_key(uint32_t h) {
  if ((h & 0x7fffu) == 0) h = 0;
  return (h & 0x8000u) ? (~h & 0xffffu) : (h | 0x8000u);
}
__device__ __forceinline__ uint32_t x_bits_of_key(uint32_t k) {
  return (k & 0x8000u) ? (k & 0x7fffu) : (~k & 0xffffu);
}

struct RowCtx {
  float m, rcp_t;
  bool temp;
};
// exp(scaled - max scaled) and the sort value of a logit; one expression everywhere, so the
// forward, the backward and both sides of a row agree bit for bit
__device__ __forceinline__ float u_of(float x, const RowCtx& c) { return (x - c.m) * c.rcp_t; }
__device__ __forceinline__ float e_of(float x, const RowCtx& c) {
  return __builtin_amdgcn_exp2f(u_of(x, c) * kLog2e);
}
__device__ __forceinline__ float ord_of(float x, const RowCtx& c) { return c.temp ? u_of(x, c) : x; }

// the value of an ordered key
__device__ __forceinline__ float value_of_key(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

__device__ __forceinline__ RowCtx ctx_of(const SideStats& s) {
  return RowCtx{s.m, s.rcp_t, (s.flags & kFlagTemp) != 0};
}
// A row's support as the passes test it: kept iff the sort value is above `bound`, or equal (-0
// equals +0) at an index <= last. A row without a filter has bound -inf and every index. A sort value
// that is NaN (0 times the infinite reciprocal of a temperature below 2^-128) is kept, so the NaN
// shows in the result.
struct Support {
  float bound;
  int32_t last;
};
__device__ __forceinline__ Support support_of(const SideStats& s) {
  return (s.flags & kFlagAll) ? Support{-INFINITY, 0x7fffffff} : Support{value_of_key(s.okey), s.last};
}
// branch-free: evaluated for every token of a pass
__device__ __forceinline__ bool kept(const Support& s, float ord, int32_t idx) {
  return !(ord < s.bound) & ((ord != s.bound) | (idx <= s.last));
}
// probability of a token after filtering (0 outside the support)
__device__ __forceinline__ float prob(const Support& s, const RowCtx& c, float zinv, uint32_t h, int32_t idx) {
  const float x = bf16f(h);
  return kept(s, ord_of(x, c), idx) ? e_of(x, c) * zinv : 0.0f;
}

// ---- block reductions over the 8 waves, fixed order, every thread gets the total ---------------
struct Red {
  double slot[2][kSampWaves];
};

__device__ __forceinline__ double join_d(uint32_t lo, uint32_t hi) {
  return __builtin_bit_cast(double, (static_cast<uint64_t>(hi) << 32) | lo);
}
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  return join_d(dpp_u32<CTRL>(static_cast<uint32_t>(b)), dpp_u32<CTRL>(static_cast<uint32_t>(b >> 32)));
}
// wave_allsum (common.h) for doubles: every lane gets the sum, added in a fixed pairing
__device__ __forceinline__ double wave_sum_d(double v) {
  v += dpp_d<0xB1>(v);
  v += dpp_d<0x4E>(v);
  v += dpp_d<0x141>(v);
  v += dpp_d<0x140>(v);
  uint64_t b = __builtin_bit_cast(uint64_t, v);
  uint32_t lo = static_cast<uint32_t>(b), hi = static_cast<uint32_t>(b >> 32);
  auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
  v = join_d(l[0], h[0]) + join_d(l[1], h[1]);
  b = __builtin_bit_cast(uint64_t, v);
  lo = static_cast<uint32_t>(b), hi = static_cast<uint32_t>(b >> 32);
  l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  return join_d(l[0], h[0]) + join_d(l[1], h[1]);
}
__device__ __forceinline__ uint32_t wave_sum_u(uint32_t v) {
  return wave_allreduce_bits(v, [](uint32_t a, uint32_t b) { return a + b; });
}
__device__ __forceinline__ uint32_t wave_max_u(uint32_t v) {
  return wave_allreduce_bits(v, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
}
// A value every lane holds alike, moved to scalar registers (the row's statistics and search
// bounds then take no vector registers beside the row itself).
__device__ __forceinline__ double uniform(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(b));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(b >> 32));
  return __builtin_bit_cast(double, (static_cast<uint64_t>(hi) << 32) | lo);
}

__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int32_t uniform(int32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float uniform(float v) { return __uint_as_float(uniform(__float_as_uint(v))); }

// Two slot sets used alternately: the barrier of the call in between separates the reads of one
// call from the writes of the call after next. Every thread adds the eight waves' slots in one
// fixed pairing.
__device__ __forceinline__ double block_total(double wave_value, Red& r, int& ph) {
  double* slot = r.slot[ph];
  ph ^= 1;
  if ((threadIdx.x & 63) == 0) slot[threadIdx.x >> 6] = wave_value;
  __syncthreads();
  return uniform(((slot[0] + slot[1]) + (slot[2] + slot[3])) + ((slot[4] + slot[5]) + (slot[6] + slot[7])));
}
__device__ __forceinline__ double block_sum(double v, Red& r, int& ph) {
  return block_total(wave_sum_d(v), r, ph);
}
__device__ __forceinline__ int64_t block_count(uint32_t v, Red& r, int& ph) {
  return static_cast<int64_t>(block_total(static_cast<double>(wave_sum_u(v)), r, ph));
}
// the row maximum, and whether any thread's `bad` is set
__device__ __forceinline__ float block_max(float v, bool bad, bool& any_bad, Red& r, int& ph) {
  double* slot = r.slot[ph];
  ph ^= 1;
  v = wave_allmax(v);
  // a NaN slot marks a wave with a bad token
  const double mine = __any(bad) ? __builtin_nan("") : static_cast<double>(v);
  if ((threadIdx.x & 63) == 0) slot[threadIdx.x >> 6] = mine;
  __syncthreads();
  double m = slot[0];
  any_bad = m != m;
#pragma unroll
  for (int w = 1; w < kSampWaves; ++w) {
    const double o = slot[w];
    any_bad |= o != o;
    m = fmax(m, o);
  }
  return uniform(static_cast<float>(m));
}

// ---- rows -------------------------------------------------------------------------------------
// Chunk c of thread t is tokens (c * 512 + t) * 8 .. + 7; tokens past V read as bf16 -inf.
__device__ __forceinline__ uint4 row_chunk(const uint16_t* row, int64_t V, int64_t base) {
  if (base + 8 <= V) return load_chunk(row + base);
  uint32_t w[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t lo = base + 2 * k < V ? row[base + 2 * k] : kNegInfBits;
    const uint32_t hi = base + 2 * k + 1 < V ? row[base + 2 * k + 1] : kNegInfBits;
    w[k] = lo | (hi << 16);
  }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

__device__ __forceinline__ int32_t opaque_t8() {
  int32_t t8 = static_cast<int32_t>(threadIdx.x) * 8;
  asm volatile("" : "+v"(t8));
  return t8;
}
__device__ __forceinline__ uint32_t half_of(const uint32_t (&w)[4], int j) {
  return (j & 1) ? w[j >> 1] >> 16 : w[j >> 1] & 0xffffu;
}

// A row held in registers (NV chunks of packed bf16 per thread: up to 98304 tokens). Each pass
// runs the words through an empty asm in place (no copy, no instruction) and rebuilds the token
// index from an opaque thread offset, so what a pass derives from them (exp values, bins, indices)
// is recomputed in that pass instead of being kept in registers from the one before.
// kWavesPerSimd: the occupancy that the row's own registers allow and the rare searches must not
// lower (they spill instead): two workgroups of a CU up to 32768 tokens, more for shorter rows.
template <int NV>
struct RegRow {
  static constexpr int kWavesPerSimd = NV == 1 ? 8 : NV == 2 ? 6 : NV <= 8 ? 4 : 2;
  const uint16_t* p;
  uint4 r[NV];
  __device__ __forceinline__ void load(const uint16_t* row, int64_t V) {
    p = row;
#pragma unroll
    for (int c = 0; c < NV; ++c)
      r[c] = row_chunk(row, V, (static_cast<int64_t>(c) * kSampThreads + threadIdx.x) * 8);
  }
  __device__ __forceinline__ uint4 first() const { return r[0]; }
  template <typename G>
  __device__ __forceinline__ void chunks(G&& g) {
    const int32_t t8 = opaque_t8();
#pragma unroll
    for (int c = 0; c < NV; ++c) {
      asm volatile("" : "+v"(r[c].x), "+v"(r[c].y), "+v"(r[c].z), "+v"(r[c].w));
      const uint32_t w[4] = {r[c].x, r[c].y, r[c].z, r[c].w};
      g(c, c * kSampThreads * 8 + t8, w);
    }
  }
};

// A row read again from global memory on every pass, for vocabularies beyond the registers' reach
// (the row stays in the caches between a workgroup's passes).
struct GlobalRow {
  static constexpr int kWavesPerSimd = 8;
  const uint16_t* p;
  int64_t V;
  int n;
  __device__ __forceinline__ void load(const uint16_t* row, int64_t V_) {
    p = row, V = V_;
    n = static_cast<int>((V + 8LL * kSampThreads - 1) / (8LL * kSampThreads));
  }
  __device__ __forceinline__ uint4 first() const { return row_chunk(p, V, static_cast<int64_t>(threadIdx.x) * 8); }
  template <typename G>
  __device__ __forceinline__ void chunks(G&& g) {
    const int32_t t8 = static_cast<int32_t>(threadIdx.x) * 8;
    for (int c = 0; c < n; ++c) {
      const int32_t base = c * kSampThreads * 8 + t8;
      const uint4 v = row_chunk(p, V, base);
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
      g(0, base, w);
    }
  }
};

// The pass's accumulators, made opaque at the end of each chunk: the chunk's contributions are
// then added before the next chunk's words are read, instead of being sunk to the pass's end with
// every token's key kept live until there.
template <typename T>
__device__ __forceinline__ void fence1(T& v) {
  asm volatile("" : "+v"(v));
}
template <typename... T>
__device__ __forceinline__ void fence(T&... v) {
  (fence1(v), ...);
}

// f(bf16 bits, token index) over the thread's tokens, in a fixed order; end() after each chunk
// (fences the pass's accumulators)
template <typename Row, typename F, typename G>
__device__ __forceinline__ void for_each(Row& row, F&& f, G&& end) {
  row.chunks([&](int c, int32_t base, const uint32_t (&w)[4]) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      f(w[k] & 0xffffu, base + 2 * k);
      f(w[k] >> 16, base + 2 * k + 1);
    }
    end();
  });
}

// LDS of one row's support search.
struct Work {
  Red red;
  float mass[kBins + kWave];  // past kBins: where the last bin's adds go, a word per lane, never read
  uint32_t count[kBins + kWave];
  union {
    struct {
      uint32_t key[kListCap];  // the list: x_key and index of the tokens of the bin looked at
      int32_t idx[kListCap];
    };
    double hist[kBins];  // the row's search: mass or count per group of keys
  };
  double part[kWave];
  float wave_mass[kSampWaves];
  uint32_t wave_count[kSampWaves];
  uint32_t n;        // tokens appended to the list
  uint32_t level;    // waves whose first tokens lie within three bins
  int32_t bin_p, bin_k;
  int32_t verdict;   // what the list's wave found: see Verdict
  uint32_t okey;
  int32_t last;
  double z;
};
enum Verdict { kFound, kLower };

// The distance of a sort value below the maximum in bins, as a float: its integer part is the bin
// (the last bin takes everything beyond). A function of the scaled value, so tokens that tie share
// a bin.
__device__ __forceinline__ float bin_of(float u) { return fminf(-u * kBinsPerNat, static_cast<float>(kBins - 1)); }

// The end of the search on one bin's list, by one wave: `above` (<= lim with top-p) is the exact mass
// and `before` the count of the tokens in higher bins, lim = top_p times the row's mass; use_k says
// whether top_k's boundary lies in this bin.
__device__ __forceinline__ void search_list(Work& w, int n, const RowCtx& cx, bool use_p, double lim, double above,
                                            bool use_k, int64_t top_k, int64_t before) {
  const int lane = threadIdx.x & 63;
  auto value = [&](int i) { return bf16f(x_bits_of_key(w.key[i])); };
  auto okey_at = [&](int i) { return ord_key(ord_of(value(i), cx)); };
  uint32_t kmin = 0xffffu, kmax = 0;
  double mass = 0.0;
  for (int i = lane; i < n; i += kWave) {
    kmin = min(kmin, w.key[i]);
    kmax = max(kmax, w.key[i]);
    mass += e_of(value(i), cx);
  }
  kmin = wave_allmin(kmin);
  kmax = wave_max_u(kmax);
  mass = wave_sum_d(mass);
  bool have_p = false;
  if (use_p) {
    have_p = above + mass > lim;
    if (!have_p && !use_k) {
      if (lane == 0) w.verdict = kLower;
      return;
    }
  }
  uint32_t okey = 0;
  int64_t keep = 0, ties = 0;
  // (sort key, kept ties, ties) of a boundary at x_key k: `room(mass, count)` gives the kept ties
  // from the mass and count of the list's tokens above it
  auto boundary = [&](uint32_t k, auto&& room) {
    const uint32_t o = ord_key(ord_of(bf16f(x_bits_of_key(k)), cx));
    double m = 0.0;
    uint32_t over = 0, same = 0;
    for (int i = lane; i < n; i += kWave) {
      const uint32_t oi = okey_at(i);
      if (oi > o) m += e_of(value(i), cx);
      over += oi > o ? 1u : 0u;
      same += oi == o ? 1u : 0u;
    }
    const int64_t c = wave_sum_u(same);
    const int64_t left = room(wave_sum_d(m), static_cast<int64_t>(wave_sum_u(over)), c,
                              e_of(bf16f(x_bits_of_key(k)), cx));
    // both filters keep a prefix of the order: the shorter one wins
    if (ties == 0 || o > okey || (o == okey && left < keep)) okey = o, keep = left, ties = c;
  };
  if (have_p) {
    uint32_t lo = kmin, hi = kmax;  // the smallest key with a strictly greater mass <= lim
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      double f = 0.0;
      for (int i = lane; i < n; i += kWave) f += w.key[i] > mid ? e_of(value(i), cx) : 0.0f;
      if (above + wave_sum_d(f) <= lim) hi = mid;
      else lo = mid + 1;
    }
    boundary(lo, [&](double m, int64_t, int64_t c, float eb) -> int64_t {
      // the j-th tie (0-based, index order) has mass above + m + j * eb before it
      if (!(eb > 0.0f)) return c;
      const double q = floor((lim - (above + m)) / static_cast<double>(eb));
      return q + 1.0 >= static_cast<double>(c) ? c : static_cast<int64_t>(q) + 1;
    });
  }
  if (use_k) {
    uint32_t lo = kmin, hi = kmax;
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      uint32_t c = 0;
      for (int i = lane; i < n; i += kWave) c += w.key[i] > mid ? 1u : 0u;
      if (before + wave_sum_u(c) <= top_k - 1) hi = mid;
      else lo = mid + 1;
    }
    boundary(lo, [&](double, int64_t over, int64_t, float) -> int64_t { return top_k - before - over; });
  }
  // the index of the last kept tie: the smallest j with `keep` ties at indices <= j
  int32_t last = 0x7fffffff;
  if (keep < ties) {
    int32_t lo = 0x7fffffff, hi = 0;
    for (int i = lane; i < n; i += kWave) {
      lo = min(lo, w.idx[i]);
      hi = max(hi, w.idx[i]);
    }
    lo = static_cast<int32_t>(wave_allmin(static_cast<uint32_t>(lo)));
    hi = static_cast<int32_t>(wave_max_u(static_cast<uint32_t>(hi)));
    while (lo < hi) {
      const int32_t mid = (lo + hi) >> 1;
      uint32_t c = 0;
      for (int i = lane; i < n; i += kWave) c += ((w.idx[i] <= mid) & (okey_at(i) == okey)) ? 1u : 0u;
      if (static_cast<int64_t>(wave_sum_u(c)) >= keep) hi = mid;
      else lo = mid + 1;
    }
    last = lo;
  }
  // the kept mass: the bins above, the list's tokens above the boundary, the kept ties
  double m = 0.0;
  float eb = 0.0f;
  for (int i = lane; i < n; i += kWave) {
    const uint32_t oi = okey_at(i);
    const float e = e_of(value(i), cx);
    if (oi > okey) m += e;
    if (oi == okey) eb = e;
  }
  m = wave_sum_d(m);
  eb = wave_allmax(eb);
  if (lane == 0) {
    w.verdict = kFound;
    w.okey = okey;
    w.last = last;
    w.z = above + m + static_cast<double>(eb) * static_cast<double>(keep);
  }
}

// The first lane at which base + the sum of the lanes' values up to it exceeds target, and that sum
// without the lane; -1 and the whole sum if there is none.
struct First {
  int at;
  double before;
};
__device__ __forceinline__ First first_lane_over(double own, double base, double target) {
  double inc = own;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const double from = __shfl_up(inc, o);
    if ((threadIdx.x & 63) >= o) inc += from;
  }
  const uint64_t over = __ballot(base + inc > target);
  if (!over) return First{-1, base + uniform(__shfl(inc, kWave - 1))};
  const int at = __ffsll(static_cast<unsigned long long>(over)) - 1;
  return First{at, base + uniform(__shfl(inc - own, at))};
}

// The same over n entries of w.hist, every wave by itself: up to a lane each; or kBins of them, first
// over the sums of 32.
__device__ __forceinline__ First first_entry_over(int n, double base, double target, Work& w) {
  const int tid = threadIdx.x, lane = tid & 63;
  if (n <= kWave) return first_lane_over(lane < n ? w.hist[lane] : 0.0, base, target);
  constexpr int kPer = kBins / kWave;
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < kBins / kSampThreads; ++i) s += w.hist[tid * (kBins / kSampThreads) + i];
#pragma unroll
  for (int o = 1; o < kSampThreads / kWave; o <<= 1) s += __shfl_xor(s, o);
  if (tid % (kSampThreads / kWave) == 0) w.part[tid / (kSampThreads / kWave)] = s;
  __syncthreads();
  const First part = first_lane_over(w.part[lane], base, target);
  if (part.at < 0) return part;
  const First f = first_lane_over(lane < kPer ? w.hist[part.at * kPer + lane] : 0.0, part.before, target);
  // (-1: the sums' rounding differs; any entry of the part is as good a proposal)
  return First{part.at * kPer + max(f.at, 0), f.at < 0 ? part.before : f.before};
}

// Keys of a row to look for a boundary in, and the mass (top-p) or count (top-k) of the tokens above.
struct KeyRange {
  uint32_t lo, hi;
  double above;
};
constexpr KeyRange kAllKeys = {0u, 0xffffu, 0.0};

// The keys of the tokens in a bin: bin_of falls as the key rises.
__device__ __forceinline__ KeyRange keys_of_bin(int bin, const RowCtx& cx, double above) {
  uint32_t edge[2];  // the lowest keys in bins <= bin and <= bin - 1
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    uint32_t lo = x_key(kNegInfBits), hi = x_key(kNegInfBits ^ 0x8000u);
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if (static_cast<int>(bin_of(u_of(bf16f(x_bits_of_key(mid)), cx))) <= bin - i) hi = mid;
      else lo = mid + 1;
    }
    edge[i] = lo;
  }
  return KeyRange{uniform(edge[0]), uniform(bin == 0 ? 0xffffu : max(edge[0], edge[1] - 1)), above};
}

// The key in a range, or below it, at which mass or count pass `target`, from fp64 sums over groups of
// keys (added in any order: a proposal in the last digits): a pass for up to 2048 keys, or two. A thread
// adds up tokens of one group before it goes to LDS, so rows of few distinct values (masked, all
// equal) do not queue up on one address.
__device__ __forceinline__ uint32_t likely_key(GlobalRow& r, const RowCtx& cx, KeyRange range, bool by_mass,
                                               double target, Work& w) {
  while (true) {
    int shift = 0;
    while (((range.hi - range.lo) >> shift) >= static_cast<uint32_t>(kBins)) ++shift;
    const int groups = static_cast<int>((range.hi - range.lo) >> shift) + 1;
    __syncthreads();
    for (int i = threadIdx.x; i < (groups <= kWave ? kWave : kBins); i += kSampThreads) w.hist[i] = 0.0;
    __syncthreads();
    uint32_t group = 0;
    double sum = 0.0;
    auto flush = [&] {
      if (sum > 0.0) __hip_atomic_fetch_add(&w.hist[group], sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      sum = 0.0;
    };
    for_each(r, [&](uint32_t h, int32_t) {
      const uint32_t k = x_key(h);
      if (k >= range.lo && k <= range.hi) {
        const uint32_t g = (range.hi - k) >> shift;
        if (g != group) flush();
        group = g;
        sum += by_mass ? e_of(bf16f(h), cx) : 1.0f;
      }
      fence(group, sum);  // token by token: this path is rare, its registers are every row's
    }, [] {});
    flush();
    __syncthreads();
    const First f = first_entry_over(groups, range.above, target, w);
    if (f.at < 0) {
      if (range.lo == 0) return 0;
      range = KeyRange{0u, range.lo - 1, f.before};
      continue;
    }
    const uint32_t top = range.hi - (static_cast<uint32_t>(f.at) << shift);
    if (shift == 0) return top;
    range = KeyRange{max(range.lo, top - ((1u << shift) - 1)), top, f.before};
  }
}

// One pass around a boundary at x_key k: the mass or count of the keys above k and from k on, and
// of the boundary's ties in scaled values the mass and count above them and their number, this also
// per step of 4096 tokens (V > 2^18: several steps) in w.count. Sums in a fixed order.
struct Around {
  double gt, ge, mass;
  int64_t over, same;
};
constexpr int kStepShift = 12;  // log2 of the tokens a workgroup's chunks cover
static_assert(kSampThreads * 8 == 1 << kStepShift, "one chunk per thread");
// (log2 of the tokens that an entry of w.count covers: at most a lane's worth of entries)
__device__ __forceinline__ int tie_shift(int64_t V) {
  int shift = kStepShift;
  while (((V - 1) >> shift) >= kWave) ++shift;
  return shift;
}

__device__ __forceinline__ Around around(GlobalRow& r, uint32_t k, const RowCtx& cx, bool by_mass, Work& w, int& ph) {
  const uint32_t o = ord_key(ord_of(bf16f(x_bits_of_key(k)), cx));
  const int shift = tie_shift(r.V);
  __syncthreads();
  if (threadIdx.x < kWave) w.count[threadIdx.x] = 0u;
  __syncthreads();
  double gt = 0.0, ge = 0.0, mass = 0.0;
  uint32_t over = 0, same = 0;
  r.chunks([&](int, int32_t base, const uint32_t (&v)[4]) {
    uint32_t ties = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t h = half_of(v, j), key = x_key(h);
      const uint32_t oi = ord_key(ord_of(bf16f(h), cx));
      const float e = e_of(bf16f(h), cx), by = by_mass ? e : 1.0f;
      gt += key > k ? by : 0.0f;
      ge += key >= k ? by : 0.0f;
      mass += oi > o ? e : 0.0f;
      over += oi > o ? 1u : 0u;
      ties += oi == o ? 1u : 0u;
      fence(gt, ge, mass, over, ties);
    }
    same += ties;
    const uint32_t all = wave_sum_u(ties);
    if ((threadIdx.x & 63) == 0 && all) atomicAdd(&w.count[base >> shift], all);
  });
  Around a;
  a.gt = block_sum(gt, w.red, ph);
  a.ge = block_sum(ge, w.red, ph);
  a.mass = block_sum(mass, w.red, ph);
  a.over = block_count(over, w.red, ph);
  a.same = block_count(same, w.red, ph);
  return a;
}

// The index of the keep-th tie of the boundary that around() last saw: its step from w.count, then
// a scan of that step's tokens.
__device__ __forceinline__ int32_t tie_index(const GlobalRow& r, uint32_t o, int64_t keep, const RowCtx& cx, Work& w) {
  const int tid = threadIdx.x, shift = tie_shift(r.V);
  const First f = first_lane_over(static_cast<double>(w.count[tid & 63]), 0.0, static_cast<double>(keep - 1));
  int64_t left = keep - static_cast<int64_t>(f.before);  // 1-based in the group
  const int64_t begin = static_cast<int64_t>(f.at) << shift, end = begin + (int64_t{1} << shift);
  for (int64_t start = begin; start < end; start += 1 << kStepShift) {
    const int32_t base = static_cast<int32_t>(start) + tid * 8;
    const uint4 c = row_chunk(r.p, r.V, base);
    const uint32_t v[4] = {c.x, c.y, c.z, c.w};
    uint32_t own = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) own += ord_key(ord_of(bf16f(half_of(v, j)), cx)) == o ? 1u : 0u;
    uint32_t upto = own;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const uint32_t from = __shfl_up(upto, d);
      if ((tid & 63) >= d) upto += from;
    }
    if ((tid & 63) == 63) w.wave_count[tid >> 6] = upto;
    __syncthreads();
    uint32_t total = 0;
#pragma unroll
    for (int i = 0; i < kSampWaves; ++i) {
      if (i < (tid >> 6)) upto += w.wave_count[i];
      total += w.wave_count[i];
    }
    if (left > upto - own && left <= upto) {
      int64_t n = left - (upto - own);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (ord_key(ord_of(bf16f(half_of(v, j)), cx)) == o && --n == 0) w.last = base + j;
    }
    __syncthreads();
    left -= total;
    if (left <= 0) break;
  }
  return w.last;
}

// The support from passes over the row in global memory (rolled loops: unrolled over a row's
// registers this rare path was most of the file's code), for a boundary that the list cannot hold.
// A key per filter is proposed from a histogram, and one exact pass around it shows that the mass (or
// count) above is <= the limit and with it is not; else a binary search over the 16-bit keys goes on
// from what that pass showed. in_p and in_k: where to look first. Two or three passes, against the
// some thirty of binary searches over keys and indices, in registers up to 98304 tokens:
// sampling_logits of 512 x 98304, sigma 0.3, top-p 877 -> 509 us; 400 x 151936 all equal 1458 -> 311;
// 1024 x 32000 with 41 tokens not masked, top-k 50, 472 -> 154; 2048 x 2560 all equal 139 -> 76.
__device__ __forceinline__ void search_row(GlobalRow& r, const SideParams& P, const RowCtx& cx, double total,
                                           KeyRange in_p, KeyRange in_k, SideStats& st, Work& w, int& ph) {
  const double lim = uniform(static_cast<double>(P.top_p) * total);
  uint32_t key = 0, okey = 0, seen = 0;  // the shorter prefix's boundary, and the key last looked at
  int64_t keep = 0, ties = 0;
  double mass = 0.0;
#pragma unroll 1
  for (int filter = 0; filter < 2; ++filter) {  // top-k, then top-p
    const bool by_mass = filter == 1;
    if (!(by_mass ? P.use_p : P.use_k)) continue;
    uint32_t lo = 0, hi = 0xffffu;  // the smallest key with at most `target` above it lies here
    KeyRange in = {by_mass ? in_p.lo : in_k.lo, by_mass ? in_p.hi : in_k.hi, by_mass ? in_p.above : in_k.above};
    if (by_mass && P.use_k) {
      // top-p matters where it ends before top-k's last token
      if (mass + static_cast<double>(e_of(bf16f(x_bits_of_key(key)), cx)) * static_cast<double>(keep - 1) <= lim) break;
      lo = key;
    }
    const double target = by_mass ? lim : uniform(static_cast<double>(P.top_k - 1));
    uint32_t mid = max(likely_key(r, cx, in, by_mass, target, w), lo);
    Around a;
    while (true) {
      a = around(r, mid, cx, by_mass, w, ph);
      if (a.gt > target && mid < hi) lo = mid + 1;
      else if (a.ge <= target && mid > lo) hi = mid - 1;
      else break;
      mid = (lo + hi) >> 1;
    }
    seen = mid;
    const float xb = bf16f(x_bits_of_key(mid));
    const uint32_t o = uniform(ord_key(ord_of(xb, cx)));
    int64_t n = a.same;
    if (by_mass) {
      const float eb = e_of(xb, cx);
      if (eb > 0.0f) {
        // the j-th tie (0-based, index order) has mass a.mass + j * eb before it
        const double q = floor((lim - a.mass) / static_cast<double>(eb));
        if (q + 1.0 < static_cast<double>(a.same)) n = static_cast<int64_t>(uniform(q)) + 1;
      }
    } else {
      n = P.top_k - a.over;
    }
    // both filters keep a prefix of the order: the shorter one wins
    if (ties == 0 || o > okey || (o == okey && n < keep)) key = mid, okey = o, keep = n, ties = a.same, mass = a.mass;
  }
  st.okey = uniform(okey);
  st.last = 0x7fffffff;
  if (keep < ties) {
    if (seen != key) around(r, key, cx, false, w, ph);
    st.last = uniform(tie_index(r, okey, keep, cx, w));
  }
  const float eb = e_of(bf16f(x_bits_of_key(key)), cx);
  st.zinv = uniform(static_cast<float>(1.0 / (mass + static_cast<double>(eb) * static_cast<double>(keep))));
}

// One side's support and normaliser. Rows with a NaN or no finite maximum get kFlagNaN (the
// reference's softmax gives NaN there).
template <bool FILTER, typename Row>
__device__ __forceinline__ SideStats compute_support(Row& r, int64_t V, const SideParams P, Work& w, int& ph) {
  const int tid = threadIdx.x;
  SideStats st = {};
  if (tid == 0) w.level = 0;
  float mx = -INFINITY;
  uint32_t mag = 0;  // the largest magnitude bits: above 0x7f80 is a NaN
  for_each(r, [&](uint32_t h, int32_t) {
    mag = max(mag, h & 0x7fffu);
    mx = fmaxf(mx, bf16f(h));
  }, [&] { fence(mx, mag); });
  bool has_nan;
  const float m = block_max(mx, mag > 0x7f80u, has_nan, w.red, ph);
  st.m = m;
  st.rcp_t = P.temp ? P.rcp_t : 1.0f;
  st.flags = P.temp ? kFlagTemp : 0u;
  if (has_nan || !(m > -INFINITY && m < INFINITY)) {
    st.flags |= kFlagNaN;
    return st;
  }
  const RowCtx cx{m, st.rcp_t, P.temp != 0};
  const bool filter = FILTER && (P.use_p || P.use_k);
  if (filter) {
    for (int i = tid; i < kBins; i += kSampThreads) w.mass[i] = 0.0f, w.count[i] = 0u;
    if (tid == 0) w.n = 0, w.bin_p = kBins - 1, w.bin_k = kBins - 1;
    // A level row, most of whose first tokens lie within three bins: its adds would queue up on these,
    // and the list could not hold their bin. The histogram stays empty and the row's search decides.
    const uint4 c = r.first();
    const uint32_t v[4] = {c.x, c.y, c.z, c.w};
    const float b0 = uniform(bin_of(u_of(bf16f(half_of(v, 0)), cx)));
    bool near = b0 < kBins - 1;
#pragma unroll
    for (int j = 0; j < 8; ++j) near &= fabsf(bin_of(u_of(bf16f(half_of(v, j)), cx)) - b0) < 3.0f;
    if (__popcll(__ballot(near)) >= 48 && (tid & 63) == 0) atomicAdd(&w.level, 1u);
    __syncthreads();
  }
  const bool level = filter && V > kListCap && uniform(w.level) > kSampWaves / 2;
  const bool hist_p = P.use_p && !level, hist_k = P.use_k && !level;
  // the total mass, the tokens equal to the maximum and the histogram
  double se = 0.0;
  uint32_t nm = 0;
  // (one branch per filter and chunk, none per token)
  const int sink = kBins + (tid & 63);
  r.chunks([&](int, int32_t base, const uint32_t (&v)[4]) {
    float e[8];
    int at[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float x = bf16f(half_of(v, j));
      e[j] = e_of(x, cx);
      se += e[j];
      nm += x == m ? 1u : 0u;
      const int b = static_cast<int>(bin_of(u_of(x, cx)));
      at[j] = b < kBins - 1 ? b : sink;
    }
    if (hist_p && base < V) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        __hip_atomic_fetch_add(&w.mass[at[j]], e[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    if (hist_k && base < V) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        __hip_atomic_fetch_add(&w.count[at[j]], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    fence(se, nm);
  });
  const double total = block_sum(se, w.red, ph);  // its barrier also completes the histogram
  st.nmax = uniform(static_cast<int32_t>(block_count(nm, w.red, ph)));
  if (!FILTER || !filter) {
    st.flags |= kFlagAll;
    st.last = 0x7fffffff;
    st.zinv = uniform(static_cast<float>(1.0 / total));
    return st;
  }
  // The bins that hold the top-p and top-k boundaries: thread t scans bins 4t .. 4t+3.
  const double lim = uniform(static_cast<double>(P.top_p) * total);
  constexpr int kPer = kBins / kSampThreads;
  float own_m[kPer];
  uint32_t own_c[kPer];
  float sum_m = 0.0f;
  uint32_t sum_c = 0;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    own_m[i] = w.mass[tid * kPer + i];
    own_c[i] = w.count[tid * kPer + i];
    sum_m += own_m[i];
    sum_c += own_c[i];
  }
  float inc_m = sum_m;
  uint32_t inc_c = sum_c;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const float fm = __shfl_up(inc_m, o);
    const uint32_t fc = __shfl_up(inc_c, o);
    if ((tid & 63) >= o) inc_m += fm, inc_c += fc;
  }
  if ((tid & 63) == 63) w.wave_mass[tid >> 6] = inc_m, w.wave_count[tid >> 6] = inc_c;
  __syncthreads();
  float run_m = inc_m - sum_m;
  uint32_t run_c = inc_c - sum_c;
#pragma unroll
  for (int i = 0; i < kSampWaves - 1; ++i) {
    run_m += i < (tid >> 6) ? w.wave_mass[i] : 0.0f;
    run_c += i < (tid >> 6) ? w.wave_count[i] : 0u;
  }
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    run_m += own_m[i];
    if (P.use_p && static_cast<double>(run_m) > lim) atomicMin(&w.bin_p, tid * kPer + i);
    if (P.use_k) {
      const uint32_t next = run_c + own_c[i];
      if (static_cast<int64_t>(next) >= P.top_k) atomicMin(&w.bin_k, tid * kPer + i);
      w.count[tid * kPer + i] = run_c;  // now the count of the tokens in higher bins
      run_c = next;
    }
  }
  __syncthreads();
  const int bin_k = uniform(P.use_k ? w.bin_k : kBins);
  int bin = uniform(P.use_p ? min(w.bin_p, bin_k) : bin_k);
  const int64_t before_k = P.use_k ? static_cast<int64_t>(uniform(w.count[min(bin_k, kBins - 1)])) : 0;
  KeyRange in_p = kAllKeys;
  // The histogram's bin, then one neighbour, then the search over the row: bounded, because the two
  // sides of a bin's edge are sums in different orders. In the last digits of top_p they can each
  // name the other bin, for ever; and there the histogram's fp32 sum can be tens of bins off.
  for (int tries = 0; tries < kBinTries && bin >= 0 && bin < kBins - 1; ++tries) {
    const float lo = static_cast<float>(bin), hi = static_cast<float>(bin + 1);
    // A bin that the histogram shows to hold more tokens than the list is only summed up: its tokens'
    // appends, one counter for all, would take longer than the search they cannot help.
    const float crowd = P.use_p ? w.mass[bin] * __builtin_amdgcn_exp2f(lo * (kLog2e / kBinsPerNat))
                                : static_cast<float>(w.count[bin + 1] - w.count[bin]);
    const bool crowded = uniform(crowd) > 1.01f * kListCap;
    double f = 0.0;
    r.chunks([&](int, int32_t base, const uint32_t (&v)[4]) {
      uint32_t in_bin = 0;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float x = bf16f(half_of(v, j));
        const float b = bin_of(u_of(x, cx));
        f += b < lo ? e_of(x, cx) : 0.0f;
        in_bin |= ((b >= lo) & (b < hi)) ? 1u << j : 0u;
      }
      if (crowded) in_bin = 0;
      for (; in_bin; in_bin &= in_bin - 1) {  // few tokens of a row
        const int j = __ffs(in_bin) - 1;
        const uint32_t word = (j & 4) ? ((j & 2) ? v[3] : v[2]) : ((j & 2) ? v[1] : v[0]);
        const uint32_t h = (j & 1) ? word >> 16 : word & 0xffffu;
        const uint32_t at = __hip_atomic_fetch_add(&w.n, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (at < kListCap) w.key[at] = x_key(h), w.idx[at] = base + j;
      }
      fence(f);
    });
    const double above = block_sum(f, w.red, ph);  // its barrier also completes the list
    const uint32_t n = uniform(w.n);
    const bool higher = P.use_p && above > lim;
    if (!higher) {
      if (crowded || n > kListCap) {
        in_p = keys_of_bin(bin, cx, above);
        break;
      }
      if (tid < kWave)
        search_list(w, static_cast<int>(n), cx, P.use_p, lim, above, bin == bin_k, P.top_k, before_k);
      __syncthreads();
      if (uniform(w.verdict) == kFound) {
        st.okey = uniform(w.okey);
        st.last = uniform(w.last);
        st.zinv = uniform(static_cast<float>(1.0 / w.z));
        __syncthreads();  // w is reused by the row's other side
        return st;
      }
    }
    bin += higher ? -1 : 1;
    __syncthreads();
    if (tid == 0) w.n = 0;
    __syncthreads();
  }
  const KeyRange in_k = P.use_k && bin_k < kBins - 1 ? keys_of_bin(bin_k, cx, static_cast<double>(before_k)) : kAllKeys;
  GlobalRow again;
  again.load(r.p, V);
  search_row(again, P, cx, total, in_p, in_k, st, w, ph);
  __syncthreads();  // w is reused by the row's other side
  return st;
}

__device__ __forceinline__ void store_side(float* dst, const SideStats& s) {
  dst[0] = s.m;
  dst[1] = s.rcp_t;
  dst[2] = __uint_as_float(s.okey);
  dst[3] = __int_as_float(s.last);
  dst[4] = s.zinv;
  dst[5] = __uint_as_float(s.flags);
  dst[6] = __int_as_float(s.nmax);
  dst[7] = 0.0f;
}
__device__ __forceinline__ SideStats load_side(const float* src) {
  SideStats s;
  s.m = src[0];
  s.rcp_t = src[1];
  s.okey = __float_as_uint(src[2]);
  s.last = __float_as_int(src[3]);
  s.zinv = src[4];
  s.flags = __float_as_uint(src[5]);
  s.nmax = __float_as_int(src[6]);
  s.pad = 0;
  return s;
}

// ---- host side ----------------------------------------------------------------------------------
int side_params(double temperature, double top_p, int64_t top_k, int64_t V, SideParams* p) {
  if (!(temperature > 0.0) || !std::isfinite(temperature))
    return set_error(ASPEC_ERR_INVALID, "sampling temperature must be finite and > 0");
  if (!(top_p > 0.0 && top_p <= 1.0))
    return set_error(ASPEC_ERR_INVALID, "sampling top_p must lie in (0, 1]");
  if (top_k == 0 || top_k < -1)
    return set_error(ASPEC_ERR_INVALID, "sampling top_k must be -1 or >= 1");
  p->temp = temperature != 1.0;
  // the reference's (x - max) / T on CUDA multiplies by the fp32 reciprocal of T
  p->rcp_t = p->temp ? 1.0f / static_cast<float>(temperature) : 1.0f;
  p->top_p = static_cast<float>(top_p);
  p->use_p = top_p < 1.0;
  p->top_k = top_k;
  p->use_k = top_k > 0 && top_k < V;
  return ASPEC_OK;
}

// register chunks per thread for a vocabulary; 0: the row is read from global memory per pass
int chunks_for(int64_t V) {
  const int64_t per = (V + 8LL * kSampThreads - 1) / (8LL * kSampThreads);
  for (int nv : {1, 2, 4, 8, 16, 24})
    if (per <= nv) return nv;
  return 0;
}

// Calls launch(RowType<Row>{}) with the row type of a vocabulary.
template <typename T>
struct RowType {
  using Row = T;
};
template <typename F>
void with_row(int64_t V, F&& launch) {
  switch (chunks_for(V)) {
    case 1: launch(RowType<RegRow<1>>{}); break;
    case 2: launch(RowType<RegRow<2>>{}); break;
    case 4: launch(RowType<RegRow<4>>{}); break;
    case 8: launch(RowType<RegRow<8>>{}); break;
    case 16: launch(RowType<RegRow<16>>{}); break;
    case 24: launch(RowType<RegRow<24>>{}); break;
    default: launch(RowType<GlobalRow>{}); break;
  }
}
bool filters(const SideParams& p) { return p.use_p || p.use_k; }

int check_rows(int64_t rows, int64_t V, const void* x) {
  if (rows <= 0 || V <= 0 || !x) return set_error(ASPEC_ERR_INVALID, "sampling needs nonempty bf16 logits");
  if (rows > 0x7fffffffLL) return set_error(ASPEC_ERR_UNSUPPORTED, "sampling takes at most 2^31 - 1 rows");
  if (V > (1LL << 24))
    return set_error(ASPEC_ERR_UNSUPPORTED, "sampling covers vocabularies up to 2^24 tokens");
  return ASPEC_OK;
}

}  // namespace
}  // namespace aspec
