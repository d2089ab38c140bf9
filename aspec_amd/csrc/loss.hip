// Vocabulary-sliced loss kernels: softmax-L1 (tiled_l1.py semantics) and cross-entropy, forward
// and backward, alone or fused. HBM-bound streaming reductions.
//
// Forward:
//   row walk (V % 8 == 0, V <= 512*8*8): one or two 512-thread workgroups per CU walk the rows; each row
//   of draft and teacher logits is read from HBM exactly once into registers while the previous
//   row is reduced (max / sum / |p - q| / sign masses);
//   streaming path (any V, any alignment): one workgroup per row, two passes over the row in
//   16-byte chunks.
// Backward: elementwise over rows x V from the saved per-row statistics (one read of x and y,
// one write of dx).
//
// Identical draft and teacher rows go through the same instruction sequence, so their
// probabilities are bitwise equal and both the L1 loss and its subgradient are exactly zero.
#include <algorithm>

#include "common.h"

namespace aspec {
namespace {

constexpr int kStats = 8;  // per-row: mx, 1/sx, my, 1/sy, mass(p>q), mass(p<q), mass(p==q), lse_x

struct LossArgs {
  const uint16_t* x;
  const uint16_t* y;
  const int64_t* yidx;
  int64_t trows;
  const int64_t* target;
  int64_t ignore_index;
  int64_t rows, V;
  float* l1;
  float* ce;
  float* stats;
  int32_t* flags;
  int64_t* amax;  // row argmax (torch.argmax semantics), optional
  const float* g_l1;
  const float* g_ce;
  uint16_t* dx;
};

__device__ __forceinline__ float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Block-wide sums of NVAL floats, broadcast to every thread.
template <int NVAL>
__device__ __forceinline__ void block_reduce(float (&v)[NVAL], float* scratch) {
#pragma unroll
  for (int i = 0; i < NVAL; ++i)
    for (int off = 32; off > 0; off >>= 1) v[i] += __shfl_xor(v[i], off);
  const int wave = threadIdx.x >> 6;
  const int nwaves = blockDim.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int i = 0; i < NVAL; ++i) scratch[i * 32 + wave] = v[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NVAL; ++i) {
    float r = scratch[i * 32];
    for (int w = 1; w < nwaves; ++w) r += scratch[i * 32 + w];
    v[i] = r;
  }
}

__device__ __forceinline__ int64_t teacher_row(const LossArgs& a, int64_t row) {
  if (!a.yidx) return row;
  const int64_t t = a.yidx[row];
  if (t < 0 || t >= a.trows) {
    atomicOr(a.flags, 1);
    return -1;
  }
  return t;
}

__device__ __forceinline__ float bf(uint16_t v) { return bf16_to_f32(v); }

// Wave-uniform reads of kernel inputs through the scalar cache (constant address space): they
// are counted by lgkmcnt, so no wait for them also waits for the vector loads in flight.
template <typename T>
__device__ __forceinline__ T scalar_read(const T* p) {
  return *(const __attribute__((address_space(4))) T*)(p);
}
// The bf16 at p (wave-uniform address), read as its aligned 32-bit word.
__device__ __forceinline__ float scalar_read_bf16(const uint16_t* p) {
  const uintptr_t a = reinterpret_cast<uintptr_t>(p);
  const uint32_t w = scalar_read(reinterpret_cast<const uint32_t*>(a & ~static_cast<uintptr_t>(3)));
  return __uint_as_float((a & 2) ? (w & 0xffff0000u) : (w << 16));
}

// log2-domain exponent of a logit against its row maximum: p = exp2(v*log2e - max*log2e) * (1/sum).
// Forward and backward evaluate e and the product e * (1/sum) alike and compare these two rounded
// values, p against q, so a token that the forward counts in one of the three masses gets that
// case's weight in the backward. For a token that holds nearly all of p and of q the two differ by
// rounding only, and the weight of another case would be off by as much as twice its probability.
// (The row walk forms p from its thread's maximum: the same bits wherever that is the row's, which
// is where a row's largest tokens are.) Identical draft/teacher rows give bitwise equal
// probabilities.
__device__ __forceinline__ float neg_scaled_max(float m) { return -(m * kLog2e); }
__device__ __forceinline__ float scaled_exp2(float v, float nm) { return fexp2(fmaf(v, kLog2e, nm)); }

// Sums over part of a row are taken relative to that part's maximum m, with the offset
// part_offset(m). Its rounding does not cancel at v == m: the exponent there is off by up to half an
// ulp of m log2e, 64 at m = -2^30. Below that (logits masked with -1e10, -1e30 or the type's lowest
// value) the sum would overflow, so there the offset is 0 and every exp2 0: the part adds nothing to
// a row that has anything larger, as in the row's own softmax.
constexpr float kMaskedBelow = -0x1p30f;
__device__ __forceinline__ float part_offset(float m) { return m < kMaskedBelow ? 0.f : neg_scaled_max(m); }

// The part's sum relative to a maximum with the offset `to` instead: scaled by the quotient of the
// two offsets as they were rounded, so a row's sum is that of scaled_exp2 at the row's own offset,
// whatever maxima its parts met. A masked part holds 0, or NaN of a NaN logit, and is not scaled
// (the factor may be infinite).
__device__ __forceinline__ float rebased_sum(float m, float s, float to) {
  return m < kMaskedBelow ? s : s * fexp2(to - neg_scaled_max(m));
}

// The exponent that scaled_exp2 has at the maximum itself: the offset's rounding.
__device__ __forceinline__ float exponent_at_max(float m) { return fmaf(m, kLog2e, neg_scaled_max(m)); }

// Merges two parts' (max, sum) pairs; +inf maxima give NaN, as softmax does.
__device__ __forceinline__ void merge_max_sum(float& m, float& s, float mo, float so) {
  const float mn = fmaxf(m, mo), to = part_offset(mn);
  s = rebased_sum(m, s, to) + rebased_sum(mo, so, to);
  m = mn;
}

// Block-wide merge of NP (max, sum) pairs; the result is broadcast to every thread.
template <int NP>
__device__ __forceinline__ void block_max_sum(float (&m)[NP], float (&s)[NP], float* scratch) {
#pragma unroll
  for (int i = 0; i < NP; ++i)
    for (int off = 32; off > 0; off >>= 1)
      merge_max_sum(m[i], s[i], __shfl_xor(m[i], off), __shfl_xor(s[i], off));
  const int wave = threadIdx.x >> 6;
  const int nwaves = blockDim.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      scratch[(2 * i) * 32 + wave] = m[i];
      scratch[(2 * i + 1) * 32 + wave] = s[i];
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    float mm = scratch[(2 * i) * 32], ss = scratch[(2 * i + 1) * 32];
    for (int w = 1; w < nwaves; ++w) merge_max_sum(mm, ss, scratch[(2 * i) * 32 + w], scratch[(2 * i + 1) * 32 + w]);
    // a row of -inf (or padding only) has no softmax: NaN, as torch gives
    m[i] = mm;
    s[i] = mm == -INFINITY ? NAN : ss;
  }
}

__device__ __forceinline__ float lo_bf(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi_bf(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// The first n of eight consecutive bf16, element by element (the rest 0).
__device__ __forceinline__ uint4 load_part(const uint16_t* p, int n) {
  uint32_t w[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t lo = 2 * k < n ? p[2 * k] : 0u;
    const uint32_t hi = 2 * k + 1 < n ? p[2 * k + 1] : 0u;
    w[k] = lo | (hi << 16);
  }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

constexpr int kWalkThreads = 512;  // threads of the persistent row walk (8 waves, 2 per SIMD)
// Eight bf16 -inf: what the row walk's lanes past the end of a row load.
__device__ const uint4 kNegInfChunk = {0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u};
constexpr int kWalkWaves = kWalkThreads / 64;
// Workgroups of the walk per CU. A row of up to 16384 tokens leaves half the registers free, and a
// second workgroup works while the first waits at a row's barriers: 8192 rows x 8192 tokens 110 ->
// 93 us, x 16000 149 -> 134 us, with dlogits x 8192 160 -> 126 us (a third workgroup spills). With
// dlogits at 16384 tokens two spill already (214 against 210 us).
constexpr int walk_groups(int nv, bool grad) { return nv >= 8 || (nv == 4 && grad) ? 1 : 2; }

// Per-thread max and exp2 values of NV chunks of eight bf16 logits (chunk j of thread t holds
// row elements (j * kWalkThreads + t) * 8 .. +7; value i of `e` is element i % 8 of chunk i / 8).
// max(a, b, c) as the hardware computes it (a NaN operand is skipped, like fmaxf). Through fmaxf
// the compiler first quiets every operand with a max of the value with itself, which more than
// doubles the cost of the row maximum; a NaN logit still reaches the row sum (and so the loss)
// through its exp.
__device__ __forceinline__ float max3_raw(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// min(a, |b|) as one v_min_f32 with an absolute-value source modifier (fminf would first quiet
// both operands).
__device__ __forceinline__ float min_abs_raw(float a, float b) {
  float r;
  asm("v_min_f32_e64 %0, %1, |%2|" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// min(a, |b|, |c|), likewise.
__device__ __forceinline__ float min3_abs_raw(float a, float b, float c) {
  float r;
  asm("v_min3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

struct NoChunkHook {
  __device__ __forceinline__ void operator()(int) const {}
};

// `after_chunk(j)` runs once chunk j's exponentials are computed (the row walk issues a load of
// the next row there, so the loads enter the memory pipeline between VALU work).
template <int NV, typename Hook = NoChunkHook>
__device__ __forceinline__ void chunk_exps(const uint4 (&v)[NV], float (&e)[NV * 8], float& m,
                                           float& sum, const Hook& after_chunk = Hook{}) {
  m = -INFINITY;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const uint32_t w[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
    for (int k = 0; k < 4; ++k) m = max3_raw(m, lo_bf(w[k]), hi_bf(w[k]));
  }
  const float nm = part_offset(m);
  sum = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const uint32_t w[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      e[j * 8 + 2 * k] = scaled_exp2(lo_bf(w[k]), nm);
      e[j * 8 + 2 * k + 1] = scaled_exp2(hi_bf(w[k]), nm);
      sum += e[j * 8 + 2 * k] + e[j * 8 + 2 * k + 1];
    }
    after_chunk(j);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// A (max, sum) pair's sum relative to `to` (>= its max): a pair whose max is -inf passes its sum
// (0, or NaN from a NaN logit) unscaled, that of a part masked with a large finite value is 0 or
// NaN too; a +inf max against a +inf `to` gives NaN, as softmax does.
__device__ __forceinline__ float sum_relative_to(float m, float s, float to) {
  return m == -INFINITY ? s : s * fexp2((m - to) * kLog2e);
}

// Merges every thread's (max, sum) pair for NP quantities: within each wave in registers, then
// across the waves through `slots` (2*NP*kWalkWaves floats, one barrier).
template <int NP>
__device__ __forceinline__ void block_merge(float (&m)[NP], float (&sm)[NP], float* slots) {
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const float mw = wave_allmax(m[i]);
    sm[i] = wave_allsum(sum_relative_to(m[i], sm[i], mw));
    m[i] = mw;
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      slots[(2 * i) * kWalkWaves + wave] = m[i];
      slots[(2 * i + 1) * kWalkWaves + wave] = sm[i];
    }
  }
  lds_barrier();
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    float mm = slots[(2 * i) * kWalkWaves];
#pragma unroll
    for (int w = 1; w < kWalkWaves; ++w) mm = fmaxf(mm, slots[(2 * i) * kWalkWaves + w]);
    float ss = 0.f;
#pragma unroll
    for (int w = 0; w < kWalkWaves; ++w)
      ss += sum_relative_to(slots[(2 * i) * kWalkWaves + w], slots[(2 * i + 1) * kWalkWaves + w], mm);
    m[i] = mm;
    sm[i] = mm == -INFINITY ? NAN : ss;  // a row of -inf (or padding only): NaN, as torch gives
  }
}

// Row argmax as torch.argmax defines it: the first NaN if the row has one (NaN compares above
// everything), else the first index holding the maximum M. Keys order the candidates: NaN at
// index i -> i, maximum at i -> i | 2^31, neither -> kNoKey; the row's argmax is the minimum key.
constexpr uint32_t kNoKey = 0xffffffffu;
__device__ __forceinline__ uint32_t argmax_key(float x, float M, uint32_t idx) {
  return x != x ? idx : (x == M ? (idx | 0x80000000u) : kNoKey);
}

// Block sums of NP floats and the block minimum of one key (same barrier).
template <int NP>
__device__ __forceinline__ void block_sums(float (&v)[NP], uint32_t& key, float* slots,
                                           uint32_t* key_slots) {
#pragma unroll
  for (int i = 0; i < NP; ++i) v[i] = wave_allsum(v[i]);
  key = wave_allmin(key);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int i = 0; i < NP; ++i) slots[i * kWalkWaves + wave] = v[i];
    key_slots[wave] = key;
  }
  lds_barrier();
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    float r = slots[i * kWalkWaves];
#pragma unroll
    for (int w = 1; w < kWalkWaves; ++w) r += slots[i * kWalkWaves + w];
    v[i] = r;
  }
  key = key_slots[0];
#pragma unroll
  for (int w = 1; w < kWalkWaves; ++w) key = min(key, key_slots[w]);
}

// GRAD (with a teacher only): once a row's statistics are final, the walk also writes the row's
// dlogits for the objective sum_r (g_ce[r] ce[r] + g_l1[r] l1[r]) from the p and q it still holds,
// dx = p * (L1 case weight * g_l1 + g_ce) - g_ce at the target (the backward's formula), into `dx`
// (which may be the logits themselves: the row has been read by then).
template <int NV, bool ARGMAX, bool HAS_Y, bool GRAD = false>
__global__ void __launch_bounds__(kWalkThreads)
__attribute__((amdgpu_waves_per_eu(2 * walk_groups(NV, GRAD), 2 * walk_groups(NV, GRAD))))
loss_fwd_persistent(LossArgs args) {
  static_assert(!GRAD || HAS_Y, "the fused gradient needs a teacher");
  __shared__ float merge_slots[4 * kWalkWaves];  // (max, sum) of x and y per wave
  __shared__ float sum_slots[4 * kWalkWaves];    // |p-q|, p>q, p<q masses and sum p per wave
  __shared__ uint32_t key_slots[kWalkWaves];      // argmax key per wave
  // Every field in a local: referencing the kernel argument itself from the loop would make the
  // compiler copy it to scratch.
  const uint16_t* const xbase = args.x;
  const uint16_t* const ybase = args.y;
  const int64_t* const yidx = args.yidx;
  const int64_t trows = args.trows;
  const int64_t* const target = args.target;
  const int64_t ignore = args.ignore_index;
  const int64_t rows = args.rows, V = args.V;
  float* const l1_out = args.l1;
  float* const ce_out = args.ce;
  float* const stats = args.stats;
  int32_t* const flags = args.flags;
  int64_t* const amax_out = args.amax;
  const int tid = threadIdx.x;
  constexpr bool has_y = HAS_Y;  // a compile-time teacher: every path issues the same loads
  const uint32_t nchunks = static_cast<uint32_t>(V / 8);
  uint4 nx[NV], ny[NV];
  // Chunk j of a row (j * kWalkThreads + tid). Every lane loads: a lane past the row's end reads
  // the -inf chunk, a teacher row out of range reads row 0 (its loss is NaN), and the last row of
  // a workgroup re-reads itself as its "next" row. NV is the smallest size that covers V, so only
  // chunks j >= NV/2 can reach past the row's end.
  // (global address space throughout: a select with a generic pointer would make these flat
  // loads, which LDS waits and barriers then also wait for)
  typedef const __attribute__((address_space(1))) uint4* GlobalChunk;
  auto src = [&](const uint16_t* row_base, int j) __attribute__((always_inline)) {
    const uint32_t chunk = static_cast<uint32_t>(j) * static_cast<uint32_t>(kWalkThreads) + tid;
    GlobalChunk p = (GlobalChunk)(row_base) + chunk;
    if (NV == 2 || j >= NV / 2) p = chunk < nchunks ? p : (GlobalChunk)(&kNegInfChunk);
    return (const uint4*)p;
  };
  auto load_x = [&](int j, int64_t r) __attribute__((always_inline)) { nx[j] = *src(xbase + r * V, j); };
  auto load_y = [&](int j, int64_t tr) __attribute__((always_inline)) {
    ny[j] = *src(ybase + (tr >= 0 && tr < trows ? tr : 0) * V, j);
  };
  auto teacher = [&](int64_t r) -> int64_t {  // teacher row of draft row r, -1 when out of range
    if (!has_y) return 0;
    if (!yidx) return r;
    const int64_t t = yidx[r];
    if (t < 0 || t >= trows) {
      atomicOr(flags, 1);
      return -1;
    }
    return t;
  };
  int64_t row = blockIdx.x;
  if (row >= rows) return;
  int64_t trow = teacher(row);
  int64_t tgt = ce_out ? target[row] : ignore;
#pragma unroll
  for (int j = 0; j < NV; ++j) load_x(j, row);
  if (has_y) {
#pragma unroll
    for (int j = 0; j < NV; ++j) load_y(j, trow);
  }
  while (row < rows) {
    // The next row's teacher index and target: loaded here, first used after the next row's draft
    // logits have been requested (so waiting for them waits for nothing else).
    const int64_t next = row + gridDim.x;
    const int64_t nsafe = next < rows ? next : row;
    const int64_t tidx_n = has_y && yidx ? scalar_read(yidx + nsafe) : nsafe;
    const int64_t tgt_n = ce_out ? scalar_read(target + nsafe) : ignore;
    // the CE target logit (from cache: the row has just been read)
    const bool tgt_ok = tgt != ignore && tgt >= 0 && tgt < V;
    const float target_logit = tgt_ok ? scalar_read_bf16(xbase + row * V + tgt) : 0.f;
    float ex[NV * 8], ey[NV * 8];
    float m[2], sm[2];
    chunk_exps<NV>(nx, ex, m[0], sm[0]);
    m[1] = -INFINITY;
    sm[1] = 0.f;
    // The next row's draft logits stream in while the teacher's exponentials are computed (one
    // chunk per step, into the registers chunk_exps has just consumed), its teacher logits during
    // the L1 masses below.
    if (has_y) {
      chunk_exps<NV>(ny, ey, m[1], sm[1], [&](int j) __attribute__((always_inline)) { load_x(j, nsafe); });
    } else {
#pragma unroll
      for (int j = 0; j < NV; ++j) load_x(j, nsafe);
    }
    const float mx_local = m[0], my_local = m[1], sx_local = sm[0];
    block_merge<2>(m, sm, merge_slots);
    uint32_t key = kNoKey;
    if (ARGMAX) {
      const float M = m[0];
      if (fabsf(M) >= 0x1p-14f && M >= kMaskedBelow && M < INFINITY && sm[0] == sm[0]) {
        // A finite row without NaN whose maximum is not tiny: a thread holding M finds its first
        // maximal element among its exp values, which hold exp2(x log2e - M log2e) (chunk_exps).
        // The maximum gives exactly `emax` (same expression), and any other bf16 logit differs
        // from M by at least |M| 2^-8, far above the rounding of M log2e, so it never does.
        if (mx_local == M) {
          const float emax = scaled_exp2(M, neg_scaled_max(M));
          uint32_t i0 = 0;  // first exp value equal to emax (immediates: nothing hoisted per value)
#pragma unroll
          for (int i = NV * 8 - 1; i >= 0; --i) i0 = ex[i] == emax ? static_cast<uint32_t>(i) : i0;
          key = ((((i0 >> 3) * kWalkThreads + tid) << 3) + (i0 & 7)) | 0x80000000u;
        }
      } else {
        // a NaN, an infinity, an all masked row or a tiny maximum: rescan the (cache-resident) row
        const uint16_t* xr = xbase + row * V;
        for (int64_t i = tid; i < V; i += kWalkThreads)
          key = min(key, argmax_key(bf(xr[i]), M, static_cast<uint32_t>(i)));
      }
    }
    // p = e * 2^((m_local - M) log2e) / S per thread (0 for threads whose chunk is all -inf)
    const float cx = (mx_local == -INFINITY ? 0.f : fexp2((mx_local - m[0]) * kLog2e)) / sm[0];
    const float cy = (my_local == -INFINITY ? 0.f : fexp2((my_local - m[1]) * kLog2e)) / sm[1];
    float acc[4] = {0.f, 0.f, 0.f, 0.f};  // |p-q|, mass p>q, mass p<q, sum p
    int64_t trow_n = 0;
    if (has_y) {
      trow_n = tidx_n;
      if (yidx && next < rows && (trow_n < 0 || trow_n >= trows)) {
        if (tid == 0) atomicOr(flags, 1);
        trow_n = -1;
      }
      // Every chunk but the last (the only one that can reach past the row's end): |p - q| and,
      // unless the chunk holds an exact tie, the signed mass S = sum copysign(p, p - q), seven VALU
      // operations per element; then, with T = sum p over those chunks, mass(p > q) = (T + S) / 2
      // and mass(p < q) = (T - S) / 2. A chunk with a tie (identical rows, both logits masked)
      // and the last chunk count their masses element by element, so ties keep their own mass
      // exactly (identical rows give exactly zero masses and gradient).
      float sgn = 0.f, exact_sum = 0.f;
      bool any_fast = false;
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        float pj[8], dj[8];
        float mj = INFINITY;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          pj[k] = ex[j * 8 + k] * cx;
          dj[k] = pj[k] - ey[j * 8 + k] * cy;
          acc[0] += fabsf(dj[k]);
          mj = min_abs_raw(mj, dj[k]);
        }
        if (j < NV - 1 && mj != 0.f) {
          any_fast = true;
#pragma unroll
          for (int k = 0; k < 8; ++k) sgn += copysignf(pj[k], dj[k]);
        } else {
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            acc[1] += dj[k] > 0.f ? pj[k] : 0.f;
            acc[2] += dj[k] < 0.f ? pj[k] : 0.f;
            exact_sum += pj[k];
          }
        }
        if constexpr (!GRAD) load_y(j, trow_n);  // GRAD: after this chunk's dlogits (below)
        __builtin_amdgcn_sched_barrier(0);
      }
      const float total = cx * sx_local;
      if (any_fast) {
        const float t = total - exact_sum;
        acc[1] += 0.5f * (t + sgn);
        acc[2] += 0.5f * (t - sgn);
      }
      acc[3] = total;
    }
    block_sums<4>(acc, key, sum_slots, key_slots);
    if constexpr (GRAD) {
      // the row's objective weights (wave-uniform) and the three L1 case weights (the backward's
      // centered terms, tiled_l1.py:107-127)
      const float wl1 = trow >= 0 ? scalar_read(args.g_l1 + row) : NAN;
      const float wce = tgt != ignore ? scalar_read(args.g_ce + row) : 0.f;
      const float pos = acc[1], neg = acc[2], zero = acc[3] - acc[1] - acc[2];
      const float k_gt = (2.f * neg + zero) * wl1 + wce;
      const float k_lt = (-2.f * pos - zero) * wl1 + wce;
      const float k_eq = (neg - pos) * wl1 + wce;
      uint16_t* const drow = args.dx + row * V;
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const uint32_t chunk = static_cast<uint32_t>(j) * static_cast<uint32_t>(kWalkThreads) + tid;
        float d[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const float pv = ex[j * 8 + k] * cx, qv = ey[j * 8 + k] * cy;
          d[k] = pv * (pv > qv ? k_gt : (pv < qv ? k_lt : k_eq));
        }
        // the CE target: chunk tgt / 8 belongs to thread (tgt / 8) % kWalkThreads at step
        // (tgt / 8) / kWalkThreads (all wave-uniform but the thread)
        if (tgt_ok && (tgt >> 3) / kWalkThreads == j && static_cast<int64_t>(tid) == (tgt >> 3) % kWalkThreads) {
          switch (static_cast<int>(tgt & 7)) {
            case 0: d[0] -= wce; break;
            case 1: d[1] -= wce; break;
            case 2: d[2] -= wce; break;
            case 3: d[3] -= wce; break;
            case 4: d[4] -= wce; break;
            case 5: d[5] -= wce; break;
            case 6: d[6] -= wce; break;
            default: d[7] -= wce; break;
          }
        }
        if (chunk < nchunks)
          reinterpret_cast<uint4*>(drow)[chunk] =
              make_uint4(pack_bf16x2(d[0], d[1]), pack_bf16x2(d[2], d[3]), pack_bf16x2(d[4], d[5]),
                         pack_bf16x2(d[6], d[7]));
        // the next row's teacher chunk, into registers this row no longer needs
        load_y(j, trow_n);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (tid == 0) {
      if (ARGMAX) amax_out[row] = static_cast<int64_t>(key & 0x7fffffffu);
      const float lse = logf(sm[0]) + m[0];
      float* st = stats + row * kStats;
      st[0] = m[0]; st[1] = 1.f / sm[0]; st[2] = m[1]; st[3] = 1.f / sm[1];
      st[4] = acc[1]; st[5] = acc[2]; st[6] = acc[3] - acc[1] - acc[2]; st[7] = lse;
      if (l1_out) l1_out[row] = (has_y && trow >= 0) ? acc[0] : NAN;
      if (ce_out) {
        float v = 0.f;
        if (tgt != ignore) {
          if (!tgt_ok) { atomicOr(flags, 2); v = NAN; }
          else v = lse - target_logit;
        }
        ce_out[row] = v;
      }
    }
    row = next;
    trow = trow_n;
    tgt = tgt_n;
  }
}

// Rows the walk does not take (V > 32768, V % 8 != 0, rows off 16-byte alignment): one workgroup
// per row, two passes over it in chunks of eight logits. Pass 1 keeps each thread's running maximum
// and sum (rescaled when a chunk raises the maximum) and the chunk that holds its maximum; pass 2
// forms p and q from the row's statistics and sums the masses, last chunks first: those are still
// in the L2.
//
// A chunk starts at a multiple of eight logits of its row, so at any 2-byte address when V % 8 != 0:
// its load is one 16-byte access all the same (global memory takes any alignment on this target).
//
// What bounds it: the VALU and both passes' reads, nearly alike. A 151936-token row and its teacher are
// 608 KB, more than a CU's registers and LDS hold, so they are read twice; at 2048 rows against 1024
// teacher rows the two passes read 2.43 GB past the L2 in 375 us (6.5 TB/s), with 34 VALU instructions
// per logit pair busy 0.92 of the time (element loads in three passes took 1467 us). Kept: two chunks
// in flight per thread (one or three measured the same) and 512 threads (1024: 483 us at 2048 rows
// and no faster at 64 rows; 256: the same at 2048 rows, 57 against 41 us at 64).
template <int THREADS, bool HAS_Y>
__global__ void __launch_bounds__(THREADS) loss_fwd_streaming(LossArgs a) {
  __shared__ float scratch[4 * 32];
  __shared__ uint32_t keys[THREADS / 64];
  const int64_t row = blockIdx.x;
  constexpr bool has_y = HAS_Y;
  const int64_t trow = has_y ? teacher_row(a, row) : 0;
  const uint16_t* const xr = a.x + row * a.V;
  // a teacher row out of range: row 0 is read and q is NaN below
  const uint16_t* const yr = has_y ? a.y + max(trow, static_cast<int64_t>(0)) * a.V : nullptr;
  const uint16_t* const kNegInf = reinterpret_cast<const uint16_t*>(&kNegInfChunk);
  const int tid = threadIdx.x;
  const uint32_t full = static_cast<uint32_t>(a.V / 8);  // whole chunks
  const int tail = static_cast<int>(a.V & 7);            // logits after them: one per thread 0 .. tail - 1
  const int64_t tail_at = full * 8LL + tid;
  const bool in_tail = tid < tail;

  // ---- pass 1: (max, sum) of the thread's chunks. The sum is relative to `ref`, a maximum of the
  // thread's that is replaced only when a chunk exceeds it by more than kSlack: nearly every chunk
  // then costs one compare instead of a rescaling, and exp2 of the shifted logits stays far from
  // overflow (2^(1.44 kSlack) per element).
  struct Running {
    float max = -INFINITY, ref = -INFINITY, nref = 0.f, sum = 0.f;
  } run[2];
  uint32_t best = 0;  // the first of the thread's chunks that holds its maximum
  constexpr float kSlack = 24.f;
  auto absorb = [&](const uint4& v, Running& r) __attribute__((always_inline)) -> bool {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    float x[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) x[2 * k] = lo_bf(w[k]), x[2 * k + 1] = hi_bf(w[k]);
    const float cm = max3_raw(max3_raw(x[0], x[1], x[2]), max3_raw(x[3], x[4], x[5]), max3_raw(x[6], x[7], x[7]));
    const bool grow = cm > r.max;
    r.max = grow ? cm : r.max;
    if (__any(cm > r.ref + kSlack)) {
      if (cm > r.ref) {
        r.nref = part_offset(cm);
        r.sum = rebased_sum(r.ref, r.sum, r.nref);
        r.ref = cm;
      }
    }
    float e[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) e[k] = scaled_exp2(x[k], r.nref);
    r.sum += ((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]));
    return grow;
  };
  // Steps of THREADS chunks (one per thread), two at a time, the next two loading meanwhile. A lane
  // past the last whole chunk reads the -inf chunk, which adds nothing.
  constexpr int kSteps = 2;
  const int groups = static_cast<int>((full + kSteps * THREADS - 1) / (kSteps * THREADS));
  uint4 nx[kSteps], ny[kSteps];
  auto fetch = [&](int g) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
      const uint32_t c = static_cast<uint32_t>(g * kSteps + u) * THREADS + tid;
      nx[u] = load_chunk(c < full ? xr + c * 8LL : kNegInf);
      if (has_y) ny[u] = load_chunk(c < full ? yr + c * 8LL : kNegInf);
    }
  };
  if (groups > 0) fetch(0);
  for (int g = 0; g < groups; ++g) {
    uint4 xv[kSteps], yv[kSteps];
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
      xv[u] = nx[u];
      if (has_y) yv[u] = ny[u];
    }
    fetch(min(g + 1, groups - 1));  // the last group stays for pass 2, which begins with it
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
      if (absorb(xv[u], run[0])) best = static_cast<uint32_t>(g * kSteps + u) * THREADS + tid;
      if (has_y) absorb(yv[u], run[1]);
    }
  }
  // (max, sum relative to it); a sum that is NaN, of a NaN or +inf logit, stays so
  float m[2], s[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    m[i] = run[i].max;
    s[i] = rebased_sum(run[i].ref, run[i].sum, part_offset(m[i]));
  }
  if (in_tail) {
    const float x = bf(xr[tail_at]);
    if (x > m[0]) best = full;
    merge_max_sum(m[0], s[0], x, scaled_exp2(x, part_offset(x)));
    if (has_y) {
      const float y = bf(yr[tail_at]);
      merge_max_sum(m[1], s[1], y, scaled_exp2(y, part_offset(y)));
    }
  }
  const float own_max = m[0];
  block_max_sum<2>(m, s, scratch);

  if (a.amax) {  // first NaN, else first maximum (torch.argmax)
    uint32_t key = kNoKey;
    if (s[0] == s[0]) {
      // no NaN and a finite maximum: a thread that holds it looks for it in the chunk it noted
      if (own_max == m[0]) {
        if (best == full) {
          key = argmax_key(m[0], m[0], static_cast<uint32_t>(tail_at));
        } else {
          for (int k = 7; k >= 0; --k)
            if (bf(xr[best * 8LL + k]) == m[0]) key = argmax_key(m[0], m[0], static_cast<uint32_t>(best * 8 + k));
        }
      }
    } else {
      for (int64_t i = tid; i < a.V; i += THREADS)
        key = min(key, argmax_key(bf(xr[i]), m[0], static_cast<uint32_t>(i)));
    }
    key = wave_allmin(key);
    if ((tid & 63) == 0) keys[tid >> 6] = key;
    __syncthreads();
    if (tid == 0) {
      for (int w = 1; w < THREADS / 64; ++w) key = min(key, keys[w]);
      a.amax[row] = static_cast<int64_t>(key & 0x7fffffffu);
    }
  }

  // ---- pass 2: the L1 masses
  const float nmx = neg_scaled_max(m[0]), nmy = neg_scaled_max(m[1]);
  const float ix = 1.f / s[0], iy = trow < 0 ? NAN : 1.f / s[1];
  float acc[4] = {0.f, 0.f, 0.f, 0.f};  // |p-q|, mass p>q, mass p<q, mass p==q
  if (has_y) {
    // The masses above and below are summed each by itself, so a small one beside a large one keeps
    // its digits; a chunk with an exact tie also tells ties from the rest, and so does a row with NaN
    // probabilities on either side (every difference is NaN), whose p all counts as neither.
    auto masses = [&](const uint4& xv, const uint4& yv) __attribute__((always_inline)) {
      const uint32_t xw[4] = {xv.x, xv.y, xv.z, xv.w}, yw[4] = {yv.x, yv.y, yv.z, yv.w};
      float p[8], d[8], low = INFINITY;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t wx = xw[k >> 1], wy = yw[k >> 1];
        p[k] = scaled_exp2((k & 1) ? hi_bf(wx) : lo_bf(wx), nmx) * ix;
        d[k] = p[k] - scaled_exp2((k & 1) ? hi_bf(wy) : lo_bf(wy), nmy) * iy;
      }
#pragma unroll
      for (int k = 0; k < 8; k += 2) low = min3_abs_raw(low, d[k], d[k + 1]);
      acc[0] += ((fabsf(d[0]) + fabsf(d[1])) + (fabsf(d[2]) + fabsf(d[3]))) +
                ((fabsf(d[4]) + fabsf(d[5])) + (fabsf(d[6]) + fabsf(d[7])));
      if (low > 0.f && low < INFINITY) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const bool above = d[k] > 0.f;
          acc[1] += above ? p[k] : 0.f;
          acc[2] += above ? 0.f : p[k];
        }
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          acc[1] += d[k] > 0.f ? p[k] : 0.f;
          acc[2] += d[k] < 0.f ? p[k] : 0.f;
          acc[3] += (d[k] > 0.f) | (d[k] < 0.f) ? 0.f : p[k];
        }
      }
    };
    for (int g = groups - 1; g >= 0; --g) {
      uint4 xv[kSteps], yv[kSteps];
#pragma unroll
      for (int u = 0; u < kSteps; ++u) xv[u] = nx[u], yv[u] = ny[u];
      fetch(max(g - 1, 0));
#pragma unroll
      for (int u = 0; u < kSteps; ++u) masses(xv[u], yv[u]);
    }
    if (in_tail) {
      const float p = scaled_exp2(bf(xr[tail_at]), nmx) * ix;
      const float d = p - scaled_exp2(bf(yr[tail_at]), nmy) * iy;
      acc[0] += fabsf(d);
      acc[1] += d > 0.f ? p : 0.f;
      acc[2] += d < 0.f ? p : 0.f;
      acc[3] += (d > 0.f) | (d < 0.f) ? 0.f : p;
    }
    block_reduce<4>(acc, scratch);
  }
  if (tid == 0) {
    // less the rounding of the offset, which all of S_x carries
    const float lse = (logf(s[0]) - kLn2 * exponent_at_max(m[0])) + m[0];
    float* st = a.stats + row * kStats;
    st[0] = m[0]; st[1] = ix; st[2] = m[1]; st[3] = iy;
    st[4] = acc[1]; st[5] = acc[2]; st[6] = acc[3]; st[7] = lse;
    if (a.l1) a.l1[row] = (has_y && trow >= 0) ? acc[0] : NAN;
    if (a.ce) {
      const int64_t t = a.target[row];
      float v = 0.f;
      if (t != a.ignore_index) {
        if (t < 0 || t >= a.V) { atomicOr(a.flags, 2); v = NAN; }
        else v = lse - bf(xr[t]);
      }
      a.ce[row] = v;
    }
  }
}

// dx = g_ce * (p - onehot(t)) + g_l1 * p * centered  (tiled_l1.py:107-127 for the L1 part), of the
// eight logits of one chunk (16-byte accesses at any alignment; a row's last, partial chunk goes
// element by element). `row_read` reads what the row's chunks share.
template <typename Read>
__device__ __forceinline__ void grad_chunk(const LossArgs& a, int64_t row, int64_t chunk, bool live_chunk,
                                           const Read& row_read) {
  const bool has_y = a.y != nullptr;
  float st[kStats];
#pragma unroll
  for (int i = 0; i < kStats; ++i) st[i] = row_read(a.stats + row * kStats + i);
  const float gl1 = (has_y && a.g_l1) ? row_read(a.g_l1 + row) : 0.f;
  float gce = 0.f;
  int64_t tgt = -1;
  if (a.g_ce) {
    tgt = row_read(a.target + row);
    gce = tgt == a.ignore_index ? 0.f : row_read(a.g_ce + row);
  }
  int64_t trow = 0;
  if (has_y) {
    trow = a.yidx ? row_read(a.yidx + row) : row;
    if (trow < 0 || trow >= a.trows) trow = -1;
  }
  if (!live_chunk) return;
  // dx = p * (L1 weight of the element's case + g_ce) - g_ce at the target, p = e_x * (1/S_x) with
  // e = exp2(v log2e - max log2e) (scaled_exp2) as in the forward.
  const float nmx = neg_scaled_max(st[0]), nmy = neg_scaled_max(st[2]);
  const float pos = st[4], neg = st[5], zero = st[6];
  const float k_gt = (2.f * neg + zero) * gl1 + gce;
  const float k_lt = (-2.f * pos - zero) * gl1 + gce;
  const float k_eq = (neg - pos) * gl1 + gce;
  const int64_t col0 = chunk * 8;
  const uint16_t* xr = a.x + row * a.V;
  const uint16_t* yr = (has_y && trow >= 0) ? a.y + trow * a.V : nullptr;
  const int live = static_cast<int>(min(a.V - col0, static_cast<int64_t>(8)));
  const uint4 xs = live == 8 ? load_chunk(xr + col0) : load_part(xr + col0, live);
  const uint4 ys = !yr ? make_uint4(0, 0, 0, 0) : live == 8 ? load_chunk(yr + col0) : load_part(yr + col0, live);
  const uint32_t xw[4] = {xs.x, xs.y, xs.z, xs.w};
  const uint32_t yw[4] = {ys.x, ys.y, ys.z, ys.w};
  float d[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float x = (e & 1) ? __uint_as_float(xw[e >> 1] & 0xffff0000u) : __uint_as_float(xw[e >> 1] << 16);
    const float p = scaled_exp2(x, nmx) * st[1];
    float k = gce;  // no teacher: the CE part alone
    if (has_y) {
      if (yr) {
        const float y = (e & 1) ? __uint_as_float(yw[e >> 1] & 0xffff0000u) : __uint_as_float(yw[e >> 1] << 16);
        const float q = scaled_exp2(y, nmy) * st[3];
        k = p > q ? k_gt : (p < q ? k_lt : k_eq);
      } else {
        k = NAN;  // teacher row out of range
      }
    }
    d[e] = p * k;
  }
  // the CE target column (one lane of the row)
  if (gce != 0.f && tgt >= col0 && tgt < col0 + 8) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (col0 + e == tgt) d[e] -= gce;
  }
  uint32_t out[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) out[e] = pack_bf16x2(d[2 * e], d[2 * e + 1]);
  uint16_t* const dr = a.dx + row * a.V + col0;
  if (live == 8) {
    store_chunk(dr, make_uint4(out[0], out[1], out[2], out[3]));
  } else {
#pragma unroll
    for (int e = 0; e < 7; ++e)
      if (e < live) dr[e] = static_cast<uint16_t>(out[e >> 1] >> ((e & 1) * 16));
  }
}

// Each workgroup pass covers 256 consecutive chunks of one row, so the row's statistics, upstream
// gradients, target and teacher index are wave-uniform and read through the scalar cache; only the
// logits and dx use the vector memory path.
constexpr int kBwdThreads = 256;

__global__ void __launch_bounds__(kBwdThreads) loss_bwd_rows_kernel(LossArgs a) {
  const int64_t per_row = (a.V + 7) / 8;
  const int64_t segs_per_row = (per_row + kBwdThreads - 1) / kBwdThreads;
  const int64_t segs = a.rows * segs_per_row;
  for (int64_t seg = blockIdx.x; seg < segs; seg += gridDim.x) {
    const int64_t row = seg / segs_per_row;
    const int64_t chunk = (seg - row * segs_per_row) * kBwdThreads + threadIdx.x;
    grad_chunk(a, row, chunk, chunk < per_row, [](const auto* p) { return scalar_read(p); });
  }
}

// Short rows, which would leave most of such a workgroup idle: the chunks of all rows in one sequence,
// each thread reading its row's statistics.
__global__ void __launch_bounds__(kBwdThreads) loss_bwd_short_kernel(LossArgs a) {
  const int64_t per_row = (a.V + 7) / 8;
  const int64_t chunks = a.rows * per_row;
  for (int64_t c = static_cast<int64_t>(blockIdx.x) * kBwdThreads + threadIdx.x; c < chunks;
       c += static_cast<int64_t>(gridDim.x) * kBwdThreads) {
    const int64_t row = c / per_row;
    grad_chunk(a, row, c - row * per_row, true, [](const auto* p) { return *p; });
  }
}

template <int NV>
void launch_walk(const LossArgs& a, int cus, hipStream_t s) {
  const dim3 block(kWalkThreads);
  const dim3 walk(static_cast<uint32_t>(std::min<int64_t>(a.rows, cus * walk_groups(NV, a.dx != nullptr))));
  if (a.dx) {  // the fused forward + dlogits (teacher present, checked by the entry point)
    if (a.amax) hipLaunchKernelGGL((loss_fwd_persistent<NV, true, true, true>), walk, block, 0, s, a);
    else hipLaunchKernelGGL((loss_fwd_persistent<NV, false, true, true>), walk, block, 0, s, a);
    return;
  }
  if (a.y) {
    if (a.amax) hipLaunchKernelGGL((loss_fwd_persistent<NV, true, true>), walk, block, 0, s, a);
    else hipLaunchKernelGGL((loss_fwd_persistent<NV, false, true>), walk, block, 0, s, a);
  } else {
    if (a.amax) hipLaunchKernelGGL((loss_fwd_persistent<NV, true, false>), walk, block, 0, s, a);
    else hipLaunchKernelGGL((loss_fwd_persistent<NV, false, false>), walk, block, 0, s, a);
  }
}

// Rows up to kShortRow logits take one wave each in the two-pass forward: a workgroup's waves would be
// mostly idle and meet at every reduction. 200000 rows x 9 logits 1165 -> 314 us with 64 instead of 256
// threads, 20000 x 1001 145 -> 57, 8192 x 2047 72 -> 46; at 64 rows of 4095 it is the slower one,
// 26 against 23.6 us.
constexpr int64_t kShortRow = 2048;
// Rows up to kShortChunks chunks take the backward over all rows' chunks: 200000 rows x 9 logits
// 171 -> 10 us against a workgroup per row, 65536 x 257 63 -> 27, 20000 x 1001 31 -> 27; 8192 x 2047
// 25 -> 27.
constexpr int64_t kShortChunks = 128;
template <int THREADS>
void launch_streaming(const LossArgs& a, dim3 grid, hipStream_t s) {
  if (a.y) hipLaunchKernelGGL((loss_fwd_streaming<THREADS, true>), grid, dim3(THREADS), 0, s, a);
  else hipLaunchKernelGGL((loss_fwd_streaming<THREADS, false>), grid, dim3(THREADS), 0, s, a);
}

int launch_fwd(const LossArgs& a, hipStream_t s) {
  const bool vec = a.V % 8 == 0 && (reinterpret_cast<uintptr_t>(a.x) & 15) == 0 &&
                   (!a.y || (reinterpret_cast<uintptr_t>(a.y) & 15) == 0);
  const dim3 grid(static_cast<uint32_t>(a.rows));
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
    return set_error(ASPEC_ERR_RUNTIME, "cannot query the GPU's compute-unit count");
  if (a.dx && !(vec && a.V <= kWalkThreads * 8 * 8 && (reinterpret_cast<uintptr_t>(a.dx) & 15) == 0))
    return set_error(ASPEC_ERR_UNSUPPORTED, "the fused loss forward + dlogits needs V %% 8 == 0, V <= %d "
                     "and 16-byte aligned rows", kWalkThreads * 8 * 8);
  if (vec && a.V <= kWalkThreads * 8 * 2) {
    launch_walk<2>(a, cus, s);
  } else if (vec && a.V <= kWalkThreads * 8 * 4) {
    launch_walk<4>(a, cus, s);
  } else if (vec && a.V <= kWalkThreads * 8 * 8) {
    launch_walk<8>(a, cus, s);
  } else if (a.V <= kShortRow) {
    launch_streaming<64>(a, grid, s);
  } else if (a.V <= 8192) {  // one workgroup per row, as many threads as its chunks keep busy
    launch_streaming<256>(a, grid, s);
  } else {
    launch_streaming<512>(a, grid, s);
  }
  return check_launch("loss forward");
}

int launch_bwd(const LossArgs& a, hipStream_t s) {
  const int64_t per_row = (a.V + 7) / 8;
  const bool by_row = per_row > kShortChunks;
  const int64_t blocks = by_row ? a.rows * ((per_row + kBwdThreads - 1) / kBwdThreads)
                                : (a.rows * per_row + kBwdThreads - 1) / kBwdThreads;
  const dim3 grid(static_cast<uint32_t>(std::min<int64_t>(blocks, 256 * 64)));
  if (by_row) hipLaunchKernelGGL(loss_bwd_rows_kernel, grid, dim3(kBwdThreads), 0, s, a);
  else hipLaunchKernelGGL(loss_bwd_short_kernel, grid, dim3(kBwdThreads), 0, s, a);
  return check_launch("loss backward");
}

// Two bf16 in one word, each times s: fp32 product, one round to nearest even.
__device__ __forceinline__ uint32_t scale_bf16_pair(uint32_t w, float s) {
  return pack_bf16x2(__uint_as_float(w << 16) * s, __uint_as_float(w & 0xffff0000u) * s);
}

// x *= s in place over n bf16 values, s read on the device. When s == 1 every product equals its
// input bit for bit, so each workgroup returns before touching x (the usual upstream gradient of a
// loss: the multiply costs a launch instead of a pass over x). n8 16-byte groups, then the tail.
__global__ void __launch_bounds__(256) scale_bf16_kernel(uint16_t* x, int64_t n, int64_t n8,
                                                         const float* scalar) {
  const float s = scalar_read(scalar);
  if (s == 1.0f) return;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
  const int64_t first = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  uint4* v = reinterpret_cast<uint4*>(x);
  for (int64_t i = first; i < n8; i += stride) {
    uint4 w = v[i];
    w.x = scale_bf16_pair(w.x, s);
    w.y = scale_bf16_pair(w.y, s);
    w.z = scale_bf16_pair(w.z, s);
    w.w = scale_bf16_pair(w.w, s);
    v[i] = w;
  }
  for (int64_t i = n8 * 8 + first; i < n; i += stride)
    x[i] = f32_to_bf16_bits(bf16_to_f32(x[i]) * s);
}

int check_common(int64_t rows, int64_t V, const void* x) {
  if (rows <= 0 || V <= 0 || !x)
    return set_error(ASPEC_ERR_INVALID, "loss kernels require nonempty logits with a vocabulary dimension");
  return ASPEC_OK;
}

}  // namespace
}  // namespace aspec

using namespace aspec;

extern "C" int aspec_loss_stats_floats(void) { return kStats; }

extern "C" int aspec_ce_l1_argmax_fwd(const void* logits, const void* teacher,
                                      const int64_t* teacher_index, int64_t teacher_rows,
                                      const int64_t* targets, int64_t ignore_index, int64_t rows,
                                      int64_t vocab, float* l1_out, float* ce_out, int64_t* argmax_out,
                                      float* stats, int32_t* status_flags, void* stream) {
  int rc = check_common(rows, vocab, logits);
  if (rc) return rc;
  if (!stats || !status_flags) return set_error(ASPEC_ERR_INVALID, "stats and status buffers are required");
  if (l1_out && !teacher) return set_error(ASPEC_ERR_INVALID, "L1 needs teacher logits");
  if (ce_out && !targets) return set_error(ASPEC_ERR_INVALID, "cross-entropy needs targets");
  if (teacher_index && teacher_rows <= 0) return set_error(ASPEC_ERR_INVALID, "indexed teacher table is empty");
  LossArgs a = {};
  a.x = static_cast<const uint16_t*>(logits);
  a.y = static_cast<const uint16_t*>(teacher);
  a.yidx = teacher_index;
  a.trows = teacher_index ? teacher_rows : rows;
  a.target = targets;
  a.ignore_index = ignore_index;
  a.rows = rows;
  a.V = vocab;
  a.l1 = l1_out;
  a.ce = ce_out;
  a.stats = stats;
  a.flags = status_flags;
  a.amax = argmax_out;
  if (argmax_out && vocab > 0x7fffffffLL)
    return set_error(ASPEC_ERR_UNSUPPORTED, "argmax needs a vocabulary below 2^31");
  return launch_fwd(a, static_cast<hipStream_t>(stream));
}

extern "C" int aspec_ce_l1_fused_fwd_bwd(const void* logits, const void* teacher,
                                          const int64_t* teacher_index, int64_t teacher_rows,
                                          const int64_t* targets, int64_t ignore_index, int64_t rows,
                                          int64_t vocab, const float* grad_ce, const float* grad_l1,
                                          float* l1_out, float* ce_out, int64_t* argmax_out,
                                          float* stats, void* grad_logits, int32_t* status_flags,
                                          void* stream) {
  int rc = check_common(rows, vocab, logits);
  if (rc) return rc;
  if (!teacher || !targets || !grad_ce || !grad_l1 || !grad_logits || !stats || !status_flags || !l1_out || !ce_out)
    return set_error(ASPEC_ERR_INVALID, "the fused loss needs teacher logits, targets, both per-row "
                     "gradients, outputs, stats, a status buffer and a dlogits buffer");
  if (teacher_index && teacher_rows <= 0) return set_error(ASPEC_ERR_INVALID, "indexed teacher table is empty");
  if (argmax_out && vocab > 0x7fffffffLL)
    return set_error(ASPEC_ERR_UNSUPPORTED, "argmax needs a vocabulary below 2^31");
  LossArgs a = {};
  a.x = static_cast<const uint16_t*>(logits);
  a.y = static_cast<const uint16_t*>(teacher);
  a.yidx = teacher_index;
  a.trows = teacher_index ? teacher_rows : rows;
  a.target = targets;
  a.ignore_index = ignore_index;
  a.rows = rows;
  a.V = vocab;
  a.l1 = l1_out;
  a.ce = ce_out;
  a.stats = stats;
  a.flags = status_flags;
  a.amax = argmax_out;
  a.g_ce = grad_ce;
  a.g_l1 = grad_l1;
  a.dx = static_cast<uint16_t*>(grad_logits);
  return launch_fwd(a, static_cast<hipStream_t>(stream));
}

extern "C" int aspec_scale_bf16_by_device_scalar(void* x, int64_t n, const float* scalar,
                                                  void* stream) {
  if (n < 0 || (n > 0 && (!x || !scalar)))
    return set_error(ASPEC_ERR_INVALID, "scaling needs a buffer, a size >= 0 and a device scalar");
  if (n == 0) return ASPEC_OK;
  const int64_t n8 = (reinterpret_cast<uintptr_t>(x) & 15) == 0 ? n / 8 : 0;
  const int64_t work = std::max<int64_t>(n8, n - n8 * 8);
  const int64_t grid = std::min<int64_t>((work + 255) / 256, 1024);
  hipLaunchKernelGGL(scale_bf16_kernel, dim3(static_cast<uint32_t>(grid)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<uint16_t*>(x), n, n8, scalar);
  return check_launch("bf16 scale");
}

extern "C" int aspec_ce_l1_fwd(const void* logits, const void* teacher, const int64_t* teacher_index,
                               int64_t teacher_rows, const int64_t* targets, int64_t ignore_index,
                               int64_t rows, int64_t vocab, float* l1_out, float* ce_out,
                               float* stats, int32_t* status_flags, void* stream) {
  return aspec_ce_l1_argmax_fwd(logits, teacher, teacher_index, teacher_rows, targets, ignore_index,
                                rows, vocab, l1_out, ce_out, nullptr, stats, status_flags, stream);
}

extern "C" int aspec_ce_l1_bwd(const void* logits, const void* teacher, const int64_t* teacher_index,
                               int64_t teacher_rows, const int64_t* targets, int64_t ignore_index,
                               int64_t rows, int64_t vocab, const float* stats,
                               const float* grad_l1, const float* grad_ce, void* grad_logits,
                               void* stream) {
  int rc = check_common(rows, vocab, logits);
  if (rc) return rc;
  if (!stats || !grad_logits) return set_error(ASPEC_ERR_INVALID, "stats and gradient buffers are required");
  if (grad_l1 && !teacher) return set_error(ASPEC_ERR_INVALID, "L1 gradient needs teacher logits");
  if (grad_ce && !targets) return set_error(ASPEC_ERR_INVALID, "cross-entropy gradient needs targets");
  LossArgs a = {};
  a.x = static_cast<const uint16_t*>(logits);
  a.y = grad_l1 ? static_cast<const uint16_t*>(teacher) : nullptr;
  a.yidx = teacher_index;
  a.trows = teacher_index ? teacher_rows : rows;
  a.target = targets;
  a.ignore_index = ignore_index;
  a.rows = rows;
  a.V = vocab;
  a.stats = const_cast<float*>(stats);
  a.g_l1 = grad_l1;
  a.g_ce = grad_ce;
  a.dx = static_cast<uint16_t*>(grad_logits);
  return launch_bwd(a, static_cast<hipStream_t>(stream));
}
