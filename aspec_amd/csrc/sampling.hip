// The logits filtered by a temperature, top-k and top-p (aspec/models/ops/loss.py:57-80) and their
// gradient; the support by sampling_support.h.
#include "sampling_support.h"

namespace aspec {
namespace {

template <typename Row, bool FILTER>
__global__ void __launch_bounds__(kSampThreads) __attribute__((amdgpu_waves_per_eu(Row::kWavesPerSimd)))
sampling_fwd_kernel(SampledArgs a) {
  __shared__ Work work;
  int ph = 0;
  const int64_t row = blockIdx.x, V = a.V;
  const SideParams px = a.px;
  Row r;
  r.load(a.x + row * V, V);
  const SideStats s = compute_support<FILTER>(r, V, px, work, ph);
  const RowCtx cx = ctx_of(s);
  const Support sup = support_of(s);
  float* out = a.out + row * V;
  const bool nan_row = (s.flags & kFlagNaN) != 0;
  const bool vec_out = V % 4 == 0 && (reinterpret_cast<uintptr_t>(a.out) & 15) == 0;
  r.chunks([&](int, int32_t base, const uint32_t (&w)[4]) {
    if (base >= V) return;
    float o[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float v = ord_of(bf16f(half_of(w, j)), cx);
      o[j] = nan_row ? __builtin_nanf("") : (kept(sup, v, base + j) ? v : -INFINITY);
    }
    if (vec_out && base + 8 <= V) {
      *reinterpret_cast<float4*>(out + base) = make_float4(o[0], o[1], o[2], o[3]);
      *reinterpret_cast<float4*>(out + base + 4) = make_float4(o[4], o[5], o[6], o[7]);
    } else {
      for (int j = 0; j < 8 && base + j < V; ++j) out[base + j] = o[j];
    }
    __builtin_amdgcn_sched_barrier(0);
  });
  if (threadIdx.x == 0) store_side(a.stats + row * kSideWords, s);
}

// d logits = keep * g * (1/T), minus, with a temperature, sum(keep * g) / T shared by the tokens
// equal to the max (the gradient of the max subtraction; amax spreads it evenly over ties)
template <typename Row>
__global__ void __launch_bounds__(kSampThreads) sampling_bwd_kernel(SampledArgs a) {
  __shared__ Red red;
  int ph = 0;
  const int64_t row = blockIdx.x, V = a.V;
  Row r;
  r.load(a.x + row * V, V);
  const SideStats s = load_side(a.stats + row * kSideWords);
  const RowCtx cx = ctx_of(s);
  const Support sup = support_of(s);
  const float* g = a.gout + row * V;
  uint16_t* dx = a.dx + row * V;
  const bool nan_row = (s.flags & kFlagNaN) != 0;
  const bool vec = V % 8 == 0 && (reinterpret_cast<uintptr_t>(a.gout) & 31) == 0 &&
                   (reinterpret_cast<uintptr_t>(a.dx) & 15) == 0;
  // the chunk's eight upstream gradients (0 past the row's end)
  auto grads = [&](int32_t base, float (&gv)[8]) {
    if (vec && base + 8 <= V) {
      const float4 g0 = *reinterpret_cast<const float4*>(g + base);
      const float4 g1 = *reinterpret_cast<const float4*>(g + base + 4);
      gv[0] = g0.x, gv[1] = g0.y, gv[2] = g0.z, gv[3] = g0.w;
      gv[4] = g1.x, gv[5] = g1.y, gv[6] = g1.z, gv[7] = g1.w;
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) gv[j] = base + j < V ? g[base + j] : 0.0f;
    }
  };
  float share = 0.0f;
  if ((s.flags & kFlagTemp) && !nan_row) {
    double sg = 0.0;
    r.chunks([&](int, int32_t base, const uint32_t (&w)[4]) {
      if (base >= V) return;
      float gv[8];
      grads(base, gv);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        sg += kept(sup, ord_of(bf16f(half_of(w, j)), cx), base + j) ? gv[j] : 0.0f;
      fence(sg);
    });
    share = static_cast<float>(block_sum(sg, red, ph) * static_cast<double>(s.rcp_t) / s.nmax);
  }
  r.chunks([&](int, int32_t base, const uint32_t (&w)[4]) {
    if (base >= V) return;
    float gv[8];
    grads(base, gv);
    uint32_t packed[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float d[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const float x = bf16f(half_of(w, 2 * k + h));
        float v = kept(sup, ord_of(x, cx), base + 2 * k + h) ? gv[2 * k + h] * s.rcp_t : 0.0f;
        v -= x == s.m ? share : 0.0f;
        d[h] = nan_row ? __builtin_nanf("") : v;
      }
      packed[k] = pack_bf16x2(d[0], d[1]);
    }
    if (vec && base + 8 <= V) {
      *reinterpret_cast<uint4*>(dx + base) = make_uint4(packed[0], packed[1], packed[2], packed[3]);
    } else {
      for (int j = 0; j < 8 && base + j < V; ++j) dx[base + j] = static_cast<uint16_t>(half_of(packed, j));
    }
    __builtin_amdgcn_sched_barrier(0);
  });
}

}  // namespace
}  // namespace aspec

using namespace aspec;

extern "C" int aspec_sampling_stats_floats(void) { return kSideWords; }

extern "C" int aspec_sampling_logits_fwd(const void* logits, int64_t rows, int64_t vocab,
                                         double temperature, double top_p, int64_t top_k, float* out,
                                         float* stats, void* stream) {
  int rc = check_rows(rows, vocab, logits);
  if (rc) return rc;
  if (!out || !stats) return set_error(ASPEC_ERR_INVALID, "sampling needs output and stats buffers");
  SampledArgs a = {};
  a.x = static_cast<const uint16_t*>(logits);
  a.rows = rows;
  a.V = vocab;
  a.out = out;
  a.stats = stats;
  if ((rc = side_params(temperature, top_p, top_k, vocab, &a.px))) return rc;
  const dim3 grid(static_cast<uint32_t>(rows)), block(kSampThreads);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  with_row(vocab, [&](auto type) {
    using Row = typename decltype(type)::Row;
    if (filters(a.px)) hipLaunchKernelGGL((sampling_fwd_kernel<Row, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((sampling_fwd_kernel<Row, false>), grid, block, 0, s, a);
  });
  return check_launch("sampling logits");
}

extern "C" int aspec_sampling_logits_bwd(const void* logits, const float* grad_out, const float* stats,
                                         int64_t rows, int64_t vocab, void* grad_logits, void* stream) {
  int rc = check_rows(rows, vocab, logits);
  if (rc) return rc;
  if (!grad_out || !stats || !grad_logits)
    return set_error(ASPEC_ERR_INVALID, "sampling backward needs gradient, stats and output buffers");
  SampledArgs a = {};
  a.x = static_cast<const uint16_t*>(logits);
  a.rows = rows;
  a.V = vocab;
  a.gout = grad_out;
  a.stats = const_cast<float*>(stats);
  a.dx = static_cast<uint16_t*>(grad_logits);
  with_row(vocab, [&](auto type) {
    using Row = typename decltype(type)::Row;
    hipLaunchKernelGGL(sampling_bwd_kernel<Row>, dim3(static_cast<uint32_t>(rows)), dim3(kSampThreads), 0,
                       static_cast<hipStream_t>(stream), a);
  });
  return check_launch("sampling logits backward");
}
