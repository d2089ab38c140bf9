// Sampled L1: the DSpark L1 term between temperature / top-p / top-k filtered draft and teacher
// distributions, l1 = sum |p_draft - p_teacher| (aspec/models/ops/loss.py:57-89), and its gradient; the
// supports by sampling_support.h.
#include "sampling_support.h"

namespace aspec {
namespace {

template <typename Row, bool FILTER>
__global__ void __launch_bounds__(kSampThreads) __attribute__((amdgpu_waves_per_eu(Row::kWavesPerSimd)))
sampled_l1_fwd_kernel(SampledArgs a) {
  __shared__ Work work;
  int ph = 0;
  const int64_t row = blockIdx.x;
  int64_t yrow = row;
  if (a.yidx) {
    yrow = a.yidx[row];
    if (yrow < 0 || yrow >= a.trows) {  // the reference device-asserts; here a flag and a NaN row
      if (threadIdx.x == 0) {
        atomicOr(a.flags, 1);
        a.l1[row] = __builtin_nanf("");
        float* st = a.stats + row * kL1Words;
        for (int i = 0; i < kL1Words; ++i) st[i] = 0.0f;
        st[5] = __uint_as_float(kFlagNaN);
      }
      return;
    }
  }
  const int64_t V = a.V;
  const SideParams px = a.px, py = a.py;
  const uint16_t* xr = a.x + row * V;
  const uint16_t* yr = a.y + yrow * V;
  Row r;
  r.load(yr, V);
  const SideStats sy = compute_support<FILTER>(r, V, py, work, ph);
  r.load(xr, V);
  const SideStats sx = compute_support<FILTER>(r, V, px, work, ph);
  const bool nan_row = ((sx.flags | sy.flags) & kFlagNaN) != 0;
  double l1 = 0.0, pos = 0.0, neg = 0.0, zero = 0.0;
  if (!nan_row) {
    const RowCtx cx = ctx_of(sx), cy = ctx_of(sy);
    const Support kx = support_of(sx), ky = support_of(sy);
    r.chunks([&](int, int32_t base, const uint32_t (&wx)[4]) {
      const uint4 yc = row_chunk(yr, V, base);
      const uint32_t wy[4] = {yc.x, yc.y, yc.z, yc.w};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float p = prob(kx, cx, sx.zinv, half_of(wx, j), base + j);
        const float q = prob(ky, cy, sy.zinv, half_of(wy, j), base + j);
        l1 += fabsf(p - q);
        pos += p > q ? p : 0.0f;
        neg += p < q ? p : 0.0f;
        zero += p == q ? p : 0.0f;
      }
      fence(l1, pos, neg, zero);
    });
  }
  const double t_l1 = block_sum(l1, work.red, ph);
  const double t_pos = block_sum(pos, work.red, ph);
  const double t_neg = block_sum(neg, work.red, ph);
  const double t_zero = block_sum(zero, work.red, ph);
  if (threadIdx.x == 0) {
    float* st = a.stats + row * kL1Words;
    store_side(st, sx);
    store_side(st + kSideWords, sy);
    st[16] = static_cast<float>(t_pos);
    st[17] = static_cast<float>(t_neg);
    st[18] = static_cast<float>(t_zero);
    for (int i = 19; i < kL1Words; ++i) st[i] = 0.0f;
    a.l1[row] = nan_row ? __builtin_nanf("") : static_cast<float>(t_l1);
  }
}

// d logits = g / T_draft * p * (sign(p - q) - sum p sign(p - q)), written per case without
// cancellation: 2 neg + zero (p > q), -(2 pos + zero) (p < q), neg - pos (p == q), where pos, neg
// and zero are the draft mass on tokens with p > q, p < q and p == q. Each workgroup takes one
// 2048-token segment of a row per loop step, eight tokens per thread in 16-byte accesses.
__global__ void __launch_bounds__(256) sampled_l1_bwd_kernel(SampledArgs a) {
  const int64_t segs = (a.V + 2047) / 2048;
  for (int64_t unit = blockIdx.x; unit < a.rows * segs; unit += gridDim.x) {
    const int64_t row = unit / segs;
    const int32_t base = static_cast<int32_t>(unit - row * segs) * 2048 + static_cast<int32_t>(threadIdx.x) * 8;
    const float* st = a.stats + row * kL1Words;
    const SideStats sx = load_side(st);
    const SideStats sy = load_side(st + kSideWords);
    const RowCtx cx = ctx_of(sx), cy = ctx_of(sy);
    const Support kx = support_of(sx), ky = support_of(sy);
    const float pos = st[16], neg = st[17], zero = st[18];
    const float g = a.g_l1[row] * sx.rcp_t;
    const bool nan_row = ((sx.flags | sy.flags) & kFlagNaN) != 0;
    int64_t yrow = row;
    if (a.yidx) {
      yrow = a.yidx[row];
      if (yrow < 0 || yrow >= a.trows) yrow = 0;  // NaN row (flagged by the forward)
    }
    if (base >= a.V) continue;
    const uint4 xc = row_chunk(a.x + row * a.V, a.V, base);
    const uint4 yc = row_chunk(a.y + yrow * a.V, a.V, base);
    const uint32_t wx[4] = {xc.x, xc.y, xc.z, xc.w}, wy[4] = {yc.x, yc.y, yc.z, yc.w};
    const float w_gt = g * (2.0f * neg + zero), w_lt = -g * (2.0f * pos + zero), w_eq = g * (neg - pos);
    float d[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float p = prob(kx, cx, sx.zinv, half_of(wx, j), base + j);
      const float q = prob(ky, cy, sy.zinv, half_of(wy, j), base + j);
      d[j] = nan_row ? __builtin_nanf("") : p * (p > q ? w_gt : (p < q ? w_lt : w_eq));
    }
    const uint32_t out[4] = {pack_bf16x2(d[0], d[1]), pack_bf16x2(d[2], d[3]), pack_bf16x2(d[4], d[5]),
                             pack_bf16x2(d[6], d[7])};
    uint16_t* dr = a.dx + row * a.V + base;
    if (base + 8 <= a.V) {
      store_chunk(dr, make_uint4(out[0], out[1], out[2], out[3]));
    } else {
#pragma unroll
      for (int j = 0; j < 7; ++j)
        if (base + j < a.V) dr[j] = static_cast<uint16_t>(half_of(out, j));
    }
  }
}

}  // namespace
}  // namespace aspec

using namespace aspec;

extern "C" int aspec_sampled_l1_stats_floats(void) { return kL1Words; }

extern "C" int aspec_sampled_l1_fwd(const void* logits, const void* teacher, const int64_t* teacher_index,
                                    int64_t teacher_rows, int64_t rows, int64_t vocab,
                                    double draft_temperature, double draft_top_p, int64_t draft_top_k,
                                    double target_temperature, double target_top_p, int64_t target_top_k,
                                    float* l1_out, float* stats, int32_t* status_flags, void* stream) {
  int rc = check_rows(rows, vocab, logits);
  if (rc) return rc;
  if (!teacher || !l1_out || !stats || !status_flags)
    return set_error(ASPEC_ERR_INVALID, "sampled L1 needs teacher logits, output, stats and status buffers");
  if (teacher_index && teacher_rows <= 0) return set_error(ASPEC_ERR_INVALID, "indexed teacher table is empty");
  SampledArgs a = {};
  a.x = static_cast<const uint16_t*>(logits);
  a.y = static_cast<const uint16_t*>(teacher);
  a.yidx = teacher_index;
  a.trows = teacher_index ? teacher_rows : rows;
  a.rows = rows;
  a.V = vocab;
  a.l1 = l1_out;
  a.stats = stats;
  a.flags = status_flags;
  if ((rc = side_params(draft_temperature, draft_top_p, draft_top_k, vocab, &a.px))) return rc;
  if ((rc = side_params(target_temperature, target_top_p, target_top_k, vocab, &a.py))) return rc;
  const dim3 grid(static_cast<uint32_t>(rows)), block(kSampThreads);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  with_row(vocab, [&](auto type) {
    using Row = typename decltype(type)::Row;
    if (filters(a.px) || filters(a.py)) hipLaunchKernelGGL((sampled_l1_fwd_kernel<Row, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((sampled_l1_fwd_kernel<Row, false>), grid, block, 0, s, a);
  });
  return check_launch("sampled L1 forward");
}

extern "C" int aspec_sampled_l1_bwd(const void* logits, const void* teacher, const int64_t* teacher_index,
                                    int64_t teacher_rows, int64_t rows, int64_t vocab, const float* stats,
                                    const float* grad_l1, void* grad_logits, void* stream) {
  int rc = check_rows(rows, vocab, logits);
  if (rc) return rc;
  if (!teacher || !stats || !grad_l1 || !grad_logits)
    return set_error(ASPEC_ERR_INVALID, "sampled L1 backward needs teacher logits, stats, gradients and output");
  SampledArgs a = {};
  a.x = static_cast<const uint16_t*>(logits);
  a.y = static_cast<const uint16_t*>(teacher);
  a.yidx = teacher_index;
  a.trows = teacher_index ? teacher_rows : rows;
  a.rows = rows;
  a.V = vocab;
  a.stats = const_cast<float*>(stats);
  a.g_l1 = grad_l1;
  a.dx = static_cast<uint16_t*>(grad_logits);
  const int64_t units = rows * ((vocab + 2047) / 2048);
  const int64_t grid = units < 256 * 64 ? units : 256 * 64;
  hipLaunchKernelGGL(sampled_l1_bwd_kernel, dim3(static_cast<uint32_t>(grid)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), a);
  return check_launch("sampled L1 backward");
}
