// attention_wide.hip — launcher of attention_wide.hpp's kernels.
#include "attention_wide.hpp"

namespace sf {

template <typename T, int DW, int MK>
static int launch_wide(const AttnWideParams& wp0, bool pre, int64_t wgs, int64_t split_items, hipStream_t st) {
  using C = AttnWideCfg<DW>;
  AttnWideParams wp = wp0;
  constexpr int64_t kChunk = int64_t(1) << 30;  // workgroups per launch (grid.x < 2^31)
  for (int64_t i0 = 0; i0 < wgs; i0 += kChunk) {
    const int64_t n = (wgs - i0) < kChunk ? (wgs - i0) : kChunk;
    wp.a.item0 = i0;
    if (pre)
      hipLaunchKernelGGL((attn_wide_kernel<T, DW, MK, true>), dim3((unsigned)n), dim3(256), 0, st, wp);
    else
      hipLaunchKernelGGL((attn_wide_kernel<T, DW, MK, false>), dim3((unsigned)n), dim3(256), 0, st, wp);
    const int rc = check_launch("attention (wide)");
    if (rc != SF_OK) return rc;
  }
  if (wp.a.parts == 0) return SF_OK;
  constexpr int64_t per = 4 * C::MB;
  for (int64_t i0 = 0; i0 < split_items; i0 += kChunk / per) {
    const int64_t n = (split_items - i0) < kChunk / per ? (split_items - i0) : kChunk / per;
    wp.a.item0 = i0;
    hipLaunchKernelGGL((attn_wide_combine_kernel<T, DW, MK>), dim3((unsigned)(per * n)), dim3(64), 0, st, wp);
    const int rc = check_launch("attention (wide combine)");
    if (rc != SF_OK) return rc;
  }
  return SF_OK;
}

template <typename T>
static int launch_wide_t(int dw, int mk, const AttnWideParams& wp, bool pre, int64_t wgs, int64_t split_items,
                         hipStream_t st) {
  switch (dw * 4 + mk) {
    case 64 * 4 + 0: return launch_wide<T, 64, 0>(wp, pre, wgs, split_items, st);
    case 64 * 4 + 1: return launch_wide<T, 64, 1>(wp, pre, wgs, split_items, st);
    case 64 * 4 + 2: return launch_wide<T, 64, 2>(wp, pre, wgs, split_items, st);
    case 96 * 4 + 0: return launch_wide<T, 96, 0>(wp, pre, wgs, split_items, st);
    case 96 * 4 + 1: return launch_wide<T, 96, 1>(wp, pre, wgs, split_items, st);
    case 96 * 4 + 2: return launch_wide<T, 96, 2>(wp, pre, wgs, split_items, st);
    case 128 * 4 + 0: return launch_wide<T, 128, 0>(wp, pre, wgs, split_items, st);
    case 128 * 4 + 1: return launch_wide<T, 128, 1>(wp, pre, wgs, split_items, st);
    case 128 * 4 + 2: return launch_wide<T, 128, 2>(wp, pre, wgs, split_items, st);
  }
  return fail(SF_ERR_INVALID_ARG, "wide attention: no kernel for tile width %d, mask kind %d", dw, mk);
}

static int wide_width(int64_t D) { return D <= 64 ? 64 : (D <= 96 ? 96 : 128); }

size_t attn_wide_part_bytes(int64_t D) {
  switch (wide_width(D)) {
    case 64: return AttnWideCfg<64>::PART * sizeof(float);
    case 96: return AttnWideCfg<96>::PART * sizeof(float);
  }
  return AttnWideCfg<128>::PART * sizeof(float);
}

AttnSplit attn_wide_split_plan(const AttnShape& a, int cus) {
  return attn_split_items(a.batch * a.heads * ((a.Sq + AttnWideCfg<64>::ROWS - 1) / AttnWideCfg<64>::ROWS), a.Sk,
                          attn_wide_part_bytes(a.D), cus);
}

int launch_attention_wide(const AttnShape& a, const AttnMask& m, float scale, sf_dtype dt, const AttnSplit& sp,
                          float* ws, hipStream_t st) {
  AttnWideParams wp;
  constexpr int rows = AttnWideCfg<64>::ROWS;
  attn_fill_params(a, scale, sp, ws, rows, wp.a);
  wp.mask = m.ptr;
  wp.mB = m.sB;
  wp.mH = m.sH;
  wp.mR = m.sR;
  const int64_t split_items = sp.items - sp.full;
  const int64_t wgs = sp.full + (sp.parts > 0 ? split_items * sp.parts : 0);
  // Q pre-scaled where that cannot overflow fp16, as in launch_attention.
  const bool pre = wp.a.scale_log2e <= 1.0f;
  const int mk = m.ptr == nullptr ? 0 : (m.dt == SF_F32 ? 1 : 2);
  const int dw = wide_width(a.D);
  return dt == SF_F16 ? launch_wide_t<F16>(dw, mk, wp, pre, wgs, split_items, st)
                      : launch_wide_t<BF16>(dw, mk, wp, pre, wgs, split_items, st);
}

}  // namespace sf
