// Row normalisations of the decode step: RMSNorm and the NormCE LayerNorm.
//
// RMSNorm follows poptransformer/layers/rms_layer_norm.py:26-36 (fp32 statistics, the inverse
// RMS rounded to fp16, then two fp16 multiplies).  LayerNorm follows the NormCE custom op:
// custom_ops/NormCE.cpp:122-200 + NormCECodelets.cpp:65-112 when there is a single row, and
// the assembly kernel custom_ops/NormCE.S:243-423 (C form NormCECodelets.cpp:181-211) when
// there are several.  One workgroup normalises one row in a single pass over registers.
#include "norm_core.h"

template <int VECS>
struct RowInMemory {
  const f16* from;
  f16x8 v[VECS];
  __device__ __forceinline__ void request(int i, int c) { v[i] = *reinterpret_cast<const f16x8*>(from + (size_t)c * 8); }
  __device__ __forceinline__ f16x8 value(int i) const { return v[i]; }
  __device__ __forceinline__ void keep(int, f16x8) const {}
};

template <int MODE, bool MIX, int VECS>
__global__ __launch_bounds__(NORM_THREADS) void norm_kernel(const f16* __restrict__ x, NormArgs a, NormMix mix) {
  RowInMemory<VECS> row{x + (size_t)blockIdx.x * a.cols};
  norm_row<MODE, MIX, VECS>(a, mix, blockIdx.x, row);
}

void launch_norm(const f16* x, int rows, int mode, const NormArgs& a, const NormMix* mix, hipStream_t s) {
  const NormMix m = mix ? *mix : NormMix{};
  auto launch = [&](auto vecs) {
    constexpr int V = decltype(vecs)::value;
    if (mode == 0) hipLaunchKernelGGL((norm_kernel<0, false, V>), dim3(rows), dim3(NORM_THREADS), 0, s, x, a, m);
    else if (mode == 1 && mix) hipLaunchKernelGGL((norm_kernel<1, true, V>), dim3(rows), dim3(NORM_THREADS), 0, s, x, a, m);
    else if (mode == 1) hipLaunchKernelGGL((norm_kernel<1, false, V>), dim3(rows), dim3(NORM_THREADS), 0, s, x, a, m);
    else if (mix) hipLaunchKernelGGL((norm_kernel<2, true, V>), dim3(rows), dim3(NORM_THREADS), 0, s, x, a, m);
    else hipLaunchKernelGGL((norm_kernel<2, false, V>), dim3(rows), dim3(NORM_THREADS), 0, s, x, a, m);
  };
  // (as few pieces of a thread as the row needs)
  switch ((a.cols + 8 * NORM_THREADS - 1) / (8 * NORM_THREADS)) {
    case 1: launch(std::integral_constant<int, 1>{}); break;
    case 2: launch(std::integral_constant<int, 2>{}); break;
    case 3: launch(std::integral_constant<int, 3>{}); break;
    default: launch(std::integral_constant<int, NORM_MAX_VEC>{});
  }
}

int check_norm(const char* name, const void* x, const void* g, const void* y, int rows, int cols) {
  PTA_REQUIRE(x && g && y, "%s: null pointer", name);
  PTA_REQUIRE(rows > 0, "%s: rows = %d", name, rows);
  PTA_REQUIRE(cols > 0 && (cols % 8) == 0 && cols <= 8 * NORM_THREADS * NORM_MAX_VEC,
              "%s: the normalised size must be a multiple of 8 and at most %d, got %d", name,
              8 * NORM_THREADS * NORM_MAX_VEC, cols);
  PTA_REQUIRE(pta_aligned(x, 16) && pta_aligned(g, 16) && pta_aligned(y, 16), "%s: pointers must be 16-byte aligned", name);
  return PTA_OK;
}

// Guards of NormCEOutplaceOpx::grow (custom_ops/NormCE.cpp:541-577) and of the Python wrapper (poptransformer/ops/customized.py:81-82): fp16
// only, size < 8192.
int check_layer_norm(const char* name, const void* beta, int cols) {
  PTA_REQUIRE(beta && pta_aligned(beta, 16), "%s: beta must be a 16-byte aligned pointer", name);
  PTA_REQUIRE(cols < 8192, "%s: the normalised size must be below 8192, got %d", name, cols);
  return PTA_OK;
}

int check_grid(const char* name, const int32_t* scale, int format) {
  PTA_REQUIRE(scale, "%s: null scale", name);
  PTA_REQUIRE(format == PTA_F143 || format == PTA_F152, "%s: unsupported fp8 format %d, it must be F143 or F152", name, format);
  return PTA_OK;
}

int check_norm_mix(const char* name, const void* y, const pta_half* const* w, pta_half* const* o) {
  PTA_REQUIRE(w[0] && o[0], "%s: null pointer", name);
  PTA_REQUIRE((!w[1] || o[1]) && (!w[2] || o[2]), "%s: a mixing vector needs its output", name);
  const void* ptrs[7] = {y, w[0], w[1], w[2], o[0], o[1], o[2]};
  for (const void* q : ptrs) PTA_REQUIRE(!q || pta_aligned(q, 16), "%s: pointers must be 16-byte aligned", name);
  return PTA_OK;
}

extern "C" int pta_rmsnorm(const pta_half* x, const pta_half* weight, pta_half* y, int rows, int cols,
                           float eps, pta_stream_t stream) {
  int rc = check_norm("pta_rmsnorm", x, weight, y, rows, cols);
  if (rc) return rc;
  launch_norm((const f16*)x, rows, 0, NormArgs{(const f16*)weight, nullptr, (f16*)y, cols, eps, nullptr, 0}, nullptr, (hipStream_t)stream);
  PTA_CHECK_LAUNCH("pta_rmsnorm");
  return PTA_OK;
}

extern "C" int pta_rmsnorm_fp8_grid(const pta_half* x, const pta_half* weight, pta_half* y, const int32_t* scale,
                                    int format, int rows, int cols, float eps, pta_stream_t stream) {
  int rc = check_norm("pta_rmsnorm_fp8_grid", x, weight, y, rows, cols);
  if (!rc) rc = check_grid("pta_rmsnorm_fp8_grid", scale, format);
  if (rc) return rc;
  launch_norm((const f16*)x, rows, 0, NormArgs{(const f16*)weight, nullptr, (f16*)y, cols, eps, scale, format}, nullptr, (hipStream_t)stream);
  PTA_CHECK_LAUNCH("pta_rmsnorm_fp8_grid");
  return PTA_OK;
}

extern "C" int pta_layer_norm_ce(const pta_half* x, const pta_half* gamma, const pta_half* beta, pta_half* y,
                                 int rows, int cols, float eps, pta_stream_t stream) {
  int rc = check_norm("pta_layer_norm_ce", x, gamma, y, rows, cols);
  if (!rc) rc = check_layer_norm("pta_layer_norm_ce", beta, cols);
  if (rc) return rc;
  launch_norm((const f16*)x, rows, rows == 1 ? 1 : 2, NormArgs{(const f16*)gamma, (const f16*)beta, (f16*)y, cols, eps, nullptr, 0}, nullptr, (hipStream_t)stream);
  PTA_CHECK_LAUNCH("pta_layer_norm_ce");
  return PTA_OK;
}

extern "C" int pta_layer_norm_ce_mix(const pta_half* x, const pta_half* gamma, const pta_half* beta, pta_half* y,
                                     pta_half* prev, const pta_half* w0, const pta_half* w1, const pta_half* w2,
                                     pta_half* o0, pta_half* o1, pta_half* o2, int rows, int cols, float eps,
                                     pta_stream_t stream) {
  const char* name = "pta_layer_norm_ce_mix";
  const pta_half* w[3] = {w0, w1, w2};
  pta_half* o[3] = {o0, o1, o2};
  int rc = check_norm(name, x, gamma, prev, rows, cols);
  if (!rc) rc = check_layer_norm(name, beta, cols);
  if (!rc) rc = check_norm_mix(name, y, w, o);
  if (rc) return rc;
  const NormMix mix{(f16*)prev, {(const f16*)w0, (const f16*)w1, (const f16*)w2}, {(f16*)o0, (f16*)o1, (f16*)o2}};
  launch_norm((const f16*)x, rows, rows == 1 ? 1 : 2, NormArgs{(const f16*)gamma, (const f16*)beta, (f16*)y, cols, eps, nullptr, 0}, &mix, (hipStream_t)stream);
  PTA_CHECK_LAUNCH(name);
  return PTA_OK;
}
