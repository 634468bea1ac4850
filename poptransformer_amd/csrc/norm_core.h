// One row of the decode step's normalisations by a workgroup: RMSNorm and the NormCE LayerNorm, of rows that lie in memory or of those that a
// launch makes itself (the end of a product whose K was split).  The numerics are told in norm.hip.
#pragma once
#include "common.h"
#include "f8codec.h"

constexpr int NORM_THREADS = 256;
constexpr int NORM_MAX_VEC = 4;  // 8-element vectors per thread: rows up to 8192 columns

// N sums over the workgroup, called once by all of its threads
template <int N>
__device__ __forceinline__ void block_sums(float (&v)[N]) {
  constexpr int WAVES = NORM_THREADS / 64;
  __shared__ float sh[N][WAVES];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    v[n] = wave_total_dpp(v[n]);
    if ((threadIdx.x & 63) == 0) sh[n][threadIdx.x >> 6] = v[n];
  }
  __syncthreads();
#pragma unroll
  for (int n = 0; n < N; ++n) {
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) t += sh[n][w];
    v[n] = t;
  }
}

// The RWKV token shift behind a LayerNorm (models/rwkv/attention.py:59-72, models/rwkv/ffn.py:44-51): the
// normalised row h feeds out[i] = h * w[i] + (1 - w[i]) * prev for up to three mixing vectors, then prev <- h.
struct NormMix {
  f16* prev;          // [rows, cols], or null: no shift
  const f16* w[3];    // [cols] each; null entries are skipped
  f16* out[3];
};

// What is done with the rows: mode 0: RMSNorm.  mode 1: NormCE with one row.  mode 2: NormCE with several rows.
struct NormArgs {
  const f16* gamma;
  const f16* beta;
  f16* y;                       // [rows, cols], or null (with a mix)
  int cols;
  float eps;
  const int32_t* grid_scale;    // or null: no cast
  int grid_format;
};

// row.request(i, c), row.value(i), row.keep(c, value): a thread's i-th piece, columns 8 c to 8 c + 7 of the workgroup's row.  VECS: pieces of a thread, as few as the row
// needs.  All requests, the weights' and the cast's exponent's go before the first value is used, and without a branch round them (where paths meet
// the compiler waits for what is in flight; a thread without a piece reads the row's last one): one round trip to memory before the sums.
// Few rows are bounded by this chain: 32 rows of 4096 behind a split product 6.1 -> 5.7 us with the branches gone; a token of 32 layers of 32 rows with the
// shift 1.4 % less, of 28 layers of eight rows with the cast to the FP8 grid nothing that runs on several machines show (0 to 0.7 %, they differ by up to 2).
template <int MODE, bool MIX, int VECS, class Row>
__device__ __forceinline__ void norm_row(const NormArgs& a, const NormMix& mix, size_t r, Row& row) {
  const size_t base = r * a.cols;
  const int nvec = a.cols >> 3;
  f16x8 v[VECS], gv[VECS], bv[VECS], pv[MIX ? VECS : 1], wv[MIX ? VECS : 1][3];
  float s = 0.f, sq = 0.f;
  const int gs = *(a.grid_scale ? a.grid_scale : reinterpret_cast<const int32_t*>(a.gamma));
#pragma unroll
  for (int i = 0; i < VECS; ++i) {
    const int at = threadIdx.x + i * NORM_THREADS, c = at < nvec ? at : nvec - 1;
    row.request(i, c);
    gv[i] = *reinterpret_cast<const f16x8*>(a.gamma + (size_t)c * 8);
    if (MODE != 0) bv[i] = *reinterpret_cast<const f16x8*>(a.beta + (size_t)c * 8);
    if (MIX) {
      pv[i] = *reinterpret_cast<const f16x8*>(mix.prev + base + (size_t)c * 8);
#pragma unroll
      for (int j = 0; j < 3; ++j) wv[i][j] = *reinterpret_cast<const f16x8*>((mix.w[j] ? mix.w[j] : mix.w[0]) + (size_t)c * 8);
    }
  }
#pragma unroll
  for (int i = 0; i < VECS; ++i) {
    const int c = threadIdx.x + i * NORM_THREADS;
    v[i] = row.value(i);
    if (c < nvec) row.keep(c, v[i]);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float f = c < nvec ? (float)v[i][e] : 0.0f;      // (a branch here would draw the requests behind it)
      s += f;
      sq = __builtin_fmaf(f, f, sq);
    }
  }
  const float inv_n = 1.0f / (float)a.cols;
  f16 mean16 = (f16)0.0f, r16;
  if (MODE == 0) {
    float sums[1] = {sq};
    block_sums(sums);
    const float ms = sums[0] * inv_n;
    r16 = (f16)(1.0f / sqrtf(ms + a.eps));
  } else {
    float sums[2] = {s, sq};
    block_sums(sums);
    const float sqs = sums[1], mean = sums[0] * inv_n;
    mean16 = (f16)mean;
    float var;
    if (MODE == 1) {
      var = sqs * inv_n - mean * mean + a.eps;  // fp32 mean, no clamp
    } else {
      const float m = (float)mean16;          // the rounded mean is what gets squared
      var = fmaxf(sqs * inv_n - m * m, 0.0f) + a.eps;
    }
    r16 = (f16)(1.0f / sqrtf(var));
  }
#pragma unroll
  for (int i = 0; i < VECS; ++i) {
    const int c = threadIdx.x + i * NORM_THREADS;
    if (c < nvec) {
      const f16x8 g = gv[i];
      f16x8 o;
      if (MODE == 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (v[i][e] * r16) * g[e];
      } else {
        const f16x8 b = bv[i];
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = ((v[i][e] - mean16) * r16) * g[e] + b[e];
      }
      if (a.grid_scale) {           // the cast of the FP8 Linear that consumes these rows
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = f8_grid_value(o[e], gs, a.grid_format);
      }
      if (!MIX || a.y) *reinterpret_cast<f16x8*>(a.y + base + (size_t)c * 8) = o;
      if (MIX) {
        // each step an fp16 operation, in the order of the separate kernel: h * w + (1 - w) * prev
        const f16 one = (f16)1.0f;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          if (!mix.w[j]) continue;
          f16x8 m;
#pragma unroll
          for (int e = 0; e < 8; ++e) m[e] = o[e] * wv[i][j][e] + (one - wv[i][j][e]) * pv[i][e];
          *reinterpret_cast<f16x8*>(mix.out[j] + base + (size_t)c * 8) = m;
        }
        *reinterpret_cast<f16x8*>(mix.prev + base + (size_t)c * 8) = o;
      }
    }
  }
}

// norm.hip: the launch over rows in memory (mode: of norm_row; mix: null without a shift) and the checks of what it takes
void launch_norm(const f16* x, int rows, int mode, const NormArgs& a, const NormMix* mix, hipStream_t s);
int check_norm(const char* name, const void* x, const void* g, const void* y, int rows, int cols);
int check_layer_norm(const char* name, const void* beta, int cols);
int check_grid(const char* name, const int32_t* scale, int format);
int check_norm_mix(const char* name, const void* y, const pta_half* const* w, pta_half* const* o);
