// Epilogue shared by the fused GEMV/GEMM kernels (INT4, FP16 and FP8 weights).
//
// The reference builds these as separate fp16 graph ops after the MatMul: the bias `ops.add`
// of poptransformer/layers/linear.py:42-46, the activation of layers/mlp.py:34-41 /
// models/rwkv/ffn.py:47-59, and the residual `ops.add` of the transformer blocks
// (e.g. models/llama2/model.py:38-46).  Each step therefore rounds to fp16.
#pragma once
#include "common.h"
#include "f8codec.h"
#include "norm_core.h"

// Where and how a product of a "wide" format goes: one fp32 value per output, rounded once where it is stored.
struct WideOut {
  int ld;                   // elements between rows of Y
  int n_main;               // channels [0, n_main) go to Y; channels past n_main + tail_count are padding of the weight
  int out_f32;              // Y holds fp32 (else the format's own type)
  float* tail;              // channels [n_main, n_main + tail_count) go here, fp32 [M, tail_count], plus tail_bias
  int tail_count;
  const float* tail_bias;
  float cap;                // > 0: y = cap * tanh(y / cap)
  int clamped;              // pairs: 0 = SwiGLU, 1 = min(g, limit) sigmoid(slope g) (clamp(u, -limit, limit) + 1)
  float limit, slope;
  const float* bias;        // [n_main] or null, added to the sum (of a pair: to the gate's)
  const float* bias2;       // [n_main] or null, added to the sum of a pair's second weight
  int act;                  // PTA_ACT_*
  const void* mul;          // [M, ld] or null, fp32 (mul_f32) or bf16: y = y * mul
  int mul_f32;
  int accumulate;           // Y (fp32) += y
};

struct GemmEpilogue {
  const f16* bias;
  const f16* residual;
  int act;
  const f16* mul;
  float post_scale;
  int norm;                 // PTA_NORM_*, applied to the rows of X before the product
  const f16* norm_weight;
  const f16* norm_bias;
  float norm_eps;
  const int32_t* out_fp8_scale;   // when set: the result is left on the FP8 grid of this exponent (unscaled)
  int out_fp8_format;
  f16* mix_state;                 // [2][M, K] or null: the previous token's rows for the token-shift mixes (gemv_lds_kernel)
  const int32_t* mix_step;
};

__device__ __forceinline__ f16 sigmoid_f16(f16 x) {
  return (f16)(1.0f / (1.0f + __expf(-(float)x)));
}

// x * sigmoid(x), evaluated in fp32 from the fp16 input and rounded once.
__device__ __forceinline__ f16 swish_f16(f16 x) {
  const float v = (float)x;
  return (f16)(v / (1.0f + __expf(-v)));
}

// tanh-form GELU, evaluated in fp32 from the fp16 input and rounded once.
__device__ __forceinline__ f16 gelu_tanh_f16(f16 x) {
  const float v = (float)x;
  const float u = 0.7978845608028654f * (v + 0.044715f * v * v * v);
  return (f16)(0.5f * v * (1.0f + tanhf(u)));
}

__device__ __forceinline__ f16 apply_act(int act, f16 y) {
  switch (act) {
    case PTA_ACT_GELU_TANH: return gelu_tanh_f16(y);
    case PTA_ACT_RELU_SQUARE: { f16 r = y > (f16)0.0f ? y : (f16)0.0f; return r * r; }
    case PTA_ACT_SIGMOID: return sigmoid_f16(y);
    default: return y;
  }
}

__device__ __forceinline__ f16 apply_epilogue(const GemmEpilogue& e, f16 y, int m, int n, int N) {
  if (e.bias) y = y + e.bias[n];
  y = apply_act(e.act, y);
  if (e.mul) y = y * e.mul[(size_t)m * N + n];
  if (e.residual) y = y + e.residual[(size_t)m * N + n];
  if (e.post_scale != 0.0f) y = y * (f16)e.post_scale;
  if (e.out_fp8_scale) y = f8_grid_value(y, e.out_fp8_scale[0], e.out_fp8_format);
  return y;
}

// the SwiGLU pair's result: up * swish(gate), then the optional cast of the epilogue
__device__ __forceinline__ f16 swiglu_out(const GemmEpilogue& e, f16 gate, f16 up) {
  f16 y = up * swish_f16(gate);
  if (e.out_fp8_scale) y = f8_grid_value(y, e.out_fp8_scale[0], e.out_fp8_format);
  return y;
}

static inline int make_epilogue(const pta_fusion* in, GemmEpilogue* out, const char* name) {
  *out = GemmEpilogue{nullptr, nullptr, PTA_ACT_NONE, nullptr, 0.f, PTA_NORM_NONE, nullptr, nullptr, 0.f, nullptr, PTA_F143, nullptr, nullptr};
  if (!in) return PTA_OK;
  PTA_REQUIRE(in->act >= PTA_ACT_NONE && in->act <= PTA_ACT_SIGMOID, "%s: unknown activation %d", name, in->act);
  PTA_REQUIRE(in->norm >= PTA_NORM_NONE && in->norm <= PTA_NORM_LAYER, "%s: unknown norm %d", name, in->norm);
  PTA_REQUIRE(in->norm == PTA_NORM_NONE || in->norm_weight, "%s: fused norm needs norm_weight", name);
  PTA_REQUIRE(in->norm != PTA_NORM_LAYER || in->norm_bias, "%s: fused LayerNorm needs norm_bias", name);
  out->bias = (const f16*)in->bias; out->residual = (const f16*)in->residual; out->act = in->act;
  out->mul = (const f16*)in->mul; out->post_scale = in->post_scale;
  out->norm = in->norm; out->norm_weight = (const f16*)in->norm_weight; out->norm_bias = (const f16*)in->norm_bias;
  out->norm_eps = in->norm_eps;
  PTA_REQUIRE(!in->out_fp8_scale || in->out_fp8_format == PTA_F143 || in->out_fp8_format == PTA_F152,
              "%s: unsupported fp8 format %d, it must be F143 or F152", name, in->out_fp8_format);
  out->out_fp8_scale = in->out_fp8_scale; out->out_fp8_format = in->out_fp8_format;
  PTA_REQUIRE(!in->mix_state == !in->mix_step, "%s: mix_state and mix_step come together", name);
  out->mix_state = (f16*)in->mix_state; out->mix_step = in->mix_step;
  return PTA_OK;
}

// ------------------------------------------------------------------------------------------
// Small-M GEMM core: Y[M,N] = fp16(X[M,K] @ W^T) for M <= 64, weights streamed once.
//
// Weights are stored tiled (see the *_tile entry points): a tile is 16 output channels x 128
// input features, made of Fmt::kVec vectors of 1 KiB; in each vector lane l owns the 16 bytes
// at offset 16*l.  The tiles of one 16-channel block are contiguous over the feature axis.
// One workgroup owns one 16-channel block; its NW waves take feature tiles round-robin, each
// wave feeding the 16x16x32 fp16 MFMA with A = 16 channels x 32 features of weights (decoded
// in registers) and B = 32 features x 16 activation rows read straight from X, and the
// partial sums meet in LDS.  HBM traffic is the weight bytes, once; X comes from L2.
// ------------------------------------------------------------------------------------------
struct GemmMat {
  const void* tiled;
  const void* scale;   // fp16 [N] (INT4), device int32 exponent (FP8), unused (FP16)
  const f16* bias;     // [N] or null; used when the launch holds several matrices
  const f16* X;        // this matrix's own input, or null for the shared one
  const f16* mix;      // this matrix's token-shift mixing vector [K], or null (with GemmEpilogue::mix_state)
  int act;             // activation of this matrix's output when the launch holds several
  f16* Y;
  int N;
  int nb_begin;        // first 16-channel block of this matrix in the launch grid
  WideOut wide;        // of the formats whose epilogue works in fp32 (Fmt::kWide)
};

// The fp32 activations of the wide formats, of every kernel the same.
__device__ __forceinline__ float sigmoid_wide(float v) { return 1.0f / (1.0f + expf(-v)); }
__device__ __forceinline__ float swiglu_f32(float g, float u) { return u * g / (1.0f + expf(-g)); }
__device__ __forceinline__ float clamped_glu_f32(float g, float u, float limit, float slope) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g / (1.0f + expf(-slope * g)) * (u + 1.0f);
}

// The fp32 epilogue of the wide formats (Y is a bf16 or fp32 buffer behind the f16* of GemmMat).
__device__ __forceinline__ float wide_value(const WideOut& w, int n, float v) {
  if (w.bias) v += w.bias[n];
  if (w.cap > 0.f) v = w.cap * tanhf(v / w.cap);
  switch (w.act) {
    case PTA_ACT_GELU_TANH: return 0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
    case PTA_ACT_RELU_SQUARE: return v > 0.f ? v * v : 0.f;
    case PTA_ACT_SIGMOID: return sigmoid_wide(v);
    default: return v;
  }
}

__device__ __forceinline__ float wide_pair_value(const WideOut& w, int n, float g, float u) {
  if (w.bias) g += w.bias[n];
  if (w.bias2) u += w.bias2[n];
  return w.clamped ? clamped_glu_f32(g, u, w.limit, w.slope) : swiglu_f32(g, u);
}

__device__ __forceinline__ void wide_store(const WideOut& w, const GemmMat& mat, int m, int n, float v) {
  const size_t at = (size_t)m * w.ld + n;
  if (w.mul) v *= w.mul_f32 ? reinterpret_cast<const float*>(w.mul)[at] : (float)reinterpret_cast<const bf16*>(w.mul)[at];
  if (w.accumulate) v += reinterpret_cast<const float*>(mat.Y)[at];
  if (w.out_f32) reinterpret_cast<float*>(mat.Y)[at] = v;
  else reinterpret_cast<bf16*>(mat.Y)[at] = (bf16)v;
}

__device__ __forceinline__ void wide_put(const GemmMat& mat, int m, int n, float v) {
  const WideOut& w = mat.wide;
  if (n < w.n_main) {
    wide_store(w, mat, m, n, wide_value(w, n, v));
  } else if (n - w.n_main < w.tail_count) {
    const int c = n - w.n_main;
    w.tail[(size_t)m * w.tail_count + c] = w.tail_bias ? v + w.tail_bias[c] : v;
  }
}

__device__ __forceinline__ void wide_put_pair(const GemmMat& mat, int m, int n, float gate, float up) {
  const WideOut& w = mat.wide;
  if (n < w.n_main) wide_store(w, mat, m, n, wide_pair_value(w, n, gate, up));
}

// four consecutive channels of a row, n a multiple of four
__device__ __forceinline__ void wide_store4(const WideOut& w, const GemmMat& mat, int m, int n, f32x4 v) {
  const size_t at = (size_t)m * w.ld + n;
  if (w.mul) {
    f32x4 g;
    if (w.mul_f32) {
      g = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(w.mul) + at);
    } else {
      const bf16x4 b = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const bf16*>(w.mul) + at);
#pragma unroll
      for (int r = 0; r < 4; ++r) g[r] = (float)b[r];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] *= g[r];
  }
  if (w.accumulate) {
    const f32x4 y = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(mat.Y) + at);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] += y[r];
  }
  if (w.out_f32) {
    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(mat.Y) + at) = v;
  } else {
    bf16x4 b;
#pragma unroll
    for (int r = 0; r < 4; ++r) b[r] = (bf16)v[r];
    *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16*>(mat.Y) + at) = b;
  }
}

__device__ __forceinline__ void wide_put4(const GemmMat& mat, int m, int n, f32x4 v) {
  const WideOut& w = mat.wide;
  if (n + 4 <= w.n_main && (w.ld & 3) == 0) {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = wide_value(w, n + r, v[r]);
    wide_store4(w, mat, m, n, v);
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) wide_put(mat, m, n + r, v[r]);
  }
}

__device__ __forceinline__ void wide_put_pair4(const GemmMat& mat, int m, int n, f32x4 gate, f32x4 up) {
  const WideOut& w = mat.wide;
  if (n + 4 <= w.n_main && (w.ld & 3) == 0) {
#pragma unroll
    for (int r = 0; r < 4; ++r) gate[r] = wide_pair_value(w, n + r, gate[r], up[r]);
    wide_store4(w, mat, m, n, gate);
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) wide_put_pair(mat, m, n + r, gate[r], up[r]);
  }
}

// eight of them, n a multiple of eight
__device__ __forceinline__ void wide_put8(const GemmMat& mat, int m, int n, f32x4 v0, f32x4 v1) {
  const WideOut& w = mat.wide;
  if (n + 8 <= w.n_main && (w.ld & 7) == 0 && !w.out_f32 && !w.mul) {
    bf16x8 b;
#pragma unroll
    for (int r = 0; r < 8; ++r) b[r] = (bf16)wide_value(w, n + r, r < 4 ? v0[r & 3] : v1[r & 3]);
    *reinterpret_cast<bf16x8*>(reinterpret_cast<bf16*>(mat.Y) + (size_t)m * w.ld + n) = b;
    return;
  }
  wide_put4(mat, m, n, v0);
  wide_put4(mat, m, n + 4, v1);
}

__device__ __forceinline__ void wide_put_pair8(const GemmMat& mat, int m, int n, f32x4 g0, f32x4 g1, f32x4 u0, f32x4 u1) {
  const WideOut& w = mat.wide;
  if (n + 8 <= w.n_main && (w.ld & 7) == 0 && !w.out_f32 && !w.mul) {
    bf16x8 b;
#pragma unroll
    for (int r = 0; r < 8; ++r) b[r] = (bf16)wide_pair_value(w, n + r, r < 4 ? g0[r & 3] : g1[r & 3], r < 4 ? u0[r & 3] : u1[r & 3]);
    *reinterpret_cast<bf16x8*>(reinterpret_cast<bf16*>(mat.Y) + (size_t)m * w.ld + n) = b;
    return;
  }
  wide_put_pair4(mat, m, n, g0, u0);
  wide_put_pair4(mat, m, n + 4, g1, u1);
}

// the rows from m0 on
static inline void wide_skip_rows(GemmMat& mat, int m0) {
  WideOut& w = mat.wide;
  mat.Y = reinterpret_cast<f16*>(reinterpret_cast<unsigned char*>(mat.Y) + (size_t)m0 * w.ld * (w.out_f32 ? 4 : 2));
  if (w.tail) w.tail += (size_t)m0 * w.tail_count;
  if (w.mul) w.mul = reinterpret_cast<const unsigned char*>(w.mul) + (size_t)m0 * w.ld * (w.mul_f32 ? 4 : 2);
}

// A norm of the result's rows behind the product: where K was split the launch that adds the slices does it (done), else whoever asked for it.
struct FinishNorm {
  NormArgs norm;
  NormMix mix;
  int mode;            // of norm_row
  bool shifted;        // with the mix
  bool any_order;      // the product's sums may be taken in another order than without a norm
  bool done;
};

struct GemmArgs {
  GemmMat mat[4];
  int count;
  const f16* X;
  const int32_t* x_scale;  // device exponent of X when X holds unscaled FP8 grid values, else null
  int M, K, KT;
  GemmEpilogue epi;
  // PAIR mode (SwiGLU): mat[0] is the gate weight, mat[1] the up weight, output in mat[0].Y.
  // K split across workgroups (gemm_own_kernel and the kernels for more rows, one matrix): one of `ksplit` slices (blockIdx.y; gemm_own_kernel: part of blockIdx.z) writes its fp32
  // sums to part[slice][M][N]; splitk_finish_kernel adds the slices and applies the epilogue.
  float* part;
  size_t part_bytes;
  int ksplit;          // 0 or 1: no split
  int prefer_stream;   // host side: up to 16 rows go to gemv_stream_kernel wherever it fits
  FinishNorm* then;    // host side: see there, or null
};
// v, read from memory at this point and kept in scalar registers
template <class T>
__device__ __forceinline__ void in_register(T& v) { asm volatile("" : "+s"(v)); }

// What the end of a kernel needs of its arguments, read at this point: while the first loads are on their way, that is.  Read where it
// is used, each line of the arguments is a round trip to memory of its own, one after another behind the products.
template <class Fmt, bool PAIR>
__device__ __forceinline__ void read_end(GemmMat& mat, GemmEpilogue& epi) {
  in_register(mat.Y);
  if constexpr (Fmt::kWide) {
    WideOut& o = mat.wide;
    in_register(o.ld); in_register(o.n_main); in_register(o.out_f32);
    in_register(o.bias); in_register(o.mul); in_register(o.mul_f32); in_register(o.accumulate);
    if constexpr (PAIR) {
      in_register(o.clamped); in_register(o.limit); in_register(o.slope); in_register(o.bias2);
    } else {
      in_register(o.tail); in_register(o.tail_count); in_register(o.tail_bias); in_register(o.cap); in_register(o.act);
    }
  } else {
    if constexpr (!PAIR) {
      in_register(mat.bias); in_register(mat.act); in_register(epi.bias); in_register(epi.residual); in_register(epi.act);
      in_register(epi.mul); in_register(epi.post_scale);
    }
    in_register(epi.out_fp8_scale); in_register(epi.out_fp8_format);
  }
}

// One finished fp32 sum of a matrix, or of a gate / up pair, on its way out.
template <class Fmt>
__device__ __forceinline__ void gemm_put(const GemmEpilogue& epi, const GemmMat& mat, int m, int n, int N, float sum) {
  if constexpr (Fmt::kWide) {
    wide_put(mat, m, n, sum);
  } else {
    f16 y0 = (f16)sum;
    if (mat.bias) y0 = y0 + mat.bias[n];
    y0 = apply_act(mat.act, y0);
    mat.Y[(size_t)m * N + n] = apply_epilogue(epi, y0, m, n, N);
  }
}

template <class Fmt>
__device__ __forceinline__ void gemm_put_pair(const GemmEpilogue& epi, const GemmMat& mat, int m, int n, int N, float gate, float up) {
  if constexpr (Fmt::kWide) wide_put_pair(mat, m, n, gate, up);
  else mat.Y[(size_t)m * N + n] = swiglu_out(epi, (f16)gate, (f16)up);
}

static inline int device_compute_units();
// The kernel that the calling thread's last product took (its last launch's, where it was several; without the finish of a K split): for
// tests that are meant for one of them.
inline thread_local const char* gemm_kernel_taken = "";
// Its tiles, of gemm_block_kernel and gemm_panel_kernel: rows x channels (a pair's: of both weights), and those of the last channels where they are others; and the
// slices of K.
struct TilesTaken { int rows, channels, rest_rows, rest_channels; };
inline thread_local TilesTaken gemm_tiles_taken{};
inline thread_local int gemm_slices_taken = 1;
static inline const char* gemm_tiles_name() {
  static thread_local char name[48];
  const TilesTaken& t = gemm_tiles_taken;
  const int n = t.rows ? snprintf(name, sizeof name, "%dx%d", t.rows, t.channels) : (name[0] = 0);
  if (t.rest_rows) snprintf(name + n, sizeof name - n, " %dx%d", t.rest_rows, t.rest_channels);
  return name;
}
constexpr int GEMM_MAX_KSPLIT = 4;
constexpr int GEMM_MAX_ROWS = 4096;
// From so many features on the rows of a workgroup (up to 256, and 48 rows past the last one) take more bytes than the 32-bit offsets of
// the kernels for more than 16 rows, and of gemm_own_kernel, reach.
constexpr int GEMM_FAR = 1 << 22;

template <class Fmt, int MT, int NW, bool PAIR>
__global__ __launch_bounds__(NW * 64) void gemv_mfma_kernel(GemmArgs a) {
  constexpr int NACC = PAIR ? 2 : 1;
  constexpr int KV = Fmt::kVec;
  __shared__ float red[NW * NACC * MT * 256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int mi = 0;
  if (!PAIR) {
#pragma unroll
    for (int i = 1; i < 4; ++i)
      if (i < a.count && (int)blockIdx.x >= a.mat[i].nb_begin) mi = i;
  }
  const int nb = blockIdx.x - a.mat[mi].nb_begin;
  const int N = a.mat[mi].N;
  const int row = nb * 16 + (lane & 15);
  const int K = a.K, KT = a.KT;

  typename Fmt::Scale sc[NACC];
  const u32x4* wp[NACC];
#pragma unroll
  for (int g = 0; g < NACC; ++g) {
    const GemmMat& m = a.mat[PAIR ? g : mi];
    sc[g] = Fmt::load_scale(m.scale, a.x_scale, row, N);
    wp[g] = reinterpret_cast<const u32x4*>(m.tiled) + (size_t)nb * KT * (64 * KV) + lane;
  }
  // B operand source: row (mt*16 + lane%16) of X, clamped into range; lanes of padding rows
  // compute values that are never stored.
  const f16* xrow[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    int m = mt * 16 + (lane & 15);
    m = m < a.M ? m : a.M - 1;
    xrow[mt] = (a.mat[mi].X ? a.mat[mi].X : a.X) + (size_t)m * K + (lane >> 4) * 8;
  }

  f32x4 acc[NACC][MT];
#pragma unroll
  for (int g = 0; g < NACC; ++g)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[g][mt] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll 2
  for (int kt = wave; kt < KT; kt += NW) {
    u32x4 w[NACC][KV];
#pragma unroll
    for (int g = 0; g < NACC; ++g)
#pragma unroll
      for (int v = 0; v < KV; ++v)
        w[g][v] = __builtin_nontemporal_load(wp[g] + ((size_t)kt * KV + v) * 64);
    f16x8 xb[4][MT];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = kt * 128 + j * 32;
      const bool in = k + (lane >> 4) * 8 < K;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        f16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
        xb[j][mt] = in ? *reinterpret_cast<const f16x8*>(xrow[mt] + k) : z;
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int g = 0; g < NACC; ++g) {
        const f16x8 av = Fmt::a_operand(w[g], j, sc[g]);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[g][mt] = Fmt::mma(av, xb[j][mt], acc[g][mt]);
      }
    }
  }

  // Cross-wave reduction through LDS, then the epilogue.  The accumulator of lane l holds
  // channels (l/16)*4 + r, r = 0..3, for activation row l%16.
#pragma unroll
  for (int g = 0; g < NACC; ++g)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[(((wave * NACC + g) * MT + mt) * 4 + r) * 64 + lane] = acc[g][mt][r];
  __syncthreads();
  for (int idx = threadIdx.x; idx < MT * 256; idx += NW * 64) {
    const int nn = idx & 15;  // channel inside the block
    const int m = idx >> 4;   // activation row
    const int n = nb * 16 + nn;
    if (m >= a.M || n >= N) continue;
    const int mt = m >> 4, r = nn & 3, ln = (nn >> 2) * 16 + (m & 15);
    float sum[NACC];
#pragma unroll
    for (int g = 0; g < NACC; ++g) {
      float t = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) t += red[(((w * NACC + g) * MT + mt) * 4 + r) * 64 + ln];
      sum[g] = Fmt::finish(t, sc[g]);
    }
    if (PAIR) {
      gemm_put_pair<Fmt>(a.epi, a.mat[0], m, n, N, sum[0], sum[1]);
    } else {
      gemm_put<Fmt>(a.epi, a.mat[mi], m, n, N, sum[0]);
    }
  }
}


// ------------------------------------------------------------------------------------------
// Variant for very small M (M <= 4): the activation rows are staged once per workgroup in LDS
// (M*K*2 bytes) and the B operand comes from LDS reads, which are broadcasts when M == 1.
// The first weight tile is requested before the staging so that HBM latency overlaps it.
// ------------------------------------------------------------------------------------------
template <class Fmt, int NW, bool PAIR>
__global__ __launch_bounds__(NW * 64) void gemv_lds_kernel(GemmArgs a) {
  constexpr int NACC = PAIR ? 2 : 1;
  constexpr int KV = Fmt::kVec;
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int mi = 0;
  if (!PAIR) {
#pragma unroll
    for (int i = 1; i < 4; ++i)
      if (i < a.count && (int)blockIdx.x >= a.mat[i].nb_begin) mi = i;
  }
  const int nb = blockIdx.x - a.mat[mi].nb_begin;
  const int N = a.mat[mi].N;
  const int row = nb * 16 + (lane & 15);
  const int K = a.K, KT = a.KT, M = a.M;
  const int xstride = KT * 128 + 8;                 // +8 halves: rows land in different banks
  f16* xs = reinterpret_cast<f16*>(smem);
  float* red = reinterpret_cast<float*>(smem + (((size_t)M * xstride * 2 + 15) & ~(size_t)15));

  typename Fmt::Scale sc[NACC];
  const u32x4* wp[NACC];
#pragma unroll
  for (int g = 0; g < NACC; ++g) {
    const GemmMat& m = a.mat[PAIR ? g : mi];
    sc[g] = Fmt::load_scale(m.scale, a.x_scale, row, N);
    wp[g] = reinterpret_cast<const u32x4*>(m.tiled) + (size_t)nb * KT * (64 * KV) + lane;
  }
  // first tile of this wave: requested before anything else
  u32x4 wcur[NACC][KV];
  int kt = wave;
  if (kt < KT) {
#pragma unroll
    for (int g = 0; g < NACC; ++g)
#pragma unroll
      for (int v = 0; v < KV; ++v) wcur[g][v] = __builtin_nontemporal_load(wp[g] + ((size_t)kt * KV + v) * 64);
  }
  // (bf16, 1 row, 2048 x 2048: 4.4 against 4.6 us; the fp16 epilogue's few arguments gain nothing)
  GemmMat wide;
  GemmEpilogue none{};
  if constexpr (Fmt::kWide) {
    wide = a.mat[PAIR ? 0 : mi];
    read_end<Fmt, PAIR>(wide, none);
  }
  // stage X (zero beyond K), normalising its rows on the way when a norm is fused
  {
    const int vec_per_row = KT * 16;               // 8-half vectors per padded row
    float ps[4] = {0.f, 0.f, 0.f, 0.f}, pq[4] = {0.f, 0.f, 0.f, 0.f};
    for (int i = threadIdx.x; i < M * vec_per_row; i += NW * 64) {
      const int m = i / vec_per_row, c = i % vec_per_row;
      f16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
      if (c * 8 < K) v = *reinterpret_cast<const f16x8*>((a.mat[mi].X ? a.mat[mi].X : a.X) + (size_t)m * K + c * 8);
      *reinterpret_cast<f16x8*>(xs + (size_t)m * xstride + c * 8) = v;
      if (a.epi.norm != PTA_NORM_NONE) {
        float s1 = 0.f, s2 = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) { const float f = (float)v[e]; s1 += f; s2 = __builtin_fmaf(f, f, s2); }
#pragma unroll
        for (int mm = 0; mm < 4; ++mm) if (mm == m) { ps[mm] += s1; pq[mm] += s2; }
      }
    }
    if (a.epi.norm != PTA_NORM_NONE) {
      // per-row sums over the workgroup: over the wave by data-parallel moves (a chain of six LDS-crossbar shuffles
      // per sum took longer than the norm launch this replaces), then LDS (the reduction buffer is free here)
#pragma unroll
      for (int mm = 0; mm < 4; ++mm)
        if (mm < M) { ps[mm] = wave_total_dpp(ps[mm]); pq[mm] = wave_total_dpp(pq[mm]); }
      if (lane == 0) {
#pragma unroll
        for (int mm = 0; mm < 4; ++mm) { red[(wave * 4 + mm) * 2] = ps[mm]; red[(wave * 4 + mm) * 2 + 1] = pq[mm]; }
      }
      __syncthreads();
      const float inv_n = 1.0f / (float)K;
      for (int i = threadIdx.x; i < M * vec_per_row; i += NW * 64) {
        const int m = i / vec_per_row, c = i % vec_per_row;
        if (c * 8 >= K) continue;
        float sum = 0.f, sq = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) { sum += red[(w * 4 + m) * 2]; sq += red[(w * 4 + m) * 2 + 1]; }
        f16x8 v = *reinterpret_cast<f16x8*>(xs + (size_t)m * xstride + c * 8);
        const f16x8 gm = *reinterpret_cast<const f16x8*>(a.epi.norm_weight + c * 8);
        if (a.epi.norm == PTA_NORM_RMS) {
          const f16 r16 = (f16)(1.0f / sqrtf(sq * inv_n + a.epi.norm_eps));
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = (v[e] * r16) * gm[e];
        } else {
          const f16x8 bt = *reinterpret_cast<const f16x8*>(a.epi.norm_bias + c * 8);
          const float mean = sum * inv_n;
          const f16 mean16 = (f16)mean;
          float var;
          if (M == 1) var = sq * inv_n - mean * mean + a.epi.norm_eps;          // single-row NormCE
          else { const float mf = (float)mean16; var = fmaxf(sq * inv_n - mf * mf, 0.0f) + a.epi.norm_eps; }
          const f16 r16 = (f16)(1.0f / sqrtf(var));
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = ((v[e] - mean16) * r16) * gm[e] + bt[e];
        }
        *reinterpret_cast<f16x8*>(xs + (size_t)m * xstride + c * 8) = v;
      }
    }
    if (a.epi.mix_state) {
      // token shift: this matrix's input is x * w + (1 - w) * prev, each step an fp16 operation as in pta_rwkv_mix;
      // prev is the copy of the state that the previous token's launch wrote, x goes to the other one (first
      // workgroup) - no workgroup of this launch reads the copy that is written
      // (a thread mixes the vectors it staged and normalised itself: no barrier in between)
      const int parity = a.epi.mix_step[0] & 1;
      const f16* prev = a.epi.mix_state + (size_t)parity * M * K;
      f16* next = a.epi.mix_state + (size_t)(parity ^ 1) * M * K;
      const f16* mw = a.mat[mi].mix;
      const f16 one = (f16)1.0f;
      for (int i = threadIdx.x; i < M * vec_per_row; i += NW * 64) {
        const int m = i / vec_per_row, c = i % vec_per_row;
        if (c * 8 >= K) continue;
        f16x8 v = *reinterpret_cast<f16x8*>(xs + (size_t)m * xstride + c * 8);
        if (blockIdx.x == 0) *reinterpret_cast<f16x8*>(next + (size_t)m * K + c * 8) = v;
        if (mw) {
          const f16x8 pv = *reinterpret_cast<const f16x8*>(prev + (size_t)m * K + c * 8);
          const f16x8 wv = *reinterpret_cast<const f16x8*>(mw + c * 8);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = v[e] * wv[e] + (one - wv[e]) * pv[e];
          *reinterpret_cast<f16x8*>(xs + (size_t)m * xstride + c * 8) = v;
        }
      }
    }
  }
  __syncthreads();
  int mrow = lane & 15;
  mrow = mrow < M ? mrow : M - 1;
  const f16* xl = xs + (size_t)mrow * xstride + (lane >> 4) * 8;

  f32x4 acc[NACC];
#pragma unroll
  for (int g = 0; g < NACC; ++g) acc[g] = f32x4{0.f, 0.f, 0.f, 0.f};

  while (kt < KT) {
    const int ktn = kt + NW;
    u32x4 wnext[NACC][KV];
    if (ktn < KT) {
#pragma unroll
      for (int g = 0; g < NACC; ++g)
#pragma unroll
        for (int v = 0; v < KV; ++v) wnext[g][v] = __builtin_nontemporal_load(wp[g] + ((size_t)ktn * KV + v) * 64);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f16x8 xb = *reinterpret_cast<const f16x8*>(xl + kt * 128 + j * 32);
#pragma unroll
      for (int g = 0; g < NACC; ++g) {
        const f16x8 av = Fmt::a_operand(wcur[g], j, sc[g]);
        acc[g] = Fmt::mma(av, xb, acc[g]);
      }
    }
    if (ktn < KT) {
#pragma unroll
      for (int g = 0; g < NACC; ++g)
#pragma unroll
        for (int v = 0; v < KV; ++v) wcur[g][v] = wnext[g][v];
    }
    kt = ktn;
  }

#pragma unroll
  for (int g = 0; g < NACC; ++g)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[((wave * NACC + g) * 4 + r) * 64 + lane] = acc[g][r];
  __syncthreads();
  for (int idx = threadIdx.x; idx < 256; idx += NW * 64) {
    const int nn = idx & 15, m = idx >> 4;
    const int n = nb * 16 + nn;
    if (m >= M || n >= N) continue;
    const int r = nn & 3, ln = (nn >> 2) * 16 + m;
    float sum[NACC];
#pragma unroll
    for (int g = 0; g < NACC; ++g) {
      float t = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) t += red[((w * NACC + g) * 4 + r) * 64 + ln];
      sum[g] = Fmt::finish(t, sc[g]);
    }
    if (PAIR) {
      gemm_put_pair<Fmt>(a.epi, Fmt::kWide ? wide : a.mat[0], m, n, N, sum[0], sum[1]);
    } else {
      gemm_put<Fmt>(a.epi, Fmt::kWide ? wide : a.mat[mi], m, n, N, sum[0]);
    }
  }
}

// ------------------------------------------------------------------------------------------
// Variant for 4 < M <= 16 (F152 weights: up to 32) when all matrices of the launch share X: one workgroup of 16 waves per
// compute unit's worth of work.  A workgroup owns NB 16-channel blocks (blocks g, g + G, ... of
// the launch's G workgroups); wave w takes the feature tiles w, w + 16, ... of ALL of them, so the
// activation fragments of a tile (the B operands: 4 KiB per 16 rows, against 1 KiB of INT4
// weights) are read once and used NB times, and every wave has NB weight tiles per feature tile
// in flight.  MT = number of 16-row groups of X.
// ------------------------------------------------------------------------------------------
constexpr int WIDE_WAVES = 16;

template <class Fmt, int MT, int NB, bool PAIR, bool NORM = false>
__global__ __launch_bounds__(WIDE_WAVES * 64) void gemv_wide_kernel(GemmArgs a, int total_nb) {
  static_assert(!NORM || MT == 1, "the fused norm covers up to 16 rows");
  constexpr int NACC = PAIR ? 2 : 1;
  constexpr int KV = Fmt::kVec;
  extern __shared__ __align__(16) unsigned char smem[];
  float* red = reinterpret_cast<float*>(smem);          // [WIDE_WAVES][NB][NACC][MT][256]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int G = gridDim.x;
  const int K = a.K, KT = a.KT;

  int mi[NB], nb[NB];
  typename Fmt::Scale sc[NB][NACC];
  const u32x4* wp[NB][NACC];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    int blk = blockIdx.x + b * G;
    blk = blk < total_nb ? blk : total_nb - 1;          // a duplicate whose results are not stored
    int m_ = 0;
    if (!PAIR) {
#pragma unroll
      for (int i = 1; i < 4; ++i)
        if (i < a.count && blk >= a.mat[i].nb_begin) m_ = i;
    }
    mi[b] = m_;
    nb[b] = blk - a.mat[m_].nb_begin;
    const int row = nb[b] * 16 + (lane & 15);
#pragma unroll
    for (int g = 0; g < NACC; ++g) {
      const GemmMat& m = a.mat[PAIR ? g : m_];
      sc[b][g] = Fmt::load_scale(m.scale, a.x_scale, row, m.N);
      wp[b][g] = reinterpret_cast<const u32x4*>(m.tiled) + (size_t)nb[b] * KT * (64 * KV) + lane;
    }
  }
  const f16* xrow[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    int row = mt * 16 + (lane & 15);
    row = row < a.M ? row : a.M - 1;                    // padding rows compute values that are never stored
    xrow[mt] = a.X + (size_t)row * K + (lane >> 4) * 8;
  }

  f32x4 acc[NB][NACC][MT];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int g = 0; g < NACC; ++g)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[b][g][mt] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Fused norm: a first pass over this wave's activation fragments gives the row sums (lane l
  // holds row l % 16, features (l / 16) * 8 + 0..7 of every 32), they meet over the lane groups and, in
  // LDS, over the waves; the product pass then normalises every fragment it loads, with the numerics of
  // pta_rmsnorm / pta_layer_norm_ce (rows > 1 variant).
  f16 n_mean = (f16)0.0f, n_r = (f16)1.0f;
  auto norm_statistics = [&]() {
    float s1 = 0.f, s2 = 0.f;
    for (int kt = wave; kt < KT; kt += WIDE_WAVES)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = kt * 128 + j * 32;
        if (k + (lane >> 4) * 8 < K) {
          const f16x8 v = *reinterpret_cast<const f16x8*>(xrow[0] + k);
#pragma unroll
          for (int e = 0; e < 8; ++e) { const float f = (float)v[e]; s1 += f; s2 = __builtin_fmaf(f, f, s2); }
        }
      }
    s1 += __shfl_xor(s1, 16, 64); s2 += __shfl_xor(s2, 16, 64);
    s1 += __shfl_xor(s1, 32, 64); s2 += __shfl_xor(s2, 32, 64);
    if (lane < 16) { red[(wave * 16 + lane) * 2] = s1; red[(wave * 16 + lane) * 2 + 1] = s2; }
    __syncthreads();
    float sum = 0.f, sq = 0.f;
#pragma unroll
    for (int w = 0; w < WIDE_WAVES; ++w) { sum += red[(w * 16 + (lane & 15)) * 2]; sq += red[(w * 16 + (lane & 15)) * 2 + 1]; }
    __syncthreads();      // the buffer is reused for the partial sums of the product
    const float inv_n = 1.0f / (float)K;
    if (a.epi.norm == PTA_NORM_RMS) {
      n_r = (f16)(1.0f / sqrtf(sq * inv_n + a.epi.norm_eps));
    } else {
      const float mean = sum * inv_n;
      n_mean = (f16)mean;
      float var;
      if (a.M == 1) var = sq * inv_n - mean * mean + a.epi.norm_eps;          // single-row NormCE
      else { const float mf = (float)n_mean; var = fmaxf(sq * inv_n - mf * mf, 0.0f) + a.epi.norm_eps; }
      n_r = (f16)(1.0f / sqrtf(var));
    }
  };
  // UN feature tiles per step, all of their loads requested before the first product (a tile
  // beyond KT repeats the last one with zero activations)
  constexpr int UN = NB * NACC * KV <= 4 ? 2 : 1;
  u32x4 w[UN][NB][NACC][KV];
  f16x8 xb[UN][4];
  auto load_w = [&](int kt0) {
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int kt_ = kt0 + u * WIDE_WAVES;
      const int kt = kt_ < KT ? kt_ : KT - 1;
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int g = 0; g < NACC; ++g)
#pragma unroll
          for (int v = 0; v < KV; ++v)
            w[u][b][g][v] = __builtin_nontemporal_load(wp[b][g] + ((size_t)kt * KV + v) * 64);
    }
  };
  auto load_x = [&](int kt0) {
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int kt_ = kt0 + u * WIDE_WAVES;
      const bool there = kt_ < KT;
      const int kt = there ? kt_ : KT - 1;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = kt * 128 + j * 32;
        const f16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
        const bool in = there && k + (lane >> 4) * 8 < K;
        xb[u][j] = in ? *reinterpret_cast<const f16x8*>(xrow[0] + k) : z;
        if (NORM && in) {
          const f16x8 gm = *reinterpret_cast<const f16x8*>(a.epi.norm_weight + k + (lane >> 4) * 8);
          if (a.epi.norm == PTA_NORM_RMS) {
#pragma unroll
            for (int e = 0; e < 8; ++e) xb[u][j][e] = (xb[u][j][e] * n_r) * gm[e];
          } else {
            const f16x8 bt = *reinterpret_cast<const f16x8*>(a.epi.norm_bias + k + (lane >> 4) * 8);
#pragma unroll
            for (int e = 0; e < 8; ++e) xb[u][j][e] = ((xb[u][j][e] - n_mean) * n_r) * gm[e] + bt[e];
          }
        }
      }
    }
  };
  auto products = [&]() {
#pragma unroll
    for (int u = 0; u < UN; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int g = 0; g < NACC; ++g)
            acc[b][g][0] = Fmt::mma(Fmt::a_operand(w[u][b][g], j, sc[b][g]), xb[u][j],
                                                                     acc[b][g][0]);
  };
  int kt0 = wave;
  if constexpr (NORM) {
    // Fused norm: the first weight tiles are requested before the pass over the activations that gives the
    // row statistics (lane l holds row l % 16, features (l / 16) * 8 + 0..7 of every 32; the sums meet over
    // the lane groups and, in LDS, over the waves), so that pass runs while they are on their way.  The
    // product pass then normalises every fragment it loads, with the numerics of pta_rmsnorm /
    // pta_layer_norm_ce (rows > 1 variant).
    if (kt0 < KT) load_w(kt0);
    norm_statistics();
    if (kt0 < KT) {
      load_x(kt0);
      products();
      kt0 += WIDE_WAVES * UN;
    }
  }
  if constexpr (MT == 1) {
    for (; kt0 < KT; kt0 += WIDE_WAVES * UN) {
      load_w(kt0);
      load_x(kt0);
      products();
    }
  } else {
    // several row groups: the activations of 32 features at a time, each used for all blocks; a weight operand is decoded once for all rows
    for (; kt0 < KT; kt0 += WIDE_WAVES) {
      u32x4 wt[NB][NACC][KV];
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int g = 0; g < NACC; ++g)
#pragma unroll
          for (int v = 0; v < KV; ++v) wt[b][g][v] = __builtin_nontemporal_load(wp[b][g] + ((size_t)kt0 * KV + v) * 64);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = kt0 * 128 + j * 32;
        f16x8 xs[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) xs[mt] = k + (lane >> 4) * 8 < K ? *reinterpret_cast<const f16x8*>(xrow[mt] + k) : f16x8{};
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int g = 0; g < NACC; ++g) {
            const f16x8 av = Fmt::a_operand(wt[b][g], j, sc[b][g]);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[b][g][mt] = Fmt::mma(av, xs[mt], acc[b][g][mt]);
          }
      }
    }
  }

  // The accumulator of lane l holds channels (l/16)*4 + r, r = 0..3, for activation row l%16 of its group.
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int g = 0; g < NACC; ++g)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[((((wave * NB + b) * NACC + g) * MT + mt) * 4 + r) * 64 + lane] = acc[b][g][mt][r];
  __syncthreads();
  // The 256 outputs (16 rows x 16 channels) of row group mt of block b are finished by quarter (b * MT + mt) % 4 of the workgroup,
  // thread t of it taking row (t / 16) % 16, channel t % 16.
  const int quarter = threadIdx.x >> 8;
#pragma unroll
  for (int i = 0; i < NB * MT; ++i) {
    if ((i & 3) != quarter) continue;
    const int b = i / MT, mt = i % MT;
    const int nn = threadIdx.x & 15, m = mt * 16 + ((threadIdx.x >> 4) & 15);
    const GemmMat& mat = a.mat[PAIR ? 0 : mi[b]];
    const int N = mat.N, n = nb[b] * 16 + nn;
    if ((int)blockIdx.x + b * G >= total_nb || m >= a.M || n >= N) continue;
    const int r = nn & 3, ln = (nn >> 2) * 16 + (m & 15);
    float sum[NACC];
#pragma unroll
    for (int g = 0; g < NACC; ++g) {
      float t = 0.f;
#pragma unroll
      for (int w = 0; w < WIDE_WAVES; ++w) t += red[((((w * NB + b) * NACC + g) * MT + mt) * 4 + r) * 64 + ln];
      sum[g] = Fmt::finish(t, sc[b][g]);      // no format's finish uses the per-channel part of the scale
    }
    if (PAIR) gemm_put_pair<Fmt>(a.epi, mat, m, n, N, sum[0], sum[NACC - 1]);
    else gemm_put<Fmt>(a.epi, mat, m, n, N, sum[0]);
  }
}

template <class Fmt, int MT, int NB, bool PAIR, bool NORM>
static int launch_gemv_wide(const GemmArgs& a, int total_nb, hipStream_t s, const char* name) {
  static bool ready = false;
  const size_t smem = (size_t)WIDE_WAVES * NB * (PAIR ? 2 : 1) * MT * 256 * sizeof(float);
  if (!ready) {
    PTA_REQUIRE(hipFuncSetAttribute((const void*)gemv_wide_kernel<Fmt, MT, NB, PAIR, NORM>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) == hipSuccess,
                "%s: cannot reserve %zu bytes of LDS", name, smem);
    ready = true;
  }
  gemm_kernel_taken = "gemv_wide_kernel";
  hipLaunchKernelGGL((gemv_wide_kernel<Fmt, MT, NB, PAIR, NORM>), dim3((total_nb + NB - 1) / NB), dim3(WIDE_WAVES * 64), smem, s,
                     a, total_nb);
  return PTA_OK;
}

// blocks per workgroup: the launch's share per compute unit, capped by what the registers of a wave (weight tiles in flight) hold
template <class Fmt, bool PAIR>
constexpr int wide_cap() { return Fmt::kVec * (PAIR ? 2 : 1) <= 4 ? 3 : 2; }

template <class Fmt, int MT, bool PAIR, bool NORM>
static int launch_gemv_wide_for(const GemmArgs& a, int total_nb, int per_cu, hipStream_t s, const char* name) {
  constexpr int cap = wide_cap<Fmt, PAIR>();
  if (per_cu <= 1) return launch_gemv_wide<Fmt, MT, 1, PAIR, NORM>(a, total_nb, s, name);
  if (per_cu == 2 || cap == 2) return launch_gemv_wide<Fmt, MT, 2, PAIR, NORM>(a, total_nb, s, name);
  return launch_gemv_wide<Fmt, MT, cap, PAIR, NORM>(a, total_nb, s, name);
}

// the longest chain of channel blocks a compute unit multiplies under launch_gemv_wide_for
template <class Fmt, bool PAIR>
static int wide_block_times(int total_nb, int per_cu) {
  const int nb = per_cu < wide_cap<Fmt, PAIR>() ? per_cu : wide_cap<Fmt, PAIR>();
  const int cus = device_compute_units();
  const int wgs = (total_nb + nb - 1) / nb;
  return (wgs + cus - 1) / cus * nb;
}

// ------------------------------------------------------------------------------------------
// Variant for up to 16 rows, one shared X, K <= 4096 and several channel blocks per compute unit: one workgroup
// of 8 waves per compute unit walks a contiguous range of the launch's 16-channel blocks.  Wave w takes the
// feature tiles w, w + 8, ... of every block, U at a time (a step; a block is up to 4 / U steps long).  The
// weights of the next D - 1 steps are on their way while those of the current one are multiplied, across block
// boundaries as well, so the stream does not pause for a reduction or for a change of workgroups; the partial
// sums of a block meet in LDS (two buffers in turn, one barrier per block) and 256 threads finish its 16 x 16
// outputs while the others go on.  The activation fragments of a wave's tiles are the same for every block
// and stay in registers (x[p]: those of a block's step p).
// ------------------------------------------------------------------------------------------
constexpr int STREAM_WAVES = 8;
constexpr int STREAM_TILES = 4;          // feature tiles of a block per wave, at most: K <= 8 * 4 * 128

template <class Fmt, int U, int D, bool PAIR>
__global__ __launch_bounds__(STREAM_WAVES * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemv_stream_kernel(GemmArgs a, int total_nb) {
  constexpr int XP = STREAM_TILES / U;     // steps of a block, at most
  static_assert(D % XP == 0, "a step's place in the ring of weight sets tells its place in the block");
  constexpr int NACC = PAIR ? 2 : 1;
  constexpr int KV = Fmt::kVec;
  __shared__ float red[2][STREAM_WAVES][NACC][256];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = a.K, KT = a.KT;
  const int G = gridDim.x;
  const int b0 = (int)((long)total_nb * blockIdx.x / G), b1 = (int)((long)total_nb * (blockIdx.x + 1) / G);
  // steps per block: 1, 2 or 4 (a divisor of the ring's length; a step past the end of K multiplies zeros)
  const int spb = KT <= STREAM_WAVES * U ? 1 : KT <= 2 * STREAM_WAVES * U ? 2 : XP;
  const int steps = (b1 - b0) * spb;
  if (steps == 0) return;

  struct Set {
    u32x4 w[U][NACC][KV];
    typename Fmt::Scale sc[NACC];
    uint16_t e[4];      // epilogue operands of the output this thread finishes: the matrix's bias, then bias, mul, residual
  };
  Set ring[D];
  typename Fmt::Scale sc[NACC];
  f32x4 acc[NACC];
#pragma unroll
  for (int g = 0; g < NACC; ++g) acc[g] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto matrix_of = [&](int blk) {
    int m_ = 0;
    if (!PAIR) {
#pragma unroll
      for (int i = 1; i < 4; ++i)
        if (i < a.count && blk >= a.mat[i].nb_begin) m_ = i;
    }
    return m_;
  };

  // The requesting side runs D - 1 steps ahead of the multiplying side.  Every step issues the same loads whatever
  // the data (a wait for one set of weights then counts the loads issued after it): they go through a buffer
  // descriptor of the block's matrix, and a tile past the end of K, or a step past the end of the workgroup's
  // range, is given an offset beyond the descriptor's range - it reads as zero and touches no memory.
  const uint32_t blk_bytes = (uint32_t)KT * (KV * 1024);
  int fb = b0, fs = 0;
  auto fetch = [&](Set& st, bool live) {
    const int m_ = matrix_of(fb);
    const int nb = fb - a.mat[m_].nb_begin;
#pragma unroll
    for (int g = 0; g < NACC; ++g) {
      const GemmMat& m = a.mat[PAIR ? g : m_];
      const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<void*>(m.tiled), 0, (int)((uint32_t)((m.N + 15) / 16) * blk_bytes), 0x00020000);
      st.sc[g] = Fmt::load_scale(m.scale, a.x_scale, nb * 16 + (lane & 15), m.N);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int kt = (fs * U + u) * STREAM_WAVES + wave;
        const int voff = live && kt < KT ? lane * 16 : -1;
#pragma unroll
        for (int v = 0; v < KV; ++v)
          st.w[u][g][v] = __builtin_amdgcn_raw_buffer_load_b128(wr, voff, (int)((uint32_t)nb * blk_bytes + (uint32_t)(kt * KV + v) * 1024), 2);
      }
    }
    if constexpr (!PAIR) {
      // The operands of the epilogue travel with the weights of the block's last step: a load issued when the block
      // is finished would wait for every set of weights requested before it.  Absent operands have an empty range.
      const GemmMat& mat = a.mat[m_];
      const int nn = threadIdx.x & 15, m = threadIdx.x >> 4, n = nb * 16 + nn;
      const bool mine = live && fs == spb - 1 && threadIdx.x < 256 && m < a.M && n < mat.N;
      const f16* ptr[4] = {mat.bias, a.epi.bias, a.epi.mul, a.epi.residual};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<f16*>(ptr[i]), 0, ptr[i] ? (i < 2 ? mat.N : a.M * mat.N) * 2 : 0, 0x00020000);
        st.e[i] = __builtin_amdgcn_raw_buffer_load_b16(r, mine ? (i < 2 ? n : m * mat.N + n) * 2 : -1, 0, 0);
      }
    }
    if (++fs == spb) { fs = 0; ++fb; }
  };

  // B operands: row lane % 16 of X (clamped: padding rows compute values that are never stored), features
  // (lane / 16) * 8 + 0..7 of every 32; x[p] holds them for the tiles of a block's step p (of its only step, when
  // a block is one step long).  Requested before the first weights: loads return in the order of their issue, and
  // the first products need these and one set of weights only.
  f16x8 x[XP][U][4];
  {
    int mrow = lane & 15;
    mrow = mrow < a.M ? mrow : a.M - 1;
    const f16* xrow = a.X + (size_t)mrow * K + (lane >> 4) * 8;
#pragma unroll
    for (int p = 0; p < XP; ++p)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int kt = ((p % spb) * U + u) * STREAM_WAVES + wave;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int k = kt * 128 + j * 32;
          const f16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
          x[p][u][j] = kt < KT && k + (lane >> 4) * 8 < K ? *reinterpret_cast<const f16x8*>(xrow + k) : z;
        }
      }
  }

#pragma unroll
  for (int i = 0; i < D - 1; ++i) fetch(ring[i], i < steps);

  int cb = b0, cs = 0, par = 0;
  auto multiply = [&](Set& st, const f16x8 (&xs)[U][4]) {
    if (cs == 0) {
#pragma unroll
      for (int g = 0; g < NACC; ++g) sc[g] = st.sc[g];
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int g = 0; g < NACC; ++g)
          acc[g] = Fmt::mma(Fmt::a_operand(st.w[u][g], j, sc[g]), xs[u][j], acc[g]);
    if (++cs < spb) return;
    // the block is complete: lane l holds channels (l/16)*4 + r, r = 0..3, for activation row l%16
#pragma unroll
    for (int g = 0; g < NACC; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        red[par][wave][g][r * 64 + lane] = acc[g][r];
        acc[g][r] = 0.f;
      }
    __syncthreads();
    if (threadIdx.x < 256) {
      const int m_ = matrix_of(cb);
      const GemmMat& mat = a.mat[PAIR ? 0 : m_];
      const int nn = threadIdx.x & 15, m = threadIdx.x >> 4;
      const int N = mat.N, n = (cb - a.mat[m_].nb_begin) * 16 + nn;
      if (m < a.M && n < N) {
        const int r = nn & 3, ln = (nn >> 2) * 16 + m;
        float sum[NACC];
#pragma unroll
        for (int g = 0; g < NACC; ++g) {
          float t = 0.f;
#pragma unroll
          for (int w = 0; w < STREAM_WAVES; ++w) t += red[par][w][g][r * 64 + ln];
          sum[g] = Fmt::finish(t, sc[g]);        // no format's finish uses the per-channel part of the scale
        }
        if (PAIR) {
          gemm_put_pair<Fmt>(a.epi, a.mat[0], m, n, N, sum[0], sum[1]);
        } else if constexpr (Fmt::kWide) {
          gemm_put<Fmt>(a.epi, mat, m, n, N, sum[0]);
        } else {
          // as apply_epilogue, with the operands that came with the weights
          f16 y0 = (f16)sum[0];
          if (mat.bias) y0 = y0 + bitcast<f16>(st.e[0]);
          y0 = apply_act(mat.act, y0);
          if (a.epi.bias) y0 = y0 + bitcast<f16>(st.e[1]);
          y0 = apply_act(a.epi.act, y0);
          if (a.epi.mul) y0 = y0 * bitcast<f16>(st.e[2]);
          if (a.epi.residual) y0 = y0 + bitcast<f16>(st.e[3]);
          if (a.epi.post_scale != 0.0f) y0 = y0 * (f16)a.epi.post_scale;
          if (a.epi.out_fp8_scale) y0 = f8_grid_value(y0, a.epi.out_fp8_scale[0], a.epi.out_fp8_format);
          mat.Y[(size_t)m * N + n] = y0;
        }
      }
    }
    par ^= 1;
    cs = 0;
    ++cb;
  };

  int t = 0;
  for (; t + D <= steps; t += D) {
#pragma unroll
    for (int i = 0; i < D; ++i) {
      fetch(ring[(i + D - 1) % D], t + i + D - 1 < steps);
      multiply(ring[i], x[i % XP]);
    }
  }
  // fewer than D steps are left and their weights are on their way
#pragma unroll
  for (int i = 0; i < D - 1; ++i)
    if (t + i < steps) multiply(ring[i], x[i % XP]);
}

// the shapes the streaming kernel takes
static inline bool stream_fits(const GemmArgs& a) {
  if (a.M > 16 || a.KT < 8 || a.KT > STREAM_WAVES * STREAM_TILES || a.epi.norm != PTA_NORM_NONE) return false;
  for (int i = 0; i < a.count; ++i) {
    if (a.mat[i].X) return false;
    // a matrix's tiles sit behind one buffer descriptor (32-bit range and offsets; four vectors per tile at most)
    if ((size_t)((a.mat[i].N + 15) / 16) * (size_t)a.KT * 4096 > 0x7fffffffu) return false;
  }
  return true;
}

template <class Fmt, bool PAIR>
static int launch_gemv_stream(const GemmArgs& a, int total_nb, int cus, hipStream_t s, const char* name) {
  // tiles per step, and four steps in the ring: 96 KiB on their way per compute unit, a ring of 64 registers
  constexpr int V = Fmt::kVec * (PAIR ? 2 : 1);
  constexpr int U = V >= 4 ? 1 : V >= 2 ? 2 : 4, D = 4;
  gemm_kernel_taken = "gemv_stream_kernel";
  hipLaunchKernelGGL((gemv_stream_kernel<Fmt, U, D, PAIR>), dim3(total_nb < cus ? total_nb : cus), dim3(STREAM_WAVES * 64), 0, s, a,
                     total_nb);
  return PTA_OK;
}

// ------------------------------------------------------------------------------------------
// Variant for 16 < M <= 64 and launches that gemm_own_kernel's workgroups would be several rounds of (dispatch_gemv has the lines): the
// activation rows of a feature tile are staged in LDS once per workgroup and shared by its waves, so that the B operands (4 KiB per 16 rows and tile, against
// 1 KiB of INT4 weights) come from LDS and not from the L2.
// A workgroup of 8 (NWV; 16 where the dispatch says so) waves owns 2 * (8 / KQ) weight streams of 16 channels (consecutive channel blocks
// of one matrix; or, for a SwiGLU pair, the gate and the up weights of 8 / KQ channel blocks) and
// all rows; its waves form KQ groups that take the feature tiles g, g + KQ, ... each; a wave
// multiplies two streams, so every B fragment it reads from LDS feeds two MFMAs.  The X tiles of
// step i + 1 are fetched (global -> registers -> LDS, double-buffered) while step i is multiplied,
// and so are the weight tiles.  The partial sums of the KQ groups meet in LDS (the staging area).
// ------------------------------------------------------------------------------------------
constexpr int TILE_WAVES = 8;
constexpr int TILE_XSTRIDE = 128 + 8;      // halves per staged row: 16 consecutive rows hit 16 different bank groups

template <class Fmt, int MT, int KQ, bool PAIR, int NWV = TILE_WAVES>
__global__ __launch_bounds__(NWV * 64) void gemm_tile_kernel(GemmArgs a) {
  constexpr int KV = Fmt::kVec;
  constexpr int WPG = NWV / KQ;          // waves per K group
  constexpr int ROWS = MT * 16;
  constexpr int XBUF = ROWS * TILE_XSTRIDE;     // halves of one staged tile
  constexpr int VPT = ROWS * 16 / (WPG * 64);   // 16-byte vectors of a tile per thread of its group
  static_assert(VPT >= 1 && ROWS * 16 % (WPG * 64) == 0, "staging must divide evenly");
  extern __shared__ __align__(16) unsigned char smem[];
  f16* xs = reinterpret_cast<f16*>(smem);       // [KQ][2][ROWS][TILE_XSTRIDE]
  float* red = reinterpret_cast<float*>(smem);  // after the product: [NWV][2][MT][256]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kq = wave / WPG, wg_ = wave % WPG;  // K group, wave within the group
  const int tig = wg_ * 64 + lane;              // thread index within the group
  const int K = a.K, M = a.M;
  const int KT = a.KT;

  // the two weight streams of this wave
  int mi = 0;
  const int first_blk = PAIR ? (int)blockIdx.x * WPG : (int)blockIdx.x * 2 * WPG;
  if (!PAIR) {
#pragma unroll
    for (int i = 1; i < 4; ++i)
      if (i < a.count && first_blk >= a.mat[i].nb_begin) mi = i;
  }
  int nb[2];
  typename Fmt::Scale sc[2];
  const u32x4* wp[2];
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    const GemmMat& m = a.mat[PAIR ? st : mi];
    nb[st] = PAIR ? first_blk + wg_ : first_blk - m.nb_begin + 2 * wg_ + st;
    sc[st] = Fmt::load_scale(m.scale, a.x_scale, nb[st] * 16 + (lane & 15), m.N);
    wp[st] = reinterpret_cast<const u32x4*>(m.tiled) + (size_t)nb[st] * KT * (64 * KV) + lane;
  }
  const f16* X = a.mat[mi].X ? a.mat[mi].X : a.X;

  f32x4 acc[2][MT];
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[st][mt] = f32x4{0.f, 0.f, 0.f, 0.f};

  // thread tig of a group stages vectors tig, tig + WPG*64, ... of the tile: vector v = row * 16 + c
  auto fetch_x = [&](int kt, u32x4 (&xv)[VPT]) {
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int v = tig + i * WPG * 64;
      const int row = v >> 4, c = v & 15;
      const int k = kt * 128 + c * 8;
      xv[i] = (row < M && k < K && kt < KT) ? *reinterpret_cast<const u32x4*>(X + (size_t)row * K + k) : u32x4{0, 0, 0, 0};
    }
  };
  auto store_x = [&](f16* buf, const u32x4 (&xv)[VPT]) {
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int v = tig + i * WPG * 64;
      *reinterpret_cast<u32x4*>(buf + (v >> 4) * TILE_XSTRIDE + (v & 15) * 8) = xv[i];
    }
  };
  auto fetch_w = [&](int kt, u32x4 (&w)[2][KV]) {
    const int ktc = kt < KT ? kt : KT - 1;
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int v = 0; v < KV; ++v) w[st][v] = __builtin_nontemporal_load(wp[st] + ((size_t)ktc * KV + v) * 64);
  };

  f16* xbuf = xs + (size_t)kq * 2 * XBUF;
  const int steps = (KT + KQ - 1) / KQ;
  u32x4 w_cur[2][KV], w_nxt[2][KV], xv[VPT];
  fetch_w(kq, w_cur);
  fetch_x(kq, xv);
  store_x(xbuf, xv);
  __syncthreads();
  for (int i = 0; i < steps; ++i) {
    const int kt = kq + i * KQ, ktn = kt + KQ;
    const bool more = i + 1 < steps;
    if (more) { fetch_w(ktn, w_nxt); fetch_x(ktn, xv); }
    const f16* cur = xbuf + (i & 1) * XBUF + (lane & 15) * TILE_XSTRIDE + (lane >> 4) * 8;
    if (kt < KT) {
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        f16x8 xb[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) xb[mt] = *reinterpret_cast<const f16x8*>(cur + mt * 16 * TILE_XSTRIDE + m * 32);
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          const f16x8 av = Fmt::a_operand(w_cur[st], m, sc[st]);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[st][mt] = Fmt::mma(av, xb[mt], acc[st][mt]);
        }
      }
    }
    if (more) {
      store_x(xbuf + ((i + 1) & 1) * XBUF, xv);
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int v = 0; v < KV; ++v) w_cur[st][v] = w_nxt[st][v];
    }
    __syncthreads();
  }

  // partial sums of the K groups meet in LDS (the staging area is free after the last barrier)
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[(((wave * 2 + st) * MT + mt) * 4 + r) * 64 + lane] = acc[st][mt][r];
  __syncthreads();
  // outputs of the workgroup: WPG wave slots x 2 streams x MT row groups x 256; PAIR: one output per stream pair
  constexpr int OUTS = WPG * (PAIR ? 1 : 2) * MT * 256;
  for (int o = threadIdx.x; o < OUTS; o += NWV * 64) {
    const int nn = o & 15, m16 = (o >> 4) & 15;
    int rest = o >> 8;
    const int mt = rest % MT; rest /= MT;
    const int st = PAIR ? 0 : rest & 1;
    const int wslot = PAIR ? rest : rest >> 1;
    const int m = mt * 16 + m16;
    const GemmMat& mat = a.mat[PAIR ? 0 : mi];
    const int N = mat.N;
    const int blk = PAIR ? first_blk + wslot : first_blk - mat.nb_begin + 2 * wslot + st;
    const int n = blk * 16 + nn;
    if (m >= M || n >= N) continue;
    const int r = nn & 3, ln = (nn >> 2) * 16 + m16;
    float sum[2] = {0.f, 0.f};
#pragma unroll
    for (int g = 0; g < (PAIR ? 2 : 1); ++g) {
      float t = 0.f;
#pragma unroll
      for (int q = 0; q < KQ; ++q) t += red[((((q * WPG + wslot) * 2 + (PAIR ? g : st)) * MT + mt) * 4 + r) * 64 + ln];
      sum[g] = t;
    }
#pragma unroll
    for (int g = 0; g < (PAIR ? 2 : 1); ++g) sum[g] = Fmt::finish(sum[g], sc[0]);   // no format's finish uses the per-channel part
    if (PAIR) {
      gemm_put_pair<Fmt>(a.epi, a.mat[0], m, n, N, sum[0], sum[1]);
    } else {
      gemm_put<Fmt>(a.epi, mat, m, n, N, sum[0]);
    }
  }
}

// Second half of a K split: adds the slices' fp32 sums of one matrix and applies what the one-kernel form
// applies to its sum (the format's scale, bias, activation, epilogue).  V: channels of a thread (four where they divide: 16 bytes
// of every slice).
template <class Fmt, int V>
__global__ __launch_bounds__(256) void splitk_finish_kernel(GemmArgs a) {
  const GemmMat& mat = a.mat[0];
  const int N = mat.N;
  const size_t total = (size_t)a.M * N;
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * V;
  if (i >= total) return;
  const int m = (int)(i / N), n = (int)(i % N);
  if constexpr (V == 4) {
    f32x4 t = {0.f, 0.f, 0.f, 0.f};
    for (int sl = 0; sl < a.ksplit; ++sl) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(a.part + (size_t)sl * total + i);
#pragma unroll
      for (int r = 0; r < 4; ++r) t[r] += v[r];
    }
    if constexpr (Fmt::kWide) {
      wide_put4(mat, m, n, t);
    } else {
      f16x4 y;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        f16 y0 = (f16)Fmt::finish(t[r], Fmt::load_scale(mat.scale, a.x_scale, n + r, N));
        if (mat.bias) y0 = y0 + mat.bias[n + r];
        y[r] = apply_epilogue(a.epi, apply_act(mat.act, y0), m, n + r, N);
      }
      *reinterpret_cast<f16x4*>(mat.Y + i) = y;
    }
  } else {
    float t = 0.f;
    for (int sl = 0; sl < a.ksplit; ++sl) t += a.part[(size_t)sl * total + i];
    gemm_put<Fmt>(a.epi, mat, m, n, N, Fmt::finish(t, Fmt::load_scale(mat.scale, a.x_scale, n, N)));
  }
}

// The same with the norm of the finished rows behind it, a row a workgroup: the rows' sums are read once, and the norm's launch and its reading of
// the rows are gone.  What bounds it at few rows is the chain of a row (32 rows of 4096, four slices, residual, gate and three mixes: 9.6 -> 5.7 us), at many the
// bytes (1000 rows, two slices: 17.1 -> 11.0).  Every operation is that of the two kernels, in their order.
template <class Fmt, int VECS>
struct FinishedRow {
  const GemmArgs& a;
  size_t total, at;                               // numbers of a slice, and the row's first
  typename Fmt::Scale scale;
  f32x4 sums[VECS][GEMM_MAX_KSPLIT][2];
  f16x8 add[VECS][4];                             // bias of the weight, of the epilogue, factor, residual
  // (Loads without a branch round them, where paths meet the compiler waits for what is in flight: a slice that there is not reads the last one
  // again, what is not added the old result.)
  __device__ __forceinline__ void request(int i, int c) {
    const size_t n = (size_t)c * 8;
#pragma unroll
    for (int sl = 0; sl < GEMM_MAX_KSPLIT; ++sl) {
      const float* from = a.part + (sl < a.ksplit ? sl : a.ksplit - 1) * total + at + n;
      sums[i][sl][0] = *reinterpret_cast<const f32x4*>(from);
      sums[i][sl][1] = *reinterpret_cast<const f32x4*>(from + 4);
    }
    const f16* const old = a.mat[0].Y + at;
    const f16* const from[4] = {a.mat[0].bias ? a.mat[0].bias : old, a.epi.bias ? a.epi.bias : old, a.epi.mul ? a.epi.mul + at : old,
                                a.epi.residual ? a.epi.residual + at : old};
#pragma unroll
    for (int k = 0; k < 4; ++k) add[i][k] = *reinterpret_cast<const f16x8*>(from[k] + n);
  }
  __device__ __forceinline__ f16x8 value(int i) const {
    const GemmMat& mat = a.mat[0];
    f16x8 out;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float t = 0.f;
#pragma unroll
      for (int sl = 0; sl < GEMM_MAX_KSPLIT; ++sl)
        if (sl < a.ksplit) t += sums[i][sl][e >> 2][e & 3];
      f16 y = (f16)Fmt::finish(t, scale);
      if (mat.bias) y = y + add[i][0][e];
      if (a.epi.bias) y = y + add[i][1][e];
      if (a.epi.mul) y = y * add[i][2][e];
      if (a.epi.residual) y = y + add[i][3][e];
      if (a.epi.post_scale != 0.0f) y = y * (f16)a.epi.post_scale;
      out[e] = y;
    }
    return out;
  }
  __device__ __forceinline__ void keep(int c, f16x8 v) const { *reinterpret_cast<f16x8*>(a.mat[0].Y + at + (size_t)c * 8) = v; }
};

template <class Fmt, int MODE, bool MIX, int VECS>
__global__ __launch_bounds__(NORM_THREADS) void splitk_finish_norm_kernel(GemmArgs a, NormArgs norm, NormMix mix) {
  const int N = a.mat[0].N;
  // (no format's finish uses the per-channel part of its scale)
  FinishedRow<Fmt, VECS> row{a, (size_t)a.M * N, (size_t)blockIdx.x * N, Fmt::load_scale(a.mat[0].scale, a.x_scale, 0, 1)};
  norm_row<MODE, MIX, VECS>(norm, mix, blockIdx.x, row);
}

template <class Fmt, int VECS>
static void launch_finish_norm(const GemmArgs& a, const FinishNorm& t, hipStream_t s) {
  if (t.mode == 0) hipLaunchKernelGGL((splitk_finish_norm_kernel<Fmt, 0, false, VECS>), dim3(a.M), dim3(NORM_THREADS), 0, s, a, t.norm, t.mix);
  else if (t.shifted) hipLaunchKernelGGL((splitk_finish_norm_kernel<Fmt, 2, true, VECS>), dim3(a.M), dim3(NORM_THREADS), 0, s, a, t.norm, t.mix);
  else hipLaunchKernelGGL((splitk_finish_norm_kernel<Fmt, 2, false, VECS>), dim3(a.M), dim3(NORM_THREADS), 0, s, a, t.norm, t.mix);
}

static inline bool finish_norm_fits(const GemmArgs& a) {
  const GemmMat& mat = a.mat[0];
  const FinishNorm* t = a.then;
  const void* whole[] = {mat.Y, mat.bias, a.epi.bias, a.epi.mul, a.epi.residual};
  for (const void* p : whole)
    if (p && !pta_aligned(p, 16)) return false;
  // (no activation: a row's sixteen of each kind are more instructions than the rest of the kernel)
  if (t->norm.cols != mat.N || a.epi.out_fp8_scale || mat.act != PTA_ACT_NONE || a.epi.act != PTA_ACT_NONE || t->mode == 1) return false;
  return true;
}

template <class Fmt>
static bool launch_splitk_finish_norm(const GemmArgs& a, hipStream_t s) {
  const GemmMat& mat = a.mat[0];
  FinishNorm* t = a.then;
  if (!finish_norm_fits(a) || a.ksplit > GEMM_MAX_KSPLIT) return false;
  // (as few pieces of a thread as the row needs: what a row is made of stays in registers)
  if (mat.N <= 8 * NORM_THREADS) launch_finish_norm<Fmt, 1>(a, *t, s);
  else if (mat.N <= 16 * NORM_THREADS) launch_finish_norm<Fmt, 2>(a, *t, s);
  else launch_finish_norm<Fmt, 4>(a, *t, s);
  return t->done = true;
}

template <class Fmt>
static void launch_splitk_finish(const GemmArgs& a, hipStream_t s) {
  gemm_slices_taken = a.ksplit;
  const size_t total = (size_t)a.M * a.mat[0].N;
  if constexpr (!Fmt::kWide) {
    if (a.then && launch_splitk_finish_norm<Fmt>(a, s)) return;
  }
  // (four channels of a row at once where no four cross its end and Y's vectors are whole)
  if (a.mat[0].N % 4 == 0 && (Fmt::kWide || pta_aligned(a.mat[0].Y, 8)))
    hipLaunchKernelGGL((splitk_finish_kernel<Fmt, 4>), dim3((unsigned)((total / 4 + 255) / 256)), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((splitk_finish_kernel<Fmt, 1>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, a);
}

template <class Fmt, int MT, int KQ, bool PAIR, int NWV = TILE_WAVES>
static int launch_gemm_tile(const GemmArgs& a, int total_nb, hipStream_t s, const char* name) {
  static bool ready = false;
  constexpr int WPG = NWV / KQ;
  const size_t stage = (size_t)KQ * 2 * MT * 16 * TILE_XSTRIDE * 2;
  const size_t redb = (size_t)NWV * 2 * MT * 256 * 4;
  const size_t smem = stage > redb ? stage : redb;
  static_assert((size_t)KQ * 2 * MT * 16 * TILE_XSTRIDE * 2 <= 160 * 1024, "staging beyond the LDS of a compute unit");
  if (!ready) {
    PTA_REQUIRE(hipFuncSetAttribute((const void*)gemm_tile_kernel<Fmt, MT, KQ, PAIR, NWV>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) == hipSuccess,
                "%s: cannot reserve %zu bytes of LDS", name, smem);
    ready = true;
  }
  const int per_wg = PAIR ? WPG : 2 * WPG;
  gemm_kernel_taken = "gemm_tile_kernel";
  hipLaunchKernelGGL((gemm_tile_kernel<Fmt, MT, KQ, PAIR, NWV>), dim3(total_nb / per_wg), dim3(NWV * 64), smem, s, a);
  return PTA_OK;
}

// a pointer that is the same in every lane, in scalar registers
__device__ __forceinline__ const unsigned char* uniform_pointer(const unsigned char* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return reinterpret_cast<const unsigned char*>((uint64_t)hi << 32 | lo);
}

// ------------------------------------------------------------------------------------------
// Variant for 5 rows and more (own_takes_few_rows, dispatch_gemv, dispatch_many_rows) and few workgroups: each wave multiplies feature
// tiles of its own.
// A workgroup of 8 waves owns NB blocks of 16 channels (of one matrix; for a SwiGLU pair of both) and MT * 16 rows (all of up to
// 64, else a row block); its wave w takes
// the feature tiles w, w + 8, ... of its slice of K.  A wave's rows are loaded straight into LDS: the loads take
// 256 bytes of 4 rows each (in the matrix unit's operand order, 64 bytes of 16 rows, the same bytes take twice as long), the LDS
// area belongs to the wave alone and is read in operand order, so that nothing in the loop waits for another wave, and the rows
// and weights of the next tile are in flight (16 KiB and NB KiB a wave at 64 rows) while one is multiplied.  The waves' sums meet
// in LDS at the end.
// What bounds it is the rows: every workgroup reads all of them, and a compute unit gets 112 GB/s out of its L2 when all read
// (4.6 us for 64 rows of 4096 features).  Parts of a launch of 64 rows, 4096 x 11008 INT4 (15.5 us before the end's arguments were
// read ahead, 14.2 with it, weights from the last cache; 15.5 from HBM): 3 us an empty one, 4.1 the rows, 2 the weights, 1 products and decoding, 2 to 3 the end.
// Before (gemm_tile_kernel, whose waves wait for one another at every step): 21.8 us.  16 requests in flight a wave are enough;
// twice as many at 32 rows were slower by 0.6 us.
// ------------------------------------------------------------------------------------------
constexpr int OWN_WAVES = 8;
// weight streams of a workgroup that the registers hold (F152's decoding takes more of them), and channel blocks
template <class Fmt> struct OwnStreams { static constexpr int cap = Fmt::kVec == 4 ? 3 : 4; static constexpr bool long_decode = false; };
template <class Fmt, bool PAIR> constexpr int own_cap(int mt) { return (OwnStreams<Fmt>::cap + (Fmt::kVec == 1 && mt <= 2 ? 2 : 0)) / (PAIR ? 2 : 1); }
constexpr int own_ahead(int mt) { return mt <= 1 ? 2 : 1; }
// tiles of weights in flight or in use: a tile of 16 rows takes less time than its weights' way from memory (13696 x 4096, 8 rows: F143
// 17.4 -> 14.9 us, INT4 12.3 -> 10.9; at 32 rows no gain)
constexpr int own_depth(int mt, int vectors) { return mt == 1 && vectors <= 4 ? 4 : 2; }

template <class Fmt, int MT, int NB, bool PAIR>
__global__ __launch_bounds__(OWN_WAVES * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_own_kernel(GemmArgs a, int group0, int groups) {
  constexpr int NACC = PAIR ? 2 : 1, NS = NB * NACC;       // weight streams
  constexpr int KV = Fmt::kVec;
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = a.K;
  // Grid: 8 groups of channels (of the launch's, from group0 on), the row blocks, the slices' groups by eights.  A group's row blocks are multiples of eight apart: on one
  // XCD, whose L2 has its weights for all.  (One flat index, divided here, cost 1.5 us a launch.)
  const int row_block = blockIdx.y, eights = (groups + 7) / 8;
  int slice = 0, group = blockIdx.z;
  while (group >= eights) group -= eights, ++slice;
  group = group * 8 + blockIdx.x;
  if (group >= groups) return;
  group += group0;
  const int row0 = row_block * (MT * 16), M = a.M - row0 < MT * 16 ? a.M - row0 : MT * 16;
  int mi = 0;
  if (!PAIR) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int here = ((a.mat[i].N + 15) / 16 + NB - 1) / NB;
      if (i + 1 < a.count && mi == i && group >= here) { group -= here; mi = i + 1; }
    }
  }
  const GemmMat& mat = a.mat[mi];
  const int N = mat.N, blocks = (N + 15) / 16;
  const int nsl = a.ksplit > 1 ? a.ksplit : 1;
  const int per_slice = (a.KT + nsl - 1) / nsl;
  const int kt_first = slice * per_slice;
  const int kt_end = kt_first + per_slice < a.KT ? kt_first + per_slice : a.KT;

  typename Fmt::Scale sc[NS];
  __amdgpu_buffer_rsrc_t wr[NS];
  const int block_bytes = a.KT * KV * 1024;
#pragma unroll
  for (int st = 0; st < NS; ++st) {
    const GemmMat& m = PAIR ? a.mat[st & 1] : mat;
    int nb = group * NB + st / NACC;
    nb = nb < blocks ? nb : blocks - 1;                    // (blocks past the last one: multiplied, never stored)
    sc[st] = Fmt::load_scale(m.scale, a.x_scale, nb * 16 + (lane & 15), m.N);
    const unsigned char* from = uniform_pointer(reinterpret_cast<const unsigned char*>(m.tiled) + (size_t)nb * block_bytes);
    wr[st] = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(from), 0, block_bytes, 0x00020000);
  }
  // rows past the last one lie past the buffer's end and read as zeros
  const unsigned char* X = uniform_pointer(reinterpret_cast<const unsigned char*>((mat.X ? mat.X : a.X) + (size_t)row0 * K));
  const int row_bytes = K * 2, x_bytes = M * row_bytes;
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(X), 0, x_bytes, 0x00020000);
  const int tiles = (kt_end - kt_first - wave + OWN_WAVES - 1) / OWN_WAVES;
  auto tile = [&](int i) { return i < tiles ? kt_first + wave + OWN_WAVES * i : kt_end; };
  // 16 rows of a tile lie in LDS with 256 bytes a row, the 16-byte vector c of row r at place c ^ r: the reads, one vector of 16
  // rows, meet in no bank.  Lane l of load j fills place l % 16 of row j * 4 + l / 16.
  constexpr int AHEAD = own_ahead(MT), RING = AHEAD * MT;   // tiles, and row groups of tiles, that the area holds
  unsigned char* const area = smem + wave * (RING * 4096);
  int xlane[4], xfeature[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = j * 4 + (lane >> 4), c = (lane & 15) ^ r;
    xlane[j] = r * row_bytes + c * 16;
    xfeature[j] = c * 8;
  }
  // requests for tiles and features past the last one lie past the buffers' ends: they read as zeros from nowhere, and the loop
  // has no branch round them
  auto x_at = [&](int kt, int (&at)[4]) {
    const int left = kt < kt_end ? K - kt * 128 : 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) at[j] = xfeature[j] < left ? xlane[j] : x_bytes;
  };
  int x_tile, x_lane[4];                                   // the tile whose rows are requested
  auto next_x = [&](int kt) { x_tile = kt; x_at(kt, x_lane); };
  auto fetch_x = [&](int mt, int place) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (__attribute__((address_space(3))) void*)(area + place * 4096 + j * 1024), 16,
                                               x_lane[j] + mt * 16 * row_bytes, x_tile * 256, 0, 0);
  };
  auto fetch_w = [&](int kt, u32x4 (&to)[NS][KV]) {
    const int at = kt < kt_end ? lane * 16 : block_bytes;
#pragma unroll
    for (int st = 0; st < NS; ++st)
#pragma unroll
      for (int v = 0; v < KV; ++v) to[st][v] = __builtin_amdgcn_raw_buffer_load_b128(wr[st], at, (kt * KV + v) * 1024, 2);
  };

  f32x4 acc[NS][MT];
#pragma unroll
  for (int st = 0; st < NS; ++st)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[st][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Requests are made in the order x(0), w(n), x(1), w(n + 1), ...: this many follow those of a row group when it is waited for
  constexpr int BEHIND = 4 * (RING - 1) + AHEAD * NS * KV;
  static_assert(BEHIND < 64, "the counter of requests");
  constexpr int DEPTH = own_depth(MT, NS * KV);
  u32x4 w[DEPTH][NS][KV];
  f16x8 xb[2][4];
  auto read_x = [&](int place, f16x8 (&to)[4], auto behind) {
    constexpr int N = decltype(behind)::value;
    __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | (N >> 4) << 14);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 4; ++j) to[j] = *reinterpret_cast<const f16x8*>(area + place * 4096 + (lane & 15) * 256 + (((j * 4 + (lane >> 4)) ^ (lane & 15)) * 16));
  };
  // tile i: TURN is i modulo what makes the places in the area and the buffers of w and xb come round again; LAST: how many of the
  // last tiles, which request no more weights, came before it (-1: it is none of them)
  auto step = [&](int i, auto turn, auto last) {
    constexpr int TURN = decltype(turn)::value, LAST = decltype(last)::value;
    constexpr int SHORT = LAST > AHEAD ? AHEAD : LAST < 0 ? 0 : LAST, SHORT_NEXT = LAST + 1 > AHEAD ? AHEAD : LAST + 1;
    f16x8 av[NS][4];
#pragma unroll
    for (int st = 0; st < NS; ++st)
#pragma unroll
      for (int j = 0; j < 4; ++j) av[st][j] = Fmt::a_operand(w[TURN][st], j, sc[st]);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      constexpr int Q0 = TURN * MT;
      const int q = Q0 + mt, place = (q + 1) % RING;        // the next row group: read while this one is multiplied, then requested anew
      if (mt == MT - 1) {
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (LAST < 0) fetch_w(tile(i + DEPTH), w[TURN]);
        next_x(tile(i + 1 + AHEAD));
        __builtin_amdgcn_sched_barrier(0);
      }
      if (mt == MT - 1) read_x(place, xb[(q + 1) & 1], std::integral_constant<int, BEHIND - SHORT_NEXT * NS * KV>{});
      else read_x(place, xb[(q + 1) & 1], std::integral_constant<int, BEHIND - SHORT * NS * KV>{});
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int st = 0; st < NS; ++st) acc[st][mt] = Fmt::mma(av[st][j], xb[q & 1][j], acc[st][mt]);
      __builtin_amdgcn_s_waitcnt(0xc07f);                  // lgkmcnt(0): the operands are out of LDS, their place is free
      __builtin_amdgcn_sched_barrier(0);
      fetch_x((mt + 1) % MT, place);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int t = 0; t < DEPTH - AHEAD; ++t) fetch_w(tile(t), w[t]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int t = 0; t < AHEAD; ++t) {
    next_x(tile(t));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) fetch_x(mt, t * MT + mt);
    __builtin_amdgcn_sched_barrier(0);
    fetch_w(tile(DEPTH - AHEAD + t), w[DEPTH - AHEAD + t]);
    __builtin_amdgcn_sched_barrier(0);
  }
  next_x(tile(AHEAD));
  read_x(0, xb[0], std::integral_constant<int, BEHIND>{});
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_sched_barrier(0);
  fetch_x(0, 0);
  __builtin_amdgcn_sched_barrier(0);
  // What the end needs of the arguments is read while the first rows are on their way: each line of them is a round trip to memory
  // of its own otherwise, one after another behind the products.
  GemmMat out = mat;
  GemmEpilogue epi = a.epi;
  read_end<Fmt, PAIR>(out, epi);
  // (in pairs or fours, with no way out between them: where paths meet, the compiler waits for what is in flight on either)
  using std::integral_constant;
  int i = 0;
  for (; i + DEPTH - 1 < tiles; i += DEPTH) {
    step(i, integral_constant<int, 0>{}, integral_constant<int, -1>{});
    step(i + 1, integral_constant<int, 1>{}, integral_constant<int, -1>{});
    if constexpr (DEPTH == 4) {
      step(i + 2, integral_constant<int, 2>{}, integral_constant<int, -1>{});
      step(i + 3, integral_constant<int, 3>{}, integral_constant<int, -1>{});
    }
  }
  if (i < tiles) {
    step(i, integral_constant<int, 0>{}, integral_constant<int, 0>{});
    if constexpr (DEPTH == 4) {
      if (i + 1 < tiles) {
        step(i + 1, integral_constant<int, 1>{}, integral_constant<int, 1>{});
        if (i + 2 < tiles) step(i + 2, integral_constant<int, 2>{}, integral_constant<int, 2>{});
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);                      // vmcnt(0): nothing is on its way into LDS any more

  __syncthreads();
  f32x4* red = reinterpret_cast<f32x4*>(smem);             // [OWN_WAVES][NS][MT][64]
#pragma unroll
  for (int st = 0; st < NS; ++st)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) red[((wave * NS + st) * MT + mt) * 64 + lane] = acc[st][mt];
  __syncthreads();
  constexpr int OUTS = NB * MT * 64, ITEMS = (OUTS + OWN_WAVES * 64 - 1) / (OWN_WAVES * 64);      // four channels of a row each
  f32x4 sums[ITEMS][NACC];
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    const int o = it * (OWN_WAVES * 64) + threadIdx.x, b = o / (MT * 64), at = o % (MT * 64);
    if (OUTS % (OWN_WAVES * 64) == 0 || o < OUTS) {
#pragma unroll
      for (int g = 0; g < NACC; ++g) {
        f32x4 t = red[(b * NACC + g) * MT * 64 + at];
#pragma unroll
        for (int v = 1; v < OWN_WAVES; ++v) {
          const f32x4 p = red[(v * NS + b * NACC + g) * MT * 64 + at];
#pragma unroll
          for (int r = 0; r < 4; ++r) t[r] += p[r];
        }
        sums[it][g] = t;
      }
    }
  }
  const bool vectors = (N & 3) == 0 && ((reinterpret_cast<uintptr_t>(out.Y) | reinterpret_cast<uintptr_t>(epi.residual)) & 7) == 0;
  const bool direct = !out.bias && out.act == PTA_ACT_NONE && !epi.bias && epi.act == PTA_ACT_NONE && !epi.mul &&
                      epi.post_scale == 0.0f && !epi.out_fp8_scale;
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    const int o = it * (OWN_WAVES * 64) + threadIdx.x, b = o / (MT * 64), at = o % (MT * 64);
    const int m = row0 + (at >> 6) * 16 + (at & 15), n = (group * NB + b) * 16 + ((at >> 4) & 3) * 4;
    if (o >= OUTS || m >= a.M || n >= N) continue;
    const f32x4 (&t)[NACC] = sums[it];
    if (!PAIR && nsl > 1) {                // a slice of a K split: the raw fp32 sums; the finishing kernel does the rest
      float* p = a.part + ((size_t)slice * a.M + m) * N + n;
      if ((N & 3) == 0) {
        *reinterpret_cast<f32x4*>(p) = t[0];
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < N) p[r] = t[0][r];
      }
      continue;
    }
    if constexpr (Fmt::kWide) {
      if constexpr (PAIR) wide_put_pair4(out, m, n, t[0], t[NACC - 1]);
      else wide_put4(out, m, n, t[0]);
    } else {
      f16* y = out.Y + (size_t)m * N + n;
      f16x4 v;
      if (!PAIR && direct) {               // nothing but the residual stream to add
        const f16* from = epi.residual + (size_t)m * N + n;
        f16x4 res = {0, 0, 0, 0};
        if (epi.residual && vectors) res = *reinterpret_cast<const f16x4*>(from);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (epi.residual && !vectors && n + r < N) res[r] = from[r];
          v[r] = (f16)Fmt::finish(t[0][r], sc[0]);                   // no format's finish uses the per-channel part
          if (epi.residual) v[r] = v[r] + res[r];
          if (!vectors && n + r < N) y[r] = v[r];
        }
        if (vectors) *reinterpret_cast<f16x4*>(y) = v;
        continue;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (n + r >= N) continue;
        if constexpr (PAIR) {
          v[r] = swiglu_out(epi, (f16)Fmt::finish(t[0][r], sc[0]), (f16)Fmt::finish(t[NACC - 1][r], sc[1]));
        } else {
          f16 y0 = (f16)Fmt::finish(t[0][r], sc[0]);
          if (out.bias) y0 = y0 + out.bias[n + r];
          v[r] = apply_epilogue(epi, apply_act(out.act, y0), m, n + r, N);
        }
        if (!vectors) y[r] = v[r];
      }
      if (vectors) *reinterpret_cast<f16x4*>(y) = v;
    }
  }
}

static inline int own_groups(const GemmArgs& a, int nb, bool pair) {
  int groups = 0;
  for (int i = 0; i < (pair ? 1 : a.count); ++i) groups += ((a.mat[i].N + 15) / 16 + nb - 1) / nb;
  return groups;
}

template <class Fmt, int MT, int NB, bool PAIR>
static int launch_gemm_own(const GemmArgs& a, hipStream_t s, const char* name) {
  static bool ready = false;
  constexpr int NS = NB * (PAIR ? 2 : 1), STAGE = 4 * own_ahead(MT);
  const size_t smem = (size_t)OWN_WAVES * MT * 1024 * (NS > STAGE ? NS : STAGE);
  if (!ready) {
    PTA_REQUIRE(hipFuncSetAttribute((const void*)gemm_own_kernel<Fmt, MT, NB, PAIR>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)smem) == hipSuccess, "%s: cannot reserve %zu bytes of LDS", name, smem);
    ready = true;
  }
  const int nsl = a.ksplit > 1 ? a.ksplit : 1;
  const int groups = own_groups(a, NB, PAIR), row_blocks = (a.M + MT * 16 - 1) / (MT * 16);
  gemm_kernel_taken = "gemm_own_kernel";
  const int most = 65535 / nsl * 8;                // (as many groups as a grid's z holds)
  for (int g = 0; g < groups; g += most) {
    const int here = groups - g < most ? groups - g : most;
    hipLaunchKernelGGL((gemm_own_kernel<Fmt, MT, NB, PAIR>), dim3(8, row_blocks, (here + 7) / 8 * nsl), dim3(OWN_WAVES * 64), smem, s, a, g, here);
  }
  if (nsl > 1) launch_splitk_finish<Fmt>(a, s);
  return PTA_OK;
}

// ------------------------------------------------------------------------------------------
// Variant for many rows (prompt passes): the activation fragments live in registers, the weights go through
// LDS decoded.  A workgroup of 8 waves owns 8 weight streams of 16 channels (8 channel blocks of one matrix,
// or the gate and up weights of 4 blocks) and 8 * RG * 16 rows.  Per 128-feature tile, wave w
//   - fetches the tile of stream w, decodes it ONCE into the four fp16 A operands of its MFMA steps and puts
//     them into LDS (double-buffered, one barrier per tile) - every weight is decoded once per workgroup, not
//     once per wave and row group: with the decode in the product loop a wave spends 13 VALU instructions per
//     step for RG MFMAs and the kernel is bound by those (measured: 262 TFLOP/s at 256 rows);
//   - holds the B operands of ITS RG row groups in registers (fetched with whole-row loads, turned into
//     fragment order through a strip of LDS of its own) and multiplies them with every stream's operands.
// ------------------------------------------------------------------------------------------
constexpr int ROWS_WAVES = 8;
constexpr int ROWS_CB = 8;                  // streams per workgroup: one per wave
constexpr int ROWS_XSTRIDE = 128 + 8;
constexpr int ROWS_AVEC = ROWS_CB * 4 * 64; // A operands (16 bytes each) of one feature tile: [stream][step][lane]

// Which rows a workgroup takes: all of X and Y in order; or those of a tile from a list, each tile with weights of its own
// (the same matrices, `weight_bytes` further per expert): entry a of `order` is read from row a / x_div of X and goes to row a of Y.
struct AllRows { static constexpr bool kListed = false; };
struct ListedRows {
  static constexpr bool kListed = true;
  const int32_t* n_tiles;
  const int32_t* tiles;        // [..][4]: expert, first entry, entries
  const int32_t* order;
  size_t weight_bytes;
  int x_div;
};

// (two waves per SIMD: the whole register file of 256 per lane is this kernel's to use)
template <class Fmt, int RG, bool PAIR, class Rows = AllRows>
__global__ __launch_bounds__(ROWS_WAVES * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_rows_kernel(GemmArgs a, int groups, int row_blocks, Rows rows) {
  constexpr int KV = Fmt::kVec;
  constexpr int XROWS = RG * 16;
  static_assert(ROWS_CB == ROWS_WAVES, "wave w decodes stream w");
  extern __shared__ __align__(16) unsigned char smem[];
  f16x8* abuf = reinterpret_cast<f16x8*>(smem);                                          // [2][ROWS_AVEC]
  f16* xbuf = reinterpret_cast<f16*>(smem + (size_t)2 * ROWS_AVEC * 16);                 // [waves][XROWS][ROWS_XSTRIDE]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int K = a.K;
  // Workgroups are dealt to the eight XCDs (each with an L2 of its own) in turn: workgroup id of the launch takes
  // tile (id % 8) * per + id / 8 of the list (row block, channel group), row block slowest - so an XCD works through
  // a contiguous stretch of the list, i.e. on one row block at a time, whose activations stay in its L2.
  int per = (int)gridDim.x / 8;
  if constexpr (Rows::kListed) {            // (the launch has room for the most tiles there can be)
    row_blocks = *rows.n_tiles;
    per = (groups * row_blocks + 7) / 8;
    if ((int)blockIdx.x / 8 >= per) return;
  }
  const int tile = ((int)blockIdx.x % 8) * per + (int)blockIdx.x / 8;
  if (tile >= groups * row_blocks) return;
  const int group = tile % groups, row_block = tile / groups;
  int M = a.M;
  const int32_t* order = nullptr;
  size_t weight_at = 0;
  if constexpr (Rows::kListed) {
    const int32_t* t = rows.tiles + row_block * 4;
    weight_at = (size_t)t[0] * rows.weight_bytes;
    order = rows.order + t[1];
    M = t[2];
  }
  const int nsl = a.ksplit > 1 ? a.ksplit : 1;
  const int per_slice = (a.KT + nsl - 1) / nsl;
  const int kt_first = (int)blockIdx.y * per_slice;
  const int kt_end = kt_first + per_slice < a.KT ? kt_first + per_slice : a.KT;
  const int steps = kt_end - kt_first;

  int mi = 0;
  const int first_blk = group * (PAIR ? ROWS_CB / 2 : ROWS_CB);
  if (!PAIR) {
#pragma unroll
    for (int i = 1; i < 4; ++i)
      if (i < a.count && first_blk >= a.mat[i].nb_begin) mi = i;
  }
  // stream st: its matrix and channel block
  auto stream_mat = [&](int st) -> const GemmMat& { return a.mat[PAIR ? (st < ROWS_CB / 2 ? 0 : 1) : mi]; };
  auto stream_blk = [&](int st) { return PAIR ? first_blk + st % (ROWS_CB / 2) : first_blk - a.mat[mi].nb_begin + st; };
  const GemmMat& own = stream_mat(wave);
  int own_blk = stream_blk(wave);
  if constexpr (Rows::kListed) own_blk = own_blk < own.N / 16 ? own_blk : own.N / 16 - 1;      // (channels past N go nowhere)
  const typename Fmt::Scale own_sc = Fmt::load_scale(own.scale, a.x_scale, own_blk * 16 + (lane & 15), own.N);
  const u32x4* own_w = reinterpret_cast<const u32x4*>(reinterpret_cast<const unsigned char*>(own.tiled) + weight_at) +
                       (size_t)own_blk * a.KT * (KV * 64) + lane;
  const f16* X = a.mat[mi].X ? a.mat[mi].X : a.X;
  const int row0 = ((Rows::kListed ? 0 : row_block) * ROWS_WAVES + wave) * XROWS;      // first row of this wave
  int listed[RG * 4];                                            // (the rows of X this lane fetches)
  if constexpr (Rows::kListed) {
#pragma unroll
    for (int j = 0; j < RG * 4; ++j) {
      const int row = row0 + j * 4 + (lane >> 4);
      listed[j] = row < M ? order[row] / rows.x_div : -1;
    }
  }
  auto result_row = [&](int m) {
    if constexpr (Rows::kListed) return order[m];
    else return m;
  };
  f16* xw = xbuf + (size_t)wave * XROWS * ROWS_XSTRIDE;

  auto fetch_w = [&](int kt, u32x4 (&wv)[KV]) {
#pragma unroll
    for (int v = 0; v < KV; ++v) wv[v] = __builtin_nontemporal_load(own_w + ((size_t)kt * KV + v) * 64);
  };
  auto decode_w = [&](f16x8* buf, const u32x4 (&wv)[KV]) {
#pragma unroll
    for (int m = 0; m < 4; ++m) buf[(wave * 4 + m) * 64 + lane] = Fmt::a_operand(wv, m, own_sc);
  };
  // whole-row loads: instruction j covers rows 4 j .. 4 j + 3 of the wave, 256 bytes each
  auto fetch_x = [&](int kt, u32x4 (&xr)[RG * 4]) {
#pragma unroll
    for (int j = 0; j < RG * 4; ++j) {
      const int row = Rows::kListed ? listed[j] : row0 + j * 4 + (lane >> 4), k = kt * 128 + (lane & 15) * 8;
      const bool there = Rows::kListed ? row >= 0 : row < M;
      xr[j] = (there && k < K) ? *reinterpret_cast<const u32x4*>(X + (size_t)row * K + k) : u32x4{0, 0, 0, 0};
    }
  };
  // through the wave's own strip of LDS into fragment order (a wave's LDS accesses complete in order)
  auto to_fragments = [&](const u32x4 (&xr)[RG * 4], f16x8 (&xf)[RG][4]) {
#pragma unroll
    for (int j = 0; j < RG * 4; ++j)
      *reinterpret_cast<u32x4*>(xw + (j * 4 + (lane >> 4)) * ROWS_XSTRIDE + (lane & 15) * 8) = xr[j];
#pragma unroll
    for (int rg = 0; rg < RG; ++rg)
#pragma unroll
      for (int m = 0; m < 4; ++m)
        xf[rg][m] = *reinterpret_cast<const f16x8*>(xw + (rg * 16 + (lane & 15)) * ROWS_XSTRIDE + m * 32 + (lane >> 4) * 8);
  };

  f32x4 acc[RG][ROWS_CB];
#pragma unroll
  for (int rg = 0; rg < RG; ++rg)
#pragma unroll
    for (int st = 0; st < ROWS_CB; ++st) acc[rg][st] = f32x4{0.f, 0.f, 0.f, 0.f};

  u32x4 wv[KV], xr[RG * 4];
  f16x8 xf[RG][4];
  if (steps > 0) {
    fetch_w(kt_first, wv);
    fetch_x(kt_first, xr);
    decode_w(abuf, wv);
    to_fragments(xr, xf);
  }
  __syncthreads();
  for (int i = 0; i < steps; ++i) {
    const bool more = i + 1 < steps;
    if (more) { fetch_w(kt_first + i + 1, wv); fetch_x(kt_first + i + 1, xr); }
    const f16x8* cur = abuf + (size_t)(i & 1) * ROWS_AVEC;
    // the operands of stream st + 1 are read while stream st is multiplied (left to itself the compiler reads two
    // operands, waits, multiplies, and the LDS latency shows after every fourth MFMA)
    f16x8 av[4], avn[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) av[m] = cur[m * 64 + lane];
#pragma unroll
    for (int st = 0; st < ROWS_CB; ++st) {
      if (st + 1 < ROWS_CB) {
#pragma unroll
        for (int m = 0; m < 4; ++m) avn[m] = cur[((st + 1) * 4 + m) * 64 + lane];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) acc[rg][st] = Fmt::mma(av[m], xf[rg][m], acc[rg][st]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < 4; ++m) av[m] = avn[m];
    }
    if (more) {
      decode_w(abuf + (size_t)((i + 1) & 1) * ROWS_AVEC, wv);
      to_fragments(xr, xf);
    }
    __syncthreads();
  }

  // Lane l holds channels (l / 16) * 4 + r, r = 0..3, of row l % 16 of each row group, for every stream.  The sums
  // go to the wave's strip of LDS first (the operand buffers are free after the last barrier) and one copy of the
  // epilogue walks over them: unrolled RG * 8 * 4 times the epilogue is too large to unroll, and an accumulator
  // array that is indexed by a loop counter lives in scratch memory - for the whole kernel.
  f32x4* sums = reinterpret_cast<f32x4*>(smem) + (size_t)wave * (RG * ROWS_CB * 64);
#pragma unroll
  for (int rg = 0; rg < RG; ++rg)
#pragma unroll
    for (int st = 0; st < ROWS_CB; ++st) sums[(rg * ROWS_CB + st) * 64 + lane] = acc[rg][st];
  if constexpr (PAIR) {
    const GemmMat& mat = a.mat[0];
    const typename Fmt::Scale sg = Fmt::load_scale(a.mat[0].scale, a.x_scale, 0, 1), su = Fmt::load_scale(a.mat[1].scale, a.x_scale, 0, 1);
#pragma unroll 1
    for (int i = 0; i < RG * ROWS_CB / 2; ++i) {
      const int rg = i / (ROWS_CB / 2), st = i % (ROWS_CB / 2);
      const int m = row0 + rg * 16 + (lane & 15);
      const f32x4 g4 = sums[(rg * ROWS_CB + st) * 64 + lane], u4 = sums[(rg * ROWS_CB + st + ROWS_CB / 2) * 64 + lane];
      if constexpr (Fmt::kWide) {
        if (m < M) wide_put_pair4(mat, result_row(m), (first_blk + st) * 16 + (lane >> 4) * 4, g4, u4);
        continue;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = (first_blk + st) * 16 + (lane >> 4) * 4 + r;
        if (m >= M || n >= mat.N) continue;
        gemm_put_pair<Fmt>(a.epi, a.mat[0], m, n, mat.N, Fmt::finish(g4[r], sg), Fmt::finish(u4[r], su));
      }
    }
  } else {
    const GemmMat& mat = a.mat[mi];
    const int N = mat.N;
    const typename Fmt::Scale s1 = Fmt::load_scale(mat.scale, a.x_scale, 0, 1);      // no format's finish uses the per-channel part
#pragma unroll 1
    for (int i = 0; i < RG * ROWS_CB; ++i) {
      const int rg = i / ROWS_CB, st = i % ROWS_CB;
      const int m = row0 + rg * 16 + (lane & 15);
      const f32x4 v4 = sums[i * 64 + lane];
      if constexpr (Fmt::kWide) {
        if (nsl == 1) {
          if (m < M) wide_put4(mat, result_row(m), stream_blk(st) * 16 + (lane >> 4) * 4, v4);
          continue;
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = stream_blk(st) * 16 + (lane >> 4) * 4 + r;
        if (m >= M || n >= N) continue;
        if (nsl > 1) { a.part[((size_t)blockIdx.y * M + m) * N + n] = v4[r]; continue; }
        gemm_put<Fmt>(a.epi, mat, m, n, N, Fmt::finish(v4[r], s1));
      }
    }
  }
}

template <class Fmt, int RG, bool PAIR, class Rows>
static int reserve_gemm_rows(size_t* smem, const char* name) {
  static bool ready = false;
  *smem = (size_t)2 * ROWS_AVEC * 16 + (size_t)ROWS_WAVES * RG * 16 * ROWS_XSTRIDE * 2;
  static_assert((size_t)2 * ROWS_AVEC * 16 + (size_t)ROWS_WAVES * RG * 16 * ROWS_XSTRIDE * 2 <= 160 * 1024, "LDS");
  if (!ready) {
    PTA_REQUIRE(hipFuncSetAttribute((const void*)gemm_rows_kernel<Fmt, RG, PAIR, Rows>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)*smem) == hipSuccess,
                "%s: cannot reserve %zu bytes of LDS", name, *smem);
    ready = true;
  }
  return PTA_OK;
}

// As launch_gemm_block_listed, where the rows lie further apart than its 32-bit offsets reach.
template <class Fmt, int RG, bool PAIR>
static int launch_gemm_listed(const GemmArgs& a, int total_nb, int max_tiles, const ListedRows& rows, hipStream_t s, const char* name) {
  size_t smem;
  const int rc = reserve_gemm_rows<Fmt, RG, PAIR, ListedRows>(&smem, name);
  if (rc) return rc;
  constexpr int per_wg = PAIR ? ROWS_CB / 2 : ROWS_CB;
  const int groups = (total_nb + per_wg - 1) / per_wg;
  gemm_kernel_taken = "gemm_rows_kernel";
  hipLaunchKernelGGL((gemm_rows_kernel<Fmt, RG, PAIR, ListedRows>), dim3((groups * max_tiles + 7) / 8 * 8), dim3(ROWS_WAVES * 64), smem, s, a,
                     groups, max_tiles, rows);
  return PTA_OK;
}

template <class Fmt, int RG, bool PAIR>
static int launch_gemm_rows(const GemmArgs& a, int total_nb, hipStream_t s, const char* name) {
  size_t smem;
  const int rc = reserve_gemm_rows<Fmt, RG, PAIR, AllRows>(&smem, name);
  if (rc) return rc;
  const int groups = total_nb / (PAIR ? ROWS_CB / 2 : ROWS_CB);
  const int row_blocks = (a.M + ROWS_WAVES * RG * 16 - 1) / (ROWS_WAVES * RG * 16);
  const int nsl = a.ksplit > 1 ? a.ksplit : 1;
  const int per = (groups * row_blocks + 7) / 8;
  gemm_kernel_taken = "gemm_rows_kernel";
  hipLaunchKernelGGL((gemm_rows_kernel<Fmt, RG, PAIR>), dim3(per * 8, nsl), dim3(ROWS_WAVES * 64), smem, s, a, groups, row_blocks, AllRows{});
  if (nsl > 1) launch_splitk_finish<Fmt>(a, s);
  return PTA_OK;
}

// a's second and fourth sixteen lanes change places with b's first and third
__device__ __forceinline__ void swap_sixteens(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// Of sums of two neighbouring channel blocks (as panel_store has them, four channels a lane) rounded to 16 bits, eight consecutive channels
// a lane: of block (lane / 16) % 2, from lane / 32 * 8 on.
template <class T4>
__device__ __forceinline__ u32x4 eight_channels(T4 first, T4 second) {
  u32x2 a = bitcast<u32x2>(first), b = bitcast<u32x2>(second);
  uint32_t a0 = a[0], a1 = a[1], b0 = b[0], b1 = b[1];
  swap_sixteens(a0, b0);
  swap_sixteens(a1, b1);
  return u32x4{a0, a1, b0, b1};
}

// swish_f16 for the tiles, bit for bit: the quotient by the hardware's reciprocal and one step of what is left of it, in half the instructions of a division
// (a reciprocal alone has another result for one gate of 65536, and that is enough for other tokens' logits some layers on).
__device__ __forceinline__ f16 tile_swish_f16(f16 x) {
  const float v = (float)x, d = 1.0f + __expf(-v), r = __builtin_amdgcn_rcpf(d), q = v * r;
  return (f16)__builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-d, q, v), r, q), d, v);
}

// The ends of a tile that most products have, straight from the registers and without a loop; false: another one (panel_store).  What bounds
// them is what they wait for: through LDS, row group by row group, each stretch of a residual, a gate or an old sum was a round trip to memory
// of its own behind the one before; here all that a tile adds is requested together.  A launch of 2048 x 4096 without its products 10.3 -> 8.2 us
// (an empty one 2.6), 2048 x 8192 11.0 -> 9.2; with them, weights from HBM: fp16, 2048 rows, 4096 x 8192 117 -> 114, 4096 x 4096 74 -> 72; bf16, 2048
// rows, 11008 x 4096 with gate and fp32 residual 215 -> 201, a pair of 4096 x 11008 341 -> 310, two of 4096 x 4096 with biases and sigmoids in turn 151.
// Not kept: sigmoid and swish of fp32 sums by the hardware's exponential and reciprocal (the pair 299, the two 143): their error is 4 to 60 units of the
// 24-bit result where the exact exponential and a division make two, and results would depend on the kernel that the number of rows selects.
template <class Fmt, int NST, int RG, bool PAIR>
__device__ __forceinline__ bool straight_store(const GemmMat& mat, const GemmEpilogue& epi, const f32x4 (&acc)[RG][NST], int blk0, int row0, int nsl,
                                               typename Fmt::Scale s0, typename Fmt::Scale s1, int M, const int32_t* order) {
  static_assert(NST == 4 && (RG % 2 == 0 || !Fmt::kWide), "tile");
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int N = mat.N, n0 = blk0 * 16;
  // A slice's sums wait for nothing, and go out as whole lines from LDS faster than a quarter of a line a lane group from here: bf16, with straight stores and
  // without, 198 rows of 4096, four slices 25.2 and 24.2 us, 166 of 5120 18.3 and 16.9, 731 of 3584, three slices 81.4 and 78.3
  if (!PAIR && nsl > 1) return false;
  const int c8 = (g & 1) * 16 + (g >> 1) * 8;               // a lane's eight channels of two blocks
  if constexpr (!Fmt::kWide) {
    if ((N & 7) || epi.out_fp8_scale || (reinterpret_cast<uintptr_t>(mat.Y) & 15)) return false;
    if constexpr (PAIR) {
      f16* y = mat.Y + (size_t)(row0 + r) * N + n0 + c8;
      const bool in = n0 + c8 < N;
#pragma unroll
      for (int rg = 0; rg < RG; ++rg) {
        f16x4 v[2];
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            v[st][e] = (f16)Fmt::finish(acc[rg][2 + st][e], s1) * tile_swish_f16((f16)Fmt::finish(acc[rg][st][e], s0));
        const u32x4 out = eight_channels(v[0], v[1]);
        if (in && row0 + rg * 16 + r < M) *reinterpret_cast<u32x4*>(y + (size_t)rg * 16 * N) = out;
      }
    } else {
      const f16* bias = mat.bias ? mat.bias : epi.bias;
      if ((mat.bias && epi.bias) || mat.act != PTA_ACT_NONE || epi.act != PTA_ACT_NONE || epi.mul || epi.post_scale != 0.0f ||
          ((reinterpret_cast<uintptr_t>(bias) | reinterpret_cast<uintptr_t>(epi.residual)) & 15))
        return false;
      const size_t at = (size_t)(row0 + r) * N + n0 + c8;
      const f16* from = epi.residual + at;
      f16x8 b[2], res[RG][2];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const bool in = n0 + p * 32 + c8 < N;
        b[p] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
        if (bias && in) b[p] = *reinterpret_cast<const f16x8*>(bias + n0 + p * 32 + c8);
        if (epi.residual) {
#pragma unroll
          for (int rg = 0; rg < RG; ++rg)
            if (in && row0 + rg * 16 + r < M) res[rg][p] = *reinterpret_cast<const f16x8*>(from + (size_t)rg * 16 * N + p * 32);
        }
      }
#pragma unroll
      for (int rg = 0; rg < RG; ++rg)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          f16x4 v[2];
#pragma unroll
          for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[st][e] = (f16)Fmt::finish(acc[rg][p * 2 + st][e], s0);
          f16x8 out = bitcast<f16x8>(eight_channels(v[0], v[1]));
          if (bias) out = out + b[p];
          if (epi.residual) out = out + res[rg][p];
          if (n0 + p * 32 + c8 < N && row0 + rg * 16 + r < M) *reinterpret_cast<f16x8*>(mat.Y + at + (size_t)rg * 16 * N + p * 32) = out;
        }
    }
  } else {
    const WideOut& w = mat.wide;
    const bool tail = !PAIR && w.tail_count && n0 + NST * 16 > w.n_main;
    if ((w.ld & 7) || (w.n_main & 7) || w.mul_f32 ||
        (tail && ((w.tail_count & 3) || ((reinterpret_cast<uintptr_t>(w.tail) | reinterpret_cast<uintptr_t>(w.tail_bias)) & 15))) ||
        ((reinterpret_cast<uintptr_t>(mat.Y) | reinterpret_cast<uintptr_t>(w.bias) | reinterpret_cast<uintptr_t>(w.mul) | (PAIR ? reinterpret_cast<uintptr_t>(w.bias2) : 0)) & 15))
      return false;
    int m[RG];
    bool on[RG];
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) {
      on[rg] = row0 + rg * 16 + r < M;
      m[rg] = on[rg] ? (order ? order[row0 + rg * 16 + r] : row0 + rg * 16 + r) : 0;
    }
    const int c4 = n0 + g * 4;
    auto channels = [&](const float* p, int c) { return p && c < w.n_main ? *reinterpret_cast<const f32x4*>(p + c) : f32x4{0.f, 0.f, 0.f, 0.f}; };
    if constexpr (PAIR) {
      if (w.out_f32 || w.mul) return false;
      f32x4 b1[2], b2[2];
#pragma unroll
      for (int st = 0; st < 2; ++st) { b1[st] = channels(w.bias, c4 + st * 16); b2[st] = channels(w.bias2, c4 + st * 16); }
      auto all = [&](auto value) {
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) {
          bf16x4 v[2];
#pragma unroll
          for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[st][e] = (bf16)value(acc[rg][st][e] + b1[st][e], acc[rg][2 + st][e] + b2[st][e]);
          const u32x4 out = eight_channels(v[0], v[1]);
          if (on[rg] && n0 + c8 < w.n_main) *reinterpret_cast<u32x4*>(reinterpret_cast<bf16*>(mat.Y) + (size_t)m[rg] * w.ld + n0 + c8) = out;
        }
      };
      const float limit = w.limit, slope = w.slope;
      if (w.clamped) all([=](float a, float b) { return clamped_glu_f32(a, b, limit, slope); });
      else all([](float a, float b) { return swiglu_f32(a, b); });
    } else {
      if (w.cap > 0.f || (w.act != PTA_ACT_NONE && (w.act != PTA_ACT_SIGMOID || w.out_f32))) return false;
      if (!w.out_f32 && (w.mul || w.accumulate)) return false;
      if (tail) {
#pragma unroll
        for (int st = 0; st < NST; ++st) {
          const int c = c4 + st * 16 - w.n_main;
          if (c < 0 || c >= w.tail_count) continue;
          f32x4 add = {0.f, 0.f, 0.f, 0.f};
          if (w.tail_bias) add = *reinterpret_cast<const f32x4*>(w.tail_bias + c);
#pragma unroll
          for (int rg = 0; rg < RG; ++rg)
            if (on[rg]) *reinterpret_cast<f32x4*>(w.tail + (size_t)m[rg] * w.tail_count + c) = acc[rg][st] + add;
        }
      }
      f32x4 b[NST];
#pragma unroll
      for (int st = 0; st < NST; ++st) b[st] = channels(w.bias, c4 + st * 16);
      if (!w.out_f32) {
        auto all = [&](auto value) {
#pragma unroll
          for (int rg = 0; rg < RG; ++rg)
#pragma unroll
            for (int p = 0; p < 2; ++p) {
              bf16x4 v[2];
#pragma unroll
              for (int st = 0; st < 2; ++st)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[st][e] = (bf16)value(acc[rg][p * 2 + st][e] + b[p * 2 + st][e]);
              const u32x4 out = eight_channels(v[0], v[1]);
              if (on[rg] && n0 + p * 32 + c8 < w.n_main)
                *reinterpret_cast<u32x4*>(reinterpret_cast<bf16*>(mat.Y) + (size_t)m[rg] * w.ld + n0 + p * 32 + c8) = out;
            }
        };
        if (w.act == PTA_ACT_SIGMOID) all([](float v) { return sigmoid_wide(v); });
        else all([](float v) { return v; });
      } else {
        // (some row groups at a time, as many as the registers hold: what they are multiplied by and added to is requested together)
        constexpr int AT = RG == 4 ? 4 : 2;
#pragma unroll
        for (int h = 0; h < RG; h += AT) {
          f32x4 old[AT][NST];
          bf16x4 by[AT][NST];
#pragma unroll
          for (int i = 0; i < AT; ++i)
#pragma unroll
            for (int st = 0; st < NST; ++st) {
              const bool in = on[h + i] && c4 + st * 16 < w.n_main;
              const size_t at = (size_t)m[h + i] * w.ld + c4 + st * 16;
              if (w.accumulate && in) old[i][st] = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(mat.Y) + at);
              if (w.mul && in) by[i][st] = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const bf16*>(w.mul) + at);
            }
#pragma unroll
          for (int i = 0; i < AT; ++i)
#pragma unroll
            for (int st = 0; st < NST; ++st) {
              f32x4 v;
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                v[e] = acc[h + i][st][e] + b[st][e];
                if (w.mul) v[e] *= (float)by[i][st][e];
                if (w.accumulate) v[e] += old[i][st][e];
              }
              if (on[h + i] && c4 + st * 16 < w.n_main) *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(mat.Y) + (size_t)m[h + i] * w.ld + c4 + st * 16) = v;
            }
        }
      }
    }
  }
  return true;
}

// The sums of a wave's tile (RG row groups x NST channel blocks; lane l holds channels st * 16 + (l / 16) * 4 + r of
// row l % 16 of each row group) go out: unit cw of the workgroup, first block blk0 of matrix `mat`, rows from row0 of M,
// to the rows of Y that `order` lists (null: the same).
template <class Fmt, int NST, int RG, bool PAIR>
__device__ __forceinline__ void panel_store(const GemmMat& mat, const GemmEpilogue& epi, float* part, f32x4 (&acc)[RG][NST], unsigned char* smem, int cw, int blk0,
                                            int row0, int nsl, typename Fmt::Scale s0, typename Fmt::Scale s1, int M, const int32_t* order = nullptr) {
  if (straight_store<Fmt, NST, RG, PAIR>(mat, epi, acc, blk0, row0, nsl, s0, s1, M, order)) return;
  constexpr int SW = NST * 16 + 4;                // floats per row of a wave's epilogue strip
  const int lane = threadIdx.x & 63;
  // Lane l holds channels st * 16 + (l / 16) * 4 + r of row l % 16 of each row group.  Row group by row group the
  // sums pass through a strip of LDS of the wave's own (the row buffers are free after the last barrier) and come
  // back with eight consecutive channels of one row per lane: one 16-byte store per lane, whole 128-byte stretches
  // of a row per wave.  (A wave's LDS accesses complete in order.)
  float* strip = reinterpret_cast<float*>(smem) + (size_t)cw * (16 * SW);
  const int N = mat.N;
  const bool direct = !mat.bias && mat.act == PTA_ACT_NONE && !epi.bias && epi.act == PTA_ACT_NONE && !epi.mul &&
                      epi.post_scale == 0.0f && !epi.out_fp8_scale;
  auto put = [&](const f32x4 (&sums)[NST]) {
#pragma unroll
    for (int st = 0; st < NST; ++st)
      *reinterpret_cast<f32x4*>(strip + (lane & 15) * SW + st * 16 + (lane >> 4) * 4) = sums[st];
  };
  // (one copy of the epilogue code: unrolled over the row groups it is too large to unroll, and an accumulator
  // array indexed by a loop counter lives in scratch memory for the whole kernel - hence the chain of comparisons)
#pragma unroll 1
  for (int rg = 0; rg < RG; ++rg) {
#pragma unroll
    for (int r = 0; r < RG; ++r)
      if (r == rg) put(acc[r]);
    if constexpr (PAIR) {
      constexpr int LPR = NST / 2 * 16 / 8;                      // lanes per row: eight output channels each
      constexpr int RPP = 64 / LPR;                              // rows per pass
#pragma unroll 1
      for (int it = 0; it < 16 / RPP; ++it) {
        const int rr = it * RPP + lane / LPR, c0 = (lane % LPR) * 8;
        const int m = row0 + rg * 16 + rr, n = blk0 * 16 + c0;
        if (rr >= 16) continue;
        const f32x4 g0 = *reinterpret_cast<const f32x4*>(strip + rr * SW + c0), g1 = *reinterpret_cast<const f32x4*>(strip + rr * SW + c0 + 4);
        const f32x4 u0 = *reinterpret_cast<const f32x4*>(strip + rr * SW + NST / 2 * 16 + c0), u1 = *reinterpret_cast<const f32x4*>(strip + rr * SW + NST / 2 * 16 + c0 + 4);
        if (m >= M) continue;
        if constexpr (Fmt::kWide) {
          wide_put_pair8(mat, order ? order[m] : m, n, g0, g1, u0, u1);
          continue;
        }
        f16x8 y;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          y[j] = swiglu_out(epi, (f16)Fmt::finish(j < 4 ? g0[j & 3] : g1[j & 3], s0), (f16)Fmt::finish(j < 4 ? u0[j & 3] : u1[j & 3], s1));
        if (n + 8 <= N && (N & 7) == 0) {
          *reinterpret_cast<f16x8*>(mat.Y + (size_t)m * N + n) = y;
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (n + j < N) mat.Y[(size_t)m * N + n + j] = y[j];
        }
      }
    } else {
      constexpr int LPR = NST * 16 / 8;
      constexpr int RPP = 64 / LPR;
#pragma unroll 1
      for (int it = 0; it < (16 + RPP - 1) / RPP; ++it) {
        const int rr = it * RPP + lane / LPR, c0 = (lane % LPR) * 8;
        const int m = row0 + rg * 16 + rr, n = blk0 * 16 + c0;
        if (rr >= 16) continue;
        const f32x4 v0 = *reinterpret_cast<const f32x4*>(strip + rr * SW + c0), v1 = *reinterpret_cast<const f32x4*>(strip + rr * SW + c0 + 4);
        if (m >= M) continue;
        if (nsl > 1) {
          float* p = part + ((size_t)blockIdx.y * M + m) * N + n;
          if (n + 8 <= N && (N & 3) == 0) {
            *reinterpret_cast<f32x4*>(p) = v0;
            *reinterpret_cast<f32x4*>(p + 4) = v1;
          } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
              if (n + j < N) p[j] = j < 4 ? v0[j & 3] : v1[j & 3];
          }
          continue;
        }
        if constexpr (Fmt::kWide) {
          wide_put8(mat, order ? order[m] : m, n, v0, v1);
          continue;
        }
        f16x8 y;
        if (direct && n + 8 <= N && (N & 7) == 0) {                // nothing but the residual stream to add: whole vectors
          f16x8 res;
          if (epi.residual) res = *reinterpret_cast<const f16x8*>(epi.residual + (size_t)m * N + n);
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            y[j] = (f16)Fmt::finish(j < 4 ? v0[j & 3] : v1[j & 3], s0);
            if (epi.residual) y[j] = y[j] + res[j];
          }
          *reinterpret_cast<f16x8*>(mat.Y + (size_t)m * N + n) = y;
          continue;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          f16 y0 = (f16)Fmt::finish(j < 4 ? v0[j & 3] : v1[j & 3], s0);
          if (n + j < N) {
            if (mat.bias) y0 = y0 + mat.bias[n + j];
            y0 = apply_act(mat.act, y0);
            y0 = apply_epilogue(epi, y0, m, n + j, N);
          }
          y[j] = y0;
        }
        if (n + 8 <= N && (N & 7) == 0) {
          *reinterpret_cast<f16x8*>(mat.Y + (size_t)m * N + n) = y;
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (n + j < N) mat.Y[(size_t)m * N + n + j] = y[j];
        }
      }
    }
  }
}

// ------------------------------------------------------------------------------------------
// Variant for hundreds of rows: the roles turned round.  The tiled weight format IS the A operand order, so a
// wave fetches the tiles of its own NST channel blocks straight into registers (1 KiB per instruction, no LDS)
// and decodes them there; the RG * 16 activation rows of the workgroup (48 to 128) go through LDS once per 128-feature tile
// (whole-row loads, double-buffered, one barrier per tile) and every wave reads all of them as B operands.
// A wave's tile is RG * 16 rows x NST * 16 channels: one B operand read from LDS feeds NST MFMAs and one decoded
// A operand feeds RG (8 in a launch that fills the chip), which is what keeps both LDS (128 bytes per clock and compute unit) and the vector ALU
// behind the matrix unit.  (With the weights through LDS and the rows in registers - gemm_rows_kernel - every
// wave reads every decoded weight: 1 KiB of LDS per 2 MFMAs, more than the LDS delivers.)
// PAIR: a wave owns NST / 2 gate blocks and the same blocks of the up weight.
// ------------------------------------------------------------------------------------------
constexpr int PANEL_WAVES = 8;
// units of `blocks` channel blocks of a matrix, the last one's perhaps fewer
constexpr int panel_units(int N, int blocks) { return ((N + 15) / 16 + blocks - 1) / blocks; }

// RG: row groups of 16 per workgroup (every wave multiplies all of them); KH: parts of K inside the workgroup - the
// waves are 8 / KH channel units x KH parts, part kh takes the feature tiles kh, kh + KH, ... of the workgroup's
// range and the parts' sums meet in LDS at the end.  KH > 1 is for launches of few tiles: it halves or
// quarters the channels of a workgroup tile, so more workgroups, without the fp32 round trip through memory that
// slices of workgroups (ksplit) cost, and fewer steps for each wave.  plan_gemm_panel chooses.
template <class Fmt, int NST, int RG, int KH, bool PAIR>
__global__ __launch_bounds__(PANEL_WAVES * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_panel_kernel(GemmArgs a, int groups, int row_blocks, int unit0, int units) {
  constexpr int KV = Fmt::kVec;
  constexpr int CW = PANEL_WAVES / KH;            // channel units (waves side by side) per workgroup
  constexpr int ROWS = RG * 16;
  constexpr int XPART = ROWS * 128;               // halves of one feature tile of the workgroup's rows
  constexpr int XSTAGE = KH * XPART;              // one stage: a tile per part
  constexpr int LOADS = KH * RG * 4, QN = (LOADS + PANEL_WAVES - 1) / PANEL_WAVES;      // row loads (4 rows each) per stage, and per wave
  constexpr int SW = NST * 16 + 4;                // floats per row of a wave's epilogue strip
  static_assert(!PAIR || NST % 2 == 0, "gate and up blocks in equal numbers");
  static_assert(KH == 1 || KH == 2 || KH == 4, "parts of K");
  static_assert(RG <= 8, "registers");
  static_assert(KH == 1 || (KH - 1) * CW * RG * NST * 1024 <= 2 * XSTAGE * 2, "the parts' sums meet in the row buffers");
  extern __shared__ __align__(16) unsigned char smem[];
  f16* xbuf = reinterpret_cast<f16*>(smem);                                              // [2][KH][ROWS][128], pieces exchanged (see fetch_x)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cw = wave % CW, kh = wave / CW;
  const int K = a.K, M = a.M;
  // workgroup id -> tile as in gemm_rows_kernel (contiguous stretches of the tile list per XCD); the row block runs
  // fastest, so the workgroups that are resident together multiply the same weights and those come from L2
  const int per = (int)gridDim.x / 8;
  const int tile = ((int)blockIdx.x % 8) * per + (int)blockIdx.x / 8;
  if (tile >= groups * row_blocks) return;
  const int row_block = tile % row_blocks, group = tile / row_blocks;
  const int nsl = a.ksplit > 1 ? a.ksplit : 1;
  const int per_slice = (a.KT + nsl - 1) / nsl;
  const int kt_first = (int)blockIdx.y * per_slice;
  const int kt_end = kt_first + per_slice < a.KT ? kt_first + per_slice : a.KT;
  const int steps = kt_end > kt_first ? (kt_end - kt_first + KH - 1) / KH : 0;      // a tile per part and step

  // this wave's channel blocks: unit `wu` of the matrices (the launch covers units unit0 .. units - 1); waves past the
  // last unit only help with the rows
  const int wu = unit0 + group * CW + cw;
  const bool active = wu < units;
  constexpr int NBW = PAIR ? NST / 2 : NST;                        // consecutive blocks of a unit
  int mi = 0, unit = active ? wu : 0;
  if (!PAIR) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int there = panel_units(a.mat[i].N, NBW);
      if (mi == i && i + 1 < a.count && unit >= there) unit -= there, mi = i + 1;
    }
  }
  const int blk0 = unit * NBW;                                    // first block within its matrix
  const int have = (a.mat[mi].N + 15) / 16 - blk0;                // blocks from there on (at least one)
  // Loads through buffer descriptors: the descriptor and the tile's offset travel in scalar registers and one
  // 32-bit offset per lane serves all streams, another all rows (with 64-bit addresses per lane the loop keeps a
  // pointer per stream and row in vector registers, which this kernel does not have).  Rows past M lie past
  // the end of the rows' descriptor and read as zero.
  const uint32_t blk_bytes = (uint32_t)a.KT * (KV * 1024);
  const unsigned char* w0 = reinterpret_cast<const unsigned char*>(a.mat[PAIR ? 0 : mi].tiled) + (size_t)blk0 * blk_bytes;
  const unsigned char* w1 = reinterpret_cast<const unsigned char*>(a.mat[PAIR ? 1 : mi].tiled) + (size_t)blk0 * blk_bytes;
  const __amdgpu_buffer_rsrc_t wr0 = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(w0), 0, (int)((have < NBW ? have : NBW) * blk_bytes), 0x00020000);
  const __amdgpu_buffer_rsrc_t wr1 = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(w1), 0, (int)((have < NBW ? have : NBW) * blk_bytes), 0x00020000);
  const int wlane = lane * 16;
  const int row0 = row_block * ROWS;
  const int rows_here = M - row0 < ROWS ? M - row0 : ROWS;
  const __amdgpu_buffer_rsrc_t xr0 = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<f16*>(a.X + (size_t)row0 * K), 0, (int)((size_t)rows_here * K * 2), 0x00020000);

  // this wave's weight tiles of step i (past the end of the range: zeros - the rows of that tile are zeros too; past the matrix's last block: that one again,
  // whose sums go nowhere)
  auto fetch_w = [&](int i, u32x4 (&wv)[NST][KV]) {
    const int kt = kt_first + i * KH + kh;
#pragma unroll
    for (int st = 0; st < NST; ++st)
#pragma unroll
      for (int v = 0; v < KV; ++v)
        wv[st][v] = kt < kt_end ? __builtin_amdgcn_raw_buffer_load_b128(PAIR && st >= NST / 2 ? wr1 : wr0, wlane,
                                      (int)((st % NBW < have ? st % NBW : have - 1) * blk_bytes + (uint32_t)(kt * KV + v) * 1024), 0)
                                : u32x4{0, 0, 0, 0};
  };
  // The rows go from memory into LDS without passing through registers: load q = 8 j + w (w: the wave) of a stage
  // brings rows 4 (q % (4 RG)) .. + 3 of the tile of part q / (4 RG), 256 bytes each, lane l the 16 bytes that
  // belong at position l % 16 of row l / 16 - LDS receives the lanes' data one after the other, so a row takes 256
  // bytes and its 16-byte pieces are stored exchanged among themselves: piece c of row r at position c ^ (r % 16).
  // The sixteen rows of a B operand read then fall into sixteen different groups of four banks, without padding.
  auto fetch_x = [&](int i, f16* stage) {
#pragma unroll
    for (int j = 0; j < QN; ++j) {
      const int q = j * PANEL_WAVES + wave;
      if (LOADS % PANEL_WAVES != 0 && q >= LOADS) break;
      const int part = q / (4 * RG), rb = q % (4 * RG);
      const int row = rb * 4 + (lane >> 4);
      const int piece = (lane & 15) ^ (row & 15);
      const int kt = kt_first + i * KH + part;
      const bool in_k = kt < kt_end && kt * 128 + piece * 8 < K;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr0, (__attribute__((address_space(3))) void*)(stage + part * XPART + rb * 4 * 128), 16,
                                               in_k ? row * K * 2 + piece * 16 : -1, kt * 256, 0, 0);
    }
  };

  f32x4 acc[RG][NST];
#pragma unroll
  for (int rg = 0; rg < RG; ++rg)
#pragma unroll
    for (int st = 0; st < NST; ++st) acc[rg][st] = f32x4{0.f, 0.f, 0.f, 0.f};

  // The product runs as one pipeline over all steps: 4 * NST blocks of RG MFMAs per tile (one decoded A operand
  // each); the A operand of the next block is decoded among the MFMAs of this one, and during the last block of a
  // 32-feature step every B operand is replaced by the next one's as soon as its MFMA has been issued - across the
  // tile boundary too.  So the tile's one barrier stands before its last 32 features: by then every wave has read
  // the last B operands from this stage (which the loads of the stage after next may then overwrite) and the next
  // stage's rows, requested when this one began, must have landed.
  u32x4 wa[NST][KV], wb[NST][KV];
  f16x8 xf[RG];
  f16x8 avc;
  const int xat = kh * XPART + (lane & 15) * 128;                  // this lane's row within a row group of its part, in halves
  auto b_piece = [&](int m) { return ((m * 4 + (lane >> 4)) ^ (lane & 15)) * 8; };
  if (steps > 0) {
    if (active) fetch_w(0, wa);
    fetch_x(0, xbuf);
  }
  typename Fmt::Scale sc[NST];             // (requested behind the first tile: one round trip to memory, not two)
#pragma unroll
  for (int st = 0; st < NST; ++st) {
    const GemmMat& mt = a.mat[PAIR ? (st < NST / 2 ? 0 : 1) : mi];
    sc[st] = Fmt::load_scale(mt.scale, a.x_scale, (blk0 + (PAIR ? st % (NST / 2) : st)) * 16 + (lane & 15), mt.N);
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);      // vmcnt(0): the rows have landed in LDS
  __syncthreads();
  if (active && steps > 0) {
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) xf[rg] = *reinterpret_cast<const f16x8*>(xbuf + xat + rg * 16 * 128 + b_piece(0));
    avc = Fmt::a_operand(wa[0], 0, sc[0]);
  }
  auto feature_tile = [&](int i, const u32x4 (&wc)[NST][KV], u32x4 (&wn)[NST][KV]) {
    const bool more = i + 1 < steps;
    const f16* xc = xbuf + (size_t)(i & 1) * XSTAGE + xat;
    const f16* xn = xbuf + (size_t)((i + 1) & 1) * XSTAGE + xat;
    if (more) {
      if (active) fetch_w(i + 1, wn);
      fetch_x(i + 1, xbuf + (size_t)((i + 1) & 1) * XSTAGE);
    }
    auto blocks = [&](int first, int last) {
#pragma unroll
      for (int blk = first; blk < last; ++blk) {
        const int m = blk / NST, st = blk % NST;
        f16x8 avn = avc;
        if (blk + 1 < 4 * NST) avn = Fmt::a_operand(wc[(blk + 1) % NST], (blk + 1) / NST, sc[(blk + 1) % NST]);
        else if (more) avn = Fmt::a_operand(wn[0], 0, sc[0]);
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) {
          acc[rg][st] = Fmt::mma(avc, xf[rg], acc[rg][st]);
          if (st == NST - 1) {
            if (m < 3) xf[rg] = *reinterpret_cast<const f16x8*>(xc + rg * 16 * 128 + b_piece(m + 1));
            else if (more) xf[rg] = *reinterpret_cast<const f16x8*>(xn + rg * 16 * 128 + b_piece(0));
          }
        }
        avc = avn;
      }
    };
    if (active) blocks(0, 3 * NST);
    __builtin_amdgcn_s_waitcnt(0x0f70);    // vmcnt(0): the next stage's rows have landed (and its weights)
    __syncthreads();
    if (active) blocks(3 * NST, 4 * NST);
  };
  for (int i = 0; i < steps; i += 2) {
    feature_tile(i, wa, wb);
    if (i + 1 < steps) feature_tile(i + 1, wb, wa);
  }
  __syncthreads();                         // (what follows reuses the row buffers)
  if constexpr (KH > 1) {
    // the sums of parts 1 .. KH - 1 go to part 0's wave of the same channel unit
    f32x4* ex = reinterpret_cast<f32x4*>(smem);                   // [(KH - 1) * CW][RG * NST][64]
    if (kh > 0 && active) {
#pragma unroll
      for (int rg = 0; rg < RG; ++rg)
#pragma unroll
        for (int st = 0; st < NST; ++st) ex[(((kh - 1) * CW + cw) * (RG * NST) + rg * NST + st) * 64 + lane] = acc[rg][st];
    }
    __syncthreads();
    if (kh == 0 && active) {
#pragma unroll
      for (int k = 1; k < KH; ++k)
#pragma unroll
        for (int rg = 0; rg < RG; ++rg)
#pragma unroll
          for (int st = 0; st < NST; ++st) {
            const f32x4 other = ex[(((k - 1) * CW + cw) * (RG * NST) + rg * NST + st) * 64 + lane];
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[rg][st][r] += other[r];
          }
    }
    __syncthreads();
    if (kh > 0) return;
  }
  if (!active) return;

  const typename Fmt::Scale s0 = Fmt::load_scale(a.mat[PAIR ? 0 : mi].scale, a.x_scale, 0, 1);   // no format's finish uses the per-channel part
  const typename Fmt::Scale s1 = Fmt::load_scale(a.mat[PAIR ? 1 : mi].scale, a.x_scale, 0, 1);
  panel_store<Fmt, NST, RG, PAIR>(a.mat[PAIR ? 0 : mi], a.epi, a.part, acc, smem, cw, blk0, row0, nsl, s0, s1, M);
}

// ------------------------------------------------------------------------------------------
// Variant for hundreds of rows of formats with more than one vector per tile (16-bit and FP8 weights): both operands
// through LDS.  A workgroup of 8 waves owns 256, 192 or 128 rows and 256 channels (a pair: 128 gate and 128 up channels), or 128 rows and
// 128 channels; loads that write LDS directly bring stages of 64 features of both.
// At 256 x 256 a 64-feature step is 64 KiB for 8.4 MFLOP, a quarter of the bytes per product that gemm_rows_kernel's
// workgroups (256 x 128, weights through registers) take.
// What bounds it: the loads.  A compute unit has about 32 KiB of them on their way, 128 bytes a line, so what counts is lines and how long each takes:
// 110 GB/s from L2, 37 weights from memory, 54 to 60 both as they come - 1.2, 0.77 and 0.53 us for a step's 64 KiB (256 x 256), 48 (128 x 256) and 32 (128 x 128),
// against 1.1, 0.64 and 0.35 of the products alone at the clock that the power leaves.  Hence stages of 64 features, whole lines of the rows (with 32,
// half lines: as many requests for half the bytes), tiles of a die that share rows and weights both (BLOCK_BAND), and requests all the time (APART; one load
// per block of MFMAs: a wave that asks for more at once is held).  bf16, weights from memory, with stages of 32 and now: 2048 rows, 8192 x 8192 203 -> 193 us (256 x
// 256), 1920 rows, 8192 x 6144 175 -> 148 (192 x 256), 2048 rows, 11008 x 4096 183 -> 150 (128 x 256), 5632 x 2048 63 -> 51 (128 x 128).
// Not kept: the order of a stage's loads turned by the workgroup, so that each line is asked for early by another one (the scalar arithmetic between the products
// costs 5 %); wave priorities round the products or for half of the waves (0 to 3 % slower); the next operand converted among this one's products (2 to 6 % slower).
// Channels need not divide: blocks past a matrix's last one lie past its descriptor and read as zeros.
// ------------------------------------------------------------------------------------------
constexpr int BLOCK_WAVES = 8;
constexpr int BLOCK_BAND = 4;               // channel groups that a die's workgroups share the rows of (one: 2 to 5 % slower at 128 rows a tile and 2048 rows)
// The tile of a wave's RG row groups x 4 channel blocks: 2 x 4 waves of 8, 6 or 4 groups (256, 192 or 128 rows by 256 channels), or 4 x 2 of 2 (128 x 128)
constexpr int block_row_parts(int rg) { return rg == 2 ? 4 : 2; }
constexpr int block_rows(int rg) { return block_row_parts(rg) * rg * 16; }
constexpr int block_cb(int rg) { return 8 / block_row_parts(rg) * 4; }         // channel blocks of a workgroup
// us of a step of 64 features (measured, all compute units at work), and of a tile's begin and end.  16-bit weights take 0.88 to 0.92 of theirs, as F143 ones do: these
// figures are those of stages of 32 features, and stay because slices of K, and with them the order of a product's sums, follow from them.
constexpr double block_step_us(int rg, bool f143) {
  return f143 ? (rg == 8 ? 1.45 : rg == 6 ? 1.1 : rg == 4 ? 0.84 : 0.55) : rg == 8 ? 1.6 : rg == 6 ? 1.25 : rg == 4 ? 0.92 : 0.6;
}
constexpr double block_ends_us(int rg) { return rg == 8 ? 9.0 : rg == 6 ? 7.5 : rg == 4 ? 6.0 : 5.0; }

// v, of which the compiler no longer knows where it is from
__device__ __forceinline__ u32x4 as_computed(u32x4 v) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t e = v[i];
    asm volatile("" : "+v"(e));
    v[i] = e;
  }
  return v;
}

// Bytes of a stage (64 features) of the rows and of the weights, and how many stages of each LDS holds
constexpr int block_x_bytes(int rg) { return block_rows(rg) * 128; }
template <class Fmt>
constexpr int block_w_bytes(int rg) { return block_cb(rg) * Fmt::kVec * 512; }
// whether the weights are asked for in a step's first half (to the place that the stage before has left) and only the rows in its second
template <class Fmt>
constexpr bool block_apart(int rg) { return Fmt::kVec == 4 || rg != 8; }
template <class Fmt>
constexpr int block_x_stages(int rg) {
  const int both = 160 * 1024 / (block_x_bytes(rg) + block_w_bytes<Fmt>(rg));
  return both < 5 ? both : 5;
}
template <class Fmt>
constexpr int block_w_stages(int rg) {            // one more where it fits
  const int x = block_x_stages<Fmt>(rg);
  return block_apart<Fmt>(rg) && x < 5 && x * block_x_bytes(rg) + (x + 1) * block_w_bytes<Fmt>(rg) <= 160 * 1024 ? x + 1 : x;
}
template <class Fmt>
constexpr int block_lds_bytes(int rg) { return block_x_stages<Fmt>(rg) * block_x_bytes(rg) + block_w_stages<Fmt>(rg) * block_w_bytes<Fmt>(rg); }

// waits until at most N of this wave's loads from memory are on their way, and (LDS) for all of its LDS requests
template <int N, bool LDS = false>
__device__ __forceinline__ void wait_loads() {
  static_assert(N < 64, "the counter of requests");
  __builtin_amdgcn_s_waitcnt((LDS ? 0x0070 : 0x0f70) | (N & 15) | (N >> 4) << 14);
}

template <class Fmt, int RG, bool PAIR, class Rows = AllRows>
__global__ __launch_bounds__(BLOCK_WAVES * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_block_kernel(GemmArgs a, int group0, int groups, int row_blocks, Rows rows) {
  constexpr int KV = Fmt::kVec, NST = 4;
  constexpr int WVEC = KV * 512;                  // bytes of a channel block's features of a stage
  constexpr int ROWS = block_rows(RG), WR = block_row_parts(RG), WC = BLOCK_WAVES / WR;
  constexpr int CB = block_cb(RG), BPW = CB / BLOCK_WAVES;      // channel blocks of the workgroup, and how many a wave brings
  constexpr int XB = block_x_bytes(RG), WB = block_w_bytes<Fmt>(RG), NX = block_x_stages<Fmt>(RG), NW = block_w_stages<Fmt>(RG);
  constexpr int XL = XB / (BLOCK_WAVES * 1024);   // loads per wave and stage: rows (eight of them each)
  constexpr int WPB = WVEC / 1024, WL = BPW * WPB;              // and weights, of a channel block and in all
  constexpr bool APART = block_apart<Fmt>(RG);
  // loads that may be on their way when the next stage must have landed: those asked for behind its weights, and behind its rows
  constexpr int BEHIND_W = (NW - 2) * (XL + WL), BEHIND_X = APART ? (NX - 2) * XL + (NX - 1) * WL : BEHIND_W;
  constexpr int WAIT = BEHIND_W < BEHIND_X ? BEHIND_W : BEHIND_X;
  constexpr int W_BEGIN = APART ? NW - 1 : NW;    // stages of weights that are asked for at the begin
  static_assert(XB % (BLOCK_WAVES * 1024) == 0 && WVEC % 1024 == 0 && NX >= 2 && (APART ? NW >= 3 : NW == NX) && block_lds_bytes<Fmt>(RG) <= 160 * 1024, "stages");
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave / WC, wc = wave % WC;
  const int K = a.K;
  // workgroup id -> tile: contiguous stretches of the tile list per die, in bands of BLOCK_BAND channel groups, within a band the group fastest
  int per = (int)gridDim.x / 8;
  if constexpr (Rows::kListed) {                  // (the launch has room for the most tiles there can be)
    row_blocks = *rows.n_tiles;
    per = (groups * row_blocks + 7) / 8;
    if ((int)blockIdx.x / 8 >= per) return;
  }
  const int tile = ((int)blockIdx.x % 8) * per + (int)blockIdx.x / 8;
  if (tile >= groups * row_blocks) return;
  const int band = tile / (BLOCK_BAND * row_blocks), in_band = tile - band * (BLOCK_BAND * row_blocks);
  const int band_groups = groups - band * BLOCK_BAND < BLOCK_BAND ? groups - band * BLOCK_BAND : BLOCK_BAND;
  const int row_block = in_band / band_groups;
  int group = group0 + band * BLOCK_BAND + in_band - row_block * band_groups;
  int M = a.M;
  const int32_t* order = nullptr;
  size_t weight_at = 0;
  if constexpr (Rows::kListed) {
    const int32_t* t = rows.tiles + row_block * 4;
    weight_at = (size_t)t[0] * rows.weight_bytes;
    order = rows.order + t[1];
    M = t[2];
  }
  const int row0 = Rows::kListed ? 0 : row_block * ROWS;
  int mi = 0;
  if constexpr (!PAIR) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int g = i < a.count ? (a.mat[i].N + CB * 16 - 1) / (CB * 16) : 0;
      if (mi == i && i + 1 < a.count && group >= g) { group -= g; mi = i + 1; }
    }
  }
  const int blk0 = group * (PAIR ? CB / 2 : CB);  // first block within its matrix
  // the slice's features in steps of 64
  const int nsl = a.ksplit > 1 ? a.ksplit : 1;
  const int all = (K + 63) / 64, per_slice = ((a.KT + nsl - 1) / nsl) * 2;
  const int first = (int)blockIdx.y * per_slice;
  const int last = first + per_slice < all ? first + per_slice : all;
  // this wave brings blocks BPW * wave and on of the workgroup's (of a pair: first the gate's, then the up blocks)
  const GemmMat& wm = a.mat[PAIR ? wave >> 2 : mi];
  const int wb = blk0 + BPW * (PAIR ? wave & 3 : wave);
  const uint32_t blk_bytes = (uint32_t)a.KT * (KV * 1024);
  int there = (wm.N + 15) / 16 - wb;
  there = __builtin_amdgcn_readfirstlane(there < 0 ? 0 : there < BPW ? there : BPW);
  const unsigned char* wp = uniform_pointer(reinterpret_cast<const unsigned char*>(wm.tiled) + weight_at + (size_t)(there ? wb : 0) * blk_bytes);
  const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(wp), 0, (int)(there * blk_bytes), 0x00020000);
  const f16* X = a.mat[mi].X ? a.mat[mi].X : a.X;
  const int rows_here = M - row0 < ROWS ? M - row0 : ROWS;
  const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<f16*>(X + (size_t)row0 * K), 0, Rows::kListed ? 0x7fffffff : (int)((size_t)rows_here * K * 2), 0x00020000);

  // A row's 128 bytes of a stage are eight pieces of 16, exchanged: piece c of row r at c ^ swap(r), so that no sixteen lanes of an operand read that
  // the LDS serves at once (0-3, 12-15, 20-23, 24-27, ...) meet in a bank.
  auto swap = [](int r) { return ((r >> 1) & 7) ^ ((r & 1) << 2); };
  const int lane_row = lane >> 3;
  const int piece = (lane & 7) ^ swap((wave & 1) * 8 + lane_row);               // (the same in all loads of a lane)
  const int x0 = (wave * 8 + lane_row) * (K * 2) + piece * 16;    // byte offset of its first row (past the last row: past the descriptor)
  int listed[XL];
  if constexpr (Rows::kListed) {
#pragma unroll
    for (int j = 0; j < XL; ++j) {
      const int r = (j * BLOCK_WAVES + wave) * 8 + lane_row;
      listed[j] = r < M ? order[r] / rows.x_div * (K * 2) + piece * 16 : -1;
    }
  }
  // load q of stage s (of the K axis) into LDS at byte `at`; past the slice's end: zeros, from nowhere
  auto bring_x = [&](int s, int at, int q) {
    const int off = Rows::kListed ? listed[q] : x0 + q * (BLOCK_WAVES * 16) * K;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(xres, (__attribute__((address_space(3))) void*)(smem + at + (q * BLOCK_WAVES + wave) * 1024), 16,
                                             s < last && s * 64 + piece * 8 < K ? off : -1, s * 128, 0, 0);
  };
  auto bring_w = [&](int s, int at, int q) {
    const int b = q / WPB, v = q % WPB;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(wres, (__attribute__((address_space(3))) void*)(smem + at + (BPW * wave + b) * WVEC + v * 1024), 16,
                                             s < last ? (int)(b * blk_bytes) + lane * 16 : -1, s * WVEC + v * 1024, 0, 0);
  };

  f32x4 acc[RG][NST];

  // operands of 32 features: half m of the stage at byte `at`
  typedef typename Fmt::Piece Piece;              // a lane's bytes of a weight operand
  const int a_at = (PAIR ? wc * 2 : wc * 4) * WVEC + lane * 16;
  auto a_piece = [&](int at, int m, int st) {
    const int blk = PAIR ? st % 2 + (st / 2) * (CB / 2) : st;
    return *reinterpret_cast<const Piece*>(smem + at + a_at + blk * WVEC + Fmt::piece_at(m));
  };
  const int b_row = (wr * (RG * 16) + (lane & 15)) * 128;
  const int b0 = b_row + ((lane >> 4) ^ swap(lane & 15)) * 16, b1 = b_row + ((4 + (lane >> 4)) ^ swap(lane & 15)) * 16;
  auto b_operand = [&](int at, int m, int rg) { return *reinterpret_cast<const f16x8*>(smem + at + (m ? b1 : b0) + rg * 2048); };

  // One pipeline over all steps: a step is two halves of 32 features, a half four blocks of RG MFMAs with one weight operand
  // each.  The row operands of the next half are requested in this one's first blocks (two sets of registers), the weight operand four blocks
  // ahead.  The barrier stands where everything of a stage has been requested: behind it
  // the stage takes what is some stages on, its weights (APART) half a step later, so that requests go out all the time.  (The last
  // half requests operands of a stage that does not exist and drops them: a condition here would stand between the MFMAs.)
  constexpr int W0 = NX * XB;                     // where the weights' stages begin
#pragma unroll
  for (int n = 0; n < NX || n < W_BEGIN; ++n) {
#pragma unroll
    for (int q = 0; q < XL; ++q)
      if (n < NX) bring_x(first + n, n * XB, q);
#pragma unroll
    for (int q = 0; q < WL; ++q)
      if (n < W_BEGIN) bring_w(first + n, W0 + n * WB, q);
  }
  uint32_t codes = 0;                             // (a lane's share) whether this wave's weights hold codes that the fast conversion does not know
  if constexpr (Fmt::kCodes) {
    if constexpr (PAIR) codes = Fmt::codes(a.mat[0], blk0 + wc * 2, 2, K, a.KT, lane) | Fmt::codes(a.mat[1], blk0 + wc * 2, 2, K, a.KT, lane);
    else codes = Fmt::codes(a.mat[mi], blk0 + wc * 4, 4, K, a.KT, lane);
  }
  // (the wide epilogue's many arguments, read while the first stages are on their way: bf16, 1024 x 8192, 1000 rows 29.5 -> 28.1 us; 2048 x 8192 46.9 -> 45.4; the
  // fp16 one's few gain nothing)
  GemmMat wide;
  GemmEpilogue none{};
  if constexpr (Fmt::kWide) {
    wide = a.mat[PAIR ? 0 : mi];
    read_end<Fmt, PAIR>(wide, none);
  }
  wait_loads<(NX - 1) * XL + (W_BEGIN - 1) * WL>();             // the first stage has landed
  __syncthreads();
  auto products = [&](auto fast) {
    constexpr bool FAST = decltype(fast)::value;
    // blocks of a half that its reads of row operands are spread over: two (four 1 % slower), but the vector unit's conversion beside reads of 256 rows takes all
    // four (F143, 2048 rows, 8192 x 8192 with codes in every block 229 -> 216 us, pair of 4096 x 13696 387 -> 363)
    constexpr int OVER = !FAST && RG == 8 ? 4 : 2;
    f16x8 xf[2][RG];
    Piece ahead[NST];
#pragma unroll
    for (int rg = 0; rg < RG; ++rg)
#pragma unroll
      for (int st = 0; st < NST; ++st) acc[rg][st] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) xf[0][rg] = b_operand(0, 0, rg);
#pragma unroll
    for (int st = 0; st < NST; ++st) ahead[st] = a_piece(W0, 0, st);
    // (the compiler would otherwise make one load of these and of the same ones at the end of a step, at the step's begin)
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) xf[0][rg] = bitcast<f16x8>(as_computed(bitcast<u32x4>(xf[0][rg])));
    __builtin_amdgcn_s_waitcnt(0xc07f);             // lgkmcnt(0): where the loop begins, nothing is on its way that its end does not know of
    int xat = 0, wat = W0, wfree = W0 + (NW - 1) * WB;            // the stage whose operands are multiplied; the place of the weights before it
    for (int i = first; i < last; ++i) {
      const int xnext = xat + XB == W0 ? 0 : xat + XB, wnext = wat + WB == W0 + NW * WB ? W0 : wat + WB;
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        if (m == 1) {
          wait_loads<WAIT, true>();                 // the next stage has landed, and this wave's requests from this one
          __builtin_amdgcn_s_barrier();
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int st = 0; st < NST; ++st) {
          const int from = APART && m == 0 ? XL : 0, n = APART ? (m == 0 ? WL : XL) : m == 0 ? 0 : XL + WL;      // requests of this half: rows, then weights
#pragma unroll
          for (int q = from + st * n / NST; q < from + (st + 1) * n / NST; ++q) {
            if (q < XL) bring_x(i + NX, xat, q);
            else bring_w(i + (APART ? NW - 1 : NW), APART ? wfree : wat, q - XL);
          }
          const f16x8 av = Fmt::template operand<FAST>(ahead[st]);
          ahead[st] = a_piece(m ? wnext : wat, 1 - m, st);
#pragma unroll
          for (int r = st * RG / OVER; r < (st + 1) * RG / OVER && r < RG; ++r) xf[1 - m][r] = b_operand(m ? xnext : xat, 1 - m, r);
#pragma unroll
          for (int rg = 0; rg < RG; ++rg) acc[rg][st] = Fmt::mma(av, xf[m][rg], acc[rg][st]);
          __builtin_amdgcn_sched_barrier(0);        // (the requests stay where they are)
        }
      }
      xat = xnext;
      wfree = wat;
      wat = wnext;
    }
  };
  if constexpr (Fmt::kCodes) {
    if (__any(codes != 0)) {
      products(std::false_type{});
    } else {
      products(std::true_type{});
    }
  } else {
    products(std::true_type{});
  }
  __builtin_amdgcn_s_waitcnt(0x0070);
  __syncthreads();                                // (what follows reuses the stages)
  const typename Fmt::Scale s0 = Fmt::load_scale(a.mat[PAIR ? 0 : mi].scale, a.x_scale, 0, 1);   // no format's finish uses the per-channel part
  const typename Fmt::Scale s1 = Fmt::load_scale(a.mat[PAIR ? 1 : mi].scale, a.x_scale, 0, 1);
  panel_store<Fmt, NST, RG, PAIR>(Fmt::kWide ? wide : a.mat[PAIR ? 0 : mi], a.epi, a.part, acc, smem, wave, blk0 + wc * (PAIR ? 2 : 4), row0 + wr * (RG * 16), nsl, s0, s1, M, order);
}

template <class Fmt, int RG, bool PAIR, class Rows>
static int reserve_gemm_block(const char* name) {
  static bool ready = false;
  constexpr int smem = block_lds_bytes<Fmt>(RG);
  static_assert(smem <= 160 * 1024 && smem >= BLOCK_WAVES * 16 * 68 * 4, "LDS");
  if (!ready) {
    PTA_REQUIRE(hipFuncSetAttribute((const void*)gemm_block_kernel<Fmt, RG, PAIR, Rows>, hipFuncAttributeMaxDynamicSharedMemorySize, smem) == hipSuccess,
                "%s: cannot reserve %d bytes of LDS", name, smem);
    ready = true;
  }
  return PTA_OK;
}

// channel groups of the launch, of `channels` each (of a pair: of half as many of both)
static inline int block_groups(const GemmArgs& a, bool pair, int channels = 256) {
  int g = 0;
  for (int i = 0; i < (pair ? 1 : a.count); ++i) g += pair ? (a.mat[i].N + channels / 2 - 1) / (channels / 2) : (a.mat[i].N + channels - 1) / channels;
  return g;
}

// channel groups [group0, group1) of the launch
template <class Fmt, int RG, bool PAIR>
static int launch_gemm_block(const GemmArgs& a, int group0, int group1, hipStream_t s, const char* name) {
  const int rc = reserve_gemm_block<Fmt, RG, PAIR, AllRows>(name);
  if (rc) return rc;
  const int groups = group1 - group0, row_blocks = (a.M + block_rows(RG) - 1) / block_rows(RG);
  const int nsl = a.ksplit > 1 ? a.ksplit : 1;
  const int per = (groups * row_blocks + 7) / 8;
  gemm_kernel_taken = "gemm_block_kernel";
  hipLaunchKernelGGL((gemm_block_kernel<Fmt, RG, PAIR>), dim3(per * 8, nsl), dim3(BLOCK_WAVES * 64), block_lds_bytes<Fmt>(RG), s, a,
                     group0, groups, row_blocks, AllRows{});
  if (nsl > 1) launch_splitk_finish<Fmt>(a, s);
  return PTA_OK;
}

// Tiles of listed rows (at most RG * 32 each, up to max_tiles of them) of a matrix, or of a gate / up pair; wide formats.  x_rows:
// rows of X.  (2048 rows, 6 of 32 experts of 4096 x 1376 each: pairs 579 -> 334 us, downs 373 -> 241, against gemm_rows_kernel)
template <class Fmt, int RG, bool PAIR>
static int launch_gemm_block_listed(const GemmArgs& a, size_t x_rows, int max_tiles, const ListedRows& rows, hipStream_t s, const char* name) {
  if (x_rows * a.K * 2 > 0x7fffffffu) return launch_gemm_listed<Fmt, RG / 4, PAIR>(a, (a.mat[0].N + 15) / 16, max_tiles, rows, s, name);
  const int rc = reserve_gemm_block<Fmt, RG, PAIR, ListedRows>(name);
  if (rc) return rc;
  const int groups = block_groups(a, PAIR);
  gemm_kernel_taken = "gemm_block_kernel";
  hipLaunchKernelGGL((gemm_block_kernel<Fmt, RG, PAIR, ListedRows>), dim3((groups * max_tiles + 7) / 8 * 8), dim3(BLOCK_WAVES * 64),
                     block_lds_bytes<Fmt>(RG), s, a, 0, groups, max_tiles, rows);
  return PTA_OK;
}

// How a launch is cut: the cheapest of the four tiles, K in slices of workgroups (one matrix, a workspace at hand; tiles of 256 and 128 rows by 256
// channels), or the channel groups of the whole rounds with 256 rows and the rest with a smaller tile - more workgroups, each shorter.
// What bounds most launches of one to three rounds is the compute units that the last round leaves idle: 144 tiles of 256 x 256 keep 112 of
// them from work, the same rows in 198 of 192 x 256 58; 64 tiles of 128 x 256 192, in 128 x 128 128 of them.  A smaller tile reads more
// bytes of LDS a product (a step of 64 features, MFMAs alone 1.2, 0.9, 0.6, 0.3 us), so it wins by its rounds only.
// us, with two tiles (256 and 128 by 256) and with four, weights from HBM: fp16, 1960 rows, 2048 x 2048 33.4 -> 25.0, 2048 x 4608 50.6 -> 45.0,
// 5632 x 2048 73.2 -> 58.2; 300 rows, 4096 x 4096 53.1 -> 38.2; 1656 rows, 11008 x 2048 117 -> 90; pair of 5632 x 5632, 791 rows 126 -> 109;
// bf16 pair of 11008 x 1024, 1100 rows 115 -> 81; F143, 2040 rows, 4096 x 4608 83.6 -> 77.9, 1601 rows, 5632 x 5632 118 -> 104.  Of 215 launches
// of 140 to 2000 rows that changed their tile, the slowest ratio was 0.98 (bf16, 1837 rows, 3072 x 11008: 136 -> 139), the middle one 1.1; of 160
// of 45 to 2000 rows by any channels and features two were below 0.98 (0.95: bf16, 692 rows, 2456 x 2200, scratch for three slices; 0.97: fp16, 229 rows, 5408 x 824).
// Not kept: 192 rows with K in slices (F143, 1583 rows, 11008 x 2304 94 -> 146), 192 rows for the rest at 4 us (0.97 to 1.04; hence 8), as many
// tiles of 192 as of 256 rows (three fp16 weights, 372 rows, 4288 x 7744 92 -> 99).
template <class Fmt, bool PAIR>
static int dispatch_gemm_block(const GemmArgs& a, hipStream_t s, const char* name) {
  const int cus = device_compute_units(), groups = block_groups(a, PAIR), narrow = block_groups(a, PAIR, 128);
  const double steps = (a.K + 63) / 64;
  auto blocks = [&](int rg) { return (a.M + block_rows(rg) - 1) / block_rows(rg); };
  auto cost = [&](int rg, int tiles, int nsl) {
    const double finish = nsl > 1 ? 5.0 + (double)a.M * a.mat[0].N * (4.0 * nsl + 6.0) / 4.5e6 : 0.0;
    return ((tiles * nsl + cus - 1) / cus) * (block_step_us(rg, Fmt::kVec == 2) * steps / nsl + block_ends_us(rg)) + finish;
  };
  const int whole = (groups * blocks(8) / cus) * cus / blocks(8);               // channel groups within whole rounds
  double best = cost(8, groups * blocks(8), 1);
  int rg = 8, rest = 0, slices = 1;               // the tile; that of the channel groups beyond the whole rounds (0: the same)
  for (int r = 6; r >= 2; r -= 2) {
    const double c = cost(r, (r == 2 ? narrow : groups) * blocks(r), 1);
    if (r == 6 && blocks(8) > 1 && blocks(6) == blocks(8)) continue;            // (as many tiles: what a tile of 256 rows lacks it does not load either)
    if (c < best) { best = c; rg = r; rest = 0; }
    if (whole == 0 || whole >= groups || (r == 2 && !PAIR && a.count > 1)) continue;      // (several matrices: their groups are counted differently)
    const double both = cost(8, whole * blocks(8), 1) + cost(r, (r == 2 ? narrow - 2 * whole : groups - whole) * blocks(r), 1) + (r == 6 ? 8.0 : 4.0);
    if (both < best) { best = both; rg = 8; rest = r; }
  }
  if (!PAIR && a.count == 1 && a.part)
    for (int nsl = 2; nsl <= GEMM_MAX_KSPLIT; ++nsl) {
      if (a.KT < nsl * 4 || a.part_bytes < (size_t)nsl * a.M * a.mat[0].N * sizeof(float)) break;
      for (int r = 8; r >= 4; r -= 4) {
        const double c = cost(r, groups * blocks(r), nsl);
        if (c < best) { best = c; rg = r; rest = 0; slices = nsl; }
      }
    }
  GemmArgs b = a;
  b.ksplit = slices;
  auto launch = [&](int r, int group0, int group1) {                            // groups of 256 channels; to the last one: -1
    switch (r) {
      case 8: return launch_gemm_block<Fmt, 8, PAIR>(b, group0, group1 < 0 ? groups : group1, s, name);
      case 6: return launch_gemm_block<Fmt, 6, PAIR>(b, group0, group1 < 0 ? groups : group1, s, name);
      case 4: return launch_gemm_block<Fmt, 4, PAIR>(b, group0, group1 < 0 ? groups : group1, s, name);
      default: return launch_gemm_block<Fmt, 2, PAIR>(b, 2 * group0, group1 < 0 ? narrow : 2 * group1, s, name);
    }
  };
  gemm_tiles_taken = {block_rows(rg), block_cb(rg) * 16, rest ? block_rows(rest) : 0, rest ? block_cb(rest) * 16 : 0};
  int rc = launch(rg, 0, rest ? whole : -1);
  if (!rc && rest) rc = launch(rest, whole, -1);
  if (rc) return rc;
  PTA_CHECK_LAUNCH(name);
  return PTA_OK;
}

// whether every matrix of the launch is a whole number of wave tiles of `nst` channel blocks and all share one input
static inline bool panel_fits(const GemmArgs& a, int nst, bool pair) {
  if (a.epi.norm != PTA_NORM_NONE || a.KT < 2) return false;
  if (pair) return ((a.mat[0].N + 15) / 16) % (nst / 2) == 0;
  for (int i = 0; i < a.count; ++i) {
    if (((a.mat[i].N + 15) / 16) % nst != 0) return false;
    if (a.mat[i].X && a.mat[i].X != a.X) return false;
  }
  return true;
}

// gemm_panel_kernel's launches: panel_fits, and channels that do not divide into its units, up to 24576 a matrix (64 rows in turn before: INT4, 1964 rows, 6336 x 1296
// 383 -> 50 us, 662 rows, three of 2304 x 1264 85 -> 22).  More channels than that still go 64 rows in turn, which is the slower: INT4, 32008 channels, 1032 features, 200
// rows 67 and 23 here, 4096 features, 1000 rows 466 and 202; F152, 32040 channels, 520 features, 136 rows 80 and 48.  That path is what they have had; the line is no
// line of speed.
static inline bool panel_takes(const GemmArgs& a, bool pair) {
  if (panel_fits(a, 4, pair)) return true;
  if (a.epi.norm != PTA_NORM_NONE || a.KT < 2) return false;
  for (int i = 0; i < (pair ? 1 : a.count); ++i)
    if (a.mat[i].N > 24576 || (!pair && a.mat[i].X && a.mat[i].X != a.X)) return false;
  return true;
}

static inline int panel_units(const GemmArgs& a, bool pair) {
  if (pair) return panel_units(a.mat[0].N, 2);
  int n = 0;
  for (int i = 0; i < a.count; ++i) n += panel_units(a.mat[i].N, 4);
  return n;
}

// units [unit0, unit1) of the launch's matrices (a unit: NST channel blocks, or NST / 2 gate and up blocks)
template <class Fmt, int NST, int RG, int KH, bool PAIR>
static int launch_gemm_panel(const GemmArgs& a, int unit0, int unit1, hipStream_t s, const char* name) {
  static bool ready = false;
  constexpr int CW = PANEL_WAVES / KH;
  constexpr size_t rows_bytes = (size_t)2 * KH * RG * 16 * 128 * 2, strips = (size_t)CW * 16 * (NST * 16 + 4) * 4;
  constexpr size_t smem = rows_bytes > strips ? rows_bytes : strips;
  static_assert(smem <= 160 * 1024, "LDS");
  if (!ready) {
    PTA_REQUIRE(hipFuncSetAttribute((const void*)gemm_panel_kernel<Fmt, NST, RG, KH, PAIR>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)smem) == hipSuccess,
                "%s: cannot reserve %zu bytes of LDS", name, smem);
    ready = true;
  }
  const int groups = (unit1 - unit0 + CW - 1) / CW;
  const int row_blocks = (a.M + RG * 16 - 1) / (RG * 16);
  const int nsl = a.ksplit > 1 ? a.ksplit : 1;
  const int per = (groups * row_blocks + 7) / 8;
  gemm_kernel_taken = "gemm_panel_kernel";
  hipLaunchKernelGGL((gemm_panel_kernel<Fmt, NST, RG, KH, PAIR>), dim3(per * 8, nsl), dim3(PANEL_WAVES * 64), smem, s, a, groups, row_blocks, unit0, unit1);
  if (nsl > 1) launch_splitk_finish<Fmt>(a, s);
  return PTA_OK;
}

// Formats with a form of gemm_block_kernel
template <class Fmt> struct BlockFormat { static constexpr bool ok = false; };
// Formats whose launches of more than 128 rows gemm_panel_kernel takes (those without a form of gemm_block_kernel)
template <class Fmt> struct PanelFormat { static constexpr bool ok = Fmt::kVec <= 2 && !BlockFormat<Fmt>::ok; };

// A launch of gemm_panel_kernel: row groups of a tile, parts of K inside a workgroup, slices of workgroups; and those of the channel groups beyond
// the first `whole` (0: all alike).
struct PanelPlan { int rg, kh, slices, whole, rest_rg, rest_kh; double us; };
// the tiles there are (F152 not with 128 rows: their decoding's registers spill)
constexpr int PANEL_TILES[][2] = {{8, 1}, {7, 1}, {6, 1}, {5, 1}, {8, 2}, {7, 2}, {6, 2}, {5, 2}, {4, 2}, {5, 4}, {4, 4}, {3, 4}};

// How a launch is cut: the tile, and the slices of K (one matrix, a workspace at hand), that come out shortest, or tiles of one kind for the whole rounds and
// another kind for the rest.  What bounds most launches is that a wave goes through its part of K alone, tile by tile: the step of 128 features of 8 waves
// takes what its products and its decoding take one after the other, whether the other compute units have work or not.  So fewer rows a tile and more parts
// of K make a launch of few tiles shorter, and one of several rounds where these come out even.  us of a step and of a tile's begin and end (INT4, weights from
// HBM): 5 to 8 row groups 1.76 to 2.37 and 6.5, two parts 1.72 (4 groups) to 2.77 and 5.5, four 2.0 (3) to 2.8 and 2.7; up to a quarter more where all
// compute units work; F152 6.4 a step more.  For 130 shapes (1024 to 11008 channels, 130 to 2000 rows), each measured with all of them, the plan's is within 2 % of the best
// in all but one (4.5 %).  us with 128 rows and one or two parts only, and now: INT4, three of 4096 x 4096, 160 rows 49 -> 28, 1000 rows 90 -> 85; 8192 x 6144, 256 rows 93 -> 42;
// pair of 2048 x 5632, 400 rows 28.8 -> 22.3; 4096 x 4096 with scratch, 500 rows 37 -> 23, 1000 rows 50 -> 36; pair of 4096 x 11008, 320 rows 83 -> 64; F152, 8192 x 6144, 160 rows 480 -> 134.
template <class Fmt, bool PAIR>
static PanelPlan plan_gemm_panel(const GemmArgs& a) {
  constexpr bool F152 = OwnStreams<Fmt>::long_decode;
  // A norm's launch, in whose place the slices are added.  Without a norm behind the product as much again, but no more than 4 % of the time, which these estimates do not
  // tell apart: a product that this leaves in slices has its sums in the order that they have before a norm (11008 x 4096, 1000 rows: 95 us, 92 whole).
  constexpr double NORM = 4.3;
  const bool normed = a.then && a.then->any_order && finish_norm_fits(a);
  const int cus = device_compute_units(), all = panel_units(a, PAIR);
  auto time = [&](int rg, int kh, int slices, int units) {
    const double step = (F152 ? 6.4 : 0.0) + (kh == 1 ? 0.7 + 0.21 * rg : kh == 2 ? 0.68 + 0.26 * rg : 0.83 + 0.39 * rg), ends = kh == 1 ? 6.5 : kh == 2 ? 5.5 : 2.7;
    // (each die its share of a slice's tiles: 84 tiles in three slices are 33 for the 32 compute units of most, and twice as long, 53 us against 35)
    const int cw = PANEL_WAVES / kh, tiles = ((units + cw - 1) / cw * ((a.M + rg * 16 - 1) / (rg * 16)) + 7) / 8 * 8 * slices;
    const double last = (double)(tiles % cus) / cus, load = 0.03 * rg;
    const double one = ends + ((a.KT + slices - 1) / slices + kh - 1) / kh * step;
    return one * (tiles / cus * (1.0 + load) + (last > 0.0 ? 1.0 + load * last * last : 0.0)) + (slices > 1 ? 3.0 + (double)a.M * a.mat[0].N * (4.0 * slices + 6.0) / 5.5e6 - (normed ? NORM : 0.0) : 0.0);
  };
  PanelPlan best{F152 ? 7 : 8, 1, 1, 0, 0, 0, 1e30};
  double least = best.us;
  auto choose = [&](const PanelPlan& p) {
    const double us = p.slices > 1 && !normed ? p.us - (0.04 * p.us < NORM ? 0.04 * p.us : NORM) : p.us;
    if (us < least) least = us, best = p;
  };
  for (const auto& t : PANEL_TILES) {
    if (F152 && t[0] == 8) continue;
    for (int slices = 1; slices <= (!PAIR && a.count == 1 && a.part ? GEMM_MAX_KSPLIT : 1); ++slices) {
      if (t[1] * slices > 1 && a.KT < t[1] * slices * 4) break;
      if (slices > 1 && a.part_bytes < (size_t)slices * a.M * a.mat[0].N * sizeof(float)) break;
      choose(PanelPlan{t[0], t[1], slices, 0, 0, 0, time(t[0], t[1], slices, all)});
    }
    if (t[1] > 1) continue;
    const int groups = (all + PANEL_WAVES - 1) / PANEL_WAVES, row_blocks = (a.M + t[0] * 16 - 1) / (t[0] * 16), whole = groups * row_blocks / cus * cus / row_blocks;
    if (whole == 0 || whole >= groups) continue;
    const double first = time(t[0], 1, 1, whole * PANEL_WAVES);
    for (const auto& r : PANEL_TILES) {
      if ((F152 && r[0] == 8) || (r[1] > 1 && a.KT < r[1] * 4)) continue;
      choose(PanelPlan{t[0], 1, 1, whole, r[0], r[1], first + time(r[0], r[1], 1, all - whole * PANEL_WAVES) + 1.0});
    }
  }
  return best;
}

template <class Fmt, bool PAIR>
static int launch_gemm_panel_plan(const GemmArgs& a, const PanelPlan& p, hipStream_t s, const char* name) {
  const int units = panel_units(a, PAIR);
  GemmArgs b = a;
  b.ksplit = p.slices;
  auto launch = [&](int rg, int kh, int unit0, int unit1) {
    switch (rg * 10 + kh) {
      case 71: return launch_gemm_panel<Fmt, 4, 7, 1, PAIR>(b, unit0, unit1, s, name);
      case 61: return launch_gemm_panel<Fmt, 4, 6, 1, PAIR>(b, unit0, unit1, s, name);
      case 51: return launch_gemm_panel<Fmt, 4, 5, 1, PAIR>(b, unit0, unit1, s, name);
      case 72: return launch_gemm_panel<Fmt, 4, 7, 2, PAIR>(b, unit0, unit1, s, name);
      case 62: return launch_gemm_panel<Fmt, 4, 6, 2, PAIR>(b, unit0, unit1, s, name);
      case 52: return launch_gemm_panel<Fmt, 4, 5, 2, PAIR>(b, unit0, unit1, s, name);
      case 42: return launch_gemm_panel<Fmt, 4, 4, 2, PAIR>(b, unit0, unit1, s, name);
      case 54: return launch_gemm_panel<Fmt, 4, 5, 4, PAIR>(b, unit0, unit1, s, name);
      case 44: return launch_gemm_panel<Fmt, 4, 4, 4, PAIR>(b, unit0, unit1, s, name);
      case 34: return launch_gemm_panel<Fmt, 4, 3, 4, PAIR>(b, unit0, unit1, s, name);
      default: break;
    }
    if constexpr (!OwnStreams<Fmt>::long_decode) {
      if (rg == 8) return kh == 1 ? launch_gemm_panel<Fmt, 4, 8, 1, PAIR>(b, unit0, unit1, s, name) : launch_gemm_panel<Fmt, 4, 8, 2, PAIR>(b, unit0, unit1, s, name);
    }
    pta_set_error("%s: no tile of %d rows and %d parts", name, rg * 16, kh);
    return (int)PTA_EINVAL;
  };
  gemm_tiles_taken = {p.rg * 16, PANEL_WAVES / p.kh * 64, p.whole ? p.rest_rg * 16 : 0, p.whole ? PANEL_WAVES / p.rest_kh * 64 : 0};
  int rc = launch(p.rg, p.kh, 0, p.whole ? p.whole * PANEL_WAVES : units);
  if (!rc && p.whole) rc = launch(p.rest_rg, p.rest_kh, p.whole * PANEL_WAVES, units);
  if (rc) return rc;
  PTA_CHECK_LAUNCH(name);
  return PTA_OK;
}

template <class Fmt, int MT, bool PAIR>
static int launch_gemm_own_for(const GemmArgs& a, int nb, hipStream_t s, const char* name) {
  constexpr int CAP = own_cap<Fmt, PAIR>(MT);
  if (CAP >= 6 && nb == 6) return launch_gemm_own<Fmt, MT, CAP >= 6 ? 6 : 1, PAIR>(a, s, name);
  if (CAP >= 5 && nb == 5) return launch_gemm_own<Fmt, MT, CAP >= 5 ? 5 : 1, PAIR>(a, s, name);
  if (CAP >= 4 && nb == 4) return launch_gemm_own<Fmt, MT, CAP >= 4 ? 4 : 1, PAIR>(a, s, name);
  if (CAP >= 3 && nb == 3) return launch_gemm_own<Fmt, MT, CAP >= 3 ? 3 : 1, PAIR>(a, s, name);
  if (CAP >= 2 && nb == 2) return launch_gemm_own<Fmt, MT, CAP >= 2 ? 2 : 1, PAIR>(a, s, name);
  return launch_gemm_own<Fmt, MT, 1, PAIR>(a, s, name);
}

struct OwnPlan { int mt, nb, slices, rounds; double us; };

// The row groups and channel blocks of a workgroup and the slices of K that come out shortest.  The constants (us a tile of a wave: its
// own, of a row group, of a channel block - its products, and its weights, which the row blocks share; of the second launch of a
// split) are fitted to measured launches: they order the choices.  64 rows, INT4, 11008 x 4096, blocks x slices: 1 x 1 23.5, 2 x 2
// 19.2, 4 x 4 20.5 us; 4096 x 11008: 1 block 29.3, 2 21.9, 3 14.5, 4 16.4; 4096 x 4096: 1 x 1 11.1, 1 x 2 16.3, 2 x 2 11.9, 4 x 4 13.4.
// A launch with a norm behind it takes a second kernel however K is cut (splitk_finish_norm_kernel in the norm kernel's place), so that
// slices cost it little more than their sums' bytes, and a workgroup of fewer features reads fewer bytes of X.  Up to 128 rows and a block
// a compute unit, by a grid of 3600 plans (12 shapes of 768 to 5120 channels, 9 to 128 rows, weights from HBM), launch and norm, us, with the plan of launches
// without a norm and with this: F143, 13696 x 4096, 64 rows 26.4 -> 23.4, 16 rows 18.4 -> 17.3, 16384 x 4096, 16 rows 23.3 ->
// 19.6; INT4, 8192 x 2048, 32 rows 10.8 -> 9.6, 4096 x 4096, 64 rows 13.9 -> 12.9, 3072 x 768, 32 rows 8.6 -> 7.2, 96 rows 9.9 -> 8.6; fp16, 11008 x 4096, 32 rows
// 29.0 -> 24.7, 2048 x 2048, 32 rows 9.1 -> 8.4.  9 to 16 rows only with 80 feature tiles and more (INT4 from 13 rows on): 4096 x 4096, 16 rows, F143
// 9.8 and 10.7, INT4 8.8 and 9.8; 11008 x 4096, 9 rows, INT4 12.9 and 13.5.  5120 x 5120 keeps the dearer estimate: 17 rows, INT4 12.0 and 13.4.
template <class Fmt, bool PAIR>
static OwnPlan plan_gemm_own(const GemmArgs& a) {
  constexpr double PRODUCTS = Fmt::kVec == 1 ? 0.48 : Fmt::kVec == 2 ? 0.6 : 0.7, WEIGHTS = Fmt::kVec == 1 ? 0.0 : Fmt::kVec == 2 ? 0.36 : 0.9;
  const int cus = device_compute_units();
  const int row_blocks = (a.M + 63) / 64;
  const int mt = ((a.M + 15) / 16 + row_blocks - 1) / row_blocks;
  const bool slices = !PAIR && a.count == 1 && a.part;
  // (of a die, which has its share of each slice's groups: 84 blocks in three slices are 33 workgroups for the 32 compute units of most; 6144 x 1336, 33 rows, F143 14.4 us
  // against 11.0 in two slices)
  auto die_rounds = [&](int nb, int sl) { return ((own_groups(a, nb, PAIR) + 7) / 8 * 8 * row_blocks * sl + cus - 1) / cus; };
  auto time = [&](int nb, int sl, bool normed, int& rounds) {
    const double rows = normed ? a.M / 16.0 / row_blocks : mt;         // groups of them that a workgroup reads
    const int tiles = ((a.KT + sl - 1) / sl + OWN_WAVES - 1) / OWN_WAVES;
    rounds = (own_groups(a, nb, PAIR) * row_blocks * sl + cus - 1) / cus;
    const int turns = normed ? die_rounds(nb, sl) : rounds;
    double us = 3.2 + turns * tiles * (0.5 + 0.29 * rows + (PRODUCTS + WEIGHTS / row_blocks) * nb * (PAIR ? 2 : 1));
    if (normed && OwnStreams<Fmt>::long_decode) us = 3.2 + turns * tiles * (0.13 * rows + 1.8 * nb);
    if (sl > 1) {
      const double size = (double)a.M * a.mat[0].N / 262144;
      us += normed ? sl * (0.35 + 0.5 * size) + (Fmt::kVec > 1 ? 1.0 : 0.8) : 2.7 * sl - 0.9 + (size > 1 ? 0.5 * sl * (size - 1) : 0.0);
    }
    return us;
  };
  auto room = [&](int sl) { return sl == 1 || (a.KT >= sl * OWN_WAVES && a.part_bytes >= (size_t)sl * a.M * a.mat[0].N * sizeof(float)); };
  OwnPlan best{mt, 1, 1, 0, 0.0};
  for (int nb = 1; nb <= own_cap<Fmt, PAIR>(mt); ++nb)
    for (int sl = 1; sl <= (slices && a.M > 16 ? GEMM_MAX_KSPLIT : 1) && room(sl); ++sl) {
      int rounds;
      const double us = time(nb, sl, false, rounds);
      if (best.rounds == 0 || us < best.us) best = OwnPlan{mt, nb, sl, rounds, us};
    }
  // (up to 128 rows and a block of channels a compute unit)
  if (!slices || !a.then || !a.then->any_order || a.M > 128 || a.mat[0].N > 16 * cus || !finish_norm_fits(a)) return best;
  // with a norm behind it: that plan, or one that is shorter by the other estimate.  F152's is one of its own, of blocks: their decoding bounds a workgroup, not its rows'
  // bytes (548 launches, rms 1 us; with the others' constants 8904 x 1584, 24 rows, 16.5 -> 19.8 us, 5632 x 3072, 17 rows, 16.0 -> 21.4), half a us shorter and of no fewer slices
  // (11008 x 2048, 100 rows, 1 x 1 33.5 against 2 x 2 31.3).
  best.us = time(best.nb, best.slices, true, best.rounds) - (OwnStreams<Fmt>::long_decode ? 0.5 : 0.0);
  if (a.M <= (Fmt::kVec == 1 ? 12 : 8) || (a.M <= 16 && a.KT < 80)) return best;
  const bool sliced = best.slices > 1;
  const int fewest = OwnStreams<Fmt>::long_decode ? best.slices : 1;
  // Not taken, though their estimates are shorter: beyond 64 rows four blocks, and four slices (INT4, 6144 x 4096, 80 rows, 4 x 2 16.0 against 2 x 1 15.4; 11008 x 2048, 112
  // rows, 4 x 3 18.2 against 2 x 2 16.9; F143, 16384 x 2048, 112 rows, 2 x 2 26.1 against 4 x 4 22.4, which is the plan without a norm); of fewer feature tiles, four blocks
  // and more in place of fewer with slices (INT4, 8192 x 4096, 40 rows, 4 x 4 14.6 against 2 x 2 14.0, 11008 x 4096, 20 rows 14.3 against 13.9, F143 8192 x 4096, 40 rows 17.1
  // against 16.5; 13696 x 4096 17.6 against 19.0), and of INT4 for up to 16 rows (11008 x 4096, 13 rows, 4 x 4 13.6 against 13.1); of 16-bit weights three blocks in their
  // place (6144 x 3072, 56 rows, 3 x 3 18.4 against 2 x 2 17.9).
  const int most = row_blocks > 1 || ((sliced || (Fmt::kVec == 1 && a.M <= 16)) && a.KT < (Fmt::kVec == 1 ? 96 : 80)) ? Fmt::kVec > 2 && sliced ? 2 : 3 : own_cap<Fmt, PAIR>(mt);
  for (int nb = 1; nb <= own_cap<Fmt, PAIR>(mt) && nb <= most; ++nb)
    for (int sl = fewest; sl <= (row_blocks > 1 ? 3 : GEMM_MAX_KSPLIT) && room(sl); ++sl) {
      if (die_rounds(nb, sl) > 1) break;          // (a second round begins with nothing on its way)
      int rounds;
      const double us = time(nb, sl, true, rounds);
      if (us < best.us) best = OwnPlan{mt, nb, sl, rounds, us};
    }
  return best;
}

template <class Fmt, bool PAIR>
static int launch_gemm_own_plan(const GemmArgs& a, const OwnPlan& p, hipStream_t s, const char* name) {
  GemmArgs b = a;
  b.ksplit = p.slices;
  const int rc = p.mt <= 1   ? launch_gemm_own_for<Fmt, 1, PAIR>(b, p.nb, s, name)
                 : p.mt == 2 ? launch_gemm_own_for<Fmt, 2, PAIR>(b, p.nb, s, name)
                 : p.mt == 3 ? launch_gemm_own_for<Fmt, 3, PAIR>(b, p.nb, s, name)
                             : launch_gemm_own_for<Fmt, 4, PAIR>(b, p.nb, s, name);
  if (rc) return rc;
  PTA_CHECK_LAUNCH(name);
  return PTA_OK;
}

// 33 to 128 rows by INT4 weights, several rounds of gemm_own_kernel: gemm_panel_kernel, if its plan is that much shorter (both plans' us a little long, the
// latter's begin with nothing on its way).  us, gemm_own_kernel and it, weights from HBM: three of 4096 x 4096, 65 rows 24.0 and 20.6, 128
// rows 28.1 and 24.9; pair of 4096 x 11008, 48 rows 25.4 and 22.5, 64 rows 29.3 and 25.8, 128 rows 42.3 and 36.3 (96 rows 35.7 and 36.0, plans 42.7 and 34.9);
// 4096 x 11008, 65 rows 21.3 and 20.2.  K of up to 2048 stays with gemm_own_kernel, which it has had; where the plans differ as much this would be the faster there too (pair
// of 2048 x 5632, 65 rows 16.9 and 12.8, 128 rows 19.6 and 15.2; 2048 x 12288, 65 rows 16.4 and 13.1; pair of 1792 x 10608, 114 rows 28.2 and 19.9).
template <class Fmt, bool PAIR>
static bool panel_before_own(const GemmArgs& a, const OwnPlan& own, PanelPlan& panel) {
  if constexpr (PanelFormat<Fmt>::ok && Fmt::kVec == 1) {
    if (a.M <= 32 || a.KT <= 16 || own.rounds < 2 || !panel_takes(a, PAIR)) return false;
    panel = plan_gemm_panel<Fmt, PAIR>(a);
    return panel.us < 0.8 * own.us;
  }
  return false;
}

// whether the launch fits gemm_tile_kernel with `per_wg` channel blocks per workgroup: every matrix
// a whole number of workgroups, enough feature tiles for the K groups
static inline bool tile_fits(const GemmArgs& a, int per_wg, int kq, bool pair) {
  if (a.KT < 2 * kq) return false;
  if (pair) return ((a.mat[0].N + 15) / 16) % per_wg == 0;
  for (int i = 0; i < a.count; ++i)
    if (((a.mat[i].N + 15) / 16) % per_wg != 0) return false;
  return true;
}

static inline int device_compute_units() {
  static int cus = 0;
  if (cus == 0) {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0)
      cus = n;
    else
      cus = 256;
  }
  return cus;
}

template <class Fmt, int NW, bool PAIR>
static void launch_gemv_lds(const GemmArgs& a, int total_nb, hipStream_t s) {
  const size_t xbytes = (((size_t)a.M * (a.KT * 128 + 8) * 2) + 15) & ~(size_t)15;
  const size_t smem = xbytes + (size_t)NW * (PAIR ? 2 : 1) * 256 * sizeof(float);
  gemm_kernel_taken = "gemv_lds_kernel";
  hipLaunchKernelGGL((gemv_lds_kernel<Fmt, NW, PAIR>), dim3(total_nb), dim3(NW * 64), smem, s, a);
}

template <class Fmt, int MT, bool PAIR>
static void launch_gemv(const GemmArgs& a, int total_nb, hipStream_t s) {
  // Waves per block: enough to split K finely when there are few channel blocks, fewer when
  // the grid alone already fills the machine.  The LDS reduction buffer caps the wide cases.
  // (more than 16 rows in 16 waves: F152 weights only, which go to gemm_own_kernel later than the others)
  constexpr bool FINE = !PAIR && (MT == 1 || (MT == 2 && OwnStreams<Fmt>::long_decode));
  gemm_kernel_taken = "gemv_mfma_kernel";
  if constexpr (FINE) {
    if (a.KT >= 16 && total_nb <= 1024) {
      hipLaunchKernelGGL((gemv_mfma_kernel<Fmt, MT, 16, PAIR>), dim3(total_nb), dim3(16 * 64), 0, s, a);
      return;
    }
  }
  constexpr int NW = MT == 4 && PAIR ? 4 : 8;
  hipLaunchKernelGGL((gemv_mfma_kernel<Fmt, MT, NW, PAIR>), dim3(total_nb), dim3(NW * 64), 0, s, a);
}

template <class Fmt, bool PAIR>
static int dispatch_gemv(const GemmArgs& a, int total_nb, hipStream_t s, const char* name);

// `chunk` rows at a time through the paths for so many
template <class Fmt, bool PAIR>
static int rows_in_turn(const GemmArgs& a, int chunk, int total_nb, hipStream_t s, const char* name) {
  for (int m0 = 0; m0 < a.M; m0 += chunk) {
    GemmArgs b = a;
    b.then = nullptr;
    b.M = a.M - m0 < chunk ? a.M - m0 : chunk;
    if (b.X) b.X += (size_t)m0 * a.K;
    for (int i = 0; i < a.count; ++i) {
      if (b.mat[i].X) b.mat[i].X += (size_t)m0 * a.K;
      if constexpr (Fmt::kWide) wide_skip_rows(b.mat[i], m0);
      else if (!PAIR || i == 0) b.mat[i].Y += (size_t)m0 * a.mat[i].N;
    }
    if (PAIR) b.mat[1].Y = b.mat[0].Y;
    if (b.epi.residual) b.epi.residual += (size_t)m0 * a.mat[0].N;
    if (b.epi.mul) b.epi.mul += (size_t)m0 * a.mat[0].N;
    const int rc = dispatch_gemv<Fmt, PAIR>(b, total_nb, s, name);
    if (rc) return rc;
  }
  return PTA_OK;
}

// More than 128 rows, 16-bit weights: whether one round of gemm_rows_kernel's workgroups (128 rows, and half the channels of
// gemm_block_kernel's) is the faster launch.  gemm_block_kernel's time follows the rows that its blocks hold, gemm_rows_kernel's does not,
// and with few tiles half the chip has none; a single weight's K can be split instead, a pair's cannot.  Ratios gemm_block_kernel to
// gemm_rows_kernel, weights from HBM, pairs 2048 x 2048 to 5632: 129 rows 0.95, 160 1.04, 200 1.17, 256 1.26, 320 1.1, 400 0.9, 512 1.14, 768
// 1.08, 1000 0.95; 8192 x 5632, 256 rows 1.26.  The fp32 epilogue adds to the former (it passes through LDS in one copy of the code): with K
// of 1024 1.03 to 1.31 (pairs) and 1.0 to 1.23 for up to 192 workgroups of the latter, 2048 x 6144, 512 rows 1.18.
// Single weights whose K is not split (no workspace, or several of them), 2048 to 12288 channels: fp16, K of 8192: 160 rows 0.9, 200 1.05 to
// 1.08, 250 1.2 to 1.26, 320 1.0, 384 1.2, 500 1.11 to 1.19, 742 1.1, 1000 1.12; of 4096: 200 1.0, 250 1.12 to 1.16, 320 0.96, 384 1.1, 500
// 1.06, 742 1.0 (1000 rows, 4096 channels, a workgroup a compute unit: 0.91); of 2048: 250 1.08, 384 1.05, 500 1.0.  bf16, K from 4096 on: 160 rows 0.95 to 1.0, 200 1.15, 250 1.3, 320 1.08, 384 1.28, 500
// 1.2, 742 1.13, 1000 1.11 to 1.19; of 2048: 129 1.04, 160 1.12, 200 1.26, 250 1.33, 320 1.18, 500 1.25 (2048 channels 0.95 to 0.99).
template <class Fmt, bool PAIR>
static bool rows_before_blocks(const GemmArgs& a, int total_nb, int cus) {
  if (Fmt::kVec < 4) return false;
  const int blocks = (a.M + 127) / 128, wgs = total_nb / (PAIR ? ROWS_CB / 2 : ROWS_CB) * blocks;
  if (wgs > cus) return false;
  const double held = a.M / (128.0 * blocks), line = 0.75 + 0.04 * (blocks - 2);
  const bool whole = !PAIR && (a.count > 1 || !a.part || a.part_bytes < 2 * (size_t)a.M * a.mat[0].N * sizeof(float));      // K is not split
  if (Fmt::kWide && a.KT <= 8) return PAIR || wgs <= cus * 3 / 4 || held >= line;
  if (Fmt::kWide && a.KT <= 16) return PAIR || (whole && wgs >= cus / 4) ? held >= line - 0.15 : wgs >= cus * 5 / 8 && held >= line;
  if (whole) {
    if (Fmt::kWide) return held >= 0.75 + 0.03 * (blocks - 2);
    if (a.KT < 24) return a.KT >= 16 && blocks <= 3 && held >= 0.9 && wgs >= cus / 4;
    return wgs <= cus * 3 / 4 && held >= (a.KT >= 48 ? 0.77 + 0.03 * (blocks - 2) : 0.85 + 0.02 * (blocks - 2));
  }
  return PAIR && held >= line;
}

// More than 64 rows: gemm_own_kernel where its workgroups are few rounds; beyond 128 rows gemm_block_kernel (16-bit and F143 weights) or
// gemm_panel_kernel (INT4, F152), and up to 128, or by rows_before_blocks, gemm_rows_kernel, where
// the channel blocks divide into their workgroup tiles; a single matrix with few channels also splits K when a workspace is at hand.  Otherwise
// the rows go through the smaller paths in turn, 64 at a time.
template <class Fmt, bool PAIR>
static int dispatch_many_rows(const GemmArgs& a, int total_nb, hipStream_t s, const char* name) {
  // One round of gemm_own_kernel's workgroups: it (us, against the kernels below; a launch of theirs takes 15 and more however small).
  // INT4: 4096 x 4096, 72 rows 11.4 against 23.1, 256 rows 18.3 against 37.5; 768 x 3072, 205 rows 8.8 against 24.7; 11008 x 4096,
  // 256 rows 36 against 49.  fp16: 768 x 3072, 205 rows 9.8 against 15.5; 2048 x 2048, 256 rows 11.2 against 19.4; F143 4096 x 4096,
  // 256 rows 20.6 against 29.6.  More rounds: to 128 rows two (4096 x 11008, 128 rows, INT4 29.8 against 40.9, F143 35.8 against 44.3,
  // fp16 44 against 47), of INT4 weights three (their pair of 11008 channels 41.5 against 48.0), and small launches (768 x 3072,
  // 512 rows, INT4 16.0 against 25.1); beyond, these lose: 4096 x 11008, 160 rows, INT4 42.8 against 39.8, fp16 60 against 44.  The plan's
  // time does not see what a round's begin and end take, so with short K the rounds are counted too: INT4 768 x 32000, 65 rows, four rounds
  // 26.8 against 21.3; pair 768 x 11008, three, 17.7 against 13.7; bf16 256 x 11008, 65 rows, two, 1.14 times; 512 x 4096, 1000 rows, four,
  // 1.14 times; 1024 x 6144, 768 rows, five, 1.10.  And 16-bit weights of long K, two rounds: 8192 x 8192, 65 to 128 rows, 1.08 to 1.18 times,
  // 11008 x 8192 1.2 to 1.34 (4096 x 8192 0.83 to 0.97).
  PanelPlan panel{};                              // (made where it is first asked for)
  const bool paneled = PanelFormat<Fmt>::ok && a.M > 128 && panel_takes(a, PAIR);
  auto panel_plan = [&]() -> const PanelPlan& {
    if (panel.rg == 0) panel = plan_gemm_panel<Fmt, PAIR>(a);
    return panel;
  };
  if (a.epi.norm == PTA_NORM_NONE) {
    const OwnPlan plan = plan_gemm_own<Fmt, PAIR>(a);
    const int most = a.M <= 128 ? ((Fmt::kWide && a.KT <= 2) || (Fmt::kVec > 2 && a.KT >= 56) ? 1 : Fmt::kVec == 1 && a.KT >= 12 ? 3 : 2) : a.KT >= 8 || PAIR ? 4 : 3;
    // (a round after the first begins with nothing on its way: 3.6 us more than the plan says; 768 rows of three 1024 x 1024 21.5 against gemm_panel_kernel's 20.8,
    // 1200 rows 27.8 against 21.3, the pair of 1024 x 2816, 640 rows 25.1 against 20.4; two rounds, and short K, stay)
    bool own = plan.rounds == 1 || (plan.rounds <= most && (a.M <= 128 || plan.us <= (Fmt::kVec == 1 ? 22.0 : 11.0)));
    if (own && a.M > 128) own = !(paneled && a.KT >= 8 && plan.rounds > 2 && plan.us + 3.6 * (plan.rounds - 1) > 1.2 * panel_plan().us);
    if constexpr (PanelFormat<Fmt>::ok) {
      if (own && a.M <= 128 && panel_before_own<Fmt, PAIR>(a, plan, panel)) return launch_gemm_panel_plan<Fmt, PAIR>(a, panel, s, name);
    }
    if (own) return launch_gemm_own_plan<Fmt, PAIR>(a, plan, s, name);
  }
  const int cus = device_compute_units();
  const int per_wg = PAIR ? 4 : 8;
  // (few features: the wide formats only, whose other path would take 64 rows per launch)
  const bool tiles = a.epi.norm == PTA_NORM_NONE && tile_fits(a, per_wg, Fmt::kWide ? 0 : 2, PAIR);
  // More than 128 rows (measured on whole prompt passes of the 7B shape, gemm_rows_kernel against this: 6.5 against
  // 7.2 ms at 128 rows, 7.7 against 7.3 at 192, 8.1 against 7.5 at 256): 128-row panels through LDS, the weights
  // straight into registers.
  // Formats with a form of gemm_block_kernel: launches of more than 128 rows.  Measured against the kernels they had before (us):
  // FP8, 1000 rows: 4096 x 2 x 13696 pair 500 -> 198, 13696 x 4096 311 -> 110, 4096 x 4608 145 -> 60 (gemm_panel_kernel, whose two
  // vectors per tile spill); bf16, 2048 rows: 4096 x 4096 102 -> 70, 11008 x 4096 261 -> 190; fp16 4096 x 2 x 11008 pair, 2048
  // rows 564 -> 326, 512 rows 176 -> 103, 160 rows 83 -> 60 (gemm_rows_kernel).  At 65 to 128 rows the pair and 11008 features
  // lose (0.75 to 0.9) what small matrices win (1.3): those stay.
  if constexpr (BlockFormat<Fmt>::ok) {
    if (a.M > 128 && a.epi.norm == PTA_NORM_NONE && !(tiles && rows_before_blocks<Fmt, PAIR>(a, total_nb, cus)))
      return dispatch_gemm_block<typename BlockFormat<Fmt>::type, PAIR>(a, s, name);
  }
  if constexpr (PanelFormat<Fmt>::ok) {
    if (paneled) return launch_gemm_panel_plan<Fmt, PAIR>(a, panel_plan(), s, name);
  }
  if (tiles) {
    // fragments in registers, weights through LDS: 256 rows per workgroup where that still fills the machine,
    // else 128; few workgroups and one matrix: K in slices as well
    const int groups = total_nb / per_wg;
    const bool two = !BlockFormat<Fmt>::ok && a.M > 128 && (long)groups * ((a.M + 255) / 256) * 2 >= (long)cus;
    const int wgs = groups * (two ? (a.M + 255) / 256 : (a.M + 127) / 128);
    GemmArgs b = a;
    int nsl = wgs > 0 ? cus / wgs : 1;
    nsl = nsl > GEMM_MAX_KSPLIT ? GEMM_MAX_KSPLIT : nsl;
    while (nsl > 1 && a.KT < nsl * 8) --nsl;
    if (!PAIR && a.count == 1 && a.part && nsl > 1 && a.part_bytes >= (size_t)nsl * a.M * a.mat[0].N * sizeof(float)) b.ksplit = nsl;
    int rc;
    if constexpr (BlockFormat<Fmt>::ok) rc = launch_gemm_rows<Fmt, 1, PAIR>(b, total_nb, s, name);
    else rc = two ? launch_gemm_rows<Fmt, 2, PAIR>(b, total_nb, s, name) : launch_gemm_rows<Fmt, 1, PAIR>(b, total_nb, s, name);
    if (rc) return rc;
    PTA_CHECK_LAUNCH(name);
    return PTA_OK;
  }
  return rows_in_turn<Fmt, PAIR>(a, 64, total_nb, s, name);
}

// 5 to 16 rows without a norm: gemm_own_kernel, or (false) gemv_wide_kernel and gemv_stream_kernel.  Where its workgroups are one round and
// there are 16 feature tiles and more.  gemv_wide_kernel takes 16 or 32 tiles a step and is at its best where they fill its steps (K about
// 4096, 8192, 12288); gemm_own_kernel's lead grows with the rows and with K.  Ratios of its time to theirs, K of 2048 to 13696 by 1024 to
// 12288 channels, medians of runs in turn, weights from HBM and from the last cache alike:
//   9 to 16 rows: INT4 0.71 to 1.05.  F143 0.74 to 1.02; K of 3300 to 5000, and more than two blocks a compute unit, from 12 rows on 0.88 to
//   1.01 (9 rows 1.08).  16-bit weights, up to a block a compute unit (4096 x 12288 1.06): 0.79 to 1.04; K of 3300 to 5000 from 16 rows on
//   0.92 to 1.02 (14 rows 1.08, 9 rows 1.14), about 8192 and 12288 from 12 rows on 0.91 to 1.01 (9 rows 1.06).  Pairs 0.81 to 1.04; K of
//   3300 to 5000 from 14 rows on (9 rows 1.12).
//   7 and 8 rows, K past 5120 (pairs and 16-bit weights 6000): 0.83 to 1.02; not 16-bit and single F143 weights about 8192 and 12288 (1.05 to
//   1.07).
//   5 and 6 rows: K from 8192 on INT4 0.89 to 0.99, from 10240 on F143 and pairs 0.87 to 1.02 (8192 1.07); not 16-bit weights.
//   5 to 8 rows, INT4: short K and pairs of up to two blocks a compute unit 0.89 to 1.02 (2048 x 11008 1.11), single weights of more than
//   four blocks a compute unit (4096 x 24576 0.84).
//   F152 (16 instructions a decoded operand): 9 rows and more, K up to 3072, two blocks a compute unit 0.74 to 1.0; else up to 1.21.
template <class Fmt, bool PAIR>
static bool own_takes_few_rows(const GemmArgs& a, int total_nb, int cus, bool one_round) {
  const int KT = a.KT;
  if (a.prefer_stream || !one_round || KT < 16 || a.K >= GEMM_FAR) return false;
  if (OwnStreams<Fmt>::long_decode) return a.M > 8 && !PAIR && KT <= 24 && total_nb <= 2 * cus;
  if (Fmt::kVec > 2 && (PAIR || total_nb > cus)) return false;
  const bool full = KT > 40 && ((KT + 4) & 31) <= 8;         // whole steps of gemv_wide_kernel, or nearly
  if (a.M <= 8) {
    if (Fmt::kVec == 1 && (PAIR ? KT <= 24 && total_nb <= 2 * cus : total_nb > 4 * cus)) return true;
    if (a.M <= 6) return Fmt::kVec == 1 && !PAIR ? KT >= 64 : Fmt::kVec <= 2 && KT >= 80 && (PAIR || !full);
    return KT > (PAIR || Fmt::kVec > 2 ? 47 : 40) && (Fmt::kVec == 1 || PAIR || !full);
  }
  const bool middle = KT > 24 && KT < 40;
  if (Fmt::kVec > 2) return a.M >= (middle ? 16 : full ? 12 : 9);
  if (PAIR) return !middle || a.M >= 14;
  return Fmt::kVec == 1 || a.M >= 12 || (!middle && total_nb <= 2 * cus);
}

// 17 to 32 rows by single F152 weights over one X: gemv_wide_kernel, whose 16 waves decode side by side where gemm_own_kernel has eight, as
// long as its workgroups (of up to three blocks) are one round and K is not split.  Ratios of its time to that of the other kernels
// (gemm_own_kernel, gemm_tile_kernel, up to 3072 features gemv_mfma_kernel), weights from HBM, 496 to 11008 channels: 1920 features 0.83 to
// 1.05, 2048 0.82 to 0.98, 3072 0.76 to 0.95, 4096 to 13696 0.86 to 0.99; 1536 to 1792 with a block a compute unit 0.94 to 1.02, with more
// 0.86 to 1.17; 1024 0.91 to 1.12; 29 rows and more, a block a compute unit, 5120 features 1.0, 8192 and more 1.03 to 1.09.  Two rounds: 14336
// and 16384 channels 1.17 to 1.35, 32000 1.13 to 1.28 (20480 0.77 to 0.92).  K in slices: 11008 x 1000 to 4104 1.07 to 1.55.
static inline bool wide_takes_some_rows(const GemmArgs& a, int total_nb, int cus, int blocks, bool split) {
  return a.M > 16 && a.M <= 32 && a.KT >= (total_nb <= cus ? 12 : 15) && !split && total_nb <= blocks * cus && !(a.M > 28 && a.KT > 40 && total_nb <= cus);
}

template <class Fmt, bool PAIR>
static int dispatch_gemv(const GemmArgs& a, int total_nb, hipStream_t s, const char* name) {
  if (a.M > 16 && a.K >= GEMM_FAR && a.epi.norm == PTA_NORM_NONE) return rows_in_turn<Fmt, PAIR>(a, 16, total_nb, s, name);
  if (a.M > 64) return dispatch_many_rows<Fmt, PAIR>(a, total_nb, s, name);
  const size_t xbytes = (size_t)a.M * (a.KT * 128 + 8) * 2;
  bool all_shared_x = true;
  for (int i = 0; i < a.count; ++i) all_shared_x = all_shared_x && a.mat[i].X == nullptr;
  const bool norm_small = a.M <= 4 && xbytes <= 40 * 1024;
  const bool norm_wide = a.M <= 16 && all_shared_x && a.KT >= 8;
  if (a.epi.norm != PTA_NORM_NONE && !norm_small && !norm_wide) {
    pta_set_error("%s: the fused norm needs M <= 4 with M*K <= 20480, or M <= 16 with one shared X and K >= 1024 "
                  "(got M=%d K=%d)", name, a.M, a.K);
    return PTA_EUNSUPPORTED;
  }
  if (a.M <= 4 && xbytes <= 40 * 1024) {
    if (a.KT >= 16 && total_nb <= 1024 && !PAIR) launch_gemv_lds<Fmt, 16, PAIR>(a, total_nb, s);
    else launch_gemv_lds<Fmt, 8, PAIR>(a, total_nb, s);
  } else {
    const int cus = device_compute_units();
    const int per_cu = (total_nb + cus - 1) / cus;
    const int mt = (a.M + 15) / 16;
    if (a.epi.norm == PTA_NORM_NONE && a.M > 4) {
      // gemm_own_kernel or gemm_tile_kernel (up to 16 rows: own_takes_few_rows).  Both sides in us, INT4 unless named.
      // One round of gemm_own_kernel's workgroups: it.  64 rows, 4096 x 11008: 14.5 against 21.8, 4096 x 4096 11.1 against 15.2,
      // 2048 x 2048 7.1 against 11.8; 32 rows 11.1 against 14.3, 8.0 against 11.2, 5.6 against 9.4; F143, 64 rows, 4096 x 4096
      // 11.9 against 16.2; bf16 14.5 against 18.2; with odd channel counts, which gemm_tile_kernel cannot take, 1000 channels at
      // 64 rows 9.6 against 19.5.
      // Several rounds: each begins with nothing on its way.  Weights of one vector a tile lose a little (32000 channels, 64 rows
      // 32.4 against 31.4), those of two win beyond 32 rows (F143 41.8 against 51.6), so does a pair of either (11008 channels, 64
      // rows 29.2 against 39.7; F143 40.8 against 46.9), fp16 ones lose (72.5 against 68.3).  Pairs of up to 32 rows: INT4, one round and
      // K of 3072 and more (11008 channels, 32 rows 16.9 against 21.5; 2048 x 5632 9.1 against 8.9).
      const int wgs4 = total_nb / (PAIR ? 2 : 4);
      const OwnPlan plan = plan_gemm_own<Fmt, PAIR>(a);
      const bool one_round = plan.rounds == 1;
      bool own, tile = false;
      if (a.M <= 16) {
        own = own_takes_few_rows<Fmt, PAIR>(a, total_nb, cus, one_round);
      } else {
        tile = tile_fits(a, PAIR ? 2 : 4, 4, PAIR) && 2 * wgs4 >= cus;
        constexpr bool F152 = OwnStreams<Fmt>::long_decode;
        if (tile && PAIR) own = mt > 2 ? Fmt::kVec <= 2 && !(F152 && a.KT <= 16 && wgs4 <= cus) : Fmt::kVec == 1 && one_round && a.KT >= 24;
        else if (tile) own = one_round || (mt > 2 && Fmt::kVec == 2);
        // Launches that gemm_tile_kernel cannot take (odd numbers of blocks, few of them, few feature tiles): gemm_own_kernel or
        // gemv_mfma_kernel, whose workgroups of one block come and go.  Few feature tiles, more than 32 rows: a wave has one or none, and
        // the end is all (us, 33 rows: 128 features 1.17 times; pairs 256 x 1024 fp16 4.4 against 5.5, 768 x 11008 13.3 against 19.0, F143 11.8
        // against 16.2; 768 x 2048 it wins).  Up to 32 rows, against the kernel before them: 16-bit pairs of several rounds 1024 x 5608 0.88
        // and 1.19, 2048 x 5608 0.93 and 1.09, 3072 x 5608 0.96 and 1.0, one round of 1024 features 0.92 and 1.03; F152 singles 1024 x 4104
        // 0.9 and 1.1, pairs 2048 x 4104 0.73 and 0.99, 4096 x 2056 0.97 and 0.9.
        else if (mt > 2) own = PAIR ? a.KT >= 8 || (one_round && a.KT > 4) : a.KT > 2;
        else if (F152) own = a.KT > (PAIR ? 16 : 24) && (!PAIR || total_nb <= cus);
        else own = a.KT >= 8 && !(PAIR && Fmt::kVec > 2 && (a.KT == 8 || (!one_round && a.KT < 24)));
      }
      if constexpr (OwnStreams<Fmt>::long_decode && !PAIR) {
        if (all_shared_x && wide_takes_some_rows(a, total_nb, cus, wide_cap<Fmt, PAIR>(), plan.slices > 1)) {
          const int rc = launch_gemv_wide_for<Fmt, 2, PAIR, false>(a, total_nb, per_cu, s, name);
          if (rc) return rc;
          PTA_CHECK_LAUNCH(name);
          return PTA_OK;
        }
      }
      if constexpr (PanelFormat<Fmt>::ok) {
        PanelPlan panel;
        if (own && panel_before_own<Fmt, PAIR>(a, plan, panel)) return launch_gemm_panel_plan<Fmt, PAIR>(a, panel, s, name);
      }
      if (own) return launch_gemm_own_plan<Fmt, PAIR>(a, plan, s, name);
      int rc = 1;
      if (tile) {
        // What bounds these launches is the bytes through the busiest compute unit: a workgroup reads all rows of X
        // beside its weights.  More workgroups than compute units (20480 channels: 320 of 64 channels): workgroups
        // of 16 waves and 128 channels where their rounds come out shorter - 160 of 768 KiB against two rounds of
        // 640 at 64 rows.  INT4, weights from HBM: 4096 x 20480, 64 rows 28.0 against 41.9 us, 48 rows 26.6 against 40.3; 4096 x
        // 32000, 64 rows 32.0 against 44.9, 32 rows 23.3 against 24.3, 17 rows 21.8 against 22.4; F143, 4096 x 20480, 32 rows 27.5
        // against 28.4.
        bool wide = false;
        if constexpr (!PAIR && Fmt::kVec <= 2) {
          // (beyond 32 rows with INT4 weights only: with two vectors per tile the 16 waves' registers do not hold it)
          if (tile_fits(a, 8, 4, false) && wgs4 > cus && (a.M <= 32 || Fmt::kVec == 1)) {
            const double xb = (double)a.M * a.K * 2, wb = (double)a.KT * Fmt::kVec * 1024;
            const int wgs_wide = total_nb / 8;
            wide = ((wgs_wide + cus - 1) / cus) * (xb + 8 * wb) < ((wgs4 + cus - 1) / cus) * (xb + 4 * wb);
          }
          if (wide) {
            if (a.M <= 32) rc = launch_gemm_tile<Fmt, 2, 4, false, 16>(a, total_nb, s, name);
            else if constexpr (Fmt::kVec == 1) rc = launch_gemm_tile<Fmt, 4, 4, false, 16>(a, total_nb, s, name);
          }
        }
        if (!wide && a.M <= 32) rc = launch_gemm_tile<Fmt, 2, 4, PAIR>(a, total_nb, s, name);
        else if constexpr (PAIR ? Fmt::kVec > 2 || OwnStreams<Fmt>::long_decode : Fmt::kVec != 2) {
          if (!wide) rc = launch_gemm_tile<Fmt, 4, 4, PAIR>(a, total_nb, s, name);
        }
      }
      if (rc < 0) return rc;
      if (rc == 0) { PTA_CHECK_LAUNCH(name); return PTA_OK; }
    }
    if (all_shared_x && a.M <= 16 && a.KT >= 8) {
      int rc;
      bool streamed = false;
      if constexpr (Fmt::kVec * (PAIR ? 2 : 1) <= 4) {
        // gemv_stream_kernel where gemv_wide_kernel's rounds of workgroups come out longer than an even share of the
        // blocks (856 blocks: 286 workgroups of 3 = two rounds = 6 block times, against 4), or on request
        if (stream_fits(a) && total_nb >= cus && (a.prefer_stream || wide_block_times<Fmt, PAIR>(total_nb, per_cu) > per_cu)) {
          rc = launch_gemv_stream<Fmt, PAIR>(a, total_nb, cus, s, name);
          streamed = true;
        }
      }
      if (streamed) {}
      else if (a.epi.norm != PTA_NORM_NONE) rc = launch_gemv_wide_for<Fmt, 1, PAIR, true>(a, total_nb, per_cu, s, name);
      else rc = launch_gemv_wide_for<Fmt, 1, PAIR, false>(a, total_nb, per_cu, s, name);
      if (rc) return rc;
    } else if (a.M <= 16) launch_gemv<Fmt, 1, PAIR>(a, total_nb, s);
    else if (a.M <= 32) launch_gemv<Fmt, 2, PAIR>(a, total_nb, s);
    else launch_gemv<Fmt, 4, PAIR>(a, total_nb, s);
  }
  PTA_CHECK_LAUNCH(name);
  return PTA_OK;
}

static inline int check_gemv_common(const char* name, const void* X, int M, int K) {
  PTA_REQUIRE(X, "%s: null X", name);
  PTA_REQUIRE(M >= 1 && M <= GEMM_MAX_ROWS, "%s: M must be in [1, %d], got %d", name, GEMM_MAX_ROWS, M);
  PTA_REQUIRE(K > 0 && (K % 8) == 0, "%s: K must be a positive multiple of 8, got %d", name, K);
  PTA_REQUIRE(pta_aligned(X, 16), "%s: X must be 16-byte aligned", name);
  return PTA_OK;
}

static inline size_t gemv_tiled_bytes(int N, int K, int kvec) {
  if (N <= 0 || K <= 0) return 0;
  return (size_t)((N + 15) / 16) * (size_t)((K + 127) / 128) * 1024 * kvec;
}
