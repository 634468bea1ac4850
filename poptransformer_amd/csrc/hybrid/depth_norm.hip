// The end of a layer whose result takes a normed addition and is then averaged with the residuals of all depths before it, with the
// next layer's norm and routing in the same launch; and the step before: a mixture's parts added to the residual.
#include "attention.h"
#include "routing.h"

typedef pta_depth_norm_args DN;

// Row r by a workgroup; a thread owns the columns c, c + 4 * THREADS, ... (four at a time) from the result to h.  y: the row of the result, or null;
// u_row: LDS, h_ld floats, the average, then what h holds.
template <typename T, int THREADS>
__device__ __forceinline__ void depth_row(const DN& a, int r, const float* y, float* u_row) {
  constexpr int WAVES = THREADS / 64;
  __shared__ float red[3][WAVES];
  __shared__ float z[ROUTE_FLOATS];
  const int d = a.width;
  const bool vec = (d & 3) == 0;
  const int span = vec ? 4 : 1, step = THREADS * span, first = threadIdx.x * span;
  T* h = reinterpret_cast<T*>(a.h) + (size_t)r * a.h_ld;
  const float* base = a.history + (size_t)r * d;
  float* newest = a.history + (size_t)(a.depth > 0 ? a.depth - 1 : 0) * a.depth_stride + (size_t)r * d;
  float* next = a.next ? a.next + (size_t)r * d : nullptr;
  const T* row = nullptr;
  if (a.table) {
    int col = a.ids_index ? *a.ids_index : 0;
    col = col < 0 ? 0 : (col >= a.ids_stride ? a.ids_stride - 1 : col);
    int id = a.ids[(size_t)r * a.ids_stride + col];
    id = id < 0 ? 0 : (id >= a.vocab ? a.vocab - 1 : id);
    row = reinterpret_cast<const T*>(a.table) + (size_t)id * d;
    if (a.pos_out && threadIdx.x == 0) a.pos_out[r] = a.ids_index ? *a.ids_index : 0;
    if (a.side) {                                            // the token's parts of all layers, one behind the other
      const T* e = reinterpret_cast<const T*>(a.side_table) + (size_t)id * a.side_layers * a.side_ld;
      for (int c = threadIdx.x * 8; c < a.side_layers * a.side_ld; c += THREADS * 8) {
        float v[8];
        load8(e + c, true, 8, v);
        store8(reinterpret_cast<T*>(a.side) + (size_t)(c / a.side_ld) * a.side_stride + (size_t)r * a.side_ld + c % a.side_ld, v);
      }
    }
  }
  float inv = 0.f;
  if (y) {
    float sq = 0.f;
    if (vec) {
      for (int c = first; c < d; c += step) {
        const f32x4 t = *reinterpret_cast<const f32x4*>(y + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) sq = __builtin_fmaf(t[e], t[e], sq);
      }
    } else {
      for (int c = first; c < d; c += step) sq = __builtin_fmaf(y[c], y[c], sq);
    }
    inv = 1.0f / sqrtf(workgroup_sum<WAVES>(sq, red[0]) / (float)d + a.eps);
  }
  float sum = 0.f;
  auto column = [&](auto width_tag, int c) {
    constexpr int V = decltype(width_tag)::value;
    auto load = [&](const float* p, float (&v)[V]) {
      if constexpr (V == 4) {
        const f32x4 t = *reinterpret_cast<const f32x4*>(p + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = t[e];
      } else {
        v[0] = p[c];
      }
    };
    auto store = [&](float* p, const float (&v)[V]) {
      if constexpr (V == 4) *reinterpret_cast<f32x4*>(p + c) = f32x4{v[0], v[1], v[2], v[3]};
      else p[c] = v[0];
    };
    float v[V], u[V] = {};
    if (row) {
#pragma unroll
      for (int e = 0; e < V; ++e) u[e] = (float)row[c + e] * a.embed_scale;
      store(newest, u);
    } else {
      load(newest, v);
      constexpr int AHEAD = 8;                               // depths requested together
      for (int j0 = 0; j0 < a.depth - 1; j0 += AHEAD) {
        float t[AHEAD][V];
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) load(base + (size_t)(j0 + j < a.depth - 1 ? j0 + j : j0) * a.depth_stride, t[j]);
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
          const float f = j0 + j < a.depth - 1 ? a.weights[j0 + j] : 0.f;
#pragma unroll
          for (int e = 0; e < V; ++e) u[e] = __builtin_fmaf(f, t[j][e], u[e]);
        }
      }
      if (y) {
        float t[V], w[V];
        load(y, t);
        load(a.y_weight, w);
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] += t[e] * inv * w[e];
        store(newest, v);
      }
      const float f = a.weights ? a.weights[a.depth - 1] : 1.0f;
#pragma unroll
      for (int e = 0; e < V; ++e) u[e] = __builtin_fmaf(f, v[e], u[e]);
    }
    if (next) store(next, u);
#pragma unroll
    for (int e = 0; e < V; ++e) {
      u_row[c + e] = u[e];
      sum += u[e];
    }
  };
  if (vec) for (int c = first; c < d; c += step) column(std::integral_constant<int, 4>{}, c);
  else for (int c = first; c < d; c += step) column(std::integral_constant<int, 1>{}, c);
  const float mean = a.centred ? workgroup_sum<WAVES>(sum, red[1]) / (float)d : 0.f;
  float sq = 0.f;
  for (int c = first; c < d; c += step)
    for (int e = 0; e < span; ++e) {
      const float t = u_row[c + e] - mean;
      sq = __builtin_fmaf(t, t, sq);
    }
  const float f = 1.0f / sqrtf(workgroup_sum<WAVES>(sq, red[2]) / (float)d + a.eps);
  if (vec && (a.h_ld & 3) == 0) {
    typedef T vecT __attribute__((ext_vector_type(4)));
    for (int c = first; c < d; c += step) {
      const f32x4 u = *reinterpret_cast<const f32x4*>(u_row + c), w = *reinterpret_cast<const f32x4*>(a.norm_weight + c);
      vecT o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[e] = (T)((u[e] - mean) * f * w[e]);
        u_row[c + e] = (float)o[e];
      }
      *reinterpret_cast<vecT*>(h + c) = o;
    }
  } else {
    for (int c = first; c < d; c += step)
      for (int e = 0; e < span; ++e) {
        const T o = (T)((u_row[c + e] - mean) * f * a.norm_weight[c + e]);
        h[c + e] = o;
        u_row[c + e] = (float)o;
      }
  }
  for (int c = d + threadIdx.x; c < a.h_ld; c += THREADS) h[c] = (T)0.0f;
  if (!a.router) return;
  router_logits<T, WAVES>(a.router, a.h_ld, d, u_row, a.routing, z);
  route_row<THREADS>(a.routing, z, r, threadIdx.x, true);
}

template <typename T, int THREADS>
__global__ __launch_bounds__(THREADS) void depth_norm_kernel(DN a) {
  extern __shared__ __align__(16) float u_row[];
  depth_row<T, THREADS>(a, blockIdx.x, a.y ? a.y + (size_t)blockIdx.x * a.width : nullptr, u_row);
}

static int check_depth_norm(const DN& a, const char* name) {
  PTA_REQUIRE(a.dtype == PTA_BF16 || a.dtype == PTA_FP32, "%s: unknown type %d", name, a.dtype);
  PTA_REQUIRE(a.rows > 0 && a.width > 0 && a.width <= 14000, "%s: rows %d, width %d (1 .. 14000)", name, a.rows, a.width);
  PTA_REQUIRE(a.history && pta_aligned(a.history, 16) && a.depth_stride >= (size_t)a.rows * a.width && a.depth_stride % 4 == 0 && pta_aligned(a.next, 16),
              "%s: the history is missing, unaligned, or too narrow", name);
  PTA_REQUIRE(a.h && pta_aligned(a.h, 16) && a.h_ld >= a.width && a.h_ld <= a.width + 7 && a.norm_weight && pta_aligned(a.norm_weight, 16),
              "%s: h or its norm's weight null or unaligned, h rows of %d", name, a.h_ld);
  PTA_REQUIRE(a.table ? (a.ids && a.vocab > 0 && a.ids_stride > 0 && a.depth == 0 && !a.y) : (a.depth >= 1 && (a.weights || a.depth == 1)),
              "%s: either an embedding with ids, or depths with their weights", name);
  PTA_REQUIRE(!a.y || (a.y_weight && pta_aligned(a.y, 16) && pta_aligned(a.y_weight, 16)), "%s: unaligned result, or without its norm's weight", name);
  PTA_REQUIRE(!a.side || (a.table && a.side_table && a.side_layers > 0 && a.side_ld > 0 && a.side_ld % 8 == 0 && pta_aligned(a.side, 16) &&
                          pta_aligned(a.side_table, 16) && a.side_stride % 8 == 0 && a.side_stride >= (size_t)a.rows * a.side_ld),
              "%s: the tokens' own parts (%d layers of %d) do not fit", name, a.side_layers, a.side_ld);
  if (a.router) {
    const int rc = check_routing(a.routing, name);
    if (rc) return rc;
    PTA_REQUIRE(a.h_ld % 8 == 0 && pta_aligned(a.router, 16), "%s: a router reads h, in whole pieces of eight", name);
  }
  return PTA_OK;
}

extern "C" int pta_depth_norm(const DN* args, pta_stream_t stream) {
  const char* name = "pta_depth_norm";
  PTA_REQUIRE(args, "%s: null arguments", name);
  const DN& a = *args;
  const int rc = check_depth_norm(a, name);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  const size_t smem = (size_t)a.h_ld * sizeof(float);
  // few rows: a whole row of 1024 threads shortens the chain of a row; many rows: the machine is full either way
  auto launch = [&](auto threads) {
    constexpr int N = decltype(threads)::value;
    if (a.dtype == PTA_BF16) hipLaunchKernelGGL((depth_norm_kernel<bf16, N>), dim3(a.rows), dim3(N), smem, s, a);
    else hipLaunchKernelGGL((depth_norm_kernel<float, N>), dim3(a.rows), dim3(N), smem, s, a);
  };
  if (a.rows <= 64 && a.width >= 2048) launch(std::integral_constant<int, 1024>{});
  else launch(std::integral_constant<int, 256>{});
  PTA_CHECK_LAUNCH(name);
  return PTA_OK;
}

// columns c to c + 7 of row r of x with the weighted parts (zeros past the width)
template <typename T>
__device__ __forceinline__ void with_parts(const pta_add_parts_args& a, size_t r, int c, float (&v)[8]) {
  const int left = a.width - c;
  const bool vec = left >= 8 && (a.width & 7) == 0;
  load8(a.x + r * a.width + c, vec, left, v);
  if (a.parts) {
    const size_t at = r * a.parts_ld * a.width + c;
    const float* w = a.part_weight + r * a.weights_ld;
#pragma unroll 4
    for (int p = 0; p < a.n_parts; ++p) {
      float t[8];
      if (a.part_f32) load8(reinterpret_cast<const float*>(a.parts) + at + (size_t)p * a.width, vec, left, t);
      else load8(reinterpret_cast<const T*>(a.parts) + at + (size_t)p * a.width, vec, left, t);
      const float f = w[p];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = __builtin_fmaf(f, t[e], v[e]);
    }
  }
}
__device__ __forceinline__ void store_sum(const pta_add_parts_args& a, size_t r, int c, const float (&v)[8]) {
  const int left = a.width - c;
  float* x = a.x + r * a.width + c;
  if (left >= 8 && (a.width & 7) == 0) store8(x, v);
  else for (int e = 0; e < 8 && e < left; ++e) x[e] = v[e];
}

// Eight columns of a row per thread: x += the weighted parts, h = x.
template <typename T>
__global__ __launch_bounds__(256) void add_parts_kernel(pta_add_parts_args a, int pieces) {
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t r = idx / pieces;
  if (r >= (size_t)a.rows) return;
  const int c = (int)(idx % pieces) * 8;
  float v[8];
  with_parts<T>(a, r, c, v);
  if (a.parts) store_sum(a, r, c, v);
  store8(reinterpret_cast<T*>(a.h) + r * a.h_ld + c, v);        // (zeros past the width)
}

static int check_add_parts(const pta_add_parts_args& a, const char* name) {
  PTA_REQUIRE(a.dtype == PTA_BF16 || a.dtype == PTA_FP32, "%s: unknown type %d", name, a.dtype);
  PTA_REQUIRE(a.rows > 0 && a.width > 0 && a.x && a.h && pta_aligned(a.x, 16) && pta_aligned(a.h, 16) && a.h_ld == (a.width + 7) / 8 * 8,
              "%s: rows %d, width %d, h rows of %d", name, a.rows, a.width, a.h_ld);
  PTA_REQUIRE(!a.parts || (a.n_parts >= 1 && a.parts_ld >= a.n_parts && a.part_weight && a.weights_ld >= a.n_parts && pta_aligned(a.parts, 16)),
              "%s: %d parts of %d", name, a.n_parts, a.parts_ld);
  return PTA_OK;
}

extern "C" int pta_add_parts(const pta_add_parts_args* args, pta_stream_t stream) {
  const char* name = "pta_add_parts";
  PTA_REQUIRE(args, "%s: null arguments", name);
  const pta_add_parts_args& a = *args;
  const int rc = check_add_parts(a, name);
  if (rc) return rc;
  const int pieces = a.h_ld / 8;
  const dim3 grid((unsigned)(((size_t)a.rows * pieces + 255) / 256));
  if (a.dtype == PTA_BF16) hipLaunchKernelGGL((add_parts_kernel<bf16>), grid, dim3(256), 0, (hipStream_t)stream, a, pieces);
  else hipLaunchKernelGGL((add_parts_kernel<float>), grid, dim3(256), 0, (hipStream_t)stream, a, pieces);
  PTA_CHECK_LAUNCH(name);
  return PTA_OK;
}

// ------------------------------------------------------------------------------------------
// The whole end of a layer of few bf16 rows as one launch: the parts added, the token's gate (gelu, times its own part), the projection of it, and
// depth_row.  Four launches of it took what their chain takes (one row of 2048: 3.8, 4.6, 3.5 and 5.0 us, an empty one 1.9), each a few KiB.  Here their
// workgroups are one grid in the order of the chain: a workgroup's ticket is its place in it, it requests its weights, and what it waits
// for is written by workgroups with smaller tickets, which have started before it - no launch has to fit the machine as a whole.
//
// A value travels as a word that holds the launch's number beside it (16 bits beside a bf16 one, 32 beside an fp32 one), stored and read at device
// scope: a word with another number has not arrived.  Tickets are never reset: a launch takes a power of two of them, the rest of its workgroups
// end at once, so that the count may wrap and nothing is divided; every word is written once a launch, and launches with one workspace follow each other.  Every wait is bounded: if one gives up, that launch's h and those of
// all later launches with the workspace are NaN.
// One row of 2048 with 256 features, us: the four launches 16.9, this one 10.3 (14 before de_row had what does not depend on y at hand when y arrives, and with a
// 64-bit division in front of everything); a token of eight layers 528 -> 486.
// ------------------------------------------------------------------------------------------
constexpr int DE_THREADS = 1024, DE_WAVES = 16, DE_ROWS = 4, DE_BLOCKS = 4;      // DE_BLOCKS: blocks of 16 channels of a projection's workgroup
constexpr int DE_POLLS = 1 << 22;
typedef pta_depth_end_args DE;

struct DepthEndShape { int gates, projections, grid, log_grid, gate_tiles, proj_tiles; };
__host__ __device__ static inline DepthEndShape depth_end_shape(const DE& a) {
  DepthEndShape s;
  s.gates = (a.side + 15) / 16;
  s.projections = (a.add.width + 16 * DE_BLOCKS - 1) / (16 * DE_BLOCKS);
  s.log_grid = 1;
  while (1 << s.log_grid < s.gates + s.projections + a.add.rows) ++s.log_grid;
  s.grid = 1 << s.log_grid;
  s.gate_tiles = (a.add.width + 127) / 128;
  s.proj_tiles = (a.side + 127) / 128;
  return s;
}
// workspace: the tickets, the failure, the gate's words, the projection's
static inline size_t depth_end_bytes(int rows, int width, int side) { return 64 + ((size_t)rows * side * 4 + 15) / 16 * 16 + (size_t)rows * width * 8; }

__device__ __forceinline__ bool de_arrived(bool there, int tries, uint32_t* failed) {
  if (there) return true;
  if (tries == DE_POLLS || ((tries & 1023) == 1023 && __hip_atomic_load(failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
    __hip_atomic_store(failed, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
  }
  __builtin_amdgcn_s_sleep(1);
  return false;
}

// Products of a wave's tile of 16 channels x 128 features with the rows in LDS: sums of channels (lane / 16) * 4 + 0..3 of row lane % 16
__device__ __forceinline__ f32x4 de_tile(const u32x4 (&w)[4], const bf16* rows, f32x4 acc) {
#pragma unroll
  for (int j = 0; j < 4; ++j)
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bitcast<bf16x8>(w[j]), *reinterpret_cast<const bf16x8*>(rows + j * 32), acc, 0, 0, 0);
  return acc;
}

// depth_row for a workgroup that waits for its y, by whole pieces of four columns: all that does not depend on y - the residual with its parts, the
// older depths' sum, the weights - is there before it.
__device__ __forceinline__ void de_row(const DE& a, int r, const unsigned long long* ys, uint32_t launch, uint32_t* failed, float* u_row) {
  constexpr int PER = 8192 / (DE_THREADS * 4);
  __shared__ float red[3][DE_WAVES];
  __shared__ float z[ROUTE_FLOATS];
  const DN& n = a.norm;
  const int d = n.width;
  f32x4 x[PER], older[PER], yw[PER], nw[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = (k * DE_THREADS + (int)threadIdx.x) * 4;
    if (c >= d) break;
    x[k] = *reinterpret_cast<const f32x4*>(a.add.x + (size_t)r * d + c);
    yw[k] = *reinterpret_cast<const f32x4*>(n.y_weight + c);
    nw[k] = *reinterpret_cast<const f32x4*>(n.norm_weight + c);
    if (a.add.parts) {
      const float* w = a.add.part_weight + (size_t)r * a.add.weights_ld;
      const size_t at = (size_t)r * a.add.parts_ld * d + c;
#pragma unroll 4
      for (int p = 0; p < a.add.n_parts; ++p) {
        f32x4 t;
        if (a.add.part_f32) {
          t = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(a.add.parts) + at + (size_t)p * d);
        } else {
          const bf16x4 b = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const bf16*>(a.add.parts) + at + (size_t)p * d);
          t = f32x4{(float)b[0], (float)b[1], (float)b[2], (float)b[3]};
        }
        const float f = w[p];
#pragma unroll
        for (int e = 0; e < 4; ++e) x[k][e] = __builtin_fmaf(f, t[e], x[k][e]);
      }
    }
    older[k] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int j = 0; j < n.depth - 1; ++j) {
      const f32x4 t = *reinterpret_cast<const f32x4*>(n.history + (size_t)j * n.depth_stride + (size_t)r * d + c);
      const float f = n.weights[j];
#pragma unroll
      for (int e = 0; e < 4; ++e) older[k][e] = __builtin_fmaf(f, t[e], older[k][e]);
    }
  }
  const float f_new = n.weights ? n.weights[n.depth - 1] : 1.0f;
  f32x4 y[PER];
  float sq = 0.f;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = (k * DE_THREADS + (int)threadIdx.x) * 4;
    if (c >= d) break;
    unsigned long long v[4];
    for (int t = 0;; ++t) {
      bool all = true;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = __hip_atomic_load(ys + c + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int e = 0; e < 4; ++e) all = all && (uint32_t)(v[e] >> 32) == launch;
      if (de_arrived(all, t, failed)) break;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y[k][e] = bitcast<float>((uint32_t)v[e]);
      sq = __builtin_fmaf(y[k][e], y[k][e], sq);
    }
  }
  const float inv = 1.0f / sqrtf(workgroup_sum<DE_WAVES>(sq, red[0]) / (float)d + n.eps);
  float* newest = a.add.x + (size_t)r * d;
  float sum = 0.f;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = (k * DE_THREADS + (int)threadIdx.x) * 4;
    if (c >= d) break;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[k][e] += y[k][e] * inv * yw[k][e];
      older[k][e] = __builtin_fmaf(f_new, x[k][e], older[k][e]);
      sum += older[k][e];
    }
    *reinterpret_cast<f32x4*>(newest + c) = x[k];
    if (n.next) *reinterpret_cast<f32x4*>(n.next + (size_t)r * d + c) = older[k];
  }
  const float mean = n.centred ? workgroup_sum<DE_WAVES>(sum, red[1]) / (float)d : 0.f;
  sq = 0.f;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    if ((k * DE_THREADS + (int)threadIdx.x) * 4 >= d) break;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float t = older[k][e] - mean;
      sq = __builtin_fmaf(t, t, sq);
    }
  }
  const float f = 1.0f / sqrtf(workgroup_sum<DE_WAVES>(sq, red[2]) / (float)d + n.eps);
  const bool gave_up = __hip_atomic_load(failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
  bf16* h = reinterpret_cast<bf16*>(n.h) + (size_t)r * n.h_ld;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = (k * DE_THREADS + (int)threadIdx.x) * 4;
    if (c >= d) break;
    bf16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[e] = gave_up ? (bf16)NAN : (bf16)((older[k][e] - mean) * f * nw[k][e]);
      u_row[c + e] = (float)o[e];
    }
    *reinterpret_cast<bf16x4*>(h + c) = o;
  }
  for (int c = d + threadIdx.x; c < n.h_ld; c += DE_THREADS) h[c] = (bf16)0.0f;
  if (!n.router) return;
  router_logits<bf16, DE_WAVES>(n.router, n.h_ld, d, u_row, n.routing, z);
  route_row<DE_THREADS>(n.routing, z, r, threadIdx.x, true);
}

__global__ __launch_bounds__(DE_THREADS) void depth_end_kernel(DE a) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ uint32_t start[3];
  const DepthEndShape g = depth_end_shape(a);
  uint32_t* tickets = reinterpret_cast<uint32_t*>(a.workspace);
  uint32_t* failed = tickets + 2;
  uint32_t* acts = reinterpret_cast<uint32_t*>(a.workspace) + 16;
  const int M = a.add.rows, width = a.add.width, side = a.side;
  unsigned long long* ys = reinterpret_cast<unsigned long long*>(acts + ((size_t)M * side + 3) / 4 * 4);
  if (threadIdx.x == 0) {
    start[2] = __hip_atomic_load(failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t n = __hip_atomic_fetch_add(tickets, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    start[0] = n & (uint32_t)(g.grid - 1);
    start[1] = (n >> g.log_grid) + 1;
  }
  __syncthreads();
  const int id = __builtin_amdgcn_readfirstlane((int)start[0]);
  const uint32_t launch = __builtin_amdgcn_readfirstlane(start[1]), tag = launch & 0xffffu;
  const bool given_up = __builtin_amdgcn_readfirstlane(start[2]) != 0;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = (lane & 15) < M ? lane & 15 : M - 1;

  if (id < g.gates + g.projections) {
    if (given_up) return;
    const bool gate = id < g.gates;
    const int tiles = gate ? g.gate_tiles : g.proj_tiles, blocks = gate ? 1 : DE_BLOCKS, blk0 = gate ? id : (id - g.gates) * DE_BLOCKS;
    const int all = gate ? g.gates : (width + 15) / 16, units = (all - blk0 < blocks ? all - blk0 : blocks) * tiles, stride = tiles * 128 + 8;
    bf16* xs = reinterpret_cast<bf16*>(smem);                                    // [M][stride]
    float* red = reinterpret_cast<float*>(smem + (size_t)M * stride * 2);        // [units, or (the gate's) waves][M][16]
    // (unit u: tile u % tiles of block blk0 + u / tiles, which lie one behind the other)
    const u32x4* from = reinterpret_cast<const u32x4*>(gate ? a.gate : a.proj) + (size_t)blk0 * tiles * 256 + lane;
    u32x4 w[4];
    const int u0 = wave < units ? wave : 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = __builtin_nontemporal_load(from + ((size_t)u0 * 4 + j) * 64);
    if (gate) {
      const int pieces = tiles * 16;
      for (int i = threadIdx.x; i < M * pieces; i += DE_THREADS) {
        const int m = i / pieces, c = i % pieces * 8;
        float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (c < width) with_parts<bf16>(a.add, m, c, v);
        store8(xs + (size_t)m * stride + c, v);
      }
    } else {
      for (int i = threadIdx.x; i < M * tiles * 128; i += DE_THREADS) {
        const int m = i / (tiles * 128), c = i % (tiles * 128);
        uint32_t v = 0;
        if (c < side) {
          const uint32_t* p = acts + (size_t)m * side + c;
          v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          for (int n = 0; !de_arrived((v >> 16) == tag, n, failed); ++n) v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        xs[(size_t)m * stride + c] = bitcast<bf16>((uint16_t)v);
      }
    }
    __syncthreads();
    const bf16* mine = xs + (size_t)row * stride + (lane >> 4) * 8;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int u = wave; u < units; u += DE_WAVES) {
      if (u != wave)
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = __builtin_nontemporal_load(from + ((size_t)u * 4 + j) * 64);
      acc = de_tile(w, mine + (size_t)(u % tiles) * 128, gate ? acc : f32x4{0.f, 0.f, 0.f, 0.f});
      if (!gate && (lane & 15) < M) *reinterpret_cast<f32x4*>(red + ((size_t)u * M + (lane & 15)) * 16 + (lane >> 4) * 4) = acc;
    }
    if (gate && (lane & 15) < M) *reinterpret_cast<f32x4*>(red + ((size_t)wave * M + (lane & 15)) * 16 + (lane >> 4) * 4) = acc;
    __syncthreads();
    for (int o = threadIdx.x; o < M * blocks * 16; o += DE_THREADS) {
      const int c = o % (blocks * 16), m = o / (blocks * 16), n = blk0 * 16 + c;
      if (n >= (gate ? side : width)) continue;
      const int parts = gate ? DE_WAVES : tiles;
      float v = 0.f;
      for (int k = 0; k < parts; ++k) v += red[((size_t)((gate ? 0 : (c >> 4) * tiles) + k) * M + m) * 16 + (c & 15)];
      if (gate) {
        v = 0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
        v *= (float)reinterpret_cast<const bf16*>(a.own)[(size_t)m * side + n];
        __hip_atomic_store(acts + (size_t)m * side + n, tag << 16 | bitcast<uint16_t>((bf16)v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      } else {
        __hip_atomic_store(ys + (size_t)m * width + n, (unsigned long long)launch << 32 | bitcast<uint32_t>(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    return;
  }
  const int r = id - g.gates - g.projections;
  if (r >= M) return;
  if (!given_up && (width & 3) == 0 && (a.norm.h_ld & 3) == 0) {                // (whole pieces of a row, and of a row of h)
    de_row(a, r, ys + (size_t)r * width, launch, failed, reinterpret_cast<float*>(smem));
    return;
  }
  float* u_row = reinterpret_cast<float*>(smem);
  float* y = u_row + a.norm.h_ld;                                                // (h_ld: a multiple of eight)
  if (!given_up) {
    if (a.add.parts)
      for (int c = threadIdx.x * 8; c < width; c += DE_THREADS * 8) {            // (read by nobody else any more once y has arrived, and stored behind that)
        float v[8];
        with_parts<bf16>(a.add, r, c, v);
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (c + e < width) u_row[c + e] = v[e];
      }
    for (int c = threadIdx.x; c < width; c += DE_THREADS) {
      const unsigned long long* p = ys + (size_t)r * width + c;
      unsigned long long v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      for (int n = 0; !de_arrived((uint32_t)(v >> 32) == launch, n, failed); ++n) v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      y[c] = bitcast<float>((uint32_t)v);
    }
    __syncthreads();
    if (a.add.parts) {
      for (int c = threadIdx.x; c < width; c += DE_THREADS) a.add.x[(size_t)r * width + c] = u_row[c];
      __syncthreads();
    }
    depth_row<bf16, DE_THREADS>(a.norm, r, y, u_row);
    __syncthreads();
  }
  if (given_up || __hip_atomic_load(failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    for (int c = threadIdx.x; c < width; c += DE_THREADS) reinterpret_cast<bf16*>(a.norm.h)[(size_t)r * a.norm.h_ld + c] = (bf16)NAN;
}

extern "C" size_t pta_depth_end_workspace_bytes(int rows, int width, int side) {
  return rows < 1 || rows > DE_ROWS || width < 1 || width > 8192 || side < 8 || side > 1024 || side % 8 ? 0 : depth_end_bytes(rows, width, side);
}

extern "C" int pta_depth_end(const DE* args, pta_stream_t stream) {
  const char* name = "pta_depth_end";
  PTA_REQUIRE(args, "%s: null arguments", name);
  const DE& a = *args;
  int rc = check_add_parts(a.add, name);
  if (!rc) rc = check_depth_norm(a.norm, name);
  if (rc) return rc;
  const size_t need = pta_depth_end_workspace_bytes(a.add.rows, a.add.width, a.side);
  if (!need || a.add.dtype != PTA_BF16 || a.norm.dtype != PTA_BF16) {
    pta_set_error("%s: %d rows of %d, %d features of the token's own: bf16, at most %d rows of 8192, a multiple of 8 up to 1024", name, a.add.rows, a.add.width, a.side, DE_ROWS);
    return PTA_EUNSUPPORTED;
  }
  PTA_REQUIRE(a.norm.rows == a.add.rows && a.norm.width == a.add.width && !a.norm.table && !a.norm.y && a.norm.y_weight && pta_aligned(a.norm.y_weight, 16) &&
                  a.norm.depth >= 1 && a.add.x == a.norm.history + (size_t)(a.norm.depth - 1) * a.norm.depth_stride,
              "%s: the two halves are not of one layer", name);
  PTA_REQUIRE(a.gate && a.proj && a.own && pta_aligned(a.gate, 16) && pta_aligned(a.proj, 16), "%s: a weight or the token's own part null or unaligned", name);
  PTA_REQUIRE(a.workspace && pta_aligned(a.workspace, 64) && a.workspace_bytes >= need, "%s: the workspace needs %zu bytes", name, need);
  const DepthEndShape g = depth_end_shape(a);
  const size_t rows = a.add.rows, gate = rows * (g.gate_tiles * 128 + 8) * 2 + DE_WAVES * rows * 64,
               proj = rows * (g.proj_tiles * 128 + 8) * 2 + (size_t)DE_BLOCKS * g.proj_tiles * rows * 64, norm = (size_t)(a.norm.h_ld + a.add.width) * 4;
  const size_t smem = gate > proj ? (gate > norm ? gate : norm) : (proj > norm ? proj : norm);
  static bool ready = false;
  if (!ready) {
    PTA_REQUIRE(hipFuncSetAttribute((const void*)depth_end_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024) == hipSuccess, "%s: cannot reserve LDS", name);
    ready = true;
  }
  PTA_REQUIRE(smem <= 128 * 1024, "%s: %zu bytes of LDS", name, smem);
  hipLaunchKernelGGL(depth_end_kernel, dim3(g.grid), dim3(DE_THREADS), smem, (hipStream_t)stream, a);
  PTA_CHECK_LAUNCH(name);
  return PTA_OK;
}

extern "C" int pta_depth_end_failed(const void* workspace, int* failed, pta_stream_t stream) {
  PTA_REQUIRE(workspace && failed, "pta_depth_end_failed: null pointer");
  uint32_t word = 0;
  hipError_t e = hipMemcpyAsync(&word, reinterpret_cast<const uint32_t*>(workspace) + 2, sizeof(word), hipMemcpyDeviceToHost, (hipStream_t)stream);
  if (e == hipSuccess) e = hipStreamSynchronize((hipStream_t)stream);
  if (e != hipSuccess) {
    pta_set_error("pta_depth_end_failed: %s", hipGetErrorString(e));
    return PTA_EHIP;
  }
  *failed = word != 0;
  return PTA_OK;
}
