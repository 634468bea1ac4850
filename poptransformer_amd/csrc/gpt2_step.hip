// One loop iteration of a GPT-2 decoder (fp16 weights, head size 64, up to eight sequences) as one launch.
//
// Reference graph: models/gpt2/model.py, models/gpt2/attention.py:50-90, layers/mlp.py:34-41, layers/lm_head.py:47-57 and the loop
// bookkeeping of models/base_model.py:313-355.  The rounding points are those of the per-operator entry points.
//
// What bounds the iteration of a model this small is the chain of its launches: GPT-2 small has 60 products and attentions a token, each
// waiting for the one before, at 4.5 us a launch of which 3 are an empty one's; its 247 MB take 52 us.  Here the workgroups of all of
// them are one grid, in the order of the chain.  A workgroup takes a ticket when it starts, and the ticket is its place in the
// chain: which product, and which of its channels.  It requests its weights into registers, then waits for the values that it multiplies.
// It only ever waits for workgroups with smaller tickets, which have started before it: no launch has to fit the machine as a whole, and
// launches of several decoders, streams and processes may share it in any proportion.
//
// A value travels from workgroup to workgroup as a 32-bit word: its fp16 bits, and above them the number of the iteration.  Words are
// stored and read at device scope; one whose upper half is not this iteration's has not arrived.  Nothing is counted, cleared or
// fenced: a slot's words are written once an iteration, and the last workgroup moves the number on when all others are done.
//
// The workgroups are few (24 to 48 a product at a width of 768; where the registers hold fewer channels of one more of them, at 2048 up to 128; the head 390
// to 790) and of 16 waves: a compute unit has one at a time, so about six products' workgroups are
// there at once, each with its weights on their way, and the machine starts some 100 workgroups a microsecond at most (a link of the
// chain with nothing to multiply: 48 workgroups 1.25 us, 96 1.7, 256 3.2; in one launch that stays 0.93).
//
// GPT-2 small, us a token, per operator and here: batch 1, context 16 314 -> 184, 400 324 -> 198, 900 340 -> 226; batch 2 336 -> 209, 4 362 ->
// 239, 8 395 -> 298 (context 900 467 -> 345); width 256 267 -> 150; 8 layers of width 1280 276 -> 173.  A link takes 2.0 (attention) to 3.0
// us: 1.0 to 1.6 until the last producer's words have come, 0.4 to 0.6 the norm, 0.4 the products, 0.4 to 0.5 the sums and the end; the head 20.
// Measured and not kept: eight copies of every word, each for an eighth of the readers (no gain: the lines are not what is
// contended); two workgroups a compute unit by half the registers (176 -> 213: twice the waiting ones); the norm applied to the
// operands of the matrix instructions (every wave of a unit repeats it: +1.3 us a link); v_rsq_f32 for the norms' reciprocal root (184 -> 179, but it
// rounds some variances to the other fp16 neighbour than 1 / sqrtf, which the operators take).
#include "common.h"
#include "formats.h"

constexpr int G2_WAVES = 16, G2_THREADS = G2_WAVES * 64;
constexpr int G2_MAX_BATCH = 8;
constexpr int G2_MAX_HIDDEN = 2048;
constexpr int G2_MAX_TILES = 4;            // feature tiles (of 16 channels x 128 features) that a wave keeps in registers
constexpr int G2_HEAD = 64;                // head size
constexpr int G2_CTL_WORDS = 64;           // workspace: ticket, failure, iteration (pta_decode_step_failed reads word 1)
constexpr int G2_POLLS = 1 << 22;

// a product of the chain: its workgroups, and the blocks of 16 channels and feature tiles of each
struct G2Part { int wgs, blocks, all_blocks, tiles; };

struct G2Args {
  pta_gpt2_model m;
  pta_decode_state s;
  uint32_t* ctl;
  uint32_t* slots;
  unsigned long long* best;              // [workgroups of the head][batch]
  G2Part qkv, out, fc, down, logits;
  int per_layer, total, xstride;
  float inv_hidden;
  size_t layer_words, at_qkv, at_ctx, at_mid, at_act;      // words of a layer's slots, and where they begin behind its input
};

__device__ __forceinline__ uint32_t g2_load(const uint32_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void g2_store(uint32_t* p, uint32_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

struct G2Wait {
  uint32_t tag;
  uint32_t* failed;
  // the word at p once it is this iteration's (v: what it held last)
  __device__ __forceinline__ f16 word(const uint32_t* p, uint32_t v) const {
    for (int n = 0; (v >> 16) != tag; ++n) {
      if (n == G2_POLLS || ((n & 1023) == 1023 && g2_load(failed))) {      // (no producer is ever missing; a wait ends all the same)
        g2_store(failed, 1);
        break;
      }
      __builtin_amdgcn_s_sleep(1);
      v = g2_load(p);
    }
    return bitcast<f16>((uint16_t)v);
  }
  __device__ __forceinline__ f16 word(const uint32_t* p) const { return word(p, g2_load(p)); }
  // Called by a whole workgroup: returns when the link before the one it waits for has (begun to) put its words, of which `p` is one.  Until then one
  // lane looks, now and then: hundreds of workgroups that look at all their words take the memory's time from those whose turn it is.
  __device__ __forceinline__ void near(const uint32_t* p) const {
    if (threadIdx.x == 0) {
      for (int n = 0; (g2_load(p) >> 16) != tag; ++n) {
        if (n == G2_POLLS || ((n & 1023) == 1023 && g2_load(failed))) { g2_store(failed, 1); break; }
        __builtin_amdgcn_s_sleep(8);
      }
    }
    __builtin_amdgcn_s_barrier();
  }
  __device__ __forceinline__ void put(uint32_t* p, f16 v) const { g2_store(p, tag << 16 | bitcast<uint16_t>(v)); }
  // four words, `stride` apart from each other, the first `n` of them (n > 0): what has not arrived is looked at again
  __device__ __forceinline__ void words(const uint32_t* p, int stride, int n, uint32_t (&v)[4]) const {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = i < n ? g2_load(p + i * stride) : tag << 16;
    for (int t = 0;; ++t) {
      bool all = true;
#pragma unroll
      for (int i = 0; i < 4; ++i) all = all && (v[i] >> 16) == tag;
      if (all) return;
      if (t == G2_POLLS || ((t & 1023) == 1023 && g2_load(failed))) {
        g2_store(failed, 1);
        return;
      }
      __builtin_amdgcn_s_sleep(1);
      uint32_t u[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if ((v[i] >> 16) != tag) u[i] = g2_load(p + i * stride);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if ((v[i] >> 16) != tag) v[i] = u[i];
    }
  }
};

// the sum over each N (2, 4, 8 or 16) consecutive lanes, in each of them
template <int N>
__device__ __forceinline__ float lanes_total(float v) {
  if constexpr (N >= 8) return lane_group_sum<N>(v);
  v += bitcast<float>(__builtin_amdgcn_update_dpp(0, bitcast<int>(v), 0xB1, 0xF, 0xF, true));
  if (N == 4) v += bitcast<float>(__builtin_amdgcn_update_dpp(0, bitcast<int>(v), 0x4E, 0xF, 0xF, true));
  return v;
}

struct G2Product {
  G2Part part;
  int K, N;
  const void* weights;
  const f16 *bias, *gamma, *beta;        // gamma null: the rows as they are
  const uint32_t* before;                // a word of the link before the one that x comes from, or null
  const uint32_t* x;                     // words of the rows; null: from the tables, whose sum goes to x_out
  uint32_t* x_out;
  const uint32_t* residual;              // words, or null
  uint32_t* y;                           // words; null: the logits
  bool gelu;
};

// Y = act(norm(X) W^T + b) + residual for the channels of workgroup wg of a product.  (One copy of the code for all products of as many
// tiles a wave: a compute unit runs them in turn, and instructions it does not hold come at half a microsecond a stretch.  Behind the
// wait every instruction counts: four waves a SIMD wait for each other's, so divisions and addresses come before it.)
template <int MB, int R>
__device__ __forceinline__ void g2_product(const G2Args& a, const G2Product& q, int wg, int step, const G2Wait& wait, unsigned char* smem) {
  constexpr int WPR = G2_WAVES / MB, SPAN = WPR * 64, OWN = G2_MAX_HIDDEN / SPAN;      // waves of a row, what they read at a time, a lane's features of a normed row
  const G2Part& part = q.part;
  const int K = q.K, N = q.N;
  const bool norm = q.gamma != nullptr;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int M = a.m.batch, KT = part.tiles, units = part.blocks * KT;
  f16* xs = reinterpret_cast<f16*>(smem);                                        // [MB][xstride]
  float* sums = reinterpret_cast<float*>(xs + (size_t)MB * a.xstride);           // [16][2]
  float* red = sums + 2 * G2_WAVES;                                              // [units][MB][16]

  // the weights: unit u of the workgroup is feature tile u % KT of its block u / KT; wave w has the units w, w + 16, ...
  const int blk0 = wg * part.blocks;
  const uint32_t weight_bytes = (uint32_t)part.all_blocks * KT * 4096;
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(q.weights), 0, (int)weight_bytes, 0x00020000);
  u32x4 w[R][4];
  int x_at[R];                                                                   // bytes of the unit's tile in a row
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int u = wave + G2_WAVES * i;
    const uint32_t at = (uint32_t)(blk0 * KT + u) * 4096;                        // (past the workgroup's units, or the last block: from nowhere)
    const int off = u < units && at < weight_bytes ? lane * 16 : -1;
#pragma unroll
    for (int v = 0; v < 4; ++v) w[i][v] = __builtin_amdgcn_raw_buffer_load_b128(wr, off, (int)at + v * 1024, 2);
    x_at[i] = u % KT * 256;
    in_register(x_at[i]);
  }
  // the rows
  const int row = wave / WPR, first = (wave % WPR) * 64 + lane;
  f16* to = xs + (size_t)row * a.xstride;
  if (norm) {
    f16 h[OWN], gm[OWN], bt[OWN];
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
      const int c = first + i * SPAN < K ? first + i * SPAN : K - 1;             // (a row may be shorter than what its waves read at a time)
      gm[i] = q.gamma[c];
      bt[i] = q.beta[c];
    }
    if (q.before) wait.near(q.before);
    float s1 = 0.f, s2 = 0.f;
    if (row < M) {
      if (q.x == nullptr) {
        const int at = step < 0 ? 0 : (step >= a.m.max_len ? a.m.max_len - 1 : step);
        int id = a.s.container[(size_t)row * a.m.max_len + at];
        id = id < 0 ? 0 : (id >= a.m.vocab ? a.m.vocab - 1 : id);
        const f16* e = (const f16*)a.m.embed + (size_t)id * K;
        const f16* p = (const f16*)a.m.positions + (size_t)(step < a.m.n_positions ? step : a.m.n_positions - 1) * K;
#pragma unroll
        for (int i = 0; i < OWN; ++i) {
          const int c = first + i * SPAN;
          if (c < K) {
            h[i] = e[c] + p[c];
            if (wg == 0) wait.put(q.x_out + (size_t)row * K + c, h[i]);
          }
        }
      } else {
        const uint32_t* from = q.x + (size_t)row * K;
#pragma unroll
        for (int i = 0; i < OWN; i += 4) {
          const int c0 = first + i * SPAN;
          if (c0 >= K) break;
          uint32_t v[4];
          if (OWN > 1 && c0 + SPAN < K) wait.words(from + c0, SPAN, (K - c0 + SPAN - 1) / SPAN, v);
          else v[0] = bitcast<uint16_t>(wait.word(from + c0));
#pragma unroll
          for (int j = 0; j < 4 && i + j < OWN; ++j) h[i + j] = bitcast<f16>((uint16_t)v[j]);
        }
      }
#pragma unroll
      for (int i = 0; i < OWN; ++i)
        if (first + i * SPAN < K) {
          const float f = (float)h[i];
          s1 += f;
          s2 = __builtin_fmaf(f, f, s2);
        }
    }
    s1 = wave_total_dpp(s1);
    s2 = wave_total_dpp(s2);
    if (lane == 0) *reinterpret_cast<f32x2*>(sums + wave * 2) = f32x2{s1, s2};
    __syncthreads();
    if (row < M) {
      const f32x2 part_sum = *reinterpret_cast<const f32x2*>(sums + (row * WPR + lane % WPR) * 2);
      const float mean = lanes_total<WPR>(part_sum[0]) * a.inv_hidden, sq = lanes_total<WPR>(part_sum[1]) * a.inv_hidden;
      const f16 mean16 = (f16)mean;
      const float about = MB == 1 ? mean : (float)mean16;                        // (as the norm of a single row, and of several)
      const float var = (MB == 1 ? sq - about * about : fmaxf(sq - about * about, 0.0f)) + a.m.eps;
      const f16 r16 = (f16)(1.0f / sqrtf(var));
#pragma unroll
      for (int i = 0; i < OWN; ++i) {
        const int c = first + i * SPAN;
        if (c < KT * 128) to[c] = c < K ? ((h[i] - mean16) * r16) * gm[i] + bt[i] : (f16)0.0f;
      }
    }
  } else {
    if (q.before) wait.near(q.before);
    if (row < M) {
      const uint32_t* from = q.x + (size_t)row * K;
      for (int c0 = first; c0 < K; c0 += 4 * SPAN) {
        uint32_t v[4];
        if (c0 + SPAN < K) wait.words(from + c0, SPAN, (K - c0 + SPAN - 1) / SPAN, v);
        else v[0] = bitcast<uint16_t>(wait.word(from + c0));
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (c0 + i * SPAN < K) to[c0 + i * SPAN] = bitcast<f16>((uint16_t)v[i]);
      }
      for (int c = K + first; c < KT * 128; c += SPAN) to[c] = (f16)0.0f;
    }
  }
  // An output a thread, channels first (one store instruction of a wave is whole stretches of a row); of a single row, whose outputs are few,
  // one to eight lanes, which add its tiles side by side (0.55 -> 0.41 us).  What an output adds is requested now.
  constexpr int LPO = MB == 1 ? 8 : 1;
  const int outs = part.blocks * 16, o0 = (int)threadIdx.x / LPO, m0 = MB == 1 ? 0 : o0 / outs, c0 = MB == 1 ? o0 : o0 % outs;
  uint32_t res = 0;
  f16 b0 = (f16)0.0f;
  if (q.y && m0 < M && c0 < outs && blk0 * 16 + c0 < N) {
    b0 = q.bias[blk0 * 16 + c0];
    if (q.residual) res = g2_load(q.residual + (size_t)m0 * N + blk0 * 16 + c0);
  }
  __syncthreads();

  // the products
  const unsigned char* xl = reinterpret_cast<const unsigned char*>(xs + (size_t)((lane & 15) < M ? lane & 15 : M - 1) * a.xstride + (lane >> 4) * 8);
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int u = wave + G2_WAVES * i;
    if (u >= units) break;
    f16x8 xv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) xv[j] = *reinterpret_cast<const f16x8*>(xl + x_at[i] + j * 64);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = FmtF16::mma(bitcast<f16x8>(w[i][j]), xv[j], acc);
    if ((lane & 15) < MB) *reinterpret_cast<f32x4*>(red + ((size_t)u * MB + (lane & 15)) * 16 + (lane >> 4) * 4) = acc;
  }
  __syncthreads();
  auto total = [&](bool here, int m, int c) {
    float t = 0.f;
    if constexpr (LPO == 8) {
      if (here)
        for (int k = threadIdx.x & 7; k < KT; k += 8) t += red[((c >> 4) * KT + k) * 16 + (c & 15)];
      t = lane_group_sum<8>(t);
    } else if (here) {
      const float* r = red + ((c >> 4) * KT * MB + m) * 16 + (c & 15);
      for (int k = 0; k < KT; k += 8) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = r[(k + j < KT ? k + j : k) * (MB * 16)];
#pragma unroll
        for (int j = 0; j < 8; ++j) t += k + j < KT ? v[j] : 0.f;
      }
    }
    return t;
  };
  constexpr int STEP = G2_THREADS / LPO;
  if (q.y) {
    for (int o = o0; o < (outs * M + STEP - 1) / STEP * STEP; o += STEP) {
      const bool again = o != o0;
      const int m = MB == 1 ? 0 : again ? o / outs : m0, c = MB == 1 ? o : again ? o % outs : c0, n = blk0 * 16 + c;
      const bool here = o < outs * M && n < N;
      const size_t at = (size_t)m * N + n;
      if (again && here) {
        b0 = q.bias[n];
        if (q.residual) res = g2_load(q.residual + at);
      }
      f16 v = (f16)total(here, m, c) + b0;
      if (!here || threadIdx.x % LPO != 0) continue;
      if (q.gelu) v = gelu_tanh_f16(v);
      if (q.residual) v = v + wait.word(q.residual + at, res);
      wait.put(q.y + at, v);
    }
  } else {
    float* val = reinterpret_cast<float*>(smem);                                 // (over the rows, which have been multiplied)
    for (int o = o0; o < (outs * M + STEP - 1) / STEP * STEP; o += STEP) {
      const int m = MB == 1 ? 0 : o / outs, c = MB == 1 ? o : o % outs, n = blk0 * 16 + c;
      const bool here = o < outs * M;
      const f16 v = (f16)total(here, m, c);
      if (!here || threadIdx.x % LPO != 0) continue;
      if (n < N) ((f16*)a.s.logits)[(size_t)m * N + n] = v;
      val[o] = n < N ? (float)v : -INFINITY;
    }
    __syncthreads();
    if (wave < M) {                                                              // the best of the workgroup's channels: of equal ones the first
      float best = -INFINITY;
      int bi = 0x7fffffff;
      for (int c = lane; c < outs; c += 64) {
        const float v = val[wave * outs + c];
        if (blk0 * 16 + c < N && (v > best || (v == best && bi == 0x7fffffff))) { best = v; bi = blk0 * 16 + c; }
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const float ov = __shfl_xor(best, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
      }
      if (lane == 0)
        __hip_atomic_store(a.best + (size_t)wg * M + wave,
                           (unsigned long long)(wait.tag << 16 | bitcast<uint16_t>((f16)best)) << 32 | (uint32_t)bi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// of each row of sixteen lanes: the value of the lane eight further on, and the largest value
__device__ __forceinline__ float row_ror8(float v) { return bitcast<float>(__builtin_amdgcn_update_dpp(0, bitcast<int>(v), 0x128, 0xF, 0xF, true)); }
__device__ __forceinline__ float row_max(float v) {
  v = fmaxf(v, bitcast<float>(__builtin_amdgcn_update_dpp(0, bitcast<int>(v), 0xB1, 0xF, 0xF, true)));       // quad_perm [1, 0, 3, 2]
  v = fmaxf(v, bitcast<float>(__builtin_amdgcn_update_dpp(0, bitcast<int>(v), 0x4E, 0xF, 0xF, true)));       // quad_perm [2, 3, 0, 1]
  v = fmaxf(v, bitcast<float>(__builtin_amdgcn_update_dpp(0, bitcast<int>(v), 0x141, 0xF, 0xF, true)));      // row_half_mirror
  return fmaxf(v, bitcast<float>(__builtin_amdgcn_update_dpp(0, bitcast<int>(v), 0x140, 0xF, 0xF, true)));   // row_mirror
}

// The attention of one head of one sequence: 8 lanes a cache row, 128 rows at a time; arithmetic as in attn_partial_kernel.  The first
// 256 rows are on their way while q, k and v are waited for.
__device__ __forceinline__ void g2_attention(const G2Args& a, int bh, void* ring, const uint32_t* before, const uint32_t* qkv, uint32_t* ctx, int step, const G2Wait& wait, unsigned char* smem) {
  constexpr int D = G2_HEAD, AHEAD = 2, ROWS = G2_WAVES * 8, PAIRS = G2_WAVES * 4;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int H = a.m.n_head, L = a.m.max_len, d = a.m.hidden, B = a.m.batch;
  const int b = bh / H, h = bh % H, d0 = (lane & 7) * 8, mine = wave * 8 + (lane >> 3);
  const int valid = step + 1 < L ? step + 1 : L, pos = step % L;
  f16* kb = (f16*)ring + ((size_t)b * H + h) * L * D;
  f16* vb = kb + (size_t)B * H * L * D;
  f16* now = reinterpret_cast<f16*>(smem);                      // [3][64]
  float* sm_m = reinterpret_cast<float*>(smem + 3 * D * 2);     // [64]
  float* sm_l = sm_m + PAIRS;                                   // [64]
  float* sm_acc = sm_l + PAIRS;                                 // [64][64 + 4]
  f16x8 k8[AHEAD], v8[AHEAD];
  auto fetch = [&](int p0) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const int p = p0 + u * ROWS + mine, pc = p < valid ? p : valid - 1;
      k8[u] = __builtin_nontemporal_load(reinterpret_cast<const f16x8*>(kb + (size_t)pc * D + d0));
      v8[u] = __builtin_nontemporal_load(reinterpret_cast<const f16x8*>(vb + (size_t)pc * D + d0));
    }
  };
  fetch(0);
  wait.near(before);
  if (threadIdx.x < 3 * D) {
    const int which = threadIdx.x / D, e = threadIdx.x % D;
    now[threadIdx.x] = wait.word(qkv + (size_t)b * 3 * d + (size_t)which * d + h * D + e);
  }
  __syncthreads();
  if (threadIdx.x >= D && threadIdx.x < 3 * D) (threadIdx.x < 2 * D ? kb : vb)[(size_t)pos * D + threadIdx.x % D] = now[threadIdx.x];
  float qf[8];
  {
    const f16x8 q8 = *reinterpret_cast<const f16x8*>(now + d0);
#pragma unroll
    for (int e = 0; e < 8; ++e) qf[e] = (float)q8[e];
  }
  float m = -INFINITY, l = 0.f, acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
  for (int p0 = 0; p0 < valid; p0 += AHEAD * ROWS) {
    if (p0 > 0) fetch(p0);
    float x[AHEAD], mn = m;
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const int p = p0 + u * ROWS + mine;
      if (p == pos) {                                           // this step's row: its ring copy is being written
        k8[u] = *reinterpret_cast<const f16x8*>(now + D + d0);
        v8[u] = *reinterpret_cast<const f16x8*>(now + 2 * D + d0);
      }
      float s = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) s = __builtin_fmaf(qf[e], (float)k8[u][e], s);
      s = lane_group_sum<8>(s);
      x[u] = p < valid ? (float)(f16)s : -INFINITY;             // fp16 output of the q.K^T MatMul
      mn = fmaxf(mn, x[u]);
    }
    if (mn != -INFINITY) {
      const float corr = m == -INFINITY ? 0.f : __expf(m - mn);
      l *= corr;
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] *= corr;
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        const float pe = p0 + u * ROWS + mine < valid ? __expf(x[u] - mn) : 0.f;
        l += pe;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = __builtin_fmaf(pe, (float)v8[u][e], acc[e]);
      }
      m = mn;
    }
  }
  // The two row groups of sixteen lanes merge by data-parallel moves; the 64 pairs of groups of the workgroup in LDS, sixteen lanes an output
  // that merge four of them each.
  {
    const float mo = row_ror8(m), lo = row_ror8(l), mn = fmaxf(m, mo);
    const float ca = m == -INFINITY ? 0.f : __expf(m - mn), cb = mo == -INFINITY ? 0.f : __expf(mo - mn);
    l = l * ca + lo * cb;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = acc[e] * ca + row_ror8(acc[e]) * cb;
    m = mn;
  }
  const int pair = wave * 4 + (lane >> 4);
  if ((lane & 15) == 0) { sm_m[pair] = m; sm_l[pair] = l; }
  if ((lane & 15) < 8) {
    *reinterpret_cast<f32x4*>(sm_acc + pair * (D + 4) + d0) = f32x4{acc[0], acc[1], acc[2], acc[3]};
    *reinterpret_cast<f32x4*>(sm_acc + pair * (D + 4) + d0 + 4) = f32x4{acc[4], acc[5], acc[6], acc[7]};
  }
  __syncthreads();
  const int out = threadIdx.x >> 4, from = threadIdx.x & 15;
  float mi[4], top = -INFINITY;
#pragma unroll
  for (int i = 0; i < 4; ++i) { mi[i] = sm_m[from + 16 * i]; top = fmaxf(top, mi[i]); }
  top = row_max(top);
  float den = 0.f, num = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float w = mi[i] == -INFINITY ? 0.f : __expf(mi[i] - top);
    den = __builtin_fmaf(sm_l[from + 16 * i], w, den);
    num = __builtin_fmaf(sm_acc[(from + 16 * i) * (D + 4) + out], w, num);
  }
  den = lane_group_sum<16>(den);
  num = lane_group_sum<16>(num);
  if (from == 0) wait.put(ctx + (size_t)b * d + h * D + out, (f16)(num / den));
}

// The last workgroup: the best token of every row, the loop's bookkeeping (step_update_kernel), and the next iteration's number.
__device__ __forceinline__ void g2_end(const G2Args& a, int step, const G2Wait& wait, unsigned char* smem) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, M = a.m.batch;
  int* next = reinterpret_cast<int*>(smem);
  if (wave < M) {
    float best = -INFINITY;
    int bi = 0x7fffffff;
    for (int g = lane; g < a.logits.wgs; g += 64) {
      const unsigned long long* p = a.best + (size_t)g * M + wave;
      unsigned long long v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      for (int n = 0; (uint32_t)(v >> 48) != wait.tag; ++n) {
        if (n == G2_POLLS || ((n & 1023) == 1023 && g2_load(wait.failed))) { g2_store(wait.failed, 1); break; }
        __builtin_amdgcn_s_sleep(1);
        v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      const float f = (float)bitcast<f16>((uint16_t)(v >> 32));
      const int i = (int)(uint32_t)v;
      if (f > best || (f == best && i < bi)) { best = f; bi = i; }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(best, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
    }
    if (lane == 0) next[wave] = bi == 0x7fffffff ? 0 : bi;      // (a row without any comparable value selects index 0)
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  a.ctl[0] = 0;
  a.ctl[2] = wait.tag;
  if (g2_load(wait.failed)) return;
  for (int b = 0; b < M; ++b) a.s.next_ids[b] = next[b];
  if (*a.s.keep_going == 0) return;
  int stopped = 0;
  for (int b = 0; b < M; ++b) {
    if (a.s.stop_mask[b]) ++stopped;
    int id = next[b];
    if (step + 1 < a.m.max_len) {
      const size_t at = (size_t)b * a.m.max_len + step + 1;
      ((f16*)a.s.mask)[at] = (f16)0.0f;
      const int slot = a.s.container[at];
      id = slot == a.m.pad_id ? id : slot;
      a.s.container[at] = id;
    }
    a.s.stop_mask[b] |= id == a.m.eos_id ? 1 : 0;
  }
  *a.s.keep_going = a.m.early_stop ? (stopped < M ? 1 : 0) : 1;
  *a.s.step = step + 1;
}

template <int MB>
__global__ __launch_bounds__(G2_THREADS) void gpt2_step_kernel(G2Args a) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ uint32_t start[4];
  if (threadIdx.x == 0) {
    start[1] = g2_load(a.ctl + 1);
    start[2] = a.ctl[2];
    start[3] = (uint32_t)*a.s.step;
    start[0] = __hip_atomic_fetch_add(a.ctl, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  int id = __builtin_amdgcn_readfirstlane((int)start[0]);
  const int step = __builtin_amdgcn_readfirstlane((int)start[3]);
  G2Wait wait{(__builtin_amdgcn_readfirstlane(start[2]) + 1) & 0xffffu, a.ctl + 1};     // (a workspace begins with zeros, which are no iteration)
  if (__builtin_amdgcn_readfirstlane(start[1])) {                // a wait gave up: nothing is done until that is cleared
    if (id == a.total - 1 && threadIdx.x == 0) {                 // (nor is this iteration's number used again: words of it may be there)
      a.ctl[0] = 0;
      a.ctl[2] = wait.tag;
    }
    return;
  }
  if (id == a.total - 1) {
    g2_end(a, step, wait, smem);
    return;
  }
  const int d = a.m.hidden, layer = id < a.m.n_layer * a.per_layer ? id / a.per_layer : a.m.n_layer;
  uint32_t* in = a.slots + (size_t)layer * a.layer_words;
  const uint32_t* last = in - a.layer_words;                      // (of the layer before, if there is one)
  id -= layer * a.per_layer;
  const pta_gpt2_layer& w = reinterpret_cast<const pta_gpt2_layer*>(a.m.layers)[layer < a.m.n_layer ? layer : 0];
  G2Product q{};
  if (layer == a.m.n_layer) {
    q = G2Product{a.logits, d, a.m.vocab, a.m.head, nullptr, (const f16*)a.m.norm_weight, (const f16*)a.m.norm_bias, last + a.at_act, in, nullptr, nullptr, nullptr, false};
  } else if (id < a.qkv.wgs) {
    q = G2Product{a.qkv, d, 3 * d, w.qkv, (const f16*)w.qkv_bias, (const f16*)w.norm1_weight, (const f16*)w.norm1_bias, layer ? last + a.at_act : nullptr,
                  layer ? in : nullptr, in, nullptr,
                  in + a.at_qkv, false};
  } else if ((id -= a.qkv.wgs) < a.m.batch * a.m.n_head) {
    g2_attention(a, id, w.kv_ring, in, in + a.at_qkv, in + a.at_ctx, step, wait, smem);
    return;
  } else if ((id -= a.m.batch * a.m.n_head) < a.out.wgs) {
    q = G2Product{a.out, d, d, w.out, (const f16*)w.out_bias, nullptr, nullptr, in + a.at_qkv, in + a.at_ctx, nullptr, in, in + a.at_mid, false};
  } else if ((id -= a.out.wgs) < a.fc.wgs) {
    q = G2Product{a.fc, d, a.m.ffn, w.fc, (const f16*)w.fc_bias, (const f16*)w.norm2_weight, (const f16*)w.norm2_bias, in + a.at_ctx, in + a.at_mid, nullptr, nullptr, in + a.at_act,
                  true};
  } else {
    id -= a.fc.wgs;
    q = G2Product{a.down, a.m.ffn, d, w.down, (const f16*)w.down_bias, nullptr, nullptr, in + a.at_mid, in + a.at_act, nullptr, in + a.at_mid, in + a.layer_words, false};
  }
  switch ((q.part.blocks * q.part.tiles + G2_WAVES - 1) / G2_WAVES) {
    case 1: g2_product<MB, 1>(a, q, id, step, wait, smem); break;
    case 2: g2_product<MB, 2>(a, q, id, step, wait, smem); break;
    case 3: g2_product<MB, 3>(a, q, id, step, wait, smem); break;
    default: g2_product<MB, 4>(a, q, id, step, wait, smem); break;
  }
}

// Blocks of 16 channels of a workgroup: as few workgroups as `most`, if the waves' registers hold that many tiles.
static G2Part g2_part(int channels, int features, int most) {
  G2Part p;
  p.tiles = (features + 127) / 128;
  p.all_blocks = (channels + 15) / 16;
  const int cap = G2_WAVES * G2_MAX_TILES / p.tiles;
  p.blocks = (p.all_blocks + most - 1) / most;
  if (p.blocks > cap) p.blocks = cap;
  p.wgs = p.blocks ? (p.all_blocks + p.blocks - 1) / p.blocks : 0;
  return p;
}

static int g2_rows(int batch) { return batch <= 1 ? 1 : batch <= 2 ? 2 : batch <= 4 ? 4 : 8; }

// false: a shape that the kernel does not cover
static bool g2_plan(const pta_gpt2_model* m, G2Args* a, size_t* lds, size_t* bytes) {
  if (!m || m->n_layer < 1 || m->batch < 1 || m->batch > G2_MAX_BATCH || m->n_head < 1 || m->hidden != m->n_head * G2_HEAD || m->ffn < 8 || m->ffn % 8 ||
      m->vocab < 1 || m->max_len < 1 || m->n_positions < m->max_len)
    return false;
  const int d = m->hidden, B = m->batch;
  if (d > G2_MAX_HIDDEN || m->ffn > 8192) return false;
  a->m = *m;
  a->inv_hidden = 1.0f / (float)d;
  a->qkv = g2_part(3 * d, d, 48);
  a->out = g2_part(d, d, 24);
  a->fc = g2_part(m->ffn, d, 48);
  a->down = g2_part(d, m->ffn, 48);
  a->logits = g2_part(m->vocab, d, 400);
  const G2Part* parts[] = {&a->qkv, &a->out, &a->fc, &a->down, &a->logits};
  int units = 0;
  for (const G2Part* p : parts) {
    if (p->blocks < 1 || (size_t)p->all_blocks * p->tiles * 4096 > 0x7fffffffu) return false;
    if (p->blocks * p->tiles > units) units = p->blocks * p->tiles;
  }
  const int widest = d > m->ffn ? d : m->ffn, rows = g2_rows(B);
  a->xstride = (widest + 127) / 128 * 128 + 8;
  *lds = (size_t)rows * a->xstride * 2 + 2 * G2_WAVES * 4 + (size_t)units * rows * 64;
  const size_t attention = 3 * G2_HEAD * 2 + 4 * G2_WAVES * 4 * (2 + G2_HEAD + 4), values = (size_t)a->logits.blocks * 16 * B * 4;
  if (*lds < attention) *lds = attention;
  if (values > (size_t)rows * a->xstride * 2 || *lds > 150 * 1024) return false;
  a->per_layer = a->qkv.wgs + B * m->n_head + a->out.wgs + a->fc.wgs + a->down.wgs;
  a->total = m->n_layer * a->per_layer + a->logits.wgs + 1;
  const size_t row = (size_t)B * d;
  a->at_qkv = row;
  a->at_ctx = 4 * row;
  a->at_mid = 5 * row;
  a->at_act = 6 * row;
  a->layer_words = 6 * row + (size_t)B * m->ffn;
  const size_t words = (G2_CTL_WORDS + (size_t)m->n_layer * a->layer_words + row + 63) & ~(size_t)63;
  *bytes = words * 4 + (size_t)a->logits.wgs * B * 8;
  return true;
}

extern "C" size_t pta_gpt2_step_workspace_bytes(const pta_gpt2_model* model) {
  G2Args a;
  size_t lds, bytes;
  return g2_plan(model, &a, &lds, &bytes) ? bytes : 0;
}

template <int MB>
static int g2_launch(const G2Args& a, size_t lds, hipStream_t s) {
  static bool ready = false;
  if (!ready) {
    PTA_REQUIRE(hipFuncSetAttribute((const void*)gpt2_step_kernel<MB>, hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024) == hipSuccess,
                "pta_gpt2_step: cannot reserve LDS");
    ready = true;
  }
  hipLaunchKernelGGL(gpt2_step_kernel<MB>, dim3(a.total), dim3(G2_THREADS), lds, s, a);
  PTA_CHECK_LAUNCH("pta_gpt2_step");
  return PTA_OK;
}

extern "C" int pta_gpt2_step(const pta_gpt2_model* model, const pta_decode_state* state, void* workspace, pta_stream_t stream) {
  G2Args a;
  size_t lds, bytes;
  PTA_REQUIRE(model && state && workspace, "pta_gpt2_step: null pointer");
  if (!g2_plan(model, &a, &lds, &bytes)) {
    pta_set_error("pta_gpt2_step: unsupported shape (batch %d, %d heads, hidden %d, ffn %d, vocabulary %d)", model->batch, model->n_head, model->hidden, model->ffn,
                  model->vocab);
    return PTA_EUNSUPPORTED;
  }
  PTA_REQUIRE(model->layers && model->embed && model->positions && model->norm_weight && model->norm_bias && model->head, "pta_gpt2_step: null pointer");
  PTA_REQUIRE(state->container && state->mask && state->stop_mask && state->step && state->keep_going && state->next_ids && state->logits,
              "pta_gpt2_step: null pointer");
  PTA_REQUIRE(pta_aligned(workspace, 256) && pta_aligned(model->head, 16) && pta_aligned(model->norm_weight, 16) && pta_aligned(model->norm_bias, 16),
              "pta_gpt2_step: unaligned pointer");
  a.s = *state;
  a.ctl = (uint32_t*)workspace;
  a.slots = a.ctl + G2_CTL_WORDS;
  a.best = (unsigned long long*)((unsigned char*)workspace + bytes) - (size_t)a.logits.wgs * model->batch;
  switch (g2_rows(model->batch)) {
    case 1: return g2_launch<1>(a, lds, (hipStream_t)stream);
    case 2: return g2_launch<2>(a, lds, (hipStream_t)stream);
    case 4: return g2_launch<4>(a, lds, (hipStream_t)stream);
    default: return g2_launch<8>(a, lds, (hipStream_t)stream);
  }
}
