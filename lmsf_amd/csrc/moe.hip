// Experts chosen by a table: token id t runs the ``top`` experts table[t, 0 .. top-1], each a gated feed-forward
//     y_e(h) = Wd_e (silu(Wg_e h) * (Wu_e h)),
// and the layer's output is base + weight * sum_k y_{table[t, k]}(h) (base: what runs for every token, or nothing).
// The choice is read on the device from the step's token ids, so a step needs nothing from the host and can be
// replayed from a graph. The experts' matrices lie stacked: Wgu [E, 2 F, W] (gate rows, then up rows), Wd [E, W, F].
//
// Few tokens (decoding), and float32 at any number: every (token, choice) streams its expert's rows, a wave per
// output, the token's vector in LDS, 16-byte loads where the rows allow them.
// Many tokens in bfloat16: the (token, choice) pairs are grouped by expert on the device (one small kernel: counts,
// offsets, an order, a list of tiles of up to 160 pairs of one expert), and each tile runs on the matrix cores
// against 256 rows of its expert's matrix (A = 16 rows of W x 32 k, B = 16 pairs x 32 k; in the gated product the gate
// and the up rows of the same outputs), operands through LDS. The down product leaves float32 rows per pair; a last kernel adds a token's pairs and the shared part. A pair's result
// does not depend on where in its tile it lies, so the order inside an expert's group (atomic counters) is free.
// Accumulation in float32 throughout.
//
// The same kernels serve experts that a router chooses: ``ids`` null makes row n of the table token n's own choice (a
// table [n_tokens, top] that a kernel of the step has just written, lmsf_moe_route below); ``pair_scale`` gives every
// (token, choice) a float32 factor on the expert's *input*, y_e(s h), which the gate and up products take as a factor on
// their results before these are rounded (W (s h) = s (W h)); ``base_scale`` a float32 factor per token on ``base``;
// ``out_scale`` a float32 factor per (token, choice) on what the expert returns. Experts may also be of one matrix in,
// y_e(h) = Wd_e relu(Wu_e h)^2 with Wgu [E, F, W], or gated with bounded operands, and experts after the last may have no
// matrices and return their input (lmsf_table_moe_act). A second router (lmsf_moe_route_groups) takes softmax scores,
// chooses within the best groups of neighbouring experts and may choose by corrected scores.
#include "common.h"

#include <math.h>

#define MOE_THREADS 256
#define MOE_WAVES (MOE_THREADS / LMSF_WAVE)
#define MOE_OUT_PER_WAVE 4

// NR rows of a matrix against one vector: out[r] = sum_i w[r * ld + i] x[i] over W entries, the lanes of a wave
// together; x in LDS as float32. The loads of all rows are asked for before any is used (rows beyond ``valid`` repeat
// the last valid one).
template <typename T, int NR>
__device__ __forceinline__ void moe_rows_dot(const T* __restrict__ w, long ld, int valid, const float* __restrict__ x,
                                             int W, int lane, bool vec, float* out) {
  float a[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) a[r] = 0.f;
  if (vec) {
    constexpr int V = Vec16<T>::N;
    for (int i = lane * V; i < W; i += LMSF_WAVE * V) {
      Vec16<T> p[NR];
#pragma unroll
      for (int r = 0; r < NR; ++r) p[r].load(w + (long)min(r, valid - 1) * ld + i);
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const float xv = x[i + e];
#pragma unroll
        for (int r = 0; r < NR; ++r) a[r] += p[r].get(e) * xv;
      }
    }
  } else {
    for (int i = lane; i < W; i += LMSF_WAVE) {
      const float xv = x[i];
#pragma unroll
      for (int r = 0; r < NR; ++r) a[r] += to_f32<T>(w[(long)min(r, valid - 1) * ld + i]) * xv;
    }
  }
#pragma unroll
  for (int r = 0; r < NR; ++r) out[r] = wave_sum(a[r]);
}

// act[(n * top + k), f] = silu(Wg_e[f] . h[n]) * (Wu_e[f] . h[n]),  e = table[ids[n], k]
template <typename T>
__global__ __launch_bounds__(MOE_THREADS) void moe_gate_up_kernel(
    const T* __restrict__ h, long h_stride, const T* __restrict__ Wgu, const int* __restrict__ ids,
    const int* __restrict__ table, int vocab, int top, int E, T* __restrict__ act, int F, int W, int vec,
    const float* __restrict__ pair_scale, int gated, float limit, int identity) {
  extern __shared__ float sh[];   // [W]
  const int nk = blockIdx.x, n = nk / top, k = nk - n * top;
  const int id = min(max(ids ? ids[n] : n, 0), vocab - 1);
  const int e = min(max(table[(long)id * top + k], 0), E + identity - 1);
  if (e >= E) return;             // (what an expert without matrices returns is its input: the kernel below)
  const float ps = pair_scale ? pair_scale[nk] : 1.f;
  for (int i = threadIdx.x; i < W; i += MOE_THREADS) sh[i] = ps * to_f32<T>(h[(long)n * h_stride + i]);
  __syncthreads();
  const int wave = threadIdx.x / LMSF_WAVE, lane = threadIdx.x % LMSF_WAVE;
  const int f0 = (blockIdx.y * MOE_WAVES + wave) * MOE_OUT_PER_WAVE;
  const T* We = Wgu + (long)e * (gated ? 2 : 1) * F * W;
  if (f0 >= F) return;
  const int valid = min(MOE_OUT_PER_WAVE, F - f0);
  float ag[MOE_OUT_PER_WAVE], au[MOE_OUT_PER_WAVE];
  moe_rows_dot<T, MOE_OUT_PER_WAVE>(We + (long)f0 * W, W, valid, sh, W, lane, vec, ag);
  if (!gated) {
    // one matrix an expert: act = relu(W_up h)^2, the product rounded as a stored activation is
    if (lane < valid) {
      float uu = 0.f;
#pragma unroll
      for (int r = 0; r < MOE_OUT_PER_WAVE; ++r)
        if (r == lane) uu = fmaxf(to_f32<T>(from_f32<T>(ag[r])), 0.f);
      act[(long)nk * F + f0 + lane] = from_f32<T>(uu * uu);
    }
    return;
  }
  moe_rows_dot<T, MOE_OUT_PER_WAVE>(We + (long)(F + f0) * W, W, valid, sh, W, lane, vec, au);
  if (lane < valid) {
    // the two products are rounded as stored activations are, then the activation in float32
    float gg = 0.f, uu = 0.f;
#pragma unroll
    for (int r = 0; r < MOE_OUT_PER_WAVE; ++r)
      if (r == lane) {
        gg = to_f32<T>(from_f32<T>(ag[r]));
        uu = to_f32<T>(from_f32<T>(au[r]));
      }
    act[(long)nk * F + f0 + lane] = from_f32<T>(limit > 0.f ? bounded_gate(gg, uu, limit) : gg / (1.f + expf(-gg)) * uu);
  }
}

// total + f v for output o: rounded once, and for every fourth output with the product rounded first, so that the two
// kernels that add up a token's experts give the same bits (left to itself the compiler shares one addition between the
// kinds of experts for the last output that a wave owns, which is not the same one in both).
__device__ __forceinline__ float moe_add(float total, float f, float v, int o) {
  float p = f * v;
  asm volatile("" : "+v"(p));
  return (o & 3) == 3 ? total + p : fmaf(f, v, total);
}

// out[n, o] = base[n, o] + weight * sum_k Wd_{e_k}[o] . act[n * top + k]
template <typename T>
__global__ __launch_bounds__(MOE_THREADS) void moe_down_kernel(
    const T* __restrict__ act, const T* __restrict__ Wd, const int* __restrict__ ids, const int* __restrict__ table,
    int vocab, int top, int E, float weight, const T* __restrict__ base, long base_stride, T* __restrict__ out,
    long out_stride, int F, int W, int vec, const float* __restrict__ base_scale,
    const float* __restrict__ out_scale, int identity, const T* __restrict__ h, long h_stride,
    const float* __restrict__ pair_scale) {
  extern __shared__ float sa[];   // [top, F]
  const int n = blockIdx.x;
  const int id = min(max(ids ? ids[n] : n, 0), vocab - 1);
  for (int i = threadIdx.x; i < top * F; i += MOE_THREADS) sa[i] = to_f32<T>(act[(long)n * top * F + i]);
  __syncthreads();
  const int wave = threadIdx.x / LMSF_WAVE, lane = threadIdx.x % LMSF_WAVE;
  const int o0 = (blockIdx.y * MOE_WAVES + wave) * MOE_OUT_PER_WAVE;
  if (o0 >= W) return;
  const int valid = min(MOE_OUT_PER_WAVE, W - o0);
  float total[MOE_OUT_PER_WAVE];
#pragma unroll
  for (int r = 0; r < MOE_OUT_PER_WAVE; ++r) total[r] = 0.f;
  for (int k = 0; k < top; ++k) {
    const int e = min(max(table[(long)id * top + k], 0), E + identity - 1);
    float part[MOE_OUT_PER_WAVE];
    const float os = out_scale ? out_scale[(long)n * top + k] : 1.f;
    if (e >= E) {      // an expert without matrices returns its input
      const float f = os * (pair_scale ? pair_scale[(long)n * top + k] : 1.f);
#pragma unroll
      for (int r = 0; r < MOE_OUT_PER_WAVE; ++r)
        total[r] = moe_add(total[r], f, to_f32<T>(h[(long)n * h_stride + o0 + min(r, valid - 1)]), o0 + r);
      continue;
    }
    moe_rows_dot<T, MOE_OUT_PER_WAVE>(Wd + ((long)e * W + o0) * F, F, valid, sa + k * F, F, lane, vec, part);
#pragma unroll
    for (int r = 0; r < MOE_OUT_PER_WAVE; ++r) total[r] = moe_add(total[r], os, part[r], o0 + r);
  }
  if (lane < valid) {
    float mine = 0.f;
#pragma unroll
    for (int r = 0; r < MOE_OUT_PER_WAVE; ++r)
      if (r == lane) mine = total[r];
    float b = base ? to_f32<T>(base[(long)n * base_stride + o0 + lane]) : 0.f;
    if (base_scale) b *= base_scale[n];
    out[(long)n * out_stride + o0 + lane] = from_f32<T>(b + weight * mine);
  }
}

// ---------------------------------------------------------------- few tokens, rows that allow 16-byte loads
//
// The same two products with everything that comes from memory asked for in one go, and a read of an expert's rows
// shared by up to MOE_SHARED_PAIRS of the pairs that have chosen it (where more have, other workgroups take the next ones
// side by side). A wave reads its rows of the matrix and the same entries of the vectors (which the caches hold) with
// 16-byte loads, MOE_AHEAD pieces of 512 or 256 entries of each row on their way at a time; nothing goes through LDS and
// no wave waits for another. Every output is added up in the order of the kernels above. In the first product the outputs
// vary fastest over the workgroups, so that an expert's rows are read by all eight dies (with the pairs fastest, a pair's
// whole expert falls to one die: gate and up 26.5 us). In the second the tokens vary fastest within a die, so that a row
// that several tokens need comes to a die once: 32 tokens in float32, 4,096 -> 2 x 1,536 -> 4,096, with one pair of
// experts 268 -> 203 us, with experts of their own choice 380 -> 305. What bounds them is memory and, for an expert of
// several pairs, the multiply-adds of a wave. Both products of 2,048 -> 2 x 1,024 -> 2,048 in bfloat16, kernels above ->
// these: 8 tokens with 2 of 16 experts each 40.6 -> 33.1 us, 31 tokens with one expert 38.6 -> 28.3 (in float32 44.3 ->
// 34.3); of one matrix 28.9 -> 22.4 and 30.0 -> 22.7; 4 pieces ahead, 2 pairs a read, 1 or 4 outputs a wave: up to a
// third slower.
#define MOE_AHEAD 2
#define MOE_FEW_PAIRS 64      // a lane each
#define MOE_SHARED_PAIRS 4    // pairs of one expert that share a read of its rows
#define MOE_FEW_OUT 2         // outputs a wave owns
// Smaller experts stay with the kernels above, which share a vector between a workgroup's waves: what counts there is the
// way from a wave's first load to its last sum (2 x 512 x 256 entries, 30 pairs of two experts from memory: 10.6 -> 12.6
// us here; 2 x 1,024 x 512 level to 1.14 times as long with all pairs on one expert, 0.75 times with the pairs spread). From
// 1,536 x 512 on everything measured is faster but 31 pairs on one expert of one matrix of that size, 18.5 -> 20.9 us in
// float32 (spread over 16 experts 32.3 -> 19.4).
#define MOE_FEW_ENTRIES (3L << 18)

// a[q][r] += sum over this lane's entries of rows r against the vectors of the pairs, each times its scale
template <typename T, int ROWS, int PAIRS>
__device__ __forceinline__ void moe_few_dot(const T* const (&w)[ROWS], const T* const (&x)[PAIRS], const float (&scale)[PAIRS],
                                            int n_pairs, int W, int lane, float (&a)[PAIRS][ROWS]) {
  constexpr int V = Vec16<T>::N, STEP = LMSF_WAVE * V;
  for (int i0 = lane * V; i0 < W; i0 += MOE_AHEAD * STEP) {
    Vec16<T> p[MOE_AHEAD][ROWS], xv[PAIRS][MOE_AHEAD];
#pragma unroll
    for (int u = 0; u < MOE_AHEAD; ++u) {
      const int i = i0 + u * STEP;
      if (i < W) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) p[u][r].load(w[r] + i);
      }
    }
#pragma unroll
    for (int q = 0; q < PAIRS; ++q) {
      if (q >= n_pairs) break;
#pragma unroll
      for (int u = 0; u < MOE_AHEAD; ++u)
        if (i0 + u * STEP < W) xv[q][u].load(x[q] + i0 + u * STEP);
    }
#pragma unroll
    for (int q = 0; q < PAIRS; ++q) {
      if (q >= n_pairs) break;
#pragma unroll
      for (int u = 0; u < MOE_AHEAD; ++u) {
        if (i0 + u * STEP >= W) break;
#pragma unroll
        for (int e = 0; e < V; ++e) {
          const float f = scale[q] * xv[q][u].get(e);
#pragma unroll
          for (int r = 0; r < ROWS; ++r) a[q][r] += p[u][r].get(e) * f;
        }
      }
    }
  }
}

template <typename T, bool GATED>
__global__ __launch_bounds__(MOE_THREADS, 4) void moe_gate_up_few_kernel(
    const T* __restrict__ h, long h_stride, const T* __restrict__ Wgu, const int* __restrict__ ids,
    const int* __restrict__ table, int vocab, int top, int E, T* __restrict__ act, int F, int W, int n_pairs,
    const float* __restrict__ pair_scale, float limit, int identity) {
  const int wave = threadIdx.x / LMSF_WAVE, lane = threadIdx.x % LMSF_WAVE;
  const int f0 = (blockIdx.x * MOE_WAVES + wave) * MOE_FEW_OUT;
  if (f0 >= F) return;
  int mine = -1;                  // the expert of pair ``lane``
  if (lane < n_pairs) {
    const int n = lane / top, id = min(max(ids ? ids[n] : n, 0), vocab - 1);
    mine = min(max(table[(long)id * top + lane - n * top], 0), E + identity - 1);
  }
  const int e = __shfl(mine, blockIdx.y, LMSF_WAVE);
  if (e >= E) return;             // (what an expert without matrices returns is its input: the kernel below)
  // of an expert's pairs every MOE_SHARED_PAIRS-th stands for itself and the ones up to the next such pair
  unsigned long long pairs = __ballot(mine == e);
  const unsigned long long before = pairs & ((1ull << blockIdx.y) - 1);
  if (__popcll(before) % MOE_SHARED_PAIRS) return;
  pairs ^= before;
  const T* We = Wgu + (long)e * (GATED ? 2 : 1) * F * W;
  const int valid = min(MOE_FEW_OUT, F - f0);
  constexpr int ROWS = (GATED ? 2 : 1) * MOE_FEW_OUT;
  const T* w[ROWS];
#pragma unroll
  for (int r = 0; r < MOE_FEW_OUT; ++r) {
    w[r] = We + (long)(f0 + min(r, valid - 1)) * W;
    if (GATED) w[ROWS - MOE_FEW_OUT + r] = w[r] + (long)F * W;
  }
  const T* x[MOE_SHARED_PAIRS];
  float scale[MOE_SHARED_PAIRS], a[MOE_SHARED_PAIRS][ROWS];
  int pair[MOE_SHARED_PAIRS], count = 0;
#pragma unroll
  for (int q = 0; q < MOE_SHARED_PAIRS; ++q) {
    pair[q] = 0;
    if (pairs) {
      pair[q] = __ffsll(pairs) - 1;
      pairs &= pairs - 1;
      ++count;
    }
    x[q] = h + (long)(pair[q] / top) * h_stride;
    scale[q] = pair_scale ? pair_scale[pair[q]] : 1.f;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) a[q][r] = 0.f;
  }
  moe_few_dot<T, ROWS, MOE_SHARED_PAIRS>(w, x, scale, count, W, lane, a);
#pragma unroll
  for (int q = 0; q < MOE_SHARED_PAIRS; ++q) {
    if (q >= count) break;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) a[q][r] = wave_sum(a[q][r]);
    if (lane < valid) {
      // the products are rounded as stored activations are, then the activation in float32
      const float gg = to_f32<T>(from_f32<T>(lane == 0 ? a[q][0] : a[q][1]));
      const float uu = to_f32<T>(from_f32<T>(lane == 0 ? a[q][ROWS - 2] : a[q][ROWS - 1]));
      float y;
      if (!GATED) {
        const float up = fmaxf(gg, 0.f);      // one matrix an expert: relu(W_up h)^2
        y = up * up;
      } else {
        y = limit > 0.f ? bounded_gate(gg, uu, limit) : gg / (1.f + expf(-gg)) * uu;
      }
      act[(long)pair[q] * F + f0 + lane] = from_f32<T>(y);
    }
  }
}

template <typename T>
__global__ __launch_bounds__(MOE_THREADS) void moe_down_few_kernel(
    const T* __restrict__ act, const T* __restrict__ Wd, const int* __restrict__ ids, const int* __restrict__ table,
    int vocab, int top, int E, float weight, const T* __restrict__ base, long base_stride, T* __restrict__ out,
    long out_stride, int F, int W, const float* __restrict__ base_scale, const float* __restrict__ out_scale,
    int identity, const T* __restrict__ h, long h_stride, const float* __restrict__ pair_scale, int n_tokens) {
  const int wave = threadIdx.x / LMSF_WAVE, lane = threadIdx.x % LMSF_WAVE;
  const int i = blockIdx.x / 8, n = i % n_tokens;
  const int o0 = ((i / n_tokens * 8 + blockIdx.x % 8) * MOE_WAVES + wave) * MOE_FEW_OUT;
  if (o0 >= W) return;
  const int valid = min(MOE_FEW_OUT, W - o0);
  const int id = min(max(ids ? ids[n] : n, 0), vocab - 1);
  float total[MOE_FEW_OUT];
#pragma unroll
  for (int r = 0; r < MOE_FEW_OUT; ++r) total[r] = 0.f;
  float b = 0.f;
  if (lane < valid && base) b = to_f32<T>(base[(long)n * base_stride + o0 + lane]);
#pragma unroll 2
  for (int k = 0; k < top; ++k) {
    const int e = min(max(table[(long)id * top + k], 0), E + identity - 1);
    const float os = out_scale ? out_scale[(long)n * top + k] : 1.f;
    if (e >= E) {      // an expert without matrices returns its input
      const float f = os * (pair_scale ? pair_scale[(long)n * top + k] : 1.f);
#pragma unroll
      for (int r = 0; r < MOE_FEW_OUT; ++r)
        total[r] = moe_add(total[r], f, to_f32<T>(h[(long)n * h_stride + o0 + min(r, valid - 1)]), o0 + r);
      continue;
    }
    const T* w[MOE_FEW_OUT];
    const T* x[1] = {act + ((long)n * top + k) * F};
    const float one[1] = {1.f};
    float a[1][MOE_FEW_OUT];
#pragma unroll
    for (int r = 0; r < MOE_FEW_OUT; ++r) {
      w[r] = Wd + ((long)e * W + o0 + min(r, valid - 1)) * F;
      a[0][r] = 0.f;
    }
    moe_few_dot<T, MOE_FEW_OUT, 1>(w, x, one, 1, F, lane, a);
#pragma unroll
    for (int r = 0; r < MOE_FEW_OUT; ++r) total[r] = moe_add(total[r], os, wave_sum(a[0][r]), o0 + r);
  }
  if (lane < valid) {
    if (base_scale) b *= base_scale[n];
    out[(long)n * out_stride + o0 + lane] = from_f32<T>(b + weight * (lane == 0 ? total[0] : total[1]));
  }
}

// ---------------------------------------------------------------- many tokens: grouped by expert, matrix cores

#define MOE_TILE 160         // pairs a tile holds

// Groups the P = N * top pairs by expert. order[i]: the pair at place i of the grouped sequence; tiles: for every
// tile (of up to ``tile_pairs`` pairs) its expert, its first place and its number of pairs; n_tiles[0]: how many
// tiles there are. One workgroup.
__global__ __launch_bounds__(1024) void moe_group_kernel(const int* __restrict__ ids, const int* __restrict__ table,
                                                        int vocab, int top, int E, int identity, int P, int tile_pairs,
                                                        int* __restrict__ order, int* __restrict__ tiles,
                                                        int* __restrict__ n_tiles) {
  extern __shared__ int sm[];   // [E] counts, [E] first places, [E] fill counters
  constexpr int HELD = 8;       // pairs whose experts a thread keeps between the two walks
  int* cnt = sm;
  int* first = sm + E;
  int* fill = sm + 2 * E;
  const int tid = threadIdx.x, step = blockDim.x;
  const auto expert_of = [&](int p) {
    const int id = min(max(ids ? ids[p / top] : p / top, 0), vocab - 1);
    return min(max(table[(long)id * top + p % top], 0), E + identity - 1);
  };
  int held[HELD];
#pragma unroll
  for (int i = 0; i < HELD; ++i) held[i] = tid + i * step < P ? expert_of(tid + i * step) : E;
  for (int e = tid; e < E; e += step) cnt[e] = fill[e] = 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < HELD; ++i)
    if (held[i] < E) atomicAdd(&cnt[held[i]], 1);
  for (int p = tid + HELD * step; p < P; p += step) {
    const int e = expert_of(p);
    if (e < E) atomicAdd(&cnt[e], 1);
  }
  __syncthreads();
  if (tid < LMSF_WAVE) {
    // places and tiles of 64 experts at a time: running sums over the lanes
    int at = 0, t = 0;
    for (int e0 = 0; e0 < E; e0 += LMSF_WAVE) {
      const int e = e0 + tid, n = e < E ? cnt[e] : 0, mine = (n + tile_pairs - 1) / tile_pairs;
      int places = n, tl = mine;
      for (int o = 1; o < LMSF_WAVE; o <<= 1) {
        const int up = __shfl_up(places, o, LMSF_WAVE), ut = __shfl_up(tl, o, LMSF_WAVE);
        if (tid >= o) {
          places += up;
          tl += ut;
        }
      }
      const int begin = at + places - n;
      if (e < E) first[e] = begin;
      for (int i = 0; i < mine; ++i) {
        int* to = tiles + 3 * (t + tl - mine + i);
        to[0] = e;
        to[1] = begin + i * tile_pairs;
        to[2] = min(tile_pairs, n - i * tile_pairs);
      }
      at += __shfl(places, LMSF_WAVE - 1, LMSF_WAVE);
      t += __shfl(tl, LMSF_WAVE - 1, LMSF_WAVE);
    }
    if (tid == 0) n_tiles[0] = t;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < HELD; ++i)
    if (held[i] < E) order[first[held[i]] + atomicAdd(&fill[held[i]], 1)] = tid + i * step;
  for (int p = tid + HELD * step; p < P; p += step) {
    const int e = expert_of(p);
    if (e < E) order[first[e] + atomicAdd(&fill[e], 1)] = p;
  }
}

// One tile of up to 160 pairs against 256 rows of its expert's matrix, operands through LDS: 128 outputs with gate and up (KIND
// 1: x = the tokens' vectors, row of pair p: p / top, Wm = Wgu, K = W, O = F, y = act [P, F] bfloat16 = silu(gate) * up), or 256
// outputs (KIND 0: x = act, row of pair p: p, Wm = Wd, K = F, O = W, y = float32 rows [P, W]; KIND 2: one matrix an expert, Wm
// [E, O, K], with relu(.)^2). In a step of 64 k the 256 rows of W and the 160 pairs' rows, 128 bytes of each (whole cache lines:
// with 64 every line came to the compute unit twice), travel from memory straight into LDS (global_load_lds_dwordx4), two
// of MOE_STAGES steps on their way at a time, one barrier a step. The 16-byte piece c of row r lies in slot (c + r) mod 8 of
// its row, so that the fragments' reads meet distinct banks. Eight waves, two a SIMD, wait for LDS in turn: two rows of them
// over the pairs, four columns over W; a wave leaves out the 16s of pairs that its tile does not have. The blocks of outputs vary
// fastest over the workgroups and fall to the dies in turn, so that an expert's rows are read by one die, whose tiles of
// that expert share them in its L2. What bounds the kernel is these rows' way into the compute units.
// 3,994 pairs of 16 experts, 2,048 -> 2 x 1,024 -> 2,048, all four kernels, with tiles of 128 pairs by 128 outputs copied through
// registers 32 k at a time 217 -> 116 us; 66 pairs 77 -> 55; 8,192 pairs of 8, 4,096 -> 2 x 1,536 -> 4,096, 766 -> 583. Many or small experts,
// most of whose tiles are nearly empty, gain as well (weights not in cache): 64 of 2,048 -> 2 x 1,024, 32 / 256 / 2,048 pairs 133 / 226 / 256 ->
// 96 / 195 / 220; 128 of 1,024 -> 2 x 256 59 / 76 / 91 -> 35 / 57 / 66; 512 of these 75 / 141 / 258 -> 41 / 97 / 186; 8 of 256 -> 2 x 256 24 / 36 / 49
// -> 21 / 27 / 42; 64 of 512 -> 256, one matrix in, 32 / 36 / 47 -> 27 / 28 / 37. Least where the experts' rows are all there is: 32 of 4,096 ->
// 2 x 2,048, 64 to 256 pairs 0.92 to 0.94 of the time.
#define MOE_TILE_ROWS 256
#define MOE_TILE_WAVES 8
#define MOE_STAGES 3
#define MOE_STAGE_BYTES ((MOE_TILE_ROWS + MOE_TILE) * 128)

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"   // m0 is named as clobbered on purpose
// (inline assembly: through the compiler's builtin every LDS read that follows would wait for all transfers in flight; the
// waits are explicit)
__device__ __forceinline__ void moe_global_to_lds_16(const void* src, unsigned lds_base_uniform) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds_base_uniform)
               : "memory", "m0");
}
#pragma clang diagnostic pop

template <int KIND>
__global__ __launch_bounds__(MOE_TILE_WAVES * 64) void moe_tile_lds_kernel(
    const bf16_t* __restrict__ x, long x_stride, int top, const bf16_t* __restrict__ Wm, const int* __restrict__ order,
    const int* __restrict__ tiles, const int* __restrict__ n_tiles, void* __restrict__ y, int O, int K, int o_blocks,
    const float* __restrict__ pair_scale, float limit) {
  constexpr bool GATED = KIND == 1, UP = KIND != 0;
  constexpr int OUTS = GATED ? MOE_TILE_ROWS / 2 : MOE_TILE_ROWS;    // outputs a workgroup
  constexpr int OW = OUTS / (MOE_TILE_WAVES / 2);  // and a wave
  constexpr int NA = MOE_TILE_ROWS / (MOE_TILE_WAVES / 2) / 16;      // fragments of W a wave
  constexpr int NB = MOE_TILE / 32;                // and of the pairs
  constexpr int STAGES = MOE_STAGES, STAGE = MOE_STAGE_BYTES;
  constexpr int ROWS8 = STAGE / 1024;              // transfers of 8 rows a step
  constexpr int LOADS = (ROWS8 + MOE_TILE_WAVES - 1) / MOE_TILE_WAVES;   // and those of a wave
  extern __shared__ __align__(16) unsigned char lds[];
  const int t = blockIdx.x / o_blocks, o_base = (blockIdx.x - t * o_blocks) * OUTS;
  if (t >= n_tiles[0] || o_base >= O) return;
  const int e = tiles[3 * t], place = tiles[3 * t + 1], count = tiles[3 * t + 2];
  const int tid = threadIdx.x, wave = tid / LMSF_WAVE, lane = tid % LMSF_WAVE;
  const int fr = lane % 16, fg = lane / 16;
  const int wr = wave / (MOE_TILE_WAVES / 2), wc = wave % (MOE_TILE_WAVES / 2);   // the wave's half of the pairs and OW outputs
  // what this lane moves: slot lane % 8 of row lane / 8 of a transfer's 8 rows (transfers beyond the last are the last again)
  const int piece = ((lane & 7) - (lane >> 3)) & 7;
  const bf16_t* src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int r = min(wave * LOADS + i, ROWS8 - 1) * 8 + (lane >> 3);    // W (gated: 128 gate rows, 128 up rows), then the pairs
    if (r < MOE_TILE_ROWS) {
      const int o = min(o_base + (r & (OUTS - 1)), O - 1);
      src[i] = Wm + ((long)e * (GATED ? 2 : 1) * O + (r >= OUTS ? O : 0) + o) * K + piece * 8;
    } else {
      const int p = order[place + min(r - MOE_TILE_ROWS, count - 1)];
      src[i] = x + (long)(UP ? p / top : p) * x_stride + piece * 8;
    }
  }
  f32x4_t acc[NA][NB];
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int mt = 0; mt < NB; ++mt) acc[a][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // 16s of pairs that the wave has: an expert's last tile may be nearly empty
  const int mine = __builtin_amdgcn_readfirstlane((count - wr * (MOE_TILE / 2) + 15) / 16);
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) const unsigned char*)lds;
  const int n_steps = (K + 63) / 64;               // K is a multiple of 32: the last step may be half a one
  auto issue = [&](int step, int stage_byte) {
    // (the second half of a last half step is fetched from the first half's place and not multiplied)
    const int k = step * 64 - (step * 64 + 32 >= K && piece >= 4 ? 32 : 0);
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      moe_global_to_lds_16(src[i] + k, __builtin_amdgcn_readfirstlane(lds0 + stage_byte + min(wave * LOADS + i, ROWS8 - 1) * 1024));
  };
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < n_steps) issue(s, s * STAGE);
  int consume = 0, produce = (STAGES - 1) * STAGE;
  for (int it = 0; it < n_steps; ++it) {
    // step ``it`` has arrived when at most the transfers of the later steps are outstanding
    if (it + STAGES - 2 < n_steps)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 2) * LOADS) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();      // everybody's part of step ``it`` is there, and everybody is done with step ``it - 1``
    if (it + STAGES - 1 < n_steps) issue(it + STAGES - 1, produce);
    produce = produce + STAGE == STAGES * STAGE ? 0 : produce + STAGE;
    const unsigned char* buf = lds + consume;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (it * 64 + s * 32 >= K) break;
      const int at = fr * 128 + (((s * 4 + fg) + fr) & 7) * 16;
      bf16x8_t fa[NA], fb[NB];
#pragma unroll
      for (int a = 0; a < NA; ++a)       // fragment a: outputs wc * OW + (a * 16) mod OW ..; gated: the second half are the up rows of the same outputs
        fa[a] = *reinterpret_cast<const bf16x8_t*>(buf + ((a * 16 >= OW ? OUTS : 0) + wc * OW + (a * 16) % OW) * 128 + at);
#pragma unroll
      for (int mt = 0; mt < NB; ++mt)
        if (mt < mine) fb[mt] = *reinterpret_cast<const bf16x8_t*>(buf + (MOE_TILE_ROWS + wr * (MOE_TILE / 2) + mt * 16) * 128 + at);
#pragma unroll
      for (int mt = 0; mt < NB; ++mt)
        if (mt < mine) {
#pragma unroll
          for (int a = 0; a < NA; ++a) acc[a][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[a], fb[mt], acc[a][mt], 0, 0, 0);
        }
    }
    consume = consume + STAGE == STAGES * STAGE ? 0 : consume + STAGE;
  }
  // lane: pair wr * (MOE_TILE / 2) + mt * 16 + fr, outputs o_base + wc * OW + a * 16 + fg * 4 .. + 3 (O is a multiple of 32)
  const bool wide = ((uintptr_t)y & 15) == 0;
#pragma unroll
  for (int mt = 0; mt < NB; ++mt) {
    const int slot = wr * (MOE_TILE / 2) + mt * 16 + fr;
    if (slot >= count) continue;
    const int p = order[place + slot];
    const float ps = UP && pair_scale ? pair_scale[p] : 1.f;
#pragma unroll
    for (int a = 0; a < OW / 16; ++a) {
      const int o = o_base + wc * OW + a * 16 + fg * 4;
      if (o >= O) continue;
      float r[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (GATED) {
          const float g = bf16_to_f32(f32_to_bf16(ps * acc[a][mt][j])), u = bf16_to_f32(f32_to_bf16(ps * acc[NA - OW / 16 + a][mt][j]));
          r[j] = limit > 0.f ? bounded_gate(g, u, limit) : g / (1.f + expf(-g)) * u;
        } else if (UP) {
          const float u = fmaxf(bf16_to_f32(f32_to_bf16(ps * acc[a][mt][j])), 0.f);
          r[j] = u * u;
        } else {
          r[j] = acc[a][mt][j];
        }
      }
      if (UP) {
        bf16_t* to = reinterpret_cast<bf16_t*>(y) + (long)p * O + o;
        if (wide) {
          *reinterpret_cast<uint2*>(to) = make_uint2(pack2_bf16(r[0], r[1]), pack2_bf16(r[2], r[3]));
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) to[j] = f32_to_bf16(r[j]);
        }
      } else {
        float* to = reinterpret_cast<float*>(y) + (long)p * O + o;
        if (wide) {
          *reinterpret_cast<float4*>(to) = make_float4(r[0], r[1], r[2], r[3]);
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) to[j] = r[j];
        }
      }
    }
  }
}

template <int KIND>
static int launch_moe_tiles(int max_tiles, hipStream_t stream, const bf16_t* x, long x_stride, int top, const bf16_t* Wm,
                            const int* order, const int* tiles, const int* n_tiles, void* y, int O, int K,
                            const float* pair_scale, float limit) {
  constexpr int smem = MOE_STAGES * MOE_STAGE_BYTES, OUTS = KIND == 1 ? MOE_TILE_ROWS / 2 : MOE_TILE_ROWS;
  static bool configured = false;   // per instantiation
  if (!configured) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(moe_tile_lds_kernel<KIND>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    if (e != hipSuccess) {
      lmsf_set_error("table_moe: cannot reserve %d bytes of LDS: %s", smem, hipGetErrorString(e));
      return 2;
    }
    configured = true;
  }
  // (blocks of outputs up to a multiple of 8, one for every die in turn; the surplus ends at once)
  const int blocks = (O + OUTS - 1) / OUTS, o_blocks = blocks > 4 ? (blocks + 7) / 8 * 8 : blocks;
  LMSF_CHECK((long)max_tiles * o_blocks < 2147483647L, "table_moe: too many tiles");
  hipLaunchKernelGGL((moe_tile_lds_kernel<KIND>), dim3((unsigned)(max_tiles * o_blocks)),
                     dim3(MOE_TILE_WAVES * 64), smem, stream, x, x_stride,
                     top, Wm, order, tiles, n_tiles, y, O, K, o_blocks, pair_scale, limit);
  return 0;
}

// out[n, o] = base[n, o] + weight * sum_k rows[n * top + k, o]; the choices of ``table`` (row ids[n], or n) from E on are
// experts without matrices, which return their input. VEC: four neighbours a thread (W and the strides multiples of 4).
template <bool VEC>
__global__ __launch_bounds__(256) void moe_combine_kernel(const float* __restrict__ rows, int top, float weight,
                                                          const bf16_t* __restrict__ base, long base_stride,
                                                          bf16_t* __restrict__ out, long out_stride, int W,
                                                          const float* __restrict__ base_scale,
                                                          const float* __restrict__ out_scale,
                                                          const int* __restrict__ ids, const int* __restrict__ table,
                                                          int vocab, int E, int identity,
                                                          const bf16_t* __restrict__ h, long h_stride,
                                                          const float* __restrict__ pair_scale) {
  const int n = blockIdx.x;
  const int* chosen = table + (long)(identity > 0 ? min(max(ids ? ids[n] : n, 0), vocab - 1) : 0) * top;
  const float bs = base_scale ? base_scale[n] : 1.f;
  constexpr int V = VEC ? 4 : 1;
  for (int o = threadIdx.x * V; o < W; o += 256 * V) {
    float s[4], x[4];
#pragma unroll
    for (int j = 0; j < V; ++j) s[j] = 0.f;
    auto bf4 = [&](const bf16_t* p) {
      if (VEC) {
        const uint2 v = *reinterpret_cast<const uint2*>(p);
        x[0] = __uint_as_float(v.x << 16), x[1] = __uint_as_float(v.x & 0xffff0000u);
        x[2] = __uint_as_float(v.y << 16), x[3] = __uint_as_float(v.y & 0xffff0000u);
      } else {
        x[0] = bf16_to_f32(p[0]);
      }
    };
    for (int k = 0; k < top; ++k) {
      float f = out_scale ? out_scale[(long)n * top + k] : 1.f;
      if (identity > 0 && chosen[k] >= E) {
        bf4(h + (long)n * h_stride + o);
        if (pair_scale) f *= pair_scale[(long)n * top + k];
      } else {
        const float* p = rows + ((long)n * top + k) * W + o;
        if (VEC) {
          const float4 v = *reinterpret_cast<const float4*>(p);
          x[0] = v.x, x[1] = v.y, x[2] = v.z, x[3] = v.w;
        } else {
          x[0] = p[0];
        }
      }
#pragma unroll
      for (int j = 0; j < V; ++j) s[j] += f * x[j];
    }
#pragma unroll
    for (int j = 0; j < V; ++j) s[j] *= weight;
    if (base) {
      bf4(base + (long)n * base_stride + o);
#pragma unroll
      for (int j = 0; j < V; ++j) s[j] = bs * x[j] + s[j];
    }
    bf16_t* y = out + (long)n * out_stride + o;
    if (VEC) *reinterpret_cast<uint2*>(y) = make_uint2(pack2_bf16(s[0], s[1]), pack2_bf16(s[2], s[3]));
    else y[0] = f32_to_bf16(s[0]);
  }
}

// ints and floats of scratch that the grouped form needs for n_tokens tokens
extern "C" long lmsf_table_moe_scratch_ints(int n_tokens, int top, int E) {
  const long P = (long)n_tokens * top;
  return P + 3 * (P / MOE_TILE + E + 1) + 4;
}

// whether lmsf_table_moe takes the grouped form for these sizes (then it needs the scratch: ints as above,
// floats n_tokens * top * W)
extern "C" int lmsf_table_moe_grouped(int dtype, int n_tokens, int top, int E, int F, int W, long h_stride) {
  return dtype == LMSF_BF16 && (long)n_tokens * top >= 32 && W % 32 == 0 && F % 32 == 0 && h_stride % 8 == 0 &&
         E <= 4096;
}

// ``act_kind`` 0: gated experts, Wgu [E, 2 F, W]; 1: experts of one matrix, Wgu [E, F, W], y_e(h) = Wd_e relu(Wu_e h)^2.
// 2: gated experts whose activation has both operands bounded by ``limit`` (common.h: bounded_gate).
// ``out_scale``: a float32 factor per (token, choice) on what the expert returns (null: none). ``identity``: so many
// experts after the E with matrices (choices E .. E + identity - 1) have none and return their input.
extern "C" int lmsf_table_moe_act(const void* h, int dtype, long h_stride, const void* Wgu, const void* Wd,
                                  const int* ids, const int* table, int vocab, int top, int E, float weight,
                                  const void* base, long base_stride, const float* pair_scale,
                                  const float* base_scale, const float* out_scale, int act_kind, float limit,
                                  int identity, void* act, void* out,
                                  long out_stride, int n_tokens, int F, int W, int* scratch_ints,
                                  float* scratch_rows, hipStream_t stream) {
  LMSF_CHECK(act_kind >= 0 && act_kind <= 2, "table_moe: unknown kind of expert %d", act_kind);
  LMSF_CHECK((act_kind == 2) == (limit > 0.f) && identity >= 0, "table_moe: a limit goes with bounded experts");
  const int gated = act_kind != 1;
  LMSF_CHECK(h && Wgu && Wd && table && act && out, "table_moe: null pointer");
  LMSF_CHECK(ids || vocab >= n_tokens, "table_moe: without token ids the table has a row per token");
  LMSF_CHECK(dtype == LMSF_F32 || dtype == LMSF_BF16, "table_moe: unknown dtype code %d", dtype);
  LMSF_CHECK(vocab > 0 && top > 0 && E > 0 && F > 0 && W > 0, "table_moe: bad sizes");
  LMSF_CHECK(h_stride >= W && out_stride >= W && (!base || base_stride >= W), "table_moe: rows overlap");
  LMSF_CHECK((size_t)W * 4 <= 64 * 1024 && (size_t)top * F * 4 <= 64 * 1024, "table_moe: a row does not fit LDS");
  LMSF_CHECK((long)n_tokens * top < 2147483647L, "table_moe: too many rows");
  if (n_tokens <= 0) return 0;
  if (lmsf_table_moe_grouped(dtype, n_tokens, top, E, F, W, h_stride) && scratch_ints && scratch_rows &&
      lmsf_aligned16(h) && lmsf_aligned16(Wgu) && lmsf_aligned16(Wd) && lmsf_aligned16(act)) {
    const int P = n_tokens * top, max_tiles = P / MOE_TILE + E;
    int* order = scratch_ints;
    int* tiles = order + P;
    int* n_tiles = tiles + 3 * (max_tiles + 1);
    hipLaunchKernelGGL(moe_group_kernel, dim3(1), dim3(1024), (size_t)3 * E * 4, stream, ids, table, vocab, top, E, identity,
                       P, MOE_TILE, order, tiles, n_tiles);
    int rc = gated ? launch_moe_tiles<1>(max_tiles, stream, (const bf16_t*)h, h_stride, top, (const bf16_t*)Wgu, order, tiles, n_tiles,
                                         act, F, W, pair_scale, limit)
                   : launch_moe_tiles<2>(max_tiles, stream, (const bf16_t*)h, h_stride, top, (const bf16_t*)Wgu, order, tiles, n_tiles,
                                         act, F, W, pair_scale, limit);
    if (rc == 0)
      rc = launch_moe_tiles<0>(max_tiles, stream, (const bf16_t*)act, (long)F, top, (const bf16_t*)Wd, order, tiles, n_tiles,
                               scratch_rows, W, F, nullptr, 0.f);
    if (rc) return rc;
    const bool vec = W % 4 == 0 && out_stride % 4 == 0 && h_stride % 4 == 0 && (!base || base_stride % 4 == 0) &&
                     ((uintptr_t)out) % 8 == 0 && ((uintptr_t)base) % 8 == 0 && lmsf_aligned16(scratch_rows);
#define MOE_COMBINE(V)                                                                                                \
  hipLaunchKernelGGL((moe_combine_kernel<V>), dim3(n_tokens), dim3(256), 0, stream, scratch_rows, top, weight,        \
                     (const bf16_t*)base, base_stride, (bf16_t*)out, out_stride, W, base_scale, out_scale, ids, table, \
                     vocab, E, identity, (const bf16_t*)h, h_stride, pair_scale)
    if (vec) MOE_COMBINE(true); else MOE_COMBINE(false);
#undef MOE_COMBINE
    LMSF_LAUNCH_CHECK("table_moe (grouped)");
    return 0;
  }
  const int es16 = 16 / lmsf_elem_size(dtype);
  if ((long)n_tokens * top <= MOE_FEW_PAIRS && (long)W * F >= MOE_FEW_ENTRIES && W % es16 == 0 && F % es16 == 0 &&
      h_stride % es16 == 0 && lmsf_aligned16(h) && lmsf_aligned16(Wgu) && lmsf_aligned16(Wd) && lmsf_aligned16(act)) {
    const int outs = MOE_WAVES * MOE_FEW_OUT, P = n_tokens * top;
    const dim3 f1((F + outs - 1) / outs, P), f2((W + 8 * outs - 1) / (8 * outs) * 8 * n_tokens);
#define MOE_GATE_UP_FEW(T_, GATED_)                                                                                   \
  hipLaunchKernelGGL((moe_gate_up_few_kernel<T_, GATED_>), f1, dim3(MOE_THREADS), 0, stream, (const T_*)h, h_stride,  \
                     (const T_*)Wgu, ids, table, vocab, top, E, (T_*)act, F, W, P, pair_scale, limit, identity)
#define MOE_FEW(T_)                                                                                                   \
  do {                                                                                                                \
    if (gated) MOE_GATE_UP_FEW(T_, true); else MOE_GATE_UP_FEW(T_, false);                                            \
    hipLaunchKernelGGL((moe_down_few_kernel<T_>), f2, dim3(MOE_THREADS), 0, stream, (const T_*)act, (const T_*)Wd,    \
                       ids, table, vocab, top, E, weight, (const T_*)base, base_stride, (T_*)out, out_stride, F, W,   \
                       base_scale, out_scale, identity, (const T_*)h, h_stride, pair_scale, n_tokens);                \
  } while (0)
    if (dtype == LMSF_F32) MOE_FEW(float); else MOE_FEW(bf16_t);
#undef MOE_FEW
#undef MOE_GATE_UP_FEW
    LMSF_LAUNCH_CHECK("table_moe (few)");
    return 0;
  }
  const int per_block = MOE_WAVES * MOE_OUT_PER_WAVE;
  const dim3 g1(n_tokens * top, (F + per_block - 1) / per_block), g2(n_tokens, (W + per_block - 1) / per_block);
  const int es = lmsf_elem_size(dtype), vn = 16 / es;
  const int vec1 = W % vn == 0 && lmsf_aligned16(Wgu), vec2 = F % vn == 0 && lmsf_aligned16(Wd);
  if (dtype == LMSF_F32) {
    hipLaunchKernelGGL((moe_gate_up_kernel<float>), g1, dim3(MOE_THREADS), (size_t)W * 4, stream, (const float*)h,
                       h_stride, (const float*)Wgu, ids, table, vocab, top, E, (float*)act, F, W, vec1, pair_scale, gated, limit,
                       identity);
    hipLaunchKernelGGL((moe_down_kernel<float>), g2, dim3(MOE_THREADS), (size_t)top * F * 4, stream, (const float*)act,
                       (const float*)Wd, ids, table, vocab, top, E, weight, (const float*)base, base_stride,
                       (float*)out, out_stride, F, W, vec2, base_scale, out_scale, identity, (const float*)h, h_stride,
                       pair_scale);
  } else {
    hipLaunchKernelGGL((moe_gate_up_kernel<bf16_t>), g1, dim3(MOE_THREADS), (size_t)W * 4, stream, (const bf16_t*)h,
                       h_stride, (const bf16_t*)Wgu, ids, table, vocab, top, E, (bf16_t*)act, F, W, vec1, pair_scale, gated, limit,
                       identity);
    hipLaunchKernelGGL((moe_down_kernel<bf16_t>), g2, dim3(MOE_THREADS), (size_t)top * F * 4, stream,
                       (const bf16_t*)act, (const bf16_t*)Wd, ids, table, vocab, top, E, weight, (const bf16_t*)base,
                       base_stride, (bf16_t*)out, out_stride, F, W, vec2, base_scale, out_scale, identity,
                       (const bf16_t*)h, h_stride, pair_scale);
  }
  LMSF_LAUNCH_CHECK("table_moe");
  return 0;
}

extern "C" int lmsf_table_moe(const void* h, int dtype, long h_stride, const void* Wgu, const void* Wd, const int* ids,
                              const int* table, int vocab, int top, int E, float weight, const void* base,
                              long base_stride, const float* pair_scale, const float* base_scale, void* act, void* out,
                              long out_stride, int n_tokens, int F, int W, int* scratch_ints, float* scratch_rows,
                              hipStream_t stream) {
  return lmsf_table_moe_act(h, dtype, h_stride, Wgu, Wd, ids, table, vocab, top, E, weight, base, base_stride,
                            pair_scale, base_scale, nullptr, 0, 0.f, 0, act, out, out_stride, n_tokens, F, W, scratch_ints,
                            scratch_rows, stream);
}

// ---------------------------------------------------------------- a router's choice
// From float32 router logits z [n_tokens, >= E]: scores s = sigmoid(z); choice[n, 0 .. top-1] the experts with the
// largest scores (the largest first; of equal scores the lower index), weight[n, k] their scores, divided by their sum
// if ``renorm``. ``extra`` >= 0: also gate[n] = sigmoid(z[n, extra]) (a column beside the experts': the gate of a
// shared expert). A wave a token; top times a pass over the E scores.
__global__ __launch_bounds__(256) void moe_route_kernel(const float* __restrict__ z, long z_stride, int n_tokens, int E,
                                                        int top, int renorm, int extra, int* __restrict__ choice,
                                                        float* __restrict__ weight, float* __restrict__ gate) {
  const int n = blockIdx.x * (256 / LMSF_WAVE) + threadIdx.x / LMSF_WAVE, lane = threadIdx.x % LMSF_WAVE;
  if (n >= n_tokens) return;
  const float* row = z + (long)n * z_stride;
  float last = INFINITY, total = 0.f, mine = 0.f;
  int last_e = -1, mine_e = 0;
  for (int k = 0; k < top; ++k) {
    // the largest (score, -index) below the one taken before
    float best = -INFINITY;
    int best_e = E;
    for (int e = lane; e < E; e += LMSF_WAVE) {
      const float sc = row[e];
      const bool below = sc < last || (sc == last && e > last_e);
      if (below && (sc > best || (sc == best && e < best_e))) {
        best = sc;
        best_e = e;
      }
    }
#pragma unroll
    for (int o = LMSF_WAVE / 2; o > 0; o >>= 1) {
      const float ob = __shfl_xor(best, o, LMSF_WAVE);
      const int oe = __shfl_xor(best_e, o, LMSF_WAVE);
      if (ob > best || (ob == best && oe < best_e)) {
        best = ob;
        best_e = oe;
      }
    }
    last = best;
    last_e = best_e;
    const float sg = 1.f / (1.f + expf(-best));
    total += sg;
    if (lane == k) {      // lane k keeps the k-th choice
      mine = sg;
      mine_e = min(best_e, E - 1);
    }
  }
  if (lane < top) {
    choice[(long)n * top + lane] = mine_e;
    weight[(long)n * top + lane] = renorm ? mine / total : mine;
  }
  if (extra >= 0 && lane == 0) gate[n] = 1.f / (1.f + expf(-row[extra]));
}

extern "C" int lmsf_moe_route(const float* z, long z_stride, int n_tokens, int E, int top, int renorm, int extra,
                              int* choice, float* weight, float* gate, hipStream_t stream) {
  LMSF_CHECK(z && choice && weight && (extra < 0 || gate), "moe_route: null pointer");
  LMSF_CHECK(E > 0 && top > 0 && top <= E && top <= LMSF_WAVE && z_stride >= E && extra < z_stride, "moe_route: bad sizes");
  if (n_tokens <= 0) return 0;
  hipLaunchKernelGGL(moe_route_kernel, dim3((n_tokens + 3) / 4), dim3(256), 0, stream, z, z_stride, n_tokens, E, top,
                     renorm, extra, choice, weight, gate);
  LMSF_LAUNCH_CHECK("moe_route");
  return 0;
}

// The same with the scores a softmax over all experts (``softmax`` 1; 0: sigmoid) and a limit on where the choice may
// fall: the experts form ``groups`` equal groups of neighbours, a group's score is its best expert's, and only experts
// of the ``keep`` best groups can be chosen (groups = keep = 1: no limit). weight[n, k]: the chosen experts' scores
// (over their sum with ``renorm``). A wave a token; a lane keeps the best score and the "kept" flag of the groups
// lane, lane + 64, ... (at most 256 groups).
__global__ __launch_bounds__(256) void moe_route_groups_kernel(const float* __restrict__ z, long z_stride, int n_tokens,
                                                               int E, int top, int softmax, int groups, int keep,
                                                               int renorm, const float* __restrict__ correction,
                                                               float scale, int extra, int* __restrict__ choice,
                                                               float* __restrict__ weight, float* __restrict__ gate) {
  const int n = blockIdx.x * (256 / LMSF_WAVE) + threadIdx.x / LMSF_WAVE, lane = threadIdx.x % LMSF_WAVE;
  if (n >= n_tokens) return;
  const float* row = z + (long)n * z_stride;
  float mx = -INFINITY, sum = 0.f;
  if (softmax) {
    for (int e = lane; e < E; e += LMSF_WAVE) mx = fmaxf(mx, row[e]);
    mx = wave_max(mx);
    for (int e = lane; e < E; e += LMSF_WAVE) sum += expf(row[e] - mx);
    sum = wave_sum(sum);
  }
  // what a choice compares: the logit, which orders as its score does, or the score plus the expert's correction
  auto score = [&](float x) { return softmax ? expf(x - mx) / sum : 1.f / (1.f + expf(-x)); };
  auto key = [&](int e) { return correction ? score(row[e]) + correction[e] : row[e]; };
  const int per = E / groups;
  float gbest[4];
  unsigned kept = 0;           // bit i: group lane + 64 i is kept
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int g = lane + LMSF_WAVE * i;
    gbest[i] = -INFINITY;
    if (g < groups && keep < groups)
      for (int e = g * per; e < (g + 1) * per; ++e) gbest[i] = fmaxf(gbest[i], key(e));
  }
  if (keep >= groups) kept = 0xFu;
  else
    for (int k = 0; k < keep; ++k) {
      float best = -INFINITY;
      int best_g = groups;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int g = lane + LMSF_WAVE * i;
        if (g < groups && !((kept >> i) & 1u) && (gbest[i] > best || (gbest[i] == best && g < best_g))) {
          best = gbest[i];
          best_g = g;
        }
      }
#pragma unroll
      for (int o = LMSF_WAVE / 2; o > 0; o >>= 1) {
        const float ob = __shfl_xor(best, o, LMSF_WAVE);
        const int og = __shfl_xor(best_g, o, LMSF_WAVE);
        if (ob > best || (ob == best && og < best_g)) {
          best = ob;
          best_g = og;
        }
      }
      if (best_g < groups && (best_g % LMSF_WAVE) == lane) kept |= 1u << (best_g / LMSF_WAVE);
    }
  float last = INFINITY, total = 0.f, mine = 0.f;
  int last_e = -1, mine_e = 0;
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int best_e = E;
    for (int e0 = 0; e0 < E; e0 += LMSF_WAVE) {      // (every lane takes part in the shuffle)
      const int e = e0 + lane;
      const int g = min(e, E - 1) / per;
      const unsigned flags = __shfl(kept, g % LMSF_WAVE, LMSF_WAVE);
      if (e >= E || !((flags >> (g / LMSF_WAVE)) & 1u)) continue;
      const float sc = key(e);
      const bool below = sc < last || (sc == last && e > last_e);
      if (below && (sc > best || (sc == best && e < best_e))) {
        best = sc;
        best_e = e;
      }
    }
#pragma unroll
    for (int o = LMSF_WAVE / 2; o > 0; o >>= 1) {
      const float ob = __shfl_xor(best, o, LMSF_WAVE);
      const int oe = __shfl_xor(best_e, o, LMSF_WAVE);
      if (ob > best || (ob == best && oe < best_e)) {
        best = ob;
        best_e = oe;
      }
    }
    last = best;
    last_e = best_e;
    const float sc = score(row[min(best_e, E - 1)]);
    total += sc;
    if (lane == k) {
      mine = sc;
      mine_e = min(best_e, E - 1);
    }
  }
  if (lane < top) {
    choice[(long)n * top + lane] = mine_e;
    weight[(long)n * top + lane] = scale * (renorm ? mine / (total + 1e-20f) : mine);
  }
  if (extra >= 0 && lane == 0) gate[n] = 1.f / (1.f + expf(-row[extra]));
}

// ``correction`` float32 [E] or null: added to the scores for the choice alone, not for the weights. ``scale`` multiplies
// the weights. ``extra``, ``gate``: as for lmsf_moe_route.
extern "C" int lmsf_moe_route_groups(const float* z, long z_stride, int n_tokens, int E, int top, int softmax,
                                     int groups, int keep, int renorm, const float* correction, float scale, int extra,
                                     int* choice, float* weight, float* gate, hipStream_t stream) {
  LMSF_CHECK(z && choice && weight && (extra < 0 || gate), "moe_route_groups: null pointer");
  LMSF_CHECK(E > 0 && top > 0 && top <= E && top <= LMSF_WAVE && z_stride >= E && extra < z_stride,
             "moe_route_groups: bad sizes");
  LMSF_CHECK(groups > 0 && groups <= 256 && E % groups == 0 && keep > 0 && keep <= groups &&
                 (long)keep * (E / groups) >= top,
             "moe_route_groups: %d of %d groups of %d experts cannot hold %d choices", keep, groups, E, top);
  if (n_tokens <= 0) return 0;
  hipLaunchKernelGGL(moe_route_groups_kernel, dim3((n_tokens + 3) / 4), dim3(256), 0, stream, z, z_stride, n_tokens, E,
                     top, softmax, groups, keep, renorm, correction, scale, extra, choice, weight, gate);
  LMSF_LAUNCH_CHECK("moe_route_groups");
  return 0;
}
