// Paged attention, general form: any number of query tokens per request, any head size that is a
// multiple of 4 up to 1024, any page size, float32 or bfloat16 storage, float32 arithmetic.
//
// Query token t belongs to request segment seg[t] and stands at position pos[t]. It attends to
// the keys at positions j in [first_visible_key(pos, window), pos] of that request (a window of the last
// positions, the query's own chunk of positions, or everything), read from the pages
// (key j lives in page block_table[seg][j / page_size] at offset j % page_size; K pages are
// [page, kv_head, offset, d], V pages [page, kv_head, d, offset]). All keys of a step
// are written to the pages before this kernel runs, so prompts, portions of prompts and single
// decoded tokens are one case.
//
// Function computed, per query head h with kv head g = h / (nh / nkv)
// (core/src/model_executor/layers/attention.rs:91-103, :139-155 for prompts;
// vllm/kernels/attention/attention_kernels.cu:82-414 for decoding):
//   s_j = scale * <q, k_j>;  p = softmax_j(s);  out = sum_j p_j v_j
// with an exact softmax (the reference's decode kernel divides by sum + 1e-6, :279).
//
// Two kernels. Heads of up to 256 in pages of a multiple of 4 keys, both on boundaries of four elements, run with a tile of
// keys a wave (paged_attention_waves_kernel). Anything else: one workgroup of 256 threads per (token, head), keys taken
// 256 at a time, one key per thread for the scores, an online softmax across chunks, and the P V product with the threads
// arranged as (key group, output dim); a head wider than 256 has one key group and up to four output dims a thread.
#include "common.h"

#include <math.h>

#define GEN_THREADS 256

// four neighbouring elements in one load
__device__ __forceinline__ void gen_load4(const float* p, float* x) {
  const float4 v = *reinterpret_cast<const float4*>(p);
  x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
}
__device__ __forceinline__ void gen_load4(const bf16_t* p, float* x) {
  const uint2 v = *reinterpret_cast<const uint2*>(p);
  x[0] = __uint_as_float(v.x << 16); x[1] = __uint_as_float(v.x & 0xffff0000u);
  x[2] = __uint_as_float(v.y << 16); x[3] = __uint_as_float(v.y & 0xffff0000u);
}

// Keys in tiles, a wave a tile. What bounds these calls is the number of trips to memory in a row, not the bytes: a tiny
// model's tokens have 40 kB of keys and values each, and every trip costs 0.5 to 1 us. So a wave asks for a tile's keys
// AND values at once (8 loads of four elements of each a lane, 8 kB of each in float32), before it knows any score:
// position -> block table -> keys and values are three trips up to 8 tiles of keys, where the form below makes one for
// every four keys a thread. Both forms, that one -> this one, 8 heads on one kv head in float32, 32 / 128 / 256 wide: 8
// tokens of 300 keys 11.0 / 27 / 48 -> 5.7 / 8.0 / 11.7 us, 1 token of 16 keys 4.6 / 6.7 / 8.3 -> 4.3 / 5.7 / 5.4, of 8,000
// keys 187 / 620 / 1,179 -> 40 / 115 / 212, a prompt of 140 tokens 11.2 / 34 / 65 -> 10.6 / 18.6 / 24, 256 tokens behind
// 768 others 151 / 536 / 1,072 -> 43 / 104 / 188, a prompt of 2,048 tokens (128 / 256 wide) 4,610 / 9,164 -> 813 / 1,557,
// heads of 160 and 192 in between; in bfloat16 alike (2,048 tokens 4,176 / 8,318 -> 581 / 1,082). LPK lanes share a key (d
// up to 32 LPK; a tile is 64 / LPK keys), every wave keeps an online softmax of its own over its tiles (w, w + 8, ...) with
// no barrier, and the waves' results are added up in their order at the end, so a token's bits hang on its own position and
// window alone.
// Values: lane = (dim, quad of keys in the page), so that consecutive lanes read consecutive 16 bytes of a page.
#define TILE_WAVES 8
// what a wave's lanes left in LDS is there for its other lanes (LDS serves a wave's accesses in order)
__device__ __forceinline__ void gen_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
template <typename T, int LPK>
__global__ __launch_bounds__(TILE_WAVES * 64) void paged_attention_waves_kernel(
    const T* __restrict__ q, long q_stride, T* __restrict__ out, long out_stride, const T* __restrict__ k_pages,
    const T* __restrict__ v_pages, const int* __restrict__ block_tables, int bt_width, const int* __restrict__ seg,
    const int* __restrict__ pos, int nh, int nkv, int d, int ps, int ps_shift, float scale, int window, float softcap,
    const float* __restrict__ bias, const float* __restrict__ sink) {
  constexpr int DMAX = 32 * LPK, KEYS = 64 / LPK, QUADS = KEYS / 4;
  constexpr int G = QUADS < 4 ? QUADS : 4;          // lanes side by side on the quads of a dim
  constexpr int DSTEP = 64 / G, DPL = DMAX / DSTEP; // dims a load covers, dims a lane owns: lane / G + DSTEP e
  constexpr int QPL = QUADS / G;                    // quads a lane takes: lane % G + G i
  static_assert(DPL * QPL == 8, "eight loads of values a lane");
  __shared__ __align__(16) float sq[TILE_WAVES][DMAX];   // the query, scaled (a copy a wave: no barrier), then the waves' outputs
  __shared__ __align__(16) float sp[TILE_WAVES][KEYS];   // a tile's probabilities
  __shared__ float sm[TILE_WAVES], sl[TILE_WAVES];

  const int t = blockIdx.x, h = blockIdx.y;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int s = seg[t], p = pos[t];
  const int lo = first_visible_key(p, window);
  const int g = h / (nh / nkv);
  const int* bt = block_tables + (long)s * bt_width;
  const float r1 = bias ? bias[h] : 0.f, r2 = bias ? bias[nh + h] : 0.f;
  const auto page_of = [&](int j) { return ps_shift >= 0 ? j >> ps_shift : j / ps; };

  for (int i = lane; i < DMAX; i += 64) sq[w][i] = i < d ? to_f32<T>(q[(long)t * q_stride + h * d + i]) * scale : 0.f;
  gen_wave_sync();

  float m = -INFINITY, l = 0.f, acc[DPL];
#pragma unroll
  for (int e = 0; e < DPL; ++e) acc[e] = 0.f;

  const int part = lane % LPK;
  // (tiles begin at a multiple of 4, in the page of the first visible key: a quad never crosses a page)
  for (int j0 = (lo & ~3) + w * KEYS; j0 <= p; j0 += TILE_WAVES * KEYS) {
    const int j = j0 + lane / LPK, jc = min(j, p);   // keys beyond the token's own are read as its own and masked
    const int block = page_of(jc), off = jc - block * ps;
    int vblock[QPL], voff[QPL];
#pragma unroll
    for (int i = 0; i < QPL; ++i) {
      const int jq = min(j0 + 4 * (lane % G + G * i), p & ~3);
      vblock[i] = page_of(jq);
      voff[i] = jq - vblock[i] * ps;
    }
    const T* kr = k_pages + (((long)bt[block] * nkv + g) * ps + off) * d;
    const T* vr[QPL];
#pragma unroll
    for (int i = 0; i < QPL; ++i) vr[i] = v_pages + ((long)bt[vblock[i]] * nkv + g) * d * ps + voff[i];
    float k4[8][4], v4[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int o = (i * LPK + part) * 4;
      gen_load4(kr + (o < d ? o : 0), k4[i]);
    }
#pragma unroll
    for (int i = 0; i < QPL; ++i)
#pragma unroll
      for (int e = 0; e < DPL; ++e) gen_load4(vr[i] + (long)min(lane / G + DSTEP * e, d - 1) * ps, v4[i * DPL + e]);

    float dot = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int o = (i * LPK + part) * 4;
      const float4 q4 = *reinterpret_cast<const float4*>(&sq[w][o]);
      const float x = q4.x * k4[i][0] + q4.y * k4[i][1] + q4.z * k4[i][2] + q4.w * k4[i][3];
      dot += o < d ? x : 0.f;
    }
#pragma unroll
    for (int o = 1; o < LPK; o <<= 1) dot += __shfl_xor(dot, o, 64);
    float sc = softcap > 0.f ? softcap * tanhf(dot / softcap) : dot;   // scores bounded by cap tanh(s / cap)
    if (bias) sc -= r1 * log1pf(r2 * (float)(p - j));                  // what the distance takes off
    const bool visible = j >= lo && j <= p;
    if (!visible) sc = -INFINITY;
    float tile_max = sc;
#pragma unroll
    for (int o = LPK; o < 64; o <<= 1) tile_max = fmaxf(tile_max, __shfl_xor(tile_max, o, 64));
    const float m_new = fmaxf(m, tile_max);
    // (a score of -inf, or an unseen key's, adds nothing, also where nothing stands beside it; one that is no number stays one)
    const float pr = sc == -INFINITY ? 0.f : expf(sc - m_new);
    const float corr = m == -INFINITY ? 0.f : expf(m - m_new);
    float tile_sum = pr;
#pragma unroll
    for (int o = LPK; o < 64; o <<= 1) tile_sum += __shfl_xor(tile_sum, o, 64);
    l = l * corr + tile_sum;
    m = m_new;
    gen_wave_sync();
    if (part == 0) sp[w][lane / LPK] = pr;
    gen_wave_sync();
#pragma unroll
    for (int e = 0; e < DPL; ++e) acc[e] *= corr;
#pragma unroll
    for (int i = 0; i < QPL; ++i) {
      const int quad = lane % G + G * i;
      const float4 p4 = *reinterpret_cast<const float4*>(&sp[w][4 * quad]);
      const float pq[4] = {p4.x, p4.y, p4.z, p4.w};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int ju = j0 + 4 * quad + u;
        const bool in = ju >= lo && ju <= p;       // what lies in a page outside these was never written
#pragma unroll
        for (int e = 0; e < DPL; ++e) acc[e] += pq[u] * (in ? v4[i * DPL + e][u] : 0.f);
      }
    }
  }
#pragma unroll
  for (int e = 0; e < DPL; ++e)
#pragma unroll
    for (int o = 1; o < G; o <<= 1) acc[e] += __shfl_xor(acc[e], o, 64);
  gen_wave_sync();
  if (lane % G == 0) {
#pragma unroll
    for (int e = 0; e < DPL; ++e) sq[w][lane / G + DSTEP * e] = acc[e];
  }
  if (lane == 0) {
    sm[w] = m;
    sl[w] = l;
  }
  __syncthreads();
  if (tid < d) {
    // (a sink: exp(sink_h) stands in the denominator beside the keys' exponentials)
    float top = sink ? sink[h] : -INFINITY;
#pragma unroll
    for (int i = 0; i < TILE_WAVES; ++i) top = fmaxf(top, sm[i]);
    float den = sink ? expf(sink[h] - top) : 0.f, o = 0.f;
#pragma unroll
    for (int i = 0; i < TILE_WAVES; ++i) {
      const float f = sm[i] == -INFINITY ? 0.f : expf(sm[i] - top);
      den += f * sl[i];
      o += f * sq[i][tid];
    }
    out[(long)t * out_stride + h * d + tid] = from_f32<T>(o / den);
  }
}

// VEC: the key pages start on a boundary of four elements (every row does then: d is a multiple of 4), and a key is read
// four elements a load. WAVES: waves a SIMD that registers are kept for: 1 (about 110 registers, so that as many loads as
// possible are on their way together; four workgroups run on a compute unit) or 5 (72 registers, seven workgroups).
template <typename T, bool VEC, int WAVES>
__global__ __launch_bounds__(GEN_THREADS, WAVES) void paged_attention_generic_kernel(
    const T* __restrict__ q, long q_stride, T* __restrict__ out, long out_stride, const T* __restrict__ k_pages,
    const T* __restrict__ v_pages, const int* __restrict__ block_tables, int bt_width, const int* __restrict__ seg,
    const int* __restrict__ pos, int nh, int nkv, int d, int ps, float scale, int window, float softcap,
    const float* __restrict__ bias, const float* __restrict__ sink) {
  extern __shared__ float smem[];
  float* sq = smem;                       // [d] query, pre-scaled
  float* sp = sq + d;                     // [256] scores, then probabilities
  int* shead = (int*)(sp + GEN_THREADS);  // [256] page * nkv + g of each key
  int* soff = shead + GEN_THREADS;        // [256] its offset in the page
  float* sacc = (float*)(soff + GEN_THREADS);  // [256] partial outputs of the key groups
  __shared__ float red[16];

  const int t = blockIdx.x, h = blockIdx.y;
  const int tid = threadIdx.x;
  const int s = seg[t], p = pos[t];
  const int lo = first_visible_key(p, window);
  const int g = h / (nh / nkv);
  const int* bt = block_tables + (long)s * bt_width;

  const float r1 = bias ? bias[h] : 0.f, r2 = bias ? bias[nh + h] : 0.f;

  for (int i = tid; i < d; i += GEN_THREADS) sq[i] = to_f32<T>(q[(long)t * q_stride + h * d + i]) * scale;

  const int ngroups = GEN_THREADS / d > 0 ? GEN_THREADS / d : 1;
  const int og = tid / d, oi = tid % d;                            // (key group, output dim) of this thread
  const bool pv_active = og < ngroups;
  // (a sink: exp(sink_h) stands in the denominator beside the keys' exponentials, so the online softmax begins with it)
  float acc = 0.f, m = sink ? sink[h] : -INFINITY, l = sink ? 1.f : 0.f;
  float wide[3] = {0.f, 0.f, 0.f};                                 // output dims tid + 256, + 512, + 768 (d > 256)
  __syncthreads();

  for (int j0 = lo; j0 <= p; j0 += GEN_THREADS) {
    const int j = j0 + tid;
    float sc = -INFINITY;
    if (j <= p) {
      const int block = j / ps, off = j - block * ps;
      const int head_base = bt[block] * nkv + g;
      shead[tid] = head_base;
      soff[tid] = off;
      const T* kr = k_pages + ((long)head_base * ps + off) * d;
      float dot = 0.f;
#pragma unroll 8
      for (int i = 0; i < d; i += 4) {
        float k4[4];
        if (VEC) {
          gen_load4(kr + i, k4);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) k4[e] = to_f32<T>(kr[i + e]);
        }
        dot += sq[i] * k4[0] + sq[i + 1] * k4[1] + sq[i + 2] * k4[2] + sq[i + 3] * k4[3];
      }
      sc = softcap > 0.f ? softcap * tanhf(dot / softcap) : dot;   // scores bounded by cap tanh(s / cap)
      if (bias) sc -= r1 * log1pf(r2 * (float)(p - j));            // what the distance takes off
    }
    const float cmax = block_max(sc, red);
    const float m_new = fmaxf(m, cmax);
    const float e = (j <= p) ? expf(sc - m_new) : 0.f;
    sp[tid] = e;
    const float csum = block_sum(e, red);  // has barriers: sp, shead and soff are visible afterwards
    const float corr = (m == -INFINITY) ? 0.f : expf(m - m_new);
    l = l * corr + csum;
    acc *= corr;
    if (d > GEN_THREADS) {
      wide[0] *= corr; wide[1] *= corr; wide[2] *= corr;
    }
    m = m_new;
    __syncthreads();
    if (pv_active) {
      const int n = min(GEN_THREADS, p - j0 + 1);
      int jj = og;
      // (up to 256 output dims: four values of a group's keys are asked for at a time; one by one every value waits for
      // the one before it)
      if (d <= GEN_THREADS)
        for (; jj + 3 * ngroups < n; jj += 4 * ngroups) {
          float v[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int key = jj + u * ngroups;
            v[u] = to_f32<T>(v_pages[((long)shead[key] * d + oi) * ps + soff[key]]);
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) acc += sp[jj + u * ngroups] * v[u];
        }
      for (; jj < n; jj += ngroups) {
        const int head_base = shead[jj], off = soff[jj];
        acc += sp[jj] * to_f32<T>(v_pages[((long)head_base * d + oi) * ps + off]);
        if (d > GEN_THREADS) {
#pragma unroll
          for (int r = 0; r < 3; ++r) {
            const int o2 = tid + (r + 1) * GEN_THREADS;
            if (o2 < d) wide[r] += sp[jj] * to_f32<T>(v_pages[((long)head_base * d + o2) * ps + off]);
          }
        }
      }
    }
    __syncthreads();
  }
  sacc[tid] = pv_active ? acc : 0.f;
  __syncthreads();
  if (tid < d) {
    float o = 0.f;
    for (int gg = 0; gg < ngroups; ++gg) o += sacc[gg * d + tid];
    out[(long)t * out_stride + h * d + tid] = from_f32<T>(o / l);
  }
  if (d > GEN_THREADS) {
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const int o2 = tid + (r + 1) * GEN_THREADS;
      if (o2 < d) out[(long)t * out_stride + h * d + o2] = from_f32<T>(wide[r] / l);
    }
  }
}

// ``softcap`` c > 0: a score s (after the scale) becomes c tanh(s / c) before the softmax; 0: scores as they are.
// ``bias`` float32 [2, nh] or null: r1_h ln(1 + r2_h (i - j)) comes off the score of query i and key j (r2 >= 0),
// after the cap. ``sink`` float32 [nh] or null: exp(sink_h) stands in head h's denominator.
extern "C" int lmsf_paged_attention_generic_biased(const void* q, long q_stride, void* out, long out_stride,
                                                   const void* k_pages, const void* v_pages, long num_pages,
                                                   const int* block_tables, int bt_width, const int* seg,
                                                   const int* pos, int n_tokens, int nh, int nkv, int d, int ps,
                                                   float scale, int window, float softcap, const float* bias, const float* sink,
                                                   int dtype, hipStream_t stream) {
  LMSF_CHECK(softcap >= 0.f, "paged_attention: the soft cap must be >= 0, got %g", (double)softcap);
  LMSF_CHECK(q && out && k_pages && v_pages && block_tables && seg && pos, "paged_attention: null pointer");
  LMSF_CHECK(dtype == LMSF_F32 || dtype == LMSF_BF16, "paged_attention: unknown dtype code %d", dtype);
  LMSF_CHECK(nh > 0 && nkv > 0 && nh % nkv == 0, "paged_attention: heads %d not a multiple of kv heads %d", nh, nkv);
  LMSF_CHECK(d > 0 && d % 4 == 0 && d <= 1024, "paged_attention: head size %d not supported (multiple of 4, <= 1024)", d);
  LMSF_CHECK(ps > 0 && bt_width > 0 && num_pages > 0, "paged_attention: bad page geometry");
  LMSF_CHECK(num_pages * nkv * ps < 2147483647L, "paged_attention: cache too large for 32-bit row indices");
  LMSF_CHECK(q_stride >= (long)nh * d && out_stride >= (long)nh * d, "paged_attention: row strides too small");
  LMSF_CHECK(nh <= 65535, "paged_attention: too many heads");
  if (n_tokens == 0) return 0;
  const size_t smem = (size_t)(d + 4 * GEN_THREADS) * 4;
  dim3 grid(n_tokens, nh), block(GEN_THREADS);
#define GENERIC_W(T_, VEC_, WAVES_)                                                                                     \
  hipLaunchKernelGGL((paged_attention_generic_kernel<T_, VEC_, WAVES_>), grid, block, smem, stream, (const T_*)q,       \
                     q_stride, (T_*)out, out_stride, (const T_*)k_pages, (const T_*)v_pages, block_tables, bt_width,    \
                     seg, pos, nh, nkv, d, ps, scale, window, softcap, bias, sink)
#define GENERIC(T_, VEC_)                                                                                               \
  do {                                                                                                                  \
    if (many) GENERIC_W(T_, VEC_, 5); else GENERIC_W(T_, VEC_, 1);                                                      \
  } while (0)
  const size_t quad = 4 * lmsf_elem_size(dtype);
  if (d <= 256 && ps % 4 == 0 && (size_t)k_pages % quad == 0 && (size_t)v_pages % quad == 0) {
    const int shift = (ps & (ps - 1)) == 0 ? __builtin_ctz((unsigned)ps) : -1;
#define TILES_OF(T_, LPK_)                                                                                              \
  hipLaunchKernelGGL((paged_attention_waves_kernel<T_, LPK_>), grid, dim3(TILE_WAVES * 64), 0, stream, (const T_*)q, q_stride, \
                     (T_*)out, out_stride, (const T_*)k_pages, (const T_*)v_pages, block_tables, bt_width, seg, pos, nh, \
                     nkv, d, ps, shift, scale, window, softcap, bias, sink)
#define TILES(T_)                                                                                                       \
  do {                                                                                                                  \
    if (d <= 32) TILES_OF(T_, 1); else if (d <= 64) TILES_OF(T_, 2); else if (d <= 128) TILES_OF(T_, 4); else TILES_OF(T_, 8); \
  } while (0)
    if (dtype == LMSF_F32) TILES(float); else TILES(bf16_t);
#undef TILES
#undef TILES_OF
    LMSF_LAUNCH_CHECK("paged_attention_generic");
    return 0;
  }
  const bool vec = (size_t)k_pages % (4 * lmsf_elem_size(dtype)) == 0;
  // What is left: wider heads, pages of other sizes, unaligned ones. More workgroups than the chip takes at once with four
  // on a compute unit: fewer registers, seven on a unit. Both sides in float32, 8 heads on one kv head, of 32 / 256 in
  // pages of 18 and of 512 in pages of 16, four -> seven a unit: 64 tokens of a prompt 6.4 / 15.9 / 40 -> 6.9 / 18.5 / 45
  // us, 100 tokens 8.0 / 27 / 77 -> 8.0 / 28 / 78, 140 tokens (beyond the line) 11.3 / 44 / 131 -> 9.4 / 42 / 126, 200
  // tokens 14.8 / 73 / 238 -> 14.1 / 74 / 226, 512 tokens 56 / 376 / 1,344 -> 53 / 429 / 1,406: ahead while seven a unit
  // hold all that four do not, and with narrow heads; wide heads of many tokens lose 5 to 14 %.
  const bool many = (long)n_tokens * nh > 4L * lmsf_compute_units();
  if (dtype == LMSF_F32) {
    if (vec) GENERIC(float, true); else GENERIC(float, false);
  } else {
    if (vec) GENERIC(bf16_t, true); else GENERIC(bf16_t, false);
  }
#undef GENERIC
#undef GENERIC_W
  LMSF_LAUNCH_CHECK("paged_attention_generic");
  return 0;
}

extern "C" int lmsf_paged_attention_generic(const void* q, long q_stride, void* out, long out_stride,
                                            const void* k_pages, const void* v_pages, long num_pages,
                                            const int* block_tables, int bt_width, const int* seg, const int* pos,
                                            int n_tokens, int nh, int nkv, int d, int ps, float scale, int window,
                                            int dtype, hipStream_t stream) {
  return lmsf_paged_attention_generic_biased(q, q_stride, out, out_stride, k_pages, v_pages, num_pages, block_tables,
                                             bt_width, seg, pos, n_tokens, nh, nkv, d, ps, scale, window, 0.f, nullptr,
                                             nullptr, dtype, stream);
}
