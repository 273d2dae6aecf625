// Linear layer C[M, N] = A[M, K] W[N, K]^T (+ bias[N]) with float32 multiply-adds.
//
// This is the true 32-bit matrix product of the float32 path (no matrix-core instruction, no
// reduced-precision input mode), and the fallback of the bfloat16 path for shapes the fast kernels
// refuse. Inputs may be float32 or bfloat16; products and sums are float32. The reference calls cuBLASLt with
// float32 compute (tops/csrc/tops/tensorrt_llm/common/cublasMMWrapper.cpp:182-210) and adds the bias afterwards
// (core/src/model_executor/layers/linear.rs:101-104).
//
// Two forms: K split over the waves of a workgroup (further down), or a 64x64 tile per workgroup of 256 threads, 4x4
// outputs per thread, K in slabs of 16 staged through LDS. Both add up an output in one order, so that which of them runs,
// and with it the number of rows multiplied together, changes no bit: the ceil(K / 32) steps of 32 k are cut into eight
// consecutive parts (gp_part), the even and the odd k of a part are two chains of fused multiply-adds, and the parts' sums
// (even + odd) are added in turn. Any M, N, K; rows may be strided (lda, ldw, ldc in elements).
#include "common.h"

#define GP_TILE 64
#define GP_BK 16
#define GP_STEP 32      // k of a step
#define GP_PARTS 8

// the first k of part p (of part GP_PARTS: K)
__device__ __forceinline__ int gp_part(int p, int K) {
  const unsigned steps = ((unsigned)K + GP_STEP - 1) / GP_STEP;      // (below 2^26)
  return (int)min(p * steps / GP_PARTS * GP_STEP, (unsigned)K);
}

// The tiles. Up to K the four entries that a thread reads of a row carry no test; with one for every entry, rows outside the
// matrix included, the tests took half of the time (2,048 x 2,048 x 512 in float32 123 us, now 68).
template <typename TA, typename TW, typename TO>
__global__ __launch_bounds__(256) void gemm_plain_kernel(const TA* __restrict__ A, long lda, const TW* __restrict__ W,
                                                         long ldw, const TW* __restrict__ bias, TO* __restrict__ C,
                                                         long ldc, int M, int N, int K) {
  __shared__ __align__(16) float As[GP_BK][GP_TILE + 4];
  __shared__ __align__(16) float Ws[GP_BK][GP_TILE + 4];
  const int tid = threadIdx.x;
  const int tx = tid % 16, ty = tid / 16;
  const int m0 = blockIdx.y * GP_TILE, n0 = blockIdx.x * GP_TILE;
  const int lrow = tid / 4, lk = (tid % 4) * 4;
  const TA* arow = A + (long)min(m0 + lrow, M - 1) * lda + lk;    // rows beyond the matrix repeat the last: not written
  const TW* wrow = W + (long)min(n0 + lrow, N - 1) * ldw + lk;
  float sum[4][4], acc[4][4][2];      // the parts so far; the even and the odd k of the present one
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) sum[i][j] = acc[i][j][0] = acc[i][j][1] = 0.f;

  for (int p = 0, k0 = 0; p < GP_PARTS; ++p) {
    const int end = gp_part(p + 1, K);
    if (k0 >= end) continue;      // a part without a step
    for (; k0 < end; k0 += GP_BK) {
      float av[4], wv[4];
      if (k0 + GP_BK <= K) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          av[e] = to_f32<TA>(arow[k0 + e]);
          wv[e] = to_f32<TW>(wrow[k0 + e]);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // (all loads are made, beyond K of the last entry: behind a test each they would be waited for one by one)
          const int at = min(k0 + e, K - 1 - lk);
          const float a1 = to_f32<TA>(arow[at]), w1 = to_f32<TW>(wrow[at]);
          av[e] = k0 + lk + e < K ? a1 : 0.f;
          wv[e] = k0 + lk + e < K ? w1 : 0.f;
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        As[lk + e][lrow] = av[e];
        Ws[lk + e][lrow] = wv[e];
      }
      __syncthreads();
      float a[2][4], w[2][4];      // the next k's operands are read while the present one's are multiplied
      auto read = [&](int kk) {
        *reinterpret_cast<float4*>(a[kk & 1]) = *reinterpret_cast<const float4*>(&As[kk][ty * 4]);
        *reinterpret_cast<float4*>(w[kk & 1]) = *reinterpret_cast<const float4*>(&Ws[kk][tx * 4]);
      };
      read(0);
#pragma unroll
      for (int kk = 0; kk < GP_BK; ++kk) {
        if (kk + 1 < GP_BK) read(kk + 1);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[i][j][kk & 1] = fmaf(a[kk & 1][i], w[kk & 1][j], acc[i][j][kk & 1]);
      }
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        sum[i][j] += acc[i][j][0] + acc[i][j][1];
        acc[i][j][0] = acc[i][j][1] = 0.f;
      }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int gm = m0 + ty * 4 + i;
    if (gm >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int gn = n0 + tx * 4 + j;
      if (gn >= N) continue;
      float r = sum[i][j];
      if (bias) r += to_f32<TW>(bias[gn]);
      C[(long)gm * ldc + gn] = from_f32<TO>(r);
    }
  }
}

// The same product for up to 16 rows of bfloat16 operands that the weight-streaming kernels refuse (a K that is no
// multiple of 8, rows that do not start on 16-byte boundaries): with so few rows the tiles above leave most of the
// chip idle (N / 64 workgroups, each walking all of K: 4,160 x 11,100 at 8 rows 1,290 us). Here a wave owns one output
// column; lane l takes k = l, l + 64, ... with 2-byte loads, which need no alignment, and the lanes' sums are added
// up in a fixed order. float32 products and sums.
#define GP_FEW_ROWS 16
// MT: rows the kernel walks (M rounded up to 1, 2, 4, 8 or 16; the rows beyond M repeat row M - 1 and are not written),
// so that the loop has no tests and the loads of several steps are in flight together. VEC: elements a load (2 where K
// and the row strides are even and the operands start on 4-byte boundaries, else 1). COLS: output columns a wave owns,
// more with more rows: every column's wave reads all of x from the caches, and with 16 rows and one column a wave that
// is 16 loads of x for each of W (4,160 x 11,100 at 16 rows: 1.5 GB through the caches).
template <typename TO, int MT, int VEC, int COLS>
__global__ __launch_bounds__(256) void gemm_plain_few_kernel(const bf16_t* __restrict__ A, long lda,
                                                             const bf16_t* __restrict__ W, long ldw,
                                                             const bf16_t* __restrict__ bias, TO* __restrict__ C,
                                                             long ldc, int M, int N, int K) {
  const int lane = threadIdx.x & 63;
  const int n0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * COLS;
  if (n0 >= N) return;
  float acc[MT][COLS];
  const bf16_t* a[MT];
  const bf16_t* w[COLS];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    a[m] = A + (long)min(m, M - 1) * lda;
#pragma unroll
    for (int c = 0; c < COLS; ++c) acc[m][c] = 0.f;
  }
#pragma unroll
  for (int c = 0; c < COLS; ++c) w[c] = W + (long)min(n0 + c, N - 1) * ldw;   // columns beyond N repeat the last one
  if (VEC == 2) {
#pragma unroll 2
    for (int k = 2 * lane; k < K; k += 128) {   // K is even: a pair never straddles the end
      float w0[COLS], w1[COLS];
#pragma unroll
      for (int c = 0; c < COLS; ++c) {
        const unsigned wp = *reinterpret_cast<const unsigned*>(w[c] + k);
        w0[c] = __uint_as_float(wp << 16);
        w1[c] = __uint_as_float(wp & 0xffff0000u);
      }
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const unsigned xp = *reinterpret_cast<const unsigned*>(a[m] + k);
        const float x0 = __uint_as_float(xp << 16), x1 = __uint_as_float(xp & 0xffff0000u);
#pragma unroll
        for (int c = 0; c < COLS; ++c) acc[m][c] = fmaf(x1, w1[c], fmaf(x0, w0[c], acc[m][c]));
      }
    }
  } else {
#pragma unroll 2
    for (int k = lane; k < K; k += 64) {
      float wv[COLS];
#pragma unroll
      for (int c = 0; c < COLS; ++c) wv[c] = bf16_to_f32(w[c][k]);
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const float xv = bf16_to_f32(a[m][k]);
#pragma unroll
        for (int c = 0; c < COLS; ++c) acc[m][c] = fmaf(xv, wv[c], acc[m][c]);
      }
    }
  }
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int c = 0; c < COLS; ++c) {
      float r = acc[m][c];
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) r += __shfl_xor(r, off, 64);
      if (lane == 0 && m < M && n0 + c < N) {
        if (bias) r += bf16_to_f32(bias[n0 + c]);
        C[(long)m * ldc + n0 + c] = from_f32<TO>(r);
      }
    }
}

template <typename TO>
static void launch_gemm_plain_few(const void* A, long lda, const void* W, long ldw, const void* bias, void* C, long ldc,
                                  int M, int N, int K, hipStream_t stream) {
  const dim3 block(256);
  const bool pairs = K % 2 == 0 && lda % 2 == 0 && ldw % 2 == 0 && (size_t)A % 4 == 0 && (size_t)W % 4 == 0;
#define FEW(MT_, COLS_)                                                                                                \
  do {                                                                                                                 \
    const dim3 grid((N + 4 * COLS_ - 1) / (4 * COLS_));                                                                \
    if (pairs)                                                                                                         \
      hipLaunchKernelGGL((gemm_plain_few_kernel<TO, MT_, 2, COLS_>), grid, block, 0, stream, (const bf16_t*)A, lda,    \
                         (const bf16_t*)W, ldw, (const bf16_t*)bias, (TO*)C, ldc, M, N, K);                            \
    else                                                                                                               \
      hipLaunchKernelGGL((gemm_plain_few_kernel<TO, MT_, 1, COLS_>), grid, block, 0, stream, (const bf16_t*)A, lda,    \
                         (const bf16_t*)W, ldw, (const bf16_t*)bias, (TO*)C, ldc, M, N, K);                            \
  } while (0)
  if (M <= 1) FEW(1, 1); else if (M <= 2) FEW(2, 1); else if (M <= 4) FEW(4, 2); else if (M <= 8) FEW(8, 4); else FEW(16, 4);
#undef FEW
}

// The product with K split over the waves of a workgroup.
// A workgroup of eight waves owns 8 MR rows by 16 columns; wave w takes part w of K, step by step. A step's rows are read
// whole cache lines at a time (lane (r, c) = (l / 8, l % 8) reads four entries c of rows r, r + 8, ...), the next step's
// while this one is multiplied, and go through an area of LDS that belongs to the wave, from which lane (r, c) takes rows
// r, r + 8, ... and columns c, c + 8 for the outputs it holds: no barrier inside the loop. The waves' sums are added in
// wave order at the end. (Without LDS, every lane fetching the rows it multiplies, a row's 16 bytes go to eight lanes of
// every wave and each line is asked for by all eight waves: nearly twice as long for 8 rows of 128 outputs.) What bounds
// it is the trip to memory with few outputs (8 x 128 x 352 2.9 us where the tiles took 34, 8 x 4,096 x 4,096 13.5 where
// they took 398); with many the tiles are ahead, which read 2 bytes of LDS a multiply-add where 32 rows here read 3.
#define GP_ROW (GP_STEP + 4)      // floats a row takes in LDS: eight rows at a time lie on distinct banks

// four neighbouring entries; VEC: in one load (K is a multiple of 4 then), else one by one, those from K on as zeros
template <bool VEC>
__device__ __forceinline__ float4 gp_load4(const float* p, int k, int K) {
  if (VEC) return k < K ? *reinterpret_cast<const float4*>(p + k) : make_float4(0.f, 0.f, 0.f, 0.f);
  return make_float4(k < K ? p[k] : 0.f, k + 1 < K ? p[k + 1] : 0.f, k + 2 < K ? p[k + 2] : 0.f, k + 3 < K ? p[k + 3] : 0.f);
}
template <bool VEC>
__device__ __forceinline__ float4 gp_load4(const bf16_t* p, int k, int K) {
  if (VEC) {
    const uint2 v = k < K ? *reinterpret_cast<const uint2*>(p + k) : make_uint2(0u, 0u);
    return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                       __uint_as_float(v.y & 0xffff0000u));
  }
  return make_float4(k < K ? bf16_to_f32(p[k]) : 0.f, k + 1 < K ? bf16_to_f32(p[k + 1]) : 0.f,
                     k + 2 < K ? bf16_to_f32(p[k + 2]) : 0.f, k + 3 < K ? bf16_to_f32(p[k + 3]) : 0.f);
}

// What a product of the split form does beside multiplying (GP_PLAIN: nothing), float32 operands read wide only. With few
// rows a kernel between two products costs its start and end and little else (3.5 us in a captured step), so a decoder
// block's products do the work around them, to the bits of the kernels they replace:
//   GP_ADD    the product is added to C, the float32 residual stream;
//   GP_GATED  act(gate) * up of W's two halves of I rows: a workgroup's two times eight rows of W are the gate's and the up
//             projection's of eight outputs;
//   GP_QKV    the fused QKV projection: the two times eight rows are those of eight rotation pairs (i, i + d / 2) of a
//             head, which the epilogue rotates and stores, in the cache too.
// NORM: A is the residual stream and its rows are normalised on the way in, x * inv * (w + offset); every workgroup makes
// the factors of its own rows, adding up squares in the order of the norm's kernel (a wave's 64 lanes hold four
// neighbours each, the parts of 256 columns are added in turn), while its first rows of W are on their way.
enum { GP_PLAIN = 0, GP_ADD, GP_GATED, GP_QKV };

struct GpFused {
  const float* norm_weight;         // NORM: [K]
  float eps, weight_offset;
  int act;                          // GP_GATED: 1 SiLU, 2 GELU
  // GP_QKV, pages of float32 (common.h: RopeCacheArgs)
  const int* positions;
  const float* table;
  const int* slots;
  float *k_pages, *v_pages;
  int nh, nkv, d, ps;
};

template <typename TA, typename TW, typename TO, int MR, bool VEC, int FORM = GP_PLAIN, bool NORM = false>
__global__ __launch_bounds__(512, 4) void gemm_plain_split_kernel(const TA* __restrict__ A, long lda,
                                                               const TW* __restrict__ W, long ldw,
                                                               const TW* __restrict__ bias, TO* __restrict__ C,
                                                               long ldc, int M, int N, int K, GpFused fu) {
  constexpr int ROWS = 8 * MR + 16;                 // of A, then of W
  constexpr bool PAIRS = FORM == GP_GATED || FORM == GP_QKV;
  static_assert(ROWS * GP_ROW >= MR * 128, "the waves' sums lie where their steps lay");
  static_assert(FORM == GP_PLAIN ? !NORM : (VEC && sizeof(TA) == 4 && sizeof(TW) == 4 && sizeof(TO) == 4), "float32 forms");
  __shared__ __align__(16) float area[8][ROWS * GP_ROW];
  __shared__ float factor[NORM ? 8 * MR : 1];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane >> 3, c = lane & 7;
  const int m0 = blockIdx.y * (8 * MR), n0 = blockIdx.x * 16;
  float* mine = area[wave];
  // rows of W: ``first`` + 0..7 and ``second`` + 0..7 (PAIRS: outputs o0 .. o0 + 7 of either half; o0 is within one head)
  const int half = FORM == GP_QKV ? fu.d / 2 : FORM == GP_GATED ? N / 2 : 8;
  const int o0 = n0 / 2, first = FORM == GP_QKV ? o0 / half * fu.d + o0 % half : PAIRS ? o0 : n0, second = first + half;
  const TA* a[MR];
  const TW* w[2];
#pragma unroll
  for (int i = 0; i < MR; ++i) a[i] = A + (long)min(m0 + r + 8 * i, M - 1) * lda;   // rows beyond M: not written
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int row = FORM == GP_GATED ? min(first + r, half - 1) + j * half : min((j ? second : first) + r, N - 1);
    w[j] = W + (long)row * ldw;
  }
  float acc[MR][2][2];        // of the even and of the odd k: two short chains instead of one
#pragma unroll
  for (int i = 0; i < MR; ++i)
#pragma unroll
    for (int e = 0; e < 2; ++e) acc[i][0][e] = acc[i][1][e] = 0.f;
  float4 x[MR], y[2], g;
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < MR; ++i) x[i] = gp_load4<VEC>(a[i], k0 + 4 * c, K);
#pragma unroll
    for (int j = 0; j < 2; ++j) y[j] = gp_load4<VEC>(w[j], k0 + 4 * c, K);
    if (NORM) g = gp_load4<VEC>(fu.norm_weight, k0 + 4 * c, K);
  };
  int k0 = gp_part(wave, K);
  const int end = gp_part(wave + 1, K);
  if (k0 < end) fetch(k0);
  float inv[MR];
  if (NORM) {
#pragma unroll
    for (int i = 0; i < MR; ++i) {
      const float* row = reinterpret_cast<const float*>(A) + (long)min(m0 + wave * MR + i, M - 1) * lda;
      float total = 0.f;
#pragma unroll 4
      for (int k = 0; k < K; k += 256) {
        const float4 v = gp_load4<true>(row, k + 4 * lane, K);
        float ss = 0.f;
        ss += v.x * v.x;
        ss += v.y * v.y;
        ss += v.z * v.z;
        ss += v.w * v.w;
        total += wave_sum(ss);
      }
      if (lane == 0) factor[wave * MR + i] = rsqrtf(total / (float)K + fu.eps);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MR; ++i) inv[i] = factor[r + 8 * i];
  }
  for (; k0 < end; k0 += GP_STEP) {
#pragma unroll
    for (int i = 0; i < MR; ++i) {
      if (NORM) {
        x[i].x = x[i].x * inv[i] * (g.x + fu.weight_offset);
        x[i].y = x[i].y * inv[i] * (g.y + fu.weight_offset);
        x[i].z = x[i].z * inv[i] * (g.z + fu.weight_offset);
        x[i].w = x[i].w * inv[i] * (g.w + fu.weight_offset);
      }
      *reinterpret_cast<float4*>(mine + (r + 8 * i) * GP_ROW + 4 * c) = x[i];
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) *reinterpret_cast<float4*>(mine + (8 * MR + r + 8 * j) * GP_ROW + 4 * c) = y[j];
    if (k0 + GP_STEP < end) fetch(k0 + GP_STEP);
    __builtin_amdgcn_wave_barrier();                // (a wave's LDS accesses are carried out in their order)
#pragma unroll
    for (int q = 0; q < GP_STEP; q += 4) {
      float xe[MR][4], ye[2][4];
#pragma unroll
      for (int i = 0; i < MR; ++i)
        *reinterpret_cast<float4*>(xe[i]) = *reinterpret_cast<const float4*>(mine + (r + 8 * i) * GP_ROW + q);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        *reinterpret_cast<float4*>(ye[j]) = *reinterpret_cast<const float4*>(mine + (8 * MR + c + 8 * j) * GP_ROW + q);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < MR; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j][e & 1] = fmaf(xe[i][e], ye[j][e], acc[i][j][e & 1]);
    }
    __builtin_amdgcn_wave_barrier();
  }
#pragma unroll
  for (int i = 0; i < MR; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) mine[(i * 2 + j) * 64 + lane] = acc[i][j][0] + acc[i][j][1];
  __syncthreads();
  auto finished = [&](int e, int n) {      // the waves' sums of entry e, and column n's bias
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < GP_PARTS; ++v) s += area[v][e];
    if (bias) s += to_f32<TW>(bias[n]);
    return s;
  };
  if constexpr (!PAIRS) {
    for (int e = tid; e < MR * 128; e += 512) {
      const int l = e & 63, j = (e >> 6) & 1, i = e >> 7;
      const int m = m0 + l / 8 + 8 * i, n = n0 + l % 8 + 8 * j;
      if (m >= M || n >= N) continue;
      const float s = finished(e, n);
      TO* to = C + (long)m * ldc + n;
      if constexpr (FORM == GP_ADD) *to = s + *to; else *to = from_f32<TO>(s);
    }
  } else {
    for (int e = tid; e < MR * 64; e += 512) {
      const int l = e & 63, i = e >> 6, at = i * 128 + l;
      const int m = m0 + l / 8 + 8 * i, o = first + l % 8;
      if (m >= M || (FORM == GP_GATED && o >= half)) continue;
      const float u = finished(at, o), v = finished(at + 64, o + half);
      if constexpr (FORM == GP_GATED) {
        C[(long)m * ldc + o] = (fu.act == 1 ? gated_product_activation<1>(u) : gated_product_activation<2>(u)) * v;
      } else {
        const int head = o / fu.d, at_d = o - head * fu.d;
        float lo = u, hi = v;
        if (head < fu.nh + fu.nkv) {
          const float* cs = fu.table + (long)fu.positions[m] * fu.d;
          rope_rotate(u, v, cs[at_d], cs[half + at_d], &lo, &hi);
        }
        C[(long)m * ldc + o] = lo;
        C[(long)m * ldc + o + half] = hi;
        const int slot = head >= fu.nh ? fu.slots[m] : -1;
        if (slot >= 0) {
          const int page = slot / fu.ps, off = slot - page * fu.ps;
          if (head < fu.nh + fu.nkv) {
            float* dst = fu.k_pages + (((long)page * fu.nkv + (head - fu.nh)) * fu.ps + off) * fu.d + at_d;
            dst[0] = lo;
            dst[half] = hi;
          } else {
            float* dst = fu.v_pages + (((long)page * fu.nkv + (head - fu.nh - fu.nkv)) * fu.d + at_d) * fu.ps + off;
            dst[0] = lo;
            dst[(long)half * fu.ps] = hi;
          }
        }
      }
    }
  }
}

// Rows of a workgroup of the split form, in eights. A workgroup of 8 rows is done soonest (its chains of multiply-adds and
// reads of LDS are a quarter of those of 32 rows), one of 32 reads W a quarter as often: 8 rows while such workgroups have
// a compute unit each (64 x 704 x 128: 32 rows 3.3 us, 16 2.8, 8 2.6; 32 x 1,024 x 2,816 15.4, 10.2, 8.2), 16 rows while
// there are two of 8 to a unit (64 x 1,024 x 2,816 15.6, 10.9, 13.8; with a short K four: 128 x 1,000 x 128 3.5, 3.1, 4.2),
// else 32 (96 x 1,024 x 2,816 16.1, 18.5, 19.5).
static int gp_rows(int M, int N, int K) {
  const long eights = ((long)M + 7) / 8 * (((long)N + 15) / 16), units = lmsf_compute_units();
  if (M <= 8 || eights <= units) return 1;
  return M <= 16 || eights <= (K <= 128 ? 4 : 2) * units ? 2 : 4;
}

template <typename TA, typename TW, typename TO, bool VEC>
static void launch_gemm_plain_split(const void* A, long lda, const void* W, long ldw, const void* bias, void* C, long ldc,
                                    int M, int N, int K, hipStream_t stream) {
  const dim3 block(512);
#define SPLIT(MR_)                                                                                                     \
  hipLaunchKernelGGL((gemm_plain_split_kernel<TA, TW, TO, MR_, VEC>), dim3((N + 15) / 16, (M + 8 * MR_ - 1) / (8 * MR_)), \
                     block, 0, stream, (const TA*)A, lda, (const TW*)W, ldw, (const TW*)bias, (TO*)C, ldc, M, N, K, GpFused())
  const int rows = gp_rows(M, N, K);
  if (rows == 1) SPLIT(1); else if (rows == 2) SPLIT(2); else SPLIT(4);
#undef SPLIT
}

template <int FORM, bool NORM>
static void launch_gemm_plain_fused(const float* A, long lda, const float* W, long ldw, const float* bias, float* C,
                                    long ldc, int M, int N, int K, const GpFused& fu, hipStream_t stream) {
  const dim3 block(512);
  constexpr int MOST = NORM ? 2 : 4;      // (many rows leave the norm to its kernel)
#define FUSED(MR_)                                                                                                     \
  hipLaunchKernelGGL((gemm_plain_split_kernel<float, float, float, MR_, true, FORM, NORM>),                            \
                     dim3((N + 15) / 16, (M + 8 * MR_ - 1) / (8 * MR_)), block, 0, stream, A, lda, W, ldw, bias, C, ldc, \
                     M, N, K, fu)
  const int rows = gp_rows(M, N, K);
  if (rows == 1) FUSED(1); else if (rows == 2) FUSED(2); else FUSED(MOST);
#undef FUSED
}

// Whether the split form runs (``wide``: rows that allow wide loads; ``half``: an operand of 16 bits). It takes rows in
// pieces of 32 x 16 outputs (8 or 16 rows where there are no more, for which a piece costs a quarter or half as much, or
// where those run side by side: gp_rows),
// which fill the chip where 64x64 tiles leave compute units without one, and K in eight parts, of which a K of one or two
// steps leaves most waves without work. The tiles are ahead from a number of pieces a compute unit on that falls with K (two
// workgroups run on a unit at once: up to K = 32 a second round already costs more than a tile's whole K) and that is
// lower for rows read entry by entry, of 16-bit entries above all. Split form -> tiles in us by the number of pieces on 256
// units: wide float32, K = 16: 512 3.2 -> 4.1, 875 4.9 -> 4.2; K = 64: 1,008 5.7 -> 7.0, 1,712 9.8 -> 8.0; K = 128: 1,712
// 11.1 -> 11.5, 2,512 14.2 -> 12.9; K = 256: 2,520 16.5 -> 19.9, 3,969 25.3 -> 21.7. Entry by entry in float32, K = 33:
// 512 4.1 -> 6.0, 1,250 9.0 -> 6.6; K = 65: 1,008 7.5 -> 8.2, 1,712 12.0 -> 9.1; K = 333: 1,250 19.7 -> 24.0, 1,827 28.1
// -> 25.0; in bfloat16, K = 15: 441 5.3 -> 4.4, 1,008 9.2 -> 4.6; K = 33: 512 5.3 -> 6.3, 875 8.6 -> 6.4; K = 333: 912
// 21.2 -> 24.9, 1,200 27.0 -> 24.8. Few rows: 8 of 50,000 columns, K = 16 6.5 -> 5.4, K = 64 6.7 -> 10.4, K = 333 20 -> 41; 16
// rows 8.0 -> 5.6, 8.6 -> 10.7, 27 -> 41; 32 rows, K = 16 13.4 -> 6.4, K = 128 17.9 -> 18.8, K = 256 21 -> 33.
static bool gp_split(int M, int N, int K, bool wide, bool half) {
  const long rows = ((long)M + 31) / 32, pieces = rows * (((long)N + 15) / 16);
  if (rows > 65535 || N > 1 << 26) return false;      // beyond what a grid takes
  if (wide ? (M <= 16 && K > 32) || (M <= 32 && K > 128) : !half && M <= 16 && K > 128) return true;
  long most;                                          // twice the pieces of a compute unit
  if (wide)
    most = K <= 32 ? 4 : K <= 64 ? 9 : K <= 128 ? 14 : 26;
  else if (half)
    most = K <= 16 ? 0 : K <= 128 ? 4 : 8;
  else
    most = K <= 64 ? 4 : K <= 128 ? 8 : 12;
  const int eighths = M <= 8 ? 2 : M <= 16 ? 4 : M <= 32 ? 6 : 8;       // what a piece costs
  return pieces * eighths <= 4 * most * lmsf_compute_units();
}

template <typename TA, typename TW, typename TO>
static void launch_gemm_plain(const void* A, long lda, const void* W, long ldw, const void* bias, void* C, long ldc,
                              int M, int N, int K, hipStream_t stream) {
  const bool wide = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && (size_t)A % (4 * sizeof(TA)) == 0 &&
                    (size_t)W % (4 * sizeof(TW)) == 0;
  if (!gp_split(M, N, K, wide, sizeof(TA) == 2 || sizeof(TW) == 2)) {
    const dim3 grid((N + GP_TILE - 1) / GP_TILE, (M + GP_TILE - 1) / GP_TILE), block(256);
    hipLaunchKernelGGL((gemm_plain_kernel<TA, TW, TO>), grid, block, 0, stream, (const TA*)A, lda, (const TW*)W, ldw,
                       (const TW*)bias, (TO*)C, ldc, M, N, K);
  } else if (wide) {
    launch_gemm_plain_split<TA, TW, TO, true>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
  } else {
    launch_gemm_plain_split<TA, TW, TO, false>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
  }
}

// Supported (a, w, c) dtypes: (f32,f32,f32), (bf16,bf16,bf16), (bf16,bf16,f32), (f32,bf16,f32),
// (bf16,f32,bf16), (bf16,f32,f32). bias has the dtype of the weight or is null.
extern "C" int lmsf_gemm_plain(const void* A, int a_dtype, long lda, const void* W, int w_dtype, long ldw,
                               const void* bias, void* C, int c_dtype, long ldc, int M, int N, int K,
                               hipStream_t stream) {
  LMSF_CHECK(A && W && C, "gemm_plain: null pointer");
  LMSF_CHECK(M >= 0 && N > 0 && K > 0, "gemm_plain: bad sizes M=%d N=%d K=%d", M, N, K);
  LMSF_CHECK(lda >= K && ldw >= K && ldc >= N, "gemm_plain: leading dimensions too small");
  LMSF_CHECK((M + GP_TILE - 1) / GP_TILE <= 65535, "gemm_plain: M=%d too large", M);
  if (M == 0) return 0;
  if (M <= GP_FEW_ROWS && a_dtype == LMSF_BF16 && w_dtype == LMSF_BF16) {
    if (c_dtype == LMSF_BF16)
      launch_gemm_plain_few<bf16_t>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
    else
      launch_gemm_plain_few<float>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
    LMSF_LAUNCH_CHECK("gemm_plain");
    return 0;
  }
  const int key = a_dtype * 100 + w_dtype * 10 + c_dtype;
  switch (key) {
    case 0: launch_gemm_plain<float, float, float>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream); break;
    case 111: launch_gemm_plain<bf16_t, bf16_t, bf16_t>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream); break;
    case 110: launch_gemm_plain<bf16_t, bf16_t, float>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream); break;
    case 10: launch_gemm_plain<float, bf16_t, float>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream); break;
    case 101: launch_gemm_plain<bf16_t, float, bf16_t>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream); break;
    case 100: launch_gemm_plain<bf16_t, float, float>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream); break;
    default:
      lmsf_set_error("gemm_plain: dtype combination a=%d w=%d c=%d not supported", a_dtype, w_dtype, c_dtype);
      return 1;
  }
  LMSF_LAUNCH_CHECK("gemm_plain");
  return 0;
}

// The split form's fused products (float32 throughout; see GpFused): whether a product of these sizes runs in the split
// form at all, and (``normed``) whether it should normalise its rows itself. N: rows of W. K and the row strides a multiple
// of 4, 16-byte aligned operands. Every workgroup makes its rows' factors anew, which pays for itself while there are two
// workgroups of 8 rows to a compute unit, one beyond K = 512 (norm, gated product with its activation -> all in one:
// 8 x 704 x 128 4.6 -> 3.2 us, 64 x 704 x 128 4.7 -> 3.8, 128 x 1,000 x 128 5.1 -> 4.9, 32 x 1,408 x 256 5.0 -> 4.0, 96 rows
// 6.3 -> 6.7; 16 x 704 x 1,024 6.3 -> 6.0, 48 rows 7.4 -> 8.6; 8 x 5,632 x 1,024 9.0 -> 8.2, x 11,264 x 2,048 20.3 -> 20.9).
extern "C" int lmsf_gemm_plain_fused_fits(int M, int N, int K, int normed) {
  if (M <= 0 || K % 4 != 0 || !gp_split(M, N, K, true, false)) return 0;
  const long eights = ((long)M + 7) / 8 * (((long)N + 15) / 16);
  return !normed || (K <= 1024 && eights <= (K <= 512 || M <= 8 ? 2 : 1) * lmsf_compute_units()) ? 1 : 0;
}

static int fused_check(const char* who, const float* x, long ldx, const float* W, long ldw, const float* y, long ldy, int M,
                       int N, int K, long width) {
  LMSF_CHECK(x && W && y, "%s: null pointer", who);
  LMSF_CHECK(M >= 0 && N > 0 && K > 0 && K % 4 == 0, "%s: bad sizes M=%d N=%d K=%d", who, M, N, K);
  LMSF_CHECK(N <= 1 << 26 && (M + 7) / 8 <= 65535, "%s: M=%d N=%d too large", who, M, N);
  LMSF_CHECK(ldx >= K && ldw >= K && ldy >= width && ldx % 4 == 0 && ldw % 4 == 0, "%s: bad row strides", who);
  LMSF_CHECK(lmsf_aligned16(x) && lmsf_aligned16(W), "%s: x and W must be 16-byte aligned", who);
  return 0;
}
static int norm_check(const char* who, const float* norm_weight, int K, float eps) {
  // (the norm's kernel adds up squares in another order beyond)
  LMSF_CHECK(norm_weight == nullptr || (lmsf_aligned16(norm_weight) && K <= 4096 && eps > 0.f),
             "%s: rows of up to 4,096 columns are normalised, by an aligned weight", who);
  return 0;
}

// stream += x W^T + bias; stream [M, N] float32 with row stride ldy.
extern "C" int lmsf_gemm_plain_add(const float* x, long ldx, const float* W, long ldw, const float* bias, float* stream_out,
                                   long ldy, int M, int N, int K, hipStream_t stream) {
  if (int rc = fused_check("gemm_plain_add", x, ldx, W, ldw, stream_out, ldy, M, N, K, N)) return rc;
  if (M == 0) return 0;
  launch_gemm_plain_fused<GP_ADD, false>(x, ldx, W, ldw, bias, stream_out, ldy, M, N, K, GpFused(), stream);
  LMSF_LAUNCH_CHECK("gemm_plain_add");
  return 0;
}

// act(x Wg^T + bg) * (x Wu^T + bu) for W [2 I, K] = [Wg; Wu]; y [M, I]; act 1 SiLU, 2 GELU. With ``norm_weight`` [K] x is
// the residual stream and its rows are normalised first, x * rsqrt(mean(x^2) + eps) * (norm_weight + weight_offset).
extern "C" int lmsf_gemm_plain_gated(const float* x, long ldx, const float* W, long ldw, const float* bias, float* y, long ldy,
                                     int M, int I, int K, int act, const float* norm_weight, float eps, float weight_offset,
                                     hipStream_t stream) {
  if (int rc = fused_check("gemm_plain_gated", x, ldx, W, ldw, y, ldy, M, 2 * I, K, I)) return rc;
  if (int rc = norm_check("gemm_plain_gated", norm_weight, K, eps)) return rc;
  LMSF_CHECK(act == 1 || act == 2, "gemm_plain_gated: activation %d (1 silu, 2 gelu)", act);
  if (M == 0) return 0;
  GpFused fu = GpFused();
  fu.norm_weight = norm_weight; fu.eps = eps; fu.weight_offset = weight_offset; fu.act = act;
  if (norm_weight)
    launch_gemm_plain_fused<GP_GATED, true>(x, ldx, W, ldw, bias, y, ldy, M, 2 * I, K, fu, stream);
  else
    launch_gemm_plain_fused<GP_GATED, false>(x, ldx, W, ldw, bias, y, ldy, M, 2 * I, K, fu, stream);
  LMSF_LAUNCH_CHECK("gemm_plain_gated");
  return 0;
}

// The fused QKV projection, the rotation of its q and k heads over the whole head (NeoX pairing, d a multiple of 16) and
// the write of k and v into float32 pages; arguments as lmsf_gemm_qkv_rope_cache, ``norm_weight`` as above.
extern "C" int lmsf_gemm_plain_qkv(const float* x, long ldx, const float* W, long ldw, const float* bias, float* y, long ldy,
                                   int M, int K, const int* positions, const float* table, int max_pos, const int* slots,
                                   float* k_pages, float* v_pages, long num_pages, int nh, int nkv, int d, int ps,
                                   const float* norm_weight, float eps, float weight_offset, hipStream_t stream) {
  LMSF_CHECK(positions && table && slots && k_pages && v_pages, "gemm_plain_qkv: null pointer");
  LMSF_CHECK(nh > 0 && nkv > 0 && d > 0 && d % 16 == 0, "gemm_plain_qkv: head size %d must be a multiple of 16", d);
  LMSF_CHECK(ps > 0 && num_pages > 0 && max_pos > 0, "gemm_plain_qkv: bad page geometry or empty table");
  const long N = (long)(nh + 2 * nkv) * d;
  LMSF_CHECK(N <= 1 << 26, "gemm_plain_qkv: %ld columns", N);
  if (int rc = fused_check("gemm_plain_qkv", x, ldx, W, ldw, y, ldy, M, (int)N, K, N)) return rc;
  if (int rc = norm_check("gemm_plain_qkv", norm_weight, K, eps)) return rc;
  if (M == 0) return 0;
  GpFused fu = GpFused();
  fu.norm_weight = norm_weight; fu.eps = eps; fu.weight_offset = weight_offset;
  fu.positions = positions; fu.table = table; fu.slots = slots; fu.k_pages = k_pages; fu.v_pages = v_pages;
  fu.nh = nh; fu.nkv = nkv; fu.d = d; fu.ps = ps;
  if (norm_weight)
    launch_gemm_plain_fused<GP_QKV, true>(x, ldx, W, ldw, bias, y, ldy, M, (int)N, K, fu, stream);
  else
    launch_gemm_plain_fused<GP_QKV, false>(x, ldx, W, ldw, bias, y, ldy, M, (int)N, K, fu, stream);
  LMSF_LAUNCH_CHECK("gemm_plain_qkv");
  return 0;
}
