// Dynamic Tanh in the place of a norm, around the float32 residual stream:
//
//   r = (residual ? residual[src] : 0) + (branch ? branch[src] : 0)       src = rows ? rows[row] : row
//   residual[row] = r                                                     (branch and residual given, no rows)
//   out[row] = tanh(alpha * r) * w + b
//
// alpha is one learned number (read from device memory), w and b vectors. No mean and no variance are computed,
// so nothing crosses a row: a thread an element (four neighbours where the row allows it). All arithmetic is
// float32; branch and out are float32 or bfloat16. The reference's only norm is RMSNorm
// (vllm/kernels/layernorm_kernels.cu:13-38), with the same fused addition (:41-68).
#include "common.h"
#include "entry_points.h"

#include <math.h>

template <typename TB, typename TO, int V>
__global__ __launch_bounds__(256) void dyt_norm_kernel(const TB* __restrict__ branch, float* __restrict__ residual,
                                                       const float* __restrict__ w, const float* __restrict__ b,
                                                       const float* __restrict__ alpha, TO* __restrict__ out,
                                                       const int* __restrict__ rows, int H) {
  const int row = blockIdx.x;
  const long src = rows ? rows[row] : row;
  const int i0 = (blockIdx.y * 256 + threadIdx.x) * V;
  if (i0 >= H) return;
  const float a = alpha[0];
  float r[V];
#pragma unroll
  for (int e = 0; e < V; ++e) {
    r[e] = residual ? residual[src * H + i0 + e] : 0.f;
    if (branch) r[e] += to_f32<TB>(branch[src * H + i0 + e]);
  }
  if (branch && residual && !rows) {
#pragma unroll
    for (int e = 0; e < V; ++e) residual[src * H + i0 + e] = r[e];
  }
#pragma unroll
  for (int e = 0; e < V; ++e) out[(long)row * H + i0 + e] = from_f32<TO>(tanhf(a * r[e]) * w[i0 + e] + b[i0 + e]);
}

// The same for many rows: a thread takes four neighbouring columns of R rows, asks for all of them at once and reads w and b,
// which are more bytes than a row of the stream and the branch, once for all of them. Memory-bound: 12 bytes an entry with
// bfloat16 around it; 2,048 rows of 2,048 22.0 -> 12.5 us (4.0 TB/s), 1,034 rows 13.4 -> 8.5, 8,000 rows 76 -> 36.
template <typename T> struct Dyt4;
template <> struct Dyt4<float> {
  static __device__ __forceinline__ float4 load(const float* p) { return *reinterpret_cast<const float4*>(p); }
  static __device__ __forceinline__ void store(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }
};
template <> struct Dyt4<bf16_t> {
  static __device__ __forceinline__ float4 load(const bf16_t* p) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                       __uint_as_float(v.y & 0xffff0000u));
  }
  static __device__ __forceinline__ void store(bf16_t* p, float4 v) {
    *reinterpret_cast<uint2*>(p) = make_uint2(pack2_bf16(v.x, v.y), pack2_bf16(v.z, v.w));
  }
};
template <typename TB, typename TO, int R>
__global__ __launch_bounds__(256) void dyt_norm_rows_kernel(const TB* __restrict__ branch, float* __restrict__ residual,
                                                            const float* __restrict__ w, const float* __restrict__ b,
                                                            const float* __restrict__ alpha, TO* __restrict__ out,
                                                            const int* __restrict__ rows, int n_rows, int H) {
  const int row0 = blockIdx.x * R, i0 = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (i0 >= H) return;
  long src[R];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int row = min(row0 + q, n_rows - 1);
    src[q] = (rows ? rows[row] : row) * (long)H + i0;
  }
  float4 r[R], y[R];
#pragma unroll
  for (int q = 0; q < R; ++q) r[q] = residual ? Dyt4<float>::load(residual + src[q]) : make_float4(0.f, 0.f, 0.f, 0.f);
  if (branch) {
#pragma unroll
    for (int q = 0; q < R; ++q) y[q] = Dyt4<TB>::load(branch + src[q]);
  }
  const float a = alpha[0];
  const float4 wv = Dyt4<float>::load(w + i0), bv = Dyt4<float>::load(b + i0);
#pragma unroll
  for (int q = 0; q < R; ++q) {
    if (branch) {
      r[q].x += y[q].x; r[q].y += y[q].y; r[q].z += y[q].z; r[q].w += y[q].w;
    }
    if (row0 + q < n_rows) {
      if (branch && residual && !rows) Dyt4<float>::store(residual + src[q], r[q]);
      Dyt4<TO>::store(out + (long)(row0 + q) * H + i0,
                      make_float4(tanhf(a * r[q].x) * wv.x + bv.x, tanhf(a * r[q].y) * wv.y + bv.y,
                                  tanhf(a * r[q].z) * wv.z + bv.z, tanhf(a * r[q].w) * wv.w + bv.w));
    }
  }
}

// 1 where n_rows rows of H columns are the kernel's of R rows a thread (where every piece is aligned): more than a workgroup a
// compute unit (fewer: level, both wait for one trip to memory), and 512 columns, or 8,000 rows: fewer columns leave a
// workgroup's waves idle, and a wave with four rows to itself is slower than four waves until the chip is full. One row a thread against four: 1,030
// rows of 64 / 256 / 384 / 512 columns 3.2 / 3.6 / 4.2 / 5.0 against 4.5 / 4.1 / 4.5 / 4.9 us, 2,048 rows of 64 / 256 / 384 3.7 / 4.6 / 5.9
// against 5.2 / 4.9 / 5.4, 8,000 rows of 8 / 64 / 256 6.9 / 6.9 / 11.7 against 5.2 / 5.1 / 7.6.
#define DYT_ROWS_A_THREAD 4
extern "C" int lmsf_dyt_norm_many(int n_rows, int H) {
  const int R = DYT_ROWS_A_THREAD;
  return H % 4 == 0 && (H >= 512 || n_rows >= 8000) && (long)((n_rows + R - 1) / R) * ((H / 4 + 255) / 256) > 256;
}

extern "C" int lmsf_dyt_norm(const void* branch, int branch_dtype, float* residual, const float* w, const float* b,
                             const float* alpha, void* out, int out_dtype, const int* rows, int n_rows, int H,
                             hipStream_t stream) {
  LMSF_CHECK(w && b && alpha && out, "dyt_norm: null pointer");
  LMSF_CHECK(branch || residual, "dyt_norm: neither a branch nor a residual");
  LMSF_CHECK(n_rows >= 0 && H > 0, "dyt_norm: bad sizes rows=%d H=%d", n_rows, H);
  LMSF_CHECK((branch_dtype == LMSF_F32 || branch_dtype == LMSF_BF16) && (out_dtype == LMSF_F32 || out_dtype == LMSF_BF16),
             "dyt_norm: unknown dtype code");
  if (n_rows == 0) return 0;
  const bool v4 = H % 4 == 0;
  const int per = v4 ? 4 : 1;
  dim3 grid(n_rows, (H / per + 255) / 256), block(256);
  constexpr int R = DYT_ROWS_A_THREAD;
  const bool many = lmsf_dyt_norm_many(n_rows, H) && lmsf_aligned16(residual) && lmsf_aligned16(w) && lmsf_aligned16(b) &&
                    lmsf_aligned16(branch) && lmsf_aligned16(out);
  if (many) {
    grid.x = (n_rows + R - 1) / R;
#define DYT_ROWS(TB, TO)                                                                                               \
  hipLaunchKernelGGL((dyt_norm_rows_kernel<TB, TO, R>), grid, block, 0, stream, (const TB*)branch, residual, w, b,     \
                     alpha, (TO*)out, rows, n_rows, H)
    if (branch_dtype == LMSF_F32 && out_dtype == LMSF_F32) DYT_ROWS(float, float);
    else if (branch_dtype == LMSF_F32) DYT_ROWS(float, bf16_t);
    else if (out_dtype == LMSF_F32) DYT_ROWS(bf16_t, float);
    else DYT_ROWS(bf16_t, bf16_t);
#undef DYT_ROWS
    LMSF_LAUNCH_CHECK("dyt_norm_rows");
    return 0;
  }
#define DYT(TB, TO)                                                                                                    \
  do {                                                                                                                 \
    if (v4)                                                                                                            \
      hipLaunchKernelGGL((dyt_norm_kernel<TB, TO, 4>), grid, block, 0, stream, (const TB*)branch, residual, w, b,      \
                         alpha, (TO*)out, rows, H);                                                                    \
    else                                                                                                               \
      hipLaunchKernelGGL((dyt_norm_kernel<TB, TO, 1>), grid, block, 0, stream, (const TB*)branch, residual, w, b,      \
                         alpha, (TO*)out, rows, H);                                                                    \
  } while (0)
  if (branch_dtype == LMSF_F32 && out_dtype == LMSF_F32) DYT(float, float);
  else if (branch_dtype == LMSF_F32) DYT(float, bf16_t);
  else if (out_dtype == LMSF_F32) DYT(bf16_t, float);
  else DYT(bf16_t, bf16_t);
#undef DYT
  LMSF_LAUNCH_CHECK("dyt_norm");
  return 0;
}
