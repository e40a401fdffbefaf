// okq_neighbours.hip -- the f32 operations on either side of the quantized
// projections, for the paths that cannot fold them into the GEMV prologue
// (batched rows on the MFMA GEMM, rows the streaming GEMV does not take).
//
//   rmsnorm: out[r, i] = (x[r, i] * (1 / sqrt(sum_i x[r, i]^2 / hidden + eps))) * w[i]
//            (crates/kernels/src/rmsnorm.rs:73-128, same order of operations;
//            the sum of squares is reduced in a fixed tree order)
//   swiglu : out[i] = (gate[i] * (1 / (1 + exp(-gate[i])))) * up[i]
//            (crates/kernels/src/mlp.rs:77-88, :233-238)
#include "okq_device.h"
#include "okq_internal.h"

namespace okq {

// A row's values stay in registers between its sum of squares and its output
// (V float4 per thread), and the norm weights are requested with them, so the
// row is read once and a call waits for memory once.  A decode call is a
// handful of rows: nothing but that latency bounds it, so a row gets as many
// threads as it has float4s, up to 1024.
//   rows x 4096, per launch: 1 row 13.8 -> 4.5 us, 32 rows 12.9 -> 4.7 us,
//   333 rows 9.7 -> 5.1 us (against 256 threads reading a row twice, one
//   value per load, which rmsnorm_kernel below still does for other shapes)
template <int V>
__global__ __launch_bounds__(1024) void rmsnorm4_kernel(const float *__restrict__ x, int hidden4,
                                                        const float *__restrict__ w, float eps,
                                                        float *__restrict__ out) {
  __shared__ float red[16];
  const int tid = (int)threadIdx.x, nt = (int)blockDim.x;
  const float4 *row = reinterpret_cast<const float4 *>(x) + (int64_t)blockIdx.x * hidden4;
  const float4 *w4 = reinterpret_cast<const float4 *>(w);
  float4 *orow = reinterpret_cast<float4 *>(out) + (int64_t)blockIdx.x * hidden4;
  float4 v[V], g[V];
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const int i = tid + j * nt;
    v[j] = i < hidden4 ? row[i] : float4{0.0f, 0.0f, 0.0f, 0.0f};
  }
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const int i = tid + j * nt;
    g[j] = i < hidden4 ? w4[i] : float4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  float ss = 0.0f;
#pragma unroll
  for (int j = 0; j < V; ++j) ss += (v[j].x * v[j].x + v[j].y * v[j].y) + (v[j].z * v[j].z + v[j].w * v[j].w);
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  // the waves' sums meet in every 16-lane row, in one fixed order
  const int i16 = tid & 15;
  float tot = i16 < nt >> 6 ? red[i16] : 0.0f;
  tot += dpp_row_f<0xB1>(tot);
  tot += dpp_row_f<0x4E>(tot);
  tot += dpp_row_f<0x141>(tot);
  tot += dpp_row_f<0x140>(tot);
  const float inv = 1.0f / sqrtf(tot / (float)(4 * hidden4) + eps);
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const int i = tid + j * nt;
    if (i < hidden4)
      orow[i] = float4{v[j].x * inv * g[j].x, v[j].y * inv * g[j].y, v[j].z * inv * g[j].z, v[j].w * inv * g[j].w};
  }
}

// Any length and alignment: one workgroup of 256 threads per row, one value
// per load.
__global__ __launch_bounds__(256) void rmsnorm_kernel(const float *__restrict__ x, int64_t hidden,
                                                      const float *__restrict__ w, float eps,
                                                      float *__restrict__ out) {
  __shared__ float red[4];
  const float *row = x + (int64_t)blockIdx.x * hidden;
  float *orow = out + (int64_t)blockIdx.x * hidden;
  const int tid = (int)threadIdx.x;
  float ss = 0.0f;
  for (int64_t i = tid; i < hidden; i += 256) {
    const float v = row[i];
    ss += v * v;
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  const float tot = (red[0] + red[1]) + (red[2] + red[3]);
  const float inv = 1.0f / sqrtf(tot / (float)hidden + eps);
  for (int64_t i = tid; i < hidden; i += 256) orow[i] = row[i] * inv * w[i];
}

__global__ __launch_bounds__(256) void swiglu_kernel(const float *__restrict__ gate, const float *__restrict__ up,
                                                     int64_t n, float *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float g = gate[i];
  const float sig = 1.0f / (1.0f + expf(-g));
  out[i] = (g * sig) * up[i];
}

hipError_t launch_rmsnorm(const float *x, int64_t rows, int64_t hidden, const float *weight, float eps, float *out,
                          hipStream_t s) {
  if (rows <= 0) return hipSuccess;
  // float4 rows of at most four float4s per thread of a full workgroup (the
  // weight is 16-byte aligned by validation); others take the loop kernel
  const bool aligned = ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) & 15u) == 0;
  if (hidden % 4 == 0 && hidden <= 4 * 4 * 1024 && aligned) {
    const int h4 = (int)(hidden / 4);
    const unsigned nt = h4 >= 1024 ? 1024u : (unsigned)(h4 + 63) / 64 * 64;
    const dim3 grid((unsigned)rows);
    if (h4 <= 1024) launch_timed(rmsnorm4_kernel<1>, grid, dim3(nt), 0u, s, x, h4, weight, eps, out);
    else if (h4 <= 2048) launch_timed(rmsnorm4_kernel<2>, grid, dim3(nt), 0u, s, x, h4, weight, eps, out);
    else launch_timed(rmsnorm4_kernel<4>, grid, dim3(nt), 0u, s, x, h4, weight, eps, out);
    return hipGetLastError();
  }
  launch_timed(rmsnorm_kernel, dim3((unsigned)rows), dim3(256), 0u, s, x, hidden, weight, eps, out);
  return hipGetLastError();
}

hipError_t launch_swiglu(const float *gate, const float *up, int64_t n, float *out, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  launch_timed(swiglu_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0u, s, gate, up, n, out);
  return hipGetLastError();
}

}  // namespace okq
