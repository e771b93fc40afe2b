// Column sums of a row-major matrix, accumulated in fp32 in a fixed order: bias gradients, and the rows of partial sums that a
// norm's backward leaves.
//
// A read of the matrix and little else: latency, not bytes, for the sizes of a training step. A workgroup of 16 waves takes 64
// columns, 8 lanes a row of 16-byte loads, 128 rows at once; rows meet by shuffles in a wave, then in LDS. Up to kColsumRows rows
// are one launch; more are split over workgroups whose fp32 sums a second launch adds. Against the general reduction (a clear
// of its counters and a kernel), us: bf16 2048 x 768 / 2304 / 3072 12.4 / 18.4 / 16.8 -> 4.8 / 4.9 / 4.9, 8192 x 3072 24.7 -> 13.6;
// fp32 512 x 768 / 4096 7.9 / 10.2 -> 3.7 / 3.8.
#pragma once
#include "sxe_common.h"

namespace sxe {

constexpr int kColsumRows = 2048;

struct ColsumArgs {  // blockIdx.z picks the matrix
  const void* in[2];
  void* out[2];
  int64_t R, N, ld, rows;  // rows of a split
  bool add[2];             // fp32 out: add to what is there
};

template <DT T, DT O, bool VEC>
__global__ void __launch_bounds__(1024) colsum_kernel(ColsumArgs a) {
  using S = typename dt_traits<T>::storage;
  __shared__ float red[16][64];
  const int c8 = (threadIdx.x & 7) * 8, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t col = (int64_t)blockIdx.x * 64 + c8, end = min(a.R, (blockIdx.y + 1) * a.rows);
  const S* in = static_cast<const S*>(a.in[blockIdx.z]);
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (col < a.N) {
    auto row = [&](int64_t r, float (&v)[8]) {
      const S* p = in + r * a.ld + col;
      if constexpr (VEC) {
        load8<T>(p, v);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = col + j < a.N ? to_f32<T>(p[j]) : 0.f;
      }
    };
    int64_t r = blockIdx.y * a.rows + (threadIdx.x >> 3);
    for (; r + 3 * 128 < end; r += 4 * 128) {
      float v[4][8];
#pragma unroll
      for (int u = 0; u < 4; ++u) row(r + u * 128, v[u]);
#pragma unroll
      for (int j = 0; j < 8; ++j) s[j] += (v[0][j] + v[1][j]) + (v[2][j] + v[3][j]);
    }
    for (; r < end; r += 128) {
      float v[8];
      row(r, v);
#pragma unroll
      for (int j = 0; j < 8; ++j) s[j] += v[j];
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    s[j] += __shfl_xor(s[j], 8, 64);
    s[j] += __shfl_xor(s[j], 16, 64);
    s[j] += __shfl_xor(s[j], 32, 64);
    if (lane < 8) red[wave][c8 + j] = s[j];
  }
  __syncthreads();
  const int64_t n = (int64_t)blockIdx.x * 64 + threadIdx.x;
  if (threadIdx.x < 64 && n < a.N) {
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < 16; ++w) t += red[w][threadIdx.x];
    auto* out = static_cast<typename dt_traits<O>::storage*>(a.out[blockIdx.z]) + (int64_t)blockIdx.y * a.N + n;
    if constexpr (O == DT::F32)
      if (a.add[blockIdx.z]) t += *out;
    *out = from_f32<O>(t);
  }
}

template <DT T, DT O>
void colsum_launch(const ColsumArgs& a, int splits, int mats) {
  const int64_t size = sizeof(typename dt_traits<T>::storage);
  bool vec = a.N % 8 == 0 && a.ld * size % 16 == 0;
  for (int i = 0; i < mats; ++i) vec = vec && reinterpret_cast<uintptr_t>(a.in[i]) % 16 == 0;
  const dim3 grid((unsigned)((a.N + 63) / 64), splits, mats);
  auto kern = vec ? colsum_kernel<T, O, true> : colsum_kernel<T, O, false>;
  hipLaunchKernelGGL(kern, grid, dim3(1024), 0, cur_stream(), a);
  SXE_LAUNCH_CHECK();
}

// one or two matrices of R > 0 rows and N > 0 columns, row stride ld; out: N elements of O each, where `add` (fp32 only) added to
template <DT T, DT O>
void colsum(const void* const (&in)[2], void* const (&out)[2], int64_t R, int64_t N, int64_t ld, int mats, const at::TensorOptions& opt,
            bool add0 = false, bool add1 = false) {
  SXE_CHECK(N <= 64ll * 0x7fffffff, "column sum: columns");
  if (R <= kColsumRows) {
    colsum_launch<T, O>({{in[0], in[1]}, {out[0], out[1]}, R, N, ld, R, {add0, add1}}, 1, mats);
    return;
  }
  const int64_t splits = std::min<int64_t>((R + 1023) / 1024, 256), rows = (R + splits - 1) / splits;
  auto part = at::empty({mats, splits, N}, opt.dtype(at::kFloat));
  float* p = part.data_ptr<float>();
  colsum_launch<T, DT::F32>({{in[0], in[1]}, {p, p + splits * N}, R, N, ld, rows, {false, false}}, (int)splits, mats);
  colsum_launch<DT::F32, O>({{p, p + splits * N}, {out[0], out[1]}, splits, N, N, splits, {add0, add1}}, 1, mats);
}

}  // namespace sxe
