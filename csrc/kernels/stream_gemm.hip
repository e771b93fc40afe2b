// Weight-streaming GEMM for batched decode on gfx950: y[M, N] = x[M, K] . W[N, K]^T (+ bias), M <= 32, bf16 or row-scaled
// e4m3 weights, fp32 accumulation; with GLU, W = [gate | up] and y[M, N / 2] = silu(gate) * up.
//
// Reference: inference/v2/kernels/core_ops/cuda_linear (FP6-LLM GEMM for small batches) and core_ops/gated_activations.
//
// What bounds it: reading W once -- and the rate at which a CU takes operand loads. In the matrix core's order neighbouring
// lanes hold different rows, and a load in that order takes ~64 cycles for its 1 KB (16 bytes a cycle and CU, measured): from
// 8 rows of x on it, not the memory, is what a kernel waits for that reads both operands that way (skinny_gemm.hip, built for
// M <= 4 with its prologues). Here the four lanes of a quad read 64 contiguous bytes of one row, four loads give them four rows,
// and a 4 x 4 exchange inside the quad (two DPP selects a register) leaves every lane with its own row.
// A workgroup takes NT tiles of 16 columns, its eight waves share K in interleaved pieces; the weight is the A operand, so a
// lane ends with 4 consecutive columns of a row. The waves' sums meet in LDS. Rates: the rules in ops/linear.py.
#include "sxe_common.h"
#include <torch/library.h>
#include <type_traits>

namespace sxe {
namespace st {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int NW = 8;  // waves of a workgroup

struct Args {
  const unsigned short* x;
  int64_t ldx;
  const void* w;
  int64_t ldw;
  const float* scale;          // fp8: of a row of w
  const unsigned short* bias;  // or null
  unsigned short* y;
  int M, N, K;
};

__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// 8 e4m3 bytes -> bf16, exact, two an instruction (at a scale of 1). By way of fp32, three for two, it took 28672 x 4096, 8 rows, gated
// 28.6 us, now 26.3, 32000 x 4096 28.8 / 26.5, 4096 x 4096 7.6 / 7.5 (with loads past the caches)
__device__ __forceinline__ u32x4 widen(unsigned lo, unsigned hi) {
  u32x4 r;
  r[0] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.f, false));
  r[1] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.f, true));
  r[2] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.f, false));
  r[3] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.f, true));
  return r;
}

// r[u] of quad lane j (row u's chunk j) -> r[c] = chunk c of row j
template <int CTRL>
__device__ __forceinline__ unsigned quad(unsigned x) { return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xf, 0xf, true); }
__device__ __forceinline__ void exchange(u32x4 (&r)[4], bool odd1, bool odd2) {
#pragma unroll
  for (int d = 0; d < 4; ++d) {
#pragma unroll
    for (int p = 0; p < 4; p += 2) {
      const unsigned a = r[p][d], b = r[p + 1][d], ax = quad<0xB1>(a), bx = quad<0xB1>(b);
      r[p][d] = odd1 ? bx : a;
      r[p + 1][d] = odd1 ? b : ax;
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const unsigned a = r[p][d], b = r[p + 2][d], ax = quad<0x4E>(a), bx = quad<0x4E>(b);
      r[p][d] = odd2 ? bx : a;
      r[p + 2][d] = odd2 ? b : ax;
    }
  }
}

// A wave's operands of one piece of K: 256 bytes of every row of W (128 columns of bf16, 256 of e4m3) and the same columns of x.
// After the exchange lane (row, g) holds chunk 4 g + c of 16 bytes of its row in register c.
template <bool FP8, int MB, int NT, bool ONCE>
struct Piece {
  static constexpr int PIECE = FP8 ? 256 : 128, XL = FP8 ? 2 : 1;
  u32x4 w[NT][4], x[MB][XL][4];
  // wr, xr: the rows 4 (row / 4) + u of this lane's quad, at chunk 4 g + j
  __device__ __forceinline__ void load(const char* const (&wr)[NT], int64_t ldw, const unsigned short* const (&xr)[MB][4], int k0, int K,
                                       int c) {
    const int kw = k0 + c * (FP8 ? 16 : 8);  // K is a multiple of 8 (16), so a lane's vector is in or out
    const bool win = kw < K;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        w[t][u] = u32x4{0u, 0u, 0u, 0u};
        const auto* p = reinterpret_cast<const u32x4*>(wr[t] + u * ldw + (int64_t)kw * (FP8 ? 1 : 2));
        if (win) w[t][u] = ONCE ? __builtin_nontemporal_load(p) : *p;
      }
#pragma unroll
    for (int h = 0; h < XL; ++h) {
      const int kx = k0 + 8 * (FP8 ? 8 * (c >> 2) + 4 * h + (c & 3) : c);
      const bool xin = kx < K;
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          x[m][h][u] = u32x4{0u, 0u, 0u, 0u};
          if (xin) x[m][h][u] = *reinterpret_cast<const u32x4*>(xr[m][u] + kx);
        }
    }
  }
  __device__ __forceinline__ void multiply(f32x4 (&acc)[MB][NT], bool odd1, bool odd2) {
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int h = 0; h < XL; ++h) exchange(x[m][h], odd1, odd2);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      exchange(w[t], odd1, odd2);
#pragma unroll
      for (int f = 0; f < 4 * XL; ++f) {
        u32x4 a;
        if constexpr (FP8) a = widen(w[t][f >> 1][2 * (f & 1)], w[t][f >> 1][2 * (f & 1) + 1]);
        else a = w[t][f];
#pragma unroll
        for (int m = 0; m < MB; ++m) acc[m][t] = mfma16(a, x[m][f >> 2][f & 3], acc[m][t]);
      }
    }
  }
};

template <bool FP8, int MB, int NT, bool GLU, bool ONCE>
__global__ void __launch_bounds__(64 * NW, 2) stream_gemm_kernel(Args a) {
  __shared__ f32x4 red[NW][NT][64];
  constexpr int OT = GLU ? NT / 2 : NT;  // tiles of output columns
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16 * OT, half = a.N / 2;
  const int j = lane & 3, quad0 = l16 & 12, c = 4 * g + j;
  // tiles start inside W (N a multiple of 4: a quad's rows all do or none); what lies past the end repeats the last rows
  const char* wr[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int n = (GLU ? n0 + 16 * (t % OT) + (t / OT) * half : n0 + 16 * t) + quad0;
    wr[t] = static_cast<const char*>(a.w) + (int64_t)min(n, a.N - 4) * a.ldw * (FP8 ? 1 : 2);
  }
  const int64_t ldw = a.ldw * (FP8 ? 1 : 2);
  const unsigned short* xr[MB][4];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int u = 0; u < 4; ++u) xr[m][u] = a.x + (int64_t)min(16 * m + quad0 + u, a.M - 1) * a.ldx;
  const bool odd1 = j & 1, odd2 = j & 2;
  f32x4 acc[MB][NT];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  // (the next piece in flight behind this one's products halves the workgroups on a CU and gains nothing)
  using P = Piece<FP8, MB, NT, ONCE>;
  for (int k0 = wave * P::PIECE; k0 < a.K; k0 += NW * P::PIECE) {
    P p;
    p.load(wr, ldw, xr, k0, a.K, c);
    p.multiply(acc, odd1, odd2);
  }
  // lane: columns 4 g .. + 3 of row l16 of every tile
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    if (16 * m >= a.M) break;
    if (m) __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; ++t) red[wave][t][lane] = acc[m][t];
    __syncthreads();
    for (int i = threadIdx.x; i < OT * 64; i += 64 * NW) {
      const int t = i >> 6, ln = i & 63, row = 16 * m + (ln & 15), n = n0 + 16 * t + 4 * (ln >> 4);
      auto sum = [&](int tile, int col) {
        f32x4 s = red[0][tile][ln];
#pragma unroll
        for (int v = 1; v < NW; ++v) s += red[v][tile][ln];
        if (FP8) {
#pragma unroll
          for (int q = 0; q < 4; ++q) s[q] *= a.scale[min(col + q, a.N - 1)];
        }
        if (a.bias != nullptr) {
#pragma unroll
          for (int q = 0; q < 4; ++q) s[q] += bf16_to_f32(a.bias[min(col + q, a.N - 1)]);
        }
        return s;
      };
      f32x4 v = sum(t, n);
      const int cols = GLU ? half : a.N;
      if constexpr (GLU) {
        const f32x4 up = sum(t + OT, n + half);
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = v[q] / (1.f + expf(-v[q])) * up[q];
      }
      if (row >= a.M) continue;
      unsigned short* yp = a.y + (int64_t)row * cols + n;
      if (n + 4 <= cols && cols % 4 == 0) {
        u16x4 o;
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = f32_to_bf16(v[q]);
        *reinterpret_cast<u16x4*>(yp) = o;
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (n + q < cols) yp[q] = f32_to_bf16(v[q]);
      }
    }
  }
}

}  // namespace st

// x [M, K] bf16, w [N, K] bf16, or e4m3 bytes with wscale fp32 [N]; bias bf16 [N] or None; glu: w = gate | up
at::Tensor stream_gemm(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& wscale,
                       const c10::optional<at::Tensor>& bias, bool glu) {
  check_beside(x, {w, wscale, bias});
  const bool fp8 = wscale.has_value() && wscale->defined();
  SXE_CHECK(x.scalar_type() == at::kBFloat16 && x.dim() == 2 && x.stride(1) == 1 && w.is_cuda() && w.dim() == 2 && w.stride(1) == 1 &&
                x.size(1) == w.size(1) && (fp8 ? w.element_size() == 1 : w.scalar_type() == at::kBFloat16),
            "stream_gemm: bf16 x [M, K], w [N, K] bf16 or e4m3 bytes");
  const int64_t M = x.size(0), N = w.size(0), K = x.size(1), unit = fp8 ? 16 : 8;
  SXE_CHECK(M >= 1 && M <= 32 && N > 0 && K > 0 && N < (1ll << 31) && K < (1ll << 31), "stream_gemm: 1 <= M <= 32");
  SXE_CHECK(K % unit == 0 && w.stride(0) % unit == 0 && x.stride(0) % 8 == 0 && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
                reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0, "stream_gemm: K and the rows must allow 16-byte loads");
  SXE_CHECK(N % 4 == 0, "stream_gemm: N a multiple of 4");
  SXE_CHECK(!glu || N % 32 == 0, "stream_gemm: gate and up of a multiple of 16 columns");
  st::Args a{};
  if (fp8) {
    SXE_CHECK(wscale->scalar_type() == at::kFloat && wscale->is_contiguous() && wscale->numel() == N, "stream_gemm: wscale fp32 [N]");
    a.scale = wscale->data_ptr<float>();
  }
  if (bias.has_value() && bias->defined()) {
    SXE_CHECK(bias->scalar_type() == at::kBFloat16 && bias->is_contiguous() && bias->numel() == N, "stream_gemm: bias bf16 [N]");
    a.bias = reinterpret_cast<const unsigned short*>(bias->data_ptr());
  }
  c10::DeviceGuard gd(x.device());
  auto y = at::empty({M, glu ? N / 2 : N}, x.options());
  a.x = reinterpret_cast<const unsigned short*>(x.data_ptr());
  a.ldx = x.stride(0);
  a.w = w.data_ptr();
  a.ldw = w.stride(0);
  a.y = reinterpret_cast<unsigned short*>(y.data_ptr());
  a.M = M;
  a.N = N;
  a.K = K;
  // tiles a workgroup: more of them for fewer reads of x, fewer for more workgroups. 28672 x 4096, us at 1 / 2 / 4 tiles: bf16,
  // 16 rows 47 / 50 / 47, 32 rows 57 / 53 / 53; e4m3, 8 rows 32 / 29 / 35; 4096 x 4096: bf16 9.7 / 12.9 / 16, e4m3 7.3 / 8.5 / 12.4
  const int64_t all = (N + 15) / 16;
  const int nt = glu ? (!fp8 && N % 64 == 0 ? 4 : 2) : all >= 384 && (fp8 || M > 16) ? 2 : 1;
  const dim3 grid((all + nt - 1) / nt);
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(64 * st::NW), 0, cur_stream(), a); };
  auto rows = [&](auto mb, auto nontemporal) {
    constexpr int MB = decltype(mb)::value;
    constexpr bool ONCE = decltype(nontemporal)::value;
    if (fp8) {
      if (glu) go(st::stream_gemm_kernel<true, MB, 2, true, ONCE>);
      else nt == 2 ? go(st::stream_gemm_kernel<true, MB, 2, false, ONCE>) : go(st::stream_gemm_kernel<true, MB, 1, false, ONCE>);
    } else if (glu) {
      nt == 4 ? go(st::stream_gemm_kernel<false, MB, 4, true, ONCE>) : go(st::stream_gemm_kernel<false, MB, 2, true, ONCE>);
    } else {
      nt == 2 ? go(st::stream_gemm_kernel<false, MB, 2, false, ONCE>) : go(st::stream_gemm_kernel<false, MB, 1, false, ONCE>);
    }
  };
  auto blocks = [&](auto nontemporal) {
    if (M <= 16) rows(std::integral_constant<int, 1>{}, nontemporal);
    else rows(std::integral_constant<int, 2>{}, nontemporal);
  };
  if (read_once(N * K * (fp8 ? 1 : 2))) blocks(std::true_type{});
  else blocks(std::false_type{});
  SXE_LAUNCH_CHECK();
  return y;
}

}  // namespace sxe

TORCH_LIBRARY_FRAGMENT(sxe, m) {
  m.def("stream_gemm(Tensor x, Tensor w, Tensor? wscale, Tensor? bias, bool glu) -> Tensor");
}
TORCH_LIBRARY_IMPL(sxe, CUDA, m) { m.impl("stream_gemm", &sxe::stream_gemm); }
