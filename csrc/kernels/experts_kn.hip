// Routed SwiGLU experts with weights as the training modules hold them, [E, K, N] (y = x @ w), for the few rows an expert
// gets at decode (gfx950): the weights are read once, the expert lists stay on the device (experts.hip), so a step needs no
// host synchronisation and can be captured.
//
// Reference: inference/v2/kernels/cutlass_ops/moe_gemm and ragged_ops/moe_gather (expert products and the weighted gather).
//
// What bounds it: reading the experts' weights. A workgroup takes 128 columns of one expert, its eight waves share K; a wave
// reads 32 rows x 256 bytes at a time (8 x 16 bytes a lane). The matrix core wants 8 consecutive k of a column in a lane, a
// row-major load has 8 columns of a row: a lane loads 8 x 8 values and swaps them in registers (32 v_perm a block, no LDS).
// Column i of a lane's octet goes to product i, so the eight products of a block have columns 8 l + i. Up to MB x 16 rows
// share a pass over the weights.
//  * gate | up: 64 gate columns and the matching 64 up columns in one workgroup, SwiGLU in its epilogue;
//  * down: K also split over the grid while there are fewer than two workgroups a CU (one token: 64 otherwise); fp32
//    partials, summed with the routing weights over a token's choices by the combine kernel.
// Mixtral-8x7B layer (8 experts of 4096 x 14336, top 2), 16 tokens, MI355X: gate | up 362 us and down 163 us, 5.2 and 5.8 TB/s;
// the loop over the experts it replaces took 1051 us with its routing. Other sizes: the dispatch in ops/moe.py.
#include "sxe_common.h"
#include "sxe_mfma.h"
#include <torch/library.h>

namespace sxe {
namespace kn {
using mf::bf16x8;
using mf::u32x4;

constexpr int NW = 8, COLS = 128, LDP = COLS + 4;  // waves, columns of a workgroup, row of a wave's sums in LDS

struct Args {
  const unsigned short *x, *w;  // x [rows, ldx]; w [E, K, N]
  int64_t ldx;
  const int *offs, *active, *token;  // token: row -> row of x, or null
  unsigned short* h;            // gate | up: [R, N / 2]
  float* part;                  // down: [splits, R, N]
  int R, E, N, K, Tx, splits;
};

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// grid (column tiles, experts that may have rows, K splits)
template <int MB, bool GATE, bool ONCE>
__global__ void __launch_bounds__(64 * NW, MB == 1 ? 4 : MB == 2 ? 3 : 2) expert_kn_kernel(Args a) {
  extern __shared__ __attribute__((aligned(16))) float part[];  // [NW][16][LDP]
  if ((int)blockIdx.y >= a.active[0]) return;
  const int e = a.active[1 + blockIdx.y], lo = a.offs[e], hi = min(a.offs[e + 1], a.R);
  if (lo < 0 || lo >= hi) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * (GATE ? COLS / 2 : COLS);
  const int col = GATE ? n0 + 8 * (l16 & 7) + (l16 >> 3) * (a.N / 2) : n0 + 8 * l16;
  const unsigned short* w = a.w + ((int64_t)e * a.K + 8 * g) * a.N + col;
  // K in steps of 32: this workgroup's share, a multiple of 32
  const int steps = a.K / 32, s0 = (int64_t)steps * blockIdx.z / a.splits, s1 = (int64_t)steps * (blockIdx.z + 1) / a.splits;
  constexpr int U = 2;
  for (int r0 = lo; r0 < hi; r0 += 16 * MB) {
    const unsigned short* xr[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const int r = min(r0 + 16 * m + l16, hi - 1);
      xr[m] = a.x + (int64_t)(a.token != nullptr ? min(max(a.token[r], 0), a.Tx - 1) : r) * a.ldx + 8 * g;
    }
    f32x4 acc[MB][8];
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[m][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = s0 + wave * U; s < s1; s += NW * U) {
      u32x4 wf[U][8], xf[MB][U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = 32 * min(s + u, s1 - 1);  // past the share: read again, not used
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const auto* p = reinterpret_cast<const u32x4*>(w + (int64_t)(k + j) * a.N);
          wf[u][j] = ONCE ? __builtin_nontemporal_load(p) : *p;
        }
#pragma unroll
        for (int m = 0; m < MB; ++m) xf[m][u] = *reinterpret_cast<const u32x4*>(xr[m] + k);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (s + u >= s1) break;
#pragma unroll
        for (int d = 0; d < 4; ++d) {  // columns 2 d and 2 d + 1 of the octet
          u32x4 b0, b1;
#pragma unroll
          for (int p = 0; p < 4; ++p) {
            b0[p] = __builtin_amdgcn_perm(wf[u][2 * p + 1][d], wf[u][2 * p][d], 0x05040100u);
            b1[p] = __builtin_amdgcn_perm(wf[u][2 * p + 1][d], wf[u][2 * p][d], 0x07060302u);
          }
#pragma unroll
          for (int m = 0; m < MB; ++m) {
            const bf16x8 xa = __builtin_bit_cast(bf16x8, xf[m][u]);
            acc[m][2 * d] = mfma16(xa, __builtin_bit_cast(bf16x8, b0), acc[m][2 * d]);
            acc[m][2 * d + 1] = mfma16(xa, __builtin_bit_cast(bf16x8, b1), acc[m][2 * d + 1]);
          }
        }
      }
    }
    // a wave's sums: row 4 g + q of the 16, column 8 l16 + i at 16 i + l16
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      if (r0 + 16 * m >= hi) break;
      __syncthreads();  // the previous sums are read
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) part[(wave * 16 + 4 * g + q) * LDP + 16 * i + l16] = acc[m][i][q];
      __syncthreads();
      auto sum = [&](int row, int at) {
        float s = 0.f;
#pragma unroll
        for (int v = 0; v < NW; ++v) s += part[(v * 16 + row) * LDP + at];
        return s;
      };
      constexpr int OUT = GATE ? COLS / 2 : COLS;
      for (int i = threadIdx.x; i < 16 * OUT; i += 64 * NW) {
        const int row = i / OUT, c = i % OUT, r = r0 + 16 * m + row, at = 16 * (c & 7) + (c >> 3);
        if (r >= hi) continue;
        if constexpr (GATE) {
          const float gt = sum(row, at), up = sum(row, at + 8);
          a.h[(int64_t)r * (a.N / 2) + n0 + c] = f32_to_bf16(gt / (1.f + expf(-gt)) * up);
        } else {
          a.part[((int64_t)blockIdx.z * a.R + r) * a.N + n0 + c] = sum(row, at);
        }
      }
    }
  }
}

// out[t] = sum_j weight[t, j] * sum_s part[s][slots[t, j]]; four columns a thread
__global__ void __launch_bounds__(256) combine_kernel(const float* __restrict__ part, const int* __restrict__ slots,
                                                      const float* __restrict__ weight, unsigned short* __restrict__ out, int T, int k,
                                                      int R, int N, int splits) {
  const int64_t i = (blockIdx.x * 256ll + threadIdx.x) * 4;
  if (i >= (int64_t)T * N) return;
  const int t = i / N, c = i - (int64_t)t * N;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int j = 0; j < k; ++j) {
    const int r = min(max(slots[t * k + j], 0), R - 1);
    f32x4 y = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < splits; ++s) y += *reinterpret_cast<const f32x4*>(part + ((int64_t)s * R + r) * N + c);
    acc += weight[t * k + j] * y;
  }
  u16x4 o;
#pragma unroll
  for (int q = 0; q < 4; ++q) o[q] = f32_to_bf16(acc[q]);
  *reinterpret_cast<u16x4*>(out + i) = o;
}

inline bool aligned16(const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

template <bool GATE>
void launch(const Args& a, hipStream_t stream) {
  const dim3 grid(a.N / COLS, std::min(a.E, a.R), a.splits);
  const size_t lds = sizeof(float) * NW * 16 * LDP;
  auto with = [&](auto mb, auto once) {
    constexpr auto kern = &expert_kn_kernel<decltype(mb)::value, GATE, decltype(once)::value>;
    allow_lds<kern>((int)lds);
    hipLaunchKernelGGL(kern, grid, dim3(64 * NW), lds, stream, a);
  };
  auto go = [&](auto mb) { read_once(2ll * a.E * a.N * a.K) ? with(mb, std::true_type{}) : with(mb, std::false_type{}); };
  // blocks of 16 rows that share a pass: twice the mean, so that an uneven routing seldom takes a second pass
  if (a.R <= 8 * a.E) go(std::integral_constant<int, 1>{});
  else if (a.R <= 16 * a.E) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 4>{});
  SXE_LAUNCH_CHECK();
}

Args args(const at::Tensor& x, const at::Tensor& w, const at::Tensor& offs, const at::Tensor& active, int64_t R) {
  SXE_CHECK_CUDA(x);
  SXE_CHECK(x.dim() == 2 && x.stride(1) == 1 && x.stride(0) % 8 == 0 && w.dim() == 3 && w.is_contiguous() && w.is_cuda() &&
                w.size(1) == x.size(1) && x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16 && aligned16(x) &&
                aligned16(w), "expert products: bf16 x [T, K], w [E, K, N], 16-byte aligned rows");
  const int64_t E = w.size(0), K = w.size(1), N = w.size(2);
  SXE_CHECK(K % 32 == 0 && N % COLS == 0 && K > 0 && N > 0 && E > 0 && R < (1ll << 31) && K < (1ll << 31) && N < (1ll << 31),
            "expert products: K a multiple of 32, N of 128");
  for (const auto* t : {&offs, &active})
    SXE_CHECK(t->is_cuda() && t->is_contiguous() && t->scalar_type() == at::kInt && t->numel() == E + 1, "expert lists int32 [E + 1]");
  Args a{};
  a.x = static_cast<const unsigned short*>(x.data_ptr());
  a.w = static_cast<const unsigned short*>(w.data_ptr());
  a.ldx = x.stride(0);
  a.offs = offs.data_ptr<int>();
  a.active = active.data_ptr<int>();
  a.R = R;
  a.E = E;
  a.N = N;
  a.K = K;
  a.Tx = x.size(0);
  a.splits = 1;
  return a;
}

}  // namespace kn

// x [T, K], w [E, K, 2 I] (gate | up), token int32 [R] -> silu(gate) * up [R, I] of the expert-sorted rows
at::Tensor expert_swiglu_kn(const at::Tensor& x, const at::Tensor& w, const at::Tensor& offs, const at::Tensor& active,
                            const at::Tensor& token) {
  const int64_t R = token.numel();
  kn::Args a = kn::args(x, w, offs, active, R);
  SXE_CHECK(token.is_cuda() && token.is_contiguous() && token.scalar_type() == at::kInt, "expert_swiglu_kn: token int32 [R]");
  auto h = at::empty({R, w.size(2) / 2}, x.options());
  if (R == 0) return h;
  c10::DeviceGuard g(x.device());
  a.token = token.data_ptr<int>();
  a.h = static_cast<unsigned short*>(h.data_ptr());
  kn::launch<true>(a, cur_stream());
  return h;
}

// h [R, K] expert-sorted rows, w [E, K, N], slots int32 [T, k] (row of each choice), weight fp32 [T, k] -> [T, N]
at::Tensor expert_down_kn(const at::Tensor& h, const at::Tensor& w, const at::Tensor& offs, const at::Tensor& active,
                          const at::Tensor& slots, const at::Tensor& weight) {
  kn::Args a = kn::args(h, w, offs, active, h.size(0));
  SXE_CHECK(slots.is_cuda() && slots.is_contiguous() && slots.scalar_type() == at::kInt && slots.dim() == 2 && slots.numel() == h.size(0) &&
                weight.is_cuda() && weight.is_contiguous() && weight.scalar_type() == at::kFloat && weight.sizes() == slots.sizes(),
            "expert_down_kn: slots int32, weight fp32 [T, k], a row of h for each");
  auto out = at::empty({slots.size(0), w.size(2)}, h.options());
  if (a.R == 0) return out.zero_();
  c10::DeviceGuard g(h.device());
  const int64_t wgs = (int64_t)(a.N / kn::COLS) * std::min(a.E, a.R);
  a.splits = std::max<int64_t>(1, std::min<int64_t>((2 * kNumCUs + wgs - 1) / wgs, a.K / 512));
  auto part = at::empty({a.splits, a.R, a.N}, h.options().dtype(at::kFloat));
  a.part = part.data_ptr<float>();
  kn::launch<false>(a, cur_stream());
  const int64_t n4 = out.numel() / 4;
  hipLaunchKernelGGL(kn::combine_kernel, dim3((n4 + 255) / 256), dim3(256), 0, cur_stream(), a.part, slots.data_ptr<int>(),
                     weight.data_ptr<float>(), static_cast<unsigned short*>(out.data_ptr()), (int)slots.size(0), (int)slots.size(1), a.R,
                     a.N, a.splits);
  SXE_LAUNCH_CHECK();
  return out;
}

}  // namespace sxe

TORCH_LIBRARY_FRAGMENT(sxe, m) {
  m.def("expert_swiglu_kn(Tensor x, Tensor w, Tensor offs, Tensor active, Tensor token) -> Tensor");
  m.def("expert_down_kn(Tensor h, Tensor w, Tensor offs, Tensor active, Tensor slots, Tensor weight) -> Tensor");
}
TORCH_LIBRARY_IMPL(sxe, CUDA, m) {
  m.impl("expert_swiglu_kn", &sxe::expert_swiglu_kn);
  m.impl("expert_down_kn", &sxe::expert_down_kn);
}
