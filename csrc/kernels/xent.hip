// Softmax cross-entropy over large vocabularies for gfx950 (forward, backward, and a fused
// forward+backward that overwrites the logits with their gradient).
//
// The reference computes the LM loss with torch (and, for sequence parallelism, a vocab/sequence
// sharded variant: deepspeed/sequence/cross_entropy.py:11-60; ALST's TiledLoss,
// runtime/sequence_parallel/ulysses_sp.py:915). Here one workgroup owns one token row
// (V up to ~256K): a single 16-byte-vectorised sweep computes the running (max, sum-exp) per lane
// (online softmax), the 4 waves merge through LDS, and the backward sweep re-reads the row
// (Infinity-Cache resident at these row sizes) and writes bf16 gradients IN PLACE, so the
// [tokens, vocab] logits tensor is never duplicated (4 GiB at 16K tokens x 128K vocab).
// The sweeps are memory-bound at 16 bytes a load, so a row that starts off a 16-byte boundary (an odd vocabulary) is swept from its
// first boundary on, the few elements around that by single lanes: 2048 x 50257 of bf16, us, element by element / so: loss
// 116 / 42, gradient 153 / 86; 256 rows 89 / 20 and 86 / 22.
#include "sxe_common.h"
#include <torch/library.h>
#include <type_traits>

namespace sxe {

constexpr float kFltMax = 3.402823466e38f;
// Running (max, sum) and another one. The products are fused as written, so that a loss does not depend on what surrounds the merge:
// a sweep rounds what it adds (LANES: what it has) before the sum.
template <bool LANES>
__device__ __forceinline__ void ms_merge(float& m, float& s, float m2, float s2) {
  // against a finite reference: nothing but masked logits so far adds nothing (a branch on it costs 10 % where rows are few)
  const float mn = fmaxf(m, m2), ref = fmaxf(mn, -kFltMax), e = __expf(m - ref), e2 = __expf(m2 - ref);
  s = LANES ? __builtin_fmaf(s2, e2, s * e) : __builtin_fmaf(s, e, s2 * e2);
  m = mn;
}

// elements of a row before its first 16-byte boundary: rows of an odd vocabulary start anywhere
template <typename S>
__device__ __forceinline__ int row_head(const S* row, int V) {
  return min(V, (int)((0 - reinterpret_cast<uintptr_t>(row) / sizeof(S)) & (16 / sizeof(S) - 1)));
}
// How a row is swept. ELEMENTS: short rows off 16 bytes, or gradients that start otherwise than their logits; WHOLE: every row is
// whole 16-byte vectors; BODY: what lies before and behind the aligned body (< 8 elements each) by single lanes.
enum Sweep { ELEMENTS, WHOLE, BODY };
// 8192 rows, us, loss + gradient by ELEMENTS / BODY: 129 columns 15.7 / 18.0, 385 17.7 / 18.4, 513 18.8 / 18.6, 1001 24.8 / 21.7
constexpr int kBodyMin = 512;
inline Sweep sweep_of(const at::Tensor& logits, int V) {
  if (V % 8 == 0 && reinterpret_cast<uintptr_t>(logits.data_ptr()) % 16 == 0) return WHOLE;
  return V >= kBodyMin ? BODY : ELEMENTS;
}
template <typename F>
void with_sweep(Sweep sw, F f) {
  if (sw == WHOLE) f(std::integral_constant<Sweep, WHOLE>{});
  else if (sw == BODY) f(std::integral_constant<Sweep, BODY>{});
  else f(std::integral_constant<Sweep, ELEMENTS>{});
}
// f8(first of 8 aligned elements), f1(element)
template <Sweep SW, typename F8, typename F1>
__device__ __forceinline__ void for_row(int V, int head, F8 f8, F1 f1) {
  if constexpr (SW == ELEMENTS) {
    for (int c = threadIdx.x; c < V; c += blockDim.x) f1(c);
    return;
  }
  if constexpr (SW == WHOLE) {
    for (int c = threadIdx.x * 8; c < V; c += blockDim.x * 8) f8(c);
    return;
  }
  const int body = (V - head) & ~7;
  for (int c = head + threadIdx.x * 8; c < head + body; c += blockDim.x * 8) f8(c);
  if ((int)threadIdx.x < head) f1(threadIdx.x);
  const int c = head + body + threadIdx.x;
  if (c < V) f1(c);
}

template <DT T, Sweep SW>
__device__ __forceinline__ float row_lse(const typename dt_traits<T>::storage* __restrict__ row, int V, int head, float* red) {
  float m = -INFINITY, s = 0.f;
  for_row<SW>(V, head, [&](int c) {
    float v[8];
    load8<T>(row + c, v);
    float lm = v[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) lm = fmaxf(lm, v[j]);
    float ls = 0.f;
    const float ref = fmaxf(lm, -kFltMax);
#pragma unroll
    for (int j = 0; j < 8; ++j) ls += __expf(v[j] - ref);
    ms_merge<false>(m, s, lm, ls);
  }, [&](int c) { ms_merge<false>(m, s, to_f32<T>(row[c]), 1.f); });
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    float m2 = __shfl_xor(m, o, 64), s2 = __shfl_xor(s, o, 64);
    ms_merge<true>(m, s, m2, s2);
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) { red[2 * w] = m; red[2 * w + 1] = s; }
  __syncthreads();
  float M = red[0], Ssum = red[1];
  for (int i = 1; i < (int)(blockDim.x >> 6); ++i) ms_merge<true>(M, Ssum, red[2 * i], red[2 * i + 1]);
  __syncthreads();
  return M + __logf(Ssum);
}

// mode: 0 = forward only; 1 = forward + in-place gradient with grad = scale * (softmax - onehot)
template <DT T, Sweep SW>
__global__ void __launch_bounds__(256) xent_kernel(typename dt_traits<T>::storage* __restrict__ logits, int64_t rows, int V,
                                                   const int64_t* __restrict__ target, int64_t ignore_index,
                                                   float* __restrict__ loss, float* __restrict__ lse_out, int mode,
                                                   const float* __restrict__ scale_t, float scale) {
  __shared__ float red[8];
  if (scale_t) scale *= *scale_t;
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    typename dt_traits<T>::storage* row = logits + r * V;
    const int64_t tgt = target[r];
    const bool ign = (tgt == ignore_index);
    const int head = SW == BODY ? row_head(row, V) : 0;
    const float lse = row_lse<T, SW>(row, V, head, red);
    if (threadIdx.x == 0) {
      const float xt = ign ? 0.f : to_f32<T>(row[tgt]);
      loss[r] = ign ? 0.f : (lse - xt);
      if (lse_out) lse_out[r] = lse;
    }
    __syncthreads();  // the target logit is read above before the gradient overwrites it
    if (mode == 1) {
      const float sc = ign ? 0.f : scale;
      for_row<SW>(V, head, [&](int c) {
        float v[8];
        load8<T>(row + c, v);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = sc * (__expf(v[j] - lse) - ((c + j) == tgt ? 1.f : 0.f));
        store8<T>(row + c, v);
      }, [&](int c) { row[c] = from_f32<T>(sc * (__expf(to_f32<T>(row[c]) - lse) - (c == tgt ? 1.f : 0.f))); });
    }
  }
}

// grad = dloss[r] * (softmax - onehot), written into grad_out (may alias logits).
template <DT T, Sweep SW>
__global__ void __launch_bounds__(256) xent_bwd_kernel(const typename dt_traits<T>::storage* __restrict__ logits,
                                                       typename dt_traits<T>::storage* __restrict__ grad, int64_t rows, int V,
                                                       const int64_t* __restrict__ target, int64_t ignore_index,
                                                       const float* __restrict__ lse, const float* __restrict__ dloss) {
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    const int64_t tgt = target[r];
    const float sc = (tgt == ignore_index) ? 0.f : dloss[r];
    const float l = lse[r];
    const typename dt_traits<T>::storage* in = logits + r * V;
    typename dt_traits<T>::storage* out = grad + r * V;
    auto one = [&](int c) { out[c] = from_f32<T>(sc * (__expf(to_f32<T>(in[c]) - l) - (c == tgt ? 1.f : 0.f))); };
    for_row<SW>(V, SW == BODY ? row_head(in, V) : 0, [&](int c) {
      float v[8];
      load8<T>(in + c, v);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = sc * (__expf(v[j] - l) - ((c + j) == tgt ? 1.f : 0.f));
      store8<T>(out + c, v);
    }, one);
  }
}

// Dual-layout LM-head gradient (bf16): g = sc[r] * (softmax - onehot) with sc = dloss * scale_a * scale_b
// (all device scalars; 0 on ignored rows), written IN PLACE over the logits (token-major, for the
// data-gradient GEMM) AND as g^T [V, rows] (vocab-major, so the weight-gradient GEMM dW = g^T h
// reads K-contiguous operands: hipBLASLt's TN layout, 12.1 vs 14.6 ms for transposes + TN at 16k
// tokens x 128256, profiles/r06/wgrad_variants_16k.log). Running in the backward, where the
// upstream scalar is known, it also replaces the forward's in-place gradient write and the
// backward's scaling pass: 16.8 GB of HBM traffic per 16k-token micro-step instead of 25.2.
// Geometry: one 1024-thread workgroup per 64-token x 256-column tile; thread t owns row t/16 and
// 16 columns from (t%16)*16 (two 16-byte vectors), stages the bf16 result in an LDS tile with a
// 258-element row stride (odd dword stride: the column-wise reads spread over the banks), then
// stores 16 tokens of one vocab row of g^T as two 16-byte vectors.
constexpr int XG_TR = 64, XG_TC = 256, XG_LD = XG_TC + 2;

__global__ void __launch_bounds__(1024) xent_grad_dual_kernel(unsigned short* __restrict__ logits,
                                                              unsigned short* __restrict__ gT, int64_t rows, int V,
                                                              const int64_t* __restrict__ target, int64_t ignore_index,
                                                              const float* __restrict__ lse, const float* __restrict__ s_a,
                                                              const float* __restrict__ s_b) {
  __shared__ __attribute__((aligned(16))) unsigned short tile[XG_TR * XG_LD];
  const int tiles_c = V / XG_TC;
  const int64_t tr = blockIdx.x / tiles_c;
  const int tc = (int)(blockIdx.x - tr * tiles_c);
  const int t = threadIdx.x, r = t >> 4, c0 = (t & 15) * 16;
  const int64_t row = tr * XG_TR + r;
  const int col = tc * XG_TC + c0;
  const int64_t tgt = target[row];
  const float sc = (tgt == ignore_index) ? 0.f : s_a[0] * (s_b ? s_b[0] : 1.f);
  const float l = lse[row];
  unsigned short* p = logits + row * V + col;
  const u16x8 a = *reinterpret_cast<const u16x8*>(p), b = *reinterpret_cast<const u16x8*>(p + 8);
  u16x8 oa, ob;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    oa[j] = f32_to_bf16(sc * (__expf(bf16_to_f32(a[j]) - l) - ((col + j) == tgt ? 1.f : 0.f)));
    ob[j] = f32_to_bf16(sc * (__expf(bf16_to_f32(b[j]) - l) - ((col + 8 + j) == tgt ? 1.f : 0.f)));
  }
  *reinterpret_cast<u16x8*>(p) = oa;
  *reinterpret_cast<u16x8*>(p + 8) = ob;
  unsigned* ld = reinterpret_cast<unsigned*>(&tile[r * XG_LD + c0]);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    ld[j] = (unsigned)oa[2 * j] | ((unsigned)oa[2 * j + 1] << 16);
    ld[4 + j] = (unsigned)ob[2 * j] | ((unsigned)ob[2 * j + 1] << 16);
  }
  __syncthreads();
  // transposed store: output row = tile column t/4, 16 tokens from (t%4)*16
  const int oc = t >> 2, r0 = (t & 3) * 16;
  u16x8 o0, o1;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    o0[j] = tile[(r0 + j) * XG_LD + oc];
    o1[j] = tile[(r0 + 8 + j) * XG_LD + oc];
  }
  unsigned short* d = gT + (int64_t)(tc * XG_TC + oc) * rows + tr * XG_TR + r0;
  *reinterpret_cast<u16x8*>(d) = o0;
  *reinterpret_cast<u16x8*>(d + 8) = o1;
}

// -> g^T [V, rows]; the logits are overwritten with g. rows % 64 == 0, V % 256 == 0, bf16.
at::Tensor xent_grad_dual(at::Tensor logits, at::Tensor target, at::Tensor lse, int64_t ignore_index, at::Tensor scale_a,
                          c10::optional<at::Tensor> scale_b) {
  SXE_CHECK_CUDA(logits);
  SXE_CHECK(logits.dim() == 2 && logits.is_contiguous() && logits.scalar_type() == at::kBFloat16,
            "xent_grad_dual: contiguous bf16 [rows, vocab] logits");
  SXE_CHECK(target.scalar_type() == at::kLong && target.numel() == logits.size(0) && target.is_contiguous(),
            "xent_grad_dual: target must be int64 [rows]");
  const int64_t rows = logits.size(0);
  const int V = (int)logits.size(1);
  SXE_CHECK(rows % XG_TR == 0 && V % XG_TC == 0, "xent_grad_dual: rows % 64 and vocab % 256 must be 0");
  SXE_CHECK(lse.scalar_type() == at::kFloat && lse.numel() == rows && lse.is_contiguous(), "xent_grad_dual: lse fp32 [rows]");
  SXE_CHECK(scale_a.scalar_type() == at::kFloat && scale_a.is_cuda() && scale_a.numel() == 1, "xent_grad_dual: scale_a fp32 [1]");
  const float* sb = nullptr;
  if (scale_b.has_value() && scale_b->defined()) {
    SXE_CHECK(scale_b->scalar_type() == at::kFloat && scale_b->is_cuda() && scale_b->numel() == 1,
              "xent_grad_dual: scale_b fp32 [1]");
    sb = scale_b->data_ptr<float>();
  }
  c10::DeviceGuard guard(logits.device());
  auto gT = at::empty({(int64_t)V, rows}, logits.options());
  const int64_t tiles = (rows / XG_TR) * (V / XG_TC);
  if (tiles == 0) return gT;
  SXE_CHECK(tiles < (1ll << 31), "xent_grad_dual: too many tiles");
  hipLaunchKernelGGL(xent_grad_dual_kernel, dim3((unsigned)tiles), dim3(1024), 0, cur_stream(),
                     reinterpret_cast<unsigned short*>(logits.data_ptr()), reinterpret_cast<unsigned short*>(gT.data_ptr()),
                     rows, V, target.data_ptr<int64_t>(), ignore_index, lse.data_ptr<float>(), scale_a.data_ptr<float>(), sb);
  SXE_LAUNCH_CHECK();
  return gT;
}

// ------------------------------------------------------------------------ vocabulary-major logits
// Logits as [V, ld] bf16 with a token per column: of an odd vocabulary the rows are whole 16-byte
// vectors only this way round (ld, the tokens rounded up, is a multiple of 64), so the head's three
// products run on aligned operands. A thread owns 8 columns and every 4th to 32nd row of its block's
// share, four in flight; both passes stream. 50257 rows, us, loss / gradient, a workgroup a row of
// token-major logits against this: 2048 tokens 34 / 89 against 47 / 94, 8192 145 / 340 against 165 /
// 310, 512 16 / 19 against 22 / 26; what the products gain is a multiple of that (see head_cross_entropy).
template <int LANES>  // of a row
struct ColBlock {
  static constexpr int COLS = 8 * LANES, ROWS = 256 / LANES;
};

template <int LANES>
__global__ void __launch_bounds__(256) xent_cols_part_kernel(const unsigned short* __restrict__ x, int64_t ld, int V, int rows_per,
                                                             float2* __restrict__ part) {
  constexpr int COLS = ColBlock<LANES>::COLS, ROWS = ColBlock<LANES>::ROWS;
  __shared__ float2 red[ROWS][COLS + 1];
  const int cx = threadIdx.x % LANES * 8, ry = threadIdx.x / LANES;
  const int64_t c = (int64_t)blockIdx.x * COLS + cx;
  const int r0 = blockIdx.y * rows_per, r1 = min(V, r0 + rows_per);
  float m[8], s[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    m[j] = -INFINITY;
    s[j] = 0.f;
  }
  if (c < ld) {
    int r = r0 + ry;
    for (; r + 3 * ROWS < r1; r += 4 * ROWS) {
      float v[4][8];
#pragma unroll
      for (int u = 0; u < 4; ++u) load8<DT::BF16>(x + (r + u * ROWS) * ld + c, v[u]);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float lm = fmaxf(fmaxf(v[0][j], v[1][j]), fmaxf(v[2][j], v[3][j])), ref = fmaxf(lm, -kFltMax);
        ms_merge<false>(m[j], s[j], lm, (__expf(v[0][j] - ref) + __expf(v[1][j] - ref)) + (__expf(v[2][j] - ref) + __expf(v[3][j] - ref)));
      }
    }
    for (; r < r1; r += ROWS) {
      float v[8];
      load8<DT::BF16>(x + r * ld + c, v);
#pragma unroll
      for (int j = 0; j < 8; ++j) ms_merge<false>(m[j], s[j], v[j], 1.f);
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) red[ry][cx + j] = float2{m[j], s[j]};
  __syncthreads();
  for (int i = threadIdx.x; i < COLS; i += 256) {
    const int64_t col = (int64_t)blockIdx.x * COLS + i;
    if (col >= ld) break;
    float2 a = red[0][i];
    for (int g = 1; g < ROWS; ++g) ms_merge<true>(a.x, a.y, red[g][i].x, red[g][i].y);
    part[blockIdx.y * ld + col] = a;
  }
}

// the shares' (max, sum) to loss and LSE: 16 tokens a block, 16 threads a token
__global__ void __launch_bounds__(256) xent_cols_loss_kernel(const unsigned short* __restrict__ x, int64_t ld, int64_t tokens, int shares,
                                                             const float2* __restrict__ part, const int64_t* __restrict__ target,
                                                             int64_t ignore_index, float* __restrict__ loss, float* __restrict__ lse) {
  __shared__ float2 red[16][17];
  const int cx = threadIdx.x & 15, ry = threadIdx.x >> 4;
  const int64_t t = (int64_t)blockIdx.x * 16 + cx;
  float2 a{-INFINITY, 0.f};
  if (t < tokens)
    for (int g = ry; g < shares; g += 16) {
      const float2 b = part[g * ld + t];
      ms_merge<true>(a.x, a.y, b.x, b.y);
    }
  red[ry][cx] = a;
  __syncthreads();
  if (ry != 0 || t >= tokens) return;
  for (int g = 1; g < 16; ++g) ms_merge<true>(a.x, a.y, red[g][cx].x, red[g][cx].y);
  const float l = a.x + __logf(a.y);
  const int64_t tgt = target[t];
  loss[t] = tgt == ignore_index ? 0.f : l - bf16_to_f32(x[tgt * ld + t]);
  lse[t] = l;
}

// dloss[t] * (softmax - onehot); columns behind the last token are zeros
template <int LANES>
__global__ void __launch_bounds__(256) xent_cols_bwd_kernel(const unsigned short* __restrict__ x, unsigned short* __restrict__ grad,
                                                            int64_t ld, int V, int64_t tokens, int rows_per,
                                                            const int64_t* __restrict__ target, int64_t ignore_index,
                                                            const float* __restrict__ lse, const float* __restrict__ dloss) {
  const int64_t c = (int64_t)blockIdx.x * ColBlock<LANES>::COLS + threadIdx.x % LANES * 8;
  if (c >= ld) return;
  float l[8], sc[8];
  int tgt[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const bool in = c + j < tokens;
    const int64_t t = in ? target[c + j] : ignore_index;
    tgt[j] = (int)t;
    sc[j] = t == ignore_index ? 0.f : dloss[c + j];
    l[j] = in ? lse[c + j] : 0.f;
  }
  const int r0 = blockIdx.y * rows_per, r1 = min(V, r0 + rows_per);
  constexpr int ROWS = ColBlock<LANES>::ROWS;
  auto put = [&](float (&v)[8], int r) {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = c + j < tokens ? sc[j] * (__expf(v[j] - l[j]) - (r == tgt[j] ? 1.f : 0.f)) : 0.f;
    store8<DT::BF16>(grad + r * ld + c, v);
  };
  int r = r0 + threadIdx.x / LANES;
  for (; r + 3 * ROWS < r1; r += 4 * ROWS) {
    float v[4][8];
#pragma unroll
    for (int u = 0; u < 4; ++u) load8<DT::BF16>(x + (r + u * ROWS) * ld + c, v[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u) put(v[u], r + u * ROWS);
  }
  for (; r < r1; r += ROWS) {
    float v[8];
    load8<DT::BF16>(x + r * ld + c, v);
    put(v, r);
  }
}

// f(blocks across, rows of a block, shares of the vocabulary) for blocks of `lanes`: 2048 blocks where there are that many of 64
// rows or more (the loss reads a (max, sum) of each column of each: 4096 blocks cost it 8 % at 2048 columns)
template <typename F>
static void col_blocks(int lanes, int V, int64_t ld, F f) {
  const int64_t across = (ld + 8 * lanes - 1) / (8 * lanes);
  const int64_t want = std::min<int64_t>(std::max<int64_t>(1, 2048 / across), (V + 63) / 64);
  const int per = (int)((V + want - 1) / want);
  f(dim3(across, (V + per - 1) / per), per);
}

static void xent_cols_checks(const at::Tensor& x, const at::Tensor& target) {
  check_beside(x, {target});
  SXE_CHECK(x.dim() == 2 && x.is_contiguous() && x.scalar_type() == at::kBFloat16 && x.size(1) % 8 == 0 && x.size(0) > 0 &&
                x.size(0) < (1ll << 30) && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0,
            "xent_cols: bf16 logits [vocab, columns], columns in multiples of 8");
  SXE_CHECK(target.is_cuda() && target.scalar_type() == at::kLong && target.is_contiguous() && target.numel() > 0 &&
                target.numel() <= x.size(1), "xent_cols: int64 targets, one for each of the first columns");
}

std::tuple<at::Tensor, at::Tensor> xent_cols_fwd(at::Tensor logits, at::Tensor target, int64_t ignore_index) {
  xent_cols_checks(logits, target);
  c10::DeviceGuard guard(logits.device());
  const int V = (int)logits.size(0);
  const int64_t ld = logits.size(1), tokens = target.numel();
  auto f = logits.options().dtype(at::kFloat);
  auto loss = at::empty({tokens}, f), lse = at::empty({tokens}, f);
  auto* x = reinterpret_cast<const unsigned short*>(logits.data_ptr());
  // pieces of 256 bytes of a row: with whole waves a row 2048 columns take 51 us for 47, 512 columns 35 for 22
  auto run = [&](auto lanes) {
    constexpr int LANES = decltype(lanes)::value;
    col_blocks(LANES, V, ld, [&](dim3 grid, int per) {
      auto part = at::empty({(int64_t)grid.y, ld, 2}, f);
      auto* pp = reinterpret_cast<float2*>(part.data_ptr<float>());
      hipLaunchKernelGGL(xent_cols_part_kernel<LANES>, grid, dim3(256), 0, cur_stream(), x, ld, V, per, pp);
      SXE_LAUNCH_CHECK();
      hipLaunchKernelGGL(xent_cols_loss_kernel, dim3((tokens + 15) / 16), dim3(256), 0, cur_stream(), x, ld, tokens, (int)grid.y, pp,
                         target.data_ptr<int64_t>(), ignore_index, loss.data_ptr<float>(), lse.data_ptr<float>());
    });
  };
  if (ld > 64) run(std::integral_constant<int, 16>{});
  else run(std::integral_constant<int, 8>{});
  SXE_LAUNCH_CHECK();
  return {loss, lse};
}

at::Tensor xent_cols_bwd(at::Tensor logits, at::Tensor target, at::Tensor lse, at::Tensor dloss, int64_t ignore_index) {
  xent_cols_checks(logits, target);
  check_beside(logits, {lse, dloss});
  for (const at::Tensor* t : {&lse, &dloss})
    SXE_CHECK(t->is_cuda() && t->scalar_type() == at::kFloat && t->is_contiguous() && t->numel() == target.numel(),
              "xent_cols: fp32 lse and dloss [tokens]");
  c10::DeviceGuard guard(logits.device());
  const int V = (int)logits.size(0);
  const int64_t ld = logits.size(1);
  auto grad = at::empty_like(logits);
  // whole waves a row where that leaves few of them idle: 8192 columns 309 us, 361 in pieces of 256 bytes
  auto run = [&](auto lanes) {
    constexpr int LANES = decltype(lanes)::value;
    col_blocks(LANES, V, ld, [&](dim3 grid, int per) {
      hipLaunchKernelGGL(xent_cols_bwd_kernel<LANES>, grid, dim3(256), 0, cur_stream(),
                         reinterpret_cast<const unsigned short*>(logits.data_ptr()), reinterpret_cast<unsigned short*>(grad.data_ptr()), ld,
                         V, target.numel(), per, target.data_ptr<int64_t>(), ignore_index, lse.data_ptr<float>(), dloss.data_ptr<float>());
    });
  };
  if (ld >= 2048 || ld % 512 == 0) run(std::integral_constant<int, 64>{});
  else if (ld > 64) run(std::integral_constant<int, 16>{});
  else run(std::integral_constant<int, 8>{});
  SXE_LAUNCH_CHECK();
  return grad;
}

static void xent_checks(const at::Tensor& logits, const at::Tensor& target) {
  SXE_CHECK(logits.dim() == 2 && logits.is_contiguous(), "xent: logits must be contiguous [rows, vocab]");
  SXE_CHECK(target.scalar_type() == at::kLong && target.numel() == logits.size(0) && target.is_contiguous(),
            "xent: target must be int64 [rows]");
}

// Returns (loss [rows] fp32, lse [rows] fp32). If `inplace_grad`, logits are overwritten with
// scale * (softmax - onehot) where scale = grad_scale * (*scale_t if given).
std::tuple<at::Tensor, at::Tensor> xent_fwd(at::Tensor logits, at::Tensor target, int64_t ignore_index, bool inplace_grad,
                                 c10::optional<at::Tensor> scale_t, double grad_scale) {
  xent_checks(logits, target);
  const int64_t rows = logits.size(0);
  const int V = (int)logits.size(1);
  c10::DeviceGuard guard(logits.device());
  auto loss = at::empty({rows}, logits.options().dtype(at::kFloat));
  auto lse = at::empty({rows}, logits.options().dtype(at::kFloat));
  if (rows == 0) return {loss, lse};
  const float* sp = nullptr;
  if (scale_t.has_value() && scale_t->defined()) {
    SXE_CHECK(scale_t->scalar_type() == at::kFloat && scale_t->is_cuda(), "xent: scale tensor fp32");
    sp = scale_t->data_ptr<float>();
  }
  const int grid = (int)std::min<int64_t>(rows, 8192);
  DT d = dtype_of(logits);
  SXE_DISPATCH_DT(d, TT, with_sweep(sweep_of(logits, V), [&](auto sw) {
    using S = typename dt_traits<TT>::storage;
    hipLaunchKernelGGL((xent_kernel<TT, decltype(sw)::value>), dim3(grid), dim3(256), 0, cur_stream(), reinterpret_cast<S*>(logits.data_ptr()),
                       rows, V, target.data_ptr<int64_t>(), ignore_index, loss.data_ptr<float>(), lse.data_ptr<float>(),
                       inplace_grad ? 1 : 0, sp, (float)grad_scale);
  }));
  SXE_LAUNCH_CHECK();
  return {loss, lse};
}

at::Tensor xent_bwd(at::Tensor logits, at::Tensor target, at::Tensor lse, at::Tensor dloss, int64_t ignore_index,
                    bool inplace) {
  xent_checks(logits, target);
  const int64_t rows = logits.size(0);
  const int V = (int)logits.size(1);
  SXE_CHECK(dloss.scalar_type() == at::kFloat && dloss.numel() == rows && dloss.is_contiguous(), "xent_bwd: dloss fp32 [rows]");
  c10::DeviceGuard guard(logits.device());
  at::Tensor grad = inplace ? logits : at::empty_like(logits);
  if (rows == 0) return grad;
  const bool alike = ((reinterpret_cast<uintptr_t>(logits.data_ptr()) ^ reinterpret_cast<uintptr_t>(grad.data_ptr())) & 15) == 0;
  const int grid = (int)std::min<int64_t>(rows, 8192);
  DT d = dtype_of(logits);
  SXE_DISPATCH_DT(d, TT, with_sweep(alike ? sweep_of(logits, V) : ELEMENTS, [&](auto sw) {
    using S = typename dt_traits<TT>::storage;
    hipLaunchKernelGGL((xent_bwd_kernel<TT, decltype(sw)::value>), dim3(grid), dim3(256), 0, cur_stream(),
                       reinterpret_cast<const S*>(logits.data_ptr()), reinterpret_cast<S*>(grad.data_ptr()), rows, V,
                       target.data_ptr<int64_t>(), ignore_index, lse.data_ptr<float>(), dloss.data_ptr<float>());
  }));
  SXE_LAUNCH_CHECK();
  return grad;
}

}  // namespace sxe

TORCH_LIBRARY_FRAGMENT(sxe, m) {
  m.def("xent_fwd(Tensor(a!) logits, Tensor target, int ignore_index, bool inplace_grad, Tensor? scale, float grad_scale) -> (Tensor, Tensor)");
  m.def("xent_bwd(Tensor(a!) logits, Tensor target, Tensor lse, Tensor dloss, int ignore_index, bool inplace) -> Tensor");
  m.def("xent_cols_fwd(Tensor logits, Tensor target, int ignore_index) -> (Tensor, Tensor)");
  m.def("xent_cols_bwd(Tensor logits, Tensor target, Tensor lse, Tensor dloss, int ignore_index) -> Tensor");
  m.def("xent_grad_dual(Tensor(a!) logits, Tensor target, Tensor lse, int ignore_index, Tensor scale_a, Tensor? scale_b) -> Tensor");
}
TORCH_LIBRARY_IMPL(sxe, CUDA, m) {
  m.impl("xent_cols_fwd", &sxe::xent_cols_fwd);
  m.impl("xent_cols_bwd", &sxe::xent_cols_bwd);
  m.impl("xent_grad_dual", &sxe::xent_grad_dual);
  m.impl("xent_fwd", &sxe::xent_fwd);
  m.impl("xent_bwd", &sxe::xent_bwd);
}
