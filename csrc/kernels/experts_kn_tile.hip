// Expert products of prefill on gfx950, weights [E, K, N] as they are trained: rows sorted by expert, one launch for all experts,
// row counts read on the device.
//   expert_swiglu_kn_tile  h[r] = silu(x[token r] . Wg) * (x[token r] . Wu),  W = [E, K, gate | up]
//   expert_down_kn_tile    y[r] = h[r] . W[E, K, N]
//
// Reference: inference/v2/kernels/cutlass_ops/moe_gemm/moe_gemm.cu (grouped GEMM over expert-sorted rows). experts_kn.hip has the
// streaming form for few rows an expert.
//
// What bounds it: the matrix cores, fed from LDS. A workgroup takes 256 rows of one expert and 2 x 128 columns (128 of gate and the
// same of up, whose sums meet in a lane's registers), eight waves of 128 rows x (32 + 32) columns, fp32 sums in registers. Slabs of
// 32 k (32 KB) arrive by direct loads in a ring of five, four ahead; x rows are gathered on the way. x is read from LDS as it
// lies, W transposed (ds_read_b64_tr_b16). The two groups of four waves (rows 0 - 127 and the rest, one wave of each on a SIMD)
// run one barrier apart, with a barrier behind either of a slab's two steps of eight products a wave, so that one group's waits
// and reads lie under the other's products: 8 experts of 2048 rows, 4096 x 14336, ms of both products 5.9 in step, 5.5 so;
// ring depth (4 or 5) and the order of loads and reads are within 2 %. The row tiles of an expert and column block run side by
// side on one XCD, so W comes from memory once. Waves whose 128 rows lie past the expert's rows run no products. 5.5 ms are 1.05
// PFLOP/s at about 1.9 GHz, matrix cores busy for a good half of the time, no LDS bank conflicts.
#include "sxe_common.h"
#include "sxe_tile.h"
#include <torch/library.h>

namespace sxe {
namespace kt {
using namespace mf;

constexpr int BM = 256, HC = 128, BK = 32, RING = 5, AHEAD = 4, NTHR = 512;
constexpr int A_BYTES = BM * BK * 2, H_BYTES = BK * HC * 2, SLOT = A_BYTES + 2 * H_BYTES;  // 16 KB, 8 KB, 32 KB: the ring is all 160 KB of LDS

struct Args {
  const unsigned short* x;
  int64_t ldx;
  const int* token;  // row of x for every sorted row; null: the row itself
  int X;             // rows of x
  const unsigned short* w;
  const int* offs;
  unsigned short* y;
  int E, R, K, N;    // N: columns of W
  int cols, half;    // columns of y; column of W that goes with column 0 in the second half of a tile
};

__device__ __forceinline__ int tiles_of(const Args& a, int e) {
  if (e >= a.E) return 0;
  const int lo = min(max(a.offs[e], 0), a.R), hi = min(max(a.offs[e + 1], 0), a.R);
  return hi > lo ? (hi - lo + BM - 1) / BM : 0;
}

template <bool GLU>
__global__ void __launch_bounds__(NTHR, 2) tile_kernel(Args a) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wr = w >> 2, wc = w & 3;
  // ---- block -> (expert, column block, row tile), row tiles fastest, consecutive ones on one XCD
  constexpr int CB = GLU ? HC : 2 * HC;
  const int tn = (a.cols + CB - 1) / CB;
  int total = 0;
  for (int e0 = 0; e0 < a.E; e0 += 64) {
    int t = tiles_of(a, e0 + lane);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
    total += t;
  }
  const int nwg = __builtin_amdgcn_readfirstlane(total) * tn, orig = blockIdx.x;
  if (orig >= nwg) return;
  const int q8 = nwg / 8, r8 = nwg % 8, xcd = orig % 8;
  const int id = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + orig / 8;
  int expert = 0, first = 0, te = 1;
  {
    int before = 0;
    for (int e0 = 0; e0 < a.E; e0 += 64) {
      const int t = tiles_of(a, e0 + lane);
      int inc = t;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(inc, o, 64);
        if (lane >= o) inc += v;
      }
      const unsigned long long hit = __ballot((before + inc) * tn > id);
      if (hit) {
        const int l = __builtin_ctzll(hit);
        expert = e0 + l;
        te = __shfl(t, l, 64);
        first = before + __shfl(inc, l, 64) - te;
        break;
      }
      before += __shfl(inc, 63, 64);
    }
  }
  expert = __builtin_amdgcn_readfirstlane(expert);
  te = __builtin_amdgcn_readfirstlane(te);
  const int local = id - __builtin_amdgcn_readfirstlane(first) * tn, nt = local / te, rt = local - nt * te;
  const int r0 = min(max(a.offs[expert], 0), a.R) + rt * BM, r1 = min(max(a.offs[expert + 1], 0), a.R);
  const int n0 = nt * CB;

  // ---- loads of a slab: wave w brings rows 16 w .. and 128 + 16 w .. of x, k rows 4 w .. of both halves of W
  const unsigned short* xp[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = min(r0 + 128 * i + 16 * w + (lane >> 2), r1 - 1);
    const int64_t row = a.token != nullptr ? min(max(a.token[r], 0), a.X - 1) : r;
    xp[i] = a.x + row * a.ldx + 8 * ((lane & 3) ^ ((lane >> 4) & 3));
  }
  const unsigned short* wp[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    // a chunk past y's columns repeats the last ones (multiples of 8): its sums are not stored
    const int c = n0 + (GLU ? 0 : i * HC) + 8 * ((lane & 15) ^ ((lane >> 4) << 2));
    wp[i] = a.w + ((int64_t)expert * a.K + 4 * w + (lane >> 4)) * a.N + min(c, a.cols - 8) + (GLU ? i * a.half : 0);
  }
  char* lds = tl::lds;
  auto load = [&](int slab, int slot) {
    char* d = lds + slot * SLOT;
#pragma unroll
    for (int i = 0; i < 2; ++i) tl::glds16(xp[i] + slab * BK, d + (i * 8 + w) * 1024);
#pragma unroll
    for (int i = 0; i < 2; ++i) tl::glds16(wp[i] + (int64_t)slab * BK * a.N, d + A_BYTES + i * H_BYTES + w * 1024);
  };

  // ---- fragment offsets: x row (lane & 31), chunk 2 s + h; W column 32 wc + (lane & 31), k rows 8 h .. + 7 of a step
  const int l32 = lane & 31, h = lane >> 5;
  int ao[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) ao[s] = (wr * 128 + l32) * (BK * 2) + 16 * ((2 * s + h) ^ ((lane >> 2) & 3));
  const int g = lane >> 4, i16 = lane & 15, q = i16 >> 2, p = i16 & 3;
  const int bo = A_BYTES + (8 * h + q) * (HC * 2) + 16 * ((4 * wc + 2 * (g & 1) + (p >> 1)) ^ (q << 2)) + 8 * (p & 1);

  f32x16 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  bf16x8 fa[2][4], fb[2][2];
  auto read = [&](int slot, int s) {
    const char* b = lds + slot * SLOT;
#pragma unroll
    for (int i = 0; i < 4; ++i) fa[s][i] = *reinterpret_cast<const bf16x8*>(b + ao[s] + i * 32 * BK * 2);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int o = bo + j * H_BYTES + s * 16 * HC * 2;
      const i16x4 lo = lds_tr(b, o), hi = lds_tr(b, o + 4 * HC * 2);
      fb[s][j] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  };
  const bool live = r0 + wr * 128 < r1;
  auto multiply = [&](int s) {
    if (!live) return;
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[s][i], fb[s][j], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
  };

  const int ns = a.K / BK;
#pragma unroll
  for (int j = 0; j < AHEAD; ++j) load(min(j, ns - 1), j);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * (AHEAD - 2)) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  read(0, 0);
  if (wr == 1) __builtin_amdgcn_s_barrier();  // one barrier behind the other group from here on
  for (int s0 = 0; s0 < ns; s0 += RING) {
#pragma unroll
    for (int j = 0; j < RING; ++j) {
      if (s0 + j >= ns) break;
      read(j, 1);
      multiply(0);
      // this wave's part of slab s + 2 has landed and all of slab s is in its registers. So behind the barrier slab s + 1 is
      // there, also the part of the group that is a barrier behind, and nobody reads slab s - 1 any more
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(4 * (AHEAD - 3)) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      load(min(s0 + j + AHEAD, ns - 1), (j + AHEAD) % RING);  // over slab s - 1 (past the end: the last slab again)
      read((j + 1) % RING, 0);
      multiply(1);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
  }
  if (wr == 0) __builtin_amdgcn_s_barrier();  // as many as the other group
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int r = r0 + wr * 128 + 32 * i + (e & 3) + 8 * (e >> 2) + 4 * h;
      if (r >= r1) continue;
      unsigned short* yp = a.y + (int64_t)r * a.cols;
      const int c = n0 + 32 * wc + l32;
      if constexpr (GLU) {
        const float v = acc[i][0][e];
        if (c < a.cols) yp[c] = f32_to_bf16(v / (1.f + expf(-v)) * acc[i][1][e]);
      } else {
        if (c < a.cols) yp[c] = f32_to_bf16(acc[i][0][e]);
        if (c + HC < a.cols) yp[c + HC] = f32_to_bf16(acc[i][1][e]);
      }
    }
}

static Args args(const at::Tensor& x, const at::Tensor& w, const at::Tensor& offs) {
  SXE_CHECK_CUDA(x);
  SXE_CHECK(x.scalar_type() == at::kBFloat16 && x.dim() == 2 && x.is_contiguous() && w.is_cuda() && w.scalar_type() == at::kBFloat16 &&
                w.dim() == 3 && w.is_contiguous() && w.size(1) == x.size(1), "expert tile product: bf16 x [T, K], w [E, K, N]");
  SXE_CHECK(offs.is_cuda() && offs.is_contiguous() && offs.scalar_type() == at::kInt && offs.numel() == w.size(0) + 1,
            "expert tile product: offs int32 [E + 1]");
  SXE_CHECK(w.size(1) > 0 && w.size(1) % BK == 0 && w.size(2) > 0 && w.size(2) % 16 == 0 && w.size(0) > 0 && w.size(1) < (1 << 30) &&
                w.size(2) < (1 << 30) && x.size(0) < (1ll << 31) && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
                reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0,
            "expert tile product: K in multiples of 32, N of 16, 16-byte aligned operands");
  Args a{};
  a.x = reinterpret_cast<const unsigned short*>(x.data_ptr());
  a.ldx = x.size(1);
  a.X = x.size(0);
  a.w = reinterpret_cast<const unsigned short*>(w.data_ptr());
  a.offs = offs.data_ptr<int>();
  a.E = w.size(0);
  a.K = w.size(1);
  a.N = w.size(2);
  return a;
}

template <bool GLU>
static void launch(const Args& a) {
  constexpr int CB = GLU ? HC : 2 * HC;
  // every expert may end in a part of a tile
  const int64_t grid = ((int64_t)a.R / BM + std::min(a.E, a.R)) * ((a.cols + CB - 1) / CB);
  SXE_CHECK(grid < (1ll << 31), "expert tile product: too many tiles");
  allow_lds<&tile_kernel<GLU>>(RING * SLOT);
  hipLaunchKernelGGL(tile_kernel<GLU>, dim3((unsigned)grid), dim3(NTHR), RING * SLOT, cur_stream(), a);
  SXE_LAUNCH_CHECK();
}

}  // namespace kt

// x [T, K], w [E, K, 2 I] (gate | up), token int32 [R] -> silu(gate) * up [R, I] of the expert-sorted rows
at::Tensor expert_swiglu_kn_tile(const at::Tensor& x, const at::Tensor& w, const at::Tensor& offs, const at::Tensor& token) {
  kt::Args a = kt::args(x, w, offs);
  SXE_CHECK(token.is_cuda() && token.is_contiguous() && token.scalar_type() == at::kInt && token.numel() < (1ll << 31),
            "expert_swiglu_kn_tile: token int32 [R]");
  auto h = at::empty({token.numel(), w.size(2) / 2}, x.options());
  if (token.numel() == 0) return h;
  SXE_CHECK(x.size(0) > 0, "expert_swiglu_kn_tile: rows without tokens");
  c10::DeviceGuard g(x.device());
  a.token = token.data_ptr<int>();
  a.R = token.numel();
  a.y = reinterpret_cast<unsigned short*>(h.data_ptr());
  a.cols = a.half = a.N / 2;
  kt::launch<true>(a);
  return h;
}

// h [R, K] expert-sorted rows, w [E, K, N] -> [R, N]
at::Tensor expert_down_kn_tile(const at::Tensor& h, const at::Tensor& w, const at::Tensor& offs) {
  kt::Args a = kt::args(h, w, offs);
  auto y = at::empty({h.size(0), w.size(2)}, h.options());
  if (h.size(0) == 0) return y;
  c10::DeviceGuard g(h.device());
  a.R = a.X;
  a.y = reinterpret_cast<unsigned short*>(y.data_ptr());
  a.cols = a.N;
  kt::launch<false>(a);
  return y;
}

}  // namespace sxe

TORCH_LIBRARY_FRAGMENT(sxe, m) {
  m.def("expert_swiglu_kn_tile(Tensor x, Tensor w, Tensor offs, Tensor token) -> Tensor");
  m.def("expert_down_kn_tile(Tensor h, Tensor w, Tensor offs) -> Tensor");
}
TORCH_LIBRARY_IMPL(sxe, CUDA, m) {
  m.impl("expert_swiglu_kn_tile", &sxe::expert_swiglu_kn_tile);
  m.impl("expert_down_kn_tile", &sxe::expert_down_kn_tile);
}
