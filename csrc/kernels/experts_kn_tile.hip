// Expert products of prefill and training on gfx950, weights [E, K, N] as they are trained: rows sorted by expert, one launch for all experts,
// row counts read on the device.
//   expert_swiglu_kn_tile  h[r] = silu(x[token r] . Wg) * (x[token r] . Wu),  W = [E, K, gate | up]
//   expert_down_kn_tile    y[r] = h[r] . W[E, K, N]
//   expert_mm_kn           y[e] = x[e] . W[e], x [E, C, K]: the same number of rows for all (training with a capacity); the rows behind
//                          those in use are cleared, not multiplied
//
// Reference: inference/v2/kernels/cutlass_ops/moe_gemm/moe_gemm.cu (grouped GEMM over expert-sorted rows). experts_kn.hip has the
// streaming form for few rows an expert.
//
// What bounds it: as in gemm_tn.hip, whose loop this is (sxe_gemm_loop.h). A workgroup takes 256 rows of one expert (128 where the
// experts have few) and 256 columns (128 of gate and the same of up, whose sums meet in a lane's registers), eight waves of 128 rows
// x 64 columns (32 + 32). x rows are gathered on the way and read from LDS as they lie, slabs of 64 k rows of W transposed
// (ds_read_b64_tr_b16). The row tiles of an expert and column block run side by side on one XCD, so W comes from memory once. Blocks
// of 16 rows past the expert's rows run no products. us, before (32-k slabs, products of 32 x 32 x 16, ring of five) / here: 8 experts of
// 2048 rows, 4096 x 2 x 14336 3620 / 2991, 14336 x 4096 1911 / 1611 (1.29 PFLOP/s); of 800 rows 1628 / 1358, 785 / 661. SwiGLU to 32 bits
// (gl::silu) has since added 1 - 2 % to the products with gate and up: of 800 rows, on one card, 1287 -> 1307.
#include "sxe_common.h"
#include "sxe_gemm_loop.h"
#include <torch/library.h>

namespace sxe {
namespace kt {
using namespace gl;

constexpr int WROW = 512;  // bytes of a slab's k row: 256 columns

struct Args {
  const unsigned short* x;
  int64_t ldx;
  const int* token;  // row of x for every sorted row; null: the row itself
  int X;             // rows of x
  const unsigned short* w;
  const int* offs;  // [E + 1]; null: C rows an expert
  int C;
  const int* rows;  // [E] of the C rows that are not zeros, the first ones; null: all
  unsigned short* y;
  int E, R, K, N;    // N: columns of W
  int cols, half;    // columns of y; column of W that goes with column 0 in the second half of a tile
};

// first row of an expert
__device__ __forceinline__ int row_of(const Args& a, int e) { return a.offs != nullptr ? min(max(a.offs[e], 0), a.R) : e * a.C; }
__device__ __forceinline__ int rows_of(const Args& a, int e) { return e < a.E ? max(row_of(a, e + 1) - row_of(a, e), 0) : 0; }
__device__ __forceinline__ int tiles_of(const Args& a, int e, int bm) { return (rows_of(a, e) + bm - 1) / bm; }

// When tiles of `bm` rows end, in slabs of a tile of 256: rounds of `whole` ones over the CUs, then what is left of them with the experts' last
// tiles, of more than 128 rows (`large`), of more than 64 or fewer. A slab of 192 rows takes 0.87 of one of 256, of 128
// 0.65, of 64 0.5.
constexpr float kClearly = 0.93f;
__host__ __device__ inline float end_of(int bm, int whole, int large, int some, int few) {
  const float w = bm == 256 ? 1.f : bm == 192 ? 0.87f : 0.65f, ws = some > 0 ? 0.65f : 0.5f;
  const int small = some + few;
  const int full = whole / kNumCUs, big = whole % kNumCUs + large, rounds = (big + kNumCUs - 1) / kNumCUs, free = rounds * kNumCUs - big;
  const auto more = [](int n) { return (n + kNumCUs - 1) / kNumCUs; };
  // the small ones on what the last round of large ones leaves free, a second time there if that is enough, else everywhere behind it
  float tail = rounds * w;
  if (rounds == 0) tail = more(small) * ws;
  else if (small > 2 * free) tail += more(small - free) * ws;
  else if (small > free) tail += 2 * ws > w ? 2 * ws - w : 0.f;
  return full * w + tail;
}

// The tile of rows r0 .. r1 of an expert (T::BM of them at most, `used` of them with products), columns from n0 on
template <typename T, bool GLU>
__device__ __forceinline__ void run_tile(const Args& a, int expert, int r0, int r1, int n0, int used) {
  constexpr int RT = T::RT, CT = T::CT, NW = T::NW, PA = T::PA, PB = T::PB, BM = T::BM, X_LDS = T::SA * T::AS, HC = T::BN / 2;
  static_assert(T::BN == 256 && NW == 8 && PB == 4);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wr = w / T::WC, wc = w % T::WC;
  // ---- loads: 8 rows of x, chunk c of row r at place c ^ ((r >> 1) & 7); 2 k rows of W, chunk c of row k at place
  // c ^ (4 (k & 3) + 2 ((k >> 3) & 1)). Slabs behind the last repeat it; the second half of one with 32 k repeats its first
  const int ns = a.K / BK, last = (a.K + BK - 1) / BK - 1;
  const bool half = a.K % BK != 0;
  unsigned xo[PA], wo[2], x_half;
  {
    const int c = (lane & 7) ^ (4 * (w & 1) + (lane >> 4));
    x_half = 16 * (c & 4);
#pragma unroll
    for (int i = 0; i < PA; ++i) {
      const int r = min(r0 + 8 * (i * NW + w) + (lane >> 3), r1 - 1);
      const int row = a.token != nullptr ? min(max(a.token[r], 0), a.X - 1) : r - r0;
      xo[i] = (unsigned)row * (unsigned)(2 * a.ldx) + 16 * c;
    }
    const int k = 2 * w + (lane >> 5), p = (lane & 31) ^ (4 * (k & 3) + 2 * ((k >> 3) & 1));
    // a chunk past y's columns repeats the last ones (multiples of 8): its sums are not stored
    const int col = GLU ? min(n0 + 8 * (p & 15), a.cols - 8) + (p >= 16 ? a.half : 0) : min(n0 + 8 * p, a.cols - 8);
    wo[0] = (unsigned)k * (unsigned)(2 * a.N) + 2 * col;
    wo[1] = wo[0] + (unsigned)(32 * a.N);  // 16 k rows on
  }
  const char* xb = reinterpret_cast<const char*>(a.token != nullptr ? a.x : a.x + r0 * a.ldx);
  const char* wb = reinterpret_cast<const char*>(a.w + (int64_t)expert * a.K * a.N);
  const unsigned l0 = lds_base();
  auto load_x = [&](int i, int slab, unsigned slot) {
    slab = min(slab, last);
    glds(xo[i] - (half && slab == last ? x_half : 0), xb + slab * 128, l0 + slot + (i * NW + w) * 1024);
  };
  auto load_w = [&](int i, int slab, unsigned slot) {
    slab = min(slab, last);
    const int k = slab * BK + (half && slab == last ? 0 : 32 * (i >> 1));
    glds(wo[i & 1], wb + (int64_t)k * (2 * a.N), l0 + X_LDS + slot + (i * NW + w) * 1024);
  };

  // ---- fragments: row (lane & 15) of a block of x, chunk 4 s + (lane >> 4) of step s; W: four columns of four k rows a lane,
  // 8 (lane >> 4) .. and the next four, of which the transposing read makes eight k of one column
  const int l16 = lane & 15, g = lane >> 4, q = l16 >> 2, p = l16 & 3;
  int ao[2], bo[CT];
#pragma unroll
  for (int s = 0; s < 2; ++s) ao[s] = (wr * RT * 16 + l16) * 128 + 16 * ((4 * s + g) ^ ((lane >> 1) & 7));
#pragma unroll
  for (int j = 0; j < CT; ++j) {
    const int ch = GLU ? 4 * wc + 2 * (j & 1) + 16 * (j >> 1) : 8 * wc + 2 * j;
    bo[j] = X_LDS + (8 * g + q) * WROW + 16 * ((ch + (p >> 1)) ^ (4 * q + 2 * (g & 1))) + 8 * (p & 1);
  }
  auto read_x = [&](bf16x8& f, int s, int i, unsigned slot) { f = *reinterpret_cast<const bf16x8*>(tl::lds + ao[s] + slot + i * 2048); };
  auto read_w = [&](bf16x8& f, int s, int j, unsigned slot) {
    const int o = bo[j] + slot + s * 32 * WROW;
    const i16x4 lo = lds_tr(tl::lds, o), hi = lds_tr(tl::lds, o + 4 * WROW);
    f = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };

  f32x4 acc[RT][CT];
  const int live = __builtin_amdgcn_readfirstlane(min(max((used - wr * RT * 16 + 15) / 16, 0), RT));
  loop<T>(acc, ns, half, used >= BM, live, load_x, load_w, read_x, read_w);

  // two blocks' four columns a lane -> eight of one: lanes of odd groups of 16 take the second block
  auto pair = [&](const float (&u)[4], const float (&v)[4]) {
    const auto lo = __builtin_amdgcn_permlane16_swap(pack(u[0], u[1]), pack(v[0], v[1]), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(pack(u[2], u[3]), pack(v[2], v[3]), false, false);
    return u32x4{lo[0], hi[0], lo[1], hi[1]};
  };
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int r = r0 + (wr * RT + i) * 16 + l16;
    float v[CT][4];
#pragma unroll
    for (int j = 0; j < (GLU ? 2 : CT); ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[j][e] = GLU ? silu<true>(acc[i][j][e]) * acc[i][j + 2][e] : acc[i][j][e];
#pragma unroll
    for (int h = 0; h < (GLU ? 1 : 2); ++h) {
      const int c = n0 + (GLU ? 32 * wc : 64 * wc + 32 * h) + 16 * (g & 1) + 8 * (g >> 1);
      const u32x4 out = pair(v[2 * h], v[2 * h + 1]);
      if (r < r1 && c < a.cols) *reinterpret_cast<u32x4*>(a.y + (int64_t)r * a.cols + c) = out;
    }
  }
}

using T256 = Tile<2, 4, 8, 4, 2, 3, 2>;
using T192 = Tile<2, 4, 6, 4, 2, 3, 2>;
using T128 = Tile<2, 4, 4, 4, 3, 3, 2>;
using T64 = Tile<2, 4, 2, 4, 3, 3, 2>;

// An expert's last tile, of fewer rows, runs as one of 64 or 128 rows (as gemm_tn.hip): six prompts of 50 to 2000
// tokens through two layers of 8 experts of 4096 x 14336, with the layers' other products, 4.48 / 4.44 ms
// EITHER: tiles of 256 or of 192 rows, whichever end sooner with the rows that the experts have
template <typename T, bool GLU, bool EITHER>
__global__ void __launch_bounds__(T::NTHR, T::WAVES) tile_kernel(Args a) {
  constexpr int HC = T::BN / 2;
  const int lane = threadIdx.x & 63;
  // ---- block -> (expert, column block, row tile), row tiles fastest, consecutive ones on one XCD
  constexpr int CB = GLU ? HC : 2 * HC;
  const int tn = (a.cols + CB - 1) / CB;
  int BM = T::BM;
  if constexpr (EITHER) {
    int n[8] = {};  // end_of's counts with tiles of 256 rows and of 192
    for (int e0 = 0; e0 < a.E; e0 += 64) {
      const int c = rows_of(a, e0 + lane);
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        const int bm = f ? 192 : 256, left = c % bm;
        n[4 * f] += c / bm;
        n[4 * f + 1] += left > 128;
        n[4 * f + 2] += left > 64 && left <= 128;
        n[4 * f + 3] += left > 0 && left <= 64;
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) n[i] += __shfl_xor(n[i], o, 64);
      n[i] *= tn;
    }
    if (end_of(192, n[4], n[5], n[6], n[7]) < kClearly * end_of(256, n[0], n[1], n[2], n[3])) BM = 192;
    BM = __builtin_amdgcn_readfirstlane(BM);
  }
  int total = 0;
  for (int e0 = 0; e0 < a.E; e0 += 64) {
    int t = tiles_of(a, e0 + lane, BM);
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
      const int t = tiles_of(a, e0 + lane, BM);
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
  const int r0 = row_of(a, expert) + rt * BM, r1 = row_of(a, expert + 1);
  const int n0 = nt * CB;
  int used = r1 - r0;  // rows of the tile with products
  if (a.rows != nullptr) used = __builtin_amdgcn_readfirstlane(min(used, a.rows[expert] - rt * BM));
  if (used <= 0 && a.rows != nullptr) {
    clear_tile(a.y + (int64_t)r0 * a.cols + n0, a.cols, min(BM, r1 - r0), min(CB, a.cols - n0));
    return;
  }
  static_assert(T64::LDS <= T::LDS && (T::BM <= 128 || T128::LDS <= T::LDS) && T64::NTHR == T::NTHR && T128::NTHR == T::NTHR);
  if (used <= (T::BM > 128 ? 128 : 64)) {
    const int there = min(BM, r1 - r0), small = used <= 64 ? T64::BM : T128::BM;
    if (there > small)  // rows that are not in use
      clear_tile(a.y + (int64_t)(r0 + small) * a.cols + n0, a.cols, there - small, min(CB, a.cols - n0));
    if (used <= 64 || T::BM <= 128) run_tile<T64, GLU>(a, expert, r0, r1, n0, used);
    else run_tile<T128, GLU>(a, expert, r0, r1, n0, used);
    return;
  }
  if constexpr (EITHER) {
    if (BM == 192) {
      run_tile<T192, GLU>(a, expert, r0, r1, n0, used);
      return;
    }
  }
  run_tile<T, GLU>(a, expert, r0, r1, n0, used);
}

static Args args(const at::Tensor& x, const at::Tensor& w) {
  SXE_CHECK_CUDA(x);
  SXE_CHECK(x.scalar_type() == at::kBFloat16 && x.dim() == 2 && x.is_contiguous() && w.is_cuda() && w.scalar_type() == at::kBFloat16 &&
                w.dim() == 3 && w.is_contiguous() && w.size(1) == x.size(1), "expert tile product: bf16 x [T, K], w [E, K, N]");
  SXE_CHECK(w.size(1) > 0 && w.size(1) % 32 == 0 && w.size(2) > 0 && w.size(2) % 16 == 0 && w.size(0) > 0 && w.size(1) < (1 << 30) &&
                w.size(2) < (1 << 30) && x.size(0) < (1ll << 31) && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
                reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0,
            "expert tile product: K in multiples of 32, N of 16, 16-byte aligned operands");
  SXE_CHECK(w.size(1) < (1 << 23) && w.size(2) < (1 << 26), "expert tile product: sizes beyond 32-bit offsets");
  Args a{};
  a.x = reinterpret_cast<const unsigned short*>(x.data_ptr());
  a.ldx = x.size(1);
  a.X = x.size(0);
  a.w = reinterpret_cast<const unsigned short*>(w.data_ptr());
  a.E = w.size(0);
  a.K = w.size(1);
  a.N = w.size(2);
  return a;
}
static Args args(const at::Tensor& x, const at::Tensor& w, const at::Tensor& offs) {
  Args a = args(x, w);
  SXE_CHECK(offs.is_cuda() && offs.is_contiguous() && offs.scalar_type() == at::kInt && offs.numel() == w.size(0) + 1,
            "expert tile product: offs int32 [E + 1]");
  a.offs = offs.data_ptr<int>();
  return a;
}

template <typename T, bool GLU, bool EITHER>
static void launch(const Args& a) {
  constexpr int CB = GLU ? T::BN / 2 : T::BN;
  // every expert may end in a part of a tile
  const int64_t grid = ((int64_t)a.R / (EITHER ? 192 : T::BM) + std::min(a.E, a.R)) * ((a.cols + CB - 1) / CB);
  SXE_CHECK(grid < (1ll << 31), "expert tile product: too many tiles");
  allow_lds<&tile_kernel<T, GLU, EITHER>>(T::LDS);
  hipLaunchKernelGGL((tile_kernel<T, GLU, EITHER>), dim3((unsigned)grid), dim3(T::NTHR), T::LDS, cur_stream(), a);
  SXE_LAUNCH_CHECK();
}
// 128 rows a tile where few column blocks make few rounds of workgroups over the CUs and theirs are the shorter ones (a round of 128 rows
// takes 0.65 of one of 256, as in `end_of`; the rule takes it for two thirds). Products with h, us, 256 / 128: 4096 columns of 14336 k, 150 rows an expert of eight 271 / 233, 250
// 318 / 382, 400 581 / 407, 800 661 / 768; 2048 of 8192, 250 170 / 118, 550 187 / 203. Many column blocks: 28672 of 4096 k, 50 rows
// 379 / 364, 150 403 / 508, 800 1358 / 1481
// 192 rows where as many for every expert would end clearly sooner in them; the kernel decides by the rows that they have (a prompt's lie near
// the mean: 697 to 751 of eight experts). us, 128 or 256 / so: 4096 columns of 14336 k, 730 rows an expert of eight 645 / 576; 300 to 1500 rows an
// expert, widths 2048, 3072 and 4096, evenly and unevenly filled, 1.03 of the speed on average, up to 1.2; but many column blocks, whose last round is one of many, and the workgroups that the grid has for 192: 28672 of 4096 k +1 % on average.
template <bool GLU>
static void launch(const Args& a) {
  const int64_t blocks = (a.cols + (GLU ? 127 : 255)) / (GLU ? 128 : 256);
  auto rounds = [&](int64_t bm) {
    const int64_t tiles = a.R < bm * a.E ? a.E : a.R / bm + a.E / 2;
    return (tiles * blocks + kNumCUs - 1) / kNumCUs;
  };
  auto even = [&](int bm) {  // all experts with as many rows
    const int c = (a.R + a.E - 1) / a.E, left = c % bm, n = (int)std::min<int64_t>(a.E * blocks, 1 << 20);
    return end_of(bm, c / bm * n, left > 128 ? n : 0, left > 64 && left <= 128 ? n : 0, left > 0 && left <= 64 ? n : 0);
  };
  const bool low = blocks <= 32 && 2 * rounds(128) <= 3 * rounds(256);
  if constexpr (!GLU) {
    if (a.offs != nullptr && blocks <= 32 && even(192) < kClearly * (low ? even(128) : even(256))) return launch<T256, GLU, true>(a);
  }
  if (low) launch<T128, GLU, false>(a);
  else launch<T256, GLU, false>(a);
}

}  // namespace kt

// x [T, K], w [E, K, 2 I] (gate | up), token int32 [R] -> silu(gate) * up [R, I] of the expert-sorted rows
at::Tensor expert_swiglu_kn_tile(const at::Tensor& x, const at::Tensor& w, const at::Tensor& offs, const at::Tensor& token) {
  kt::Args a = kt::args(x, w, offs);
  SXE_CHECK(token.is_cuda() && token.is_contiguous() && token.scalar_type() == at::kInt && token.numel() < (1ll << 31),
            "expert_swiglu_kn_tile: token int32 [R]");
  auto h = at::empty({token.numel(), w.size(2) / 2}, x.options());
  if (token.numel() == 0) return h;
  SXE_CHECK(x.size(0) > 0 && x.numel() < (1ll << 31), "expert_swiglu_kn_tile: rows without tokens, or x beyond 32-bit offsets");
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

// x [E, C, K], w [E, K, N] -> [E, C, N]; used int32 [E]: x[e, used[e]:] is zeros, and so is y
at::Tensor expert_mm_kn(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& used) {
  check_beside(x, {w, used});
  SXE_CHECK(x.dim() == 3 && x.is_contiguous() && w.dim() == 3 && x.size(0) == w.size(0) && x.device() == w.device() && x.numel() < (1ll << 40) &&
                x.size(0) * x.size(1) < (1ll << 31), "expert_mm_kn: x [E, C, K], w [E, K, N]");
  const at::Tensor rows = x.view({-1, x.size(2)});
  kt::Args a = kt::args(rows, w);
  auto y = at::empty({x.size(0), x.size(1), w.size(2)}, x.options());
  if (y.numel() == 0) return y;
  c10::DeviceGuard g(x.device());
  a.C = x.size(1);
  a.rows = used_rows(used, w.size(0));
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
  m.def("expert_mm_kn(Tensor x, Tensor w, Tensor? rows=None) -> Tensor");
}
TORCH_LIBRARY_IMPL(sxe, CUDA, m) {
  m.impl("expert_swiglu_kn_tile", &sxe::expert_swiglu_kn_tile);
  m.impl("expert_down_kn_tile", &sxe::expert_down_kn_tile);
  m.impl("expert_mm_kn", &sxe::expert_mm_kn);
}
