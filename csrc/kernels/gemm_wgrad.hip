// Weight gradients on gfx950: C[M, N] (+)= alpha * A' B, A = dY [T, M] and B = X [T, N] bf16, both row-major (the sum runs over the tokens,
// the ROWS of both operands), fp32 C; one product, or one for every expert of a layer in a launch; the tokens in one or two pieces.
//
// Why a hand-written kernel: this is the one training product whose operands both have the summed index as their rows. The vendor
// library runs it with an fp32 C at 0.8 - 1.1 PFLOP/s, and with few tokens (626 of each of 8 experts, 3072 x 16384) at 0.48. Here both
// operands stream through LDS as they lie and are read transposed (ds_read_b64_tr_b16): no operand needs a transposed copy.
//
// us, the library with fp32 C, with transposed copies or without / here, each call on another C: 28672 x 4096, 8192 tokens 1603 / 1520,
// 2048 513 / 466, 256 221 / 209; 4096 x 4096, 8192 tokens 253 / 215, 512 47 / 40; 128256 x 4096, 4096 tokens 3846 / 3644; 2048 x 2048, 4096 tokens
// 49 / 48; 8 experts of 256 tokens, 4096 x 28672 1890 / 1517.
//
// What bounds it: as in gemm_tn.hip, whose loop this is (sxe_gemm_loop.h), plus C, 128 MB of fp32 in a round of workgroups. A tile is
// 256 x 256 (128 x 256 or splits of the tokens where a plan of rounds finds them shorter), slabs of 64 tokens, rows of 256 or 128
// columns, chunk c (8 columns) of token t at place c ^ (4 (t & 3) + 2 ((t >> 3) & 1)): a transposing read takes 4 columns of 4
// tokens a lane, the four tokens' 32 bytes from four 64-byte groups of banks, neighbouring groups of lanes from the two halves of
// these. The tokens behind the last whole slab are cleared to zeros in LDS. Stores take whole cache lines.
#include "sxe_common.h"
#include "sxe_gemm_loop.h"
#include <torch/library.h>
#include <cmath>

namespace sxe {
namespace wg {
using namespace gl;

struct Args {
  const unsigned short *a, *b, *a2, *b2;  // first and second piece of the tokens
  const int *rows, *rows2;                // tokens of each expert's piece that are not zeros, the first ones; null: all
  float *c, *part;                        // part: sums of the splits, [splits, M, N]
  int64_t lda, ldb, ldc;
  int64_t ba, bb, ba2, bb2, bc;           // elements from expert to expert
  int M, N, n1, slabs, per, tail, tail2;  // slabs of the first piece, of both, of a split; tokens behind the last slab of each piece
  int tm, tn, gm, parts;                  // whole row tiles, column blocks; row tiles side by side; splits or experts
  float alpha;
};

// offset in LDS of a lane's transposing reads, rows of `bytes`, 16 columns from chunk `ch` on: tokens 8 (lane >> 4) .. and, 4 rows on,
// the next four
__device__ __forceinline__ int tr_off(int lane, int bytes, int ch) {
  const int g = lane >> 4, q = (lane >> 2) & 3, p = lane & 3;
  return (8 * g + q) * bytes + 16 * ((ch + (p >> 1)) ^ (4 * q + 2 * (g & 1))) + 8 * (p & 1);
}

template <typename T, bool ACCUM, bool SPLIT>
__global__ void __launch_bounds__(T::NTHR, T::WAVES) wgrad_kernel(Args a) {
  constexpr int RT = T::RT, CT = T::CT, NW = T::NW, PA = T::PA, PB = T::PB, BM = T::BM, BN = T::BN, X_LDS = T::SA * T::AS;
  constexpr int XROW = 2 * BM, WROW = 2 * BN, XL = XROW / 16, WL = WROW / 16, XK = 64 / XL, WK = 64 / WL;  // lanes of a row, rows of a load
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wr = w / T::WC, wc = w % T::WC;
  // ---- workgroup -> (split or expert, row tile, column block), as gemm_tn.hip
  const int whole = a.tm * a.tn * a.parts;
  const bool rest = (int)blockIdx.x >= whole;
  const int block = rest ? blockIdx.x - whole : blockIdx.x, nwg = rest ? gridDim.x - whole : whole;
  const int q8 = nwg / 8, r8 = nwg % 8, xcd = block % 8;
  const int id = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + block / 8;
  const int nt = rest ? a.tn : a.tm * a.tn, part = a.parts > 1 ? id / nt : 0, tile = id - part * nt;
  const int per_group = a.gm * a.tn, group = tile / per_group, in = tile - group * per_group, rows = min(a.tm - group * a.gm, a.gm);
  const int m0 = (rest ? a.tm : group * a.gm + in % rows) * BM, n0 = (rest ? tile : in / rows) * BN;
  const int expert = SPLIT ? 0 : part;
  // slabs with tokens other than zeros: of the first piece, of both
  int n1 = a.n1, slabs = a.slabs, tails[2] = {a.tail, a.tail2};
  if (!SPLIT && (a.rows != nullptr || a.rows2 != nullptr)) {
    auto in_use = [&](const int* rows, int n, int& tail) {
      if (rows == nullptr) return n;
      const int used = __builtin_amdgcn_readfirstlane(max(rows[expert], 0));
      if (used <= n * BK) tail = 0;
      return min(n, (used + BK - 1) / BK);
    };
    n1 = in_use(a.rows, a.n1, tails[0]);
    slabs = n1 + in_use(a.rows2, a.slabs - a.n1, tails[1]);
  }
  const int first = SPLIT ? part * a.per : 0, ns = SPLIT ? min(a.per, slabs - first) : slabs;

  // ---- loads: a wave's are XK (WK) tokens; columns behind the last repeat it
  const int xk = XK * w + lane / XL, wk = WK * w + lane / WL;
  const int xc = 2 * min(m0 + 8 * ((lane % XL) ^ (4 * (xk & 3) + 2 * ((xk >> 3) & 1))), a.M - 8);
  const int wcol = 2 * min(n0 + 8 * ((lane % WL) ^ (4 * (wk & 3) + 2 * ((wk >> 3) & 1))), a.N - 8);
  const unsigned xo = (unsigned)xk * (unsigned)(2 * a.lda) + xc, wo = (unsigned)wk * (unsigned)(2 * a.ldb) + wcol;
  const unsigned short *pa = a.a + expert * a.ba, *pb = a.b + expert * a.bb, *pa2 = a.a2 + expert * a.ba2, *pb2 = a.b2 + expert * a.bb2;
  const unsigned l0 = lds_base();
  auto tokens_a = [&](int slab) { return slab < n1 ? pa + (int64_t)slab * BK * a.lda : pa2 + (int64_t)(slab - n1) * BK * a.lda; };
  auto tokens_b = [&](int slab) { return slab < n1 ? pb + (int64_t)slab * BK * a.ldb : pb2 + (int64_t)(slab - n1) * BK * a.ldb; };
  auto load_x = [&](int i, int slab, unsigned slot) {
    glds(xo, tokens_a(first + min(slab, ns - 1)) + (int64_t)(i * NW * XK) * a.lda, l0 + slot + (i * NW + w) * 1024);
  };
  auto load_w = [&](int i, int slab, unsigned slot) {
    glds(wo, tokens_b(first + min(slab, ns - 1)) + (int64_t)(i * NW * WK) * a.ldb, l0 + X_LDS + slot + (i * NW + w) * 1024);
  };

  int ao[RT], bo[CT];
#pragma unroll
  for (int i = 0; i < RT; ++i) ao[i] = tr_off(lane, XROW, 2 * (wr * RT + i));
#pragma unroll
  for (int j = 0; j < CT; ++j) bo[j] = X_LDS + tr_off(lane, WROW, 2 * (wc * CT + j));
  auto frag = [](bf16x8& f, int o, int four) {
    const i16x4 lo = lds_tr(tl::lds, o), hi = lds_tr(tl::lds, o + four);
    f = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  auto read_x = [&](bf16x8& f, int s, int i, unsigned slot) { frag(f, ao[i] + slot + s * 32 * XROW, 4 * XROW); };
  auto read_w = [&](bf16x8& f, int s, int j, unsigned slot) { frag(f, bo[j] + slot + s * 32 * WROW, 4 * WROW); };

  f32x4 acc[RT][CT];
  const int live = __builtin_amdgcn_readfirstlane(min(max((a.M - m0 - wr * RT * 16 + 15) / 16, 0), RT));
  if (ns > 0) {
    loop<T>(acc, ns, false, !rest, live, load_x, load_w, read_x, read_w);
  } else {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < CT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // less than a slab of tokens at the end of a piece: zeros behind them, in both operands
#pragma unroll 1
  for (int piece = 0; piece < 2; ++piece) {
    const int tail = tails[piece];
    if (tail == 0 || first + ns != slabs) continue;
    __builtin_amdgcn_s_barrier();  // nobody reads the slots any more, and no load writes them
    asm volatile("" ::: "memory");
    const unsigned short* ta = piece ? pa2 + (int64_t)(a.slabs - a.n1) * BK * a.lda : pa + (int64_t)a.n1 * BK * a.lda;
    const unsigned short* tb = piece ? pb2 + (int64_t)(a.slabs - a.n1) * BK * a.ldb : pb + (int64_t)a.n1 * BK * a.ldb;
#pragma unroll
    for (int i = 0; i < PA; ++i)
      glds((unsigned)min(i * NW * XK + xk, tail - 1) * (unsigned)(2 * a.lda) + xc, ta, l0 + (i * NW + w) * 1024);
#pragma unroll
    for (int i = 0; i < PB; ++i)
      glds((unsigned)min(i * NW * WK + wk, tail - 1) * (unsigned)(2 * a.ldb) + wcol, tb, l0 + X_LDS + (i * NW + w) * 1024);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    for (int o = tail * XROW + threadIdx.x * 16; o < BK * XROW; o += T::NTHR * 16) *reinterpret_cast<u32x4*>(tl::lds + o) = u32x4{0u, 0u, 0u, 0u};
    for (int o = tail * WROW + threadIdx.x * 16; o < BK * WROW; o += T::NTHR * 16)
      *reinterpret_cast<u32x4*>(tl::lds + X_LDS + o) = u32x4{0u, 0u, 0u, 0u};
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      bf16x8 fb[CT];
#pragma unroll
      for (int j = 0; j < CT; ++j) read_w(fb[j], s, j, 0);
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        bf16x8 fa;
        read_x(fa, s, i, 0);
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa, acc[i][j], 0, 0, 0);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }

  // ---- a lane has four columns of a row in each block; two lanes with neighbouring rows change one of two neighbouring blocks, so that
  // a store writes 32 columns of 8 rows, whole lines. C is read and written around the caches, which hold the operands, and many weights
  // later is out of them anyway (the splits' sums are read next). us, through the caches / so, each call on another C: 28672 x 4096, 256 tokens
  // 231 / 209, 2048 483 / 466; 2048 x 2048, 256 18.8 / 15.8; 8 experts of 512, 4096 x 28672 2142 / 1747. (Reading C four rows of blocks ahead
  // as well: 1 - 10 % slower.)
  const int l16 = lane & 15, g = lane >> 4;
  const bool odd = lane & 1;
  auto put = [](f32x4 v, float* to) {
    if constexpr (SPLIT) *reinterpret_cast<f32x4*>(to) = v;
    else __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(to));
  };
  float* out = SPLIT ? a.part + (int64_t)part * a.M * a.N : a.c + expert * a.bc;
  const int64_t ld = SPLIT ? a.N : a.ldc;
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int r = m0 + (wr * RT + i) * 16 + (l16 & ~1);
    float* p[2];
    f32x4 old[2][2];
    bool in_row[2], in_col[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      p[h] = out + (int64_t)(r + h) * ld;
      in_row[h] = r + h < a.M;
      in_col[h] = n0 + wc * 64 + 32 * h + 16 * odd + 4 * g < a.N;
    }
    if (ACCUM) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int k = 0; k < 2; ++k)
          if (in_row[k] && in_col[h])
            old[h][k] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p[k] + n0 + wc * 64 + 32 * h + 16 * odd + 4 * g));
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4 v[2], t;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[0][e] = SPLIT ? acc[i][2 * h][e] : a.alpha * acc[i][2 * h][e];
        v[1][e] = SPLIT ? acc[i][2 * h + 1][e] : a.alpha * acc[i][2 * h + 1][e];
        t[e] = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, odd ? v[0][e] : v[1][e]), 0xB1, 0xF, 0xF, true));
      }
      f32x4 lo = odd ? t : v[0], hi = odd ? v[1] : t;
      if (ACCUM) lo += old[h][0], hi += old[h][1];
      const int c = n0 + wc * 64 + 32 * h + 16 * odd + 4 * g;
      if (in_col[h]) {
        if (in_row[0]) put(lo, p[0] + c);
        if (in_row[1]) put(hi, p[1] + c);
      }
    }
  }
}

// C (+)= alpha * the splits' sums, 4 columns a thread
template <bool ACCUM>
__global__ void __launch_bounds__(256) sum_kernel(const float* __restrict__ part, float* __restrict__ c, int64_t ldc, int M, int N, int splits,
                                                  float alpha) {
  const int64_t all = (int64_t)M * N;
  const int per = N / 4;
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < (int64_t)M * per; i += gridDim.x * 256ll) {
    const int64_t r = i / per, o = r * N + 4 * (i - r * per);
    f32x4 s = *reinterpret_cast<const f32x4*>(part + o);
    for (int k = 1; k < splits; ++k) s += *reinterpret_cast<const f32x4*>(part + k * all + o);
    f32x4* to = reinterpret_cast<f32x4*>(c + r * ldc + 4 * (i - r * per));
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] *= alpha;
    *to = ACCUM ? *to + s : s;
  }
}

using T256 = Tile<2, 4, 8, 4, 2, 3, 2>;  // 256 x 256
using T128 = Tile<2, 4, 4, 4, 3, 3, 2>;  // 128 x 256

template <typename T, bool ACCUM>
static void launch(Args a, int splits, int experts) {
  a.tm = a.M / T::BM;
  a.tn = (a.N + T::BN - 1) / T::BN;
  a.gm = std::max(1, std::min(a.tm, 8));
  a.parts = splits * experts;  // one of them is 1
  const int64_t grid = ((int64_t)a.M + T::BM - 1) / T::BM * a.tn * a.parts;
  SXE_CHECK(grid < (1ll << 30), "wgrad_gemm: too many tiles");
  if (splits > 1) {
    allow_lds<&wgrad_kernel<T, false, true>>(T::LDS);
    hipLaunchKernelGGL((wgrad_kernel<T, false, true>), dim3((unsigned)grid), dim3(T::NTHR), T::LDS, cur_stream(), a);
    hipLaunchKernelGGL(sum_kernel<ACCUM>, dim3(stream_grid((int64_t)a.M * a.N / 4, 256)), dim3(256), 0, cur_stream(), a.part, a.c, a.ldc,
                       a.M, a.N, splits, a.alpha);
  } else {
    allow_lds<&wgrad_kernel<T, ACCUM, false>>(T::LDS);
    hipLaunchKernelGGL((wgrad_kernel<T, ACCUM, false>), dim3((unsigned)grid), dim3(T::NTHR), T::LDS, cur_stream(), a);
  }
  SXE_LAUNCH_CHECK();
}

// (tile, splits of the tokens) of the least rounds of workgroups over the CUs, us: a slab 1.45 (256 x 256) or 0.82 (128 x 256), a start
// with C written 14 or 9, read first 12 or 8 more
static std::pair<int, int> plan(int64_t M, int64_t N, int64_t slabs, int64_t experts, bool accumulate) {
  std::pair<int, int> best{0, 1};
  float least = 1e30f;
  for (int f = 0; f < 2; ++f) {
    const int64_t tiles = (M + (f ? 127 : 255)) / (f ? 128 : 256) * ((N + 255) / 256) * experts;
    for (int s : {1, 2, 3, 4, 6, 8}) {
      if (s > 1 && (experts > 1 || slabs < 4 * s || tiles * s > 600)) break;
      const float one = (slabs + s) / s * (f ? 0.82f : 1.45f) + (f ? 9.f : 14.f) + (accumulate && s == 1 ? (f ? 8.f : 12.f) : 0.f);
      float us = (tiles * s + kNumCUs - 1) / kNumCUs * one;
      if (s > 1) us += 4.f + M * N * 4 * (2 * s + (accumulate ? 2 : 1)) / 3.6e6f;
      if (us < least) least = us, best = {f, s};
    }
  }
  return best;
}

// operands [T, cols] or [E, T, cols], rows that start on 16 bytes
static void check_tokens(const at::Tensor& t, int64_t d, const char* name) {
  SXE_CHECK(t.is_cuda() && t.scalar_type() == at::kBFloat16 && t.dim() == d + 2 && t.stride(d + 1) == 1 && t.size(d + 1) % 8 == 0 &&
                t.size(d + 1) >= 8 && (t.size(d) <= 1 || t.stride(d) % 8 == 0) && (!d || t.size(0) <= 1 || t.stride(0) % 8 == 0) &&
                reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 && (t.size(d) <= 1 || (t.stride(d) > 0 && t.stride(d) < (1 << 24))),
            "wgrad_gemm: ", name, " bf16 rows of multiples of 8 columns that start on 16 bytes");
}
static int64_t row_stride(const at::Tensor& t, int64_t d) { return t.size(d) > 1 ? t.stride(d) : t.size(d + 1); }

static void run(const at::Tensor& x, const at::Tensor& y, const at::Tensor* x2, const at::Tensor* y2, at::Tensor c, double alpha, bool accumulate,
                int64_t tile, int64_t splits, const c10::optional<at::Tensor>& rows = c10::nullopt,
                const c10::optional<at::Tensor>& rows2 = c10::nullopt) {
  check_beside(x, {y, c, rows, rows2});
  const int64_t d = c.dim() - 2;
  SXE_CHECK(d == 0 || d == 1, "wgrad_gemm: C [M, N] or [E, M, N]");
  check_tokens(x, d, "A");
  check_tokens(y, d, "B");
  const int64_t M = x.size(d + 1), N = y.size(d + 1), experts = d ? c.size(0) : 1;
  SXE_CHECK(c.scalar_type() == at::kFloat && c.size(d) == M && c.size(d + 1) == N && x.size(d) == y.size(d) && c.stride(d + 1) == 1 &&
                (M <= 1 || (c.stride(d) % 4 == 0 && c.stride(d) >= N)) && (!d || experts <= 1 || c.stride(0) % 4 == 0) &&
                (!d || (x.size(0) == experts && y.size(0) == experts)) && reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 == 0 &&
                M < (1 << 30) && N < (1 << 30) && x.size(d) < (1ll << 31) && experts < (1 << 16),
            "wgrad_gemm: fp32 C of rows that start on 16 bytes, as many tokens of A and B");
  c10::DeviceGuard g(x.device());
  Args a{};
  a.a = reinterpret_cast<const unsigned short*>(x.data_ptr());
  a.b = reinterpret_cast<const unsigned short*>(y.data_ptr());
  a.a2 = a.a;
  a.b2 = a.b;
  a.c = c.data_ptr<float>();
  a.lda = row_stride(x, d);
  a.ldb = row_stride(y, d);
  a.ldc = M > 1 ? c.stride(d) : N;
  a.M = M;
  a.N = N;
  a.alpha = alpha;
  if (d) {
    a.ba = x.stride(0);
    a.bb = y.stride(0);
    a.bc = c.stride(0);
  }
  if (d) {  // of experts only
    a.rows = used_rows(rows, experts);
    a.rows2 = used_rows(rows2, experts);
  }
  a.n1 = x.size(d) / BK;
  a.slabs = a.n1;
  a.tail = x.size(d) % BK;
  if (x2 != nullptr) {
    check_beside(x, {*x2, *y2});
    check_tokens(*x2, d, "A2");
    check_tokens(*y2, d, "B2");
    SXE_CHECK(x2->size(d + 1) == M && y2->size(d + 1) == N && x2->size(d) == y2->size(d) && (!d || (x2->size(0) == experts && y2->size(0) == experts)) &&
                  x2->size(d) < (1ll << 30) && x.size(d) < (1ll << 30), "wgrad_gemm: pieces of the same columns");
    if (row_stride(*x2, d) != a.lda || row_stride(*y2, d) != a.ldb) {  // one after the other
      run(x, y, nullptr, nullptr, c, alpha, accumulate, tile, splits, rows);
      run(*x2, *y2, nullptr, nullptr, c, alpha, true, tile, splits, rows2);
      return;
    }
    a.a2 = reinterpret_cast<const unsigned short*>(x2->data_ptr());
    a.b2 = reinterpret_cast<const unsigned short*>(y2->data_ptr());
    if (d) {
      a.ba2 = x2->stride(0);
      a.bb2 = y2->stride(0);
    }
    a.slabs += x2->size(d) / BK;
    a.tail2 = x2->size(d) % BK;
  }
  if (c.numel() == 0) return;
  if (a.slabs == 0 && a.tail == 0 && a.tail2 == 0) {
    if (!accumulate) c.zero_();
    return;
  }
  const auto p = plan(M, N, a.slabs, experts, accumulate);
  if (tile < 0) tile = p.first;
  if (splits <= 0) splits = p.second;
  splits = std::max<int64_t>(1, std::min<int64_t>(splits, a.slabs));
  SXE_CHECK(tile < 2 && (splits == 1 || experts == 1), "wgrad_gemm: tile 0 or 1, experts or splits");
  a.per = splits > 1 ? (a.slabs + splits - 1) / splits : a.slabs;
  if (splits > 1) splits = (a.slabs + a.per - 1) / a.per;  // none of them empty
  at::Tensor part;
  if (splits > 1) {
    part = at::empty({splits, M, N}, c.options());
    a.part = part.data_ptr<float>();
  }
  if (tile == 0) accumulate ? launch<T256, true>(a, splits, experts) : launch<T256, false>(a, splits, experts);
  else accumulate ? launch<T128, true>(a, splits, experts) : launch<T128, false>(a, splits, experts);
}

}  // namespace wg

// c (+)= alpha * a' b, a [T, M], b [T, N], c [M, N], or all with a leading expert index
// (rows int32 [E]: a[e, rows[e]:] or b[e, rows[e]:] is zeros, as far as 64 tokens go from there on both are)
void wgrad_gemm_(const at::Tensor& a, const at::Tensor& b, at::Tensor c, double alpha, bool accumulate, const c10::optional<at::Tensor>& rows) {
  wg::run(a, b, nullptr, nullptr, c, alpha, accumulate, -1, 0, rows);
}
// The same with a tile (0: 256 x 256, 1: 128 x 256, else the plan's) and splits of the tokens (0: the plan's) of the caller's, for comparisons
void wgrad_gemm_variant_(const at::Tensor& a, const at::Tensor& b, at::Tensor c, double alpha, bool accumulate, int64_t variant) {
  const int64_t tile = variant & 15;
  wg::run(a, b, nullptr, nullptr, c, alpha, accumulate, tile < 2 ? tile : -1, variant >> 4);
}
// c (+)= alpha * [a; a2]' [b; b2] (one after the other along the tokens) without the concatenation
void wgrad_gemm2_(const at::Tensor& a, const at::Tensor& b, const at::Tensor& a2, const at::Tensor& b2, at::Tensor c, double alpha,
                  bool accumulate, const c10::optional<at::Tensor>& rows, const c10::optional<at::Tensor>& rows2) {
  wg::run(a, b, &a2, &b2, c, alpha, accumulate, -1, 0, rows, rows2);
}

}  // namespace sxe

TORCH_LIBRARY_FRAGMENT(sxe, m) {
  m.def("wgrad_gemm_(Tensor a, Tensor b, Tensor(a!) c, float alpha, bool accumulate, Tensor? rows=None) -> ()");
  m.def("wgrad_gemm_variant_(Tensor a, Tensor b, Tensor(a!) c, float alpha, bool accumulate, int variant) -> ()");
  m.def("wgrad_gemm2_(Tensor a, Tensor b, Tensor a2, Tensor b2, Tensor(a!) c, float alpha, bool accumulate, Tensor? rows=None, "
        "Tensor? rows2=None) -> ()");
}
TORCH_LIBRARY_IMPL(sxe, CUDA, m) {
  m.impl("wgrad_gemm_", &sxe::wgrad_gemm_);
  m.impl("wgrad_gemm_variant_", &sxe::wgrad_gemm_variant_);
  m.impl("wgrad_gemm2_", &sxe::wgrad_gemm2_);
}
