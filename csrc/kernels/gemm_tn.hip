// Products of many rows on gfx950: y[M, N] = x[M, K] . w[N, K]' (+ bias), both operands with K contiguous, and the same with SwiGLU
// over w = [gate | up] in the epilogue (y[M, N / 2] = silu(x . gate') * (x . up'), one rounding, of the result). bf16 in and out, fp32
// sums; also a batch of them in one launch. skinny_gemm.hip and stream_gemm.hip have the forms for up to 32 rows.
//
// What bounds it: at 256 x 256 the card's power. Products of 16 x 16 x 32 run at 1.85 GHz where those of 32 x 32 x 16 run at
// 1.65 (they read and write half as many sums a flop); behind them LDS, which is busy for 80 % of the products' time.
//  * Slabs of 64 k, 128-byte rows (a whole cache line a row: with slabs of 32 the L2 answers twice the requests, 1.28 against 1.5
//    PFLOP/s), by direct-to-LDS loads through the loop of sxe_gemm_loop.h. Of 160 KB, 256 x 256 has room for two slabs of x and three
//    of w, which comes from memory where x is in a cache (1040 rows, 28672 x 4096 with SwiGLU 218 us the other way, 200 so).
//  * w rows lie in LDS so that a lane's sums of neighbouring 16-row blocks are 8 neighbouring columns of y: 16-byte stores (8-byte
//    ones cost 3 % at K = 4096). A round's workgroups end together, and their stores are what is left of its start: 5 % at K = 4096,
//    13 % at 2048.
//  * The row tiles of a column block run side by side on one XCD.
// us, the library / here: 8192 rows, 28672 x 4096 1255 / 1285 (with SwiGLU 1376 / 1290), 4096 x 14336 604 / 630, 4096 x 4096 174 / 184;
// 7588 rows, 28672 x 4096 with SwiGLU 1390 / 1250, 4096 x 14336 1010 / 620; 1040 rows 238 / 200 and 142 / 110.
#include "sxe_common.h"
#include "sxe_gemm_loop.h"
#include <torch/library.h>
#include <cmath>

namespace sxe {
namespace tn {
using namespace gl;

constexpr int ROW = 2 * BK;

struct Args {
  const unsigned short *x, *w, *bias;
  unsigned short* y;
  const int* rows;       // of a batch: rows of each product that are not zeros, the first ones; null: all
  float* part;           // splits of K: their sums, [splits, M, N]; or, of one split, `into`
  float* into;           // y in fp32; add: added to what is there
  bool add;
  int64_t ldx, ldw, bx, bw, by;  // elements from row to row, and from product to product of a batch
  int M, cols, half, slabs, per, parts;  // columns of y (SwiGLU: half the rows of w); w row that goes with row 0 as up; slabs of K, of a split;
                                         // splits of K, or products of a batch
  int tm, tn, gm;        // whole row tiles, column blocks; row tiles that run side by side
};

// Column of a tile that LDS row r of w holds (SwiGLU: of gate for even blocks of 16 rows, of up for odd ones)
template <bool GLU>
__device__ __forceinline__ int column(int r) {
  const int p = r & 15, b = GLU ? (r >> 5) & 1 : (r >> 4) & 1;
  return (GLU ? (r >> 6) * 32 : r & ~31) + 8 * (p >> 2) + 4 * b + (p & 3);
}

// The tile of `used` rows from row m0 on (T::BM rows are stored, as far as there are), columns from n0 on, ns slabs from `first` on
template <typename T, bool GLU, bool SPLIT>
__device__ __forceinline__ void run_tile(const Args& a, int m0, int n0, int part, int first, int ns, int used) {
  constexpr int RT = T::RT, CT = T::CT, NW = T::NW, PA = T::PA, PB = T::PB, BM = T::BM, X_LDS = T::SA * T::AS;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wr = w / T::WC, wc = w % T::WC;
  // ---- loads: a wave's load is 8 rows, chunk c of row r at place c ^ ((r >> 1) & 7). Rows and columns behind the last, and slabs,
  // repeat it
  unsigned xo[PA], wo[PB];
  const int lr = lane >> 3, lc = 16 * ((lane & 7) ^ (4 * (w & 1) + (lane >> 4)));
#pragma unroll
  for (int i = 0; i < PA; ++i) xo[i] = (unsigned)min(8 * (i * NW + w) + lr, a.M - 1 - m0) * (unsigned)(2 * a.ldx) + lc;
#pragma unroll
  for (int i = 0; i < PB; ++i) {
    const int r = 8 * (i * NW + w) + lr, c = min(column<GLU>(r), a.cols - 1 - n0);
    wo[i] = (unsigned)(c + (GLU && (r & 16) ? a.half : 0)) * (unsigned)(2 * a.ldw) + lc;
  }
  const char* xb = reinterpret_cast<const char*>(a.x + m0 * a.ldx + (SPLIT ? first * BK : part * a.bx));
  const char* wb = reinterpret_cast<const char*>(a.w + n0 * a.ldw + (SPLIT ? first * BK : part * a.bw));
  const unsigned l0 = lds_base();
  auto load_x = [&](int i, int slab, unsigned slot) { glds(xo[i], xb + min(slab, ns - 1) * ROW, l0 + slot + (i * NW + w) * 1024); };
  auto load_w = [&](int i, int slab, unsigned slot) {
    glds(wo[i], wb + min(slab, ns - 1) * ROW, l0 + X_LDS + slot + (i * NW + w) * 1024);
  };

  // ---- fragments: row (lane & 15) of a block, chunk 4 s + (lane >> 4) of step s
  const int l16 = lane & 15, g = lane >> 4;
  int ao[2], bo[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int ch = 16 * ((4 * s + g) ^ ((lane >> 1) & 7));
    ao[s] = (wr * RT * 16 + l16) * ROW + ch;
    bo[s] = X_LDS + (wc * CT * 16 + l16) * ROW + ch;
  }
  auto read_x = [&](bf16x8& f, int s, int i, unsigned slot) { f = *reinterpret_cast<const bf16x8*>(tl::lds + ao[s] + slot + i * 16 * ROW); };
  auto read_w = [&](bf16x8& f, int s, int j, unsigned slot) { f = *reinterpret_cast<const bf16x8*>(tl::lds + bo[s] + slot + j * 16 * ROW); };

  f32x4 acc[RT][CT];
  // a tile of fewer rows skips the products of the others
  const int live = __builtin_amdgcn_readfirstlane(min(max((used - wr * RT * 16 + 15) / 16, 0), RT));
  loop<T>(acc, ns, false, used >= BM, live, load_x, load_w, read_x, read_w);

  if constexpr (SPLIT || GLU) {
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int r = m0 + (wr * RT + i) * 16 + l16;
      if (r >= a.M) continue;
      if constexpr (SPLIT) {
        float* p = a.part + ((int64_t)part * a.M + r) * (GLU ? 2 * a.cols : a.cols);
#pragma unroll
        for (int j = 0; j < CT; ++j) {
          const int b = GLU ? (j >> 1) & 1 : j & 1, c = n0 + (GLU ? wc * CT * 8 : (wc * CT + (j & ~1)) * 16) + 8 * g + 4 * b;
          if (c >= a.cols) continue;
          f32x4* to = reinterpret_cast<f32x4*>(p + c + (GLU && (j & 1) ? a.cols : 0));
          *to = a.add ? *to + acc[i][j] : acc[i][j];  // (of one split)
        }
      } else {
        const int c = n0 + wc * CT * 8 + 8 * g;
        if (c >= a.cols) continue;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          v[e] = silu<false>(acc[i][2 * (e >> 2)][e & 3]) * acc[i][2 * (e >> 2) + 1][e & 3];
        }
        *reinterpret_cast<u32x4*>(a.y + part * a.by + (int64_t)r * a.cols + c) = u32x4{pack(v[0], v[1]), pack(v[2], v[3]), pack(v[4], v[5]), pack(v[6], v[7])};
      }
    }
  } else {
    float b[2][8] = {};
    if (a.bias != nullptr)
#pragma unroll
      for (int h = 0; h < 2; ++h) load8<DT::BF16>(a.bias + min(n0 + wc * CT * 16 + 32 * h + 8 * g, a.cols - 8), b[h]);
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      u32x4 v[2];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[h][e] = pack(acc[i][2 * h + (e >> 1)][2 * (e & 1)] + b[h][2 * e], acc[i][2 * h + (e >> 1)][2 * (e & 1) + 1] + b[h][2 * e + 1]);
      store_lines(a.y + part * a.by, a.cols, m0 + (wr * RT + i) * 16 + l16, a.M, n0 + wc * CT * 16, a.cols, v);
    }
  }
}

// The last tiles, of fewer rows, run as tiles of 64 or 128 rows: one of 256 with empty blocks of rows takes 0.93 of a whole one's time, as
// its loads and barriers stay. 28672 x 4096 with SwiGLU, us: 1040 rows 202 / 184, 1088 214 / 188, 1152 234 / 201 (1024: 181).
using T256 = Tile<2, 4, 8, 4, 2, 3, 2>;   // 256 x 256
using T192 = Tile<2, 4, 6, 4, 2, 3, 2>;   // 192 x 256
using T128 = Tile<2, 4, 4, 4, 3, 3, 2>;   // 128 x 256
using T64 = Tile<2, 4, 2, 4, 3, 3, 2>;    // 64 x 256
using N128 = Tile<2, 2, 4, 4, 2, 2, 2>;   // 128 x 128, two a CU

template <typename T, bool GLU, bool SPLIT>
__global__ void __launch_bounds__(T::NTHR, T::WAVES) gemm_kernel(Args a) {
  constexpr int BM = T::BM, CB = GLU ? T::BN / 2 : T::BN;
  // ---- workgroup -> (split or product, row tile, column block): neighbours in an XCD's run share w, gm row tiles at a time. The tiles of the
  // last rows, if these are no whole tile, come behind all others: they take less time and fill the last round
  const int whole = a.tm * a.tn * a.parts;
  const bool rest = (int)blockIdx.x >= whole;
  const int block = rest ? blockIdx.x - whole : blockIdx.x, nwg = rest ? gridDim.x - whole : whole;
  const int q8 = nwg / 8, r8 = nwg % 8, xcd = block % 8;
  const int id = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + block / 8;
  const int nt = rest ? a.tn : a.tm * a.tn, part = a.parts > 1 ? id / nt : 0, tile = id - part * nt;
  const int per_group = a.gm * a.tn, group = tile / per_group, in = tile - group * per_group, rows = min(a.tm - group * a.gm, a.gm);
  const int m0 = (rest ? a.tm : group * a.gm + in % rows) * BM, n0 = (rest ? tile : in / rows) * CB;
  const int first = SPLIT ? part * a.per : 0, ns = SPLIT ? min(a.per, a.slabs - first) : a.slabs;
  int used = a.M - m0;  // rows of the tile with products
  if (!SPLIT && a.rows != nullptr) {
    used = __builtin_amdgcn_readfirstlane(min(used, a.rows[part] - m0));
    if (used <= 0) {
      clear_tile(a.y + part * a.by + (int64_t)m0 * a.cols + n0, a.cols, min(BM, a.M - m0), min(CB, a.cols - n0));
      return;
    }
  }
  if constexpr (T::BN == 256) {
    static_assert(T64::LDS <= T::LDS && (BM <= 128 || T128::LDS <= T::LDS) && T64::NTHR == T::NTHR && T128::NTHR == T::NTHR);
    if (used <= (BM > 128 ? 128 : 64)) {
      const int there = min(BM, a.M - m0), small = used <= 64 ? T64::BM : T128::BM;
      if (!SPLIT && there > small)  // rows that are not in use
        clear_tile(a.y + part * a.by + (int64_t)(m0 + small) * a.cols + n0, a.cols, there - small, min(CB, a.cols - n0));
      if (used <= 64 || BM <= 128) run_tile<T64, GLU, SPLIT>(a, m0, n0, part, first, ns, used);
      else run_tile<T128, GLU, SPLIT>(a, m0, n0, part, first, ns, used);
      return;
    }
  }
  run_tile<T, GLU, SPLIT>(a, m0, n0, part, first, ns, used);
}

// y from the sums of the splits, 8 columns a thread; INTO: in fp32, with `add` added to what is there
template <bool GLU, bool INTO>
__global__ void __launch_bounds__(256) sum_kernel(const float* __restrict__ part, const unsigned short* __restrict__ bias,
                                                  void* __restrict__ y, int M, int cols, int splits, bool add) {
  const int64_t row = GLU ? 2 * (int64_t)cols : cols, all = M * row;
  const int per = cols / 8;
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < (int64_t)M * per; i += gridDim.x * 256ll) {
    const int64_t r = i / per;
    const int c = 8 * (int)(i - r * per);
    float v[8], u[8] = {};
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 0.f;
    for (int s = 0; s < splits; ++s) {
      const float* p = part + s * all + r * row + c;
      float t[8];
      load8<DT::F32>(p, t);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] += t[e];
      if (GLU) {
        load8<DT::F32>(p + cols, t);
#pragma unroll
        for (int e = 0; e < 8; ++e) u[e] += t[e];
      }
    }
    if (GLU) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = silu<false>(v[e]) * u[e];
    } else if (bias != nullptr) {
      load8<DT::BF16>(bias + c, u);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] += u[e];
    }
    if constexpr (INTO) {
      float* to = static_cast<float*>(y) + r * cols + c;
      if (add) {
        load8<DT::F32>(to, u);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += u[e];
      }
      store8<DT::F32>(to, v);
    } else {
      store8<DT::BF16>(static_cast<unsigned short*>(y) + r * cols + c, v);
    }
  }
}

// The tile and the splits of K that take least by this account: rounds of workgroups over the CUs, each its slabs and a start (with the
// stores of a round, which all its workgroups issue at once); the tiles of the last, fewer rows take what those of 64 or 128 rows take, or
// 0.93 of a whole one's time and up, and run on the CUs that the last round of whole ones leaves idle before they lengthen it. us a slab
// and a start, fitted to 32 weights of 2048 x 2048 to 28672 x 4096 at 33 to 13000 rows with every tile and split (433 sizes); with the
// small last tiles the choice is 0.3 % behind the best on average and 11 % at the most over 200 sizes of 260 to 12000 rows.
// 256 x 128 and 192 x 128 were never the best.
struct Form {
  int bm, bn, at_once;
  float slab, start;
};
constexpr Form kForms[4] = {{256, 256, 256, 1.24f, 0.4f}, {192, 256, 256, 0.96f, 2.5f}, {128, 256, 256, 0.79f, 2.4f}, {128, 128, 512, 1.02f, 1.7f}};
constexpr float kAlone = 0.87f;  // a slab's time of a tile of the last form that has a CU to itself
struct Plan {
  int form, splits;
  float us;
};
// when `rest` tiles of `part` rounds each, on `slots` of which `idle` are free a round earlier, end behind `rounds` rounds
static float end_of(int64_t rounds, int64_t idle, int64_t slots, int64_t rest, float part) {
  if (rest == 0) return rounds;
  const auto fit = [&](float end) {
    const auto of = [&](float time) { return time > 0 ? (int64_t)(time / part + 1e-4f) : 0; };
    return idle * of(end - rounds + 1) + (slots - idle) * of(end - rounds) >= rest;
  };
  // The last to end is the k-th on a slot that was idle, or the k-th on another. An idle slot takes 3 more at the most, as no part is below 0.5
  float first = 1e30f, second = 1e30f;
  for (int64_t k = std::max<int64_t>(1, rest / slots); idle > 0 && first > 1e29f; ++k)
    if (fit(rounds - 1 + k * part)) first = rounds - 1 + k * part;
  for (int64_t k = std::max<int64_t>(1, rest / slots - 3); second > 1e29f; ++k)
    if (fit(rounds + k * part)) second = rounds + k * part;
  return std::max<float>(rounds, std::min(first, second));
}
static Plan plan(int64_t M, int64_t N, int64_t slabs, bool may_split, int64_t batch) {
  Plan best{0, 1, 1e30f};
  for (int f = 0; f < 4; ++f) {
    const Form& t = kForms[f];
    const int64_t cols = (N + t.bn - 1) / t.bn * batch, rest = M % t.bm;
    for (int s : {1, 2, 3, 4, 6, 8}) {
      const int64_t tiles = (M + t.bm - 1) / t.bm * cols * s;
      if (s > 1 && (!may_split || slabs < 4 * s || tiles > 600)) break;
      const float one = (slabs + s - 1) / s * t.slab * (f == 3 && tiles <= kNumCUs ? kAlone : 1.f) + t.start;
      const int64_t whole = M / t.bm * cols * s, rounds = (whole + t.at_once - 1) / t.at_once;
      const float part = f == 3 || rest > (t.bm > 128 ? 128 : 64)
                             ? 0.93f + 0.07f * rest / t.bm
                             : ((slabs + s - 1) / s * (rest <= 64 ? 0.62f : kForms[2].slab) + kForms[2].start) / one;
      float us = one * end_of(rounds, rounds * t.at_once - whole, t.at_once, rest ? cols * s : 0, part);
      if (s > 1) us += 6.8f + M * N * 4 * (2 * s + 0.5f) / 6.9e6f;
      if (us < best.us) best = {f, s, us};
    }
  }
  return best;
}

template <typename T, bool GLU>
static void launch(Args a, int splits, int batch) {
  constexpr int CB = GLU ? T::BN / 2 : T::BN;
  a.tm = a.M / T::BM;
  a.tn = (a.cols + CB - 1) / CB;
  a.gm = std::max(1, std::min(a.tm, 8));
  a.parts = splits * batch;  // one of them is 1
  const int64_t grid = ((int64_t)a.M + T::BM - 1) / T::BM * a.tn * a.parts;
  SXE_CHECK(grid < (1ll << 30), "gemm_tn: too many tiles");
  if (a.part != nullptr) {
    const bool add = a.add;
    a.add = add && splits == 1;
    allow_lds<&gemm_kernel<T, GLU, true>>(T::LDS);
    hipLaunchKernelGGL((gemm_kernel<T, GLU, true>), dim3((unsigned)grid), dim3(T::NTHR), T::LDS, cur_stream(), a);
    auto sum = [&](auto kernel, void* y) {
      hipLaunchKernelGGL(kernel, dim3(stream_grid((int64_t)a.M * a.cols / 8, 256)), dim3(256), 0, cur_stream(), a.part, a.bias, y, a.M, a.cols, splits, add);
    };
    if (splits > 1) {
      if constexpr (GLU) sum(sum_kernel<true, false>, a.y);
      else if (a.into != nullptr) sum(sum_kernel<false, true>, a.into);
      else sum(sum_kernel<false, false>, a.y);
    }
  } else {
    allow_lds<&gemm_kernel<T, GLU, false>>(T::LDS);
    hipLaunchKernelGGL((gemm_kernel<T, GLU, false>), dim3((unsigned)grid), dim3(T::NTHR), T::LDS, cur_stream(), a);
  }
  SXE_LAUNCH_CHECK();
}

}  // namespace tn

// x, w [.., rows, K], one product or a batch; out: y's sizes where they are not those of one product; into: y in fp32, written or added to
static at::Tensor gemm_tn_run(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& bias, bool glu, int64_t tile, int64_t splits,
                              at::IntArrayRef out = {}, const c10::optional<at::Tensor>& rows = c10::nullopt,
                              const c10::optional<at::Tensor>& into = c10::nullopt, bool add = false) {
  check_beside(x, {w, bias, rows, into});
  const int64_t d = x.dim() - 2, batch = d ? x.size(0) : 1, M = x.size(d), K = x.size(d + 1), N = w.size(d), cols = glu ? N / 2 : N;
  SXE_CHECK(x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16 && w.size(d + 1) == K && (!d || w.size(0) == batch),
            "gemm_tn: bf16 x [M, K], w [N, K]");
  SXE_CHECK(K > 0 && K % tn::BK == 0 && N > 0 && N % (glu ? 16 : 8) == 0, "gemm_tn: K in multiples of 64, columns of 8");
  for (const at::Tensor* t : {&x, &w})
    SXE_CHECK((t->size(d) <= 1 || (t->stride(d) % 8 == 0 && t->stride(d) >= 0)) && (!d || batch <= 1 || t->stride(0) % 8 == 0) &&
                  t->stride(d + 1) == 1 && reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 == 0,
              "gemm_tn: rows of neighbouring elements that start on 16 bytes");
  const int64_t ldx = M > 1 ? x.stride(d) : K, ldw = N > 1 ? w.stride(d) : K;
  SXE_CHECK(M < (1ll << 30) && N < (1ll << 30) && K < (1ll << 30) && 512 * ldx < (1ll << 32) && (glu ? 2 * N * ldw : 512 * ldw) < (1ll << 32),
            "gemm_tn: sizes beyond 32-bit offsets");
  const bool has_bias = bias.has_value() && bias->defined();
  SXE_CHECK(!has_bias || (!glu && bias->scalar_type() == at::kBFloat16 && bias->dim() == 1 && bias->size(0) == N && bias->is_contiguous() &&
                          reinterpret_cast<uintptr_t>(bias->data_ptr()) % 16 == 0), "gemm_tn: bias bf16 [N]");
  SXE_CHECK(tile < 4 && splits >= 0 && splits <= 64, "gemm_tn: tile 0 - 3 or -1, splits 0 - 64");
  c10::DeviceGuard g(x.device());
  auto y = into.has_value() ? *into : d ? at::empty({batch, M, cols}, x.options()) : out.empty() ? at::empty({M, cols}, x.options()) : at::empty(out, x.options());
  if (y.numel() == 0) return y;
  tn::Args a{};
  a.x = reinterpret_cast<const unsigned short*>(x.data_ptr());
  a.w = reinterpret_cast<const unsigned short*>(w.data_ptr());
  a.bias = has_bias ? reinterpret_cast<const unsigned short*>(bias->data_ptr()) : nullptr;
  if (into.has_value()) {
    a.into = a.part = y.data_ptr<float>();
    a.add = add;
  } else {
    a.y = reinterpret_cast<unsigned short*>(y.data_ptr());
  }
  a.ldx = ldx;
  a.ldw = ldw;
  a.rows = used_rows(rows, batch);
  if (d) {
    a.bx = x.stride(0);
    a.bw = w.stride(0);
    a.by = M * cols;
  }
  a.M = M;
  a.cols = cols;
  a.half = cols;
  a.slabs = K / tn::BK;
  if (tile < 0) {
    const tn::Plan p = tn::plan(M, N, a.slabs, splits != 1, batch);
    tile = p.form;
    if (splits == 0) splits = p.splits;
  }
  splits = std::max<int64_t>(1, splits);
  SXE_CHECK(splits == 1 || batch == 1, "gemm_tn: a batch or splits");
  a.per = (a.slabs + splits - 1) / splits;
  const int parts = (a.slabs + a.per - 1) / a.per;  // none of them empty
  at::Tensor part;
  if (parts > 1) {
    part = at::empty({parts, M, N}, x.options().dtype(at::kFloat));
    a.part = part.data_ptr<float>();
  }
  auto run = [&](auto t) {
    using T = decltype(t);
    glu ? tn::launch<T, true>(a, parts, batch) : tn::launch<T, false>(a, parts, batch);
  };
  switch (tile) {
    case 0: run(tn::T256{}); break;
    case 1: run(tn::T192{}); break;
    case 2: run(tn::T128{}); break;
    default: run(tn::N128{});
  }
  return y;
}

// x [M, K] (rows may lie apart) or contiguous [.., K], w [N, K] (rows may lie apart), bias [N] or none -> [.., N], glu: [.., N / 2], a tensor
// of its own. tile, splits of K: -1, 0: the plan's
at::Tensor gemm_tn(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& bias, bool glu, int64_t tile, int64_t splits) {
  SXE_CHECK((x.dim() == 2 || (x.dim() > 2 && x.is_contiguous())) && w.dim() == 2, "gemm_tn: bf16 x [M, K] or contiguous [.., K], w [N, K]");
  if (x.dim() == 2) return gemm_tn_run(x, w, bias, glu, tile, splits);
  std::vector<int64_t> out(x.sizes().vec());
  out.back() = glu ? w.size(0) / 2 : w.size(0);
  return gemm_tn_run(x.view({-1, x.size(-1)}), w, bias, glu, tile, splits, out);
}

// c [M, N] fp32 (+)= x [M, K] . w [N, K]^T: a weight gradient whose operands lie with the tokens side by side; splits by the plan of the
// product in bf16: 515 x 768, 8192 tokens 72 us in one, 26 so, 5003 x 768 84, 66
void gemm_tn_into(const at::Tensor& x, const at::Tensor& w, at::Tensor c, bool add, int64_t tile, int64_t splits) {
  SXE_CHECK(x.dim() == 2 && w.dim() == 2 && c.dim() == 2 && c.size(0) == x.size(0) && c.size(1) == w.size(0) && c.scalar_type() == at::kFloat &&
                c.is_contiguous() && reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 == 0, "gemm_tn_into: bf16 x [M, K], w [N, K], fp32 c [M, N]");
  gemm_tn_run(x, w, c10::nullopt, false, tile, splits, {}, c10::nullopt, c, add);
}

// x [B, M, K], w [B, N, K] -> [B, M, N], one launch; rows int32 [B]: x[b, rows[b]:] is zeros, and so is y
at::Tensor gemm_tn_batch(const at::Tensor& x, const at::Tensor& w, int64_t tile, const c10::optional<at::Tensor>& rows) {
  SXE_CHECK(x.dim() == 3 && w.dim() == 3, "gemm_tn_batch: bf16 x [B, M, K], w [B, N, K]");
  return gemm_tn_run(x, w, c10::nullopt, false, tile, 1, {}, rows);
}

}  // namespace sxe

TORCH_LIBRARY_FRAGMENT(sxe, m) {
  m.def("gemm_tn(Tensor x, Tensor w, Tensor? bias, bool glu, int tile=-1, int splits=0) -> Tensor");
  m.def("gemm_tn_into(Tensor x, Tensor w, Tensor(a!) c, bool add, int tile=-1, int splits=0) -> ()");
  m.def("gemm_tn_batch(Tensor x, Tensor w, int tile=-1, Tensor? rows=None) -> Tensor");
}
TORCH_LIBRARY_IMPL(sxe, CUDA, m) {
  m.impl("gemm_tn", &sxe::gemm_tn);
  m.impl("gemm_tn_into", &sxe::gemm_tn_into);
  m.impl("gemm_tn_batch", &sxe::gemm_tn_batch);
}
