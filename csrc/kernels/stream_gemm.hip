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

// What is done with the sums: EPI_PLAIN bf16 (+ bias); EPI_GLU silu(gate) * up; and those of a decoder's layer, whose norms and RoPE are no
// launches of their own: EPI_RES adds the residual stream, EPI_ROPE rotates q and k and appends k and v to the paged cache, EPI_NGLU and
// EPI_HEAD (fp32 result) are the other two products behind a norm. A norm between two products is split over both: the first one's
// epilogue holds the new residual stream and leaves (stream x norm weight) in bf16 for the next product and its tiles' sums of squares; the
// next one asks for those (rows x tiles of 4 bytes: 32 rows of hidden 4096 32 KB, of 8192 64) in front of its first operand loads, adds them up
// behind these and multiplies its sums by 1 / rms. The operand is
// rounded once, as a norm's result is; the product and the sum are no longer rounded before they meet the stream.
// A launch costs a step ~4.7 us whatever it does: a layer of 4096 x 4096 / 28672 x 4096 has 6 of them, 9 before.
enum Epi { EPI_PLAIN, EPI_GLU, EPI_RES, EPI_ROPE, EPI_NGLU, EPI_HEAD };

struct Args {
  const unsigned short* x;
  int64_t ldx;
  const void* w;
  int64_t ldw;
  const float* scale;          // fp8: of a row of w
  const unsigned short* bias;  // or null
  unsigned short* y;
  int M, N, K;
  // behind a norm (ROPE, NGLU, HEAD; part null: x is normed): sums of squares [parts, mp] of the rows' tiles
  const float* part;
  int parts, mp;  // mp: M rounded up to 8, 16 or 32
  float eps;
  float* yf;  // HEAD
  // RES: y = bf16(stream * gw)
  const unsigned short *res, *gw;
  int64_t ldr;
  // RES of one row that attention has left in splits (null: x): unnormalised sums [splits, K] and (max, sum) [splits, K / dim, 2], log2
  const float *po, *pml;
  int splits, dim;
  unsigned short* h;  // [M, N], the new stream
  float* sums;        // [N / 16, mp]; half tiles: [N / 8, mp]
  // ROPE: w's rows are nq + 2 nkv heads of 128
  const float *rcos, *rsin;  // [positions, 64]
  const int64_t *pos, *slots;
  unsigned short* cache;  // [blocks, 2, nkv, bs, 128]
  int nq, nkv, bs;
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
// X8 (up to 8 rows): 256 columns, of which the matrix core's columns 0 - 7 have the one half of x and 8 - 15 the other one. A half of W goes to
// sums of its own with the same registers of x, eight columns of which count: half the loads of x and half of its exchange.
template <bool FP8, int MB, int NT, bool ONCE, bool X8 = false>
struct Piece {
  static constexpr int PIECE = FP8 || X8 ? 256 : 128, XL = FP8 && !X8 ? 2 : 1, WL = X8 && !FP8 ? 2 : 1;
  u32x4 w[NT * WL][4], x[MB][XL][4];
  // wr, xr: the rows 4 (row / 4) + u of this lane's quad, at chunk 4 g + j
  __device__ __forceinline__ void load_w(const char* const (&wr)[NT], int64_t ldw, int k0, int K, int c) {
#pragma unroll
    for (int t = 0; t < NT * WL; ++t) {
      const int kw = k0 + 128 * (t % WL) + c * (FP8 ? 16 : 8);  // K is a multiple of 8 (16), so a lane's vector is in or out
      const bool win = kw < K;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        w[t][u] = u32x4{0u, 0u, 0u, 0u};
        const auto* p = reinterpret_cast<const u32x4*>(wr[t / WL] + u * ldw + (int64_t)kw * (FP8 ? 1 : 2));
        if (win) w[t][u] = ONCE ? __builtin_nontemporal_load(p) : *p;
      }
    }
  }
  __device__ __forceinline__ void load_x(const unsigned short* const (&xr)[MB][4], int k0, int K, int c) {
#pragma unroll
    for (int h = 0; h < XL; ++h) {
      const int hx = X8 ? (threadIdx.x >> 3) & 1 : h;
      const int kx = k0 + 8 * (FP8 ? 8 * (c >> 2) + 4 * hx + (c & 3) : X8 ? 16 * hx + c : c);
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
  // one row in LDS for all of them, as the exchange would leave it
  __device__ __forceinline__ void row_x(const unsigned short* row, int k0, int K, int g) {
#pragma unroll
    for (int h = 0; h < XL; ++h)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int kx = k0 + 8 * (4 * (XL * g + h) + u);
        x[0][h][u] = u32x4{0u, 0u, 0u, 0u};
        if (kx < K) x[0][h][u] = *reinterpret_cast<const u32x4*>(row + kx);
      }
  }
  template <bool ROW = false>
  __device__ __forceinline__ void multiply(f32x4 (&acc)[MB][NT * (X8 ? 2 : 1)], bool odd1, bool odd2) {
    if constexpr (!ROW) {
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int h = 0; h < XL; ++h) exchange(x[m][h], odd1, odd2);
    }
#pragma unroll
    for (int t = 0; t < NT * WL; ++t) {
      exchange(w[t], odd1, odd2);
#pragma unroll
      for (int f = 0; f < (FP8 ? 8 : 4); ++f) {
        u32x4 a;
        if constexpr (FP8) a = widen(w[t][f >> 1][2 * (f & 1)], w[t][f >> 1][2 * (f & 1) + 1]);
        else a = w[t][f];
        const int at = !X8 ? t : FP8 ? 2 * t + (f >> 2) : t;
#pragma unroll
        for (int m = 0; m < MB; ++m) acc[m][at] = mfma16(a, x[m][X8 ? 0 : f >> 2][f & 3], acc[m][at]);
      }
    }
  }
};

constexpr int MERGE_K = 2048;  // columns of a row that is merged on its way in

// The row of attention's splits, sum_s 2^(M_s - M) o_s / sum_s 2^(M_s - M) L_s, in bf16 as a launch of its own would leave it. A split
// without keys has a maximum of -inf and nothing behind it. Four columns a thread, the loads of eight splits at once.
__device__ __forceinline__ void merge_row(const Args& a, unsigned short* row) {
  constexpr int U = 8;
  const int heads = a.K / a.dim;
  for (int k = 4 * threadIdx.x; k < a.K; k += 4 * 64 * NW) {
    float top = -INFINITY, den = 0.f;
    f32x4 num = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < a.splits; s0 += U) {
      float ms[U], ls[U];
      f32x4 o[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t s = min(s0 + u, a.splits - 1), at = 2 * (s * heads + k / a.dim);
        ms[u] = a.pml[at];
        ls[u] = a.pml[at + 1];
        o[u] = *reinterpret_cast<const f32x4*>(a.po + s * a.K + k);
      }
      float most = top;
#pragma unroll
      for (int u = 0; u < U; ++u) most = fmaxf(most, ms[u]);
      const float r = top == -INFINITY ? 0.f : exp2f(top - most);
      top = most;
      den *= r;
#pragma unroll
      for (int q = 0; q < 4; ++q) num[q] *= r;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (s0 + u >= a.splits || ms[u] == -INFINITY) continue;
        const float f = exp2f(ms[u] - top);
        den += f * ls[u];
#pragma unroll
        for (int q = 0; q < 4; ++q) num[q] += f * o[u][q];
      }
    }
    u16x4 v;
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = f32_to_bf16(den > 0.f ? num[q] / den : 0.f);
    *reinterpret_cast<u16x4*>(row + k) = v;
  }
}

// HALF (up to 8 rows): a tile of 8 columns, each twice. The matrix core's rows 0 - 7 have one half of a piece's K, rows 8 - 15 the other one,
// of W and of x alike, and the two blocks of the result that belong together are added: no lane loads what another one does, and there are
// twice the workgroups, each with half the pieces one behind the other.
template <bool FP8, int MB, int NT, int EPI, bool ONCE, bool HALF = false, bool MERGE = false, int DEEP = 1, bool X8 = false>
__global__ void __launch_bounds__(64 * NW, 2) stream_gemm_kernel(Args a) {
  static_assert(!HALF || (MB == 1 && NT == 1), "");
  static_assert(!MERGE || (EPI == EPI_RES && HALF), "");
  static_assert(!X8 || (MB == 1 && !HALF), "");
  constexpr bool GLU = EPI == EPI_GLU || EPI == EPI_NGLU, NORMED = EPI >= EPI_ROPE;
  constexpr int OT = GLU ? NT / 2 : NT;  // tiles of output columns
  constexpr int TC = HALF ? 8 : 16, PAIRS = TC * NT / 2;
  __shared__ f32x4 red[NW][NT][64];
  __shared__ __attribute__((aligned(16))) unsigned short merged[MERGE ? MERGE_K : 8];
  __shared__ __attribute__((aligned(16))) float squares[NORMED ? NW : 1][NORMED ? 32 : 1];  // written four at a time
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, g = lane >> 4;
  const int half = a.N / 2;
  const int j = lane & 3, quad0 = l16 & (TC - 4), c = 4 * g + j;
  // ROPE: a workgroup has both halves of what it rotates, as two tiles or as the halves of one; else NT tiles side by side
  const int n0 = EPI == EPI_ROPE ? (int)(blockIdx.x / (64 / PAIRS)) * 128 + (int)(blockIdx.x % (64 / PAIRS)) * PAIRS : (int)blockIdx.x * TC * OT;
  auto column = [&](int t, int q) {  // of column q (a multiple of 4) of tile t
    if constexpr (EPI == EPI_ROPE) return NT == 2 ? n0 + 64 * t + q : HALF ? n0 + 16 * q : n0 + (q & 4) + 8 * (q & 8);
    return GLU ? n0 + 16 * (t % OT) + (t / OT) * half + q : n0 + 16 * t + q;
  };
  // what this lane finishes: 4 columns of row frow of tile `wave` (HALF: the four groups of 16 lanes do the same)
  const int frow = HALF ? lane & 7 : l16, fq = HALF ? (lane & 8) / 2 : 4 * g;
  // tiles start inside W (N a multiple of 4: a quad's rows all do or none); what lies past the end repeats the last rows
  const char* wr[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) wr[t] = static_cast<const char*>(a.w) + (int64_t)min(column(t, quad0), a.N - 4) * a.ldw * (FP8 ? 1 : 2);
  const int64_t ldw = a.ldw * (FP8 ? 1 : 2);
  const unsigned short* xr[MB][4];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int u = 0; u < 4; ++u) xr[m][u] = a.x + (int64_t)min(16 * m + (X8 ? quad0 & 4 : quad0) + u, a.M - 1) * a.ldx;
  const bool odd1 = j & 1, odd2 = j & 2;
  constexpr int AL = X8 ? 2 : 1;
  f32x4 acc[MB][NT * AL];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int t = 0; t < NT * AL; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  // DEEP 2: the next piece is in flight behind this one's products. It halves the workgroups on a CU: only where a launch has few
  using P = Piece<FP8, MB, NT, ONCE, X8>;
  constexpr int STEP = HALF ? 2 * P::PIECE : P::PIECE;
  int k0 = wave * STEP + (HALF ? (l16 >> 3) * P::PIECE : 0);
  P p[DEEP];
  auto load = [&](P& q, int ahead) {  // the piece `ahead` of the one that is next
    q.load_w(wr, ldw, k0 + ahead * NW * STEP, a.K, c);
    if constexpr (!MERGE) q.load_x(xr, k0 + ahead * NW * STEP, a.K, c);
  };
  // what the epilogue reads is on its way beside the first piece
  u16x4 res[MB], gw;
  f32x4 cs[MB], sn[MB];
  int64_t slot[MB];
  if constexpr (EPI >= EPI_RES) {
    int64_t at[MB];
    if constexpr (EPI == EPI_ROPE) {
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const int row = min(16 * m + frow, a.M - 1);
        at[m] = a.pos[row];
        slot[m] = a.slots[row];
      }
    }
    // First the sums of squares: loaded after the piece they came last, and each load of a loop
    // over them waited for the one before. Asked for at once and in front, they are added up while
    // the piece is on its way. Head of 32000 x 4096: 47.9 to 44.4 us at 8 rows, 57.8 to 56.4 at 32;
    // gate and up of 28672 x 4096 at 32 rows: 51.3 to 49.4; QKV of 6144 in e4m3 at 8: 10.8 to 10.3.
    constexpr int AHEAD = 4;  // loads of a thread: 256 tiles of 32 rows
    f32x4 sq[AHEAD];
    const int quads = a.mp / 4, pieces = NORMED && a.part != nullptr ? a.parts * quads : 0;
    if constexpr (NORMED) {
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) {
        sq[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (64 * NW * i + (int)threadIdx.x < pieces) sq[i] = reinterpret_cast<const f32x4*>(a.part)[64 * NW * i + threadIdx.x];
      }
    }
    load(p[0], 0);
    if (EPI == EPI_RES && wave < OT) {
      const int n = min(column(wave, fq), a.N - 4);
      gw = *reinterpret_cast<const u16x4*>(a.gw + n);
#pragma unroll
      for (int m = 0; m < MB; ++m) res[m] = *reinterpret_cast<const u16x4*>(a.res + (int64_t)min(16 * m + frow, a.M - 1) * a.ldr + n);
    }
    if (EPI == EPI_ROPE && wave < OT) {
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const int64_t o = at[m] * 64 + (column(wave, fq) & 63);
        cs[m] = *reinterpret_cast<const f32x4*>(a.rcos + o);
        sn[m] = *reinterpret_cast<const f32x4*>(a.rsin + o);
      }
    }
    if constexpr (NORMED) {
      if (pieces > 0) {  // a thread always has the same 4 rows: 512 is a multiple of mp / 4
        f32x4 s = (sq[0] + sq[1]) + (sq[2] + sq[3]);
        for (int i = 64 * NW * AHEAD + threadIdx.x; i < pieces; i += 64 * NW) s += reinterpret_cast<const f32x4*>(a.part)[i];
        for (int d = quads; d < 64; d *= 2)
#pragma unroll
          for (int q = 0; q < 4; ++q) s[q] += __shfl_xor(s[q], d, 64);
        if (lane < quads) *reinterpret_cast<f32x4*>(&squares[wave][4 * lane]) = s;
      }
    }
    if constexpr (MERGE) {
      merge_row(a, merged);
      __syncthreads();
    }
  }
  auto multiply = [&](P& q) {
    if constexpr (MERGE) q.row_x(merged, k0, a.K, g);
    q.template multiply<MERGE>(acc, odd1, odd2);
    k0 += NW * STEP;
  };
  if constexpr (DEEP == 1) {
    if constexpr (EPI >= EPI_RES) multiply(p[0]);
    while (k0 - (HALF ? (l16 >> 3) * P::PIECE : 0) < a.K) {
      load(p[0], 0);
      multiply(p[0]);
    }
  } else {
    static_assert(DEEP == 2, "");
    if constexpr (EPI < EPI_RES) load(p[0], 0);
    for (int ku = wave * STEP; ku < a.K; ku += 2 * NW * STEP) {
      load(p[1], 1);
      multiply(p[0]);
      if (ku + NW * STEP >= a.K) break;
      load(p[0], 1);
      multiply(p[1]);
    }
  }
  // lane: columns 4 g .. + 3 of row l16 of every tile
  auto finish = [&](int m, int t) {
    const int row = 16 * m + frow, n = column(t, fq);
    float rinv = 1.f;
    if constexpr (NORMED) {
      if (a.part != nullptr) {
        float s = 0.f;
#pragma unroll
        for (int v = 0; v < NW; ++v) s += squares[v][min(row, a.mp - 1)];
        rinv = rsqrtf(s / (float)a.K + a.eps);
      }
    }
    auto sum = [&](int tile, int other, int col) {  // other: of the other half of the tile's columns
      f32x4 s;
      if constexpr (HALF) {  // of the waves 2 (lane / 16) and the next, then of all
        const int at = frow + 16 * ((fq >> 2) ^ other), v = lane >> 4;
        s = red[2 * v][tile][at] + red[2 * v][tile][at + 40] + red[2 * v + 1][tile][at] + red[2 * v + 1][tile][at + 40];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          s[q] += __shfl_xor(s[q], 16, 64);
          s[q] += __shfl_xor(s[q], 32, 64);
        }
      } else {
        const int at = other ? lane ^ 32 : lane;
        s = red[0][tile][at];
#pragma unroll
        for (int v = 1; v < NW; ++v) s += red[v][tile][at];
      }
      if (FP8) {
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q] *= a.scale[min(col + q, a.N - 1)];
      }
      if (NORMED) {
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q] *= rinv;
      } else if (a.bias != nullptr) {
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q] += bf16_to_f32(a.bias[min(col + q, a.N - 1)]);
      }
      return s;
    };
    f32x4 v = sum(t, 0, n);
    const int cols = GLU ? half : a.N;
    if constexpr (GLU) {
      const f32x4 up = sum(t + OT, 0, n + half);
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = v[q] / (1.f + expf(-v[q])) * up[q];
    }
    if constexpr (EPI == EPI_ROPE) {
      const f32x4 other = NT == 2 ? sum(1 - t, 0, n ^ 64) : sum(0, 1, n ^ 64);
      if (n < (a.nq + a.nkv) * 128) {
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = v[q] * cs[m][q] + (n & 64 ? other[q] : -other[q]) * sn[m][q];
      }
    }
    u16x4 o;
    if constexpr (EPI == EPI_RES) {
      float s = 0.f;
      u16x4 hs;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        hs[q] = f32_to_bf16(v[q] + bf16_to_f32(res[m][q]));
        const float h = bf16_to_f32(hs[q]);
        s += h * h;
        o[q] = f32_to_bf16(h * bf16_to_f32(gw[q]));
      }
      if constexpr (HALF) {
        s += __shfl_xor(s, 8, 64);
      } else {
        s += __shfl_xor(s, 16, 64);
        s += __shfl_xor(s, 32, 64);
      }
      if (n >= a.N || row >= a.mp) return;  // a whole tile, or rows that have no place
      if (HALF && lane >= 16) return;
      if (fq == 0) a.sums[(int64_t)(n / TC) * a.mp + row] = row < a.M ? s : 0.f;
      if (row < a.M) *reinterpret_cast<u16x4*>(a.h + (int64_t)row * a.N + n) = hs;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) o[q] = f32_to_bf16(v[q]);
    }
    if (row >= a.M || (HALF && lane >= 16)) return;
    if constexpr (EPI == EPI_HEAD) {
      if (n < a.N) *reinterpret_cast<f32x4*>(a.yf + (int64_t)row * a.N + n) = v;
      return;
    }
    if constexpr (EPI == EPI_ROPE) {
      const int head = n >> 7;
      if (head >= a.nq && slot[m] >= 0) {
        const int kv = head >= a.nq + a.nkv ? 1 : 0, hh = head - a.nq - kv * a.nkv;
        const int64_t blk = slot[m] / a.bs, off = slot[m] - blk * a.bs;
        *reinterpret_cast<u16x4*>(a.cache + (((blk * 2 + kv) * a.nkv + hh) * a.bs + off) * 128 + (n & 127)) = o;
      }
    }
    unsigned short* yp = a.y + (int64_t)row * cols + n;
    if (n + 4 <= cols && cols % 4 == 0) {
      *reinterpret_cast<u16x4*>(yp) = o;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (n + q < cols) yp[q] = o[q];
    }
  };
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    if (16 * m >= a.M) break;
    if (m) __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if constexpr (X8) {
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[m][2 * t][q] += __shfl_xor(acc[m][2 * t + 1][q], 8, 64);
      }
      red[wave][t][lane] = acc[m][AL * t];
    }
    __syncthreads();
    if (wave < OT) finish(m, wave);
  }
}

}  // namespace st

namespace {
// w [N, K] bf16, or e4m3 bytes with wscale fp32 [N], for M rows of K; -> whether w is e4m3
bool weights(st::Args& a, int64_t M, int64_t K, const at::Tensor& w, const c10::optional<at::Tensor>& wscale,
             const c10::optional<at::Tensor>& bias) {
  const bool fp8 = wscale.has_value() && wscale->defined();
  SXE_CHECK(w.is_cuda() && w.dim() == 2 && w.stride(1) == 1 && w.size(1) == K && (fp8 ? w.element_size() == 1 : w.scalar_type() == at::kBFloat16),
            "stream_gemm: w [N, K] bf16 or e4m3 bytes");
  check_beside(w, {wscale, bias});
  const int64_t N = w.size(0), unit = fp8 ? 16 : 8;
  SXE_CHECK(M >= 1 && M <= 32 && N > 0 && K > 0 && N < (1ll << 31) && K < (1ll << 31), "stream_gemm: 1 <= M <= 32");
  SXE_CHECK(K % unit == 0 && w.stride(0) % unit == 0 && reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0,
            "stream_gemm: K and the rows must allow 16-byte loads");
  SXE_CHECK(N % 4 == 0, "stream_gemm: N a multiple of 4");
  if (fp8) {
    SXE_CHECK(wscale->scalar_type() == at::kFloat && wscale->is_contiguous() && wscale->numel() == N, "stream_gemm: wscale fp32 [N]");
    a.scale = wscale->data_ptr<float>();
  }
  if (bias.has_value() && bias->defined()) {
    SXE_CHECK(bias->scalar_type() == at::kBFloat16 && bias->is_contiguous() && bias->numel() == N, "stream_gemm: bias bf16 [N]");
    a.bias = reinterpret_cast<const unsigned short*>(bias->data_ptr());
  }
  a.w = w.data_ptr();
  a.ldw = w.stride(0);
  a.M = M;
  a.N = N;
  a.K = K;
  a.mp = M <= 8 ? 8 : M <= 16 ? 16 : 32;
  return fp8;
}

// x [M, K] bf16 and w
bool operands(st::Args& a, const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& wscale,
              const c10::optional<at::Tensor>& bias) {
  check_beside(x, {w, wscale, bias});
  SXE_CHECK(x.scalar_type() == at::kBFloat16 && x.dim() == 2 && x.stride(1) == 1 && x.stride(0) % 8 == 0 &&
                reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0, "stream_gemm: bf16 x [M, K] in rows that allow 16-byte loads");
  a.x = reinterpret_cast<const unsigned short*>(x.data_ptr());
  a.ldx = x.stride(0);
  return weights(a, x.size(0), x.size(1), w, wscale, bias);
}

// the sums of squares that stream_gemm_res left for x's rows, or none: x is normed
void normed_by(st::Args& a, const at::Tensor& x, const c10::optional<at::Tensor>& part, double eps) {
  if (!part.has_value() || !part->defined()) return;
  check_beside(x, {*part});
  SXE_CHECK(part->scalar_type() == at::kFloat && part->dim() == 2 && part->is_contiguous() && part->size(1) == a.mp && part->size(0) > 0 &&
                part->size(0) < (1 << 24) && reinterpret_cast<uintptr_t>(part->data_ptr()) % 16 == 0, "stream_gemm: sums fp32 [tiles, rows]");
  a.part = part->data_ptr<float>();
  a.parts = part->size(0);
  a.eps = (float)eps;
}

// the kernel of M's rows and of weights that are read past the caches or through them: run(one or two blocks of rows, past the caches)
template <class F>
void by_rows(const st::Args& a, bool fp8, F run) {
  auto blocks = [&](auto nontemporal) {
    if (a.M <= 16) run(std::integral_constant<int, 1>{}, nontemporal);
    else run(std::integral_constant<int, 2>{}, nontemporal);
  };
  if (read_once((int64_t)a.N * a.K * (fp8 ? 1 : 2))) blocks(std::true_type{});
  else blocks(std::false_type{});
  SXE_LAUNCH_CHECK();
}

// tiles a workgroup: more of them for fewer reads of x, fewer for more workgroups. e4m3, 28672 x 4096, 8 rows, us at 1 / 2 / 4 tiles 32 / 29 /
// 35, 4096 x 4096 7.3 / 8.5 / 12.4; bf16, 4096 x 4096, 16 rows 9.7 / 12.9 / 16
int plain_tiles(const st::Args& a, bool fp8) { return (a.N + 15) / 16 >= 384 && (fp8 || a.M > 16) ? 2 : 1; }

// Half tiles where whole ones give half of the CUs no work: 2048 columns, up to 8 rows, a decode step of three layers of hidden 2048, ff 8192 with
// the head 189 / 180 us bf16, 148 / 142 e4m3; but 2560 columns (160 tiles) 230 / 236 and 180 / 187, 4096 (256) 367 / 380 and 266 / 284
bool halves(const st::Args& a) { return a.M <= 8 && a.N <= 2048; }

// A piece in flight behind the products of the one before, where a CU has one workgroup (more: `x8`) and a wave three or more pieces: bf16, us,
// so off / on: 4096 x 4096 1 row 10.6 / 9.4, 8 rows 10.5 / 9.5, 3072 x 8192 14.8 / 13.9, 4096 x 14336 23.4 / 22.5; but two pieces, 3072 x 2048
// 6.6 / 7.0; 16 rows and more, whose pieces are larger, 4096 x 14336 24.4 / 24.6, 5120 x
// 3072 15.4 / 17.8, and e4m3 4096 x 14336 16.2 / 16.9. Three pieces in flight are slower than two everywhere.
bool deep(const st::Args& a, bool fp8, int64_t workgroups) {
  return !fp8 && a.M <= 8 && workgroups <= 256 && a.K > 2 * st::NW * 128 * (halves(a) ? 2 : 1);
}

// The two halves of x side by side (see Piece) in whole tiles of up to 8 rows. e4m3, 8 rows, us, so off / on: 4096 x 14336 17.5 / 15.4, 3072 x 8192
// 10.7 / 9.7, 4096 x 4096 8.0 / 7.6, QKV of 6144 x 4096 10.4 / 9.9, gate and up of 28672 x 4096 27.5 / 26.3, 1 row 26.9 / 25.9. bf16 has twice the bytes
// in a piece then, which takes turns with the other form: 8 rows, 1 or 2 pieces in flight as `deep` has it / so, 6144 x 4096 14.7 / 13.8, 8192 x
// 4096 14.2 / 13.7, 3072 x 2048 6.8 / 6.5, but 4096 x 4096 9.4 / 10.0, 3072 x 8192 13.9 / 14.9, gate and up of 28672 x 4096 41.7 / 43.7
bool x8(const st::Args& a, bool fp8, int64_t workgroups) {
  return a.M <= 8 && (fp8 || (workgroups <= 512 && (workgroups > 256 || a.K <= 2 * st::NW * 128)));
}

template <int EPI>
void launch(const st::Args& a, bool fp8, int nt) {
  if constexpr (EPI != st::EPI_GLU && EPI != st::EPI_NGLU) {
    if (halves(a)) {
      const dim3 grid((a.N + 7) / 8);
      auto go = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(64 * st::NW), 0, cur_stream(), a); };
      by_rows(a, fp8, [&](auto, auto nontemporal) {
        constexpr bool ONCE = decltype(nontemporal)::value;
        if (deep(a, fp8, grid.x)) go(st::stream_gemm_kernel<false, 1, 1, EPI, ONCE, true, false, 2>);
        else fp8 ? go(st::stream_gemm_kernel<true, 1, 1, EPI, ONCE, true>) : go(st::stream_gemm_kernel<false, 1, 1, EPI, ONCE, true>);
      });
      return;
    }
  }
  const dim3 grid(((a.N + 15) / 16 + nt - 1) / nt);
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(64 * st::NW), 0, cur_stream(), a); };
  constexpr bool GLU = EPI == st::EPI_GLU || EPI == st::EPI_NGLU;
  by_rows(a, fp8, [&](auto mb, auto nontemporal) {
    constexpr int MB = decltype(mb)::value;
    constexpr bool ONCE = decltype(nontemporal)::value;
    if constexpr (GLU) {
      // a tile of gate and one of up; two of each leave a workgroup a CU, steps of three layers, us, two / one: 4096, 14336 1 row 358 / 340, 8
      // rows 372 / 355, 16 397 / 379, 32 467 / 455; 4096, 11008 32 rows 544 / 509; 3072, 8192 235 / 234, 300 / 297; 2048, 8192 180 / 177, 218 / 216
      if (MB == 1 && fp8 && x8(a, fp8, grid.x)) go(st::stream_gemm_kernel<true, 1, 2, EPI, ONCE, false, false, 1, true>);
      else fp8 ? go(st::stream_gemm_kernel<true, MB, 2, EPI, ONCE>) : go(st::stream_gemm_kernel<false, MB, 2, EPI, ONCE>);
    } else if (MB == 1 && x8(a, fp8, grid.x)) {
      if (fp8) nt == 2 ? go(st::stream_gemm_kernel<true, 1, 2, EPI, ONCE, false, false, 1, true>) : go(st::stream_gemm_kernel<true, 1, 1, EPI, ONCE, false, false, 1, true>);
      else go(st::stream_gemm_kernel<false, 1, 1, EPI, ONCE, false, false, 1, true>);
    } else if (MB == 1 && deep(a, fp8, grid.x)) {
      go(st::stream_gemm_kernel<false, 1, 1, EPI, ONCE, false, false, 2>);
    } else if (fp8) {
      nt == 2 ? go(st::stream_gemm_kernel<true, MB, 2, EPI, ONCE>) : go(st::stream_gemm_kernel<true, MB, 1, EPI, ONCE>);
    } else {
      nt == 2 ? go(st::stream_gemm_kernel<false, MB, 2, EPI, ONCE>) : go(st::stream_gemm_kernel<false, MB, 1, EPI, ONCE>);
    }
  });
}
}  // namespace

// (+ bias bf16 [N] or None); glu: w = gate | up
at::Tensor stream_gemm(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& wscale,
                       const c10::optional<at::Tensor>& bias, bool glu) {
  st::Args a{};
  const bool fp8 = operands(a, x, w, wscale, bias);
  SXE_CHECK(!glu || a.N % 32 == 0, "stream_gemm: gate and up of a multiple of 16 columns");
  c10::DeviceGuard gd(x.device());
  auto y = at::empty({a.M, glu ? a.N / 2 : a.N}, x.options());
  a.y = reinterpret_cast<unsigned short*>(y.data_ptr());
  if (glu) launch<st::EPI_GLU>(a, fp8, 2);
  else launch<st::EPI_PLAIN>(a, fp8, plain_tiles(a, fp8));
  return y;
}

// one row of attention's splits for x (part_ml given): [splits, 1, heads, dim] and (max, sum) [splits, 1, heads, 2], fp32; x is not read
static void split_row(st::Args& a, const at::Tensor& part_o, const at::Tensor& part_ml) {
  SXE_CHECK(part_o.scalar_type() == at::kFloat && part_o.dim() == 4 && part_o.is_contiguous() && part_ml.scalar_type() == at::kFloat &&
                part_ml.dim() == 4 && part_ml.is_contiguous() && part_o.size(0) > 0 && part_o.size(1) == 1 && part_o.size(3) % 4 == 0 &&
                part_ml.size(0) == part_o.size(0) && part_ml.size(1) == 1 && part_ml.size(2) == part_o.size(2) && part_ml.size(3) == 2 &&
                reinterpret_cast<uintptr_t>(part_o.data_ptr()) % 16 == 0, "stream_gemm_res: splits fp32 [S, 1, heads, dim], [S, 1, heads, 2]");
  a.po = part_o.data_ptr<float>();
  a.pml = part_ml.data_ptr<float>();
  a.splits = part_o.size(0);
  a.dim = part_o.size(3);
}

// h = res + x . w^T (+ bias), and what a product of rms_norm(h) * gw needs: -> [bf16(h * gw), h, sums of h^2 [tiles of 16 or 8 columns, rows]]
static std::vector<at::Tensor> residual(st::Args a, bool fp8, const at::Tensor& w, const at::Tensor& res, const at::Tensor& gw) {
  check_beside(w, {res, gw});
  SXE_CHECK(a.N % 16 == 0, "stream_gemm_res: whole tiles of 16 columns");
  SXE_CHECK(res.scalar_type() == at::kBFloat16 && res.dim() == 2 && res.size(0) == a.M && res.size(1) == a.N && res.stride(1) == 1 &&
                res.stride(0) % 4 == 0 && reinterpret_cast<uintptr_t>(res.data_ptr()) % 8 == 0, "stream_gemm_res: res bf16 [M, N]");
  SXE_CHECK(gw.scalar_type() == at::kBFloat16 && gw.is_contiguous() && gw.numel() == a.N && reinterpret_cast<uintptr_t>(gw.data_ptr()) % 8 == 0,
            "stream_gemm_res: gw bf16 [N]");
  c10::DeviceGuard gd(w.device());
  auto y = at::empty({a.M, a.N}, res.options()), h = at::empty({a.M, a.N}, res.options());
  auto sums = at::empty({a.N / (halves(a) ? 8 : 16), a.mp}, res.options().dtype(at::kFloat));
  a.y = reinterpret_cast<unsigned short*>(y.data_ptr());
  a.h = reinterpret_cast<unsigned short*>(h.data_ptr());
  a.sums = sums.data_ptr<float>();
  a.res = reinterpret_cast<const unsigned short*>(res.data_ptr());
  a.ldr = res.stride(0);
  a.gw = reinterpret_cast<const unsigned short*>(gw.data_ptr());
  if (a.po == nullptr) {
    launch<st::EPI_RES>(a, fp8, plain_tiles(a, fp8));
  } else {
    auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(a.N / 8), dim3(64 * st::NW), 0, cur_stream(), a); };
    fp8 ? go(st::stream_gemm_kernel<true, 1, 1, st::EPI_RES, false, true, true>) : go(st::stream_gemm_kernel<false, 1, 1, st::EPI_RES, false, true, true>);
    SXE_LAUNCH_CHECK();
  }
  return {y, h, sums};
}

std::vector<at::Tensor> stream_gemm_res(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& wscale,
                                        const c10::optional<at::Tensor>& bias, const at::Tensor& res, const at::Tensor& gw) {
  st::Args a{};
  const bool fp8 = operands(a, x, w, wscale, bias);
  return residual(a, fp8, w, res, gw);
}

// the same of one row that attention has left in splits: the flash-decoding merge runs before the product's own loads arrive. Every workgroup
// reads all splits, so small products only: a step of three layers of hidden 2048, ff 8192, 1000 / 3000 keys, us with a merge launch / so 173 /
// 168, 175 / 172, e4m3 134 / 130, 142 / 140; but hidden 4096 342 / 342, 355 / 358, 12000 keys 394 / 418
std::vector<at::Tensor> stream_gemm_res_splits(const at::Tensor& part_o, const at::Tensor& part_ml, const at::Tensor& w,
                                               const c10::optional<at::Tensor>& wscale, const at::Tensor& res, const at::Tensor& gw) {
  st::Args a{};
  check_beside(w, {part_o, part_ml});
  split_row(a, part_o, part_ml);
  const bool fp8 = weights(a, 1, part_o.size(2) * part_o.size(3), w, wscale, c10::nullopt);
  SXE_CHECK(a.K <= st::MERGE_K && halves(a), "stream_gemm_res_splits: w of up to 2048 x 2048");
  return residual(a, fp8, w, res, gw);
}

// of x . w^T / rms (sums of stream_gemm_res; None: x is normed): silu(gate) * up in bf16 (glu), or the product in fp32
at::Tensor stream_gemm_normed(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& wscale,
                              const c10::optional<at::Tensor>& part, double eps, bool glu) {
  st::Args a{};
  const bool fp8 = operands(a, x, w, wscale, c10::nullopt);
  normed_by(a, x, part, eps);
  SXE_CHECK(!glu || a.N % 32 == 0, "stream_gemm_normed: gate and up of a multiple of 16 columns");
  c10::DeviceGuard gd(x.device());
  auto y = at::empty({a.M, glu ? a.N / 2 : a.N}, glu ? x.options() : x.options().dtype(at::kFloat));
  if (glu) {
    a.y = reinterpret_cast<unsigned short*>(y.data_ptr());
    launch<st::EPI_NGLU>(a, fp8, 2);
  } else {
    a.yf = y.data_ptr<float>();
    launch<st::EPI_HEAD>(a, fp8, plain_tiles(a, fp8));
  }
  return y;
}

// the q, k and v of nq + 2 nkv heads of 128 (bf16 [M, heads * 128]) of x . w^T / rms, q and k rotated, k and v in the cache as well
at::Tensor stream_gemm_rope(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& wscale,
                            const c10::optional<at::Tensor>& part, double eps, const at::Tensor& cos_t, const at::Tensor& sin_t,
                            const at::Tensor& pos, const at::Tensor& slots, at::Tensor cache, int64_t nq, int64_t nkv) {
  st::Args a{};
  const bool fp8 = operands(a, x, w, wscale, c10::nullopt);
  normed_by(a, x, part, eps);
  check_beside(x, {cos_t, sin_t, pos, slots, cache});
  SXE_CHECK(nq > 0 && nkv > 0 && a.N == (nq + 2 * nkv) * 128, "stream_gemm_rope: w rows = (nq + 2 nkv) * 128");
  SXE_CHECK(cos_t.scalar_type() == at::kFloat && sin_t.scalar_type() == at::kFloat && cos_t.is_contiguous() && sin_t.is_contiguous() &&
                cos_t.size(-1) == 64 && sin_t.sizes() == cos_t.sizes() && reinterpret_cast<uintptr_t>(cos_t.data_ptr()) % 16 == 0 &&
                reinterpret_cast<uintptr_t>(sin_t.data_ptr()) % 16 == 0, "stream_gemm_rope: cos / sin fp32 [positions, 64]");
  SXE_CHECK(pos.scalar_type() == at::kLong && slots.scalar_type() == at::kLong && pos.is_contiguous() && slots.is_contiguous() &&
                pos.numel() == a.M && slots.numel() == a.M, "stream_gemm_rope: pos / slots int64 [M]");
  SXE_CHECK(cache.scalar_type() == at::kBFloat16 && cache.dim() == 5 && cache.is_contiguous() && cache.size(1) == 2 && cache.size(2) == nkv &&
                cache.size(4) == 128 && reinterpret_cast<uintptr_t>(cache.data_ptr()) % 8 == 0,
            "stream_gemm_rope: cache bf16 [blocks, 2, nkv, bs, 128]");
  c10::DeviceGuard gd(x.device());
  auto y = at::empty({a.M, a.N}, x.options());
  a.y = reinterpret_cast<unsigned short*>(y.data_ptr());
  a.rcos = cos_t.data_ptr<float>();
  a.rsin = sin_t.data_ptr<float>();
  a.pos = pos.data_ptr<int64_t>();
  a.slots = slots.data_ptr<int64_t>();
  a.cache = reinterpret_cast<unsigned short*>(cache.data_ptr());
  a.nq = nq;
  a.nkv = nkv;
  a.bs = cache.size(3);
  launch<st::EPI_ROPE>(a, fp8, plain_tiles(a, fp8));
  return y;
}

}  // namespace sxe

TORCH_LIBRARY_FRAGMENT(sxe, m) {
  m.def("stream_gemm(Tensor x, Tensor w, Tensor? wscale, Tensor? bias, bool glu) -> Tensor");
  m.def("stream_gemm_res(Tensor x, Tensor w, Tensor? wscale, Tensor? bias, Tensor res, Tensor gw) -> Tensor[]");
  m.def("stream_gemm_res_splits(Tensor part_o, Tensor part_ml, Tensor w, Tensor? wscale, Tensor res, Tensor gw) -> Tensor[]");
  m.def("stream_gemm_normed(Tensor x, Tensor w, Tensor? wscale, Tensor? part, float eps, bool glu) -> Tensor");
  m.def("stream_gemm_rope(Tensor x, Tensor w, Tensor? wscale, Tensor? part, float eps, Tensor cos, Tensor sin, Tensor pos, Tensor slots, "
        "Tensor(a!) cache, int nq, int nkv) -> Tensor");
}
TORCH_LIBRARY_IMPL(sxe, CUDA, m) {
  m.impl("stream_gemm", &sxe::stream_gemm);
  m.impl("stream_gemm_res", &sxe::stream_gemm_res);
  m.impl("stream_gemm_res_splits", &sxe::stream_gemm_res_splits);
  m.impl("stream_gemm_normed", &sxe::stream_gemm_normed);
  m.impl("stream_gemm_rope", &sxe::stream_gemm_rope);
}
