// Evoformer attention (DS4Sci_EvoformerAttention) on gfx950: O = softmax(Q K^T / sqrt(D) + bias1 +
// bias2) V over Q/K/V [B, N, L, H, D] with bias1 [B, N, 1, 1, L] (MSA row mask) and bias2
// [B, 1, H, L, L] (pair bias), head dims 32 / 64; backward with dQ, dK, dV, dbias1, dbias2.
//
// Reference: ops/deepspeed4science/evoformer_attn.py (CUTLASS kernels of csrc/deepspeed4science,
// not in the snapshot; kMax = 64 there too).
//
// What bounds it: with D = 32 the vector work of a score (exponent 8 clocks a wave's instruction, every other 4) beside two to four
// products of it, and how little of the two the waves of a SIMD overlap: at 1 x 128 x 384, 8 heads of 32, the vector units are busy 69 % of the
// forward's clocks, 53 % of dK-dV's and 34 % of dQ's (fewer than two waves a SIMD), the matrix cores 19, 29 and 16 %. Structure:
//  * swapped products (S^T = K Q^T: one lane = one query's scores, lane-local softmax) on v_mfma_f32_32x32x16_bf16, the
//    score accumulator reused as the B operand of O^T += V^T P^T; 128 queries (or keys) a workgroup, K / V (Q / dO) rows
//    direct to LDS, two slots;
//  * the scores' accumulator starts at the pair bias: packed once a call (pack_kernel: 2 x [H, L, L]) in the accumulator's order and the
//    type it came in. fp32 is packed in the products' domain, so that adding it costs no instruction, but 64 KB a tile of 128 x 128 and
//    row, which two of the N rows share where the grid is large (evo_single); bf16 is widened, and at heads of 32 scaled, per
//    score, at half the bytes and registers;
//  * the row mask of the kernels with queries on the lanes, and LSE and delta of those with keys on them, come in by one more product
//    each (of 8 k): three bf16 parts of the fp32 number times ones, 16 bytes a key, and a query and head. As rows of LDS floats they
//    cost four broadcast reads and 16 instructions a tile each; at 32 bytes a number they took dbias2 of heads of 64 from 136 to 142 us;
//  * the mask is -inf behind the last key, which is all the tail masking there is; rows behind L are read as zeros;
//  * dbias2 = sum of dS over the N rows stays in registers while a workgroup walks the rows; up to 384 keys of head dim 32 together
//    with dQ (dq_pair_kernel), else in a kernel of its own (dpair_kernel). Where that gives too few workgroups the rows are split and the
//    parts added up by a last pass. dbias1: per-lane sums, one atomic a key;
//  * delta = rowsum(dO O) is formed in the dQ kernels, which leave it and the LSE to the others.
// MSA row attention 1 x 128 x 384, 8 heads of 32, bf16 biases, MI355X, forward + backward: 278 us with biases added per score, dQ and
// dbias2 apart (forward 62, dQ 68, dK / dV 76, dbias2 79); 230 now (forward 55, dQ + dbias2 91, dK / dV 74). 8 heads of 64, the same
// way: 450 us; with fp32 packed biases and wide statistics 458; 423 now (forward 69, dQ 97, dK / dV 118, dbias2 130).
#include "sxe_gemm_loop.h"
#include <torch/library.h>
#include <type_traits>

namespace sxe {
namespace evo {
using namespace tl;
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

constexpr int NW = 4, QB = 32 * NW, KT = 64;  // waves, rows of a workgroup, streamed rows of a step
constexpr float FAR = 1.1e9f;                 // biases beyond it are this far: sums of them stay finite, exp() of them stays 0

__device__ const __attribute__((aligned(128))) unsigned short kZeroRow[64] = {0};

struct Args {
  const unsigned short *q, *k, *v, *dout, *o;
  const unsigned short* km;  // row mask as an MFMA operand [B N, Lp, 8]
  const float* mask;         // row mask [B N, Lp], log2 domain
  const void *pq, *pk;       // packed pair bias, lane = query / lane = key; null: none
  float* lse;                // [B N, H, Lp], log2 domain
  unsigned short* stats;     // -LSE and -delta as MFMA operands [B N, H, Lp, 2, 4]
  int B, N, L, H, Lp;
  float c;                   // log2(e) / sqrt(D)
};

// A number as four k of an operand: three bf16 parts, which is all of its 24 bits (inf and NaN in the first), and a zero
__device__ __forceinline__ u32x2 split(float x) {
  const unsigned short a = f32_to_bf16(x);
  const float hi = bf16_to_f32(a), rest = fabsf(hi) < INFINITY ? x - hi : 0.f;
  const unsigned short b = f32_to_bf16(rest);
  return u32x2{a | (unsigned)b << 16, f32_to_bf16(rest - bf16_to_f32(b))};
}
// Lane half hf holds k = 4 hf ..: a row of such parts, the same in both halves or zeros in the second, times `ones` is the number.
__device__ __forceinline__ u32x2 ones(int hf) { return hf ? u32x2{0u, 0u} : u32x2{0x3f803f80u, 0x3f80u}; }
__device__ __forceinline__ f32x16 mfma8(u32x2 a, u32x2 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(__builtin_bit_cast(i16x4, a), __builtin_bit_cast(i16x4, b), c, 0, 0, 0);
}
__device__ __forceinline__ float bounded(float x) {  // inf and NaN stay
  return x < -FAR && x > -INFINITY ? -FAR : x > FAR && x < INFINITY ? FAR : x;
}

// ------------------------------------------------------------------------------------ bias packing
// One launch for both. bias1 (null: none) [B N, L] -> mask [B N, Lp] * log2(e) and km [B N, Lp, 8] * sqrt(D), -inf behind L: the first
// mask_y rows of the grid, a row a workgroup. bias2 [B H, L, L] * scale -> 32 x 32 tiles in accumulator order, a workgroup each: element
// (tile (a, b), group i / W, lane, i % W) is the value of register i of that lane, W values of type P in 16 bytes. pq: lane =
// query of tile row a, registers = keys of b; pk (may be null): lane = key of tile row a, registers = queries of b. nt = Lp / 32.
// A row of either whose largest bias is far below zero (every key masked by a large finite number) is moved up to zero, one of
// bias1 far above it down: the softmax is the same, and its scores keep their fractions. (One of bias2 is read whole only where a
// tile's part of it lies there.)
constexpr float MASKED = 1e4f;
__device__ __forceinline__ float lift(float top) { return top < -MASKED && top > -INFINITY ? top : 0.f; }
template <typename P>
__global__ void __launch_bounds__(256) pack_kernel(const void* __restrict__ b1, int b1_bf16, float* __restrict__ mask,
                                                   unsigned short* __restrict__ km, int64_t rows, const P* __restrict__ b2,
                                                   P* __restrict__ pq, P* __restrict__ pk, int L, int nt, float root, float scale,
                                                   int mask_y) {
  auto value = [](auto t) { return sizeof(t) == 2 ? bf16_to_f32((unsigned short)t) : (float)t; };
  if ((int)blockIdx.y < mask_y) {
    __shared__ float tops[4];
    const int Lp = 32 * nt;
    for (int64_t row = blockIdx.y * (int64_t)gridDim.x + blockIdx.x; row < rows; row += mask_y * (int64_t)gridDim.x) {
      auto at = [&](int key) {
        if (key >= L) return -INFINITY;
        const int64_t i = row * L + key;
        const float x = b1 == nullptr ? 0.f : b1_bf16 ? bf16_to_f32(reinterpret_cast<const unsigned short*>(b1)[i])
                                                      : reinterpret_cast<const float*>(b1)[i];
        return x * LOG2E == -INFINITY ? -INFINITY : x;
      };
      float up = 0.f;
      if (b1 != nullptr) {
        float top = -INFINITY;
        for (int key = threadIdx.x; key < L; key += 256) top = fmaxf(top, at(key));
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) top = fmaxf(top, __shfl_xor(top, o));
        __syncthreads();  // of the row before
        if ((threadIdx.x & 63) == 0) tops[threadIdx.x >> 6] = top;
        __syncthreads();
        top = fmaxf(fmaxf(tops[0], tops[1]), fmaxf(tops[2], tops[3]));
        up = top > MASKED && top < INFINITY ? top : lift(top);
      }
      for (int key = threadIdx.x; key < Lp; key += 256) {
        const float x = bounded(at(key) - up);
        mask[row * Lp + key] = x * LOG2E;
        const u32x2 parts = split(x * root);
        *reinterpret_cast<u32x4*>(km + (row * Lp + key) * 8) = u32x4{parts[0], parts[1], 0u, 0u};
      }
    }
    return;
  }
  __shared__ float t[32][33];
  const int a = blockIdx.x / nt, b = blockIdx.x - a * nt;
  const int64_t bh = blockIdx.y - mask_y;
  const int r0 = threadIdx.x / 8, q = 32 * a + r0, k0 = 4 * (threadIdx.x % 8), k = 32 * b + k0;  // eight threads a row
  const P* row = b2 + bh * L * L + (int64_t)q * L;
  P x[4] = {0, 0, 0, 0};
  if (q < L) {
    typedef P P4 __attribute__((ext_vector_type(4)));
    if (L % 4 == 0 && reinterpret_cast<uintptr_t>(b2) % sizeof(P4) == 0) {
      if (k < L) {
        const P4 y = *reinterpret_cast<const P4*>(row + k);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = y[e];
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (k + e < L) x[e] = row[k + e];
    }
  }
  auto row_top = [](float y) {
#pragma unroll
    for (int o = 4; o > 0; o >>= 1) y = fmaxf(y, __shfl_xor(y, o));
    return y;
  };
  float top = -INFINITY;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (k + e < L) top = fmaxf(top, value(x[e]));
  float up = lift(row_top(top));
  if (up != 0.f) {  // (so q < L: the others' values are zeros)
    for (int i = threadIdx.x % 8; i < L; i += 8) top = fmaxf(top, value(row[i]));
    up = lift(row_top(top));
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) t[r0][k0 + e] = bounded(value(x[e]) - up) * scale;  // behind L they meet a mask of -inf, or zeros
  __syncthreads();
  // W values a thread; of 16 bits the first threads' are pq's, the others' pk's
  constexpr int W = 16 / sizeof(P), NT = 1024 / W;
  typedef typename std::conditional<W == 4, f32x4, u16x8>::type V;
  const int64_t tiles = bh * nt * nt;
  const int i = threadIdx.x % NT, g = i >> 6, hf = threadIdx.x >> 5 & 1, r = threadIdx.x & 31;
  auto store = [&](P* to, auto at) {
    V y;
#pragma unroll
    for (int e = 0; e < W; ++e) {
      const float z = at(acc_row(W * g + e, hf));
      if constexpr (W == 4) y[e] = z;
      else y[e] = f32_to_bf16(z);
    }
    *reinterpret_cast<V*>(to + i * W) = y;
  };
  if (NT == 256 || threadIdx.x < NT) store(pq + (tiles + blockIdx.x) * 1024, [&](int e) { return t[r][e]; });
  if (pk != nullptr && (NT == 256 || threadIdx.x >= NT)) store(pk + (tiles + (int64_t)b * nt + a) * 1024, [&](int e) { return t[e][r]; });
}

// waves a SIMD: what the registers allow without spills
template <int D>
constexpr int min_waves() { return D == 32 ? 3 : 2; }
// A lane's 16 biases of one 32 x 32 tile as they arrive, and where the accumulator of the scores starts with them
struct NoPair {};
template <typename P>
struct Bias {
  f32x16 x;
  __device__ __forceinline__ void load(const void* packed, int64_t tile, int lane) {
    const float* p = static_cast<const float*>(packed) + tile * 1024 + lane * 4;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 y = *reinterpret_cast<const f32x4*>(p + 256 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[4 * g + e] = y[e];
    }
  }
  template <int D>
  __device__ __forceinline__ f32x16 start() const { return x; }
};
template <>
struct Bias<unsigned short> {
  u32x4 v[2];
  __device__ __forceinline__ void load(const void* packed, int64_t tile, int lane) {
    const unsigned short* p = static_cast<const unsigned short*>(packed) + tile * 1024 + lane * 8;
#pragma unroll
    for (int g = 0; g < 2; ++g) v[g] = *reinterpret_cast<const u32x4*>(p + 512 * g);
  }
  template <int D>
  __device__ __forceinline__ f32x16 start() const {
    f32x16 x;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const unsigned y = v[i >> 3][(i & 7) >> 1];
      x[i] = __uint_as_float(i & 1 ? y & 0xffff0000u : y << 16);
      if (D == 32) x[i] *= 5.65685425f;  // sqrt(32); sqrt(64) is in the packed ones already
    }
    return x;
  }
};
template <>
struct Bias<NoPair> {
  __device__ __forceinline__ void load(const void*, int64_t, int) {}
  template <int D>
  __device__ __forceinline__ f32x16 start() const { return zero16(); }
};

// Rows of one (b, n), head h, that arrive 16 bytes a lane through a buffer resource: its length is the rows that are there, and what
// is read behind it is zeros. A lane's offset and a wave's resource stay, the base moves: nothing is left to do a load.
struct Rows {
  const unsigned short* x;
  int left;  // rows from x on
  __device__ __forceinline__ u32x4 resource(int most, int64_t rs) const {
    const uint64_t p = reinterpret_cast<uint64_t>(x);
    auto uniform = [](unsigned v) { return (unsigned)__builtin_amdgcn_readfirstlane(v); };
    return u32x4{uniform((unsigned)p), uniform((unsigned)(p >> 32) & 0xffffu), uniform((unsigned)(min(max(left, 0), most) * (int)rs) * 2u),
                 0x00020000u};
  }
};
// 1 KB: as gl::glds, from a resource
__device__ __forceinline__ void blds(unsigned off, const u32x4& res, unsigned dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(dst), "v"(off), "s"(res) : "memory", "m0");
}
// a lane's byte offset for KB i of a tile: 1024 / (2 D) rows each
template <int D>
__device__ __forceinline__ unsigned row_off(int i, int lane, int64_t rs) {
  const int r = i * (512 / D) + lane / (D / 8);
  return (unsigned)(r * (int)rs + (lane % (D / 8) ^ swz<D>(r)) * 8) * 2;
}

// Streamed rows: a step takes KT / NN rows of two arrays from each of NN of the N rows, 2 NN tiles in LDS. A wave's loads of a
// step are LOADS KB of one tile.
template <int D, int NN>
struct Stream {
  static constexpr int ROWS = KT / NN, TILE = ROWS * 2 * D, SLOT = 2 * NN * TILE, PART = TILE / 1024, LOADS = 2 * NN * PART / NW;
  static_assert(LOADS * NW == 2 * NN * PART && PART % LOADS == 0);
  Rows rows;
  unsigned off[LOADS];
  int at;
  int64_t rs;
  // x, y: the first rows of the first of the NN; step: elements from one to the next, the last of them `last`
  __device__ __forceinline__ void init(const unsigned short* x, const unsigned short* y, int64_t step, int last, int64_t rs_, int L, int w,
                                       int lane) {
    at = LOADS * w, rs = rs_;
    const int tile = at / PART;
    rows = {(tile & 1 ? y : x) + min(tile >> 1, last) * step, L};
#pragma unroll
    for (int i = 0; i < LOADS; ++i) off[i] = row_off<D>(at % PART + i, lane, rs);
  }
  // the next ROWS rows
  __device__ __forceinline__ void load(char* slot) {
    const unsigned dst = gl::lds_base() + (unsigned)(slot - lds) + at * 1024;
    const u32x4 res = rows.resource(ROWS, rs);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) blds(off[i], res, dst + i * 1024);
    rows.x += ROWS * rs, rows.left -= ROWS;
  }
};
// Said to be global memory: a load through a pointer chosen between the two would be a flat one, and every wait for LDS would
// wait for it, too.
template <typename T>
using Global = __attribute__((address_space(1))) T;
template <int D>
__device__ __forceinline__ void frags(bf16x8 (&f)[D / 16], const unsigned short* x, int64_t rs, int row, int L, int hf) {
#pragma unroll
  for (int t = 0; t < D / 16; ++t)
    f[t] = *reinterpret_cast<const Global<bf16x8>*>((row < L ? (const Global<unsigned short>*)(x + (int64_t)row * rs)
                                                             : (const Global<unsigned short>*)kZeroRow) + 16 * t + 8 * hf);
}

// where a lane's half of its row is in the row mask's operand rows [8]
__device__ __forceinline__ int lane_row(int lane) { return (lane & 31) * 8 + (lane >> 5) * 4; }
// log2-domain LSE from the reference exponent and the sum. Without a key, behind L, and where the pair bias alone puts every
// score of the row so far out that fp32 has no fractions there, it is large: the probabilities of the backward are 0.
__device__ __forceinline__ float row_lse(bool in, float m, float l) {
  return in && l > 0.f && fabsf(m) < 1.6e7f ? m + log2f(l) : 1e30f;
}

struct Place {
  int b, n, h, blk, bn, last;  // n, bn: the first of the workgroup's rows, n + last its last
  int64_t rs, base, row;       // row stride; element of (b, n, 0, h, 0); row of the [B N, H, Lp] arrays
  int64_t step, srow;          // from one n to the next
};
// The N rows that share a pair-bias tile are neighbours in the grid. (A row's blocks and heads on one XCD instead measured
// the same: K / V traffic does not bound these kernels.)
template <int D, int NN>
__device__ __forceinline__ Place place(const Args& a) {
  Place p;
  int idx = blockIdx.x;
  const int nn = (a.N + NN - 1) / NN;
  p.n = idx % nn * NN;
  idx /= nn;
  const int nblk = a.Lp / QB;
  p.blk = idx % nblk;
  idx /= nblk;
  p.h = idx % a.H;
  p.b = idx / a.H;
  p.bn = p.b * a.N + p.n;
  p.last = min(NN - 1, a.N - 1 - p.n);
  p.rs = (int64_t)a.H * D;
  p.step = a.L * p.rs;
  p.srow = (int64_t)a.H * a.Lp;
  p.base = p.bn * p.step + (int64_t)p.h * D;
  p.row = p.bn * p.srow + (int64_t)p.h * a.Lp;
  return p;
}

template <int D>
__device__ __forceinline__ void store_rows(const f32x16 (&acc)[D / 32], unsigned short* out, float s, int hf) {
#pragma unroll
  for (int t = 0; t < D / 32; ++t) store_acc_t(acc[t], out + 32 * t + 4 * hf, s);
}

// ------------------------------------------------------------------------------------ forward
// A workgroup takes the same 128 queries of NN of the N rows; a step is two 32 x 32 tiles a wave, one of each row (NN = 2) or two of
// the one. Which: evo_single.
template <int D, typename P, int NN>
__global__ void __launch_bounds__(256, 3) fwd_kernel(Args a, unsigned short* __restrict__ out) {
  using St = Stream<D, NN>;
  constexpr int SUB = 2 / NN;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, hf = lane >> 5;
  const Place p = place<D, NN>(a);
  const int q0 = p.blk * QB + 32 * w, q = q0 + r, nt32 = a.Lp / 32;
  const int64_t tiles = (((int64_t)p.b * a.H + p.h) * nt32 + q0 / 32) * nt32;
  const unsigned short* km = a.km + (int64_t)p.bn * a.Lp * 8;
  const int lr = lane_row(lane);
  bf16x8 qf[NN][D / 16];
  f32x16 o[NN][D / 32];
  float m[NN], l[NN];
#pragma unroll
  for (int i = 0; i < NN; ++i) {
    frags<D>(qf[i], a.q + p.base + min(i, p.last) * p.step, p.rs, q, a.L, hf);
#pragma unroll
    for (int t = 0; t < D / 32; ++t) o[i][t] = zero16();
    m[i] = -INFINITY, l[i] = 0.f;
  }
  const int n = (a.L + St::ROWS - 1) / St::ROWS;
  St st;
  st.init(a.k + p.base, a.v + p.base, p.step, p.last, p.rs, a.L, w, lane);
  Bias<P> bias[SUB];
  u32x2 kmf[2];
  auto load = [&](int t) {
    st.load(lds + (t & 1) * St::SLOT);
#pragma unroll
    for (int j = 0; j < SUB; ++j) bias[j].load(a.pq, tiles + SUB * t + j, lane);
#pragma unroll
    for (int u = 0; u < 2; ++u)
      kmf[u] = *reinterpret_cast<const u32x2*>(km + (int64_t)min(u % NN, p.last) * a.Lp * 8 + 256 * (SUB * t + u / NN) + lr);
  };
  load(0);
  wait_loads();
  __syncthreads();
  LaneOffs<D> lo;
  lo.init(lane);
  for (int t = 0; t < n; ++t) {
    const char* slot = lds + (t & 1) * St::SLOT;
    f32x16 s[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) s[u] = mfma8(kmf[u], ones(hf), bias[u / NN].template start<D>());
    if (t + 1 < n) load(t + 1);
    if (q0 < a.L) {
      constexpr bool EARLY = D == 32;  // else operands one product ahead: 167 registers, three waves a SIMD
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if constexpr (!EARLY) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t2 = 0; t2 < D / 16; ++t2)
          s[u] = mfma(row_at(slot + 2 * St::TILE * (u % NN) + 64 * D * (u / NN), lo.row[t2]), qf[u % NN][t2], s[u]);
      }
      bf16x8 vf[2][2][D / 32];  // read here where registers allow: in front of their products the wave would wait for each
      auto values = [&](int u, int s2) {
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
          vf[u][s2][dt] = tr_at(slot + 2 * St::TILE * (u % NN) + St::TILE + (32 * (u / NN) + 16 * s2) * 2 * D, lo.tr[dt]);
      };
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (EARLY || i < 1) values(i / 2, i % 2);
      if constexpr (D == 32) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < NN; ++i) {
        float mx = -INFINITY;
#pragma unroll
        for (int u = i; u < 2; u += NN)
#pragma unroll
          for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[u][e]);
        mx = fmaxf(mx, xor32(mx)) * a.c;
        const bool grow = mx > m[i] + 8.f;  // lazy rescale: p <= 2^8
        const float mnew = grow ? mx : m[i], mref = mnew == -INFINITY ? 0.f : mnew, alpha = fast_exp2(m[i] - mref);
        float ps = 0.f;
#pragma unroll
        for (int u = i; u < 2; u += NN)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            s[u][e] = fast_exp2(__builtin_fmaf(s[u][e], a.c, -mref));
            ps += s[u][e];
          }
        l[i] = l[i] * alpha + ps;
        m[i] = mnew;
        if (__any(grow)) {
          asm volatile("");  // stays a branch
#pragma unroll
          for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[i][dt][e] *= alpha;
        }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          if constexpr (!EARLY) {
            __builtin_amdgcn_sched_barrier(0);
            const int next = 2 * u + s2 + 1;
            if (next < 4) values(next / 2, next % 2);
          }
          const bf16x8 pb = acc_to_b(s[u], s2);
#pragma unroll
          for (int dt = 0; dt < D / 32; ++dt)
            o[u % NN][dt] = mfma(vf[u][s2][dt], pb, o[u % NN][dt]);
        }
    }
    wait_loads();
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < NN; ++i) {
    if (i > p.last) break;
    l[i] += xor32(l[i]);
    if (q < a.L) store_rows<D>(o[i], out + p.base + i * p.step + (int64_t)q * p.rs, l[i] > 0.f ? 1.f / l[i] : 0.f, hf);
    if (hf == 0) a.lse[p.row + i * p.srow + q] = row_lse(q < a.L, m[i], l[i]);
  }
}

// ----------------------------------------------------------------------------------------- dQ
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
// delta = rowsum(dO O) of a lane's query, and what the kernels with keys on the lanes read of it
template <int D>
__device__ __forceinline__ float row_delta(const bf16x8 (&df)[D / 16], const bf16x8 (&of)[D / 16]) {
  float delta = 0.f;
#pragma unroll
  for (int t = 0; t < D / 16; ++t)
#pragma unroll
    for (int e = 0; e < 8; e += 2)
      delta = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{df[t][e], df[t][e + 1]}, bf16x2{of[t][e], of[t][e + 1]}, delta, false);
  return delta + xor32(delta);
}
__device__ __forceinline__ void store_stats(const Args& a, int64_t row, float lse, float delta, int hf) {
  *reinterpret_cast<u32x2*>(a.stats + row * 8 + 4 * hf) = split(hf ? -delta : -lse / a.c);
}

template <int D, typename P, int NN>
__global__ void __launch_bounds__(256, 2) dq_kernel(Args a, unsigned short* __restrict__ dq) {
  using St = Stream<D, NN>;
  constexpr int SUB = 2 / NN;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, hf = lane >> 5;
  const Place p = place<D, NN>(a);
  const int q0 = p.blk * QB + 32 * w, q = q0 + r, nt32 = a.Lp / 32;
  const int64_t tiles = (((int64_t)p.b * a.H + p.h) * nt32 + q0 / 32) * nt32;
  const unsigned short* km = a.km + (int64_t)p.bn * a.Lp * 8;
  const int lr = lane_row(lane);
  bf16x8 qf[NN][D / 16], df[NN][D / 16];
  f32x16 acc[NN][D / 32];
  float lse[NN], delta[NN];
  const int n = (a.L + St::ROWS - 1) / St::ROWS;
  St st;
  st.init(a.k + p.base, a.v + p.base, p.step, p.last, p.rs, a.L, w, lane);
  Bias<P> bias[SUB];
  u32x2 kmf[2];
  auto load = [&](int t) {
    st.load(lds + (t & 1) * St::SLOT);
#pragma unroll
    for (int j = 0; j < SUB; ++j) bias[j].load(a.pq, tiles + SUB * t + j, lane);
#pragma unroll
    for (int u = 0; u < 2; ++u)
      kmf[u] = *reinterpret_cast<const u32x2*>(km + (int64_t)min(u % NN, p.last) * a.Lp * 8 + 256 * (SUB * t + u / NN) + lr);
  };
  load(0);
#pragma unroll
  for (int i = 0; i < NN; ++i) {
    const int64_t base = p.base + min(i, p.last) * p.step, row = p.row + min(i, p.last) * p.srow + q;
    bf16x8 of[D / 16];
    frags<D>(qf[i], a.q + base, p.rs, q, a.L, hf);
    frags<D>(df[i], a.dout + base, p.rs, q, a.L, hf);
    frags<D>(of, a.o + base, p.rs, q, a.L, hf);
    lse[i] = a.lse[row], delta[i] = row_delta<D>(df[i], of);
    store_stats(a, row, lse[i], delta[i], hf);
#pragma unroll
    for (int t = 0; t < D / 32; ++t) acc[i][t] = zero16();
  }
  wait_loads();
  __syncthreads();
  LaneOffs<D> lo;
  lo.init(lane);
  for (int t = 0; t < n; ++t) {
    const char* slot = lds + (t & 1) * St::SLOT;
    f32x16 s[2], dp[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) s[u] = mfma8(kmf[u], ones(hf), bias[u / NN].template start<D>());
    if (t + 1 < n) load(t + 1);
    if (q0 < a.L) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const char* kt = slot + 2 * St::TILE * (u % NN) + 64 * D * (u / NN);
        dp[u] = zero16();
#pragma unroll
        for (int t2 = 0; t2 < D / 16; ++t2) {
          s[u] = mfma(row_at(kt, lo.row[t2]), qf[u % NN][t2], s[u]);
          dp[u] = mfma(row_at(kt + St::TILE, lo.row[t2]), df[u % NN][t2], dp[u]);
        }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int e = 0; e < 16; ++e) s[u][e] = fast_exp2(__builtin_fmaf(s[u][e], a.c, -lse[u % NN])) * (dp[u][e] - delta[u % NN]);  // dS^T
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const bf16x8 db = acc_to_b(s[u], s2);
#pragma unroll
          for (int dt = 0; dt < D / 32; ++dt)
            acc[u % NN][dt] = mfma(tr_at(slot + 2 * St::TILE * (u % NN) + (32 * (u / NN) + 16 * s2) * 2 * D, lo.tr[dt]), db, acc[u % NN][dt]);
        }
      }
    }
    wait_loads();
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < NN; ++i)
    if (i <= p.last && q < a.L) store_rows<D>(acc[i], dq + p.base + i * p.step + (int64_t)q * p.rs, a.c * LN2, hf);
}

// -------------------------------------------------------------------------------------- dK, dV
// Keys on the lanes; Q / dO tiles and their -LSE / -delta rows stream by.
template <int D, int NN>
struct QueryStream : Stream<D, NN> {
  using S = Stream<D, NN>;
  static constexpr int SLOT = S::SLOT + 1024;  // KT rows of both statistics, 16 bytes each
  const unsigned short* stat;
  unsigned soff;
  // base: element of the first row and head; row: of the [B N, H, Lp] arrays
  __device__ __forceinline__ void init(const Args& a, int64_t base, int64_t row, int64_t step, int64_t srow, int last, int64_t rs, int w,
                                       int lane) {
    S::init(a.q + base, a.dout + base, step, last, rs, a.L, w, lane);
    stat = a.stats + row * 8;
    soff = 16u * (unsigned)(lane % S::ROWS + min(lane / S::ROWS, last) * srow);
  }
  __device__ __forceinline__ void load(char* slot, int w) {
    S::load(slot);
    if (w == 0) gl::glds(soff, stat, gl::lds_base() + (unsigned)(slot - lds) + S::SLOT);
    stat += S::ROWS * 8;
  }
};

// The operands of tile u of a slot, 32 queries, and its products: S - LSE and dP - delta [query][key], keys on the lanes (queries behind
// L: LSE large, so P = 0)
template <int D, int NN>
struct QueryTile {
  using St = QueryStream<D, NN>;
  u32x4 stats;
  bf16x8 q[D / 16], d[D / 16];
  __device__ __forceinline__ void read(const char* slot, int u, const LaneOffs<D>& lo, int r) {
    const char* tile = slot + 2 * St::TILE * (u % NN) + 64 * D * (u / NN);
    stats = *reinterpret_cast<const u32x4*>(slot + St::S::SLOT + 512 * u + 16 * r);
#pragma unroll
    for (int t = 0; t < D / 16; ++t) {
      q[t] = row_at(tile, lo.row[t]);
      d[t] = row_at(tile + St::TILE, lo.row[t]);
    }
  }
  __device__ __forceinline__ void products(f32x16& pr, f32x16& ds, const bf16x8 (&kf)[D / 16], const bf16x8 (&vf)[D / 16],
                                           const f32x16& bias, int hf) const {
    pr = mfma8(u32x2{stats[0], stats[1]}, ones(hf), bias);
    ds = mfma8(u32x2{stats[2], stats[3]}, ones(hf), zero16());
#pragma unroll
    for (int t = 0; t < D / 16; ++t) {
      pr = mfma(q[t], kf[t], pr);
      ds = mfma(d[t], vf[t], ds);
    }
  }
};
__device__ __forceinline__ void score_grads(f32x16& pr, f32x16& ds, float mask, float c) {
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    pr[i] = fast_exp2(__builtin_fmaf(pr[i], c, mask));
    ds[i] *= pr[i];
  }
}

template <int D, typename P, int NN, bool DB1>
__global__ void __launch_bounds__(256, (NN == 1 ? min_waves<D>() : 2)) dkdv_kernel(Args a, unsigned short* __restrict__ dk,
                                                                     unsigned short* __restrict__ dv, float* __restrict__ db1) {
  using St = QueryStream<D, NN>;
  constexpr int SUB = 2 / NN;
  constexpr bool ONE = NN == 1 && (D == 32 || std::is_same<P, float>::value);  // a tile after the other, where registers are short
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, hf = lane >> 5;
  const Place p = place<D, NN>(a);
  const int k0 = p.blk * QB + 32 * w, key = k0 + r, nt32 = a.Lp / 32;
  const int64_t tiles = (((int64_t)p.b * a.H + p.h) * nt32 + k0 / 32) * nt32;
  bf16x8 kf[NN][D / 16], vf[NN][D / 16];
  f32x16 dka[NN][D / 32], dva[NN][D / 32];
  float mask[NN], b1acc[NN];
  St st;
  st.init(a, p.base, p.row, p.step, p.srow, p.last, p.rs, w, lane);
  Bias<P> bias[SUB];
  auto load = [&](int t) {
    st.load(lds + (t & 1) * St::SLOT, w);
#pragma unroll
    for (int j = 0; j < SUB; ++j) bias[j].load(a.pk, tiles + SUB * t + j, lane);
  };
  load(0);
#pragma unroll
  for (int i = 0; i < NN; ++i) {
    const int64_t base = p.base + min(i, p.last) * p.step;
    frags<D>(kf[i], a.k + base, p.rs, key, a.L, hf);
    frags<D>(vf[i], a.v + base, p.rs, key, a.L, hf);
    mask[i] = a.mask[(int64_t)(p.bn + min(i, p.last)) * a.Lp + key];
    b1acc[i] = 0.f;
#pragma unroll
    for (int t = 0; t < D / 32; ++t) dka[i][t] = dva[i][t] = zero16();
  }
  const int n = (a.L + St::ROWS - 1) / St::ROWS;
  wait_loads();
  __syncthreads();
  LaneOffs<D> lo;
  lo.init(lane);
  for (int t = 0; t < n; ++t) {
    const char* slot = lds + (t & 1) * St::SLOT;
    auto products = [&](int u, f32x16& pr, f32x16& ds) __attribute__((always_inline)) {
      QueryTile<D, NN> x;
      x.read(slot, u, lo, r);
      __builtin_amdgcn_sched_barrier(0);
      x.products(pr, ds, kf[u % NN], vf[u % NN], bias[u / NN].template start<D>(), hf);
    };
    auto sums = [&](int u, f32x16& pr, f32x16& ds) __attribute__((always_inline)) {
      const char* tile = slot + 2 * St::TILE * (u % NN) + 64 * D * (u / NN);
      bf16x8 df[2][D / 32], qf[2][D / 32];  // read here: in front of their products the wave would wait for each
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt) {
          df[s2][dt] = tr_at(tile + St::TILE + 32 * D * s2, lo.tr[dt]);
          qf[s2][dt] = tr_at(tile + 32 * D * s2, lo.tr[dt]);
        }
      if constexpr (D == 32) __builtin_amdgcn_sched_barrier(0);
      score_grads(pr, ds, mask[u % NN], a.c);
      if constexpr (DB1) {
#pragma unroll
        for (int i = 0; i < 16; ++i) b1acc[u % NN] += ds[i];
      }
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        const bf16x8 pb = acc_to_b(pr, s2), db = acc_to_b(ds, s2);
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt) {
          dva[u % NN][dt] = mfma(df[s2][dt], pb, dva[u % NN][dt]);  // dV^T += dO^T P
          dka[u % NN][dt] = mfma(qf[s2][dt], db, dka[u % NN][dt]);  // dK^T += Q^T dS
        }
      }
    };
    if constexpr (ONE) {
      if (t + 1 < n) st.load(lds + (t + 1 & 1) * St::SLOT, w);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        f32x16 pr, ds;
        products(u, pr, ds);
        if (t + 1 < n) bias[u].load(a.pk, tiles + 2 * (t + 1) + u, lane);
        if (k0 < a.L) sums(u, pr, ds);
      }
    } else {
      f32x16 pr[2], ds[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) products(u, pr[u], ds[u]);
      if (t + 1 < n) load(t + 1);
      if (k0 < a.L) {
#pragma unroll
        for (int u = 0; u < 2; ++u) sums(u, pr[u], ds[u]);
      }
    }
    wait_loads();
    __syncthreads();
  }
  if (key >= a.L) return;
#pragma unroll
  for (int i = 0; i < NN; ++i) {
    if (i > p.last) break;
    if constexpr (DB1) {
      b1acc[i] += xor32(b1acc[i]);
      if (hf == 0) atomicAdd(db1 + (int64_t)(p.bn + i) * a.L + key, b1acc[i]);
    }
    store_rows<D>(dka[i], dk + p.base + i * p.step + (int64_t)key * p.rs, a.c * LN2, hf);
    store_rows<D>(dva[i], dv + p.base + i * p.step + (int64_t)key * p.rs, 1.f, hf);
  }
}

// ------------------------------------------------------------------------------ dQ and dbias2 together
// A workgroup has 32 QW queries of one (b, h) and all keys (KEYS of them are Lp), and walks rows_per of the N rows: QW x KG waves, each 32 queries x J tiles
// of 32 keys, whose biases and dbias2 stay in its registers; the scores are formed once for both gradients. The KG partial sums of
// dQ go through LDS, and are added up while the next row's scores are formed. part: fp32 [parts, B H, tiles, tiles, 1024], the
// packed order of pq. Grid: (query tiles * B H, parts), heads fastest.
template <int J>
struct DqPair {
  static constexpr int D = 32, QW = 2, KG = 4, NWG = QW * KG, QUERIES = 32 * QW, KEYS = 32 * KG * J, ROWS = KEYS * 2 * D, QROWS = QUERIES * 2 * D;
  static constexpr int SLOT = 2 * ROWS + 3 * QROWS, RED = NWG * 4096;  // K, V, Q, dO, O
  static constexpr int NR = 2 * SLOT + 2 * RED <= 160 * 1024 ? 2 : 1, LDS = 2 * SLOT + NR * RED;
  static_assert(NWG == 8 && LDS <= 160 * 1024);
};
template <int J, typename P>
__global__ void __launch_bounds__(512, 2) dq_pair_kernel(Args a, unsigned short* __restrict__ dq, float* __restrict__ part, int rows_per) {
  using C = DqPair<J>;
  constexpr int D = 32, QW = C::QW, KG = C::KG;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), hf = lane >> 5;
  const int qw = w % QW, kg = w / QW, nt32 = a.Lp / 32, nbh = a.B * a.H, bh = blockIdx.x % nbh, h = bh % a.H, b = bh / a.H;
  const int qb = C::QUERIES * (blockIdx.x / nbh), q = qb + 32 * qw + (lane & 31), t0 = kg * J;
  const int64_t rs = (int64_t)a.H * D, step = a.L * rs;
  const int n0 = blockIdx.y * rows_per, n1 = min(a.N, n0 + rows_per);
  const int64_t tiles = ((int64_t)bh * nt32 + qb / 32 + qw) * nt32 + t0;
  const unsigned lbase = gl::lds_base();
  f32x16 bias[J], dpair[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    Bias<P> packed;
    packed.load(a.pq, tiles + j, lane);
    bias[j] = packed.template start<D>();
    dpair[j] = zero16();
  }
  u32x2 kmn[J];
  float lsen;
  // A wave loads K's or V's rows 16 (w / 2) .. of every 64, 16 rows of Q or dO and, the first waves, 16 of O
  constexpr int QP = C::QUERIES / 16;
  const int64_t first = ((int64_t)b * a.N + n0) * step + (int64_t)h * D;
  Rows kv = {(w & 1 ? a.v : a.k) + first, a.L}, qd = {(w < QP ? a.q : a.dout) + first + qb * rs, a.L - qb}, oo = {a.o + first + qb * rs, a.L - qb};
  const unsigned koff = row_off<D>(w / 2, lane, rs), qoff = row_off<D>(w % QP, lane, rs);
  const float* lsep = a.lse + (((int64_t)b * a.N + n0) * a.H + h) * a.Lp + q;
  const unsigned short* kmp = a.km + (((int64_t)b * a.N + n0) * a.Lp + 32 * t0) * 8 + lane_row(lane);
  auto load = [&](int n) {
    const unsigned dst = lbase + ((n - n0) & 1) * C::SLOT;
    const u32x4 kres = kv.resource(C::KEYS, rs), qres = qd.resource(C::QUERIES, rs);
#pragma unroll
    for (int i = 0; i < C::KEYS / 64; ++i)
      blds(koff + i * (unsigned)(128 * rs), kres, dst + (w & 1) * C::ROWS + (w / 2 + 4 * i) * 1024);
    if (w < 2 * QP) blds(qoff, qres, dst + 2 * C::ROWS + w * 1024);
    if (w < QP) blds(qoff, oo.resource(C::QUERIES, rs), dst + 2 * C::ROWS + (2 * QP + w) * 1024);
    lsen = *lsep;
#pragma unroll
    for (int j = 0; j < J; ++j) kmn[j] = *reinterpret_cast<const u32x2*>(kmp + 256 * j);
    kv.x += step, qd.x += step, oo.x += step, lsep += (int64_t)a.H * a.Lp, kmp += a.Lp * 8;
  };
  // dQ of row n: four values a thread
  auto reduce = [&](int n) {
    if (threadIdx.x >= 256 * QW) return;
    const int qt = threadIdx.x >> 8, i = threadIdx.x & 255, qq = qb + 32 * qt + (i & 31);
    const char* red = lds + 2 * C::SLOT + (C::NR == 2 ? (n - n0) & 1 : 0) * C::RED + 16 * i;
    f32x4 x = *reinterpret_cast<const f32x4*>(red + qt * 4096);
#pragma unroll
    for (int g = 1; g < KG; ++g) x += *reinterpret_cast<const f32x4*>(red + (g * QW + qt) * 4096);
    if (qq >= a.L) return;
    const float s = a.c * LN2;
    const unsigned lo = gl::pack(x[0] * s, x[1] * s), hi = gl::pack(x[2] * s, x[3] * s);
    unsigned short* to = dq + ((int64_t)b * a.N + n) * step + (int64_t)h * D + (int64_t)qq * rs + 8 * (i >> 6) + 4 * (i >> 5 & 1);
    *reinterpret_cast<unsigned long long*>(to) = (unsigned long long)lo | (unsigned long long)hi << 32;
  };
  LaneOffs<D> lo;
  lo.init(lane);
  if (n0 < n1) load(n0);
  wait_loads();
  __syncthreads();
  for (int n = n0; n < n1; ++n) {
    const char* slot = lds + ((n - n0) & 1) * C::SLOT;
    const char *kt = slot + t0 * 2048, *qt = slot + 2 * C::ROWS + qw * 2048;
    bf16x8 qf[2], df[2], of[2];
    u32x2 km[J];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      df[t] = row_at(qt + C::QROWS, lo.row[t]);
      of[t] = row_at(qt + 2 * C::QROWS, lo.row[t]);
      qf[t] = row_at(qt, lo.row[t]);
    }
    const float lse = lsen, delta = row_delta<D>(df, of);
    const u32x2 nd = split(-delta);
    if (kg == 0) {
      const int64_t row = (((int64_t)b * a.N + n) * a.H + h) * a.Lp + q;
      *reinterpret_cast<u32x2*>(a.stats + row * 8 + 4 * hf) = hf ? nd : split(-lse / a.c);
    }
#pragma unroll
    for (int j = 0; j < J; ++j) km[j] = kmn[j];
    if (n + 1 < n1) load(n + 1);
    if (n > n0) reduce(n - 1);
    f32x16 acc = zero16();
    // operands are read one use ahead: left to itself the compiler reads each in front of its product and waits
    bf16x8 kf[2], vf[2], tr[2];
    auto read = [&](int j) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        kf[t] = row_at(kt + 2048 * j, lo.row[t]);
        vf[t] = row_at(kt + C::ROWS + 2048 * j, lo.row[t]);
      }
    };
    read(0);
#pragma unroll
    for (int j = 0; j < J; ++j) {
      f32x16 s = mfma8(km[j], ones(hf), bias[j]), dp = mfma8(ones(hf), nd, zero16());
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        s = mfma(kf[t], qf[t], s);
        dp = mfma(vf[t], df[t], dp);
      }
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) tr[s2] = tr_at(kt + 2048 * j + 1024 * s2, lo.tr[0]);
      if (j + 1 < J) read(j + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = fast_exp2(__builtin_fmaf(s[e], a.c, -lse));
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        s[e] *= dp[e];  // dS^T
        dpair[j][e] += s[e];
      }
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) acc = mfma(tr[s2], acc_to_b(s, s2), acc);
    }
    if constexpr (C::NR == 1) __syncthreads();
    char* red = lds + 2 * C::SLOT + (C::NR == 2 ? (n - n0) & 1 : 0) * C::RED + w * 4096 + 16 * lane;
#pragma unroll
    for (int g = 0; g < 4; ++g) *reinterpret_cast<f32x4*>(red + 1024 * g) = f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
    wait_loads();
    __syncthreads();
  }
  if (n0 < n1) reduce(n1 - 1);
  float* out = part + ((int64_t)blockIdx.y * nbh * nt32 * nt32 + tiles) * 1024 + 4 * lane;
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(out + 1024 * j + 256 * g) = f32x4{dpair[j][4 * g], dpair[j][4 * g + 1], dpair[j][4 * g + 2], dpair[j][4 * g + 3]};
}

// packed parts -> dbias2 [B H, L, L]; a 32 x 32 tile a workgroup, grid (tiles * tiles, B H) with tiles = ceil(L / 32)
template <typename T>
__global__ void __launch_bounds__(256) dpair_tiles_kernel(const float* __restrict__ part, T* __restrict__ out, int64_t stride, int parts, int L,
                                                          int nt32) {
  __shared__ float t[32][33];
  const int tl = (L + 31) / 32, ta = blockIdx.x / tl, tb = blockIdx.x - ta * tl, g = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const float* src = part + (((int64_t)blockIdx.y * nt32 + ta) * nt32 + tb) * 1024 + 4 * threadIdx.x;
  f32x4 x = {0.f, 0.f, 0.f, 0.f};
  for (int p = 0; p < parts; ++p) x += *reinterpret_cast<const f32x4*>(src + p * stride);
#pragma unroll
  for (int e = 0; e < 4; ++e) t[lane & 31][acc_row(4 * g + e, lane >> 5)] = x[e];
  __syncthreads();
  for (int i = threadIdx.x; i < 1024; i += 256) {
    const int q = 32 * ta + i / 32, k = 32 * tb + i % 32;
    if (q >= L || k >= L) continue;
    T* to = out + ((int64_t)blockIdx.y * L + q) * L + k;
    if constexpr (sizeof(T) == 2) *to = f32_to_bf16(t[i / 32][i % 32]);
    else *to = t[i / 32][i % 32];
  }
}

// -------------------------------------------------------------------------------------- dbias2
// A workgroup holds dbias2 of 64 queries x 128 keys of one (b, h) and walks rows_per of the N rows. part: fp32 [parts,
// B H, L, L]. Grid: (query tiles * key blocks * B H, parts), heads fastest: with 8 heads an XCD walks one head's rows
// (82 us at 128 x 384 x 8 heads of 32; 103 us with the tiles of a head spread over the XCDs).
template <int D, typename P>
__global__ void __launch_bounds__(256, (min_waves<D>())) dpair_kernel(Args a, float* __restrict__ part, int rows_per) {
  using St = QueryStream<D, 1>;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, hf = lane >> 5;
  const int nqt = (a.L + KT - 1) / KT, nkb = a.Lp / QB, nt32 = a.Lp / 32;
  const int nbh = a.B * a.H, bh = blockIdx.x % nbh, kb = blockIdx.x / nbh % nkb, qt = blockIdx.x / nbh / nkb;
  const int h = bh % a.H, b = bh / a.H;
  const int k0 = kb * QB + 32 * w, key = k0 + r, q0 = qt * KT;
  const int64_t rs = (int64_t)a.H * D;
  f32x16 bias[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    Bias<P> packed;
    packed.load(a.pk, ((int64_t)bh * nt32 + k0 / 32) * nt32 + 2 * qt + j, lane);
    bias[j] = packed.template start<D>();
  }
  const int n0 = blockIdx.y * rows_per, n1 = min(a.N, n0 + rows_per);
  f32x16 acc[2] = {zero16(), zero16()};
  bf16x8 kf[D / 16], vf[D / 16], kn[D / 16], vn[D / 16];
  float mask = 0.f, maskn = 0.f;
  auto load = [&](int n, char* slot) {
    const int bn = b * a.N + n;
    const int64_t base = (int64_t)bn * a.L * rs + (int64_t)h * D;
    St st;
    st.init(a, base, ((int64_t)bn * a.H + h) * a.Lp, 0, 0, 0, rs, w, lane);
    st.rows.x += q0 * rs, st.rows.left -= q0, st.stat += q0 * 8;
    st.load(slot, w);
    frags<D>(kn, a.k + base, rs, key, a.L, hf);
    frags<D>(vn, a.v + base, rs, key, a.L, hf);
    maskn = a.mask[(int64_t)bn * a.Lp + key];
  };
  if (n0 < n1) load(n0, lds);
  wait_loads();
  __syncthreads();
  LaneOffs<D> lo;
  lo.init(lane);
  for (int n = n0; n < n1; ++n) {
    const int cur = (n - n0) & 1;
#pragma unroll
    for (int t = 0; t < D / 16; ++t) {
      kf[t] = kn[t];
      vf[t] = vn[t];
    }
    mask = maskn;
    if (n + 1 < n1) load(n + 1, lds + (cur ^ 1) * St::SLOT);
    if (k0 < a.L) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        f32x16 pr, ds;
        QueryTile<D, 1> x;
        x.read(lds + cur * St::SLOT, j, lo, r);
        x.products(pr, ds, kf, vf, bias[j], hf);
        score_grads(pr, ds, mask, a.c);
        acc[j] += ds;
      }
    }
    wait_loads();
    __syncthreads();
  }
  if (key >= a.L) return;
  float* out = part + ((int64_t)blockIdx.y * a.B * a.H + bh) * a.L * a.L + key;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int qq = q0 + 32 * j + acc_row(i, hf);
      if (qq < a.L) out[(int64_t)qq * a.L] = acc[j][i];
    }
}

template <typename T>
__global__ void __launch_bounds__(256) dpair_sum_kernel(const float* __restrict__ part, T* __restrict__ out, int64_t n, int parts) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n; i += gridDim.x * 256ll) {
    float s = 0.f;
    for (int p = 0; p < parts; ++p) s += part[p * n + i];
    if constexpr (sizeof(T) == 2) out[i] = f32_to_bf16(s);
    else out[i] = s;
  }
}

}  // namespace evo

// ------------------------------------------------------------------------------- host side
// 16-byte aligned storage (a view of a larger tensor may start anywhere)
static at::Tensor evo_aligned(const at::Tensor& t) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 ? t.clone() : t;
}
static bool evo_has(const c10::optional<at::Tensor>& t) { return t.has_value() && t->defined(); }

struct EvoCall {
  evo::Args a{};
  at::Tensor q, k, v;  // keep what the pointers look at
  at::ScalarType pair = at::ScalarType::Undefined;  // of the packed bias2
};

static EvoCall evo_call(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v) {
  SXE_CHECK(q.dim() == 5 && q.sizes() == k.sizes() && q.sizes() == v.sizes(), "evoformer: q/k/v [B, N, L, H, D]");
  for (const at::Tensor* t : {&q, &k, &v})
    SXE_CHECK(t->is_contiguous() && t->scalar_type() == at::kBFloat16, "evoformer: contiguous bf16 q/k/v");
  const int D = q.size(4);
  SXE_CHECK(D == 32 || D == 64, "evoformer: head dim 32 or 64");
  EvoCall c;
  evo::Args& a = c.a;
  a.B = q.size(0);
  a.N = q.size(1);
  a.L = q.size(2);
  a.H = q.size(3);
  a.Lp = (a.L + evo::QB - 1) / evo::QB * evo::QB;
  a.c = mf::LOG2E / std::sqrt((float)D);
  c.q = evo_aligned(q);
  c.k = evo_aligned(k);
  c.v = evo_aligned(v);
  a.q = reinterpret_cast<const unsigned short*>(c.q.data_ptr());
  a.k = reinterpret_cast<const unsigned short*>(c.k.data_ptr());
  a.v = reinterpret_cast<const unsigned short*>(c.v.data_ptr());
  return c;
}

static int evo_grid(const evo::Args& a, int rows) { return a.B * ((a.N + rows - 1) / rows) * a.H * (a.Lp / evo::QB); }

// Whether the grid is small enough for one of the N rows a workgroup where two could share the pair bias: three workgroups of two rows a
// CU or fewer are better off as twice as many. It matters for fp32 biases of heads of 32, and for dQ of heads of 64; bf16 biases are
// half the bytes and need fewer registers, and one row at a time is the better form of everything else. us, two rows of fp32 packed
// biases / one of bf16 ones, heads of 32 (8 of them; workgroups of two rows): 20 x 500 (320) forward 31.2 / 27.2, backward 88 / 83;
// 128 x 384 (1536) 61.9 / 58.0, dK / dV 79.8 / 74.5; 100 x 500 (1600) 95 / 78, 318 / 299; 200 x 512 165 / 149, 602 / 568; 256 x 512
// (4096) 195 / 194, 828 / 820; but 256 x 400 143 / 147, 605 / 612. Heads of 64, forward, two rows / one: 128 x 384 75.6 / 69, 256 x 512
// 254 / 238, fp32 biases 77 / 72, 257 / 264; dQ 97 / 101, 314 / 336, but 21 x 428 (336) 35.5 / 31.4. No pair bias: 200 x 450, 4 heads
// of 32, forward and backward 230 / 208, 512 x 64 74.5 / 72.1, 256 x 512 582 / 581, heads of 64 916 / 906.
static bool evo_single(const evo::Args& a) { return evo_grid(a, 2) <= 3 * kNumCUs; }

// bias1 and bias2 as the kernels read them: [mask, pair]; mask fp32 [5, B N, Lp]: the mask, then km; pair [1 or 2, B H, Lp, Lp]: pq
// and, where a backward is to come, pk, in the type of bias2: fp32 times sqrt(D), bf16 as it is or, at heads of 64, times 8, which is
// exact; undefined without bias2
static std::vector<at::Tensor> evo_pack(const evo::Args& a, const at::TensorOptions& opt, const c10::optional<at::Tensor>& b1,
                                        const c10::optional<at::Tensor>& b2, bool backward, int64_t D) {
  const int64_t rows = (int64_t)a.B * a.N;
  const bool pair = evo_has(b2), has1 = evo_has(b1);
  auto ok = [](const at::Tensor& t) { return t.is_contiguous() && (t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16); };
  if (has1) SXE_CHECK(ok(*b1) && b1->numel() == rows * a.L, "evoformer: bias1 fp32 / bf16 [B, N, 1, 1, L]");
  if (pair) SXE_CHECK(ok(*b2) && b2->numel() == (int64_t)a.B * a.H * a.L * a.L, "evoformer: bias2 fp32 / bf16 [B, 1, H, L, L]");
  const bool narrow = pair && b2->scalar_type() == at::kBFloat16;
  at::Tensor mask = at::empty({5, rows, a.Lp}, opt.dtype(at::kFloat)), packed;
  if (pair) packed = at::empty({backward ? 2 : 1, (int64_t)a.B * a.H, a.Lp, a.Lp}, opt.dtype(narrow ? at::kBFloat16 : at::kFloat));
  if (mask.numel() == 0) return {mask, packed};
  const int nt = a.Lp / 32;
  auto pack = [&](auto t) {
    using P = decltype(t);
    P* pq = pair ? static_cast<P*>(packed.data_ptr()) : nullptr;
    const int64_t bh = pair ? (int64_t)a.B * a.H : 0, most = std::min<int64_t>(rows, 8 * kNumCUs), x = pair ? (int64_t)nt * nt : most;
    const int mask_y = std::max<int64_t>(1, std::min<int64_t>((most + x - 1) / x, 65535 - bh));
    hipLaunchKernelGGL((evo::pack_kernel<P>), dim3((unsigned)x, (unsigned)(mask_y + bh)), dim3(256), 0, cur_stream(),
                       has1 ? b1->data_ptr() : nullptr, has1 && b1->scalar_type() == at::kBFloat16, mask.data_ptr<float>(),
                       reinterpret_cast<unsigned short*>(mask.data_ptr<float>() + rows * a.Lp), rows,
                       pair ? reinterpret_cast<const P*>(b2->data_ptr()) : nullptr, pq,
                       pair && backward ? pq + packed.numel() / 2 : nullptr, a.L, nt, mf::LOG2E / a.c,
                       narrow && D == 32 ? 1.f : mf::LOG2E / a.c, mask_y);
  };
  if (narrow) pack((unsigned short)0);
  else pack(0.f);
  SXE_LAUNCH_CHECK();
  return {mask, packed};
}

static void evo_set_packed(EvoCall& c, const at::Tensor& mask, const c10::optional<at::Tensor>& pair) {
  c.a.mask = mask.data_ptr<float>();
  c.a.km = reinterpret_cast<const unsigned short*>(c.a.mask + mask.numel() / 5);
  if (!evo_has(pair)) return;
  c.pair = pair->scalar_type();
  c.a.pq = pair->data_ptr();
  c.a.pk = pair->size(0) == 2 ? static_cast<const char*>(c.a.pq) + pair->nbytes() / 2 : nullptr;
}

// f(head dim constant, tag of the packed pair bias)
template <typename F>
static void evo_dispatch(int D, at::ScalarType pair, F f) {
  auto with = [&](auto d) {
    if (pair == at::kBFloat16) f(d, (unsigned short)0);
    else if (pair == at::kFloat) f(d, 0.f);
    else f(d, evo::NoPair{});
  };
  if (D == 32) with(std::integral_constant<int, 32>{});
  else with(std::integral_constant<int, 64>{});
}

// -> [o, lse, packed biases of evo_pack]: the backward reads these, not the biases, which the caller may have changed by then
std::vector<at::Tensor> evoformer_fwd(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                                      const c10::optional<at::Tensor>& b1, const c10::optional<at::Tensor>& b2, bool backward) {
  check_beside(q, {k, v, b1, b2});
  c10::DeviceGuard g(q.device());
  EvoCall c = evo_call(q, k, v);
  evo::Args& a = c.a;
  auto packed = evo_pack(a, q.options(), b1, b2, backward, q.size(4));
  evo_set_packed(c, packed[0], packed[1]);
  auto o = at::empty_like(q);
  auto lse = at::empty({(int64_t)a.B * a.N, a.H, a.Lp}, q.options().dtype(at::kFloat));
  const int grid = evo_grid(a, 1);
  packed.insert(packed.begin(), {o, lse});
  if (grid == 0) return packed;
  a.lse = lse.data_ptr<float>();
  evo_dispatch(q.size(4), c.pair, [&](auto d, auto t) {
    constexpr int D = decltype(d)::value;
    using P = decltype(t);
    auto rows = [&](auto nn) {
      constexpr int NN = decltype(nn)::value, LDS = 2 * evo::Stream<D, NN>::SLOT;
      hipLaunchKernelGGL((evo::fwd_kernel<D, P, NN>), dim3(evo_grid(a, NN)), dim3(256), LDS, cur_stream(), a,
                         reinterpret_cast<unsigned short*>(o.data_ptr()));
    };
    if constexpr (D == 32 && std::is_same<P, float>::value) if (!evo_single(a)) return rows(std::integral_constant<int, 2>{});
    rows(std::integral_constant<int, 1>{});
  });
  SXE_LAUNCH_CHECK();
  return packed;
}

std::vector<at::Tensor> evoformer_bwd(const at::Tensor& dout, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                                      const at::Tensor& o, const at::Tensor& lse, const at::Tensor& mask,
                                      const c10::optional<at::Tensor>& pair, bool need_db1, c10::optional<at::ScalarType> db2_type) {
  const bool need_db2 = db2_type.has_value();
  check_beside(q, {dout, k, v, o, lse, mask, pair});
  c10::DeviceGuard g(q.device());
  EvoCall c = evo_call(q, k, v);
  evo::Args& a = c.a;
  auto packed = [](const at::Tensor& t, int64_t numel) {
    return t.numel() == numel && t.is_contiguous() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  SXE_CHECK(packed(mask, 5 * (int64_t)a.B * a.N * a.Lp) && mask.scalar_type() == at::kFloat, "evoformer_bwd: mask as the forward packed it");
  if (evo_has(pair))
    SXE_CHECK(pair->dim() == 4 && pair->size(0) == 2 && packed(*pair, 2 * (int64_t)a.B * a.H * a.Lp * a.Lp) &&
                  (pair->scalar_type() == at::kFloat || pair->scalar_type() == at::kBFloat16),
              "evoformer_bwd: bias2 as the forward packed it, in both forms");
  SXE_CHECK(!need_db2 || *db2_type == at::kFloat || *db2_type == at::kBFloat16, "evoformer_bwd: gradient of bias2 in fp32 / bf16");
  evo_set_packed(c, mask, pair);
  for (const at::Tensor* t : {&dout, &o})
    SXE_CHECK(t->sizes() == q.sizes() && t->is_contiguous() && t->scalar_type() == at::kBFloat16, "evoformer_bwd: dout / o like q");
  SXE_CHECK(lse.numel() == (int64_t)a.B * a.N * a.H * a.Lp && lse.scalar_type() == at::kFloat && lse.is_contiguous(),
            "evoformer_bwd: lse fp32 [B*N, H, Lp]");
  SXE_CHECK(!need_db2 || evo_has(pair), "evoformer_bwd: gradient of a bias2 that is not there");
  const at::Tensor d = evo_aligned(dout), oo = evo_aligned(o);
  auto stats = at::empty({lse.numel(), 2, 4}, q.options());
  a.dout = reinterpret_cast<const unsigned short*>(d.data_ptr());
  a.o = reinterpret_cast<const unsigned short*>(oo.data_ptr());
  a.lse = lse.data_ptr<float>();
  a.stats = reinterpret_cast<unsigned short*>(stats.data_ptr());
  auto dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
  at::Tensor db1, db2;
  if (need_db1) db1 = at::zeros({a.B, a.N, 1, 1, a.L}, q.options().dtype(at::kFloat));
  if (need_db2) db2 = at::empty({a.B, 1, a.H, a.L, a.L}, q.options().dtype(*db2_type));
  const int grid = evo_grid(a, 1);
  if (grid == 0) {
    if (need_db2) db2.zero_();
    return {dq, dk, dv, need_db1 ? db1 : at::Tensor(), need_db2 ? db2 : at::Tensor()};
  }
  auto* dqp = reinterpret_cast<unsigned short*>(dq.data_ptr());
  auto* dkp = reinterpret_cast<unsigned short*>(dk.data_ptr());
  auto* dvp = reinterpret_cast<unsigned short*>(dv.data_ptr());
  evo_dispatch(q.size(4), c.pair, [&](auto dd, auto t) {
    constexpr int D = decltype(dd)::value;
    using P = decltype(t);
    constexpr bool PAIR = !std::is_same<P, evo::NoPair>::value;
    bool both = false;
    if constexpr (PAIR && D == 32) {
      both = need_db2 && a.L <= 384;
      auto run = [&](auto j) {
        using C = evo::DqPair<decltype(j)::value>;
        constexpr auto kernel = &evo::dq_pair_kernel<decltype(j)::value, P>;
        allow_lds<kernel>(C::LDS);
        const int wgs = (a.L + C::QUERIES - 1) / C::QUERIES * a.B * a.H, most = std::max(1, std::min(a.N, kNumCUs / wgs));
        const int rows_per = (a.N + most - 1) / most, parts = (a.N + rows_per - 1) / rows_per;
        const int64_t stride = (int64_t)a.B * a.H * a.Lp * a.Lp;
        auto part = at::empty({parts, stride}, q.options().dtype(at::kFloat));
        hipLaunchKernelGGL(kernel, dim3(wgs, parts), dim3(512), C::LDS, cur_stream(), a, dqp, part.template data_ptr<float>(), rows_per);
        const int tl = (a.L + 31) / 32;
        const dim3 gs(tl * tl, a.B * a.H);
        if (db2.scalar_type() == at::kFloat)
          hipLaunchKernelGGL(evo::dpair_tiles_kernel<float>, gs, dim3(256), 0, cur_stream(), part.template data_ptr<float>(),
                             db2.data_ptr<float>(), stride, parts, a.L, a.Lp / 32);
        else
          hipLaunchKernelGGL(evo::dpair_tiles_kernel<unsigned short>, gs, dim3(256), 0, cur_stream(), part.template data_ptr<float>(),
                             reinterpret_cast<unsigned short*>(db2.data_ptr()), stride, parts, a.L, a.Lp / 32);
      };
      if (both) {
        if (a.L <= 128) run(std::integral_constant<int, 1>{});
        else if (a.L <= 256) run(std::integral_constant<int, 2>{});
        else run(std::integral_constant<int, 3>{});
      }
    }
    auto dq_rows = [&](auto nn) {
      constexpr int NN = decltype(nn)::value, LDS = 2 * evo::Stream<D, NN>::SLOT;
      hipLaunchKernelGGL((evo::dq_kernel<D, P, NN>), dim3(evo_grid(a, NN)), dim3(256), LDS, cur_stream(), a, dqp);
    };
    if (!both) {
      constexpr bool TWO = std::is_same<P, float>::value || (PAIR && D == 64);
      bool two = false;
      if constexpr (TWO) {
        two = !evo_single(a);
        if (two) dq_rows(std::integral_constant<int, 2>{});
      }
      if (!two) dq_rows(std::integral_constant<int, 1>{});
    }
    auto dkdv = [&](auto nn, auto db) {
      constexpr int NN = decltype(nn)::value, LDS = 2 * evo::QueryStream<D, NN>::SLOT;
      hipLaunchKernelGGL((evo::dkdv_kernel<D, P, NN, decltype(db)::value>), dim3(evo_grid(a, NN)), dim3(256), LDS, cur_stream(), a, dkp, dvp,
                         need_db1 ? db1.data_ptr<float>() : nullptr);
    };
    auto dkdv_rows = [&](auto db) {
      if constexpr (D == 32 && std::is_same<P, float>::value) if (!evo_single(a)) return dkdv(std::integral_constant<int, 2>{}, db);
      dkdv(std::integral_constant<int, 1>{}, db);
    };
    if (need_db1) dkdv_rows(std::true_type{});
    else dkdv_rows(std::false_type{});
    if constexpr (PAIR) if (need_db2 && !both) {
      constexpr int LDSP = 2 * evo::QueryStream<D, 1>::SLOT;
      // as many parts as all run at once (a part of at least 8 rows): a second, part-filled round costs more than the
      // longer walk
      const int wgs = (a.L + evo::KT - 1) / evo::KT * (a.Lp / evo::QB) * a.B * a.H;
      const int most = std::max(1, std::min((a.N + 7) / 8, evo::min_waves<D>() * kNumCUs / wgs));
      const int rows_per = (a.N + most - 1) / most, parts = (a.N + rows_per - 1) / rows_per;
      const bool direct = parts == 1 && db2.scalar_type() == at::kFloat;
      auto part = direct ? db2 : at::empty({parts, db2.numel()}, q.options().dtype(at::kFloat));
      hipLaunchKernelGGL((evo::dpair_kernel<D, P>), dim3(wgs, parts), dim3(256), LDSP, cur_stream(), a, part.template data_ptr<float>(),
                         rows_per);
      if (!direct) {
        const dim3 gs(stream_grid(db2.numel(), 256));
        if (db2.scalar_type() == at::kFloat)
          hipLaunchKernelGGL(evo::dpair_sum_kernel<float>, gs, dim3(256), 0, cur_stream(), part.template data_ptr<float>(),
                             db2.data_ptr<float>(), db2.numel(), parts);
        else
          hipLaunchKernelGGL(evo::dpair_sum_kernel<unsigned short>, gs, dim3(256), 0, cur_stream(), part.template data_ptr<float>(),
                             reinterpret_cast<unsigned short*>(db2.data_ptr()), db2.numel(), parts);
      }
    }
  });
  SXE_LAUNCH_CHECK();
  return {dq, dk, dv, need_db1 ? db1 : at::Tensor(), need_db2 ? db2 : at::Tensor()};
}

}  // namespace sxe

TORCH_LIBRARY_FRAGMENT(sxe, m) {
  m.def("evoformer_fwd(Tensor q, Tensor k, Tensor v, Tensor? bias1, Tensor? bias2, bool backward=False) -> Tensor[]");
  m.def("evoformer_bwd(Tensor dout, Tensor q, Tensor k, Tensor v, Tensor o, Tensor lse, Tensor mask, Tensor? pair, "
        "bool need_db1, ScalarType? db2) -> Tensor[]");
}
TORCH_LIBRARY_IMPL(sxe, CUDA, m) {
  m.impl("evoformer_fwd", &sxe::evoformer_fwd);
  m.impl("evoformer_bwd", &sxe::evoformer_bwd);
}
