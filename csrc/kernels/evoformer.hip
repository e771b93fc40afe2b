// Evoformer attention (DS4Sci_EvoformerAttention) on gfx950: O = softmax(Q K^T / sqrt(D) + bias1 +
// bias2) V over Q/K/V [B, N, L, H, D] with bias1 [B, N, 1, 1, L] (MSA row mask) and bias2
// [B, 1, H, L, L] (pair bias), head dims 32 / 64; backward with dQ, dK, dV, dbias1, dbias2.
//
// Reference: ops/deepspeed4science/evoformer_attn.py (CUTLASS kernels of csrc/deepspeed4science,
// not in the snapshot; kMax = 64 there too).
//
// What bounds it: with D = 32 a score costs 4 matrix-core cycles and ~11 VALU ones (bias, exponent, sums, rounding), so
// every access and instruction a score has to pay for counts. Structure:
//  * swapped products (S^T = K Q^T: one lane = one query's scores, lane-local softmax) on v_mfma_f32_32x32x16_bf16, the
//    score accumulator reused as the B operand of O^T += V^T P^T; 128 queries (or keys) a workgroup, K / V (Q / dO) tiles
//    of 64 rows direct to LDS in rows of D elements, two slots;
//  * the pair bias is brought into the accumulator's order once a call (pack_kernel: 2 x [H, L, L]), in the type it came in:
//    a lane then reads its 16 scores' biases as 16-byte vectors (lane = query for the forward and dQ, lane = key for
//    dK / dV and dbias2) one tile ahead. Read in place they are 16 loads of one value, each over 32 rows of the matrix;
//  * the row mask is packed to fp32 in the log2 domain with -inf behind the last key, which is all the tail masking there
//    is; rows behind L are read from a row of zeros;
//  * dbias2 = sum of dS over the N rows has a kernel of its own that keeps a 64 x 128 tile of it in registers while it
//    walks the rows (a third recomputation of dS costs less than L x L atomics a row and is deterministic); where that
//    gives too few workgroups the rows are split and the parts added up by a last pass. dbias1: per-lane sums, one atomic
//    a key;
//  * delta = rowsum(dO O) is formed in the dQ kernel, which leaves it and the log2-domain LSE to the other two.
// MSA row attention 1 x 128 x 384, 8 heads of 32, bf16 biases, MI355X, forward + backward: 1595 us with biases read in
// place, dbias2 by atomics and delta by torch; see the kernels below for what each takes now.
#include "sxe_common.h"
#include "sxe_tile.h"
#include <torch/library.h>
#include <type_traits>

namespace sxe {
namespace evo {
using namespace tl;

constexpr int NW = 4, QB = 32 * NW, KT = 64;  // waves, rows of a workgroup, rows of a streamed tile
constexpr int TAIL = 2 * KT * 4;              // bytes of a slot's two fp32 rows

__device__ const __attribute__((aligned(128))) unsigned short kZeroRow[64] = {0};

struct Args {
  const unsigned short *q, *k, *v, *dout, *o;
  const float* b1;        // packed row mask [B N, Lp]
  const void *pq, *pk;    // packed pair bias, lane = query / lane = key; null: none
  float *lse, *lse2, *ndelta;  // [B N, H, Lp]: natural log; log2 domain, -delta
  int B, N, L, H, Lp;
  float c;                // log2(e) / sqrt(D)
};

// ------------------------------------------------------------------------------------ bias packing
// One launch for both. bias1 (null: none) [B N, L] -> [B N, Lp] fp32 * log2(e), -inf behind L: the blocks of the last grid row.
// bias2 [B H, L, L] -> 32 x 32 tiles in accumulator order: element (tile (a, b), half i / 8, lane, i % 8) is the value of
// register i of that lane. pq: lane = query of tile row a, registers = keys of b; pk (may be null): lane = key of tile row
// a, registers = queries of b. Grid: (nt * nt, B H + 1), nt = Lp / 32; without bias2 (64, 1).
template <typename T>
__global__ void __launch_bounds__(256) pack_kernel(const void* __restrict__ b1, int b1_bf16, float* __restrict__ mask, int64_t n1,
                                                   const T* __restrict__ b2, T* __restrict__ pq, T* __restrict__ pk, int L, int nt) {
  if (blockIdx.y == gridDim.y - 1) {
    const int Lp = 32 * nt;
    for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n1; i += gridDim.x * 256ll) {
      const int key = i % Lp;
      const int64_t at = i / Lp * L + key;
      float x = 0.f;
      if (b1 != nullptr && key < L)
        x = b1_bf16 ? bf16_to_f32(reinterpret_cast<const unsigned short*>(b1)[at]) : reinterpret_cast<const float*>(b1)[at];
      mask[i] = key < L ? x * LOG2E : -INFINITY;
    }
    return;
  }
  __shared__ T t[32][33];
  const int a = blockIdx.x / nt, b = blockIdx.x - a * nt;
  const T* src = b2 + (int64_t)blockIdx.y * L * L;
  for (int i = threadIdx.x; i < 1024; i += 256) {
    const int q = 32 * a + i / 32, k = 32 * b + i % 32;
    t[i / 32][i % 32] = q < L && k < L ? src[(int64_t)q * L + k] : (T)0;
  }
  __syncthreads();
  const int64_t tiles = (int64_t)blockIdx.y * nt * nt;
  for (int i = threadIdx.x; i < 1024; i += 256) {
    const int reg = (i >> 9) * 8 + (i & 7), lane = (i >> 3) & 63, r = acc_row(reg, lane >> 5);
    pq[(tiles + (int64_t)a * nt + b) * 1024 + i] = t[lane & 31][r];
    if (pk != nullptr) pk[(tiles + (int64_t)b * nt + a) * 1024 + i] = t[r][lane & 31];
  }
}

struct NoBias {};
// waves a SIMD: what the registers allow without spills
template <int D, typename BT>
constexpr int min_waves() { return D == 32 && !std::is_same<BT, float>::value ? 3 : 2; }
// a lane's 16 biases of one 32 x 32 tile
template <typename BT>
struct Bias {
  u32x4 v[sizeof(BT)];
  __device__ __forceinline__ void load(const void* packed, int64_t tile, int lane) {
    const char* p = reinterpret_cast<const char*>(packed) + (tile * 1024 + lane * 8) * sizeof(BT);
#pragma unroll
    for (int i = 0; i < (int)sizeof(BT); ++i)  // halves are 512 elements apart, a half is sizeof(BT) / 2 vectors
      v[i] = *reinterpret_cast<const u32x4*>(p + (sizeof(BT) == 2 ? i * 1024 : (i >> 1) * 2048 + (i & 1) * 16));
  }
  __device__ __forceinline__ float at(int i) const {
    if constexpr (sizeof(BT) == 2) {
      const unsigned x = v[i >> 3][(i & 7) >> 1];
      return __uint_as_float(i & 1 ? x & 0xffff0000u : x << 16);
    } else {
      return __uint_as_float(v[i >> 2][i & 3]);
    }
  }
};
template <>
struct Bias<NoBias> {
  __device__ __forceinline__ void load(const void*, int64_t, int) {}
};
// (bias1 + bias2) * log2(e); m: the packed bias1
template <typename BT>
__device__ __forceinline__ float bias_term(const Bias<BT>& b, int i, float m) {
  if constexpr (std::is_same<BT, NoBias>::value) return m;
  else return __builtin_fmaf(b.at(i), LOG2E, m);
}

__device__ __forceinline__ void glds4(const void* src, char* dst) {
  const unsigned a = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)lds +
                                                    (unsigned)(dst - lds));
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(a), "v"(src) : "memory", "m0");
}

// rows row0 .. of x (rows of one (b, n), head h) to LDS; rows behind L are zeros
template <int D>
__device__ __forceinline__ void load_rows(char* dst, const unsigned short* x, int64_t rs, int row0, int L) {
  load_tile<KT, D, NW>(dst, D / 8, [&](int r) { return row0 + r < L ? x + (int64_t)(row0 + r) * rs : kZeroRow; });
}
template <int D>
__device__ __forceinline__ void frags(bf16x8 (&f)[D / 16], const unsigned short* x, int64_t rs, int row, int L, int hf) {
#pragma unroll
  for (int t = 0; t < D / 16; ++t)
    f[t] = *reinterpret_cast<const bf16x8*>((row < L ? x + (int64_t)row * rs : kZeroRow) + 16 * t + 8 * hf);
}
// four floats of each register group of a lane half: rows 8 g + 4 hf .. of an LDS row of floats
struct Rows16 {
  f32x4 x[4];
  __device__ __forceinline__ void load(const char* p, int first, int hf) {
#pragma unroll
    for (int g = 0; g < 4; ++g) x[g] = *reinterpret_cast<const f32x4*>(p + 4 * (first + 8 * g + 4 * hf));
  }
  __device__ __forceinline__ float at(int i) const { return x[i >> 2][i & 3]; }
};

struct Place {
  int b, n, h, blk, bn;
  int64_t rs, base, row;  // row stride; element of (b, n, 0, h, 0); row of the [B N, H, Lp] arrays
};
// The N rows that share a pair-bias tile are neighbours in the grid. (A row's blocks and heads on one XCD instead measured
// the same: K / V traffic does not bound these kernels.)
template <int D>
__device__ __forceinline__ Place place(const Args& a) {
  Place p;
  int idx = blockIdx.x;
  p.n = idx % a.N;
  idx /= a.N;
  const int nblk = a.Lp / QB;
  p.blk = idx % nblk;
  idx /= nblk;
  p.h = idx % a.H;
  p.b = idx / a.H;
  p.bn = p.b * a.N + p.n;
  p.rs = (int64_t)a.H * D;
  p.base = (int64_t)p.bn * a.L * p.rs + (int64_t)p.h * D;
  p.row = ((int64_t)p.bn * a.H + p.h) * a.Lp;
  return p;
}

template <int D>
__device__ __forceinline__ void store_rows(const f32x16 (&acc)[D / 32], unsigned short* out, float s, int hf) {
#pragma unroll
  for (int t = 0; t < D / 32; ++t) store_acc_t(acc[t], out + 32 * t + 4 * hf, s);
}

// ------------------------------------------------------------------------------------ forward
template <int D, typename BT>
__global__ void __launch_bounds__(256, (min_waves<D, BT>())) fwd_kernel(Args a, unsigned short* __restrict__ out) {
  constexpr int TILE = KT * 2 * D, SLOT = 2 * TILE + TAIL;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, hf = lane >> 5;
  const Place p = place<D>(a);
  const int q0 = p.blk * QB + 32 * w, q = q0 + r, nt32 = a.Lp / 32;
  const int64_t tiles = (((int64_t)p.b * a.H + p.h) * nt32 + q0 / 32) * nt32;
  bf16x8 qf[D / 16];
  frags<D>(qf, a.q + p.base, p.rs, q, a.L, hf);
  f32x16 o[D / 32];
#pragma unroll
  for (int t = 0; t < D / 32; ++t) o[t] = zero16();
  float m = -INFINITY, l = 0.f;
  const int n = (a.L + KT - 1) / KT;
  auto load = [&](int t, char* slot) {
    load_rows<D>(slot, a.k + p.base, p.rs, t * KT, a.L);
    load_rows<D>(slot + TILE, a.v + p.base, p.rs, t * KT, a.L);
    if (w == 0) glds4(a.b1 + (int64_t)p.bn * a.Lp + t * KT + lane, slot + 2 * TILE);
  };
  Bias<BT> bias[2], next[2];
  load(0, lds);
#pragma unroll
  for (int j = 0; j < 2; ++j) next[j].load(a.pq, tiles + j, lane);
  wait_loads();
  __syncthreads();
  LaneOffs<D> lo;
  lo.init(lane);
  for (int t = 0; t < n; ++t) {
    const char* kt = lds + (t & 1) * SLOT;
    const char* vt = kt + TILE;
#pragma unroll
    for (int j = 0; j < 2; ++j) bias[j] = next[j];
    if (t + 1 < n) {
      load(t + 1, lds + ((t & 1) ^ 1) * SLOT);
#pragma unroll
      for (int j = 0; j < 2; ++j) next[j].load(a.pq, tiles + 2 * (t + 1) + j, lane);
    }
    if (q0 < a.L) {
      f32x16 s[2];
      float mx = -INFINITY;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        s[j] = zero16();
#pragma unroll
        for (int t2 = 0; t2 < D / 16; ++t2) s[j] = mfma(row_at(kt + 32 * j * 2 * D, lo.row[t2]), qf[t2], s[j]);
        Rows16 mask;
        mask.load(vt + TILE, 32 * j, hf);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[j][i] = __builtin_fmaf(s[j][i], a.c, bias_term(bias[j], i, mask.at(i)));
          mx = fmaxf(mx, s[j][i]);
        }
      }
      mx = fmaxf(mx, xor32(mx));
      const bool grow = mx > m + 8.f;  // lazy rescale: p <= 2^8
      const float mnew = grow ? mx : m, mref = mnew == -INFINITY ? 0.f : mnew, alpha = fast_exp2(m - mref);
      float ps = 0.f;
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[j][i] = fast_exp2(s[j][i] - mref);
          ps += s[j][i];
        }
      l = l * alpha + ps;
      m = mnew;
      if (__any(grow)) {
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
      }
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const bf16x8 pb = acc_to_b(s[j], s2);
#pragma unroll
          for (int dt = 0; dt < D / 32; ++dt) o[dt] = mfma(tr_at(vt + (32 * j + 16 * s2) * 2 * D, lo.tr[dt]), pb, o[dt]);
        }
    }
    wait_loads();
    __syncthreads();
  }
  l += xor32(l);
  if (q < a.L) store_rows<D>(o, out + p.base + (int64_t)q * p.rs, l > 0.f ? 1.f / l : 0.f, hf);
  if (hf == 0) a.lse[p.row + q] = q < a.L && l > 0.f ? (m + log2f(l)) * LN2 : INFINITY;
}

// ----------------------------------------------------------------------------------------- dQ
template <int D, typename BT>
__global__ void __launch_bounds__(256, (min_waves<D, BT>())) dq_kernel(Args a, unsigned short* __restrict__ dq) {
  constexpr int TILE = KT * 2 * D, SLOT = 2 * TILE + TAIL;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, hf = lane >> 5;
  const Place p = place<D>(a);
  const int q0 = p.blk * QB + 32 * w, q = q0 + r, nt32 = a.Lp / 32;
  const int64_t tiles = (((int64_t)p.b * a.H + p.h) * nt32 + q0 / 32) * nt32;
  bf16x8 qf[D / 16], df[D / 16], of[D / 16];
  frags<D>(qf, a.q + p.base, p.rs, q, a.L, hf);
  frags<D>(df, a.dout + p.base, p.rs, q, a.L, hf);
  frags<D>(of, a.o + p.base, p.rs, q, a.L, hf);
  const int n = (a.L + KT - 1) / KT;
  auto load = [&](int t, char* slot) {
    load_rows<D>(slot, a.k + p.base, p.rs, t * KT, a.L);
    load_rows<D>(slot + TILE, a.v + p.base, p.rs, t * KT, a.L);
    if (w == 0) glds4(a.b1 + (int64_t)p.bn * a.Lp + t * KT + lane, slot + 2 * TILE);
  };
  Bias<BT> bias[2], next[2];
  load(0, lds);
#pragma unroll
  for (int j = 0; j < 2; ++j) next[j].load(a.pq, tiles + j, lane);
  const float lse2 = a.lse[p.row + q] * LOG2E;
  float delta = 0.f;
#pragma unroll
  for (int t = 0; t < D / 16; ++t)
#pragma unroll
    for (int e = 0; e < 8; ++e) delta += (float)df[t][e] * (float)of[t][e];
  delta += xor32(delta);
  if (hf == 0) {
    a.lse2[p.row + q] = lse2;
    a.ndelta[p.row + q] = -delta;
  }
  f32x16 acc[D / 32], nd;
#pragma unroll
  for (int t = 0; t < D / 32; ++t) acc[t] = zero16();
#pragma unroll
  for (int i = 0; i < 16; ++i) nd[i] = -delta;
  wait_loads();
  __syncthreads();
  LaneOffs<D> lo;
  lo.init(lane);
  for (int t = 0; t < n; ++t) {
    const char* kt = lds + (t & 1) * SLOT;
    const char* vt = kt + TILE;
#pragma unroll
    for (int j = 0; j < 2; ++j) bias[j] = next[j];
    if (t + 1 < n) {
      load(t + 1, lds + ((t & 1) ^ 1) * SLOT);
#pragma unroll
      for (int j = 0; j < 2; ++j) next[j].load(a.pq, tiles + 2 * (t + 1) + j, lane);
    }
    if (q0 < a.L) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        f32x16 s = zero16(), dp = nd;
#pragma unroll
        for (int t2 = 0; t2 < D / 16; ++t2) {
          s = mfma(row_at(kt + 32 * j * 2 * D, lo.row[t2]), qf[t2], s);
          dp = mfma(row_at(vt + 32 * j * 2 * D, lo.row[t2]), df[t2], dp);
        }
        Rows16 mask;
        mask.load(vt + TILE, 32 * j, hf);
#pragma unroll
        for (int i = 0; i < 16; ++i)
          s[i] = fast_exp2(__builtin_fmaf(s[i], a.c, bias_term(bias[j], i, mask.at(i))) - lse2) * dp[i];  // dS^T
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const bf16x8 db = acc_to_b(s, s2);
#pragma unroll
          for (int dt = 0; dt < D / 32; ++dt) acc[dt] = mfma(tr_at(kt + (32 * j + 16 * s2) * 2 * D, lo.tr[dt]), db, acc[dt]);
        }
      }
    }
    wait_loads();
    __syncthreads();
  }
  if (q < a.L) store_rows<D>(acc, dq + p.base + (int64_t)q * p.rs, a.c * LN2, hf);
}

// -------------------------------------------------------------------------------------- dK, dV
// Keys on the lanes; Q / dO tiles and their LSE / -delta stream by.
template <int D>
__device__ __forceinline__ void load_query_tile(const Args& a, const unsigned short* q, const unsigned short* d, int64_t rs,
                                                int64_t row, int q0, char* slot, int w, int lane) {
  constexpr int TILE = KT * 2 * D;
  load_rows<D>(slot, q, rs, q0, a.L);
  load_rows<D>(slot + TILE, d, rs, q0, a.L);
  if (w == 0) glds4(a.lse2 + row + q0 + lane, slot + 2 * TILE);
  if (w == 1) glds4(a.ndelta + row + q0 + lane, slot + 2 * TILE + KT * 4);
}

// P and dS [query][key] of 32 queries of a slot, keys on the lanes (queries behind L: LSE inf, so P = 0)
template <int D, typename BT>
__device__ __forceinline__ void score_grads(f32x16& pr, f32x16& ds, const char* slot, int j, const LaneOffs<D>& lo,
                                            const bf16x8 (&kf)[D / 16], const bf16x8 (&vf)[D / 16], const Bias<BT>& bias, float mask,
                                            float c, int hf) {
  constexpr int TILE = KT * 2 * D;
  Rows16 ls, nd;
  ls.load(slot + 2 * TILE, 32 * j, hf);
  nd.load(slot + 2 * TILE + KT * 4, 32 * j, hf);
  pr = zero16();
#pragma unroll
  for (int i = 0; i < 16; ++i) ds[i] = nd.at(i);
#pragma unroll
  for (int t = 0; t < D / 16; ++t) {
    pr = mfma(row_at(slot + 32 * j * 2 * D, lo.row[t]), kf[t], pr);
    ds = mfma(row_at(slot + TILE + 32 * j * 2 * D, lo.row[t]), vf[t], ds);
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    pr[i] = fast_exp2(__builtin_fmaf(pr[i], c, bias_term(bias, i, mask)) - ls.at(i));
    ds[i] *= pr[i];
  }
}

template <int D, typename BT>
__global__ void __launch_bounds__(256, (min_waves<D, BT>())) dkdv_kernel(Args a, unsigned short* __restrict__ dk,
                                                                   unsigned short* __restrict__ dv, float* __restrict__ db1) {
  constexpr int TILE = KT * 2 * D, SLOT = 2 * TILE + TAIL;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, hf = lane >> 5;
  const Place p = place<D>(a);
  const int k0 = p.blk * QB + 32 * w, key = k0 + r, nt32 = a.Lp / 32;
  const int64_t tiles = (((int64_t)p.b * a.H + p.h) * nt32 + k0 / 32) * nt32;
  bf16x8 kf[D / 16], vf[D / 16];
  frags<D>(kf, a.k + p.base, p.rs, key, a.L, hf);
  frags<D>(vf, a.v + p.base, p.rs, key, a.L, hf);
  const float mask = a.b1[(int64_t)p.bn * a.Lp + key];
  f32x16 dka[D / 32], dva[D / 32];
#pragma unroll
  for (int t = 0; t < D / 32; ++t) dka[t] = dva[t] = zero16();
  float b1acc = 0.f;
  const int n = (a.L + KT - 1) / KT;
  Bias<BT> bias[2], next[2];
  load_query_tile<D>(a, a.q + p.base, a.dout + p.base, p.rs, p.row, 0, lds, w, lane);
#pragma unroll
  for (int j = 0; j < 2; ++j) next[j].load(a.pk, tiles + j, lane);
  wait_loads();
  __syncthreads();
  LaneOffs<D> lo;
  lo.init(lane);
  for (int t = 0; t < n; ++t) {
    const char* slot = lds + (t & 1) * SLOT;
#pragma unroll
    for (int j = 0; j < 2; ++j) bias[j] = next[j];
    if (t + 1 < n) {
      load_query_tile<D>(a, a.q + p.base, a.dout + p.base, p.rs, p.row, (t + 1) * KT, lds + ((t & 1) ^ 1) * SLOT, w, lane);
#pragma unroll
      for (int j = 0; j < 2; ++j) next[j].load(a.pk, tiles + 2 * (t + 1) + j, lane);
    }
    if (k0 < a.L) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        f32x16 pr, ds;
        score_grads<D>(pr, ds, slot, j, lo, kf, vf, bias[j], mask, a.c, hf);
        if (db1 != nullptr) {
#pragma unroll
          for (int i = 0; i < 16; ++i) b1acc += ds[i];
        }
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const bf16x8 pb = acc_to_b(pr, s2), db = acc_to_b(ds, s2);
#pragma unroll
          for (int dt = 0; dt < D / 32; ++dt) {
            dva[dt] = mfma(tr_at(slot + TILE + (32 * j + 16 * s2) * 2 * D, lo.tr[dt]), pb, dva[dt]);  // dV^T += dO^T P
            dka[dt] = mfma(tr_at(slot + (32 * j + 16 * s2) * 2 * D, lo.tr[dt]), db, dka[dt]);         // dK^T += Q^T dS
          }
        }
      }
    }
    wait_loads();
    __syncthreads();
  }
  if (key >= a.L) return;
  if (db1 != nullptr) {
    b1acc += xor32(b1acc);
    if (hf == 0) atomicAdd(db1 + (int64_t)p.bn * a.L + key, b1acc);
  }
  store_rows<D>(dka, dk + p.base + (int64_t)key * p.rs, a.c * LN2, hf);
  store_rows<D>(dva, dv + p.base + (int64_t)key * p.rs, 1.f, hf);
}

// -------------------------------------------------------------------------------------- dbias2
// A workgroup holds dbias2 of 64 queries x 128 keys of one (b, h) and walks rows_per of the N rows. part: fp32 [parts,
// B H, L, L]. Grid: (query tiles * key blocks * B H, parts), heads fastest: with 8 heads an XCD walks one head's rows
// (82 us at 128 x 384 x 8 heads of 32; 103 us with the tiles of a head spread over the XCDs).
template <int D, typename BT>
__global__ void __launch_bounds__(256, (min_waves<D, BT>())) dpair_kernel(Args a, float* __restrict__ part, int rows_per) {
  constexpr int TILE = KT * 2 * D, SLOT = 2 * TILE + TAIL;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, hf = lane >> 5;
  const int nqt = (a.L + KT - 1) / KT, nkb = a.Lp / QB, nt32 = a.Lp / 32;
  const int nbh = a.B * a.H, bh = blockIdx.x % nbh, kb = blockIdx.x / nbh % nkb, qt = blockIdx.x / nbh / nkb;
  const int h = bh % a.H, b = bh / a.H;
  const int k0 = kb * QB + 32 * w, key = k0 + r, q0 = qt * KT;
  const int64_t rs = (int64_t)a.H * D;
  Bias<BT> bias[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) bias[j].load(a.pk, ((int64_t)bh * nt32 + k0 / 32) * nt32 + 2 * qt + j, lane);
  const int n0 = blockIdx.y * rows_per, n1 = min(a.N, n0 + rows_per);
  f32x16 acc[2] = {zero16(), zero16()};
  bf16x8 kf[D / 16], vf[D / 16], kn[D / 16], vn[D / 16];
  float mask = 0.f, maskn = 0.f;
  auto load = [&](int n, char* slot) {
    const int bn = b * a.N + n;
    const int64_t base = (int64_t)bn * a.L * rs + (int64_t)h * D;
    load_query_tile<D>(a, a.q + base, a.dout + base, rs, ((int64_t)bn * a.H + h) * a.Lp, q0, slot, w, lane);
    frags<D>(kn, a.k + base, rs, key, a.L, hf);
    frags<D>(vn, a.v + base, rs, key, a.L, hf);
    maskn = a.b1[(int64_t)bn * a.Lp + key];
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
    if (n + 1 < n1) load(n + 1, lds + (cur ^ 1) * SLOT);
    if (k0 < a.L) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        f32x16 pr, ds;
        score_grads<D>(pr, ds, lds + cur * SLOT, j, lo, kf, vf, bias[j], mask, a.c, hf);
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
  at::ScalarType pair = at::ScalarType::Undefined;
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

// bias1 and bias2 as the kernels read them: [mask, pq, pk], pq undefined without bias2, pk without a backward to come, too
static std::vector<at::Tensor> evo_pack(const evo::Args& a, const at::TensorOptions& opt, const c10::optional<at::Tensor>& b1,
                                        const c10::optional<at::Tensor>& b2, bool backward) {
  const int64_t rows = (int64_t)a.B * a.N;
  const bool pair = evo_has(b2), has1 = evo_has(b1);
  auto ok = [](const at::Tensor& t) { return t.is_contiguous() && (t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16); };
  if (has1) SXE_CHECK(ok(*b1) && b1->numel() == rows * a.L, "evoformer: bias1 fp32 / bf16 [B, N, 1, 1, L]");
  if (pair) SXE_CHECK(ok(*b2) && b2->numel() == (int64_t)a.B * a.H * a.L * a.L, "evoformer: bias2 fp32 / bf16 [B, 1, H, L, L]");
  at::Tensor mask = at::empty({rows, a.Lp}, opt.dtype(at::kFloat)), pq, pk;
  if (pair) pq = at::empty({(int64_t)a.B * a.H, a.Lp, a.Lp}, b2->options());
  if (pair && backward) pk = at::empty_like(pq);
  if (mask.numel() == 0) return {mask, pq, pk};
  const int nt = a.Lp / 32;
  auto pack = [&](auto* t) {
    using T = std::remove_pointer_t<decltype(t)>;
    hipLaunchKernelGGL(evo::pack_kernel<T>, pair ? dim3(nt * nt, a.B * a.H + 1) : dim3(64, 1), dim3(256), 0, cur_stream(),
                       has1 ? b1->data_ptr() : nullptr, has1 && b1->scalar_type() == at::kBFloat16, mask.data_ptr<float>(), mask.numel(),
                       pair ? reinterpret_cast<const T*>(b2->data_ptr()) : nullptr,
                       pair ? reinterpret_cast<T*>(pq.data_ptr()) : nullptr,
                       pk.defined() ? reinterpret_cast<T*>(pk.data_ptr()) : nullptr, a.L, nt);
  };
  if (pair && b2->scalar_type() == at::kBFloat16) pack((unsigned short*)nullptr);
  else pack((float*)nullptr);
  SXE_LAUNCH_CHECK();
  return {mask, pq, pk};
}

static void evo_set_packed(EvoCall& c, const at::Tensor& mask, const c10::optional<at::Tensor>& pq, const c10::optional<at::Tensor>& pk) {
  c.a.b1 = mask.data_ptr<float>();
  if (!evo_has(pq)) return;
  c.pair = pq->scalar_type();
  c.a.pq = pq->data_ptr();
  c.a.pk = evo_has(pk) ? pk->data_ptr() : nullptr;
}

// f(head dim constant, pair bias type tag)
template <typename F>
static void evo_dispatch(int D, at::ScalarType pair, F f) {
  auto with = [&](auto d) {
    if (pair == at::kBFloat16) f(d, (unsigned short)0);
    else if (pair == at::kFloat) f(d, 0.f);
    else f(d, evo::NoBias{});
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
  auto packed = evo_pack(a, q.options(), b1, b2, backward);
  evo_set_packed(c, packed[0], packed[1], packed[2]);
  auto o = at::empty_like(q);
  auto lse = at::empty({(int64_t)a.B * a.N, a.H, a.Lp}, q.options().dtype(at::kFloat));
  const int grid = a.B * a.N * a.H * (a.Lp / evo::QB);
  packed.insert(packed.begin(), {o, lse});
  if (grid == 0) return packed;
  a.lse = lse.data_ptr<float>();
  evo_dispatch(q.size(4), c.pair, [&](auto d, auto t) {
    constexpr int D = decltype(d)::value;
    hipLaunchKernelGGL((evo::fwd_kernel<D, decltype(t)>), dim3(grid), dim3(256), 2 * (2 * evo::KT * 2 * D + evo::TAIL), cur_stream(),
                       a, reinterpret_cast<unsigned short*>(o.data_ptr()));
  });
  SXE_LAUNCH_CHECK();
  return packed;
}

std::vector<at::Tensor> evoformer_bwd(const at::Tensor& dout, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                                      const at::Tensor& o, const at::Tensor& lse, const at::Tensor& mask,
                                      const c10::optional<at::Tensor>& pq, const c10::optional<at::Tensor>& pk, bool need_db1,
                                      bool need_db2) {
  check_beside(q, {dout, k, v, o, lse, mask, pq, pk});
  c10::DeviceGuard g(q.device());
  EvoCall c = evo_call(q, k, v);
  evo::Args& a = c.a;
  SXE_CHECK(mask.numel() == (int64_t)a.B * a.N * a.Lp && mask.scalar_type() == at::kFloat && mask.is_contiguous(),
            "evoformer_bwd: mask as the forward packed it");
  SXE_CHECK(evo_has(pq) == evo_has(pk), "evoformer_bwd: both forms of bias2");
  if (evo_has(pq))
    for (const at::Tensor* t : {&*pq, &*pk})
      SXE_CHECK(t->numel() == (int64_t)a.B * a.H * a.Lp * a.Lp && t->is_contiguous() && t->scalar_type() == pq->scalar_type() &&
                    (t->scalar_type() == at::kFloat || t->scalar_type() == at::kBFloat16) &&
                    reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 == 0, "evoformer_bwd: bias2 as the forward packed it");
  evo_set_packed(c, mask, pq, pk);
  for (const at::Tensor* t : {&dout, &o})
    SXE_CHECK(t->sizes() == q.sizes() && t->is_contiguous() && t->scalar_type() == at::kBFloat16, "evoformer_bwd: dout / o like q");
  SXE_CHECK(lse.numel() == (int64_t)a.B * a.N * a.H * a.Lp && lse.scalar_type() == at::kFloat && lse.is_contiguous(),
            "evoformer_bwd: lse fp32 [B*N, H, Lp]");
  SXE_CHECK(!need_db2 || evo_has(pq), "evoformer_bwd: gradient of a bias2 that is not there");
  const at::Tensor d = evo_aligned(dout), oo = evo_aligned(o);
  auto stats = at::empty({2, lse.numel()}, lse.options());
  a.dout = reinterpret_cast<const unsigned short*>(d.data_ptr());
  a.o = reinterpret_cast<const unsigned short*>(oo.data_ptr());
  a.lse = lse.data_ptr<float>();
  a.lse2 = stats.data_ptr<float>();
  a.ndelta = a.lse2 + lse.numel();
  auto dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
  at::Tensor db1, db2;
  if (need_db1) db1 = at::zeros({a.B, a.N, 1, 1, a.L}, q.options().dtype(at::kFloat));
  if (need_db2) db2 = at::empty({a.B, 1, a.H, a.L, a.L}, pq->options());
  const int grid = a.B * a.N * a.H * (a.Lp / evo::QB);
  if (grid == 0) {
    if (need_db2) db2.zero_();
    return {dq, dk, dv, need_db1 ? db1 : at::Tensor(), need_db2 ? db2 : at::Tensor()};
  }
  auto* dqp = reinterpret_cast<unsigned short*>(dq.data_ptr());
  auto* dkp = reinterpret_cast<unsigned short*>(dk.data_ptr());
  auto* dvp = reinterpret_cast<unsigned short*>(dv.data_ptr());
  evo_dispatch(q.size(4), c.pair, [&](auto dd, auto t) {
    constexpr int D = decltype(dd)::value;
    using BT = decltype(t);
    const size_t lds = 2 * (2 * evo::KT * 2 * D + evo::TAIL);
    hipLaunchKernelGGL((evo::dq_kernel<D, BT>), dim3(grid), dim3(256), lds, cur_stream(), a, dqp);
    hipLaunchKernelGGL((evo::dkdv_kernel<D, BT>), dim3(grid), dim3(256), lds, cur_stream(), a, dkp, dvp,
                       need_db1 ? db1.data_ptr<float>() : nullptr);
    if constexpr (!std::is_same<BT, evo::NoBias>::value) if (need_db2) {
      // as many parts as all run at once (a part of at least 8 rows): a second, part-filled round costs more than the
      // longer walk
      const int wgs = (a.L + evo::KT - 1) / evo::KT * (a.Lp / evo::QB) * a.B * a.H;
      const int most = std::max(1, std::min((a.N + 7) / 8, evo::min_waves<D, BT>() * kNumCUs / wgs));
      const int rows_per = (a.N + most - 1) / most, parts = (a.N + rows_per - 1) / rows_per;
      const bool direct = parts == 1 && db2.scalar_type() == at::kFloat;
      auto part = direct ? db2 : at::empty({parts, db2.numel()}, q.options().dtype(at::kFloat));
      hipLaunchKernelGGL((evo::dpair_kernel<D, BT>), dim3(wgs, parts), dim3(256), lds, cur_stream(), a, part.template data_ptr<float>(),
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
  m.def("evoformer_bwd(Tensor dout, Tensor q, Tensor k, Tensor v, Tensor o, Tensor lse, Tensor mask, Tensor? pq, Tensor? pk, "
        "bool need_db1, bool need_db2) -> Tensor[]");
}
TORCH_LIBRARY_IMPL(sxe, CUDA, m) {
  m.impl("evoformer_fwd", &sxe::evoformer_fwd);
  m.impl("evoformer_bwd", &sxe::evoformer_bwd);
}
