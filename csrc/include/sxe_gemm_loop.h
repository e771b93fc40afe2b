// The inner loop of the 16 x 16 x 32 bf16 products (gemm_tn.hip, experts_kn_tile.hip, gemm_wgrad.hip): WR x WC waves, each RT x CT blocks of 16 x 16
// fp32 sums, whose operands x and w stream through LDS in slabs of 64 k, SA and SB of them at once.
//  * The loads of a slab (a wave's are PA of x and PB of w, 1 KB each) are spread over three quarters of a slab's time: a wave that
//    issues them at once waits in front of the full address queue with its products behind it (8192 rows, 28672 x 4096, 1.20 against
//    1.32 PFLOP/s), and issued later they arrive late.
//  * Fragments of a step of 32 k are read while the step before runs: the second half of x's rows and, behind the barrier in the
//    middle of a slab's last step, the next step's first half and w's. x's replace what the step has used up, w's have two sets.
//  * Of a SIMD's two waves the one that is further waits (s_setprio by progress): in the order of their age one runs ahead to the
//    barrier and the other then runs alone, with its latencies: 2 %.
#pragma once
#include "sxe_tile.h"
#include <type_traits>

namespace sxe {
namespace gl {
using namespace mf;

constexpr int BK = 64;

// SA, SB: slots of x and of w; WAVES: of a SIMD; a slab's row of BM values of x or BN of w is BK values long
template <int WR_, int WC_, int RT_, int CT_, int SA_, int SB_, int WAVES_>
struct Tile {
  static constexpr int WR = WR_, WC = WC_, RT = RT_, CT = CT_, SA = SA_, SB = SB_, WAVES = WAVES_;
  static constexpr int NW = WR * WC, NTHR = 64 * NW, BM = WR * RT * 16, BN = WC * CT * 16;
  static constexpr int PA = BM / 8 / NW, PB = BN / 8 / NW, AS = BM * 2 * BK, BS = BN * 2 * BK, LDS = SA * AS + SB * BS;
  static_assert(PA * 8 * NW == BM && PB * 8 * NW == BN && NW % 2 == 0 && RT % 2 == 0 && CT == 4 && SB >= SA && SA >= 2 && LDS <= 160 * 1024);
};

// 16 bytes a lane, at `base` + the lane's `off`, to 1 KB of LDS at the wave-uniform byte address `dst`; as tl::glds16
__device__ __forceinline__ void glds(unsigned off, const void* base, unsigned dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ unsigned lds_base() {
  return __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)tl::lds);
}
__device__ __forceinline__ unsigned pack(float a, float b) { return (unsigned)f32_to_bf16(a) | ((unsigned)f32_to_bf16(b) << 16); }
// x / (1 + exp(-x)). FULL: to 32 bits, off by less than 5 * 2^-24 of itself (x / (1.f + expf(-x)): 3, but the quotient costs 10 % of a
// tile of 4096 k): what rounding -LOG2E * x and LOG2E left out is put back behind the exponent; below -87 it goes to -0. Else as
// x / (1.f + __expf(-x)), whose exponent is off as -LOG2E * x is rounded: 17 * 2^-24 at x = -16, 66 at -87.
template <bool FULL>
__device__ __forceinline__ float silu(float x) {
  constexpr float kLow = 1.92596299e-8f;  // log2(e) - LOG2E
  if constexpr (!FULL) return x * __builtin_amdgcn_rcpf(1.f + fast_exp2(-LOG2E * x));
  const float c = __builtin_amdgcn_fmed3f(x, -88.f, 150.f), t = -LOG2E * c;
  const float left = __builtin_fmaf(-kLow, c, __builtin_fmaf(-LOG2E, c, -t)), e = fast_exp2(t);
  const float d = 1.f + __builtin_fmaf(e, LN2 * left, e), r = __builtin_amdgcn_rcpf(d);
  return x * __builtin_fmaf(__builtin_fmaf(-d, r, 1.f), r, r);
}

// acc[i][j] = sums over ns slabs of (w block j)' x (x block i): a lane has row lane & 15 of x and the four rows 4 (lane >> 4) .. of w.
//   load_x(i, slab, slot), load_w(i, slab, slot): the wave's i-th load of a slab to a slot (byte offset in x's or w's part of LDS);
//     slabs behind the last are asked for, too, and may be any that can be read
//   read_x(f, s, i, slot), read_w(f, s, j, slot): fragment of block i or j, step s
//   live: x blocks of the wave whose sums are wanted, `all` of them or fewer; half: 32 k more, the first step of slab ns
template <typename T, typename LX, typename LW, typename RX, typename RW>
__device__ __forceinline__ void loop(f32x4 (&acc)[T::RT][T::CT], int ns, bool half, bool all, int live, LX load_x, LW load_w, RX read_x, RW read_w) {
  constexpr int RT = T::RT, CT = T::CT, SA = T::SA, SB = T::SB, PA = T::PA, PB = T::PB, AS = T::AS, BS = T::BS;
  constexpr int HR = RT / 2, TURN = 2 * RT;  // rows of blocks: of half a step, of a slab
  bf16x8 fa[RT], fb[2][CT];
  // the first slabs, in the order of the loop's loads: x of slab t + SA and w of slab t + SB behind the barrier of slab t. What the
  // loop issues ahead of its first barrier repeats the last of these
#pragma unroll
  for (int t = 0; t < SB; ++t) {
    if (t < SA)
#pragma unroll
      for (int i = 0; i < PA; ++i) load_x(i, t, t * AS);
#pragma unroll
    for (int i = 0; i < PB; ++i) load_w(i, t, t * BS);
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((SA - 1) * PA + (SB - 1) * PB) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < HR; ++i) read_x(fa[i], 0, i, 0);
#pragma unroll
  for (int j = 0; j < CT; ++j) read_w(fb[0][j], 0, j, 0);
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  unsigned sx = 0, sw = 0, px = (SA - 1) * AS, pw = (SB - 1) * BS;  // slots of this slab and of the one before
  auto run = [&](auto every) __attribute__((always_inline)) {
    for (int t = 0; t < ns; ++t) {
      const unsigned nx = sx + AS == SA * AS ? 0 : sx + AS, nw = sw + BS == SB * BS ? 0 : sw + BS;
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < RT; ++i) {
          __builtin_amdgcn_sched_barrier(0);
          const int behind = (s * RT + i + TURN - RT - HR) % TURN;  // rows since the barrier
          if (behind == 0) __builtin_amdgcn_s_setprio(3);
          if (behind == TURN / 4) __builtin_amdgcn_s_setprio(2);
          if (behind == TURN / 2) __builtin_amdgcn_s_setprio(1);
          if (behind == 3 * TURN / 4) __builtin_amdgcn_s_setprio(0);
          if (behind == 0) {
            // This wave's part of slab t + 1 has landed and slab t is in its registers; behind the barrier that holds for all. What
            // may be in flight still: w of slab t + 2 (with a third slot each, x of it, too), issued last
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((SA - 2) * PA + (SB - 2) * PB) : "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
          }
          if constexpr (!decltype(every)::value)
            if (i < live) {
#pragma unroll
              for (int j = 0; j < CT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[s][j], fa[i], acc[i][j], 0, 0, 0);
            }
#pragma unroll
          for (int j = 0; j < CT; ++j) {
            if constexpr (decltype(every)::value)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[s][j], fa[i], acc[i][j], 0, 0, 0);
            const int m = i * CT + j;
#pragma unroll
            for (int k = 0; k < HR; ++k)
              if (k * CT / 2 == m) read_x(fa[HR + k], s, HR + k, sx);
#pragma unroll
            for (int k = 0; k < HR + CT; ++k)
              if (HR * CT + k * HR * CT / (HR + CT) == m) {
                if (k < HR) read_x(fa[k], s ^ 1, k, s == 0 ? sx : nx);
                else read_w(fb[s ^ 1][k < HR ? 0 : k - HR], s ^ 1, k - HR, s == 0 ? sw : nw);
              }
          }
          // the slots of slab t are free behind its barrier
          const bool now = s == 1 && i >= HR;
#pragma unroll
          for (int n = 0; n < PA + PB; ++n)
            if (n * (3 * TURN / 4) / (PA + PB) == behind) {
              if (n < PA) load_x(n < PA ? n : 0, (now ? t : t - 1) + SA, now ? sx : px);
              else load_w(n < PA ? 0 : n - PA, (now ? t : t - 1) + SB, now ? sw : pw);
            }
        }
      px = sx, pw = sw, sx = nx, sw = nw;
    }
  };
  if (all) run(std::true_type{});
  else run(std::false_type{});
  if (half) {
#pragma unroll
    for (int i = HR; i < RT; ++i) read_x(fa[i], 0, i, sx);
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < CT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[0][j], fa[i], acc[i][j], 0, 0, 0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing writes LDS behind the end
  __builtin_amdgcn_s_setprio(0);
}

// 64 columns of y from column c in 16 rows, r a lane's own: v[h] are its 8 columns 32 h + 8 (lane >> 4) .. . Rows below `rows` and columns
// below `cols` exist; every lane of the wave takes part and neighbours have neighbouring rows, the even one the even row. Two lanes with neighbouring rows change halves, so that a
// store writes whole cache lines, 64 columns of 8 rows, and not halves of 16 (8192 rows, 16384 x 2048: 417 us so, 406 here)
__device__ __forceinline__ void store_lines(unsigned short* y, int64_t ld, int r, int rows, int c, int cols, const u32x4 (&v)[2]) {
  const int lane = threadIdx.x & 63;
  const bool odd = lane & 1;
  u32x4 t;
#pragma unroll
  for (int e = 0; e < 4; ++e) t[e] = __builtin_amdgcn_mov_dpp(odd ? v[0][e] : v[1][e], 0xB1, 0xF, 0xF, true);  // lane ^ 1
  r = (r & ~1), c += (odd ? 32 : 0) + 8 * (lane >> 4);
  if (c < cols) {
    unsigned short* p = y + r * ld + c;
    if (r < rows) *reinterpret_cast<u32x4*>(p) = odd ? t : v[0];
    if (r + 1 < rows) *reinterpret_cast<u32x4*>(p + ld) = odd ? v[1] : t;
  }
}

// zeros to a tile of y: rows x cols (a multiple of 8) from `y` on
__device__ __forceinline__ void clear_tile(unsigned short* y, int64_t ld, int rows, int cols) {
  const int per = cols / 8;
  for (int i = threadIdx.x; i < rows * per; i += blockDim.x) *reinterpret_cast<u32x4*>(y + (i / per) * ld + i % per * 8) = u32x4{0u, 0u, 0u, 0u};
}

}  // namespace gl

// rows in use of each of `n` blocks of rows, or null
inline const int* used_rows(const c10::optional<at::Tensor>& t, int64_t n) {
  if (!t.has_value() || !t->defined()) return nullptr;
  SXE_CHECK(t->is_cuda() && t->scalar_type() == at::kInt && t->is_contiguous() && t->numel() == n, "rows in use: int32, one number for each of ", n);
  return t->data_ptr<int>();
}
}  // namespace sxe
