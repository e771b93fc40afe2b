// Attention of many new tokens of a sequence over its paged KV cache (gfx950): prompts, chunks of prompts behind
// earlier tokens, any mixture of them in one launch. Decodes beside them share the launch, alone they run paged_attn.hip.
//
// Reference: inference/v2/kernels/ragged_ops/blocked_flash (an external flash-attn build over the blocked cache) with
// its atom builder, inference/v2/kernels/ragged_ops/atom_builder.
//
// What bounds it: at 64 keys a tile the two products and the softmax between them, as in the training forward
// (flash_attn.hip), once a K / V byte serves enough rows. So:
//  * a workgroup is 128 rows of one kv head: row = (token, query head of the group), so a GQA group shares every K / V
//    byte, a prompt of 20 tokens still fills its rows and the causal triangle wastes at most 128 / G tokens;
//  * the host hands over one list of tiles for all sequences, longest key range first, so one launch takes the whole
//    batch and short tiles fill in behind long ones; block index = (tile, kv head): with 8 kv heads every XCD keeps one
//    head's keys in its L2;
//  * K / V tiles go straight from the cache blocks to LDS, two slots, the next tile's load in flight behind this
//    tile's products; its block id is read a tile ahead;
//  * few tiles over long histories (one chunk behind 4k tokens) are split along the keys, fp32 partials, one merge.
// The longest prompts run the training forward instead, 1.0 - 1.05 PFLOP/s where this reaches 0.9 - 0.95: the rule and its figures
// are in ops/paged_attention.py.
// Llama-8B heads (32 / 8, D 128), MI355X, a layer: a 3500-token prompt in chunks of 1024 beside 16 decodes took 2170 us a
// chunk in the 16-row decode kernel (one read of the keys for every 4 tokens), 92 us with the decodes in a launch of that and the merges of both, 78 us in one launch here; 12
// fresh prompts of 20 - 3000 tokens took 630 us in one flash-attention launch a prompt with its padding copies, 172 us here.
#include "sxe_common.h"
#include "sxe_tile.h"
#include <torch/library.h>
#include <type_traits>

namespace sxe {
namespace pp {
using namespace tl;

constexpr int KT = 64;   // keys of a tile
constexpr int NW = 4;    // waves of 32 rows

struct Args {
  const unsigned short* q;
  int64_t q_tok_stride;
  const unsigned short* cache;  // [blocks, 2, nkv, bs, D]
  const int* block_table;
  int max_blocks;
  const int *q_start, *q_len, *kv_len;
  const int* tiles;  // [n][4]: sequence, first token row, tokens, row of its first partial
  int nq, nkv, bs, window;
  float c;           // scale * log2(e), > 0
  int splits, keys_per_split;
  unsigned short* out;
  int64_t out_tok_stride;
  float *part_o, *part_ml;  // [splits, rows, nq, D], [splits, rows, nq, 2]
  int64_t part_rows;
};

// One key tile of a wave's online softmax; MASK: some key of the tile lies behind a row's position or in front of its window.
template <bool MASK, int D>
__device__ __forceinline__ void tile_step(const LaneOffs<D>& lo, const char* kt, const char* vt, const bf16x8 (&qf)[D / 16],
                                          f32x16 (&o)[D / 32], float& m, float& l, float c, int k0, int qpos, int window, int hf,
                                          bool skip1) {
  f32x16 s[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    s[j] = zero16();
    if (j == 1 && skip1) break;  // the second 32 keys lie behind every row of the wave
#pragma unroll
    for (int t = 0; t < D / 16; ++t) s[j] = mfma(row_at(kt + 32 * j * 2 * D, lo.row[t]), qf[t], s[j]);
  }
  float mx = -INFINITY;
  int ahead = k0 + 4 * hf - qpos, behind = ahead + (window > 0 ? window : 1 << 30);
  if (MASK) asm volatile("" : "+v"(ahead), "+v"(behind));  // keep the row offsets immediates of the compares
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if (MASK && (ahead + 32 * j + acc_row(i, 0) > 0 || behind + 32 * j + acc_row(i, 0) <= 0)) s[j][i] = -INFINITY;
      mx = fmaxf(mx, s[j][i]);
    }
  mx = fmaxf(mx, xor32(mx)) * c;
  const bool grow = mx > m + 8.f;  // lazy rescale: p <= 2^8, see flash_attn.hip
  const float mnew = grow ? mx : m;
  const float mref = mnew == -INFINITY ? 0.f : mnew;
  const float alpha = fast_exp2(m - mref);
  float ps = 0.f;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float p = fast_exp2(__builtin_fmaf(s[j][i], c, -mref));
      s[j][i] = p;
      ps += p;
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
  for (int j = 0; j < 2; ++j) {
    if (j == 1 && skip1) break;
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const bf16x8 pb = acc_to_b(s[j], s2);
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt) o[dt] = mfma(tr_at(vt + (32 * j + 16 * s2) * 2 * D, lo.tr[dt]), pb, o[dt]);
    }
  }
}

// WHOLE: cache blocks are whole key tiles (bs % 64 == 0), so a tile lies in one block
template <int D, bool WHOLE>
__global__ void __launch_bounds__(NW * 64, D >= 256 ? 1 : 2) prefill_kernel(Args a) {
  constexpr int TILE = KT * 2 * D, SLOT = 2 * TILE;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, hf = lane >> 5;
  const int ti = blockIdx.x / a.nkv, kvh = blockIdx.x - ti * a.nkv, split = blockIdx.y;
  const int seq = a.tiles[4 * ti], t0 = a.tiles[4 * ti + 1], nt = a.tiles[4 * ti + 2], part0 = a.tiles[4 * ti + 3];
  const int kl = a.kv_len[seq], pos0 = kl - a.q_len[seq] + (t0 - a.q_start[seq]);  // position of the tile's first token
  const int G = a.nq / a.nkv, rows = nt * G;
  const int row = min(w * 32 + r, rows - 1), tok = row / G, head = kvh * G + row - tok * G, qpos = pos0 + tok;
  const bool wave_on = w * 32 < rows;
  // keys that some row of the tile sees, in this split; starts are multiples of 64
  int lo_key = a.window > 0 ? max(0, pos0 - a.window + 1) & ~(KT - 1) : 0, hi_key = min(kl, pos0 + nt);
  // all of them in one split: its result is the tile's, and (max, sum) of split 0 says so (a sum is never negative)
  const bool whole = a.splits == 1 || lo_key / a.keys_per_split == (hi_key - 1) / a.keys_per_split;
  lo_key = max(lo_key, split * a.keys_per_split);
  hi_key = min(hi_key, (split + 1) * a.keys_per_split);
  const int n = hi_key > lo_key ? (hi_key - lo_key + KT - 1) / KT : 0;
  auto partial = [&](int s, int first) { return ((int64_t)s * a.part_rows + first + tok) * a.nq + head; };
  if (n == 0) {  // the merge reads nothing else of a split whose maximum is -inf
    if (!whole && w * 32 + r < rows && hf == 0) {
      a.part_ml[partial(split, part0) * 2] = -INFINITY;
      a.part_ml[partial(split, part0) * 2 + 1] = 0.f;
    }
    return;
  }
  const int pmin = pos0 + min(w * 32, rows - 1) / G, pmax = pos0 + min(w * 32 + 31, rows - 1) / G;

  bf16x8 qf[D / 16];
  const unsigned short* qp = a.q + (int64_t)(t0 + tok) * a.q_tok_stride + (int64_t)head * D + 8 * hf;
#pragma unroll
  for (int t = 0; t < D / 16; ++t) qf[t] = *reinterpret_cast<const bf16x8*>(qp + 16 * t);
  f32x16 o[D / 32];
#pragma unroll
  for (int t = 0; t < D / 32; ++t) o[t] = zero16();
  float m = -INFINITY, l = 0.f;

  const int* bt = a.block_table + (int64_t)seq * a.max_blocks;
  const int64_t head_stride = (int64_t)a.bs * D, half_stride = a.nkv * head_stride, block_stride = 2 * half_stride;
  const unsigned short* cache = a.cache + kvh * head_stride;
  // keys at or past kl repeat the last one: they are masked, and memory past it may hold anything
  auto load = [&](int k0, int blk, char* slot) {
    if constexpr (WHOLE) {
      const unsigned short* base = cache + blk * block_stride + (int64_t)(k0 % a.bs) * D;
      const int last = kl - 1 - k0;
      load_tile<KT, D, NW>(slot, D / 8, [&](int i) { return base + min(i, last) * D; });
      load_tile<KT, D, NW>(slot + TILE, D / 8, [&](int i) { return base + half_stride + min(i, last) * D; });
    } else {
      auto at = [&](int i) {
        const int key = min(k0 + i, kl - 1), b = key / a.bs;
        return cache + bt[b] * block_stride + (int64_t)(key - b * a.bs) * D;
      };
      load_tile<KT, D, NW>(slot, D / 8, at);
      load_tile<KT, D, NW>(slot + TILE, D / 8, [&](int i) { return at(i) + half_stride; });
    }
  };
  auto block_of = [&](int t) { return WHOLE ? bt[(lo_key + KT * min(t, n - 1)) / a.bs] : 0; };
  int blk = 0;
  load(lo_key, block_of(0), lds);
  blk = block_of(1);
  wait_loads();
  __syncthreads();
  LaneOffs<D> lo;
  lo.init(lane);
  auto step = [&](int t, auto slot) {
    constexpr int CUR = decltype(slot)::value;
    if (t + 1 < n) {
      load(lo_key + KT * (t + 1), blk, lds + (CUR ^ 1) * SLOT);
      blk = block_of(t + 2);
    }
    const int k0 = lo_key + KT * t;
    if (wave_on && k0 <= pmax && (a.window <= 0 || k0 + KT - 1 > pmin - a.window)) {
      const char* kt = lds + CUR * SLOT;
      if (k0 + KT - 1 > pmin || (a.window > 0 && k0 <= pmax - a.window))
        tile_step<true, D>(lo, kt, kt + TILE, qf, o, m, l, a.c, k0, qpos, a.window, hf, k0 + 32 > pmax);
      else
        tile_step<false, D>(lo, kt, kt + TILE, qf, o, m, l, a.c, k0, qpos, 0, hf, false);
    }
    wait_loads();
    __syncthreads();
  };
  for (int t = 0; t < n; t += 2) {
    step(t, std::integral_constant<int, 0>{});
    if (t + 1 < n) step(t + 1, std::integral_constant<int, 1>{});
  }
  l += xor32(l);
  if (w * 32 + r >= rows) return;
  int first = part0;
  asm volatile("" : "+s"(first));  // the partials' rows are worked out here, not held from above
  if (whole) {
    if (a.splits > 1 && hf == 0) a.part_ml[partial(0, first) * 2 + 1] = -1.f;
    const float inv = l > 0.f ? 1.f / l : 0.f;
    unsigned short* op = a.out + (int64_t)(t0 + tok) * a.out_tok_stride + (int64_t)head * D + 4 * hf;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt) store_acc_t(o[dt], op + 32 * dt, inv);
  } else {
    const int64_t mine = partial(split, first);
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(a.part_o + mine * D + 32 * dt + 8 * g + 4 * hf) =
            f32x4{o[dt][4 * g], o[dt][4 * g + 1], o[dt][4 * g + 2], o[dt][4 * g + 3]};
    if (hf == 0) {
      a.part_ml[mine * 2] = m;
      a.part_ml[mine * 2 + 1] = l;
    }
  }
}

}  // namespace pp

// paged_attn.hip
void paged_merge(const at::Tensor& part_o, const at::Tensor& part_ml, const at::Tensor& rows, at::Tensor& out);

// q [T, nq, D], out [T, nq, D] (only the listed tokens are written); tiles int32 [n, 4] (sequence, first token row,
// tokens, partial row), tokens * (nq / nkv) <= 128; splits > 1: rows int32 [R] is the token row of every partial row.
void paged_prefill(const at::Tensor& q, const at::Tensor& cache, const at::Tensor& block_table, const at::Tensor& q_start,
                   const at::Tensor& q_len, const at::Tensor& kv_len, const at::Tensor& tiles,
                   const c10::optional<at::Tensor>& rows, double scale, int64_t window, int64_t splits, int64_t keys_per_split, at::Tensor out) {
  check_beside(q, {cache, block_table, q_start, q_len, kv_len, tiles, rows, out});
  SXE_CHECK(q.scalar_type() == at::kBFloat16 && cache.scalar_type() == at::kBFloat16 && out.scalar_type() == at::kBFloat16,
            "paged_prefill: bf16 only");
  SXE_CHECK(q.dim() == 3 && q.stride(2) == 1 && q.stride(1) == q.size(2) && q.stride(0) % 8 == 0 &&
                reinterpret_cast<uintptr_t>(q.data_ptr()) % 16 == 0,
            "paged_prefill: q [T, nq, D] with head stride D and 16-byte aligned rows");
  SXE_CHECK(out.sizes() == q.sizes() && out.is_contiguous(), "paged_prefill: out contiguous like q");
  SXE_CHECK(cache.dim() == 5 && cache.is_contiguous() && cache.size(1) == 2, "cache must be [blocks, 2, nkv, bs, D]");
  SXE_CHECK(block_table.scalar_type() == at::kInt && block_table.is_contiguous() && block_table.dim() == 2,
            "block_table int32 [S, max_blocks]");
  for (auto* t : {&q_start, &q_len, &kv_len})
    SXE_CHECK(t->scalar_type() == at::kInt && t->is_contiguous() && t->numel() == block_table.size(0),
              "q_start/q_len/kv_len: int32 [S]");
  SXE_CHECK(tiles.scalar_type() == at::kInt && tiles.is_contiguous() && tiles.dim() == 2 && tiles.size(1) == 4,
            "paged_prefill: tiles int32 [n, 4]");
  const int nq = q.size(1), D = q.size(2), nkv = cache.size(2), bs = cache.size(3);
  SXE_CHECK(cache.size(4) == D && nkv > 0 && nq % nkv == 0, "head layout mismatch");
  SXE_CHECK(scale > 0 && splits >= 1 && keys_per_split > 0 && keys_per_split % pp::KT == 0,
            "paged_prefill: scale > 0, keys_per_split a multiple of 64");
  if (tiles.size(0) == 0) return;
  c10::DeviceGuard g(q.device());
  pp::Args a{};
  a.q = reinterpret_cast<const unsigned short*>(q.data_ptr());
  a.q_tok_stride = q.stride(0);
  a.cache = reinterpret_cast<const unsigned short*>(cache.data_ptr());
  a.block_table = block_table.data_ptr<int>();
  a.max_blocks = block_table.size(1);
  a.q_start = q_start.data_ptr<int>();
  a.q_len = q_len.data_ptr<int>();
  a.kv_len = kv_len.data_ptr<int>();
  a.tiles = tiles.data_ptr<int>();
  a.nq = nq;
  a.nkv = nkv;
  a.bs = bs;
  a.window = (int)std::max<int64_t>(0, window);
  a.c = (float)scale * mf::LOG2E;
  a.splits = (int)splits;
  a.keys_per_split = (int)keys_per_split;
  a.out = reinterpret_cast<unsigned short*>(out.data_ptr());
  a.out_tok_stride = out.stride(0);
  at::Tensor part_o, part_ml;
  if (splits > 1) {
    SXE_CHECK(rows.has_value() && rows->scalar_type() == at::kInt && rows->is_contiguous(),
              "paged_prefill: rows int32 [R]");
    a.part_rows = rows->numel();
    part_o = at::empty({splits, a.part_rows, nq, D}, q.options().dtype(at::kFloat));
    part_ml = at::empty({splits, a.part_rows, nq, 2}, q.options().dtype(at::kFloat));
    a.part_o = part_o.data_ptr<float>();
    a.part_ml = part_ml.data_ptr<float>();
  }
  const dim3 grid(tiles.size(0) * nkv, splits);
  auto launch = [&](void (*kern)(pp::Args), size_t lds) {
    if (lds > 65536)  // beyond 64 KiB of dynamic LDS a kernel is opted in (gfx950: 160 KiB a CU)
      SXE_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, grid, dim3(pp::NW * 64), lds, cur_stream(), a);
  };
  const size_t lds = 4 * pp::KT * 2 * D;
  const bool whole = bs % pp::KT == 0;
  if (D == 128) launch(whole ? pp::prefill_kernel<128, true> : pp::prefill_kernel<128, false>, lds);
  else if (D == 64) launch(whole ? pp::prefill_kernel<64, true> : pp::prefill_kernel<64, false>, lds);
  else if (D == 256) launch(whole ? pp::prefill_kernel<256, true> : pp::prefill_kernel<256, false>, lds);
  else SXE_CHECK(false, "paged_prefill: head_dim must be 64, 128 or 256");
  SXE_LAUNCH_CHECK();
  if (splits > 1) paged_merge(part_o, part_ml, *rows, out);
}

// (splits, keys of a split) of a launch of tiles with these key ranges (longest first) and tokens: equal pieces of the longest range, of which a
// tile has as many as its own range reaches into, and no partials where that is one. What takes least by this account, in us: the longest
// piece, 1.6 for every 64 keys, or all of them together, 190 such steps of a kv head a us; and where tiles have more than one piece the
// merge, 5 for every 16 pieces and 0.15 each, and the fp32 partials through memory, a MB in half a us. No piece under 384 keys, and no more
// partials than `bytes`. Fitted to 450 times of heads of 128 (106 batches of prompts, chunks and decodes, heads 32 / 8, 24 / 8, 16 / 4 and 32 / 32,
// pieces from 256 keys to all of them): what it names is 2 % slower than the best piece on average; two workgroups a CU of equal key
// ranges, with the decodes in a launch of their own, 20 %. us, by that rule / by this: 1024 tokens alone 39.7 / 31.7, behind 2048 79 / 76; beside
// 16 sequences of 200 - 2500 keys 57 / 44, 97 / 88; 64 of 300 - 4000 beside 512 tokens 113 / 93, 128 of 2000 beside 32 196 / 182.
std::tuple<int64_t, int64_t> paged_prefill_plan(at::IntArrayRef keys, at::IntArrayRef tokens, int64_t nq, int64_t nkv, int64_t dim, int64_t bytes) {
  SXE_CHECK(!keys.empty() && keys.size() == tokens.size() && nq > 0 && nkv > 0 && dim > 0, "paged_prefill_plan: keys and tokens of every tile");
  int64_t most = 1, all = 0, steps = 0;
  for (size_t i = 0; i < keys.size(); ++i) {
    SXE_CHECK(keys[i] > 0 && tokens[i] > 0, "paged_prefill_plan: tiles of no keys or tokens");
    most = std::max(most, keys[i]);
    all += tokens[i];
    steps += (keys[i] + pp::KT - 1) / pp::KT;
  }
  const int64_t row = nq * dim * 4;
  std::tuple<int64_t, int64_t> best;
  double least = 1e30;
  for (int64_t s : {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20, 24, 32, 48, 64}) {
    const int64_t piece = (most + s * pp::KT - 1) / (s * pp::KT) * pp::KT, splits = (most + piece - 1) / piece;
    if (s > 1 && (piece < 384 || splits * all * row > bytes)) break;
    double us = std::max(1.6 * piece / pp::KT, steps * nkv / 190.0);
    if (splits > 1) {
      int64_t held = 0;
      for (size_t i = 0; i < keys.size(); ++i)
        if (keys[i] > piece) held += (keys[i] + piece - 1) / piece * tokens[i];
      us += 5.0 * ((splits + 15) / 16) + 0.15 * splits + (double)held * row / (1 << 21);
    }
    if (us < least) least = us, best = {splits, piece};
  }
  return best;
}

}  // namespace sxe

TORCH_LIBRARY_FRAGMENT(sxe, m) {
  m.def("paged_prefill_plan(int[] keys, int[] tokens, int nq, int nkv, int dim, int bytes) -> (int, int)", &sxe::paged_prefill_plan);
  m.def("paged_prefill(Tensor q, Tensor cache, Tensor block_table, Tensor q_start, Tensor q_len, Tensor kv_len, "
        "Tensor tiles, Tensor? rows, float scale, int window, int splits, int keys_per_split, Tensor(a!) out) -> ()");
}
TORCH_LIBRARY_IMPL(sxe, CUDA, m) { m.impl("paged_prefill", &sxe::paged_prefill); }
