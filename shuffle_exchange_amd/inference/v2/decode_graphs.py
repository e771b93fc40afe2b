"""HIP-graph replay of decode steps for the ragged engine.

A decode step of a dense model (every sequence adds ONE token) is launch-bound at serving batch
sizes: Llama-3-8B issues 6 kernels per layer up to 32 sequences (four products with norms, RoPE, KV append,
residual sums and SwiGLU inside, paged attention, split merge) and ~10 beyond, i.e. 200 - 330 launches per
token, while the HBM time of the step is ~2 ms. The reference captures CUDA graphs only in its v1 engine
(inference/engine.py ``_create_cuda_graph``); here the v2 engine captures its decode steps:

* graphs are keyed by (sequence bucket, KV-length bucket), powers of two (of sequences also 12 and 24, with experts 48, ..), and where the attention kernel splits the
  keys otherwise for them, by whether the sequences are about as long as one another; captured lazily on first use and
  sharing one memory pool;
* all per-step metadata (token ids, positions, cache slots, block tables, lengths) lives in static
  device buffers refreshed by one pinned H2D copy before ``replay()``;
* padding sequences point at a reserved scratch KV block and state slot (q_len = kv_len = 1), so every
  row the graph computes is well defined and no real cache slot is touched;
* the paged-attention grid is fixed per graph by the KV bucket (splits of at most 512 keys while their partials
  are small, ops/paged_attention.decode_plan; workgroups past a sequence's length exit at once).

MoE models whose expert counts go through the host, sliding windows narrower than the KV bucket and modules whose
weights are made anew for every generation (hybrid engine) run eagerly.
"""
import numpy as np
import torch

from ...ops.paged_attention import decode_plan, even_lengths

MIN_KV_BUCKET = 256


def _pow2_at_least(n, lo=1):
    b = lo
    while b < n:
        b *= 2
    return b


def sequence_bucket(n, experts=False):
    """Rows of the graph that runs ``n`` sequences: powers of two and, from 8 on, what lies half way. Padding rows cost their part of the products
    and of attention's workgroups, and choose experts that no sequence needs; every bucket is captured by itself. us a step of two layers at the
    next power of two / here: 9 sequences of 8b 299 / 292, in e4m3 237 / 227, 17 379 / 366; of Mixtral 20 1427 / 1245, 33 1667 / 1313. Not from 33 on
    without experts, whose products the library runs: 41 of 3b 299 / 308, 40 of 8b 444 / 461. (5 in e4m3 206, as 6 199.) Other decoders, 9 and 24
    sequences: RaggedDecoder, two layers of 8b 296 / 290, 381 / 374, of 3b 201 / 196, 263 / 257, of 1b 163.5 / 162.9, 191.9 / 192.1; eight layers of Tobinex 8b 1132
    / 1107, 1454 / 1427, 1b 655 / 650, 771 / 746; of Bipotar 8b, with experts, 1514 / 1456, 1885 / 1748, 1b 664 / 642, 800 / 744."""
    p = _pow2_at_least(n)
    return p // 4 * 3 if 8 < p <= (256 if experts else 32) and n <= p // 4 * 3 else p


class _StaticBatch:
    """RaggedBatch protocol (see ragged.py) over fixed-shape device buffers."""

    def __init__(self, S, max_blocks, kv_bucket, device, even=False):
        self.num_tokens = self.num_seqs = S
        self.max_blocks = max_blocks
        self.max_kv_len = kv_bucket
        self.even_lengths = even
        self.every_token = True  # the logits are those of every row, in order
        n64, n32 = 32 * S, 16 * S + 4 * S * max_blocks  # bytes: one copy brings both
        self.dev = torch.zeros(n64 + n32, dtype=torch.uint8, device=device)
        self.host = torch.zeros(n64 + n32, dtype=torch.uint8, pin_memory=True)
        self.d64, self.d32 = self.dev[:n64].view(torch.int64), self.dev[n64:].view(torch.int32)
        self.h64, self.h32 = self.host[:n64].view(torch.int64), self.host[n64:].view(torch.int32)
        self.input_ids, self.positions, self.slots, self.last_idx = self.d64.view(4, S).unbind(0)
        self.q_start, self.q_len, self.kv_len, self.state_slots = self.d32[:4 * S].view(4, S).unbind(0)
        self.block_table = self.d32[4 * S:].view(S, max_blocks)
        # host views read by the attention dispatch: no pure prefill, every row one query token
        self.host_seen = [1] * S
        self.host_q_len = [1] * S
        self.host_q_start = list(range(S))
        self.host_kv_len = [kv_bucket] * S
        self.rows = torch.arange(S, dtype=torch.int32, device=device)[:, None].repeat(1, 2)
        self.order = np.arange(S)
        self.copied = None  # event: last H2D copy out of the pinned buffers

    def token_rows(self, below=None):
        return self.rows


class DecodeGraphRunner:
    def __init__(self, model, kv_cache, max_seqs=256, max_context=131072):
        self.model, self.kv = model, kv_cache
        self.max_seqs = max_seqs
        self.max_context = max_context
        self.bs = kv_cache.block_size
        self.scratch_block = int(kv_cache.reserve(1)[0])
        self.scratch_state = -1
        if kv_cache.states is not None:
            self.scratch_state = kv_cache.states.reserve()
            for t in kv_cache.states.layers:
                if t is not None:
                    t[self.scratch_state].zero_()
        self._graphs = {}
        self._matters = {}
        self._pool = None
        self.replays = 0

    # ------------------------------------------------------------------------------ eligibility
    def eligible(self, seqs, lens):
        if not lens or any(n != 1 for n in lens) or len(seqs) > self.max_seqs:
            return False
        kv_max = max(s.seen_tokens + 1 for s in seqs)
        if kv_max > self.max_context:
            return False
        window = getattr(getattr(self.model, "spec", None), "sliding_window", None)
        if window is not None and self._kv_bucket(kv_max) > window:
            return False
        return True

    def _kv_bucket(self, kv_max):
        return max(_pow2_at_least(kv_max, MIN_KV_BUCKET), self.bs)

    def _even(self, S, kvb, seqs):
        """The sequences are about as long as one another, and attention splits their keys otherwise then."""
        matters = self._matters.get((S, kvb))
        if matters is None:
            nq, nkv, dim = (getattr(self.model, name, None) for name in ("nq", "nkv", "head_dim"))
            plans = [decode_plan(S, nkv, kvb, 4 * S * nq * dim, even, dim) for even in (True, False)] if nq and nkv and dim else (1, 1)
            matters = self._matters[S, kvb] = plans[0] != plans[1]
        return matters and even_lengths([s.seen_tokens + 1 for s in seqs])

    # ------------------------------------------------------------------------------------- run
    def run(self, seqs, tokens):
        S_real = len(seqs)
        S = sequence_bucket(S_real, getattr(self.model, "is_moe", False))
        kvb = self._kv_bucket(max(s.seen_tokens + 1 for s in seqs))
        even = self._even(S, kvb, seqs)
        key = (S, kvb, even)
        entry = self._graphs.get(key)
        sb = entry[1] if entry is not None else _StaticBatch(S, (kvb + self.bs - 1) // self.bs, kvb,
                                                              self.model.device, even)
        self._fill(sb, seqs, tokens)
        if entry is None:
            entry = self._capture(sb)
            self._graphs[key] = entry
        graph, _, out = entry
        graph.replay()
        self.replays += 1
        return out[:S_real].clone()

    def _fill(self, sb, seqs, tokens):
        if sb.copied is not None:
            sb.copied.synchronize()  # the previous step's copy has left the pinned buffers
        S, mb, bs, n = sb.num_seqs, sb.max_blocks, self.bs, len(seqs)
        # numpy views of the pinned buffers: a small numpy operation costs a tenth of a tensor one (24 sequences:
        # 740 us of host time with tensors, 165 us so)
        ids, pos, slots, last = sb.h64.numpy().reshape(4, S)
        qs, ql, kl, ss = sb.h32.numpy()[:4 * S].reshape(4, S)
        bt = sb.h32.numpy()[4 * S:].reshape(S, mb)
        p = np.array([s.seen_tokens for s in seqs], dtype=np.int64)
        ids[:n] = torch.cat([t.reshape(-1)[:1].to("cpu", torch.int64) for t in tokens]).numpy()
        pos[:n] = p
        slots[:n] = np.array([s.blocks[s.seen_tokens // bs] for s in seqs], dtype=np.int64) * bs + p % bs
        last[:] = qs[:] = sb.order
        ql.fill(1)
        kl[:n] = p + 1
        ss[:n] = [s.state_slot for s in seqs]
        for i, s in enumerate(seqs):
            nb = len(s.blocks)
            bt[i, :nb] = s.blocks
            bt[i, nb:] = self.scratch_block
        ids[n:] = pos[n:] = 0  # rows past the batch: one key in the scratch block
        slots[n:], kl[n:], ss[n:], bt[n:] = self.scratch_block * bs, 1, self.scratch_state, self.scratch_block
        sb.dev.copy_(sb.host, non_blocking=True)
        ev = torch.cuda.Event()
        ev.record()
        sb.copied = ev

    def _capture(self, sb):
        if self._pool is None:
            self._pool = torch.cuda.graph_pool_handle()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side), torch.no_grad():
            # warm-up: lazy inits, hipBLASLt heuristics. KV writes land where the replay writes again; a
            # recurrent state must advance once only, so this pass works on the scratch slot
            slots = sb.state_slots.clone()
            sb.state_slots.fill_(self.scratch_state)
            self.model.forward(sb, self.kv)
            sb.state_slots.copy_(slots)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, pool=self._pool), torch.no_grad():
            out = self.model.forward(sb, self.kv)
        return graph, sb, out

    @property
    def num_graphs(self):
        return len(self._graphs)
