"""Ragged (continuous-batching) forward for the Llama / Mixtral families over a paged KV cache.

Parity: reference inference/v2/model_implementations/llama_v2/model.py and mixtral/model.py
(``_forward_embed`` / ``_forward_transformer_layer`` / ``_forward_unembed``), with the module
choices the reference makes through its registry (blocked KV rotary, blocked flash, pre-RMS norm,
BLAS linear, cutlass MoE GEMM) replaced by this framework's gfx950 kernels:

  * RMSNorm with fused residual add (norm.hip), projections through hipBLASLt and, for few rows, the
    decode kernels (skinny_gemm.hip, stream_gemm.hip); up to 32 tokens the products' epilogues hold the residual
    sums, norms, RoPE and KV scatter (``_chain``), and a layer is its four products and the attention,
  * RoPE in place on the packed QKV (rope.hip), KV scatter into the blocked cache and paged
    attention (paged_attn.hip; sequences with many new tokens, with or without earlier ones, in one
    launch of the tile kernel, paged_prefill.hip; the longest prompts, flash_attn.hip),
  * SwiGLU (act.hip, or in the epilogue of the decode kernels); Mixtral experts routed on the device
    (experts_kn.hip, experts_kn_tile.hip),
  * only the last token of every sequence goes through the final norm + LM head.
The weights are the training modules' own parameters (no copy): a trained LlamaForCausalLM /
MixtralForCausalLM serves directly.

Tensor parallelism (``tp_group`` of size t; reference llama_v2/model.py:156 all-reduce after the
attention output and MLP down projections, :191 all-gather of the vocab-parallel logits): each rank
holds q heads / kv heads / FFN columns / vocab rows of its 1/t share (kv heads replicated when t
exceeds their count), its KV cache holds only its kv heads, and per layer exactly two all-reduces
(o_proj, down_proj) plus one logits all-gather per forward cross xGMI. The embedding and norms stay
replicated. MoE layers shard every expert's FFN columns (routing replicated, one all-reduce after
the experts); ``weight_quant`` quantizes each rank's slices.
"""
import os

import torch
import torch.nn.functional as F

from ....ops import native
from ....ops.activation import swiglu
from ....ops.linear import Linear, STREAM_ROWS_SMALL, TILED_GLU_ROWS, glu_faster, glu_linear, glu_tiled, is_own_forward, linear
from ....ops.linear import MERGE_COLUMNS, chain_faster, stream_glu, stream_head, stream_res, stream_res_splits, stream_rope, stream_weight
from ....ops.norm import RMSNorm
from ....ops.paged_attention import paged_attention_parts, paged_batch_attention, ragged_attention, rope_kv_cache_append
from ....ops.rows import embed_normed, gather_last


class _TPShards:
    """This rank's slices of every projection (copied once; the full weights can then be freed)."""

    def __init__(self, model, t, r, nq, nkv, D):
        assert nq % t == 0, f"query heads ({nq}) must divide by tp_size ({t})"
        assert nkv % t == 0 or t % nkv == 0, f"kv heads ({nkv}) and tp_size ({t}) must divide one another"
        self.nq = nq // t
        if nkv % t == 0:
            self.nkv, kv0 = nkv // t, r * (nkv // t)
        else:  # fewer kv heads than ranks: each rank keeps the kv head its q heads attend to
            self.nkv, kv0 = 1, (r * nq // t) // (nq // nkv)
        q0 = r * self.nq
        self.layers = []
        for layer in model.layers:
            a = layer.self_attn
            w = a.qkv_proj.weight
            q = w[q0 * D:(q0 + self.nq) * D]
            k = w[(nq + kv0) * D:(nq + kv0 + self.nkv) * D]
            v = w[(nq + nkv + kv0) * D:(nq + nkv + kv0 + self.nkv) * D]
            d = {"qkv": torch.cat([q, k, v]).contiguous(),
                 "o": a.o_proj.weight[:, q0 * D:(q0 + self.nq) * D].contiguous()}
            if hasattr(layer, "mlp"):
                mlp = layer.mlp
                inter = mlp.gate_up_proj.weight.shape[0] // 2
                assert inter % t == 0, f"intermediate size ({inter}) must divide by tp_size ({t})"
                c = inter // t
                gu = mlp.gate_up_proj.weight
                d["gu"] = torch.cat([gu[r * c:(r + 1) * c], gu[inter + r * c:inter + (r + 1) * c]]).contiguous()
                d["down"] = mlp.down_proj.weight[:, r * c:(r + 1) * c].contiguous()
            else:  # MoE: every expert's FFN columns (reference sharding/moe.py); routing replicated
                moe = (layer.block_sparse_moe if hasattr(layer, "block_sparse_moe") else layer.moe).deepspeed_moe
                ex = moe.experts
                inter = ex.w_down.shape[1]
                assert inter % t == 0, f"expert intermediate size ({inter}) must divide by tp_size ({t})"
                c = inter // t
                w = ex.w_gate_up  # [E, H, 2I]: x @ w
                d["e_gu"] = torch.cat([w[..., r * c:(r + 1) * c], w[..., inter + r * c:inter + (r + 1) * c]], -1).contiguous()
                d["e_down"] = ex.w_down[:, r * c:(r + 1) * c].contiguous()
            self.layers.append(d)
        V = model.lm_head.weight.shape[0]
        self.vshard = -(-V // t)
        self.vocab = V
        lo, hi = min(r * self.vshard, V), min((r + 1) * self.vshard, V)
        head = model.lm_head.weight[lo:hi]
        if hi - lo < self.vshard:  # pad the last shard so every rank gathers the same size
            head = torch.cat([head, head.new_zeros(self.vshard - (hi - lo), head.shape[1])])
        self.head = head.contiguous()


class RaggedLlama:
    def __init__(self, model, weight_quant=None, tp_group=None, tp_size=1, pins=None):
        from ..modules import heuristics as H
        self.model = model
        self.qw = None
        from .... import comm as dist
        self.tp_group = tp_group  # None with tp_size > 1: the world group
        self.tp = int(tp_size)
        if self.tp > 1:
            assert dist.get_world_size(tp_group) == self.tp, "tp_group size != tp_size"
        self.tp_rank = dist.get_rank(tp_group) if self.tp > 1 else 0
        p0 = next(model.parameters())
        dev = p0.device.type
        self._weight_quant, self._pins = weight_quant, pins
        if weight_quant and self.tp == 1:
            # linear implementations from the registry (modules/heuristics.py): quantized
            # weight-only GEMMs for decode-sized inputs, the bf16 weight on hipBLASLt otherwise
            self.qw = []
            for layer in model.layers:
                d = {"qkv": self._lin(layer.self_attn.qkv_proj.weight), "o": self._lin(layer.self_attn.o_proj.weight)}
                if hasattr(layer, "mlp"):
                    d["gu"] = self._lin(layer.mlp.gate_up_proj.weight)
                    d["down"] = self._lin(layer.mlp.down_proj.weight)
                self.qw.append(d)
            self.qhead = self._lin(model.lm_head.weight)
        self.cfg = model.cfg
        self.is_moe = hasattr(model.layers[0], "block_sparse_moe") or hasattr(model.layers[0], "moe")
        a0 = model.layers[0].self_attn
        self.nq, self.nkv, self.head_dim = a0.nq, a0.nkv, a0.d
        self.attn_impl = H.instantiate_attention(H.AttentionConfig(self.head_dim, self.nq, self.nkv, p0.dtype, 0, dev),
                                                 pins)
        emb = getattr(model.embed_tokens, "weight", None)
        self.embed_impl = H.instantiate_embed(H.EmbedConfig(emb.shape[0], emb.shape[1], emb.dtype, dev), emb, pins) \
            if emb is not None else None
        self.moe_impl = None
        # short passes wait for the host, those with experts for these: us a pass of two layers of 2048, experts of 8192 (0.8 GB), 2 prompts of 210
        # and 564 tokens 704, with own short products 717; of 3072 (1.2 GB), 18 and 62 710, 718
        self._host_bound = not self.is_moe
        if self.is_moe:
            l0 = model.layers[0]
            moe = (l0.block_sparse_moe if hasattr(l0, "block_sparse_moe") else l0.moe).deepspeed_moe
            self.moe_impl = H.instantiate_moe(H.MoEConfig(moe.gate.wg.weight.shape[0], moe.gate.k, dev), pins)
        self.implementations = {"attention": self.attn_impl.impl_name,
                                "embed": self.embed_impl.impl_name if self.embed_impl else "module",
                                "linear": self.qhead.impl_name if self.qw is not None else "module",
                                "moe": self.moe_impl.impl_name if self.moe_impl else None}
        self.num_layers = len(model.layers)
        self.vocab_size = self.cfg.vocab_size
        self.tps = None
        if self.tp > 1:
            self._full_heads = (self.nq, self.nkv)
            self._make_shards()
            self.nq, self.nkv = self.tps.nq, self.tps.nkv
            if self.qw is not None:
                self.implementations["linear"] = self.qhead.impl_name

    def _lin(self, w, bias=None):
        from ..modules import heuristics as H
        return H.instantiate_linear(H.LinearConfig(w.shape[1], w.shape[0], w.dtype, self._weight_quant, w.device.type),
                                    w, bias, self._pins)

    def _make_shards(self):
        self.tps = _TPShards(self.model, self.tp, self.tp_rank, *self._full_heads, self.head_dim)
        if self._weight_quant:  # quantize this rank's slices (row scales are per output row)
            self.qw = [{k: self._lin(v) for k, v in d.items() if k in ("qkv", "o", "gu", "down")}
                       for d in self.tps.layers]
            self.qhead = self._lin(self.tps.head)

    def refresh_shards(self):
        """Re-slice the tensor-parallel shards from the (updated) module weights -- the hybrid
        engine calls this before each generation, after training steps changed the weights."""
        if self.tps is not None:
            self._make_shards()

    @property
    def device(self):
        return next(self.model.parameters()).device

    @property
    def device_routing(self):
        """A MoE model's expert counts stay on the device at decode, so its steps can be captured."""
        from ....ops.moe import swiglu_experts_ok
        if not self.is_moe or self.tps is not None or self.device.type != "cuda" or not self.moe_impl.use_hip_gating:
            return False
        probe = torch.empty(0, self.cfg.hidden_size, dtype=self.dtype, device=self.device)
        moes = [(x.block_sparse_moe if hasattr(x, "block_sparse_moe") else x.moe).deepspeed_moe for x in self.model.layers]
        return all(m.ep_size == 1 and hasattr(m.experts, "w_gate_up") and m.gate.wg.weight.dtype == self.dtype
                   and swiglu_experts_ok(probe, m.experts.w_gate_up, m.experts.w_down) for m in moes)

    @property
    def dtype(self):
        return next(self.model.parameters()).dtype

    def _attention(self, qkv, kv_layer, batch):
        pinned = (self._pins or {}).get("attention") == "dense_blocked_attention"
        q, scale = qkv[:, :self.nq], self.head_dim ** -0.5
        return paged_batch_attention(q, kv_layer, batch, scale) if pinned else ragged_attention(q, kv_layer, batch, scale, kv=qkv[:, self.nq:])

    def _proj(self, mod, x, li, key):
        if self.tps is not None:
            if self.qw is not None:
                y = self.qw[li][key](x)
            else:
                y = linear(x, self.tps.layers[li][key])
            if key in ("o", "down"):  # row-parallel: partial sums over this rank's heads / FFN columns
                from .... import comm as dist
                dist.all_reduce(y, group=self.tp_group)
            return y
        # FP8 weights pay off where the GEMM is weight-streaming bound (<= 16 rows: W8A16 skinny
        # kernel); larger batches keep the module's bf16 weight on hipBLASLt
        if self.qw is not None and key in self.qw[li]:
            return self.qw[li][key](x)
        return linear(x, mod.weight, mod.bias, self._host_bound) if is_own_forward(mod, Linear) else mod(x)

    # decode (<= 4 tokens) of a model that ``_chain`` does not cover, be it for one projection that is more than its product, one norm weight
    # of another type or heads of another size: RMSNorm folded into the QKV / gate_up GEMMs as their prologue, SwiGLU into gate_up's
    # epilogue (skinny_gemm.hip) -- three latency-bound launches fewer per layer
    FUSE_MAX_T = 4

    def _fusable(self, T):
        return (self.tps is None and T <= self.FUSE_MAX_T and not self.is_moe and self.device.type == "cuda" and native.hip_available()
                and os.environ.get("SXE_DECODE_FUSE", "1") == "1")

    def _attn_o(self, attn, qkv, kv_layer, batch, li, T):
        """Attention + o_proj outside ``_chained``. One token: the KV-split merge runs inside the o_proj GEMM launch
        (paged_attention_parts + fused_merge_linear) -- one latency-bound launch fewer per layer. More tokens: every workgroup
        of that launch would read all of their partials; 4 sequences of 4000 keys, 4 layers of Llama-8B: 704 us a step so, 658
        with a merge launch (1 sequence: 548 / 547; 2: 602 / 581)."""
        if (T == 1 and self._fusable(T) and getattr(attn.o_proj, "bias", None) is None and native.use_hip(qkv)
                and os.environ.get("SXE_DECODE_FUSE_ATTN", "1") == "1"):
            from ....ops.linear import _pro_weight, fused_merge_linear
            w = self._wobj(attn.o_proj, li, "o")
            if _pro_weight(w) is not None:
                out, parts = paged_attention_parts(qkv[:, :self.nq], kv_layer, batch.block_table, batch.q_start,
                                                   batch.q_len, batch.kv_len, self.head_dim ** -0.5, batch.max_kv_len)
                if parts is not None:
                    y = fused_merge_linear(parts[0], parts[1], w)
                    if y is not None:
                        return y
                    from ....ops.paged_attention import merge_attention_parts
                    out = merge_attention_parts(parts[0], parts[1], qkv.dtype)  # keep the computed splits
                return self._proj(attn.o_proj, out.reshape(T, self.nq * self.head_dim), li, "o")
        o = self._attention(qkv, kv_layer, batch)
        return self._proj(attn.o_proj, o.reshape(T, self.nq * self.head_dim), li, "o")

    def _wobj(self, mod, li, key):
        """The weight that a fused launch reads in place of running ``mod``; None where the module is more than its product."""
        if self.qw is not None and key in self.qw[li]:
            return self._impl_weight(self.qw[li][key])
        return mod.weight if is_own_forward(mod, Linear, torch.nn.Linear) else None

    @staticmethod
    def _impl_weight(impl):
        return getattr(impl, "q", None) if getattr(impl, "q", None) is not None else getattr(impl, "weight", None)

    def _norm_proj(self, norm, x, res, mod, li, key):
        """(norm(x + res) @ W^T, h) through the fused kernel, else the separate launches."""
        if self._fusable(x.shape[0]) and getattr(mod, "bias", None) is None and is_own_forward(norm, RMSNorm):
            from ....ops.linear import fused_rms_linear
            r = fused_rms_linear(x, res, norm.weight, norm.eps, self._wobj(mod, li, key))
            if r is not None:
                return r
        a, h = (norm(x), x) if res is None else norm(x, res)
        return self._proj(mod, a, li, key), h

    def _norm_glu(self, layer, x, res, li):
        """(silu(gate) * up of the normed residual sum, the sum); the activation in the GEMM's epilogue at decode and for
        many tokens, the norm in its prologue up to 4."""
        mlp, norm, T = layer.mlp, layer.post_attention_layernorm, x.shape[0]
        w = None
        few = T <= STREAM_ROWS_SMALL  # between these and the many rows there is no such product: host-bound passes, and asking is 10 us a layer
        if (self.tps is None and (few or T > TILED_GLU_ROWS) and (T > self.FUSE_MAX_T or self._fusable(T)) and self.device.type == "cuda"
                and getattr(mlp.gate_up_proj, "bias", None) is None and native.hip_available()):
            w = self._wobj(mlp.gate_up_proj, li, "gu")
            if T > 16 and self.qw is not None:  # quantized layers run more than 16 rows on the weight as it came
                w = self.qw[li]["gu"].weight
        if w is not None and T <= self.FUSE_MAX_T and is_own_forward(norm, RMSNorm):
            from ....ops.linear import fused_rms_glu
            r = fused_rms_glu(x, res, norm.weight, norm.eps, w)
            if r is not None:
                return r
        a, h = norm(x, res)
        if w is not None:
            mid = (glu_linear(a, w) if glu_faster(T, w) else None) if few else glu_tiled(a, w)
            if mid is not None:
                return mid, h
        return swiglu(self._proj(mlp.gate_up_proj, a, li, "gu")), h

    def _chain(self, T, batch, kv_cache, rope):
        """Per layer the weights of its products, where all of them (up to 32 rows) run the streaming kernel with the residual sums, norms,
        RoPE and the cache's append in their epilogues; None otherwise. MoE layers: of the first product alone."""
        if not (0 < T <= STREAM_ROWS_SMALL and self.tps is None and self.device.type == "cuda" and self.head_dim == 128
                and native.hip_available() and rope.cos.shape[-1] == 64 and rope.cos.dtype == torch.float32
                and os.environ.get("SXE_DECODE_FUSE", "1") == "1" and os.environ.get("SXE_DECODE_FUSE_ATTN", "1") == "1"):
            return None
        small = self.qw is None or T <= 16  # quantized layers run more rows on the weight as it came

        def weight(mod, li, key, columns=16):
            if getattr(mod, "bias", None) is not None:
                return None
            w = self._wobj(mod, li, key) if small else self.qw[li][key].weight
            return None if w is None else stream_weight(w, T, columns)

        def normed(n):  # four weights a load: one may lie anywhere in a buffer of many
            return is_own_forward(n, RMSNorm) and n.weight.dtype == torch.bfloat16 and n.weight.data_ptr() % 8 == 0
        out = []
        for li, layer in enumerate(self.model.layers):
            kv, mlp = kv_cache.layer(li), getattr(layer, "mlp", None)
            if (not kv.is_contiguous() or kv.dim() != 5 or kv.dtype != torch.bfloat16 or kv.shape[2] != self.nkv
                    or not normed(layer.input_layernorm) or not normed(layer.post_attention_layernorm)):
                return None
            ws = [weight(layer.self_attn.qkv_proj, li, "qkv")]
            if mlp is not None:
                ws += [weight(layer.self_attn.o_proj, li, "o"), weight(mlp.gate_up_proj, li, "gu", 32), weight(mlp.down_proj, li, "down")]
            if any(w is None for w in ws) or not chain_faster(T, ws) or ws[0][0].shape[0] != (self.nq + 2 * self.nkv) * 128:
                return None
            out.append(ws)
        return out if normed(self.model.norm) else None

    def _embed(self, ids):
        return self.embed_impl(ids) if self.embed_impl is not None else self.model.embed_tokens(ids)

    def _chained(self, batch, kv_cache, rope, chain):
        """The layers and the head with ``_chain``'s weights: logits."""
        model, T = self.model, batch.num_tokens
        from ..modules.implementations import RaggedEmbedding
        own = type(self.embed_impl) is RaggedEmbedding
        first = embed_normed(self.embed_impl.weight, batch.input_ids, model.layers[0].input_layernorm.weight) if own and chain else None
        a, h, sums = first or (None, None, None)
        x = self._embed(batch.input_ids) if first is None else h
        for li, (layer, ws) in enumerate(zip(model.layers, chain)):
            kv_layer, norm = kv_cache.layer(li), layer.input_layernorm
            if a is None:
                a, h = (norm(x), x) if h is None else norm(x, h)
            qkv = stream_rope(a, ws[0], sums, norm.eps, rope, batch.positions, kv_layer, batch.slots, self.nq, self.nkv)
            qkv, norm = qkv.view(T, self.nq + 2 * self.nkv, self.head_dim), layer.post_attention_layernorm
            if T == 1 and len(ws) > 1 and max(ws[1][0].shape) <= MERGE_COLUMNS:  # the splits' merge in the o product's launch
                o, parts = paged_attention_parts(qkv[:, :self.nq], kv_layer, batch.block_table, batch.q_start, batch.q_len, batch.kv_len,
                                                 self.head_dim ** -0.5, batch.max_kv_len)
            else:
                o, parts = self._attention(qkv, kv_layer, batch), None
            o = o.reshape(T, self.nq * self.head_dim) if parts is None else None
            if len(ws) == 1:
                m, h = norm(self._proj(layer.self_attn.o_proj, o, li, "o"), h)
                x, a, sums = self._moe(layer, m, li), None, None
                continue
            a, h, sums = stream_res(o, ws[1], h, norm.weight) if parts is None else stream_res_splits(parts, ws[1], h, norm.weight)
            mid = stream_glu(a, ws[2], sums, norm.eps)
            after = model.layers[li + 1].input_layernorm if li + 1 < len(chain) else model.norm
            a, h, sums = stream_res(mid, ws[3], h, after.weight)
        if a is not None and getattr(batch, "every_token", False):
            w = model.lm_head.weight if self.qw is None else self._impl_weight(self.qhead)
            wk = stream_weight(w, T, 4) if w is not None else None
            if wk is not None:
                return stream_head(a, wk, sums, model.norm.eps)
        x = gather_last(x, batch.last_idx, h) if a is None else gather_last(h, batch.last_idx)
        return self._head(model.norm(x))

    def _moe(self, layer, m, li):
        moe = layer.block_sparse_moe if hasattr(layer, "block_sparse_moe") else layer.moe
        if self.tps is not None:  # this rank's expert columns -> partial sums -> one all-reduce
            d = self.tps.layers[li]
            y = self._moe_dropless(moe.deepspeed_moe, m, d["e_gu"], d["e_down"])
            from .... import comm as dist
            dist.all_reduce(y, group=self.tp_group)
            return y
        return self._moe_dropless(moe.deepspeed_moe, m)

    def _moe_dropless(self, moe, m, w_gu=None, w_down=None):
        """Exact top-k routing for inference (no capacity, no dropped tokens): tokens are grouped
        by expert, each expert runs its two GEMMs on its rows, results are gathered back weighted by the
        renormalised top-k gate probabilities (reference ragged_ops/top_k_gating + moe_scatter +
        moe_gather): on the device where the expert kernels cover the sizes (ops/moe.swiglu_experts),
        else with an argsort and a loop over the experts."""
        gate, ex = moe.gate, moe.experts
        assert moe.ep_size == 1, "ragged inference runs experts locally (ep_size == 1)"
        w_gu = ex.w_gate_up if w_gu is None else w_gu
        w_down = ex.w_down if w_down is None else w_down
        k = gate.k
        from ....ops.moe import route_logits, route_topk, swiglu_experts, swiglu_experts_ok
        if (self.moe_impl is not None and self.moe_impl.use_hip_gating and swiglu_experts_ok(m, w_gu, w_down)):
            wg = gate.wg.weight
            routing = (route_topk(m, wg, k) if wg.dtype == m.dtype and wg.is_contiguous()
                       else route_logits(F.linear(m.float(), wg.float()), k))
            return swiglu_experts(m, routing, w_gu, w_down)
        logits = F.linear(m.float(), gate.wg.weight.float())
        if self.moe_impl is not None and self.moe_impl.use_hip_gating and logits.is_cuda:
            from ....ops.moe import topk_softmax  # fused softmax + top-k kernel (moe.hip)
            probs, topi = topk_softmax(logits, k)
            topw = probs.gather(1, topi)
        else:
            probs = torch.softmax(logits, dim=-1)
            topw, topi = probs.topk(k, dim=-1)
        topw = topw / topw.sum(-1, keepdim=True)
        flat = topi.reshape(-1)
        order = torch.argsort(flat, stable=True)
        tok = order // k
        counts = torch.bincount(flat, minlength=ex.num_local_experts).tolist()
        xs = m.index_select(0, tok)
        ws = topw.reshape(-1).index_select(0, order).to(m.dtype).unsqueeze(1)
        out = torch.zeros_like(m)
        o = 0
        for e, c in enumerate(counts):
            if c == 0:
                continue
            y = torch.matmul(swiglu(torch.matmul(xs[o:o + c], w_gu[e])), w_down[e])
            out.index_add_(0, tok[o:o + c], y * ws[o:o + c])
            o += c
        return out

    @torch.no_grad()
    def forward(self, batch, kv_cache):
        model = self.model
        rope = model.rope(self.device)
        if batch.max_kv_len > rope.max_pos:  # the HIP RoPE kernels index the cos/sin table unchecked
            raise ValueError(f"sequence length {batch.max_kv_len} exceeds the model's RoPE table "
                             f"({rope.max_pos} positions, max_position_embeddings)")
        T = batch.num_tokens
        chain = self._chain(T, batch, kv_cache, rope)
        if chain is not None:
            return self._chained(batch, kv_cache, rope, chain)
        x = self._embed(batch.input_ids)
        res = None
        for li, layer in enumerate(model.layers):
            attn = layer.self_attn
            kv_layer = kv_cache.layer(li)
            r = None
            if (self._fusable(T) and self.head_dim == 128 and getattr(attn.qkv_proj, "bias", None) is None
                    and is_own_forward(layer.input_layernorm, RMSNorm) and os.environ.get("SXE_DECODE_FUSE_ATTN", "1") == "1"):
                # decode: RMSNorm prologue + QKV GEMM + RoPE / KV-append epilogue in one launch
                from ....ops.linear import fused_rms_rope_linear
                ln = layer.input_layernorm
                r = fused_rms_rope_linear(x, res, ln.weight, ln.eps, self._wobj(attn.qkv_proj, li, "qkv"), rope,
                                          batch.positions, kv_layer, batch.slots, self.nq, self.nkv)
            if r is not None:
                qkv, h = r
                qkv = qkv.view(T, self.nq + 2 * self.nkv, self.head_dim)
                o = self._attn_o(attn, qkv, kv_layer, batch, li, T)
            else:
                qkv, h = self._norm_proj(layer.input_layernorm, x, res, attn.qkv_proj, li, "qkv")
                qkv = qkv.view(T, self.nq + 2 * self.nkv, self.head_dim)
                # RoPE on q/k + append of k/v to the paged cache: one launch (paged_attn.hip)
                rope_kv_cache_append(qkv, rope, batch.positions, kv_layer, batch.slots, self.nq, self.nkv)
                o = self._attn_o(attn, qkv, kv_layer, batch, li, T)
            if hasattr(layer, "mlp"):
                mid, res = self._norm_glu(layer, o, h, li)
                x = self._proj(layer.mlp.down_proj, mid, li, "down")
            else:
                m, res = layer.post_attention_layernorm(o, h)
                x = self._moe(layer, m, li)
        last = batch.last_idx
        x = gather_last(x, last, res)
        if self._fusable(x.shape[0]) and is_own_forward(model.norm, RMSNorm):
            from ....ops.linear import RMS_GLU_BF16, RMS_GLU_FP8, _pro_weight, fused_rms_linear
            w = model.lm_head.weight if self.qw is None else self._impl_weight(self.qhead)
            wk = _pro_weight(w)
            # one launch for the norm and the head, where building its input in every workgroup costs less than a launch
            if wk is not None and x.numel() <= (RMS_GLU_BF16 if wk[1] is None else RMS_GLU_FP8):
                r = fused_rms_linear(x, None, model.norm.weight, model.norm.eps, w)
                if r is not None:
                    return r[0].float()
        h = model.norm(x)
        if self.tps is not None:  # vocab-parallel head: gather every rank's logit columns
            from .... import comm as dist
            part = (self.qhead(h) if self.qw is not None else linear(h, self.tps.head)).float()
            full = torch.empty(self.tp * part.shape[0], part.shape[1], dtype=part.dtype, device=part.device)
            dist.all_gather_into_tensor(full, part, group=self.tp_group)
            return full.view(self.tp, -1, part.shape[1]).permute(1, 0, 2).reshape(part.shape[0], -1)[:, :self.tps.vocab]
        return self._head(h)

    def _head(self, h):
        return (self.qhead(h) if self.qw is not None else linear(h, self.model.lm_head.weight)).float()
