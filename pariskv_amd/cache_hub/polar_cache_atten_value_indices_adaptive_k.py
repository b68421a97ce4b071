"""Dense-form adaptive-k variant of the retrieval cache (reference:
``cache_hub/polar_cache_atten_value_indices_adaptive_k.py``).

Like :mod:`polar_cache_adaptivek_varlen`, every decode step ranks the candidates of each (batch, kv-head) row by
``exp(logit) * ||v||`` and finds the smallest k whose mass, together with the dense sink/local tokens, reaches
``adaptive_topk_threshold`` of the total.  What differs (reference ``:1298-1589``):

* k is capped by ``adaptive_topk_max_k`` (default 2048, also the size of the gathered-row buffer) and has no lower
  clamp (``:1564-1577``);
* the attended set is dense: every row keeps ``global_k = max over rows of k`` ids of its own benefit order
  (``:1585-1589``, ``:1462-1499``), so rows with a small k still attend to the next-best candidates of their list.
  The reference reads ``global_k`` back to the host to size its tensors; here the attention takes the maximum over the
  rows on the device (with K/V on the host a one-workgroup kernel broadcasts it, for the gather too), so the step has no
  host synchronisation;
* both storage modes are supported: with ``enable_offload=False`` the K/V rows and the value norms live at their
  absolute positions on the GPU (``:377-381``, ``:1086``, ``:967``) and the selected rows are attended in place through
  the index list.
"""
from __future__ import annotations

import torch

from .. import ops, ranges
from .polar_cache import polar_cache as _polar_cache_base
from .polar_cache_adaptivek_varlen import polar_cache as _adaptive_base


class polar_cache(_adaptive_base):
    def __init__(self, valid_start, layer_num, batch_size, max_length, num_key_value_heads, num_heads, head_dim, dtype,
                 layer_mapping, max_new_length, sink_size, local_size, core=0, nprobe=0, cache_unit_size=0,
                 cache_cluster_num=0, num_gpus=1, model_size=0, codebook_path=None, collision_ratio: float = 0.3,
                 candidate_ratio: float = 0.05, final_topk: int = 100, dynamic_update_interval: int = 512,
                 full_attention_threshold: int = 2000, enable_offload: bool = True, enable_recall: bool = False,
                 adaptive_topk_threshold: float = 0.9, adaptive_topk_max_k: int = 2048) -> None:
        # the two ratios are stored (:197-198); the per-step ratios come from the retrieval length (:1825-1845)
        _polar_cache_base.__init__(self, valid_start, layer_num, batch_size, max_length, num_key_value_heads, num_heads,
                                   head_dim, dtype, layer_mapping, max_new_length, sink_size, local_size, core, nprobe,
                                   cache_unit_size, cache_cluster_num, num_gpus, model_size, codebook_path=codebook_path,
                                   final_topk=final_topk, dynamic_update_interval=dynamic_update_interval,
                                   full_attention_threshold=full_attention_threshold, enable_offload=enable_offload)
        self.collision_ratio = collision_ratio
        self.candidate_ratio = candidate_ratio
        self.enable_recall = enable_recall
        self.adaptive_topk_threshold = adaptive_topk_threshold
        self.adaptive_topk_max_k = int(adaptive_topk_max_k) if adaptive_topk_max_k is not None else final_topk  # :201
        self._init_adaptive_state(self.adaptive_topk_max_k, uniform_k=True)

    def _caps(self, cand_len):
        """(topk_cap, k_min, k_max): k in [1, min(adaptive_topk_max_k, cand_len)] (:1564, :1574-1582)."""
        cap = max(1, min(self.adaptive_topk_max_k, cand_len))
        return cap, 1, cap

    # ------------------------------------------------ value-norm bookkeeping
    def _norm_targets(self, layer_idx, b0, b1, abs0, n_encode):
        targets = super()._norm_targets(layer_idx, b0, b1, abs0, n_encode)
        if not self.enable_offload and n_encode > 0:
            # every token at its absolute position (:611-614); the retrieval zone's norms also by position (:634-637)
            targets["zone_vnorm2"] = self._sl_vnorm_cache[layer_idx][b0:b1, :, abs0:abs0 + n_encode]
        return targets

    def _on_refresh(self, layer_idx, r):
        if self.enable_offload:
            return super()._on_refresh(layer_idx, r)
        a0, n = r.encode_abs0, r.n_new
        self.value_norm_gpu[layer_idx][:, :, a0:a0 + n] = self._sl_vnorm_cache[layer_idx][:, :, a0:a0 + n]  # :967

    # ---------------------------------------------------------------- compute
    def _compute_adaptive_topk(self, query_avg, sink_local_keys, sl_vnorm, all_cand_scores, all_cand_indices, layer_idx,
                               threshold: float = 0.9):
        """The reference's return form (:1508-1589): (adaptive_k [bs,H] int64, topk_indices [bs,H,global_k] int64 in
        descending benefit order, global_k int).  Reads k back to the host; :meth:`compute` does not go through here."""
        adaptive_k, topk_ids, _ = self._adaptive_topk_device(query_avg, sink_local_keys, sl_vnorm, all_cand_scores,
                                                             all_cand_indices, layer_idx, threshold)
        global_k = int(adaptive_k.max().item())
        return adaptive_k, topk_ids[:, :, :global_k].contiguous(), global_k

    def compute(self, queries, layer_idx):
        """Decode attention for one token: [bs,1,Hq,D] -> [bs,1,Hq,D] (reference :1298-1502)."""
        if self.enable_offload:
            return super().compute(queries, layer_idx)  # the fused step, with the broadcast of max k switched on
        z = self._zones[layer_idx]
        total, n_keys = z.seq_len, z.encoded
        if total < self._min_total() or n_keys <= 0:
            return _polar_cache_base.compute(self, queries, layer_idx)  # dense branch
        q = queries if queries.is_contiguous() else queries.contiguous()
        step = self._adaptive_bound[layer_idx]
        if step is None or step[0] != n_keys or step[3] != self.adaptive_topk_max_k:
            step = self._bind_adaptive_step(layer_idx, q, n_keys)
        _, bound, local_seg, _ = step
        # what moves with every token: the local window grows by one; k goes to a tensor of its own, as the caller may keep it.
        # adaptive_topk_threshold and adaptive_topk_max_k hold for the next step, whenever they are set.
        dense = z.gpu_prefix_rows
        bound.ad.threshold = float(self.adaptive_topk_threshold)
        bound.ad.dense_rows = bound.ad.row_keys_base = dense
        bound.segs[local_seg].n_rows = z.dense_tail_len
        self.last_adaptive_k = torch.empty_like(self._adaptive_k)
        bound.ad.adaptive_k = self.last_adaptive_k.data_ptr()
        # one host call, as in the offloading form; the dense rows (two runs: sink, local) and the selected ones are read
        # where they lie
        if ranges.enabled:
            with ranges.span("collision_topk+adaptive_k+attention_varlen"):
                return bound.launch(q)
        return bound.launch(q)

    def _bind_adaptive_step(self, layer_idx, q, n_keys):
        if self.enable_offload:
            return super()._bind_adaptive_step(layer_idx, q, n_keys)
        z, S0 = self._zones[layer_idx], self.sink_size
        n_keys, n_cand, _, tiers = self.retrieval_shape(layer_idx)
        topk_cap, k_min, k_max = self._caps(n_cand)
        kg, vg = self.unified_keys_gpu[layer_idx], self.unified_values_gpu[layer_idx]
        bs, H = self.batch_size, self.kv_head
        need = ops.adaptive_topk_ws_bytes(self.batch_groups, n_cand, topk_cap)
        if self._adk_ws is None or self._adk_ws.numel() < need:
            self._adk_ws = self._larger(self._adk_ws, need, torch.uint8)
        if self._dense_vnorm_run is None:
            self._dense_vnorm_run = torch.empty_like(self._dense_logits)
        if self._topk_ids.numel() < bs * H * topk_cap:   # adaptive_topk_max_k was raised; bound steps keep the tensor they name
            self._topk_ids = self._larger(self._topk_ids, bs * H * topk_cap, torch.int64)
        local0, dense = z.local_start, z.gpu_prefix_rows
        adaptive = dict(dense_k=kg, dense_rows=dense, dense_split=S0, dense_row1=local0, dense_vnorm=self._sl_vnorm_cache[layer_idx],
                        dense_vnorm_run=self._dense_vnorm_run, dense_logits=self._dense_logits, scale=self._attn_scale,
                        value_norm=self.value_norm_gpu[layer_idx], vn_offset=S0, record_word_offset=ops.RECORD_VALUE_NORM_OFFSET,
                        threshold=self.adaptive_topk_threshold, k_out=topk_cap, k_min=k_min, k_max=k_max,
                        adaptive_k=self._adaptive_k, topk_ids=self._topk_ids, row_keys=self._row_keys, row_keys_base=dense,
                        row_keys_uniform=True, ws=self._adk_ws, src_k=None, src_v=None, dst_k=None, dst_v=None)
        ids = self._topk_ids[:bs * H * topk_cap].view(bs, H, topk_cap)
        # the selected rows come last so that the per-row key count cuts inside them (the reference gathers copies, :1481-1488)
        segments = [(kg, vg, 0, S0), (kg, vg, local0, z.dense_tail_len), (kg, vg, S0, topk_cap, ids)]  # runs may be empty
        bound = self._plan.bind_adaptive(q, self._srht_signs, self._mag_centers, self.cluster_key_counts_gpu[layer_idx],
                                         self._codes_km[layer_idx], self._nib_km[layer_idx], self._w_km[layer_idx], S0,
                                         n_keys, tiers, n_cand, adaptive, self._attention, segments)
        step = (n_keys, bound, 1, self.adaptive_topk_max_k)
        self._adaptive_bound[layer_idx] = step
        return step
