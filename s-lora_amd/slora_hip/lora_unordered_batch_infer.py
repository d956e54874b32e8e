"""The LoRA half of the reference's batch engine
(slora/models/peft/lora_unordered_batch_infer.py:16-483): per inference step the
``delta`` buffers, the choice between the segmented (prefill) kernels and the
per-token BGMV kernels, and per layer the shrink + expand of the q, k, v and o
projections on top of the base model's matmul outputs.

The base model (matmuls, rotary embedding, attention, FFN) is the caller's: it
computes ``q``, ``cache_k``, ``cache_v`` / ``o`` with its own weights and hands
them to ``lora_get_qkv`` / ``lora_get_o``, which add the adapters' deltas in
place -- exactly what the reference does between its ``torch.mm`` calls and the
rotary embedding (:254-318 decode, :321-408 prefill, :411-483 o projection).

Two ways to issue the work, same results bit for bit:

* ``fused=False``: the reference's call sequence, one ``dispatch_bgmv`` or
  ``lora_get_qkvo_fwd_*`` call per projection and direction (8 per layer),
  ``delta[0]`` shared by q and o as in the reference;
* ``fused=True`` (default): q, k and v of a layer in one call, which reads the
  activations once.  In decode steps shrink and expand are one call as well, which the
  library turns into one launch where that is faster than two; in prefill steps
  they are one launch each.

Either way the first call of a step builds the batch's plan inside the library and
the other calls of the step reuse it (the index tensors are the same objects in
every call of a step).  Nothing here waits for the device, but an object's first decode
step (``begin_step``) and what ``begin_step`` is not told (its docstring).
"""
from __future__ import annotations

from typing import List, Optional, Sequence

import torch

from ._kernels import (dispatch_bgmv, dispatch_bgmv_lora, dispatch_bgmv_qkv_expand, dispatch_bgmv_qkv_lora,
                       dispatch_bgmv_qkv_shrink, lora_get_qkvo_fwd_expand, lora_get_qkvo_fwd_expand_qkv,
                       lora_get_qkvo_fwd_shrink, lora_get_qkvo_fwd_shrink_qkv, segments_ok, store_ids)

# lora_unordered_batch_infer.py:334: in the reference the segmented kernels serve batches with a long
# request, adapters of rank >= 64 and at least two requests, and everything else is BGMV
PREFILL_MIN_SEQ_LEN = 200
PREFILL_MIN_LORA_DIM = 64
PREFILL_MIN_REQUESTS = 2
# Beyond these the segmented kernels have no plan or no vector path, and such batches stay with BGMV
SEGMENTED_MAX_REQUESTS = 256
SEGMENTED_MAX_RANK = 128


def segmented_pays(n_tok: int, n_req: int, max_rank: int, hidden: int) -> bool:
    """Whether the segmented kernels are the faster ones for a prefill batch.

    Their four launches of a layer cost the same however few rows there are, plus a share per 16 rows of each
    prompt; the per-token ones cost least at one token and grow with tokens times rank.  us per layer, token
    by token against segmented (f16, calls from Python, prompts of equal length):

    ====================  ==================  ==================  ==================  ==================
    prompts x tokens      4096, rank 8        4096, rank 16       4096, rank 64       8192, rank 64
    ====================  ==================  ==================  ==================  ==================
    1 x 1                  15.0 /  21.2        14.8 /  21.9        16.2 /  24.1        21.1 /  30.3
    1 x 16                 22.4 /  23.0        22.2 /  23.1        24.7 /  25.7        34.4 /  31.9
    1 x 64                 24.8 /  24.0        25.2 /  24.5        32.7 /  27.2        45.3 /  33.5
    4 x 16                 21.9 /  23.5        22.8 /  23.9        27.6 /  26.8        41.8 /  33.3
    16 x 4                 22.2 /  24.5        23.3 /  25.2        29.2 /  35.4        43.7 /  51.1
    64 x 16                41.6 /  47.8        55.2 /  52.5       142.8 /  96.5       245.7 / 142.2
    256 x 1                27.9 /  82.5        32.9 /  89.0        71.8 / 183.2       114.9 / 256.8
    ====================  ==================  ==================  ==================  ==================

    A prompt of fewer rows than a part of 16 pays for the whole part: 16 rows per prompt.  Wide rows (5120 and
    8192) make a token dearer than a launch: up to eight prompts from four rows (8 x 4 tokens of ranks 8 / 64 at
    hidden 5120: 0.86 / 1.01 of the per-token time; 16 x 4: 0.93 / 1.14).  Narrow rows of low rank are so cheap per
    token that several prompts need enough of them.  Rank 16: 256 tokens (8 x 16: 1.07, 8 x 32: 1.00, 4 x 64:
    0.98).  Rank 8: about 1000 tokens in prompts of 64 (64 x 36: 1.18, 64 x 56: 0.98, 64 x 66: 0.94, 100 x 40: 1.20),
    or of 40 where the kernels of more than 4096 tokens run (100 x 48: 1.00, 128 x 40: 0.97, 200 x 33: 1.06, 200 x 40:
    0.92); above 8192 tokens the per-token operator's plan costs milliseconds a step (256 x 33, a step of 8 layers:
    6.6 ms against 1.7).  Hidden 1024 and 2048 and bf16 measure the same or better for the segmented kernels."""
    if hidden > 4096 and n_req <= 8:
        return n_tok >= 4 * n_req
    if hidden > 4096 or n_req == 1 or max_rank > 16:
        return n_tok >= 16 * n_req
    if max_rank > 8:
        return n_tok >= max(256, 16 * n_req)
    return n_tok > 8192 or n_tok >= max(1024, (40 if n_tok > 4096 else 64) * n_req)


class LoraUnorderedBatchInfer:
    """One object per batch, as in the reference (model_rpc.py:234 builds it per step).

    ``infer_adapter``: the tables ``a_loc / a_start / a_len / a_scaling``, ``adapter_dirs`` /
    ``idx_map`` and the pool as ``mem_manager.key_buffer / value_buffer`` or, like the reference's
    ``NaiveInferAdapter``, as ``key_buffer / value_buffer`` of its own (``slora_hip.InferAdapter`` or
    anything with those attributes).  ``adapters``: per request an object with ``lora_dir``
    and ``r`` (the reference's ``LoraTpPartAdapter``); ``None`` entries (requests on the bare
    base model, which the reference does not support either, :35-36) are rejected."""

    def __init__(self, infer_adapter, adapters: Sequence, kv_embed_dim: Optional[int] = None, fused: bool = True,
                 delta_dtype: Optional[torch.dtype] = None):
        if any(a is None for a in adapters):
            raise ValueError("requests without an adapter are not supported (as in the reference)")
        self.infer_adapter = infer_adapter
        # the pool's buffers: on the adapter table itself (the reference's NaiveInferAdapter, :28-30)
        # or on its memory manager (:31-33)
        owner = infer_adapter if hasattr(infer_adapter, "key_buffer") else infer_adapter.mem_manager
        self.key_buffer: List[torch.Tensor] = owner.key_buffer
        self.value_buffer: List[torch.Tensor] = owner.value_buffer
        dev = self.key_buffer[0].device
        self.max_lora_dim = max((int(a.r) for a in adapters), default=0)
        idx_map = getattr(infer_adapter, "idx_map", None)
        if idx_map:  # one dictionary lookup per request; the reference searches the list (:37)
            ids = [idx_map[a.lora_dir] for a in adapters]
        else:
            ids = [infer_adapter.adapter_dirs.index(a.lora_dir) for a in adapters]
        # On the default stream the adapter indices go to the device as kernel arguments: a copy waits for everything
        # queued on the stream, i.e. for the step before, while the next one is not even begun, and a copy from pinned memory
        # needs a new block for every step that is in flight (9 prompts of 2311 tokens, 8 layers, us a step: 559, 531 and 526 in
        # this form).  `_stored`: what steps wait for until the host has.  On other streams it is the copy, which
        # is also what refuses an object that is built while a graph is being recorded, and so it is for a pool of another
        # device than the current one, whose default stream the launch would go to.
        here = dev.type == "cuda" and dev.index == torch.cuda.current_device()
        self._stored = store_ids(ids, self.key_buffer[0]) if here else None
        self._req_bins = torch.tensor(ids, dtype=torch.long, device=dev) if self._stored is None else self._stored.ids
        kb = self.key_buffer[0]
        self.page_elems = int(kb.shape[1] * kb.shape[2])
        self.kv_embed_dim = int(kv_embed_dim) if kv_embed_dim is not None else self.page_elems
        self.fused = bool(fused)
        self.delta_dtype = delta_dtype or kb.dtype
        self.delta: List[torch.Tensor] = []
        self.is_prefill = False
        self.use_segmented = False
        self.batch_req_bins: Optional[torch.Tensor] = None
        self.max_b_seq_len = 0
        self._bins: Optional[torch.Tensor] = None
        self._n_tok = self._longest = 0
        # a BGMV batch of the reference whose tokens are rows of prompts: (starts, lengths), or None
        self._prompts: Optional[tuple] = None
        self._adapters = adapters

    @property
    def req_bins(self) -> torch.Tensor:
        """Adapter index of every request, on the device (:37), there for every stream.  Steps read this tensor, recorded
        ones at every replay."""
        self._settle()
        return self._req_bins

    @req_bins.setter
    def req_bins(self, bins: torch.Tensor) -> None:
        self._req_bins, self._stored = bins, None

    def _settle(self) -> None:
        """The host waits, once, until the indices are on the device; also while this thread records a graph."""
        stored = self._stored  # (read once: another thread may have waited in between)
        if stored is not None:
            stored.wait()
            self._stored = None

    # ---- per step (forward(), :44-80) -----------------------------------------------------
    def begin_step(self, b_start_loc: torch.Tensor, b_seq_len: torch.Tensor, is_prefill: bool,
                   max_b_seq_len: Optional[int] = None, total_token_num: Optional[int] = None) -> None:
        """The per-step part of ``forward``: ``delta`` (three zeroed ``[tokens, max_lora_dim]``
        buffers, :69 / :76), per-token adapter ids for a prefill batch (:66) and the kernel choice
        (:334).  ``max_b_seq_len`` spares the read-back of ``torch.max(b_seq_len).item()`` (:61)
        and ``total_token_num`` (the sum of ``b_seq_len``, an argument of the reference's ``forward``)
        the one inside ``repeat_interleave``, when the caller knows them: the step then starts
        without waiting for the device."""
        bins, stored = self._req_bins, self._stored
        assert b_start_loc.shape[0] == b_seq_len.shape[0] == bins.shape[0]
        if stored is not None:
            if is_prefill and not torch.cuda.is_current_stream_capturing():
                stored.order()
            else:
                # A graph may be replayed on any stream.  The launches of a decode step are sized by the plan's item count,
                # which the host has in time only where the stream is nearly idle when the plan is built (23 tokens, 32
                # layers: 830 us, without the wait 1064).
                self._settle()
        self.is_prefill = bool(is_prefill)
        self.b_start_loc, self.b_seq_len = b_start_loc, b_seq_len
        self.max_b_seq_len = int(max_b_seq_len) if max_b_seq_len is not None else int(torch.max(b_seq_len).item())
        n_req = int(b_seq_len.shape[0])
        if self.is_prefill:
            self.batch_req_bins = torch.repeat_interleave(bins, b_seq_len.to(torch.long),
                                                          output_size=total_token_num)
            n_tok = int(self.batch_req_bins.shape[0])
            self.use_segmented = (self.max_b_seq_len >= PREFILL_MIN_SEQ_LEN and
                                  self.max_lora_dim >= PREFILL_MIN_LORA_DIM and n_req >= PREFILL_MIN_REQUESTS)
            self._bins = self.batch_req_bins
            self._prompts = None
            if (not self.use_segmented and n_tok > 0 and n_req <= SEGMENTED_MAX_REQUESTS and
                    segmented_pays(n_tok, n_req, self.max_lora_dim, self.page_elems) and
                    self.max_lora_dim <= SEGMENTED_MAX_RANK and all(int(a.r) % 8 == 0 for a in self._adapters) and
                    self.page_elems % 8 == 0 and self.delta_dtype == self.key_buffer[0].dtype):
                # where the rows of a prompt start follows from the lengths alone, as batch_req_bins does; like that
                # one starts and lengths are this step's own, whatever the caller writes into b_seq_len before the
                # last layer (lengths as a difference: a copy of a tensor is a transfer, 10 us dearer than a kernel)
                lens = b_seq_len.to(torch.int32)
                ends = torch.cumsum(lens, 0, dtype=torch.int32)
                starts = ends - lens
                self._prompts = (starts, ends - starts)
                # the longest prompt, if it was read here: a caller's figure has only decided the rule above, where a
                # wrong one does no harm, and no prompt is longer than the batch.  (It matters above 65536 tokens,
                # where that bound hides that a plan could be built: 70000 tokens of rank 32 in 64 prompts 1636 us
                # per layer against 1133; token by token 4036, of rank 8 1539 / 1068 / 1354 and a plan of
                # milliseconds per step)
                self._longest = self.max_b_seq_len if max_b_seq_len is None else n_tok
        else:
            self._prompts = None
            self.batch_req_bins = None
            n_tok = n_req
            self.use_segmented = False
            self._bins = bins
        self._n_tok = n_tok
        dev = bins.device
        # (one fill for all three where each starts on 16 bytes, as an allocation of its own would)
        shape = (n_tok, self.max_lora_dim)
        if self.max_lora_dim % 8 == 0:
            self.delta = list(torch.zeros((3, *shape), dtype=self.delta_dtype, device=dev).unbind(0))
        else:
            self.delta = [torch.zeros(shape, dtype=self.delta_dtype, device=dev) for _ in range(3)]

    def _segments(self, key: torch.Tensor, val: torch.Tensor, x: torch.Tensor, *outs: torch.Tensor):
        """Index tensors and longest request for the segmented kernels, or None where the per-token
        kernels serve the call: what they refuse (strided rows or pools, another row count) they still
        refuse, and what only they take (tables that are not 1-D, pools of two page widths) they still take."""
        ia = self.infer_adapter
        if self.use_segmented:
            return (ia.a_loc, ia.a_start, ia.a_len, self.b_start_loc, self.b_seq_len, self._req_bins), self.max_b_seq_len
        if self._prompts is None:
            return None
        if not segments_ok(self.key_buffer[0], key, val, ia.a_loc, ia.a_start, ia.a_len, self._n_tok, self.page_elems, x, *outs):
            return None
        return (ia.a_loc, ia.a_start, ia.a_len, *self._prompts, self._req_bins), self._longest

    def _one_call(self, key: torch.Tensor, val: torch.Tensor) -> bool:
        """Whether the per-token shrink and expand of a layer go out as one call (which wants whole 16-byte pieces of
        delta and pools of one shape): the same bits as the two."""
        return self.fused and self.max_lora_dim % 8 == 0 and key.shape == val.shape

    # ---- q, k, v of one layer (:254-318 decode, :321-408 prefill) --------------------------
    def lora_get_qkv(self, layer_id: int, input_embs: torch.Tensor, q: torch.Tensor, cache_k: torch.Tensor,
                     cache_v: torch.Tensor) -> None:
        """``q / cache_k / cache_v += scaling * (input_embs A_p) B_p`` for p = q, k, v with every
        token's own adapter.  ``input_embs``: ``[tokens, hidden]``; the three outputs 2-D views
        ``[tokens, h_out]`` that already hold the base model's projections (``cache_k`` /
        ``cache_v`` may be row slices of the pool itself, transformer_layer_infer_template.py:39-41)."""
        ia = self.infer_adapter
        key, val = self.key_buffer[layer_id], self.value_buffer[layer_id]
        d = self.delta
        outs = (q, cache_k, cache_v)
        if self.max_lora_dim == 0 or input_embs.shape[0] == 0:
            return
        segments = self._segments(key, val, input_embs, q, cache_k, cache_v) if self.is_prefill else None
        if segments is not None:
            key2, val2 = key.view(-1, self.page_elems), val.view(-1, self.page_elems)
            seg, longest = segments
            hidden = int(input_embs.shape[1])
            if self.fused:
                lora_get_qkvo_fwd_shrink_qkv(input_embs, key2, d[0], d[1], d[2], *seg, hidden, self.max_lora_dim,
                                             longest)
            else:
                for p in range(3):
                    lora_get_qkvo_fwd_shrink(input_embs, key2, d[p], *seg, hidden, p, self.max_lora_dim,
                                             longest)
            if self.fused and cache_k.shape == cache_v.shape and cache_k.stride(0) == cache_v.stride(0):
                lora_get_qkvo_fwd_expand_qkv(d[0], d[1], d[2], val2, q, cache_k, cache_v, ia.a_scaling, *seg,
                                             int(q.shape[1]), int(cache_k.shape[1]), self.max_lora_dim,
                                             longest)
                return
            for p in range(3):
                lora_get_qkvo_fwd_expand(d[p], val2, outs[p], ia.a_scaling, *seg, int(outs[p].shape[1]), p,
                                         self.max_lora_dim, longest)
            return
        tabs = (ia.a_start, ia.a_len, ia.a_loc, self._bins)
        if self._one_call(key, val):
            dispatch_bgmv_qkv_lora(q, cache_k, cache_v, d[0], d[1], d[2], input_embs, key, val, *tabs, ia.a_scaling)
        elif self.fused:
            dispatch_bgmv_qkv_shrink(d[0], d[1], d[2], input_embs, key, *tabs)
            dispatch_bgmv_qkv_expand(q, cache_k, cache_v, d[0], d[1], d[2], val, *tabs, ia.a_scaling)
        else:
            for p in range(3):
                dispatch_bgmv(d[p], input_embs, key, *tabs, p, ia.a_scaling)
                dispatch_bgmv(outs[p], d[p], val, *tabs, p, ia.a_scaling)

    # ---- o of one layer (:411-483) ---------------------------------------------------------
    def lora_get_o(self, layer_id: int, input: torch.Tensor, o: torch.Tensor) -> None:
        """``o += scaling * (input A_o) B_o``; ``delta[0]`` is reused, as in the reference (:421, :447)."""
        ia = self.infer_adapter
        key, val = self.key_buffer[layer_id], self.value_buffer[layer_id]
        d = self.delta[0]
        if self.max_lora_dim == 0 or input.shape[0] == 0:
            return
        segments = self._segments(key, val, input, o) if self.is_prefill else None
        if segments is not None:
            key2, val2 = key.view(-1, self.page_elems), val.view(-1, self.page_elems)
            seg, longest = segments
            lora_get_qkvo_fwd_shrink(input, key2, d, *seg, int(input.shape[1]), 3, self.max_lora_dim,
                                     longest)
            lora_get_qkvo_fwd_expand(d, val2, o, ia.a_scaling, *seg, int(o.shape[1]), 3, self.max_lora_dim,
                                     longest)
            return
        tabs = (ia.a_start, ia.a_len, ia.a_loc, self._bins)
        if self._one_call(key, val) and self.max_lora_dim < min(input.shape[1], o.shape[1]):
            dispatch_bgmv_lora(o, d, input, key, val, *tabs, 3, ia.a_scaling)
            return
        dispatch_bgmv(d, input, key, *tabs, 3, ia.a_scaling)
        dispatch_bgmv(o, d, val, *tabs, 3, ia.a_scaling)
