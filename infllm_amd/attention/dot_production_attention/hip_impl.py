"""Multi-stage attention on the gfx950 MFMA kernel.

Same call protocol as TorchMultiStageDotProductionAttention /
TritonMultiStageDotProductionAttention
(inf_llm/attention/dot_production_attention/torch_impl.py:6-96,
triton_impl.py:488-556): every ``append`` is one stage with its own keys,
values and sliding-window mask; ``end=True`` closes the joint softmax;
``get_result()`` returns the output and, per stage, the column sums of the
final probabilities (or None).  Each stage is one launch of infllm_attn_stage
that leaves a partial (o, lse); the merge kernel joins them, and the scores
are computed afterwards from the final lse (infllm_local_score).  A stage of few
queries is cut into as many key splits as fill the chip (infllm_attn_stage_splits),
with partial rows for each.  Scores are
returned in fp32.  Heads narrower than 128 are padded with zeros to the kernels'
width (the softmax scale stays 1/sqrt of the real head_dim) and the result is cut
back.
"""
import math

import torch
import torch.nn.functional as F

from ... import ops
from .base import MultiStageDotProductionAttention


class HipMultiStageDotProductionAttention(MultiStageDotProductionAttention):
    def __init__(self, q_shape, dtype, device):
        super().__init__(q_shape, dtype, device)
        if dtype != torch.bfloat16:
            raise TypeError(f"the HIP attention path computes in bfloat16, got {dtype}")
        self._stages = []          # (q, k, mask, offset, window, get_score)
        self._o_parts = []
        self._lse_parts = []

    def append(self, q, k, v, sliding_window=None, complement_sliding_window=False, end=False, get_score=False,
               *args, **kwargs):
        assert q.shape == self.q_shape
        assert not self.end, "append after end"
        (batch, heads, _, d), shape, dev = self.q_shape, k.shape, q.device
        if len(shape) != 4 or v.shape != shape or shape[0] != batch or shape[3] != d or shape[1] == 0 or heads % shape[1]:
            raise ValueError(f"keys {tuple(shape)} and values {tuple(v.shape)} do not fit queries {self.q_shape}")      # (read by address)
        if k.device != dev or v.device != dev:
            raise ValueError(f"q, k and v must be on one device, got {dev}, {k.device}, {v.device}")
        if d < ops.HEAD_DIM:
            q, k, v = (F.pad(t, (0, ops.HEAD_DIM - d)) for t in (q, k, v))
        q, k, v = ops._bf16_4d(q, "q"), ops._bf16_4d(k, "k"), ops._bf16_4d(v, "v")
        B, H, Lq, D = q.shape
        scale = 1.0 / math.sqrt(d)
        len_k = k.shape[2]
        if len_k > 1 and (k.stride(2) | v.stride(2)) >= 1 << 27:          # rows further apart than the kernel's offsets reach
            k, v = (t.clone(memory_format=torch.contiguous_format) for t in (k, v))
        if sliding_window is None:
            mask, offset, window = ops.MASK_NONE, 0, 0
        else:
            if isinstance(sliding_window, int):
                sliding_window = (len_k - Lq, sliding_window)
            offset, window = int(sliding_window[0]), int(sliding_window[1])
            mask = ops.MASK_COMPLEMENT if complement_sliding_window else ops.MASK_WINDOW
        o_part, lse_part = ops.attn_stage_split(q, k, v, j_lo=0, j_hi=len_k, mask=mask, offset=offset, window=window, softmax_scale=scale)
        self._o_parts.append(o_part)
        self._lse_parts.append(lse_part)
        self._stages.append((q, k, mask, offset, window, get_score, scale))
        if end:
            self._finalize()

    def _finalize(self):
        self.end = True
        B, H, Lq, d = self.q_shape
        D = max(d, ops.HEAD_DIM)
        dev = self._o_parts[0].device
        if len(self._o_parts) > 2:                             # the merge takes two sets of partials
            self._o_parts = [self._o_parts[0], torch.cat(self._o_parts[1:], dim=0)]
            self._lse_parts = [self._lse_parts[0], torch.cat(self._lse_parts[1:], dim=0)]
        self.ret = torch.empty((B, H, Lq, D), dtype=torch.bfloat16, device=dev)
        self.lse = torch.empty((B, H, Lq), dtype=torch.float32, device=dev)
        # The merge's launch takes the scores of a stage along where there are enough keys to fill it: what it refuses is not offered
        # to it (a small pass is bound by this host code).
        merged, late = None, []
        if Lq <= 2048 and sum(len(part) for part in self._lse_parts) <= 8:
            merged = next((i for i, stage in enumerate(self._stages) if stage[5] and stage[1].shape[2] > 1024), None)
        if merged is None:
            ops.attn_merge_sets(self._o_parts, self._lse_parts, self.ret, self.lse)
        for i, (q, k, mask, offset, window, want, scale) in enumerate(self._stages):
            if not want:
                self.score_list.append(None)
                continue
            score = torch.empty((B, H, k.shape[2]), dtype=torch.float32, device=dev)       # every cell is written
            if i == merged:
                if ops.merge_sets_and_score(self._o_parts, self._lse_parts, self.ret, self.lse, q, k, score, mask=mask, offset=offset, window=window,
                                            softmax_scale=scale):
                    self.score_list.append(score)
                    continue
                ops.attn_merge_sets(self._o_parts, self._lse_parts, self.ret, self.lse)
            self.score_list.append(score)
            late.append((i, score))
        for i, score in late:                     # (behind the merge, wherever it was)
            q, k, mask, offset, window, _, scale = self._stages[i]
            if k.shape[2] > 0:
                ops.local_score(q, k, self.lse, score, j_lo=0, j_hi=k.shape[2], mask=mask, offset=offset,
                                window=window, accumulate=False, softmax_scale=scale)
        if d < D:
            self.ret = self.ret[..., :d].contiguous()
        self._o_parts, self._lse_parts = [], []
