"""Mixture of experts on the gfx950 kernels of csrc/moe.hip.

    router: fp32 logits, scores, choice by groups with a correction, weights           (one launch)
    pairs (token, choice) sorted by expert                                             (one launch)
    per expert [gate | up] with the activation, then down                              (one launch each)
The weighted sum over a token's choices (identity experts: the token's own input) is left to the residual update behind the layer;
where the weight multiplies the expert's input instead, it multiplies the sums of [gate | up], ahead of the activation.
Expert weights are kept in ONE form: as the checkpoint has them in fp32, fragment-ordered in 16 bits (``finish_weights``)."""
from __future__ import annotations

import math

import torch
from torch import nn

from .. import hip_ops
from ..utils.loader import materialize
from .latent_attention import padded_parameter
from .linear import Segment, SegmentedLinear, gated_linear, pad_to

__all__ = ["ExpertMLP"]

# Rows of the tiles that a launch works on, by the pairs per expert.  Both products, us, tiles of 16 / 32 / 64 / 256 rows:
#   few pairs: 32 rows are ahead of 16 from 10 (32 experts of 2048 -> 768: 8 62 / 58, 12 67 / 62; 8 experts 24 / 22, 26 / 24).  64 rows against 32, for their longer
#   runs of a weight: of 8 experts from 28 (2048 -> 768: 24 32 / 34, 29 37 / 34; 4096 -> 1536 24 78 / 85, 29 98 / 86), of fewer not up to 40 (2 of 4096 -> 1024, 34 pairs
#   29 / 51), of 32 and more from 24 (4096 -> 1536: 17 226 / 263, 24 261 / 264, 28 314 / 269), but from 16 where their workgroups are no more than two a CU (32 of 2048 ->
#   768: 17 70 / 62, 24 80 / 63; 64 of 1024 -> 384 17 39 / 34) or the second product is the long one (32 of 768 -> 3072: 17 116 / 110; 128 408 / 363).
#   256 rows (two workgroups of 128 x 256 to a CU) against 64: ahead where the workgroups of both products fill the chip in part, half of it the gated one's, 80 CUs the
#   other's, which is the longer one where the experts are wide.  Workgroups of the two, pairs: 32 of 2048 -> 768 (192, 256) 64 pairs 100 / 66, 32 of 1024 -> 384 (96, 128)
#   64 30 / 33, (192, 256) 160 51 / 37; 4 of 2048 -> 768 (144, 192) 768 61 / 53; 8 of 768 -> 3072 (192, 24) 64 51 / 62, (768, 96) 500 110 / 98; 16 of 1024 -> 2816 (352, 64) 44
#   77 / 83; 2 of 4096 -> 1024 (192, 384) 1500 102 / 94; 1 of 1024 -> 2816 (440, 80) 2500 82 / 76.  Over 500 shapes (1 .. 128 experts, 44 .. 2500 pairs) 0.3 % behind the better
#   of the two in the mean, 17 % at worst; without the second line eleven took up to 1.2 times as long as by the 64 or 128 rows that they once had.
#   128 rows: the 256's kernel, a tile a workgroup (tiles of the 64's kind, which they were, are nowhere ahead of both).
# Up to QUARTERS pairs per expert, tiles of 64 rows sum as those of 16 and 32 do: a call's bits are those of tiles of 32 rows, which it once had.
# That costs nothing in them, but 256 rows, which have no such sums, would be ahead in the end: 32 experts of 2048 -> 768, 24 pairs 68 / 65, 40 74 / 66 (32 rows 78, 130).
FEW, WIDE_GROUPS, QUARTERS = 8, (128, 80), 40


class ExpertMLP(nn.Module):
    def __init__(self, width: int, experts: int, identity: int, top: int, groups: int, keep: int, scale: float, ff: int,
                 shared_ff: int = 0, act: hip_ops.GateAct | None = None, sigmoid: bool = False, corrected: bool = True,
                 raw_weights: bool = False, weigh_inputs: bool = False) -> None:
        """``sigmoid``: scores are sigmoids of the logits, not a softmax; ``corrected``: a number per output joins the scores in the
        choice; ``raw_weights``: the weights are the chosen scores, not divided by their sum; ``weigh_inputs``: they multiply the
        experts' inputs, not their outputs."""
        super().__init__()
        if weigh_inputs and identity:
            raise ValueError("identity experts have no product that could weigh its input")
        self.sigmoid, self.raw_weights, self.weigh_inputs = sigmoid, raw_weights, weigh_inputs
        self.experts, self.top, self.groups, self.keep, self.scale = experts, top, groups, keep, float(scale)
        self.act = act or hip_ops.GateAct(0, 0.0, 0.0)     # silu
        w, f = pad_to(width), pad_to(ff)
        self.w, self.f, self.width, self.ff = w, f, width, ff
        self.router = padded_parameter(experts + identity, w)
        self.correction = padded_parameter(experts + identity) if corrected else None
        self.gate_up, self.down = nn.Parameter(torch.zeros(experts, 2, f, w)), nn.Parameter(torch.zeros(experts, w, f))
        self.gate_up.weight_loader = self.down.weight_loader = self._load
        self.packed = False
        self.shared_gate_up = self.shared_down = None
        if shared_ff:
            self.shared_gate_up = SegmentedLinear(width, [Segment("gate", shared_ff), Segment("up", shared_ff)], split="out")
            self.shared_down = SegmentedLinear(width, [Segment("down", shared_ff)], split="in")

    def extra_repr(self) -> str:
        return f"experts={self.experts}, outputs={self.router.shape[0]}, top={self.top}, groups={self.keep} of {self.groups}, ff={self.ff}"

    def _load(self, param, tensor, shard=None, *args, **kwargs):
        """shard: (expert, "gate" | "up" | "down")."""
        e, what = shard
        t, want = materialize(tensor), (self.width, self.ff) if what == "down" else (self.ff, self.width)
        if tuple(t.shape) != want:
            raise ValueError(f"expert {e} {what}: expected {want}, got {tuple(t.shape)}")
        dst = param.data[e] if what == "down" else param.data[e, int(what == "up")]
        dst[:want[0], :want[1]].copy_(t)

    def finish_weights(self) -> None:
        """The form that the kernels read, in place of the loaded one."""
        if self.router.dtype != torch.float32 and not self.packed:
            for p in (self.gate_up, self.down):
                p.data = hip_ops.pack_weight(p.data.view(-1, p.shape[-1]))
            self.packed = True

    def _rows32(self) -> int:
        """Pairs per expert up to which tiles of 32 rows are ahead of 64."""
        if self.experts < 32:
            return 28 if self.experts >= 8 else 40
        groups = self.experts * math.ceil(max(2 * self.f, self.w) / 128)      # workgroups of the 64's larger product
        return 16 if groups <= 512 or self.f > self.w else 24

    def tile_rows(self, tokens: int) -> int:
        if self.router.dtype == torch.float32:
            return 16
        per = tokens * self.top / self.experts
        if per <= FEW:
            return 16
        if per <= self._rows32():
            return 32
        if per <= QUARTERS:
            return 64
        rows = self.experts * math.ceil(per / 128)        # workgroups of the two products
        wide = rows * math.ceil(2 * self.f / 256) >= WIDE_GROUPS[0] and rows * math.ceil(self.w / 256) >= WIDE_GROUPS[1]
        return 256 if wide else 64

    def route(self, h):
        """-> (weights [T, top], the pairs sorted by expert), for callers that have use for the parts; ``forward`` makes both in its one call."""
        ids, weights = hip_ops.moe_route(h, self.router, self.correction, self.top, self.groups, self.keep, self.scale, self.sigmoid,
                                         self.raw_weights)
        return weights, hip_ops.moe_group(ids, self.experts, self.tile_rows(h.shape[0]), weights if self.weigh_inputs else None)

    def forward(self, h):
        """-> (shared expert's output or None, the routed experts' part for ``hip_ops.residual_update``)."""
        tile = self.tile_rows(h.shape[0])
        y, place, weights = hip_ops.moe_mlp(h, self.router, self.correction, self.gate_up, self.down, self.experts, self.f, self.w, self.top, tile, self.act,
                                            self.groups, self.keep, self.scale, self.sigmoid, self.raw_weights, self.weigh_inputs,
                                            tile == 64 and h.shape[0] * self.top <= QUARTERS * self.experts)
        shared = None
        if self.shared_gate_up is not None:
            shared = self.shared_down(gated_linear(h, self.shared_gate_up, "silu"), partial_ok=True)
        return shared, (y, place, None if self.weigh_inputs else weights)
