"""The residual of a step between sublayers: streams, or sums of the embedding row and the outputs so far.

A sublayer turns the streams x_1 .. x_S into  x_t <- sum_s mix[s, t] x_s + post[t] (y + bias). mix and post are weights, so every
stream is a sum over the outputs with coefficients known at load. A step of many rows reads the outputs (bf16) in place of reading
and writing S streams (fp32): csrc/ops/stream_norm.hip.

The outputs are held to the plan's end, at most 10 S bytes an element where the streams are 4 S: 4,096 rows of mudepel-base 517 MB at
a step's peak, with streams 366, of mudepel-wide 655 and 688.
"""
from __future__ import annotations

from typing import Dict, List, NamedTuple, Optional, Sequence

import torch

from pilottai_amd import ops


class Hyper(NamedTuple):
    mix: torch.Tensor   # [S, S], from x to
    post: torch.Tensor  # [S]
    bias: Optional[torch.Tensor]  # fp32 [D], joins the sublayer's output
    units: int  # 2 bytes an element that the output takes to read: 1, or 2 where it is a sum of partials


class StreamPlan:
    """Coefficients of the streams before sublayers 0 .. end: all of them, or where streams take over.

    Sums grow with the depth: S streams are 8 S bytes an element to read and write, an output 2 or 4. So they are taken for outputs
    of 8 S bytes, half of that on average, and to the end where that is at most a quarter further on (streams to go on from are written
    once more)."""

    MAX_STREAMS, MAX_TERMS = 8, 63  # of the kernel

    def __init__(self, subs: Sequence[Hyper], device):
        S = subs[0].post.numel()
        f64 = lambda t: t.detach().double().cpu()  # noqa: E731
        units = terms = 0
        fits = []
        for h in subs:
            units, terms = units + h.units, terms + 1 + (h.bias is not None)
            fits.append((units, terms < self.MAX_TERMS))
        most = 5 * S if units <= 5 * S else 4 * S
        self.end = sum(u <= most and ok for u, ok in fits)
        self.whole, self.device = self.end == len(subs), device
        self.subs = [(f64(h.mix), f64(h.post)[None], h.bias is not None) for h in subs[:self.end]]
        self._coef: Dict[tuple, torch.Tensor] = {}

    def coef(self, summed: tuple, kept: bool) -> torch.Tensor:
        """[terms, streams] behind len(summed) outputs, in the kernel's order: biases and what is summed from partials (fp32), then the
        embedding row and the other outputs (bf16). The last one's sum is one of the first if it is `kept`, else it stands behind all."""
        if (summed, kept) not in self._coef:  # (before graph capture: the capture's warm-up runs come first)
            narrow = torch.ones(1, self.subs[0][0].shape[0], dtype=torch.float64)
            wide = last = narrow[:0]
            for partials, (mix, post, bias) in zip(summed, self.subs):
                wide, narrow, last = torch.cat([wide, last]) @ mix, narrow @ mix, narrow[:0]
                if bias:
                    wide = torch.cat([wide, post])
                if partials:
                    last = post
                else:
                    narrow = torch.cat([narrow, post])
            order = [wide, last, narrow] if kept else [wide, narrow, last]
            self._coef[summed, kept] = torch.cat(order).float().to(self.device).contiguous()
        return self._coef[summed, kept]


class Residual:
    """x by sums as far as the plan goes, or without one (plan None) and behind it by its streams."""

    def __init__(self, plan: Optional[StreamPlan], streams: int, embed: torch.Tensor, ids: torch.Tensor):
        self.plan, self.streams, self.embed, self.ids, self.at = plan, streams, embed, ids, 0
        self.f: List[torch.Tensor] = []  # terms
        self.b = [embed]
        self.summed: tuple = ()  # by output: whether it is a sum of partials
        self.x = None if plan is not None else self._rows(streams, embed.shape[1])
        self.step = dict(emb=embed, ids=ids) if plan is None else {}  # what the next norm adds first
        self.held = self.step  # (an output's memory is not the next sublayer's: 64 decoding rows, 8 layers, 1,096 us so, 1,088)

    def _rows(self, *sizes: int) -> torch.Tensor:
        return torch.empty(self.ids.numel(), *sizes, dtype=torch.float32, device=self.ids.device)

    def add(self, result: tuple, mix: torch.Tensor, post: torch.Tensor) -> None:
        """A sublayer's (y, partials, weights, bias)."""
        y, n, weights, bias = result
        self.at += 1
        self.step = dict([("y" if y.dtype == self.embed.dtype else "sums", y)], partials=n, y_weights=weights)
        if self.x is not None:
            self.step.update(bias=bias, mix=mix, post=post)
            return
        if bias is not None:
            self.f.append(bias)
        self.summed += (n > 1 or weights is not None,)
        if not self.summed[-1]:
            self.b.append(y)
            self.step = {}

    def norm(self, eps: float, rows: Optional[torch.Tensor] = None, **kw) -> torch.Tensor:
        """ops.hyper_norm's out of the next sublayer; it may be asked for again."""
        if self.x is not None:
            out = ops.hyper_norm(self.x, eps, rows=rows, **kw, **self.step)
            if rows is None:
                self.held, self.step = self.step, {}
            return out
        D, kept, x = self.embed.shape[1], None, None
        if rows is None and self.at == self.plan.end and not self.plan.whole:
            x = self._rows(self.streams, D)
        elif rows is None and self.step and self.at < self.plan.end:  # (behind the last output nobody adds to it)
            kept = self._rows(D)
        out = ops.stream_norm(self.f, self.b, self.plan.coef(self.summed, not self.step), eps, ids=self.ids, rows=rows, x=x, y_kept=kept, **kw, **self.step)
        if x is not None:
            self.x, self.f, self.b, self.step = x, [], [], {}
        elif kept is not None:
            self.f.append(kept)
            self.step = {}
        return out

    def sum(self, eps: float) -> torch.Tensor:
        """The streams' sum (fp32) behind the last sublayer, without a plan."""
        after = self.x.clone()
        ops.hyper_norm(after, eps, **self.step)
        return after.sum(1)
