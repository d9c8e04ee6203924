"""Two mixers side by side: both read the same input, each output goes through an RMSNorm of its own over the model
width (plain weights "left_out" / "right_out", eps inside the root), and the result is half their sum:

    y = 1/2 (rmsnorm(left(h)) * w_left + rmsnorm(right(h)) * w_right)

The two are any registered mixers; between them they may keep one set of keys and values (the cache gives an entry of
the schedule one).  Each may keep a state of fixed size: two float32 states addressed by the step's slot ids lie side by
side in the entry's one state row, the left mixer's first, and each mixer sees its own columns.
"""
from __future__ import annotations

import dataclasses

import torch

from .. import ops
from .base import MIXERS, AddingDelta, CacheNeed, ParamSpec, Part, PartSpec, StateNeed
from .linear import upload


@MIXERS.register("parallel")
class ParallelMixer(Part):
    gives_lazy_delta = True         # forward(..., lazy_ok=True) may return a LazyDelta

    def __init__(self, hidden: int, left: PartSpec, right: PartSpec, eps: float):
        self.hidden, self.eps = int(hidden), float(eps)
        self.left, self.right = MIXERS.build(left), MIXERS.build(right)
        needs = [self.left.cache_need(), self.right.cache_need()]
        if sum(n.kv is not None for n in needs) > 1:
            raise ValueError("parallel mixer: its two mixers may keep one set of keys and values between them")
        self.state_split = None                  # floats of the left mixer's state when both keep one
        if all(n.state is not None for n in needs):
            for n in needs:
                if len(n.state.shape) != 1 or n.state.dtype != torch.float32:
                    raise ValueError("parallel mixer: two states share a row only as flat float32 states")
            self.state_split = int(needs[0].state.shape[0])
        self.w_left = self.w_right = None

    @property
    def prompt_capturable(self) -> bool:
        return all(getattr(m, "prompt_capturable", False) for m in (self.left, self.right))

    def children(self):
        return {"left": self.left, "right": self.right}

    def tensors(self):
        t = {f"{cn}.{tn}": spec for cn, c in self.children().items() for tn, spec in c.tensors().items()}
        t.update({"left_out": ParamSpec((self.hidden,), "ones"), "right_out": ParamSpec((self.hidden,), "ones")})
        return t

    def load(self, tensors, device, dtype):
        for cn, c in self.children().items():
            c.load({k[len(cn) + 1:]: v for k, v in tensors.items() if k.startswith(cn + ".")}, device, dtype)
        self.w_left = upload(tensors["left_out"], device, torch.float32)
        self.w_right = upload(tensors["right_out"], device, torch.float32)

    def linears(self):
        return [l for c in self.children().values() for l in c.linears()]

    def cache_need(self) -> CacheNeed:
        a, b = self.left.cache_need(), self.right.cache_need()
        state = a.state or b.state
        if self.state_split is not None:
            state = StateNeed((a.state.shape[0] + b.state.shape[0],), torch.float32,
                              device_addressed=a.state.device_addressed and b.state.device_addressed)
        return CacheNeed(kv=a.kv or b.kv, state=state)

    def wants_stream_norm(self, ctx, rows: int) -> bool:
        """Whether forward is better given its rows undone (an ops.StreamNorm)."""
        ends = [getattr(m, "ends", None) for m in (self.left, self.right)]
        return all(ends) and ops.can_group_stream_norm(rows, self.hidden, [first for first, _ in ends])

    def forward(self, h, ctx, kv, lazy_ok: bool = False):
        kv_a = kv_b = kv
        if self.state_split is not None:
            kv_a = dataclasses.replace(kv, state=kv.state[:, :self.state_split])
            kv_b = dataclasses.replace(kv, state=kv.state[:, self.state_split:])
        ends = [getattr(m, "ends", None) for m in (self.left, self.right)]
        undone = isinstance(h, ops.StreamNorm)
        if undone and not (all(ends) and kv.writes):
            h, undone = h.materialize(), False
        if undone:                               # the rows are formed in the first products' kernel
            pa, pb = ops.linear_group_stream_norm(h, [(first.weight, first.streamed, None) for first, _ in ends])
        elif all(ends) and kv.writes and isinstance(h, torch.Tensor):
            # both read h, and neither's last product waits for the other: two launches instead of four where steps are short
            pa, pb = ops.linear_group([(h, first.weight, first.streamed, None) for first, _ in ends])
        if undone or (all(ends) and kv.writes and isinstance(h, torch.Tensor)):
            ya, yb = self.left.forward(h, ctx, kv_a, projected=pa), self.right.forward(h, ctx, kv_b, projected=pb)
            a, b = ops.linear_group([(y, last.weight, last.streamed, None) for y, (_, last) in zip((ya, yb), ends)])
        else:
            a = self.left.forward(h, ctx, kv_a)
            b = self.right.forward(h, ctx, kv_b)
        args = (a, self.w_left, b, self.w_right)
        if not lazy_ok or not ops.can_mean_into(*args):
            return ops.rmsnorm_mean(*args, self.eps)

        def add(x):
            if x.data_ptr() % 16:
                return False
            ops.rmsnorm_mean(*args, self.eps, into=x)
            return True
        return AddingDelta(lambda: ops.rmsnorm_mean(*args, self.eps), add)
