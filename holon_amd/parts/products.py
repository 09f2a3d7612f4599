"""Products that do not read one another's results, in one launch.

In a step of a few rows a product of 2,048 columns takes a kernel's start, end and a round of memory latency, whatever its
weights need, and a block's sublayers, or two mixers side by side, wait for one another only in the order they are written
down in. A part may therefore say what it does as a generator (`products`, with `forward`'s arguments): it yields lists of
`Product`s, is sent their results, and returns what `forward` returns. `drive` runs such parts side by side: in steps of few
rows it collects what all of them ask for and runs it as one operation (`linear_group`); in other steps, and for parts
without a generator, one after the other, each product as it always was.
"""
from __future__ import annotations

import ctypes
import dataclasses

import torch

from ..kernels.registry import KernelOp, register_kernel
from .linear import Linear

FEW_ROWS = 16                 # up to this many rows products run together
MOST = 8                      # products a launch takes


@dataclasses.dataclass
class Product:
    """x W^T of one projection: in the rows' dtype, as `dtype`, or (`relu2`) its max(z, 0)^2."""

    linear: Linear
    x: torch.Tensor
    dtype: torch.dtype | None = None
    relu2: bool = False

    def alone(self) -> torch.Tensor:
        linear, k = self.linear, self.linear.kernels
        if not self.relu2:
            return linear(self.x, self.dtype)
        y = k.linear_relu2(self.x, linear.weight, linear.tiled if linear.folded is None else None)
        return k.relu2(linear(self.x)) if y is None else y


def products_of(part, *args, **kwargs):
    """The part's generator, where the class that says what `forward` does says it as one too; else one that runs `forward`."""
    owner = next((c for c in type(part).__mro__ if "forward" in vars(c) or "products" in vars(c)), None)
    if owner is not None and "products" in vars(owner):
        return part.products(*args, **kwargs)

    def whole():
        return part(*args, **kwargs)
        yield
    return whole()


def drive(kernels, rows: int, *parts) -> list:
    """What each generator returns."""
    if rows > FEW_ROWS:
        return [_by_itself(part) for part in parts]
    results, asked = [None] * len(parts), {}

    def go(i: int, send) -> None:
        try:
            asked[i] = parts[i].send(send)
        except StopIteration as end:
            asked.pop(i, None)
            results[i] = end.value
    for i in range(len(parts)):
        go(i, None)
    while asked:
        waiting = dict(asked)
        done = iter(kernels.linear_group([p for i in waiting for p in waiting[i]]))
        for i, products in waiting.items():
            go(i, [next(done) for _ in products])
    return results


def _by_itself(part):
    send = None
    while True:
        try:
            send = [p.alone() for p in part.send(send)]
        except StopIteration as end:
            return end.value


def linear_group_plain(products: list[Product]) -> list[torch.Tensor]:
    """The results of products that do not read one another's, in order; each with the roundings it has alone."""
    return [p.alone() for p in products]


def _served(p: Product) -> bool:
    """Whether the few-row product over a tiled copy serves it (what `linear` and `linear_relu2` would run)."""
    x, w, tiled = p.x, p.linear.weight, p.linear.tiled
    return (tiled is not None and p.linear.folded is None and x.is_cuda and x.dtype == tiled.dtype == torch.bfloat16 and x.dim() == 2
            and 1 <= x.shape[0] <= FEW_ROWS and x.is_contiguous() and tiled.is_contiguous() and tiled.shape == w.shape
            and x.shape[1] == w.shape[1] and w.shape[0] % 16 == 0 and w.shape[1] % 32 == 0 and w.shape[1] >= 256
            and x.data_ptr() % 16 == 0 and p.dtype in (None, torch.bfloat16, torch.float32) and not (p.relu2 and p.dtype == torch.float32))


def _linear_group_hip(launch, products: list[Product]) -> list[torch.Tensor]:
    out: list = [None] * len(products)
    by_rows: dict[int, list[int]] = {}
    for i, p in enumerate(products):
        if _served(p):
            by_rows.setdefault(p.x.shape[0], []).append(i)
    for rows, which in by_rows.items():
        for group in (which[at: at + MOST] for at in range(0, len(which), MOST)):
            if len(group) == 1:
                continue
            items = []
            for i in group:
                p = products[i]
                form = 4 if p.relu2 else 2 if p.dtype == torch.float32 else 0
                n, k = p.linear.weight.shape
                out[i] = torch.empty((rows, n), dtype=torch.float32 if form == 2 else torch.bfloat16, device=p.x.device)
                items += [p.x.data_ptr(), p.linear.tiled.data_ptr(), out[i].data_ptr(), n, k, form]
            launch((ctypes.c_int64 * len(items))(*items), len(group), rows)
    return [y if y is not None else p.alone() for y, p in zip(out, products)]


register_kernel(KernelOp("linear_group", linear_group_plain, "holon_gemm_skinny_group_bf16",
                         [ctypes.c_void_p, ctypes.c_int, ctypes.c_int], _linear_group_hip))
