"""Products that do not read one another's results, in one launch.

In a step of a few rows a product of 2,048 columns takes a kernel's start, end and a round of memory latency, whatever its
weights need, and a block's sublayers, or two mixers side by side, wait for one another only in the order they are written
down in. A part may therefore say what it does as a generator (`products`, with `forward`'s arguments): it yields lists of
`Product`s, is sent their results, and returns what `forward` returns. `drive` runs such parts side by side: in steps of few
rows it collects what all of them ask for and runs it as one operation (`linear_group`); in other steps, and for parts
without a generator, one after the other: products of one size in one launch where they fill the chip together
(`linear_block_group`), each other product as it always was. (A list, its products and the generator's way cost the host 3 us, as
much as two launches of a step that the host bounds: a part that has one or two products to ask for runs them itself in steps that
cannot share a launch, which is what `together` says of its input, and a launch for one product alone is not asked for.)
"""
from __future__ import annotations

import ctypes
import dataclasses
import functools
import inspect
from collections.abc import Sequence
from typing import Any

import torch

from ..kernels.registry import KernelOp, register_kernel
from .linear import Linear

FEW_ROWS = 16                 # up to this many rows products run together
MOST = 8                      # products a launch takes
BLOCK_ROWS = (129, 3072)      # this many rows: products of one size run together
BLOCK_MOST = 4                # so many of them


@dataclasses.dataclass(slots=True)
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


@dataclasses.dataclass(slots=True)
class Routing:
    """A mixture's router (`moe_router_top`, or with `scale` set `moe_router`): which experts each row of x takes, and their weights."""

    kernels: Any
    x: torch.Tensor
    router: torch.Tensor
    bias: torch.Tensor | None
    experts: int
    top: int
    groups: int
    keep: int
    score: str = "softmax"
    scale: float | None = None

    def alone(self) -> torch.Tensor:
        if self.scale is not None:
            return self.kernels.moe_router(self.x, self.router, self.bias, self.top, self.groups, self.keep, self.scale)
        how = {} if self.score == "softmax" else {"score": self.score}
        return self.kernels.moe_router_top(self.x, self.router, self.bias, self.experts, self.top, self.groups, self.keep, **how)

    def served(self) -> bool:
        """Whether a launch of products takes it along: what the operation by itself would accept, at few rows and experts."""
        x, r, e = self.x, self.router, self.experts
        return (x.is_cuda and x.dtype == torch.bfloat16 and x.dim() == 2 and x.is_contiguous() and 1 <= x.shape[0] <= FEW_ROWS
                and r.dtype == torch.float32 and r.is_contiguous() and r.dim() == 2 and r.shape[1] == x.shape[1] <= 12288
                and r.shape[0] in ((e,) if self.scale is not None else (e, e + 1)) and 1 <= self.top <= e <= 64
                and (self.bias is None or (self.bias.dtype == torch.float32 and self.bias.is_contiguous() and self.bias.shape == (e,)))
                and (self.groups <= 1 or (e % self.groups == 0 and 1 <= self.keep <= self.groups
                                          and (self.scale is not None or self.top <= self.keep * (e // self.groups)))))


@dataclasses.dataclass(slots=True)
class ExpertsDown:
    """The second product of a mixture's chosen experts (`moe_down_few`) over x, their activations [T, experts ff + shared]."""

    kernels: Any
    x: torch.Tensor
    weights: torch.Tensor
    tiled: torch.Tensor
    experts: int
    ff: int
    shared: int

    def alone(self) -> torch.Tensor:
        return self.kernels.moe_down_few(self.x, self.weights, self.tiled, self.experts, self.ff, self.shared)

    def served(self) -> bool:
        """Whether a product's launch takes it along: what the operation by itself accepts."""
        x, w, t, cols = self.x, self.weights, self.tiled, self.experts * self.ff + self.shared
        return (x.is_cuda and x.dtype == t.dtype == torch.bfloat16 and x.is_contiguous() and t.is_contiguous() and w.is_contiguous()
                and w.dtype == torch.float32 and w.dim() == 2 and w.shape[0] == x.shape[0] and 1 <= x.shape[0] <= FEW_ROWS
                and w.shape[1] >= self.experts and tuple(x.shape[1:]) == (cols,) and tuple(t.shape[1:]) == (cols,) and t.shape[0] % 32 == 0
                and self.experts <= 1024 and self.ff % 32 == 0 and self.shared % 32 == 0)


def together(x, linear: Linear | None = None) -> bool:
    """Whether a product over these rows (of `linear`, if it is one's) may share a launch: few of them, in the type that it serves, over
    a tiled copy. Else whoever asks for it gains nothing from the list, and runs it."""
    return x.shape[0] <= FEW_ROWS and getattr(x, "dtype", None) == torch.bfloat16 and \
        (linear is None or getattr(linear, "tiled", None) is not None)


@functools.cache
def _says_products(cls: type) -> bool:
    """Whether the class that says what a call of the part does (the nearest that has `__call__`, `forward` or `products`) says it as a
    generator too."""
    owner = next((vars(c) for c in cls.__mro__ if not vars(c).keys().isdisjoint(("__call__", "forward", "products"))), {})
    return inspect.isgeneratorfunction(owner.get("products"))


def products_of(part, *args, **kwargs):
    """The part's generator, where the class that says what `forward` does says it as one too; else one that runs `forward`."""
    if _says_products(type(part)):
        return part.products(*args, **kwargs)

    def whole():
        return part(*args, **kwargs)
        yield
    return whole()


def drive(kernels, rows: int, *parts) -> Sequence:
    """What each generator returns."""
    if rows > FEW_ROWS or len(parts) == 1:
        return [by_itself(kernels, part) for part in parts]
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
        done = iter(_results(kernels, [p for i in waiting for p in waiting[i]]))
        for i, products in waiting.items():
            go(i, [next(done) for _ in products])
    return results


def by_itself(kernels, part):
    """What one generator returns, with nothing beside it."""
    try:
        asked = part.send(None)
        while True:
            asked = part.send(_results(kernels, asked))
    except StopIteration as end:
        return end.value


def _results(kernels, products: list[Product | Routing | ExpertsDown]) -> list[torch.Tensor]:
    if len(products) < 2:
        return [p.alone() for p in products]
    if products[0].x.shape[0] > FEW_ROWS:
        if len(products) >= BLOCK_MOST:
            return kernels.linear_block_group(products)
    elif any(isinstance(p, Product) and together(p.x, p.linear) for p in products):
        return kernels.linear_group(products)
    return [p.alone() for p in products]


def linear_group_plain(products: list[Product | Routing | ExpertsDown]) -> list[torch.Tensor]:
    """The results of products (and of a mixture's routing or its experts' second product) that do not read one another's, in order; each
    with the roundings it has alone."""
    return [p.alone() for p in products]


def group_pays(m: int, n: int, k: int) -> bool:
    """Whether a product of m rows over an [n, k] weight joins a launch of several. Not where few waves share its K and each has a long run of it:
    the launch holds two to sixteen such tiles a block and a wave four loads at a time, which leaves units idle that the product by itself fills.
    And not the widest weights, which fill the chip by themselves, in blocks that hold two tiles above eight rows. Measured, us, beside
    2,048 x 2,048, together | one after the other at 1 / 16 rows: 4,096 columns of K 2,816 (8 waves, 11 steps of 32 each) 9.9 | 10.9 and less, 1,408 (4, 11)
    10.2 | 10.1 at 16 rows, 3,840 (8, 15) 13.9 | 13.8 at 16; 4,352 (8, 17) 16.0 | 14.9 at 16, 11,008 (8, 43) 25.6 | 20.4 and 35.5 | 25.8, 5,504 (4, 43) 20.2 | 15.0
    and 33.6 | 17.1, 1,440 (1, 45) 18.9 | 10.1 and 25.5 | 11.6; two of 8,192 x 8,192 (8, 32) faster together at any rows, 12,288 x 4,096 at 4 rows, but 42.8 | 41.6 at
    16; 9,216 x 4,096 27.0 | 25.5, 16,384 x 2,048 15.0 | 15.0 at 4 rows and 19.9 | 17.6 at 16, two of 24,576 x 2,048 35.0 | 33.7 and 45.5 | 35.8."""
    waves = few_row_waves(n, k)
    return n <= (12288 if m <= 8 else 8192) and (waves == (16 if n < 5120 else 8) or k // (32 * waves) <= 15)


@functools.lru_cache(maxsize=1024)
def few_row_waves(n: int, k: int) -> int:
    """Waves a tile of 16 columns of a few-row product over an [n, k] weight, as the kernels' `skinny_waves` has them."""
    return next(w for w in (16, 8, 4, 2, 1) if w <= (16 if n < 5120 else 8) and k % (32 * w) == 0)


@functools.lru_cache(maxsize=1024)
def beside_pays(hidden: int, n: int, k: int) -> bool:
    """Whether a mixture's second product into `hidden` columns and a product of the same rows over an [n, k] weight share a launch: a block of
    eight waves for 16 of the mixture's columns, and one for one to eight tiles of the other's. It saves a launch, and where either leaves units
    idle a round of blocks. Where neither is so, the mixture's blocks full rounds of 256 and no round fewer together, the other product's blocks
    wait for the mixture's units; what they then win is that their loads follow one another without a gap, which takes more than four steps of K
    a wave. Over 21,700 steps (1,024 to 8,192 columns, 8 to 128 experts, 512 to 12,288 columns of the other, K of 256 to 8,192, 1 to 16 rows, weights from
    memory) the choice is 0.3 % from the better on average and takes 0.86 of the time apart (always together 0.6 %, never 18 %); 4 % are more than 2 %
    longer than apart, most of them beside 12,288 columns, up to 21 % beside a small mixture there. In us, 8 experts, one row unless noted, together |
    apart: 2,048 columns beside 2,048 x 2,048 12.6 | 16.3 and 31.2 | 36.3 at 16, 12,288 x 2,048 16.3 | 19.4; 2,560 beside 2,560 x 1,024 10.4 | 11.3;
    3,072 beside 2,048 x 1,024 10.7 | 12.5; 3,584 beside 1,024 x 3,584 12.7 | 17.3, 12,288 x 1,024 14.1 | 12.3; 5,120 beside 12,288 x 2,048 at three 32.7 | 42.8;
    4,096 beside 4,096 x 4,096 15.5 | 16.4, 4,096 x 8,192 at four 26.0 | 26.6, and what stays apart: 4,096 x 2,048 9.7 | 9.8 and 24.7 | 23.2 at 16,
    2,048 x 1,024 9.4 | 8.6; 8,192 beside 4,096 x 1,024 20.2 | 19.7."""
    mixture, waves = hidden // 16, few_row_waves(n, k)
    product = -(-(n // 16) // (8 // min(waves, 8)))
    return mixture % 256 != 0 or k > 4 * 32 * waves or -(-(mixture + product) // 256) < -(-mixture // 256) + -(-product // 256)


def _served(p: Product) -> bool:
    """Whether the few-row product over a tiled copy serves it (what `linear` and `linear_relu2` would run), and a launch of several pays."""
    x, w, tiled = p.x, p.linear.weight, p.linear.tiled
    return (tiled is not None and p.linear.folded is None and x.is_cuda and x.dtype == tiled.dtype == torch.bfloat16 and x.dim() == 2
            and 1 <= x.shape[0] <= FEW_ROWS and x.is_contiguous() and tiled.is_contiguous() and tiled.shape == w.shape
            and x.shape[1] == w.shape[1] and w.shape[0] % 16 == 0 and w.shape[1] % 32 == 0 and w.shape[1] >= 256
            and x.data_ptr() % 16 == 0 and p.dtype in (None, torch.bfloat16, torch.float32) and not (p.relu2 and p.dtype == torch.float32)
            and group_pays(x.shape[0], *w.shape))


SCORES = {"softmax": 0, "sigmoid": 1, "sigmoid_squared": 2}


def _linear_group_hip(launch, products: list[Product | Routing | ExpertsDown]) -> list[torch.Tensor]:
    launch, launch_beside = launch
    out: list = [None] * len(products)
    by_rows: dict[int, list[int]] = {}
    routes: dict[int, list[int]] = {}
    downs: dict[int, list[int]] = {}
    for i, p in enumerate(products):
        if isinstance(p, (Routing, ExpertsDown)):
            if p.served():
                (routes if isinstance(p, Routing) else downs).setdefault(p.x.shape[0], []).append(i)
        elif _served(p):
            by_rows.setdefault(p.x.shape[0], []).append(i)
    for rows, which in by_rows.items():
        for group in (which[at: at + MOST] for at in range(0, len(which), MOST)):
            route = routes[rows].pop(0) if routes.get(rows) else None
            if len(group) == 1 and route is None:
                p = products[group[0]]
                at = next((d for d in downs.get(rows, ()) if beside_pays(products[d].tiled.shape[0], *p.linear.weight.shape)), None)
                if at is not None:                        # a mixture's experts beside it (several products fill the chip by themselves)
                    downs[rows].remove(at)
                    out[group[0]], out[at] = _beside(launch_beside, p, products[at])
                continue
            items = []
            for i in group:
                p = products[i]
                form = 4 if p.relu2 else 2 if p.dtype == torch.float32 else 0
                n, k = p.linear.weight.shape
                out[i] = torch.empty((rows, n), dtype=torch.float32 if form == 2 else torch.bfloat16, device=p.x.device)
                items += [p.x.data_ptr(), p.linear.tiled.data_ptr(), out[i].data_ptr(), n, k, form]
            with_it, scale = None, 0.0
            if route is not None:
                p = products[route]
                out[route] = torch.empty((rows, p.router.shape[0]), dtype=torch.float32, device=p.x.device)
                score, scale = (SCORES[p.score], 0.0) if p.scale is None else (-1, float(p.scale))
                with_it = (ctypes.c_int64 * 11)(p.x.data_ptr(), p.router.data_ptr(), 0 if p.bias is None else p.bias.data_ptr(),
                                                out[route].data_ptr(), p.x.shape[1], p.experts, p.router.shape[0], p.top, p.groups, p.keep, score)
            launch((ctypes.c_int64 * len(items))(*items), len(group), rows, with_it, scale)
    return [y if y is not None else p.alone() for y, p in zip(out, products)]


def _beside(launch, p: Product, d: ExpertsDown) -> tuple[torch.Tensor, torch.Tensor]:
    """A product and a mixture's second one, in one launch."""
    form = 4 if p.relu2 else 2 if p.dtype == torch.float32 else 0
    rows, (n, k), hidden = p.x.shape[0], p.linear.weight.shape, d.tiled.shape[0]
    y = torch.empty((rows, n), dtype=torch.float32 if form == 2 else torch.bfloat16, device=p.x.device)
    out = torch.empty((rows, hidden), dtype=torch.bfloat16, device=p.x.device)
    launch(d.x.data_ptr(), d.tiled.data_ptr(), out.data_ptr(), rows, hidden, d.experts, d.ff, d.shared, d.weights.data_ptr(),
           d.weights.shape[1], p.x.data_ptr(), p.linear.tiled.data_ptr(), y.data_ptr(), n, k, form)
    return y, out


_P, _I = ctypes.c_void_p, ctypes.c_int
register_kernel(KernelOp("linear_group", linear_group_plain, ("holon_gemm_skinny_group_bf16", "holon_moe_down_beside_bf16"),
                         ([_P, _I, _I, _P, ctypes.c_float], [_P, _P, _P, _I, _I, _I, _I, _I, _P, _I, _P, _P, _P, _I, _I, _I]),
                         _linear_group_hip))


def block_group_pays(count: int, m: int, n: int, k: int) -> bool:
    """Whether `count` bfloat16 products of m rows over [n, k] weights run as one launch on 256 x 256 tiles rather than one after the
    other. A tile takes about 5 us + K / 64 however few of the 256 compute units have one, so that one product of 2,048 rows and
    columns leaves three quarters of the chip idle (36 us; the library's smaller tiles 25), and four of them take 63 us where the
    library's four take 100. Four products against the library's, inside a graph: 36 | 36 us at 129 rows of 2,048 x 2,048, 37 | 44
    at 400, 42 | 65 at 1,024, 103 | 127 at 3,000, 123 | 155 at 4,096; 2,560 x 2,560: 43 | 43 at 129, 57 | 104 at 1,024, 187 | 221 at
    4,096; 4,096 x 4,096: 71 | 88 at 129, 114 | 181 at 1,024, 308 | 347 at 3,000, then 406 | 385 at 4,096, where one product fills
    the chip by itself. Wider weights gain on the library as long, tile for tile: 8,192 x 2,048 40 | 52 at 129 rows, 102 | 135 at 1,024, 200 | 203 at 2,048 (256
    tiles a product), 244 | 306 and 288 | 343 at 2,560 and 3,072; 8,192 x 4,096 75 | 96, 197 | 253, 369 | 386, 481 | 547, 577 | 622; 8,192 x 1,024 115 | 123 at 2,048; 5,120 x
    2,560 226 | 231 at 3,072. 1,024 x 2,048 at 129 and 256 rows 34.7 | 32.7 and 35.2 | 34.5, at 400 35.9 | 38.5. Two or three gain little or lose at most sizes (three of 4,096 x 4,096 at 1,400 rows 155 | 153)."""
    return count == BLOCK_MOST and BLOCK_ROWS[0] <= m <= BLOCK_ROWS[1] and 1024 <= n <= 8192 and 1024 <= k < 8192 and k % 128 == 0 and n % 16 == 0


def _block_served(p: Product | Routing) -> bool:
    if not isinstance(p, Product) or p.relu2 or p.dtype not in (None, torch.bfloat16) or not isinstance(p.x, torch.Tensor):
        return False
    x, w = p.x, p.linear.weight
    return (x.is_cuda and w is not None and x.dtype == w.dtype == torch.bfloat16 and x.dim() == w.dim() == 2 and x.shape[1] == w.shape[1]
            and x.is_contiguous() and w.is_contiguous() and (x.data_ptr() | w.data_ptr()) % 16 == 0)


def linear_block_group_plain(products: list[Product | Routing]) -> list[torch.Tensor]:
    """What `linear_group` returns, of products of many rows."""
    return [p.alone() for p in products]


def _linear_block_group_hip(launch, products: list[Product | Routing]) -> list[torch.Tensor]:
    out: list = [None] * len(products)
    alike: dict[tuple, list[int]] = {}
    for i, p in enumerate(products):
        if _block_served(p):
            alike.setdefault((p.x.shape[0], *p.linear.weight.shape), []).append(i)
    for (m, n, k), which in alike.items():
        for at in range(0, len(which), BLOCK_MOST):
            group = which[at: at + BLOCK_MOST]
            first = products[group[0]].linear
            # (a model whose sums stay as they are keeps the library's order of them)
            if not block_group_pays(len(group), m, n, k) or first.kernels.settled or \
                    first.kernels.product_choice("group", first.weight, m, yields=True, by_rule=True) != "own":
                continue
            y = torch.empty((len(group), m, n), dtype=torch.bfloat16, device=products[group[0]].x.device)
            for i, rows in zip(group, y):
                out[i] = rows
            operands = [products[i].x.data_ptr() for i in group] + [products[i].linear.weight.data_ptr() for i in group] + \
                [out[i].data_ptr() for i in group]
            launch((ctypes.c_int64 * len(operands))(*operands), len(group), m, n, k)
    return [y if y is not None else p.alone() for y, p in zip(out, products)]


register_kernel(KernelOp("linear_block_group", linear_block_group_plain, "holon_gemm_block_group_bf16",
                         [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int], _linear_block_group_hip))
