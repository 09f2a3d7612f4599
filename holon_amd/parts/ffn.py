"""Feed-forward parts. SwiGLU: std/holon_std/ffn/units.py:12-50, activation std/holon_std/ffn/reference.py:7-12.
Beside it a dense feed-forward with the PolyNorm activation and a mixture of experts (HIP forms of their elementwise
steps: `csrc/ffn_kinds.hip`)."""
from __future__ import annotations

import ctypes

import torch

from ..kernels.registry import KernelOp, register_kernel
from ..registry import register_part
from .base import FLOAT32, Build, Part, Stream
from .linear import Linear
from .norms import Normed
from .products import ExpertsDown, Product, Routing, by_itself, together


@register_part("ffn", "swiglu")
class SwiGLU(Part):
    """down(act(gate(x)) * up(x)) with act silu, or gelu in its tanh form (`act` "gelu_tanh"); gate and up are merged into
    one product after loading (gate rows first)."""

    graph_safe = True
    ACTS = ("silu", "gelu_tanh")

    def __init__(self, build: Build, *, inter: int, hidden: int, layer: int, act: str = "silu") -> None:
        super().__init__(build)
        if act not in self.ACTS:
            raise ValueError(f"ffn swiglu: no activation {act!r} ({', '.join(self.ACTS)})")
        self.inter, self.hidden, self.act = inter, hidden, act
        self.attach("gate_proj", Linear(build, inp=hidden, out=inter))
        self.attach("up_proj", Linear(build, inp=hidden, out=inter))
        self.attach("down_proj", Linear(build, inp=inter, out=hidden))
        self.gate_up: Linear | None = None

    def finalize(self) -> None:
        self.gate_up = Linear.merge(self.build, self.gate_proj, self.up_proj)
        self.drop("gate_proj")
        self.drop("up_proj")
        self._children["gate_up"] = self.gate_up

    adds_residual = True

    def absorb_norm(self, norm: Part) -> bool:
        """Fold the norm in front of this part into its first product; it then takes `Normed` input (the kernels that do
        are silu's)."""
        return self.act == "silu" and self.gate_up.absorb(norm)

    def forward(self, x: torch.Tensor | Normed, step=None, residual: Stream | None = None) -> torch.Tensor | None:
        gate_up, y = self.gate_up, None
        if self.act == "gelu_tanh":
            x = x.value() if isinstance(x, Normed) else x
            y = self.kernels.linear_gelu_mul(x, gate_up.weight, gate_up.tiled)
            return self.down_proj(self.kernels.gelu_mul(gate_up(x)) if y is None else y, residual=residual)
        if gate_up.folds(x):
            y = self.kernels.linear_silu_mul(x.h, gate_up.weight, gate_up.tiled, row_scale=gate_up.row_scale(x))
        elif gate_up.reads_folded(x, gated=True):  # 17 to 64 rows: the folded copy over rows normed without the weight
            y = self.kernels.linear_silu_mul(x.unit_value(), gate_up.weight, gate_up.tiled)
        elif gate_up.folded is None or x.shape[0] > 128:      # fused for steps of few rows, and of many (over the weight as it is)
            x = x.value() if isinstance(x, Normed) else x
            y = self.kernels.linear_silu_mul(x, gate_up.weight, gate_up.tiled if gate_up.folded is None else None)
        if y is None:
            y = self.kernels.silu_mul(gate_up(x))
        return self.down_proj(y, residual=residual)

    __call__ = forward


# -- a dense feed-forward with the PolyNorm activation, and a mixture of experts ------------------------------------------
_P, _I, _L, _F = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_float
_DT = {torch.float32: 0, torch.bfloat16: 1}


def _need(cond: bool, what: str) -> None:
    if not cond:
        raise ValueError(what)


def gelu_mul_plain(gate_up):
    """gate_up [T, 2 F] (gates, then ups) -> gelu(gate) * up [T, F], gelu in its tanh form; the gelu is rounded to the
    rows' dtype before the product, as silu_mul rounds."""
    gate, up = gate_up.chunk(2, dim=-1)
    wide = gate if gate.dtype == torch.float64 else gate.float()
    return torch.nn.functional.gelu(wide, approximate="tanh").to(gate.dtype) * up


def _gelu_mul_hip(launch, gate_up):
    _need(gate_up.is_cuda and gate_up.is_contiguous() and gate_up.dim() == 2 and gate_up.dtype in _DT
          and gate_up.shape[1] % 2 == 0, "gelu_mul: contiguous rows of gates and ups on the GPU")
    y = torch.empty((gate_up.shape[0], gate_up.shape[1] // 2), dtype=gate_up.dtype, device=gate_up.device)
    launch(gate_up.data_ptr(), y.data_ptr(), y.shape[0], y.shape[1], _DT[gate_up.dtype])
    return y


def linear_gelu_mul_plain(x, weight, tiled=None):
    """gelu_mul(x W^T) where one kernel does both, with the roundings of the two one after the other; None where it does
    not (the caller then composes them). The plain form never does."""
    return None


def _linear_gelu_mul_hip(launch, x, weight, tiled=None):
    """Steps of up to 16 bfloat16 rows: the few-row product with the activation in its epilogue."""
    (m, k), n = x.shape, weight.shape[0]
    if not (x.is_cuda and x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and x.is_contiguous()
            and weight.is_contiguous() and weight.shape[1] == k and 1 <= m <= 16 and n % 32 == 0 and k % 128 == 0
            and k >= 256 and (tiled is None or (tiled.shape == weight.shape and tiled.dtype == weight.dtype
                                                 and tiled.is_contiguous()))):
        return None
    y = torch.empty((m, n // 2), dtype=torch.bfloat16, device=x.device)
    launch(x.data_ptr(), (tiled if tiled is not None else weight).data_ptr(), y.data_ptr(), m, n // 2, k,
           int(tiled is not None))
    return y


def linear_glu_plain(x, weight, act):
    """A gated first product of many rows with its activation: what a kernel set that has a choice of forms for it answers for itself
    (`kernels.api.Kernels.linear_glu`); the plain form is the composition."""
    return None


def polynorm_plain(z, coef, eps):
    """z [T, F], coef [4] float32 = (a, b, c, e): a N(z) + b N(z^2) + c N(z^3) + e with the powers taken element by
    element and N(v) = v / sqrt(mean(v^2) + eps) over a row. float32 inside, one rounding to z's dtype."""
    x = z.float()
    a, b, c, e = coef.float().unbind(0)

    def unit(v):
        return v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + eps)
    return (a * unit(x) + b * unit(x * x) + c * unit(x * x * x) + e).to(z.dtype)


def _polynorm_hip(launch, z, coef, eps):
    _need(z.is_cuda and z.is_contiguous() and z.dim() == 2 and z.dtype in _DT and coef.is_cuda and coef.is_contiguous()
          and coef.dtype == torch.float32 and coef.shape == (4,), "polynorm: contiguous rows and four float32 numbers")
    y = torch.empty_like(z)
    if z.shape[0]:
        launch(z.data_ptr(), coef.data_ptr(), y.data_ptr(), z.shape[0], z.shape[1], float(eps), _DT[z.dtype])
    return y


def moe_route_plain(logits, correction, top, groups, keep, scale):
    """Router logits [T, E] float32 -> weights [T, E] float32: s = sigmoid(logits); experts are chosen by s +
    `correction` [E] (None: by s): the `top` largest among the experts of the `keep` best of `groups` equal groups of
    neighbouring experts, a group's score being the sum of its two largest choice scores (groups <= 1: among all).
    A chosen expert's weight is s * scale (the score without the correction, not renormalised), every other 0."""
    s = torch.sigmoid(logits.float())
    choice = s if correction is None else s + correction.float()
    t, e = s.shape
    if groups > 1:
        size = e // groups
        score = choice.view(t, groups, size).topk(min(2, size), dim=-1).values.sum(-1)
        best = score.topk(keep, dim=-1).indices
        open_ = torch.zeros((t, groups), dtype=torch.bool, device=s.device).scatter_(1, best, True)
        choice = choice.masked_fill(~open_.repeat_interleave(size, dim=1), float("-inf"))
    chosen = choice.topk(top, dim=-1).indices
    return torch.zeros_like(s).scatter_(1, chosen, s.gather(1, chosen) * scale)


def _moe_route_hip(launch, logits, correction, top, groups, keep, scale):
    t, e = logits.shape
    _need(logits.is_cuda and logits.is_contiguous() and logits.dtype == torch.float32 and 1 <= top <= e <= 1024
          and (correction is None or (correction.dtype == torch.float32 and correction.is_contiguous()
                                      and correction.shape == (e,)))
          and (groups <= 1 or (e % groups == 0 and 1 <= keep <= groups)),
          f"moe_route: {e} experts, top {top}, {groups} groups of which {keep} (float32 logits, at most 1,024 experts)")
    w = torch.empty_like(logits)
    if t:
        launch(logits.data_ptr(), None if correction is None else correction.data_ptr(), w.data_ptr(), t, e, int(top),
               int(groups), int(keep), float(scale))
    return w


def moe_router_plain(x, router, correction, top, groups, keep, scale):
    """x [T, W] (any dtype), router [E, W] float32: the float32 logits x . router[e], then `moe_route` on them."""
    return moe_route_plain(x.float() @ router.float().T, correction, top, groups, keep, scale)


def _moe_router_hip(launch, x, router, correction, top, groups, keep, scale):
    (t, w), e = x.shape, router.shape[0]
    _need(x.is_cuda and x.is_contiguous() and x.dtype in _DT and router.is_contiguous() and router.dtype == torch.float32
          and router.shape == (e, w) and 1 <= top <= e <= 1024 and w <= 12288
          and (correction is None or (correction.dtype == torch.float32 and correction.is_contiguous()
                                      and correction.shape == (e,)))
          and (groups <= 1 or (e % groups == 0 and 1 <= keep <= groups)),
          f"moe_router: rows {tuple(x.shape)} {x.dtype}, {e} experts, top {top}, {groups} groups of which {keep}")
    weights = torch.empty((t, e), dtype=torch.float32, device=x.device)
    if t:
        launch(x.data_ptr(), router.data_ptr(), None if correction is None else correction.data_ptr(),
               weights.data_ptr(), t, w, e, int(top), int(groups), int(keep), float(scale), _DT[x.dtype])
    return weights


def moe_gate_plain(gate_up, weights, ff, shared, shared_weight=False):
    """gate_up [T, 2 C] with C = E ff + shared columns of gates, then as many of ups; weights [T, E] float32.
    -> [T, C]: silu(gate) * up (as `silu_mul` rounds it), times the weight of the column's expert (column c belongs to
    expert c // ff; the last `shared` columns to an expert that every token uses with weight 1); exactly 0 where the
    weight is 0. One more rounding for the weight. `shared_weight`: weights is [T, E + 1] and its last column is the
    weight of the shared expert's columns."""
    t, e = weights.shape[0], weights.shape[1] - int(bool(shared_weight))
    c = e * ff + shared
    g, u = gate_up[:, :c].float(), gate_up[:, c:].float()
    act = ((g * torch.sigmoid(g)).to(gate_up.dtype).float() * u).to(gate_up.dtype)
    w = weights[:, :e].repeat_interleave(ff, dim=1)
    if shared:
        last = weights[:, e:].expand(t, shared) if shared_weight else torch.ones((t, shared), dtype=w.dtype, device=w.device)
        w = torch.cat((w, last), dim=1)
    return torch.where(w == 0, torch.zeros_like(act), (act.float() * w).to(gate_up.dtype))


def _moe_gate_hip(launch, gate_up, weights, ff, shared, shared_weight=False):
    t, e = weights.shape[0], weights.shape[1] - int(bool(shared_weight))
    c = e * ff + shared
    _need(gate_up.is_cuda and gate_up.is_contiguous() and gate_up.dtype in _DT and gate_up.shape == (t, 2 * c)
          and weights.is_contiguous() and weights.dtype == torch.float32 and e >= 1,
          f"moe_gate: rows {tuple(gate_up.shape)} for {e} experts of {ff} and {shared} shared columns")
    y = torch.empty((t, c), dtype=gate_up.dtype, device=gate_up.device)
    if t:
        launch(gate_up.data_ptr(), weights.data_ptr(), y.data_ptr(), t, e, ff, shared, _DT[gate_up.dtype],
               weights.shape[1], e if shared_weight else -1)
    return y


ROUTER_SCORES = {"softmax": 0, "sigmoid": 1, "sigmoid_squared": 2}


def moe_router_top_plain(x, router, bias, experts, top, groups=1, keep=1, score="softmax"):
    """x [T, W] (any dtype), router [R, W] float32 with R = experts or experts + 1, bias [experts] float32 or None:
    the float32 logits z = x . router[e] + bias[e]; the `top` largest are chosen (equal ones: the lower index first)
    and weighted by the softmax over the chosen logits alone, every other expert 0. `groups` > 1: only experts of the
    `keep` best of as many equal groups of neighbours can be chosen, a group's score being its largest logit. A last
    row beyond the experts is a gate: its column holds sigmoid(x . router[experts]). `score` "sigmoid": a chosen expert's
    weight is sigmoid(z_e) alone, "sigmoid_squared": that squared. -> [T, R] float32."""
    z = x.float() @ router.float().T
    logits = z[:, :experts] + (bias.float() if bias is not None else 0.0)
    choice = logits
    if groups > 1:
        best = logits.view(-1, groups, experts // groups).amax(-1)
        best = torch.sort(best, dim=-1, descending=True, stable=True).indices[:, :keep]
        open_ = torch.zeros((logits.shape[0], groups), dtype=torch.bool, device=x.device).scatter_(1, best, True)
        choice = logits.masked_fill(~open_.repeat_interleave(experts // groups, dim=1), float("-inf"))
    order = torch.sort(choice, dim=-1, descending=True, stable=True).indices[:, :top]
    chosen = logits.gather(1, order)
    weigh = {"softmax": lambda z: torch.softmax(z, dim=-1), "sigmoid": torch.sigmoid,
             "sigmoid_squared": lambda z: torch.sigmoid(z).square()}[score]
    w = torch.zeros_like(logits).scatter_(1, order, weigh(chosen))
    return torch.cat((w, torch.sigmoid(z[:, experts:])), dim=1).contiguous()


def _moe_router_top_hip(launch, x, router, bias, experts, top, groups=1, keep=1, score="softmax"):
    (t, w), r = x.shape, router.shape[0]
    _need(x.is_cuda and x.is_contiguous() and x.dtype in _DT and router.is_contiguous() and router.dtype == torch.float32
          and router.shape == (r, w) and r in (experts, experts + 1) and 1 <= top <= experts <= 1024 and w <= 12288
          and (bias is None or (bias.dtype == torch.float32 and bias.is_contiguous() and bias.shape == (experts,)))
          and (groups <= 1 or (experts % groups == 0 and 1 <= keep <= groups and top <= keep * (experts // groups))),
          f"moe_router_top: rows {tuple(x.shape)} {x.dtype}, router {tuple(router.shape)}, top {top} of {experts}, "
          f"{groups} groups of which {keep}")
    weights = torch.empty((t, r), dtype=torch.float32, device=x.device)
    if t:
        launch(x.data_ptr(), router.data_ptr(), None if bias is None else bias.data_ptr(), weights.data_ptr(), t, w,
               experts, r, int(top), _DT[x.dtype], int(groups), int(keep), ROUTER_SCORES[score])
    return weights


def moe_relu2_plain(up, weights, ff, shared, shared_weight=False):
    """up [T, C] with C = E ff + shared columns -> max(up, 0)^2 times the weight of the column's expert, float32 inside and
    one rounding, exactly 0 where the weight is 0; columns and weights as for `moe_gate`."""
    t, e = weights.shape[0], weights.shape[1] - int(bool(shared_weight))
    w = weights[:, :e].repeat_interleave(ff, dim=1)
    if shared:
        last = weights[:, e:].expand(t, shared) if shared_weight else torch.ones((t, shared), dtype=w.dtype, device=w.device)
        w = torch.cat((w, last), dim=1)
    return torch.where(w == 0, torch.zeros_like(w), torch.relu(up.float()).square() * w).to(up.dtype)


def _moe_relu2_hip(launch, up, weights, ff, shared, shared_weight=False):
    t, e = weights.shape[0], weights.shape[1] - int(bool(shared_weight))
    c = e * ff + shared
    _need(up.is_cuda and up.is_contiguous() and up.dtype in _DT and up.shape == (t, c) and weights.is_contiguous()
          and weights.dtype == torch.float32 and e >= 1, f"moe_relu2: rows {tuple(up.shape)} for {e} experts of {ff} and "
          f"{shared} shared columns")
    y = torch.empty_like(up)
    if t:
        launch(up.data_ptr(), weights.data_ptr(), y.data_ptr(), t, e, ff, shared, _DT[up.dtype], weights.shape[1],
               e if shared_weight else -1)
    return y


def relu2_plain(z):
    """z [T, F] -> max(z, 0)^2, float32 inside, one rounding."""
    return torch.relu(z.float()).pow(2).to(z.dtype)


def _relu2_hip(launch, z):
    _need(z.is_cuda and z.is_contiguous() and z.dtype in _DT, "relu2: contiguous float32 or bfloat16 values on the GPU")
    y = torch.empty_like(z)
    if z.numel():
        launch(z.data_ptr(), y.data_ptr(), z.numel(), _DT[z.dtype])
    return y


register_kernel(KernelOp("polynorm", polynorm_plain, "holon_polynorm", [_P, _P, _P, _L, _I, _F, _I], _polynorm_hip))
register_kernel(KernelOp("moe_route", moe_route_plain, "holon_moe_route", [_P, _P, _P, _L, _I, _I, _I, _I, _F],
                         _moe_route_hip))
register_kernel(KernelOp("moe_router", moe_router_plain, "holon_moe_router",
                         [_P, _P, _P, _P, _L, _I, _I, _I, _I, _I, _F, _I], _moe_router_hip))
register_kernel(KernelOp("moe_gate", moe_gate_plain, "holon_moe_gate", [_P, _P, _P, _L, _I, _I, _I, _I, _I, _I],
                         _moe_gate_hip))
register_kernel(KernelOp("moe_router_top", moe_router_top_plain, "holon_moe_router_top",
                         [_P, _P, _P, _P, _L, _I, _I, _I, _I, _I, _I, _I, _I], _moe_router_top_hip))
register_kernel(KernelOp("moe_relu2", moe_relu2_plain, "holon_moe_relu2", [_P, _P, _P, _L, _I, _I, _I, _I, _I, _I],
                         _moe_relu2_hip))
register_kernel(KernelOp("gelu_mul", gelu_mul_plain, "holon_gelu_mul", [_P, _P, _L, _I, _I], _gelu_mul_hip))
register_kernel(KernelOp("linear_gelu_mul", linear_gelu_mul_plain, "holon_gemm_skinny_geglu_bf16",
                         [_P, _P, _P, _I, _I, _I, _I], _linear_gelu_mul_hip))
register_kernel(KernelOp("linear_glu", linear_glu_plain))
register_kernel(KernelOp("relu2", relu2_plain, "holon_relu2", [_P, _P, _L, _I], _relu2_hip))


def linear_relu2_plain(x, weight, tiled=None):
    """relu2(x W^T) where one kernel does both, with the roundings of the two one after the other; None where it does
    not (the caller then composes them). The plain form never does."""
    return None


def _linear_relu2_hip(launch, x, weight, tiled=None):
    """Steps of up to 16 bfloat16 rows: the few-row product with the activation in its epilogue."""
    (m, k), n = x.shape, weight.shape[0]
    if not (x.is_cuda and x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and x.is_contiguous()
            and weight.is_contiguous() and weight.shape[1] == k and 1 <= m <= 16 and n % 16 == 0 and k % 32 == 0
            and k >= 256 and (tiled is None or (tiled.shape == weight.shape and tiled.dtype == weight.dtype
                                                 and tiled.is_contiguous()))):
        return None
    y = torch.empty((m, n), dtype=torch.bfloat16, device=x.device)
    launch(x.data_ptr(), (tiled if tiled is not None else weight).data_ptr(), y.data_ptr(), m, n, k, 4,
           int(tiled is not None))
    return y


register_kernel(KernelOp("linear_relu2", linear_relu2_plain, "holon_gemm_skinny_bf16", [_P, _P, _P, _I, _I, _I, _I, _I],
                         _linear_relu2_hip))


def moe_few_serves(rows: int, hidden: int, experts: int, ff: int, shared: int) -> bool:
    """What the library's `holon_moe_few_supported` answers."""
    return 1 <= rows <= 16 and hidden % 32 == 0 and experts <= 1024 and ff % 32 == 0 and shared % 32 == 0


def moe_few_pays(rows: int, hidden: int, experts: int, ff: int, gated: bool, top: int) -> bool:
    """Whether a step is done sooner over the chosen experts' columns than over all. By a fit on MI355X over 3,016 steps of 1 to 16 rows
    (hidden 256 to 4,096, 4 to 128 experts of 64 to 4,096 columns, 1 to 8 a token, up to 1.5 choices an expert, each both ways): in us,
    what the columns that no row is expected to choose take, against a start, the search through rows x experts weights and a start an
    expert chosen. The choice is 0.6 % from the better of the two on average; the chosen ones wherever there were up to 1.5 choices an
    expert took up to 2.7 times as long as all (128 experts of 64 columns, 16 rows). Of 8 experts of 2,048 x 2,048 beside a shared one,
    2 a token, 1 / 2 / 4 rows take 21 / 29 / 37 us over the chosen ones and 48 / 49 / 50 over all; of 64 of 4,096 x 512, 6 a token, 1 / 4 /
    16 rows 28 / 57 / 137 and 133 / 129 / 155."""
    if 2 * rows * top > 3 * experts:
        return False
    left = experts * (1 - top / experts) ** rows
    column = 2e-7 * (3 if gated else 2) * hidden + 7e-4 + 4.5e-5 * rows
    return 1 + 0.01 * rows * experts + 0.25 * (experts - left) < column * ff * left


def _moe_up_few_hip(launch, x, weights, up_tiled, down_tiled, experts, ff, shared, gated, shared_weight=False):
    t, hidden = x.shape
    cols = experts * ff + shared
    if up_tiled is None or down_tiled is None or x.dtype != torch.bfloat16 or not moe_few_serves(t, hidden, experts, ff, shared):
        return None
    _need(x.is_cuda and x.is_contiguous() and weights.is_contiguous() and weights.dtype == torch.float32
          and tuple(weights.shape) == (t, experts + int(bool(shared_weight)))
          and all(w.is_contiguous() and w.dtype == x.dtype for w in (up_tiled, down_tiled))
          and tuple(up_tiled.shape) == ((2 if gated else 1) * cols, hidden) and tuple(down_tiled.shape) == (hidden, cols),
          f"moe_up_few: rows {tuple(x.shape)}, weights {tuple(weights.shape)}, projections {tuple(up_tiled.shape)} and "
          f"{tuple(down_tiled.shape)} for {experts} experts of {ff} and {shared} shared columns")
    act = torch.empty((t, cols), dtype=x.dtype, device=x.device)
    launch(x.data_ptr(), up_tiled.data_ptr(), act.data_ptr(), t, hidden, experts, ff, shared, int(bool(gated)), weights.data_ptr(),
           weights.shape[1], experts if shared_weight else -1)
    return act


def _moe_down_few_hip(launch, act, weights, down_tiled, experts, ff, shared):
    t, hidden = act.shape[0], down_tiled.shape[0]
    cols = experts * ff + shared
    _need(act.is_cuda and act.is_contiguous() and act.dtype == down_tiled.dtype == torch.bfloat16 and weights.is_contiguous()
          and weights.dtype == torch.float32 and weights.dim() == 2 and weights.shape[0] == t and weights.shape[1] >= experts
          and down_tiled.is_contiguous() and moe_few_serves(t, hidden, experts, ff, shared)
          and tuple(act.shape) == (t, cols) and tuple(down_tiled.shape) == (hidden, cols),
          f"moe_down_few: activations {tuple(act.shape)}, weights {tuple(weights.shape)}, projection {tuple(down_tiled.shape)} for {experts} "
          f"experts of {ff} and {shared} shared columns")
    y = torch.empty((t, hidden), dtype=act.dtype, device=act.device)
    launch(act.data_ptr(), down_tiled.data_ptr(), y.data_ptr(), t, hidden, experts, ff, shared, weights.data_ptr(),
           weights.shape[1])
    return y


def moe_up_few_plain(x, weights, up_tiled, down_tiled, experts, ff, shared, gated, shared_weight=False):
    """The experts' first product and the activation behind it for steps of few rows, reading the chosen experts' weights alone, with the
    roundings of `linear` and `moe_gate` (`gated`) or `moe_relu2`: [T, experts ff + shared], columns of experts that no row chose left as
    the memory was; None where the two products are not served (the caller then composes them with those). The plain form never does."""
    return None


def moe_down_few_plain(act, weights, down_tiled, experts, ff, shared):
    """The second product over what `moe_up_few` left, reading the chosen experts' weights alone, with the rounding of `linear`."""
    n, k = down_tiled.shape
    down = down_tiled.view(n // 16, k // 32, 4, 16, 8).permute(0, 3, 1, 2, 4).reshape(n, k)          # (16 rows of 32 columns lie together)
    used = torch.cat(((weights[:, :experts] != 0).repeat_interleave(ff, 1), weights.new_ones(act.shape[0], shared).bool()), 1)
    return (torch.where(used, act, 0).float() @ down.float().T).to(act.dtype)


register_kernel(KernelOp("moe_up_few", moe_up_few_plain, "holon_moe_up_few_bf16", [_P, _P, _P, _I, _I, _I, _I, _I, _I, _P, _I, _I], _moe_up_few_hip))
register_kernel(KernelOp("moe_down_few", moe_down_few_plain, "holon_moe_down_few_bf16", [_P, _P, _P, _I, _I, _I, _I, _I, _P, _I], _moe_down_few_hip))


def moe_rows_plain(x, weights, up, down, experts, top, ff, shared, gated, shared_weight=False):
    """The experts' two products and the activation between them for steps of many rows, every expert over the rows that chose
    it alone, with the roundings of `linear`, `moe_gate` (`gated`) or `moe_relu2`, and `linear` (whose sums over the experts
    are cut at the experts); None where they are not served (the caller then composes the three). The plain form never does."""
    return None


def moe_rows_serves(rows: int, hidden: int, experts: int, top: int, ff: int, shared: int) -> bool:
    """What the library's `holon_moe_rows_supported` answers."""
    def deep(k):
        return k >= 128 and k % 128 == 0
    return 1 <= rows < 1 << 22 and deep(hidden) and deep(ff) and (shared == 0 or deep(shared)) and 1 <= top <= experts <= 1024 \
        and top <= 256 and max(rows * top * ff, rows * hidden, rows * shared, (experts * ff + shared + 128) * hidden,
                               experts * rows) < 1 << 31


def moe_rows_pays(rows: int, hidden: int, experts: int, ff: int, shared: int, gated: bool, top: int) -> bool:
    """Whether a step of many rows is done sooner over every expert's own rows than with all rows over all experts, by what either
    takes in us: tiles of 256 x 256 over 256 compute units (1.6 us a round and 64 columns of K where there are several rounds, 1.3
    where there is one) and the parts' traffic against the products over all (their operations at 1.2 PFLOP/s and their weights at 4
    TB/s). Measured on MI355X, own rows / all (us): 8 experts of 3,072 x 4,096 beside a shared one, 2 a row, at 64 / 512 / 4,096 rows
    181 / 218 / 830 and 226 / 472 / 2,035; of 2,048 x 2,048 at 64 / 512 / 4,096 86 / 93 / 345 and 89 / 211 / 853; 8 of 1,024 beside a
    shared one of 2,048, 4 a row, at 64 / 512 / 1,024 / 4,096 82 / 97 / 113 / 405 and 50 / 85 / 149 / 438; 64 of 512, 6 a row, at 17 /
    32 / 64 / 1,024 89 / 115 / 128 / 168 and 124 / 125 / 131 / 496; the others at 17 / 32 / 63: of 3,072 x 4,096 167 / 178 / 181 and 224 / 215 /
    209, of 2,048 x 2,048 87 / 87 / 86 and 85 / 89 / 90, 8 of 1,024 81 / 82 / 83 and 47 / 45 / 45. A step whose parts would take more memory
    than the products over all stays with those."""
    if rows <= 16:
        return False
    cols = experts * ff + shared
    # (bytes a row: its act, parts and places in the lists, against its products over all and their activation)
    if 2 * (top * ff + shared) + 4 * (top + 1) * hidden + 4 * (experts + top) > (6 if gated else 4) * cols:
        return False
    row_tiles, all_tiles = max(min(experts, rows * top), rows * top / 256 + experts / 2), -(-rows // 256)
    width = 128 if gated else 256
    up = row_tiles * -(-ff // width) + all_tiles * -(-shared // width)
    down = (row_tiles * (0.029 * ff + 8) + (all_tiles * (0.029 * shared + 8) if shared else 0)) * -(-hidden // 256)
    own = 12 + hidden * max(0.0205, 0.029 * up / 256) + max(0.0205 * max(ff, shared), down / 256) + rows * hidden * (top + 1) / 1.1e6
    values = (3 if gated else 2) * cols * hidden
    return own < 0.93 * (20 + 2 * rows * values / 1.2e9 + 2 * values / 4e6)


def _moe_rows_hip(launch, x, weights, up, down, experts, top, ff, shared, gated, shared_weight=False):
    t, hidden = x.shape
    cols = experts * ff + shared
    if x.dtype != torch.bfloat16 or not moe_rows_serves(t, hidden, experts, top, ff, shared) \
            or any(v.data_ptr() % 16 for v in (x, up, down)):
        return None
    _need(x.is_cuda and x.is_contiguous() and weights.is_contiguous() and weights.dtype == torch.float32
          and tuple(weights.shape) == (t, experts + int(bool(shared_weight)))
          and all(w.is_contiguous() and w.dtype == x.dtype for w in (up, down))
          and tuple(up.shape) == ((2 if gated else 1) * cols, hidden) and tuple(down.shape) == (hidden, cols),
          f"moe_rows: rows {tuple(x.shape)}, weights {tuple(weights.shape)}, projections {tuple(up.shape)} and "
          f"{tuple(down.shape)} for {experts} experts of {ff} and {shared} shared columns")
    lists = torch.empty(experts * (t + 1) + t * top, dtype=torch.int32, device=x.device)
    act = torch.empty(t * (top * ff + shared), dtype=x.dtype, device=x.device)
    parts = torch.empty((t * (top + 1), hidden), dtype=torch.float32, device=x.device)
    y = torch.empty_like(x)
    launch(x.data_ptr(), up.data_ptr(), down.data_ptr(), y.data_ptr(), lists.data_ptr(), act.data_ptr(), parts.data_ptr(), t, hidden,
           experts, top, ff, shared, int(bool(gated)), weights.data_ptr(), weights.shape[1], experts if shared_weight else -1)
    return y


register_kernel(KernelOp("moe_rows", moe_rows_plain, "holon_moe_rows_bf16",
                         [_P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _I, _P, _I, _I], _moe_rows_hip))


def moe_f32_plain(x, weights, up, down, experts, top, ff, shared, gated, shared_weight=False):
    """The experts of the 32-bit path over the rows that chose them: the two products and the activation between them, the sums over
    the experts cut at the experts; None where they are not served (the caller then composes the three). The plain form never does."""
    return None


def moe_f32_serves(rows: int, hidden: int, experts: int, top: int, ff: int, shared: int) -> bool:
    """What the library's `holon_moe_f32_supported` answers (of sizes whose counts fit 31 bits)."""
    return 1 <= rows < 1 << 22 and hidden > 0 and ff > 0 and not (hidden % 16 or ff % 16 or shared % 16) and 1 <= top <= experts <= 1024 \
        and top <= 256 and (rows * top // 64 + experts + -(-rows // 64)) * (max(experts * ff + shared, hidden) // 32 + 1) < 1 << 31 \
        and max(2 * (experts * ff + shared), experts * rows, rows * top) < 1 << 31


def moe_f32_takes(hidden: int, experts: int, ff: int, shared: int, gated: bool, top: int) -> bool:
    """Whether a float32 mixture's steps go over the rows that chose an expert, by its sizes alone: the two forms' orders of sums
    differ, and a row has the same bits whatever step it comes in only if one of them takes them all. It is taken where a row chooses
    at most half of the experts and its parts (which steps of more than 16 rows keep) take no more memory than the products over all.
    Measured on MI355X, us, own rows / all: 8 experts of 2,048 x 2,048 (squared ReLU) beside a shared one, 2 a row, at 1 / 4 / 8 / 16 / 17 /
    32 / 64 / 700 rows 52 / 92 / 116 / 136 / 201 / 203 / 203 / 460 and 110 / 111 / 115 / 132 / 152 / 177 / 245 / 1,199; 8 of 1,024 (gated) beside
    one of 2,048, 4 a row, at 1 / 4 / 16 / 17 / 64 / 700 72 / 86 / 123 / 190 / 190 / 703 and 95 / 96 / 109 / 128 / 201 / 945; 64 of 512 x 1,024,
    6 a row, at 1 / 8 / 16 / 32 / 700 40 / 143 / 205 / 185 / 294 and 158 / 163 / 194 / 250 / 1,629; 8 of 3,072 x 4,096 (gated) beside a shared one,
    2 a row, at 1 / 16 / 32 161 / 441 / 561 and 533 / 588 / 659; 128 of 64 x 2,048, 8 a row, at 1 / 8 / 16 / 63 / 200 38 / 114 / 171 / 146 / 150 and
    80 / 83 / 92 / 123 / 310. Decode rows and prompts gain, some 8 to 40 rows a step of small experts lose."""
    cols = experts * ff + shared
    return 2 * top <= experts and top * ff + shared + (top + 1) * hidden + experts + top <= (3 if gated else 2) * cols


def _moe_f32_hip(launch, x, weights, up, down, experts, top, ff, shared, gated, shared_weight=False):
    t, hidden = x.shape
    cols = experts * ff + shared
    if x.dtype != torch.float32 or not moe_f32_serves(t, hidden, experts, top, ff, shared) \
            or any(v.data_ptr() % 16 for v in (x, up, down)):
        return None
    _need(x.is_cuda and x.is_contiguous() and weights.is_contiguous() and weights.dtype == torch.float32
          and tuple(weights.shape) == (t, experts + int(bool(shared_weight)))
          and all(w.is_contiguous() and w.dtype == x.dtype for w in (up, down))
          and tuple(up.shape) == ((2 if gated else 1) * cols, hidden) and tuple(down.shape) == (hidden, cols),
          f"moe_f32: rows {tuple(x.shape)}, weights {tuple(weights.shape)}, projections {tuple(up.shape)} and "
          f"{tuple(down.shape)} for {experts} experts of {ff} and {shared} shared columns")
    few = t <= 16
    lists = None if few else torch.empty(experts * (t + 1) + t * top, dtype=torch.int32, device=x.device)
    act = torch.empty(t * (cols if few else top * ff + shared), dtype=x.dtype, device=x.device)
    parts = None if few else torch.empty((t * (top + 1), hidden), dtype=torch.float32, device=x.device)
    y = torch.empty_like(x)
    launch(x.data_ptr(), up.data_ptr(), down.data_ptr(), y.data_ptr(), None if few else lists.data_ptr(), act.data_ptr(),
           None if few else parts.data_ptr(), t, hidden, experts, top, ff, shared, int(bool(gated)), weights.data_ptr(),
           weights.shape[1], experts if shared_weight else -1)
    return y


register_kernel(KernelOp("moe_f32", moe_f32_plain, "holon_moe_f32",
                         [_P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _I, _P, _I, _I], _moe_f32_hip))


@register_part("ffn", "polynorm")
class PolyNormFFN(Part):
    """down(act(up(x))) with act = a N(z) + b N(z^2) + c N(z^3) + e (`act` holds a, b, c, e; N divides a token's
    vector by its root mean square, `eps` inside the root)."""

    graph_safe = True

    def __init__(self, build: Build, *, inter: int, eps: float, hidden: int, layer: int) -> None:
        super().__init__(build)
        self.inter, self.hidden, self.eps = inter, hidden, float(eps)
        self.attach("up_proj", Linear(build, inp=hidden, out=inter))
        self.attach("down_proj", Linear(build, inp=inter, out=hidden))
        self.declare("act", (4,), kind=FLOAT32, init="unit")

    def products(self, x: torch.Tensor, step=None):
        few = together(x, self.down_proj)
        up = (yield [Product(self.up_proj, x)])[0] if few else self.up_proj(x)
        y = self.kernels.polynorm(up, self.act, self.eps)
        return (yield [Product(self.down_proj, y)])[0] if few else self.down_proj(y)

    def forward(self, x: torch.Tensor, step=None) -> torch.Tensor:
        return by_itself(self.kernels, self.products(x, step))

    __call__ = forward


@register_part("ffn", "dense")
class DenseFFN(Part):
    """down(act(up(x))) with an activation by name: `relu2`, the square of max(z, 0)."""

    graph_safe = True
    ACTS = ("relu2",)

    def __init__(self, build: Build, *, inter: int, hidden: int, layer: int, act: str = "relu2") -> None:
        super().__init__(build)
        if act not in self.ACTS:
            raise ValueError(f"ffn dense: no activation {act!r} ({', '.join(self.ACTS)})")
        self.inter, self.hidden, self.act = inter, hidden, act
        self.attach("up_proj", Linear(build, inp=hidden, out=inter))
        self.attach("down_proj", Linear(build, inp=inter, out=hidden))

    def products(self, x: torch.Tensor, step=None):
        few = together(x, self.down_proj)
        up = Product(self.up_proj, x, relu2=True)
        y = (yield [up])[0] if few else up.alone()
        return (yield [Product(self.down_proj, y)])[0] if few else self.down_proj(y)

    def forward(self, x: torch.Tensor, step=None) -> torch.Tensor:
        return by_itself(self.kernels, self.products(x, step))

    __call__ = forward


@register_part("ffn", "moe")
class MoE(Part):
    """A mixture of experts with a router, and an optional shared expert that every token uses. The experts are SiLU-gated,
    or (`act` "relu2") W_down max(W_up x, 0)^2.

    `score` "softmax_top" is the other router: float32 logits z = W_r x + b (`router_bias`), the `top` largest z are
    chosen and weighted by the softmax over the chosen z alone (no scale); with `groups` only among the `keep` groups
    whose largest z are best. (A softmax over all experts whose chosen scores are then divided by their sum gives the
    same weights: the largest score is always among the chosen, so their sum is never near zero.) `shared_gated`: the shared
    expert's output is multiplied by sigmoid(w_sg . x), one number a token; w_sg rides as one more row of the router's
    weights, so the router's kernel leaves that weight too. `score` "sigmoid_top" is the same choice with each chosen
    expert's own sigmoid(z) as its weight. `weigh_input`: the weight multiplies an expert's input, not its output; for the
    squared ReLU that is its square on the output, W_down max(W_up w x, 0)^2 = w^2 W_down max(W_up x, 0)^2 for w > 0, and
    the router's kernel squares it. What follows describes `score` "sigmoid".

    Router: float32 logits (products of the input as it is with float32 weights, summed in float32), scores s =
    sigmoid(logits); experts are chosen by s + `correction` (`bias`), optionally
    only within the `keep` best of `groups` groups of neighbouring experts, `top` per token; a chosen expert's output
    is weighted by s * `scale`. All experts' gate and up projections are one product and all down projections
    another: the activations of experts a token did not choose are set to 0 in between (`moe_gate`), so the second
    product adds up exactly the chosen experts' weighted outputs, and the shared expert's columns ride in the same two
    products. Steps of few rows take the same two products over the chosen experts' columns alone (`moe_up_few`, `moe_down_few`), steps of many
    rows each expert's over the rows that chose it (`moe_rows`), where that is done sooner; in float32 every step does the latter
    (`moe_f32`) or none, by the mixture's sizes. Steps of as many rows launch the same kernels whatever was chosen."""

    graph_safe = True

    def __init__(self, build: Build, *, experts: int, top: int, inter: int, hidden: int, layer: int,
                 scale: float = 1.0, groups: int = 1, keep: int = 1, bias: bool = True, shared: int = 0,
                 score: str = "sigmoid", shared_gated: bool = False, act: str = "silu", weigh_input: bool = False) -> None:
        super().__init__(build)
        if not 1 <= top <= experts:
            raise ValueError(f"moe: top {top} of {experts} experts")
        if score not in ("sigmoid", "softmax_top", "sigmoid_top"):
            raise ValueError(f"moe: no router score {score!r} (sigmoid, softmax_top, sigmoid_top)")
        if score != "sigmoid" and float(scale) != 1.0:
            raise ValueError("moe: the router that chooses by its logits comes without a scale")
        if shared_gated and (not shared or score == "sigmoid"):
            raise ValueError("moe: a gate on the shared expert needs a shared expert and a router that chooses by its logits")
        if act not in ("silu", "relu2"):
            raise ValueError(f"moe: no expert activation {act!r} (silu, relu2)")
        if weigh_input and (act != "relu2" or score != "sigmoid_top"):
            raise ValueError("moe: weights on the experts' inputs come with the squared ReLU and the sigmoid_top router")
        self.act, self.weigh_input = act, bool(weigh_input)
        self.score, self.shared_gated = score, bool(shared_gated)
        if groups > 1 and (experts % groups or not 1 <= keep <= groups or top > keep * (experts // groups)):
            raise ValueError(f"moe: {experts} experts in {groups} groups, {keep} kept, top {top}")
        self.experts, self.top, self.inter, self.hidden, self.shared = experts, top, inter, hidden, int(shared)
        self.scale, self.groups, self.keep = float(scale), int(groups), int(keep)
        self.declare("router", (experts, hidden), kind=FLOAT32)
        self.has_bias = bool(bias)
        if self.has_bias:
            # (sigmoid: a correction of the choice alone; softmax_top: the logits' bias)
            self.declare("correction" if score == "sigmoid" else "router_bias", (experts,), kind=FLOAT32, init="zero")
        if self.shared_gated:
            self.declare("shared_sg", (1, hidden), kind=FLOAT32)
        if act == "silu":
            self.declare("gate", (experts, inter, hidden))
        self.declare("up", (experts, inter, hidden))
        self.declare("down", (experts, hidden, inter))
        if self.shared:
            if act == "silu":
                self.declare("shared_gate", (self.shared, hidden))
            self.declare("shared_up", (self.shared, hidden))
            self.declare("shared_down", (hidden, self.shared))
        self.gate_up: Linear | None = None
        self.all_down: Linear | None = None

    def finalize(self) -> None:
        if self.up is None:
            return
        if self.shared_gated and self.router.shape[0] == self.experts:
            self.router = torch.cat((self.router, self.shared_sg)).contiguous()
            del self._decls["shared_sg"]
            self.shared_sg = None
        e, f, w = self.experts, self.inter, self.hidden
        cols = e * f + self.shared
        gated = self.act == "silu"
        gate_up, down = Linear(self.build, inp=w, out=(2 if gated else 1) * cols), Linear(self.build, inp=cols, out=w)
        gates, ups = [self.gate.reshape(e * f, w)] if gated else [], [self.up.reshape(e * f, w)]
        downs = [self.down.permute(1, 0, 2).reshape(w, e * f)]
        if self.shared:
            if gated:
                gates.append(self.shared_gate)
            ups.append(self.shared_up)
            downs.append(self.shared_down)
        gate_up.weight = torch.cat(gates + ups, dim=0).contiguous()
        down.weight = torch.cat(downs, dim=1).contiguous()
        for name in ("gate", "up", "down", "shared_gate", "shared_up", "shared_down"):
            if name in self._decls:
                del self._decls[name]
                setattr(self, name, None)
        gate_up.finalize()
        down.finalize()
        self.gate_up = self.attach("gate_up", gate_up)
        self.all_down = self.attach("all_down", down)

    def products(self, x: torch.Tensor, step=None):
        k = self.kernels
        if self.score != "sigmoid":
            score = "softmax" if self.score == "softmax_top" else "sigmoid_squared" if self.weigh_input else "sigmoid"
            route = Routing(k, x, self.router, self.router_bias if self.has_bias else None, self.experts, self.top, self.groups, self.keep,
                            score)
        else:
            route = Routing(k, x, self.router, self.correction if self.has_bias else None, self.experts, self.top, self.groups, self.keep,
                            scale=self.scale)
        weights = (yield [route])[0] if together(x) else route.alone()
        up, down = self.gate_up, self.all_down
        if x.dtype == torch.float32 and moe_f32_takes(x.shape[1], self.experts, self.inter, self.shared, self.act == "silu", self.top):
            y = k.moe_f32(x, weights, up.weight, down.weight, self.experts, self.top, self.inter, self.shared, self.act == "silu",
                          shared_weight=self.shared_gated)
            if y is not None:
                return y
        if moe_few_pays(x.shape[0], x.shape[1], self.experts, self.inter, self.act == "silu", self.top):
            act = k.moe_up_few(x, weights, up.tiled, down.tiled, self.experts, self.inter, self.shared, self.act == "silu",
                               shared_weight=self.shared_gated)
            if act is not None:
                rest = ExpertsDown(k, act, weights, down.tiled, self.experts, self.inter, self.shared)
                return (yield [rest])[0] if together(x) else rest.alone()
        if moe_rows_pays(x.shape[0], x.shape[1], self.experts, self.inter, self.shared, self.act == "silu", self.top) \
                and self._own_rows(x.shape[0]):
            y = k.moe_rows(x, weights, up.weight, down.weight, self.experts, self.top, self.inter, self.shared, self.act == "silu",
                           shared_weight=self.shared_gated)
            if y is not None:
                return y
        between = k.moe_relu2 if self.act == "relu2" else k.moe_gate
        return down(between(up(x), weights, self.inter, self.shared, shared_weight=self.shared_gated))

    def forward(self, x: torch.Tensor, step=None) -> torch.Tensor:
        return by_itself(self.kernels, self.products(x, step))

    def _own_rows(self, rows: int) -> bool:
        """Whether the engine's product choices leave a step of many rows to `moe_rows`: pins of either product over all experts keep
        those, and so does mode `vendor`."""
        choice = getattr(self.kernels, "product_choice", None)       # (a kernel set with one form a product has nothing to choose)
        if choice is None:
            return True
        shapes = [tuple(w.weight.shape) for w in (self.gate_up, self.all_down)]
        return choice("experts", self.gate_up.weight, rows, yields=[(kind, s) for kind in ("rows", "vendor") for s in shapes],
                      by_rule=True) == "own"

    __call__ = forward
