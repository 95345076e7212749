"""Dense SwiGLU feed-forward: down(silu(gate(x)) * up(x)) (clockwork/engine/model.py:52-63).

gate and up are one product over a fused [2 I, H] weight; the gate multiply is one kernel.
"""

from __future__ import annotations

import torch

from clockwork_amd import ops
from clockwork_amd.config.spec import ParamSpec
from clockwork_amd.parts.base import Part, own_method
from clockwork_amd.parts.specs import SwiGLUSpec


class SwiGLU(Part):
    graph_safe = True

    def __init__(self, spec: SwiGLUSpec) -> None:
        self.spec = spec

    @property
    def by_rows(self) -> bool:
        """A row of the output depends on that row of the input and on nothing else of the step."""
        return own_method(self, SwiGLU)

    def param_specs(self):
        H, I = self.spec.hidden_size, self.spec.intermediate_size
        return {"gate_up_weight": ParamSpec((2 * I, H)), "down_weight": ParamSpec((H, I))}

    def bind(self, params, device, dtype) -> None:
        self.gate_up = params["gate_up_weight"]
        self.down = params["down_weight"]

    def fuses_input_norm(self, n_tokens: int, dtype, delta) -> bool:
        """True if ``forward`` can take an ``ops.LazyAddNorm`` of that many rows and make the
        norm inside the gate/up product (decode: few rows)."""
        H, I = self.spec.hidden_size, self.spec.intermediate_size
        return ops.swiglu_norm_fusable(n_tokens, 2 * I, H, dtype, self.gate_up, delta)

    def takes_begun_norm(self, n_tokens: int) -> bool:
        """May ``forward``'s input be an ``ops.BegunNorm`` of that many rows?"""
        return own_method(self, SwiGLU) and ops.swiglu_begun_ok(n_tokens, self.gate_up)

    def joins_stream(self, n_tokens: int, norm) -> bool:
        """Does ``forward_joined`` add that many rows to the stream and begin ``norm``?"""
        return own_method(self, SwiGLU) and ops.linear_join_pays(n_tokens, self.down, norm.weight)

    def forward_joined(self, x, ctx, resid, norm) -> "ops.BegunNorm":
        """``forward``, its output added to ``resid`` and ``norm`` of that begun."""
        inner = ops.linear_swiglu(x, self.gate_up, policy=getattr(ctx, "products", None))
        return ops.linear_join(inner, self.down, resid, norm.weight, norm.spec.eps)

    def forward(self, x, ctx) -> torch.Tensor:
        policy = getattr(ctx, "products", None)
        return ops.linear(ops.linear_swiglu(x, self.gate_up, policy=policy), self.down, partial_ok=True, policy=policy,
                          portions_partial_ok=getattr(ctx, "reader_adds_sums", False))


class GatedMLP(Part):
    """down(act(gate(x)) * up(x)) with the activation the spec names ("silu", "relu" or "gelu_tanh"), through the
    kernels of :class:`SwiGLU`."""

    graph_safe = True
    partial_ok = False   # may the output come as ``ops.PartialSums``? A block whose next norm adds them up sets it

    def __init__(self, spec) -> None:
        self.spec = spec

    @property
    def by_rows(self) -> bool:
        return own_method(self, GatedMLP)

    def param_specs(self):
        H, I = self.spec.hidden_size, self.spec.intermediate_size
        return {"gate_up_weight": ParamSpec((2 * I, H)), "down_weight": ParamSpec((H, I))}

    def kernel_libraries(self) -> list:
        return [("rowwise", None)] if self.spec.activation == "gelu_tanh" else []

    def bind(self, params, device, dtype) -> None:
        self.gate_up = params["gate_up_weight"]
        self.down = params["down_weight"]

    def forward(self, x, ctx) -> torch.Tensor:
        policy = getattr(ctx, "products", None)
        act = {"relu": ops.RELU_GATE, "gelu_tanh": ops.GELU_GATE}.get(self.spec.activation, 0.0)
        inner = ops.linear_swiglu(x, self.gate_up, policy=policy, limit=act)
        return ops.linear(inner, self.down, partial_ok=self.partial_ok, policy=policy, portions_partial_ok=self.partial_ok)


class DenseMLP(Part):
    """down(act(up(x))) (``DenseMLPSpec``). "gelu": the up product with the erf GELU (float32
    inside) in its epilogue for few rows, as a kernel of its own behind the product otherwise;
    "gelu_tanh": its tanh form, in the epilogue for long portions as well;
    "relu2": max(z, 0)^2 on the float32 sums in the epilogue of the up product for few rows
    (the weight-streaming kernel) and for long portions (the wide-tile kernel), in place behind
    the product otherwise; the down product."""

    graph_safe = True

    def __init__(self, spec) -> None:
        self.spec = spec

    def param_specs(self):
        H, I = self.spec.hidden_size, self.spec.intermediate_size
        return {"up_weight": ParamSpec((I, H)), "down_weight": ParamSpec((H, I))}

    def kernel_libraries(self) -> list:
        return [("rowwise", None)]

    def bind(self, params, device, dtype) -> None:
        self.up = params["up_weight"]
        self.down = params["down_weight"]

    def forward(self, x, ctx) -> torch.Tensor:
        policy = getattr(ctx, "products", None)
        if self.spec.activation == "relu2":
            return ops.linear(ops.linear_relu_squared(x, self.up, policy=policy), self.down, policy=policy)
        form = "tanh" if self.spec.activation == "gelu_tanh" else "erf"
        return ops.linear(ops.linear_gelu(x, self.up, policy=policy, form=form), self.down, policy=policy)
