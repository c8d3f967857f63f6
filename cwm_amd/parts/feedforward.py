"""Dense feed-forwards: gated, and with a plain activation between two products."""

from __future__ import annotations

from typing import Any, Dict, Mapping, Optional

import torch

from .. import ops
from .base import FeedForward, Runtime, TensorSpec, register_part
from .linear import LinearWeights


class SwiGLU(FeedForward):
    """w2(silu(w1 x) * (w3 x)), no biases (cwm/fastgen/forward.py:776-782;
    cwm/model/transformer.py:214-228).  w1 and w3 are joined into one product; the
    gate's SiLU and the product with the up branch are computed in float32 and
    rounded once."""

    replayable = True

    def __init__(self, dim: int, hidden_dim: int) -> None:
        self.dim = dim
        self.hidden_dim = hidden_dim

    def tensor_specs(self) -> Dict[str, TensorSpec]:
        return {
            "w1.weight": TensorSpec((self.hidden_dim, self.dim)),
            "w2.weight": TensorSpec((self.dim, self.hidden_dim)),
            "w3.weight": TensorSpec((self.hidden_dim, self.dim)),
        }

    def bind(self, tensors: Mapping[str, torch.Tensor], runtime: Runtime) -> None:
        super().bind(tensors, runtime)
        # gate and up rows alternate in groups of 8 where the width allows, so that a decode batch
        # finishes silu(gate) * up in the product's epilogue
        self.grouped = self.hidden_dim % 8 == 0
        self.gate_up = LinearWeights.joined(
            [tensors["w1.weight"], tensors["w3.weight"]], [None, None], group=8 if self.grouped else None,
            stream_copy=runtime.stream_copies,
        )
        self.down = LinearWeights(tensors["w2.weight"], stream_copy=runtime.stream_copies)

    def forward(self, x: torch.Tensor, batch: Any) -> torch.Tensor:
        # the result (or partial sums of it) is added into the residual by the next norm.  (Forming
        # silu(gate) * up inside the down product was tried: every block recomputes it, which costs
        # more than the kernel it saves.)
        hidden = ops.gate_up_silu(x, self.gate_up.weight, self.gate_up.bias, self.grouped, streamed=self.gate_up.streamed)
        return self.down(hidden, partials_ok=True)


register_part("feed_forward", "swiglu", SwiGLU)


class ActivatedMLP(FeedForward):
    """W_down act(W_up x), no gate and no biases; `activation` is one of `ops.ACTIVATIONS` ("relu2": the square of
    relu).  The activation is computed in float32 on the product's sums (rounded before as `GatedMLP` says) and
    rounded once.  `up` and `down` are the tensors' local names."""

    replayable = True

    def __init__(self, dim: int, hidden_dim: int, activation: str = "relu2", up: str = "up", down: str = "down") -> None:
        if activation not in ops.ACTIVATIONS:
            raise ValueError(f"activation {activation!r}: known are {', '.join(ops.ACTIVATIONS)}")
        self.dim, self.hidden_dim, self.activation = dim, hidden_dim, activation
        self.up_name, self.down_name = up, down

    def tensor_specs(self) -> Dict[str, TensorSpec]:
        return {self.up_name: TensorSpec((self.hidden_dim, self.dim)), self.down_name: TensorSpec((self.dim, self.hidden_dim))}

    def bind(self, tensors: Mapping[str, torch.Tensor], runtime: Runtime) -> None:
        super().bind(tensors, runtime)
        self.up = LinearWeights(tensors[self.up_name], stream_copy=runtime.stream_copies)
        self.down = LinearWeights(tensors[self.down_name], stream_copy=runtime.stream_copies)

    def forward(self, x: torch.Tensor, batch: Any) -> torch.Tensor:
        hidden = ops.act_rows(self.up(x, partials_ok=True), self.activation, x.dtype)
        return self.down(hidden, partials_ok=True)


register_part("feed_forward", "activated_mlp", ActivatedMLP)


class GatedMLP(FeedForward):
    """W_down act(W_gate x, W_up x), no biases, with the gated activation as an argument (`ops.GatedActivation`):
    "silu": silu(g) * u;  "clamped_swish": g' * sigmoid(act_alpha * g') * (u' + 1) with g' = min(g, act_limit) and
    u' = clamp(u, -act_limit, act_limit);  "gelu_tanh": gelu(g) * u, the tanh form.  With `row_gate` (a tensor's local name, [1, dim]) the whole result is
    multiplied by sigmoid(w . x), one number a token: the gate's row rides as one more output of the joined gate/up
    product and scales the activation's rows, which the linear down product carries through.  The activation is
    computed in float32 on the product's sums and rounded once (sums that one block finishes are rounded before, to the
    activations' type, for up to 8 rows, in the tiled kernel and where that does not take the sizes, and so are the library's).  `gate`, `up`, `down`: the tensors' local names."""

    replayable = True

    def __init__(
        self, dim: int, hidden_dim: int, activation: str = "silu", act_alpha: float = 1.0, act_limit: float = 0.0,
        row_gate: Optional[str] = None, gate: str = "gate", up: str = "up", down: str = "down",
    ) -> None:
        self.dim, self.hidden_dim = dim, hidden_dim
        self.activation = ops.GatedActivation(activation, float(act_alpha), float(act_limit))
        self.activation.code()  # an unknown kind is refused here
        self.row_gate, self.gate_name, self.up_name, self.down_name = row_gate, gate, up, down

    def tensor_specs(self) -> Dict[str, TensorSpec]:
        specs = {
            self.gate_name: TensorSpec((self.hidden_dim, self.dim)),
            self.up_name: TensorSpec((self.hidden_dim, self.dim)),
            self.down_name: TensorSpec((self.dim, self.hidden_dim)),
        }
        if self.row_gate is not None:
            specs[self.row_gate] = TensorSpec((1, self.dim))
        return specs

    def bind(self, tensors: Mapping[str, torch.Tensor], runtime: Runtime) -> None:
        super().bind(tensors, runtime)
        matrices = [tensors[self.gate_name], tensors[self.up_name]]
        if self.row_gate is not None:
            # with zeros up to whole groups of 16 rows, which the wide product takes and no other number of columns (2,049 columns of
            # 2,048 at 1,500 rows: the library 23.2 us, 2,064 columns 19.0)
            row = tensors[self.row_gate]
            matrices += [row, row.new_zeros((-(2 * self.hidden_dim + 1) % 16, self.dim))]
        self.gate_up = self.gate_up_wide = LinearWeights.joined(matrices, [None] * len(matrices), stream_copy=runtime.stream_copies)
        if self.row_gate is not None:
            # Up to as many rows as the streaming product takes, the columns there are: the tiled product would take 2,064, in more time than that
            # one 2,049 (us, 2,049 / 2,064 columns without a copy: 16 rows 9.1 / 11.1; 513 / 528 of 512: 33 rows 7.4 / 10.6).  Of 65 to 256 rows
            # the library takes 2,049, in 3 to 5 us less than the tiled product 2,064, but its call costs the host 20 us more: a step of
            # four layers and 128 rows 1,548 us with 2,049 columns, 1,505 with 2,064.
            streamed = self.gate_up.streamed
            self.gate_up = self.gate_up.rows(0, 2 * self.hidden_dim + 1)
            self.gate_up.streamed = streamed  # its tiles of 16 rows end in the same zeros
        self.down = LinearWeights(tensors[self.down_name], stream_copy=runtime.stream_copies)

    def forward(self, x: torch.Tensor, batch: Any) -> torch.Tensor:
        joined = (self.gate_up if x.shape[0] <= ops.STREAM_MAX_ROWS else self.gate_up_wide)(x, partials_ok=True)
        hidden = ops.gated_act_rows(joined, self.hidden_dim, self.activation, x.dtype, 2 * self.hidden_dim if self.row_gate is not None else None)
        return self.down(hidden, partials_ok=True)


register_part("feed_forward", "gated_mlp", GatedMLP)
