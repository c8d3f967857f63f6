"""Which routers of a decode step are served by one launch: those for which it was measured to be faster."""

from __future__ import annotations

import pytest

from cwm_amd import ops


@pytest.mark.parametrize("experts,k,pays", [
    (1, 32, True), (8, 4096, True), (16, 1024, True), (16, 2048, True), (16, 4096, True), (16, 4128, False), (16, 8192, False), (8, 8192, False),
    (17, 1024, False), (32, 2048, False), (32, 3072, False), (64, 2048, False), (64, 8192, False), (16, 2056, False),
])
def test_one_launch_where_it_pays(experts, k, pays):
    assert ops.route_group_pays(experts, k) == pays


@pytest.mark.parametrize("tokens,k,pays", [(17, 4096, True), (4096, 2048, True), (4097, 2048, False), (8192, 1024, True), (8192, 1536, True), (8193, 1024, False), (65536, 3072, False)])
def test_many_tokens_of_long_rows_stay_a_product(tokens, k, pays):
    assert ops.route_rows_pays(tokens, k) == pays


@pytest.mark.gpu
@pytest.mark.parametrize("experts,pays", [(16, True), (32, False)])
def test_a_layer_asks_the_rule(experts, pays):
    """Routed experts of either size: a step of few tokens gives the rows that each expert's weights make of the chosen tokens."""
    import torch

    from cwm_amd.parts.base import Runtime
    from cwm_amd.parts.experts import RoutedExperts

    dim, hidden, top, dev = 256, 128, 3, torch.device("cuda:0")
    part = RoutedExperts(dim=dim, hidden_dim=hidden, n_experts=experts, top=top)
    g = torch.Generator(device=dev).manual_seed(experts)
    tensors = {name: (torch.randn([abs(n) for n in spec.shape], generator=g, device=dev) * abs(spec.shape[-1]) ** -0.5).bfloat16() for name, spec in part.tensor_specs().items()}
    part.bind(tensors, Runtime(device=dev, act_dtype=torch.bfloat16, stream_copies=False))
    assert (part.router_copy is not None) == pays
    x = torch.randn((9, dim), generator=g, device=dev).bfloat16()
    got = part.forward(x, None).double()
    router = next(t for t in tensors.values() if tuple(t.shape) == (experts, dim))
    logits = x.double() @ router.double().T
    best, chosen = logits.topk(top, -1)
    for t in range(9):
        want = torch.zeros(dim, dtype=torch.float64, device=dev)
        for weight, e in zip(torch.softmax(best[t], -1), chosen[t].tolist()):
            gate, up, down = (tensors[f"e{e}.{n}"].double() for n in ("gate", "up", "down"))
            want += weight * (down @ (torch.nn.functional.silu(gate @ x[t].double()) * (up @ x[t].double())))
        # the hidden row is rounded to bfloat16: 2^-8 of each of its `hidden` values, through weights of size hidden^-0.5
        assert float((got[t] - want).abs().max()) <= 2.0 ** -6 * float(want.abs().max())
