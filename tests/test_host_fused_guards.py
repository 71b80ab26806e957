"""What the fused host paths must not pass by: hooks and replaced parts of a module, second derivatives, forward mode, functorch."""
import threading

import pytest
import torch
import torch.nn as nn

from memorax_amd import functional as Fn
from memorax_amd import sequence_models as sm
from memorax_amd._lib import native
from memorax_amd.dense import Dense, dense, dense_group


def test_gradients_refuse_a_second_derivative():
    x, w = torch.randn(4, 8, requires_grad=True), torch.randn(3, 8, requires_grad=True)
    (g,) = torch.autograd.grad((dense(x, w) ** 2).sum(), x, create_graph=True)
    with pytest.raises(RuntimeError, match="differentiable once"):
        g.sum().backward()


def test_a_tangent_is_refused():
    x, w = torch.randn(4, 8), torch.randn(3, 8)
    with torch.autograd.forward_ad.dual_level():
        with pytest.raises(NotImplementedError, match="forward-mode"):
            dense(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)), w)


@pytest.mark.parametrize("at", ["weight", "bias", "second weight"])
def test_a_parameter_s_tangent_is_refused_beside_an_input_that_requires_gradients(at):
    dual = lambda t: torch.autograd.forward_ad.make_dual(t, torch.ones_like(t))  # noqa: E731
    x, w, v, b = torch.randn(4, 8, requires_grad=True), torch.randn(3, 8), torch.randn(3, 8), torch.randn(3)
    with torch.autograd.forward_ad.dual_level():
        w, v, b = dual(w) if at == "weight" else w, dual(v) if at == "second weight" else v, dual(b) if at == "bias" else b
        with pytest.raises(NotImplementedError, match="forward-mode"):
            native().dense_group(x, [w, v], [b, None])


def _acting():
    """The acting entries, with the argument that carries a tangent handed in (named as in the entry)."""
    N, done, ones = 8, torch.zeros(4, 1), torch.ones
    x, state = ones(4, 1, N), ones(4, 1, N, dtype=torch.complex64)
    lru = [ones(N), ones(N), ones(N), ones(N, N), ones(N, N), ones(N, N), ones(N, N), ones(N)]
    mlstm = [ones(2 * N, N), ones(N, 1, 4), ones(N), *[ones(2, 4, 4)] * 3, *[ones(2, 3 * N), ones(2)] * 2, ones(2, 4), ones(N), ones(N, N)]
    carry = [ones(4, 1, 2, 4, 4), ones(4, 1, 2, 1, 1), ones(4, 1, 2, 4, 1), ones(4, 1, 2, 1, 1)]
    put = lambda lst, i, t: [*lst[:i], t, *lst[i + 1:]]  # noqa: E731
    return {
        "row_dense x": (x, lambda t: native().row_dense(t, 0, None, None, 0.0, False, [ones(N, N)], [None], torch.float32, torch.float32, None)),
        "row_dense scale": (ones(N), lambda t: native().row_dense(x, 1, t, None, 0.0, False, [ones(N, N)], [None], torch.float32, torch.float32, None)),
        "row_dense weight": (ones(N, N), lambda t: native().row_dense(x, 0, None, None, 0.0, False, [ones(N, N), t], [None, None], torch.float32,
                                                                      torch.float32, None)),
        "row_dense bias": (ones(N), lambda t: native().row_dense(x, 0, None, None, 0.0, False, [ones(N, N)], [t], torch.float32, torch.float32, None)),
        "row_dense residual": (x, lambda t: native().row_dense(x, 0, None, None, 0.0, False, [ones(N, N)], [None], torch.float32, torch.float32, t)),
        "lru_act x": (x, lambda t: native().lru_act(t, 0, None, None, 0.0, lru, done, state, state)),
        "lru_act parameter": (ones(N), lambda t: native().lru_act(x, 0, None, None, 0.0, put(lru, 1, t), done, state, state)),
        "lru_act carry": (state, lambda t: native().lru_act(x, 0, None, None, 0.0, lru, done, state, t)),
        "mlstm_act x": (x, lambda t: native().mlstm_act(t, 0, None, None, 0.0, mlstm, done, carry, -60.0)),
        "mlstm_act parameter": (ones(2, 4, 4), lambda t: native().mlstm_act(x, 0, None, None, 0.0, put(mlstm, 4, t), done, carry, -60.0)),
        "mlstm_act carry": (carry[2], lambda t: native().mlstm_act(x, 0, None, None, 0.0, mlstm, done, put(carry, 2, t), -60.0)),
        "mingru_step z": (x, lambda t: native().mingru_step(t, x, None, done, x, x, False)),
        "mingru_step gate": (x, lambda t: native().mingru_step(x, x, t, done, x, x, False)),
        "mingru_step carry": (x, lambda t: native().mingru_step(x, x, None, done, x, t, False)),
    }


@pytest.mark.parametrize("name", sorted(_acting()))
def test_acting_refuses_a_tangent(name):
    """Switching gradients off leaves tangents on: the acting entries, which run without gradients, look for them."""
    t, call = _acting()[name]
    with torch.no_grad(), torch.autograd.forward_ad.dual_level():
        with pytest.raises(NotImplementedError, match="forward-mode"):
            call(torch.autograd.forward_ad.make_dual(t, torch.ones_like(t)))


@pytest.mark.parametrize("kind", ["forward", "pre", "backward", "backward_pre"])
def test_hooks_are_seen_at_any_depth(kind):
    block = sm.PreNorm(sm.Memoroid(sm.LRUCell(8, 8)), 8)
    assert not sm._hooked(block)
    m = block.module.cell
    handle = {"forward": m.register_forward_hook, "pre": m.register_forward_pre_hook, "backward": m.register_full_backward_hook,
              "backward_pre": m.register_full_backward_pre_hook}[kind](lambda *a: None)
    assert sm._hooked(block)
    handle.remove()
    assert not sm._hooked(block)
    handle = nn.modules.module.register_module_forward_hook(lambda *a: None)
    assert sm._hooked(block)
    handle.remove()


@pytest.mark.parametrize("part,method", [("", "forward"), ("module", "forward"), ("norm", "forward"), ("module.cell", "forward"), ("module.cell", "scan"),
                                         ("module.cell", "read"), ("module.cell.output_projection", "forward")])
def test_a_method_set_on_an_instance_is_seen_at_any_depth(part, method):
    block = sm.PreNorm(sm.Memoroid(sm.LinearAttentionCell(8, 4, 2)), 8)
    assert not sm._hooked(block)
    m = block.get_submodule(part)
    setattr(m, method, getattr(m, method))
    assert sm._hooked(block)
    delattr(m, method)
    assert not sm._hooked(block)


def test_a_replaced_part_is_no_row_layer():
    class Wrapped(Dense):
        def forward(self, x):
            return 2 * super().forward(x)

    x = torch.randn(4, 1, 8)
    assert sm._row_layers(x, [Dense(8, 8), nn.Linear(8, 8)])
    assert not sm._row_layers(x, [Dense(8, 8), Wrapped(8, 8)])
    cell = sm.mLSTMCell(8, hidden_dim=32, num_heads=2)
    assert cell._parts_as_written()
    cell.up_projection = Dense(8, 64)
    assert not cell._parts_as_written()


@pytest.mark.parametrize("bias", [False, True])
def test_a_mapped_dense_layer_keeps_its_gradients(bias):
    """As torch.nn.functional.linear: the mapped input, the parameters closed over, and a second path through them."""
    lin, x = nn.Linear(8, 3, bias=bias).double(), torch.randn(5, 4, 8, dtype=torch.float64, requires_grad=True)
    params = [x, *lin.parameters()]

    def loss(layer):
        return (torch.vmap(layer)(x) ** 2).sum() + (lin.weight ** 3).sum()

    got = torch.autograd.grad(loss(lambda t: dense(t, lin.weight, lin.bias)), params)
    grouped = torch.autograd.grad(loss(lambda t: dense_group(t, [lin, lin])[1]), params)
    for g, h, want in zip(got, grouped, torch.autograd.grad(loss(lin), params)):
        torch.testing.assert_close(g, want, rtol=1e-12, atol=1e-12)
        torch.testing.assert_close(h, want, rtol=1e-12, atol=1e-12)
    f = lambda layer: torch.func.grad(lambda w: layer(x.detach()[0], w).pow(2).sum())(lin.weight.detach())  # noqa: E731
    torch.testing.assert_close(f(dense), f(nn.functional.linear), rtol=1e-12, atol=1e-12)


def _operators():
    """Every operator that records a node, of one tensor that all its floating arguments are made of."""
    done, s = torch.zeros(2, 3), torch.ones(4)
    heads = lambda t: t.view(2, 3, 1, 4)  # noqa: E731
    return {
        "linear_scan": lambda t: Fn.linear_scan(t, t, done),
        "mingru_scan": lambda t: Fn.mingru_scan(t, t, done),
        "linear_attention": lambda t: native().linear_attention(heads(t), heads(t), heads(t), done, None, 0, False),
        "normalised": lambda t: native().normalised_linear_attention(heads(t), heads(t), heads(t), done, None, None, 0, 1e-6, False, False),
        "gated": lambda t: native().gated_linear_attention(heads(t), heads(t), heads(t), t[..., :1], done, None, 0, False),
        "delta_rule": lambda t: native().delta_rule(heads(t), heads(t), heads(t), t[..., :1], done, None, False, 0, False),
        "mlstm_gates": lambda t: Fn.mlstm_gates(t, t, done),
        "rms_norm": lambda t: Fn.rms_norm(t, s),
        "layer_norm": lambda t: Fn.layer_norm_fork(t, s, s)[1],
        "silu_gate": lambda t: Fn.silu_gate(t, t),
        "mamba_mix": lambda t: native().mamba_mix(t, t, t, t[..., :1], torch.ones(10, 1, 4), torch.ones(10), s[:1], s[:1], s[:1], s[:2], done,
                                                  torch.zeros(2, 1, 2, 4), torch.ones(2, 1), 1e-6, False),
    }


@pytest.mark.parametrize("name", sorted(_operators()))
def test_functorch_is_refused_by_name(name):
    f = _operators()[name]
    with pytest.raises(RuntimeError, match="functorch"):
        torch.vmap(f)(torch.randn(5, 2, 3, 4))


def test_stepping_in_place_is_a_thread_s_own():
    """A thread that captures a step in place leaves the carries of the others' steps alone."""
    seen = {}
    with Fn.step_in_place():
        t = threading.Thread(target=lambda: seen.update(other=Fn.stepping_in_place()))
        t.start()
        t.join()
        seen["own"] = Fn.stepping_in_place()
    assert seen == {"other": False, "own": True} and not Fn.stepping_in_place()
