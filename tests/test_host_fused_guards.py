"""What the fused host paths must not pass by: hooks and replaced parts of a module, second derivatives, forward mode."""
import pytest
import torch
import torch.nn as nn

from memorax_amd import sequence_models as sm
from memorax_amd.dense import Dense, dense


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
