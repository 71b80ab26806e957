"""torch.jit.trace: blocks that are compositions of array operations give graphs that compute with other inputs too; the recurrences
refuse instead of leaving their results in the graph as constants."""
import pytest
import torch

from memorax_amd import functional as Fn
from memorax_amd import sequence_models as sm

pytestmark = pytest.mark.gpu


class _Output(torch.nn.Module):
    def __init__(self, block):
        super().__init__()
        self.block = block

    def forward(self, *args):
        return self.block(*args)[1]


BLOCKS = {"ffn": lambda: sm.FFN(64), "glu": lambda: sm.GLU(64), "rms block": lambda: sm.Residual(sm.PreNorm(sm.FFN(64), 64, norm=sm.RMSNorm)),
          "layer block": lambda: sm.Residual(sm.PreNorm(sm.Projection(64, 64), 64)), "post": lambda: sm.PostNorm(sm.FFN(64), 64)}


@pytest.mark.parametrize("autocast", [False, True])
@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("name", sorted(BLOCKS))
def test_stateless_blocks_trace(name, grad, autocast):
    torch.manual_seed(0)
    block = _Output(BLOCKS[name]()).cuda()
    make = lambda: torch.randn(3, 5, 64, device="cuda", requires_grad=grad)  # noqa: E731
    with torch.set_grad_enabled(grad), torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast, cache_enabled=False):
        traced = torch.jit.trace(block, (make(),), check_trace=False)
        x = make()
        got, want = traced(x), block(x)
    assert got.dtype == want.dtype and got.requires_grad == want.requires_grad
    # the composition against the kernels: float32 sums of 256 terms, or bfloat16 roundings
    torch.testing.assert_close(got, want, rtol=0, atol=(2e-2 if autocast else 1e-5) * float(want.detach().abs().max()))


def test_gates_and_norms_trace():
    h, g = (torch.randn(4, 64, device="cuda") for _ in range(2))
    f = lambda h, g: (Fn.silu_gate(h, g), Fn.rms_norm(h.bfloat16(), g[0]), Fn.layer_norm(h, None, None, 1e-6, torch.bfloat16))  # noqa: E731
    traced = torch.jit.trace(f, (h, g), check_trace=False)
    h, g = g + 1, h
    for a, b in zip(traced(h, g), f(h, g)):
        assert a.dtype == b.dtype
        torch.testing.assert_close(a, b, rtol=1e-2 if a.dtype == torch.bfloat16 else 1e-5, atol=1e-6)


@pytest.mark.parametrize("T", [1, 6])
@pytest.mark.parametrize("cell", ["lru", "mamba", "mlstm", "linear_attention", "delta", "recurrence"])
def test_recurrences_refuse_to_be_traced(cell, T):
    make = {"lru": lambda: sm.LRUCell(64, 64), "mamba": lambda: sm.MambaCell(64, num_heads=2, head_dim=16, state_dim=16),
            "mlstm": lambda: sm.mLSTMCell(64, hidden_dim=64, num_heads=2), "linear_attention": lambda: sm.LinearAttentionCell(64, 16, 2),
            "delta": lambda: sm.DeltaNetCell(64, 16, 2)}
    model = sm.GatedLinearRecurrence(64) if cell == "recurrence" else sm.Memoroid(make[cell]())
    block = _Output(sm.Residual(sm.PreNorm(model, 64))).cuda()
    with torch.no_grad(), pytest.raises(RuntimeError, match="traced"):
        torch.jit.trace(block, (torch.randn(2, T, 64, device="cuda"), torch.zeros(2, T, dtype=torch.bool, device="cuda")), check_trace=False)
