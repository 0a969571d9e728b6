"""The autograd node of the operators."""
import pytest
import torch

import butterfly_amd  # noqa: F401  (registers the operators)
from test_gpu_multiply import say

pytestmark = pytest.mark.gpu


def perm_call(L=6, layer=False, seed=0):
    """A differentiable call with both column tables: (output, twiddle, input, in_perm, out_index)."""
    ops = torch.ops.torch_butterfly
    torch.manual_seed(seed)
    n = 1 << L
    tw = (torch.randn(1, 1, L, n // 2, 2, 2) / 2 ** 0.5).cuda().requires_grad_()
    tables = [torch.randperm(n).int().cuda() for _ in range(2)]
    if layer:
        x = torch.randn(9, n).cuda().requires_grad_()
        y = ops.butterfly_layer(tw, x, None, *tables, None, None, True, n, False, False)
    else:
        x = torch.randn(9, 1, n).cuda().requires_grad_()
        y = ops.butterfly_multiply_perm(tw, x, *tables, None, True, None)
    return y, tw, x, *tables


@pytest.mark.parametrize("layer", [False, True])
@pytest.mark.parametrize("which", [0, 1])
def test_column_tables_are_saved_variables(layer, which):
    say("tables", layer, which)
    y, tw, x, *tables = perm_call(layer=layer)
    # another permutation put into the table: the backward would follow it silently
    with torch.no_grad():
        tables[which].copy_(tables[which].flip(0))
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(y.sum(), (tw, x))

    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append((t.dtype, t.numel())) or t, lambda t: t):
        y, tw, x, *tables = perm_call(layer=layer)
    assert seen.count((torch.int32, x.shape[-1])) == 2

    # released with the graph
    y, tw, x, *tables = perm_call(L=12, layer=layer)
    loss = y.sum()
    torch.autograd.grad(loss, (tw, x))
    held = torch.cuda.memory_allocated()
    del tables
    assert held - torch.cuda.memory_allocated() >= 2 * 4 * 4096
