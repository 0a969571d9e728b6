"""The autograd node of the operators: what it saves, and the gradients nobody asks for."""
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


@pytest.mark.parametrize("base4", [False, True])
@pytest.mark.parametrize("in_size, out_size", [(64, 250), (100, 100), (2048, 5000)])
def test_gradients_nobody_asks_for(in_size, out_size, base4):
    """A layer behind an input without gradient (every first layer), and one with a frozen bias: the
    other gradients bit for bit, no column sums and no sum over the stacks."""
    from butterfly_amd import Butterfly, ButterflyBase4
    say("unwanted gradients", in_size, out_size, base4)
    torch.manual_seed(in_size)
    layer = (ButterflyBase4 if base4 else Butterfly)(in_size, out_size).cuda()
    names = [n for n, p in layer.named_parameters() if p.numel() > 0]
    params = dict(layer.named_parameters())
    x = torch.randn(33, in_size, device="cuda")
    g = torch.randn(33, out_size, device="cuda")

    def step(input_wanted, bias_wanted):
        params["bias"].requires_grad_(bias_wanted)
        a = x.clone().requires_grad_(input_wanted)
        y = layer(a)
        wanted = [params[n] for n in names if n != "bias" or bias_wanted] + ([a] if input_wanted else [])
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        grads = torch.autograd.grad(y, wanted, g)
        count = torch.cuda.memory_stats()["allocation.all.allocated"] - before
        return dict(zip([n for n in names if n != "bias" or bias_wanted] + ["input"], grads)), count

    full, most = step(True, True)
    stacks = -(-out_size // layer.n)
    for input_wanted, bias_wanted in ((False, True), (True, False), (False, False)):
        part, count = step(input_wanted, bias_wanted)
        for name, grad in part.items():
            assert torch.equal(grad, full[name]), name
        # (the one stack's kernels write their input gradient, wanted or not)
        left_out = (not bias_wanted) + (not input_wanted and stacks > 1)
        assert count == most - left_out, (input_wanted, bias_wanted, count, most)
    # asked for in one pass over the graph and not in the next
    params["bias"].requires_grad_(True)
    a = x.clone().requires_grad_()
    y = layer(a)
    (only,) = torch.autograd.grad(y, [params["bias"]], g, retain_graph=True)
    (rows,) = torch.autograd.grad(y, [a], g)
    assert torch.equal(only, full["bias"]) and torch.equal(rows, full["input"])


def test_layer_backward_without_an_input_gradient_through_the_c_abi():
    """d_input NULL: left out where the stacks' gradients would be added up, refused elsewhere."""
    import ctypes
    from butterfly_amd import _capi
    L, S, B = 5, 3, 17
    n = 1 << L
    torch.manual_seed(1)
    tw = torch.randn(S, 1, L, n // 2, 2, 2, device="cuda")
    x, g = torch.randn(B, n, device="cuda"), torch.randn(B, S * n, device="cuda")
    ptr = lambda t: None if t is None else ctypes.c_void_p(t.data_ptr())
    lib = _capi.lib()

    def run(stacks, with_input):
        layer = _capi.Layer()
        p = layer.problem
        p.dtype, p.increasing_stride, p.batch, p.nstacks, p.log_n, p.nblocks = 0, 1, B, stacks, L, 1
        p.input_size = p.output_size = n
        p.input_stride[:] = (n, 0, 1)
        p.output_stride[:] = (stacks * n, n, 1)
        p.d_input_stride[:] = (n, n, 1)
        layer.shared_input = 1
        layer.total_output = stacks * n
        layer.twiddle = tw.data_ptr()
        size = lib.bf_layer_bw_workspace_bytes(ctypes.byref(layer), 0, 0)
        ws = torch.empty(size, dtype=torch.uint8, device="cuda")
        d_tw = torch.zeros_like(tw[:stacks])
        d_x = torch.zeros_like(x) if with_input else None
        rc = lib.bf_layer_bw(ctypes.byref(layer), ptr(x), ptr(g[:, :stacks * n].contiguous()), None, 0, ptr(d_tw), None,
                             ptr(d_x), None, ptr(ws), size, None)
        torch.cuda.synchronize()
        return rc, d_tw, d_x

    rc, d_tw, d_x = run(S, True)
    assert rc == 0 and d_x.abs().sum() > 0
    rc, without, _ = run(S, False)
    assert rc == 0 and torch.equal(without, d_tw)
    rc, _, _ = run(1, False)
    assert rc == _capi.BF_ERR_INVALID
