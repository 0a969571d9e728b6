"""What a FusedSequential must not fold away, and layers whose methods a subclass overrides."""
import pytest
import torch
from torch import nn

from test_gpu_multiply import say

pytestmark = pytest.mark.gpu


def close(a, b):
    return a.shape == b.shape and a.dtype == b.dtype and (a - b).norm().item() <= 1e-5 * b.norm().item()


def chain(n=64):
    """Real rows through a permutation, a diagonal and a complex layer and back."""
    from butterfly_amd import Butterfly
    from butterfly_amd.complex_utils import Complex2Real, Real2Complex
    from butterfly_amd.diagonal import Diagonal
    from butterfly_amd.permutation import FixedPermutation, FusedSequential
    torch.manual_seed(n)
    return FusedSequential(FixedPermutation(torch.randperm(n)), Real2Complex(), Diagonal(n, complex=True),
                           Butterfly(n, n, bias=False, complex=True), Complex2Real(), FixedPermutation(torch.randperm(n))).cuda()


def compare(fused, x):
    """Outputs and every gradient against the children one after the other."""
    plain = nn.Sequential(*fused)
    a, b = (x.clone().requires_grad_() for _ in range(2))
    y, z = fused(a), plain(b)
    assert close(y, z)
    g = torch.randn_like(z)
    params = [p for p in fused.parameters()]
    for u, v in zip(torch.autograd.grad(y, [a] + params, g), torch.autograd.grad(z, [b] + params, g)):
        assert close(u, v)


@pytest.mark.parametrize("kind", ["forward", "forward_pre", "full_backward", "full_backward_pre", "global_forward",
                                  "global_forward_pre"])
@pytest.mark.parametrize("child", [1, 4], ids=["Real2Complex", "Complex2Real"])
def test_hooks_of_conversions_fire(child, kind):
    say("hooks", child, kind)
    seq = chain()
    x = torch.randn(7, 64, device="cuda")
    y0 = seq(x)
    calls = []
    hook = lambda module, *args: calls.append(module) or None
    if kind.startswith("global"):
        handle = getattr(nn.modules.module, "register_module_" + kind[len("global_"):] + "_hook")(hook)
    else:
        handle = getattr(seq[child], f"register_{kind}_hook")(hook)
    try:
        a = x.clone().requires_grad_()
        y = seq(a)
        y.sum().backward()
    finally:
        handle.remove()
    assert calls.count(seq[child]) == 1
    assert close(y.detach(), y0.detach())
    calls.clear()
    assert torch.equal(seq(x), y0) and not calls


def test_hooks_of_a_layer_see_complex_numbers():
    """A hook on the layer between two conversions is handed what the layer takes and returns."""
    seq = chain()
    seen = []
    handle = seq[3].register_forward_hook(lambda module, args, out: seen.append((args[0].dtype, out.dtype)) or 2 * out)
    x = torch.randn(7, 64, device="cuda")
    y = seq(x)
    handle.remove()
    assert seen == [(torch.complex64, torch.complex64)]
    assert close(y, 2 * seq(x))


@pytest.mark.parametrize("child", range(6))
def test_children_with_a_forward_of_their_own(child):
    """A subclass that overrides forward is run, whatever it derives from."""
    say("override", child)
    seq = chain()
    base = type(seq[child])

    class Doubled(base):
        def forward(self, input):
            return 2 * base.forward(self, input)

    x = torch.randn(7, 64, device="cuda")
    y = seq(x)
    seq[child].__class__ = Doubled
    assert close(seq(x), 2 * y)
    compare(seq, x)


def test_base4_layers_among_the_children():
    """ButterflyBase4 folds nothing: its neighbours run as modules."""
    from butterfly_amd import ButterflyBase4
    from butterfly_amd.diagonal import Diagonal
    from butterfly_amd.permutation import FixedPermutation, FusedSequential
    torch.manual_seed(3)
    seq = FusedSequential(FixedPermutation(torch.randperm(64)), ButterflyBase4(64, 100, bias=False), Diagonal(100)).cuda()
    compare(seq, torch.randn(9, 64, device="cuda"))


@pytest.mark.parametrize("width", [50, 90])
def test_rows_of_another_width(width):
    """A permutation or diagonal in front of a layer refuses (or trims) rows that are not as wide as it
    is; the layer alone takes rows of any width."""
    from butterfly_amd import Butterfly
    from butterfly_amd.diagonal import Diagonal
    from butterfly_amd.permutation import FixedPermutation, FusedSequential
    torch.manual_seed(width)
    x = torch.randn(5, width, device="cuda")
    layer = Butterfly(64, 64).cuda()
    for front in (FixedPermutation(torch.randperm(64)).cuda(), Diagonal(64).cuda()):
        fused, plain = FusedSequential(front, layer), nn.Sequential(front, layer)
        if isinstance(front, Diagonal):
            with pytest.raises(RuntimeError):
                plain(x)
            with pytest.raises(RuntimeError):
                fused(x)
        elif width > 64:
            assert close(fused(x), plain(x))
    assert close(FusedSequential(layer)(x), layer(x))


def test_a_child_that_moves_the_rows():
    """Rows that leave the GPU between two layers, and rows that arrive there."""
    from butterfly_amd.permutation import FusedSequential

    class To(nn.Module):
        def __init__(self, device):
            super().__init__()
            self.device = device

        def forward(self, input):
            return input.to(self.device)

    there, here = chain(), chain().cpu()
    x = torch.randn(7, 64)
    want = here(here(x))
    calls = []
    handles = [m.register_forward_hook(lambda m, a, o: calls.append(type(m).__name__)) for m in (here[2], there[2])]
    down = FusedSequential(*there, To("cpu"), *here)(x.cuda())
    assert close(down, want)
    assert calls == ["Diagonal"]      # folded on the GPU, run on the host
    calls.clear()
    up = FusedSequential(*here, To("cuda"), *there)(x)
    assert up.is_cuda and close(up.cpu(), want)
    assert calls == ["Diagonal"]
    for handle in handles:
        handle.remove()


# (the bias of ButterflyBase4 is added by post_process)
@pytest.mark.parametrize("kind, method", [(kind, method) for kind in ("Butterfly", "ButterflyUnitary", "ButterflyBase4")
                                          for method in ("pre_process", "post_process", "bias_rows")
                                          if (kind, method) != ("ButterflyBase4", "bias_rows")])
@pytest.mark.parametrize("of_the_class", [True, False])
def test_overridden_steps_of_a_layer(kind, method, of_the_class):
    """A layer whose rows are prepared or finished differently, by a subclass or on the object."""
    import butterfly_amd
    say("steps", kind, method, of_the_class)
    torch.manual_seed(5)
    base = getattr(butterfly_amd, kind)
    layer = base(50, 100, nblocks=2).cuda()
    x = torch.randn(6, 50, dtype=torch.complex64 if kind == "ButterflyUnitary" else torch.float32, device="cuda")
    with torch.no_grad():
        plain = layer(x)
        no_bias = plain - layer.bias
        if method == "pre_process":
            change = lambda self, input: base.pre_process(self, 3 * input)
            want = 3 * no_bias + layer.bias
        elif method == "post_process":
            change = lambda self, *args, **kw: 3 * base.post_process(self, *args, **kw)
            want = 3 * plain
        else:
            change = lambda self, *args, **kw: 3 * base.bias_rows(self, *args, **kw)
            want = no_bias + 3 * layer.bias
        if of_the_class:
            layer.__class__ = type("Changed", (base,), {method: change})
        else:
            setattr(layer, method, change.__get__(layer))
        assert close(layer(x), want)
