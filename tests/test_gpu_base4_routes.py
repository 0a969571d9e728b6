"""Base-4 rows on either side of the lines between kernels.  Rows beyond one workgroup run
in one streaming launch or in passes, by their number: the results match the oracle, and calls
that keep the activations for a backward return what calls that do not return, bit for bit.  The
backward of 512 floats takes two or four row groups at a time."""
import numpy as np
import pytest
import torch

import butterfly_amd  # noqa: F401  (registers the operators)
from conftest import randn, rel_err
from oracle import oracle
from test_gpu_multiply import BW_TOL, FW_TOL, dev, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("dtype, L, nb", [(np.float32, 11, 1), (np.float32, 11, 2), (np.float32, 12, 1), (np.float32, 12, 2),
                                          (np.complex64, 9, 1), (np.complex64, 10, 2), (np.complex64, 11, 1)],
                         ids=lambda v: v.__name__ if isinstance(v, type) else str(v))
def test_routes(dtype, L, nb, with_bias):
    ops = torch.ops.torch_butterfly
    n = 1 << L
    rng = np.random.default_rng(L + nb)
    tw4 = (randn(rng, (1, nb, L // 2, n // 4, 4, 4), dtype) / 2).astype(dtype)
    tw2 = (randn(rng, (1, nb, L % 2, n // 2, 2, 2), dtype) / np.sqrt(2)).astype(dtype)
    bias = randn(rng, (n,), dtype) if with_bias else None
    rows = 4 << (11 + (L == 12) - L)          # of a tile
    leaves = [dev(t).requires_grad_() for t in (tw4, tw2)]
    bias_d = None if bias is None else dev(bias).requires_grad_()
    for tiles in (3, 16, 17, 64, 65, 130, 257):
        batch = tiles * rows - 1
        say("routes", dtype, L, nb, with_bias, tiles)
        x = randn(rng, (batch, n), dtype)
        xd = dev(x).requires_grad_()
        with torch.no_grad():
            plain = ops.butterfly_layer_base4(*leaves, xd, bias_d, True, n)
        y = ops.butterfly_layer_base4(*leaves, xd, bias_d, True, n)
        assert torch.equal(plain, y.detach())
        y_ref = oracle.butterfly_base4_fw(tw4, tw2, x[:, None], True)[:, 0]
        assert rel_err(plain.cpu().numpy(), y_ref if bias is None else y_ref + bias) < FW_TOL
        if tiles in (17, 65):
            g = randn(rng, (batch, n), dtype)
            (d_x,) = torch.autograd.grad(y, [xd], dev(g))
            d_x_ref = oracle.butterfly_base4_bw(tw4, tw2, x[:, None], g[:, None], True)[2][:, 0]
            assert rel_err(d_x.cpu().numpy(), d_x_ref) < BW_TOL


@pytest.mark.parametrize("increasing", [True, False])
@pytest.mark.parametrize("batch", [1, 511, 1025, 1536, 1537, 2051])
def test_row_groups_of_the_backward_at_512(batch, increasing):
    say("row groups", batch, increasing)
    n, L, nb = 512, 9, 2
    rng = np.random.default_rng(batch)
    tw4 = (randn(rng, (1, nb, L // 2, n // 4, 4, 4), np.float32) / 2).astype(np.float32)
    tw2 = (randn(rng, (1, nb, 1, n // 2, 2, 2), np.float32) / np.sqrt(2)).astype(np.float32)
    bias = randn(rng, (500,), np.float32)
    x, g = randn(rng, (batch, 510), np.float32), randn(rng, (batch, 500), np.float32)
    leaves = [dev(t).requires_grad_() for t in (tw4, tw2, x, bias)]
    y = torch.ops.torch_butterfly.butterfly_layer_base4(*leaves, increasing, 500)
    grads = torch.autograd.grad(y, leaves, dev(g))
    refs = oracle.butterfly_base4_bw(tw4, tw2, x[:, None], g[:, None], increasing)
    refs = (refs[0], refs[1], refs[2][:, 0], g.astype(np.float64).sum(0))
    for got, ref in zip(grads, refs):
        assert rel_err(got.cpu().numpy(), ref) < BW_TOL
