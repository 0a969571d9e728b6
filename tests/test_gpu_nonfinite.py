"""Infinities and NaN in the rows and in the output's gradient: each kernel passes them on to the
outputs that depend on them and to no others, as the oracle does."""
import numpy as np
import pytest
import torch

import butterfly_amd  # noqa: F401  (registers the operators)
from conftest import randn, rel_err
from oracle import oracle
from test_gpu_multiply import BW_TOL, FW_TOL, dev, say

pytestmark = pytest.mark.gpu


def spoil(a, rng):
    """Infinities of either sign and a NaN in three rows of a (batch, stacks, width) operand."""
    batch, width = a.shape[0], a.shape[2]
    for row, value in ((0, np.inf), (batch // 2, -np.inf), (batch - 1, np.nan)):
        a[row, rng.integers(a.shape[1]), rng.integers(width)] = value


def same(got, ref, tol):
    """Infinities (with their sign) and NaN in the same places, the rest within tol."""
    got, ref = (np.ascontiguousarray(a) for a in (got.detach().cpu().numpy(), ref))
    assert got.shape == ref.shape and got.dtype == ref.dtype
    if got.dtype.kind == "c":
        got, ref = (a.view(a.real.dtype) for a in (got, ref))
    bad = ~np.isfinite(ref)
    assert np.array_equal(np.isnan(got), np.isnan(ref)), (np.isnan(got).sum(), np.isnan(ref).sum())
    assert np.array_equal(got[bad], ref[bad], equal_nan=True)
    assert rel_err(np.where(bad, 0, got), np.where(bad, 0, ref)) < tol


def factors(rng, shape, dtype):
    return (randn(rng, shape, dtype) / np.sqrt(shape[-1])).astype(dtype)


@pytest.mark.parametrize("dtype, B, S, L, nb, inc", [
    # the closing 2x2 stage on the top bit and on bit 0, few rows (passes) and many (one launch), one
    # plane of rows a workgroup and two
    (np.float32, 7, 1, 11, 1, True), (np.float32, 1001, 1, 11, 1, True), (np.float32, 501, 2, 11, 1, False),
    (np.float32, 2061, 1, 11, 1, False), (np.float32, 1001, 1, 11, 2, True), (np.float32, 1001, 1, 12, 1, True),
    (np.complex64, 3301, 1, 9, 1, True), (np.complex64, 3301, 1, 9, 1, False), (np.complex64, 831, 1, 11, 1, True),
    (np.complex64, 831, 1, 11, 1, False), (np.complex64, 1651, 1, 10, 1, True)],
    ids=lambda v: v.__name__ if isinstance(v, type) else str(v))
def test_base4_rows(dtype, B, S, L, nb, inc):
    say("non-finite base 4", dtype, B, S, L, nb, inc)
    rng = np.random.default_rng(B + L)
    n = 1 << L
    tw4 = factors(rng, (S, nb, L // 2, n // 4, 4, 4), dtype)
    tw2 = factors(rng, (S, nb, L % 2, n // 2, 2, 2), dtype)
    x, g = randn(rng, (B, S, n), dtype), randn(rng, (B, S, n), dtype)
    spoil(x, rng)
    leaves = [dev(t).requires_grad_() for t in (tw4, tw2, x)]
    plain = torch.ops.torch_butterfly.butterfly_multiply_base4_fw(*(t.detach() for t in leaves), inc, None)
    y = torch.ops.torch_butterfly.butterfly_multiply_base4(*leaves, inc, None)
    with np.errstate(invalid="ignore"):
        y_ref = oracle.butterfly_base4_fw(tw4, tw2, x, inc)
    same(plain, y_ref, FW_TOL)
    same(y, y_ref, FW_TOL)
    spoil(g, rng)
    wanted = [t for t in leaves if t.numel() > 0]
    grads = torch.autograd.grad(y, wanted, dev(g))
    refs = oracle.butterfly_base4_bw(tw4, tw2, x, g, inc)
    for got, ref in zip(grads, [r for r in refs if r.size > 0]):
        same(got, ref, BW_TOL)


@pytest.mark.parametrize("dtype, B, in_size, out_size, nb, inc", [
    (np.float32, 37, 256, 1000, 1, True), (np.float32, 37, 30, 120, 2, False), (np.float32, 9, 2000, 5000, 1, False),
    (np.float32, 37, 500, 512, 1, True), (np.complex64, 37, 100, 300, 1, True), (np.complex64, 9, 4096, 4096, 1, False)],
    ids=lambda v: v.__name__ if isinstance(v, type) else str(v))
def test_layer_rows(dtype, B, in_size, out_size, nb, inc):
    """Whole layers: stacks that share the input, the sum of their gradients, the bias gradient."""
    say("non-finite layer", dtype, B, in_size, out_size, nb, inc)
    rng = np.random.default_rng(B + in_size)
    L = (in_size - 1).bit_length()
    n = 1 << L
    S = -(-out_size // n)
    tw = factors(rng, (S, nb, L, n // 2, 2, 2), dtype)
    bias = randn(rng, (out_size,), dtype)
    x, g = randn(rng, (B, 1, in_size), dtype), randn(rng, (B, 1, out_size), dtype)
    spoil(x, rng)
    spoil(g, rng)
    leaves = [dev(t).requires_grad_() for t in (tw, x[:, 0], bias)]
    y = torch.ops.torch_butterfly.butterfly_layer(leaves[0], leaves[1], leaves[2], None, None, None, None, inc, out_size,
                                                  False, False)
    d_tw, d_x, d_bias = torch.autograd.grad(y, leaves, dev(g[:, 0]))
    with np.errstate(invalid="ignore"):
        rows = np.repeat(x, S, axis=1)
        y_ref = oracle.butterfly_fw(tw, rows, inc).reshape(B, S * n)[:, :out_size] + bias
        same(y, y_ref, FW_TOL)
        same(d_bias, g[:, 0].sum(0), BW_TOL)
        grad = np.zeros((B, S * n), dtype)
        grad[:, :out_size] = g[:, 0]
        d_tw_ref, d_rows = oracle.butterfly_bw(tw, rows, grad.reshape(B, S, n), inc)
        same(d_x, d_rows.sum(1), BW_TOL)
        same(d_tw, d_tw_ref, BW_TOL)


@pytest.mark.parametrize("B, L, inc", [(37, 11, True), (37, 11, False), (19, 12, True), (19, 12, False)])
def test_complex_rows_through_column_tables(B, L, inc):
    say("non-finite tables", B, L, inc)
    rng = np.random.default_rng(B + L)
    n = 1 << L
    tw = factors(rng, (1, 1, L, n // 2, 2, 2), np.complex64)
    x, g = randn(rng, (B, 1, n), np.complex64), randn(rng, (B, 1, n), np.complex64)
    spoil(x, rng)
    spoil(g, rng)
    perm = rng.permutation(n)
    inverse = np.argsort(perm)
    table = dev((perm if inc else inverse).astype(np.int32))
    leaves = [dev(t).requires_grad_() for t in (tw, x)]
    y = torch.ops.torch_butterfly.butterfly_multiply_perm(*leaves, table if inc else None, None if inc else table, None,
                                                          inc, None)
    d_tw, d_x = torch.autograd.grad(y, leaves, dev(g))
    with np.errstate(invalid="ignore"):
        if inc:
            u, gy = np.ascontiguousarray(x[:, :, perm]), g
        else:
            u, gy = x, np.ascontiguousarray(g[:, :, inverse])
        y_ref = oracle.butterfly_fw(tw, u, inc)
        d_tw_ref, d_u = oracle.butterfly_bw(tw, u, gy, inc)
        same(y, y_ref if inc else y_ref[:, :, perm], FW_TOL)
        same(d_x, d_u[:, :, inverse] if inc else d_u, BW_TOL)
        same(d_tw, d_tw_ref, BW_TOL)


@pytest.mark.parametrize("B, L, inc", [(37, 5, True), (37, 10, False), (19, 11, True), (9, 12, False)])
def test_real_rows_around_complex_factors(B, L, inc):
    say("non-finite real rows", B, L, inc)
    rng = np.random.default_rng(B + L)
    n = 1 << L
    tw = factors(rng, (1, 1, L, n // 2, 2, 2), np.complex64)
    x, g = randn(rng, (B, 1, n), np.float32), randn(rng, (B, 1, n), np.float32)
    spoil(x, rng)
    spoil(g, rng)
    leaves = [dev(t).requires_grad_() for t in (tw, x[:, 0])]
    y = torch.ops.torch_butterfly.butterfly_layer(*leaves, None, None, None, None, None, inc, n, True, True)
    d_tw, d_x = torch.autograd.grad(y, leaves, dev(g[:, 0]))
    with np.errstate(invalid="ignore"):
        xc, gc = x.astype(np.complex64), g.astype(np.complex64)
        same(y, oracle.butterfly_fw(tw, xc, inc)[:, 0].real, FW_TOL)
        d_tw_ref, d_u = oracle.butterfly_bw(tw, xc, gc, inc)
        same(d_x, d_u[:, 0].real, BW_TOL)
        same(d_tw, d_tw_ref, BW_TOL)
