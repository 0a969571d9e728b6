"""Real numbers around complex factors (rows read and written as real numbers by the layer's own
kernels), diagonals and column tables next to them, against the oracle in double precision."""
import numpy as np
import pytest
import torch

import butterfly_amd  # noqa: F401  (registers the operators)
from conftest import randn, rel_err
from oracle import oracle
from test_gpu_multiply import BW_TOL, FW_TOL, dev, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("real", ["in", "out", "both"])
@pytest.mark.parametrize("B, in_size, out_size, nb, inc, extras", [
    # every kind of pass that can stand at an end of the schedule: short rows, whole rows, chunks and
    # spans first or last, the tiles made for column tables, rows that are narrower or wider than n
    (37, 2, 2, 1, True, ""), (301, 30, 32, 2, False, "d"), (33, 64, 64, 1, True, "i"), (1030, 256, 250, 1, False, "do"),
    (129, 700, 1000, 2, True, "d"), (70, 1024, 1024, 1, False, "io"), (65, 1500, 2048, 1, True, "i"),
    (65, 2048, 2000, 1, False, "o"), (21, 4096, 4096, 1, True, "di"), (21, 4000, 4001, 1, False, "o"),
    (9, 4096, 4096, 2, True, "d"), (7, 8192, 8192, 1, False, ""), (5, 16384, 16000, 1, True, "d"),
    (45, 100, 500, 1, True, "d"), (45, 128, 300, 2, False, "i")], ids=str)
def test_against_the_oracle(B, in_size, out_size, nb, inc, extras, real):
    say("real rows", B, in_size, out_size, nb, inc, extras, real)
    rng = np.random.default_rng(B + in_size + nb)
    L = (in_size - 1).bit_length()
    n = 1 << L
    S = -(-out_size // n)
    tw = (randn(rng, (S, nb, L, n // 2, 2, 2), np.complex64) / np.sqrt(2)).astype(np.complex64)
    x = randn(rng, (B, in_size), np.float32 if real != "out" else np.complex64)
    g = randn(rng, (B, out_size), np.float32 if real != "in" else np.complex64)
    scales = [randn(rng, (k,), np.complex64) if "d" in extras else None for k in (in_size, out_size)]
    perm, order = np.arange(n), np.arange(n)
    if "i" in extras:
        perm[:in_size] = rng.permutation(in_size)
    if "o" in extras:
        order[:out_size] = rng.permutation(out_size)   # output column c is column order[c] of the product
    index = np.argsort(order)

    leaves = [dev(a).requires_grad_() for a in (tw, x)]
    diagonals = [None if a is None else dev(a).requires_grad_() for a in scales]
    tables = [dev(perm.astype(np.int32)) if "i" in extras else None, dev(index.astype(np.int32)) if "o" in extras else None]

    def call():
        return torch.ops.torch_butterfly.butterfly_layer(*leaves, None, *tables, *diagonals, inc, out_size, real != "out",
                                                         real != "in")

    with torch.no_grad():
        plain = call()
    y = call()
    wanted = leaves + [d for d in diagonals if d is not None]
    grads = torch.autograd.grad(y, wanted, dev(g))

    wide = lambda a: a.astype(np.complex128)
    one = np.ones(max(n, S * n), np.complex128)
    before, behind = one[:n].copy(), one[:S * n].copy()
    if "d" in extras:
        before[:in_size], behind[:out_size] = scales
    rows = np.zeros((B, n), np.complex128)
    rows[:, :in_size] = x
    rows = rows[:, perm]
    u = np.repeat((rows * before)[:, None], S, axis=1)
    v = oracle.butterfly_fw(wide(tw), np.ascontiguousarray(u), inc).reshape(B, S * n)
    # (the diagonal stands between the factors and the permutation)
    columns = order[:out_size] if S == 1 else np.arange(out_size)
    y_ref = (v * behind)[:, columns]
    if real != "in":
        y_ref = y_ref.real
    for got in (plain, y):
        assert got.dtype == (torch.complex64 if real == "in" else torch.float32)
        assert rel_err(got.detach().cpu().numpy(), y_ref) < FW_TOL
    gv = np.zeros((B, S * n), np.complex128)
    gv[:, columns] = g
    d_behind = (v.conj() * gv).sum(0)
    d_tw, d_u = oracle.butterfly_bw(wide(tw), np.ascontiguousarray(u), (gv * behind.conj()).reshape(B, S, n), inc)
    d_u = d_u.sum(1)
    d_before = (rows.conj() * d_u).sum(0)
    d_rows = np.zeros_like(rows)
    d_rows[:, perm] = d_u * before.conj()
    d_x = d_rows[:, :in_size]
    refs = [d_tw, d_x if real == "out" else d_x.real]
    if "d" in extras:
        refs += [d_before[:in_size], d_behind[:out_size]]
    for got, ref in zip(grads, refs):
        assert rel_err(got.cpu().numpy(), ref) < BW_TOL
