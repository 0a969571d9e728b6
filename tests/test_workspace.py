"""Room for the partial slices of a backward call: bounded, whatever the number of passes."""
import ctypes

import pytest
import torch

from butterfly_amd import _capi

MIB = 1 << 20


def problem(dtype, batch, nstacks, log_n, nblocks):
    n = 1 << log_n
    p = _capi.Problem()
    p.dtype, p.increasing_stride, p.batch, p.nstacks, p.log_n, p.nblocks = dtype, 1, batch, nstacks, log_n, nblocks
    p.input_size = p.output_size = n
    for stride in (p.input_stride, p.output_stride, p.d_input_stride):
        stride[:] = (nstacks * n, n, 1)
    return p


@pytest.mark.parametrize("base4", [False, True])
@pytest.mark.parametrize("dtype, batch, nstacks, log_n", [
    (_capi.BF_F32, 4096, 1, 10), (_capi.BF_F32, 300, 2, 5), (_capi.BF_F32, 4096, 1, 12), (_capi.BF_C64, 4096, 1, 8),
    (_capi.BF_C64, 2048, 1, 12), (_capi.BF_F32, 8, 1, 17)])
def test_backward_workspace_is_bounded(dtype, batch, nstacks, log_n, base4):
    lib = _capi.lib()
    plane = (batch * nstacks * (8 if dtype == _capi.BF_C64 else 4) << log_n) + 255 & ~255

    def partials(nblocks):
        """The workspace of a backward with kept activations is one gradient plane and the slices."""
        p = ctypes.byref(problem(dtype, batch, nstacks, log_n, nblocks))
        size = (lib.bf_butterfly_multiply_base4_bw_saved_workspace_bytes(p) if base4
                else lib.bf_butterfly_multiply_bw_saved_workspace_bytes(p, 0))
        assert size != _capi.SIZE_INVALID and size > plane
        return size - plane

    few = partials(3)
    for nblocks in (4, 7, 12, 18):
        assert partials(nblocks) <= max(few, 128 * MIB), nblocks


@pytest.mark.gpu
@pytest.mark.parametrize("dtype, batch, nstacks, log_n, nblocks", [
    (torch.float32, 16384, 1, 10, 16), (torch.float32, 9, 3, 4, 40), (torch.complex64, 700, 1, 11, 5)])
def test_factor_gradients_do_not_depend_on_the_room(dtype, batch, nstacks, log_n, nblocks):
    """Slices of all passes side by side, of some at a time, of one at a time: the same sums."""
    lib = _capi.lib()
    n = 1 << log_n
    torch.manual_seed(n)
    tw = torch.randn(nstacks, nblocks, log_n, n // 2, 2, 2, dtype=dtype, device="cuda") / 2 ** 0.5
    x, g = (torch.randn(batch, nstacks, n, dtype=dtype, device="cuda") for _ in range(2))
    p = problem(_capi.BF_C64 if dtype.is_complex else _capi.BF_F32, batch, nstacks, log_n, nblocks)
    asked = lib.bf_butterfly_multiply_bw_workspace_bytes(ctypes.byref(p))
    ws = torch.empty(asked + 600 * MIB, dtype=torch.uint8, device="cuda")
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())

    def run(size):
        d_tw, d_x = torch.full_like(tw, 7), torch.full_like(x, 7)
        rc = lib.bf_butterfly_multiply_bw(ctypes.byref(p), ptr(tw), ptr(x), ptr(g), ptr(d_tw), ptr(d_x), ptr(ws), size,
                                          _capi._stream())
        torch.cuda.synchronize()
        return rc, d_tw, d_x

    rc, d_tw, d_x = run(asked)
    assert rc == 0
    least, size = asked, asked
    # from more than is asked for down to what the call refuses (nothing is launched then)
    for size in [asked + 600 * MIB] + [asked - k * (asked // 64 & ~255) for k in range(1, 64)]:
        rc, d_tw2, d_x2 = run(size)
        if rc != 0:
            assert rc == _capi.BF_ERR_WORKSPACE
            break
        least = size
        assert torch.equal(d_tw, d_tw2) and torch.equal(d_x, d_x2), (size, asked)
    assert least < asked
