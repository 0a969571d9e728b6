"""Forward plans of complex64 rows between column tables, from the workspace they ask for."""
import ctypes

import pytest

from butterfly_amd import _capi


@pytest.mark.parametrize("increasing", [0, 1])
@pytest.mark.parametrize("log_n, nblocks, batch, single", [
    (11, 1, 1, True), (11, 1, 64, True), (11, 1, 8192, True),   # the whole block in one launch, tables or not
    (11, 2, 64, False), (11, 2, 8192, False), (12, 1, 8192, False)])
def test_inference_forward_takes_the_whole_block_kernel(log_n, nblocks, batch, single, increasing):
    """A forward call that keeps nothing reads and writes each row once where the factors of a block fit
    the registers, also through a table on the side where the passes have tiles made for it."""
    lib = _capi.lib()
    n = 1 << log_n
    sizes = []
    for table in (None, ctypes.c_void_p(16)):
        layer = _capi.Layer()
        p = layer.problem
        p.dtype, p.increasing_stride, p.batch, p.nstacks, p.log_n, p.nblocks = _capi.BF_C64, increasing, batch, 1, log_n, nblocks
        p.input_size = p.output_size = layer.total_output = n
        for stride in (p.input_stride, p.output_stride, p.d_input_stride):
            stride[:] = (n, n, 1)
        layer.shared_input = 1
        if increasing:
            layer.in_perm = table
        else:
            layer.out_index = table
        sizes.append(lib.bf_layer_fw_workspace_bytes(ctypes.byref(layer)))
    assert sizes[0] == sizes[1]
    assert (sizes[0] == 0) == single
