"""A device table written by one launch (lrq_group_upload) against the same table
copied and mapped in two steps, byte for byte but for padding: one tensor, empty tensors first,
between and last, and as many tensors as the launch's arguments hold."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from lumenrl_amd import _lib
from lumenrl_amd.quantization import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,block", [("fp8_block", (128, 128)), ("fp8_block", (1, 128)), ("mxfp4", (1, 32)),
                                       ("tensor_scale", (1, 1))])
@pytest.mark.parametrize("shapes", [[(128, 128)], [(0, 256), (384, 256), (0, 128), (1, 4096), (0, 256)],
                                    [(1 + 37 * i, 128 * (1 + i % 5)) for i in range(_lib.UPLOAD_TENSORS)]])
def test_one_launch_table_equals_copy_and_map(fmt, block, shapes):
    if fmt == "tensor_scale":
        shapes = [s for s in shapes if s[0]]
    L, dev = _lib.lib(), torch.device("cuda", 0)
    w = torch.zeros(1 << 20, dtype=torch.bfloat16, device=dev)
    descs = (_lib.LrqTensor * len(shapes))()
    for d, (r, c) in zip(descs, shapes):  # only addresses are recorded: no launch reads them
        d.in_ = d.codes = d.scales = w.data_ptr()
        d.batch, d.rows, d.cols, d.ld, d.batch_stride = 1, r, c, c, r * c
    args = (ops._FMTS[fmt], descs, len(shapes), _lib.DTYPE_BF16, *block, 0)
    need = L.lrq_group_table_bytes(*args)
    host = np.zeros(need, np.uint8)
    assert L.lrq_group_pack(*args, host.ctypes.data, need) == 0
    size = L.lrq_group_device_bytes(host.ctypes.data)
    one = torch.full((size,), 0xA5, dtype=torch.uint8, device=dev)
    two = torch.full((size,), 0xA5, dtype=torch.uint8, device=dev)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert L.lrq_group_upload(host.ctypes.data, one.data_ptr(), stream) == 0
    two[:need] = torch.from_numpy(host).to(dev)
    assert L.lrq_group_build_map(host.ctypes.data, two.data_ptr(), stream) == 0
    host[:] = 0  # the call keeps nothing of the host table
    torch.cuda.synchronize()
    one, two = one.cpu().numpy(), two.cpu().numpy()
    gaps = one != two  # only padding, which nothing reads, is left unwritten: behind the header and the descriptors
    header, first, each = 104, 256, 112
    assert not gaps[:header].any() and not gaps[first:first + each * len(shapes)].any()
    assert not gaps[need:].any() and (one[gaps] == 0xA5).all()
