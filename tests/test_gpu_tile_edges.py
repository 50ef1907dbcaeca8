"""128x128 tiles cut at the matrix's edges: every width class of the last tile
column (at most 64 columns, more, whole) against rows that end inside a tile,
bit for bit with the oracle, the extremes of each tile at its far corner."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from lumenrl_amd.quantization import fp8_block_quant
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows", [1, 31, 127, 129, 200])
@pytest.mark.parametrize("cols", [8, 56, 64, 72, 120, 128, 136, 192, 200, 264])
def test_cut_tiles_vs_oracle(dtype, rows, cols):
    g = torch.Generator().manual_seed(rows * 1000 + cols)
    x = torch.randn(2, rows, cols + 8, generator=g) * 0.02
    x[0, -1, cols - 1] = 5.0           # the last tile's largest value at its last element
    x[1, rows // 2, cols - 3] = float("inf") if cols % 16 else -3.0
    x = x.to(dtype)[..., :cols]        # rows with a pitch: what lies past the width is not read into a tile
    codes, scales = fp8_block_quant(x.cuda(), (128, 128))
    torch.cuda.synchronize()
    name = {torch.bfloat16: "bf16", torch.float16: "f16", torch.float32: "f32"}[dtype]
    for b in range(2):
        v = x[b].contiguous()
        h = v.numpy() if dtype == torch.float32 else v.view(torch.int16).numpy().view(np.uint16)
        oc, osc = O.fp8_block_quant(h, name, "f32", (128, 128))
        assert np.array_equal(codes[b].view(torch.uint8).cpu().numpy(), oc[0])
        assert np.array_equal(scales[b].cpu().numpy().view(np.uint32), osc[0].view(np.uint32))
