"""dynamic_mxfp4_quant at the edges of its grid, bit for bit against the oracle: rows around a 32-row group
and a 256-row padding block, one chunk of 512 values and its remainders, and both sides of the line between
one chunk a wave and eight."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import aklr_amd
from aklr_amd import workloads
from oracle import layouts as olayouts
from oracle import quant as oquant
from tests.helpers import bf16_bits, say, u8

pytestmark = pytest.mark.gpu


# 8192 chunks: 256 x 16384 (shuffled 256 x 32), 512 x 8192, 160 x 26112 just past it
@pytest.mark.parametrize("t,h", [(1, 32), (31, 480), (32, 512), (33, 544), (255, 2080), (256, 16384), (257, 16384),
                                 (512, 8192), (513, 8192), (160, 26112), (3, 65536)])
def test_rows_and_chunks(t, h):
    say(f"mxfp4 quant grid {t}x{h}")
    x = workloads.activations(t, h, seed=t + h, device="cuda:0")
    codes, scales = oquant.dynamic_mxfp4_quant(bf16_bits(x))
    for shuffle in (False, True):
        for _ in range(2):  # the second call may reuse the first one's memory: every padding byte is written
            q, s = aklr_amd.dynamic_mxfp4_quant(x, shuffle)
            torch.cuda.synchronize()
            want = olayouts.e8m0_scales(scales) if shuffle else scales
            assert np.array_equal(u8(q), codes) and np.array_equal(u8(s), want)
            s.view(torch.uint8).fill_(0xAB)
            del q, s
