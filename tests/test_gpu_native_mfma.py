"""BF16 rows on several tokens, through the row kernel and from 98,304 or 131,072
dots on (by tokens and columns) through the f32 matrix cores (k_native_mfma):
every dot is the oracle's dotBf16 bit for bit, on both sides of the rule, at the
edges of the 16-row tiles, of the groups of four tokens and of the token passes,
in each of the kernel's four forms, and with infinities, NaN and denormals in
the input."""
from __future__ import annotations

import numpy as np
import pytest

from colizig_amd import _lib, moe
from tests.helpers import f32_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("O,I,S", [(8192, 2048, 2), (8193, 2048, 8), (8207, 512, 5), (8208, 256, 16), (9001, 2048, 17),
                                   (8200, 4096, 9), (8191, 2048, 3), (8192, 8192, 6), (8195, 768, 13),
                                   # one group of four tokens a pass (the last: four passes)
                                   (49153, 768, 2), (32769, 768, 3), (32790, 256, 4), (65545, 2048, 3),
                                   (6145, 8192, 16),
                                   # two groups (the last: two passes)
                                   (26231, 256, 5), (16397, 512, 8), (16386, 2048, 8), (8200, 4096, 16),
                                   # three, and four over two waves a row tile
                                   (14567, 256, 9), (10925, 1024, 12), (10083, 256, 13), (8195, 512, 16),
                                   # either side of the rule
                                   (16383, 512, 8), (16384, 512, 8), (12287, 768, 8), (12288, 768, 8),
                                   (24575, 1024, 4), (24576, 1024, 4), (98304, 256, 2)])
def test_bf16_rows_many_tokens_bit_exact(gpu, oracle_lib, O, I, S):
    print(f"bf16 rows {O}x{I} S={S}", flush=True)
    moe.set_vram_budget(1 << 30)
    rng = np.random.default_rng(O + I + S)
    w = (rng.normal(0.0, 0.02, size=(O, I)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    x = rng.normal(size=(S, I)).astype(np.float32)
    x[0, :4] = [1e-40, -3e-42, 1e38, -1e38]
    x[S - 1, I - 1] = np.inf
    key = moe.Fp8Matrix.expert_key(43, (O + I) % 509, 3)
    xb, yb = moe.DeviceBuffer(S * I * 4), moe.DeviceBuffer((S * O + 64) * 4)
    try:
        moe.matrix_load_bf16(key, w)
        xb.upload(x)
        yb.upload(np.full(S * O + 64, 7.0, np.float32))
        moe.matmul_bf16_dev(yb.ptr, xb.ptr, S, I, O, key)
        assert _lib.hip().colizig_hip_sync() == 0
        y = yb.download(np.empty(S * O + 64, np.float32))
        assert (y[S * O:] == 7.0).all()  # nothing past the last row
        y, ref = y[:S * O].reshape(S, O), oracle_lib.matmul_bf16(x, w, S, I, O)
        same = (f32_bits(y) == f32_bits(ref)) | (np.isnan(y) & np.isnan(ref))
        assert same.all(), f"{np.count_nonzero(~same)} of {same.size} differ"
    finally:
        xb.free()
        yb.free()
        moe.set_vram_budget(0)
