"""Many-token FP8 products at f32 accuracy (k_gemm_f32x, k_gg_f32x): against
64-bit sums over tile edges, odd rows and columns, wide ranges of magnitude,
infinities and NaN; and layers past 8192 slots against the oracle.

The bound on the relative L2 error: the split into three bf16 terms is exact, a
K block's 128 exact products are summed in f32 (at most 24 rounded additions,
random signs: about sqrt(24) 2^-25), then one FMA per K block: about 2e-7 in
all; 6e-7 is asserted."""
from __future__ import annotations

import numpy as np
import pytest

from colizig_amd import _lib, moe, synth
from oracle import oracle as orc
from tests.helpers import f32_bits, rel_l2

pytestmark = pytest.mark.gpu

RTOL = 6e-7


def _dequant(w, s):
    import torch

    O, I = w.shape
    f = torch.from_numpy(w).view(torch.float8_e4m3fn).double().numpy()
    sc = np.repeat(np.repeat(s.astype(np.float64), 128, 0), 128, 1)[:O, :I]
    return f * sc


def _run(xs, mats, I):
    """Each matrix alone and all in one launch: the same bits."""
    S = xs.shape[0]
    hip = _lib.hip()
    xb = moe.DeviceBuffer(xs.nbytes)
    xb.upload(xs)
    yb = [moe.DeviceBuffer((S * w.shape[0] + 32) * 4) for w, _, _ in mats]
    outs = []
    try:
        for b, (w, s, key) in zip(yb, mats):
            n = S * w.shape[0]
            b.upload(np.full(n + 32, 7.0, np.float32))
            moe.matmul_fp8_dev(b.ptr, xb.ptr, S, I, w.shape[0], key)
            assert hip.colizig_hip_sync() == 0
            y = b.download(np.empty(n + 32, np.float32))
            assert (y[n:] == 7.0).all()
            outs.append(y[:n].reshape(S, -1).copy())
        moe.matmul_fp8_dev_multi([b.ptr for b in yb], xb.ptr, S, I, [w.shape[0] for w, _, _ in mats],
                                 [k for _, _, k in mats])
        assert hip.colizig_hip_sync() == 0
        for b, o in zip(yb, outs):
            y = b.download(np.empty(o.size + 32, np.float32))[:o.size].reshape(o.shape)
            assert np.array_equal(f32_bits(y), f32_bits(o))
    finally:
        xb.free()
        for b in yb:
            b.free()
    return outs


@pytest.mark.parametrize("S,I,Os", [(16, 2048, (4096, 512, 512)), (31, 128, (130, 7)), (33, 384, (300,)),
                                    (64, 896, (65, 256, 1)), (385, 512, (4097, 2048)), (97, 4096, (2048,)),
                                    (1, 2048, (512,)), (12, 2048, (512,)), (200, 768, (2048,)), (513, 512, (300, 64)),
                                    (14, 2048, (200, 70)), (15, 2048, (70,)), (8, 4096, (70,)), (9, 5120, (70,)),
                                    (128, 512, (130,)), (129, 512, (130,)), (512, 384, (130,))])
def test_many_tokens_f32_accuracy(gpu, S, I, Os):
    print(f"f32x S={S} I={I} O={Os}", flush=True)
    rng = np.random.default_rng(S * 7 + I)
    moe.set_vram_budget(1 << 30)
    try:
        x = rng.normal(size=(S, I)).astype(np.float32)
        x *= (10.0 ** rng.integers(-12, 12, size=(S, 1))).astype(np.float32)  # rows far apart
        x[:, 5] *= 1e-4  # small beside large in one K block
        mats = []
        for m, O in enumerate(Os):
            w, s = synth.block_quantize(rng.normal(0, 0.02, size=(O, I)).astype(np.float32))
            key = moe.Fp8Matrix.expert_key(60 + m, (S + I + O) % 509, 1)
            moe.matrix_load(key, w, s)
            mats.append((w, s, key))
        for (w, s, _), y in zip(mats, _run(x, mats, I)):
            x64, wd = x.astype(np.float64), _dequant(w, s)
            # against the terms' own size, so that a sum that cancels is not held to its small rest
            err = np.linalg.norm(y - x64 @ wd.T, axis=1) / np.sqrt(((x64 ** 2) @ (wd ** 2).T).sum(1))
            print(f"  {w.shape}: worst row {err.max():.2e}", flush=True)
            assert np.sqrt((err ** 2).mean()) < RTOL
    finally:
        moe.set_vram_budget(0)


@pytest.mark.parametrize("S,I", [(2, 16384), (7, 14336), (7, 4096), (8, 5120), (13, 2048), (15, 3072), (15, 1024)])
def test_fewer_tokens_keep_the_gemv(gpu, S, I):
    """Below the products' rule the GEMV runs: a token's row has the bits it has
    alone (the products sum in another order)."""
    rng = np.random.default_rng(S + I)
    O = 70
    moe.set_vram_budget(1 << 30)
    try:
        w, s = synth.block_quantize(rng.normal(0, 0.02, size=(O, I)).astype(np.float32))
        key = moe.Fp8Matrix.expert_key(73, I % 507, 1)
        moe.matrix_load(key, w, s)
        x = rng.normal(size=(S, I)).astype(np.float32)
        y = _run(x, [(w, s, key)], I)[0]
        one = np.concatenate([_run(x[t:t + 1], [(w, s, key)], I)[0] for t in range(S)])
        assert np.array_equal(f32_bits(y), f32_bits(one))
    finally:
        moe.set_vram_budget(0)


@pytest.mark.parametrize("S", [16, 40, 129, 513])
def test_extreme_values(gpu, S):
    """Infinities, NaN, zero rows, the largest and smallest floats, a NaN
    weight and a zero scale: what f32 sums of the same products give."""
    rng = np.random.default_rng(S)
    I, O = 256, 96
    moe.set_vram_budget(1 << 30)
    try:
        w, s = synth.block_quantize(np.abs(rng.normal(0, 0.02, size=(O, I))).astype(np.float32) + 0.01)
        w[3, 200] = 0x7F  # NaN
        x = np.abs(rng.normal(size=(S, I))).astype(np.float32)
        x[0, 7] = np.inf
        x[1, 7] = -np.inf
        x[2, 9], x[2, 140] = np.inf, -np.inf
        x[3, 9] = np.nan
        x[4] = 0.0
        x[5] = 1e-38
        x[6] = 3e33  # times 448 and summed: still finite before the block scale, as in f32 sums
        x[7, 3], x[7, 4] = np.inf, 3e33  # a large finite value beside an infinity stays finite
        key = moe.Fp8Matrix.expert_key(70, S, 1)
        moe.matrix_load(key, w, s)
        y = _run(x, [(w, s, key)], I)[0]
        with np.errstate(all="ignore"):
            ref = np.stack([(x.astype(np.float64)[t] * _dequant(w, s)).sum(1) for t in range(S)]).astype(np.float32)
        assert np.array_equal(np.isnan(y), np.isnan(ref))
        fin = np.isfinite(ref)
        assert np.array_equal(y[~fin & ~np.isnan(ref)], ref[~fin & ~np.isnan(ref)])
        # all terms of one sign: no cancellation
        assert (np.abs(y[fin] - ref[fin]) <= 2e-6 * np.abs(ref[fin]) + 1e-44).all()
    finally:
        moe.set_vram_budget(0)


@pytest.mark.parametrize("S,I", [(16, 2048), (129, 512), (513, 384), (24, 896)])
def test_small_elements_beside_large_ones(gpu, S, I):
    """Each row's 128-column blocks hold one element 1e6 to 1e30 times the
    rest, whose weights are zero: the result is the rest's, with all of their
    bits, as f32 sums give it.  Rows of the smallest floats keep theirs too."""
    rng = np.random.default_rng(S + I)
    O = 200
    moe.set_vram_budget(1 << 30)
    try:
        w, s = synth.block_quantize(rng.normal(0, 0.02, size=(O, I)).astype(np.float32))
        w[:, 5::128] = 0
        x = rng.normal(size=(S, I)).astype(np.float32)
        ratio = 10.0 ** np.array([6, 8, 10, 15, 20, 30])[np.arange(S) % 6]
        x[:, 5::128] = ratio[:, None] * rng.choice([-1.0, 1.0], size=(S, len(range(5, I, 128))))
        tiny = np.arange(S) % 8 == 7
        x[tiny] = 1e-37 * rng.normal(size=(int(tiny.sum()), I))  # down to subnormals; none beside them
        key = moe.Fp8Matrix.expert_key(71, S % 500, 1)
        moe.matrix_load(key, w, s)
        y = _run(x, [(w, s, key)], I)[0]
        ref = x.astype(np.float64) @ _dequant(w, s).T
        err = np.linalg.norm(y - ref, axis=1) / np.linalg.norm(ref, axis=1)
        print(f"small beside large S={S} I={I}: worst row {err.max():.2e}", flush=True)
        assert err[~tiny].max() < RTOL
        assert err[tiny].max() < 1e-6  # results near 5e-38, whose last place is 2^-149, besides
    finally:
        moe.set_vram_budget(0)


@pytest.mark.parametrize("S", [16, 129, 513])
def test_rows_do_not_depend_on_each_other(gpu, S):
    """Rows that take the large rows' path leave the bits of the others."""
    rng = np.random.default_rng(S)
    I, O = 384, 130
    moe.set_vram_budget(1 << 30)
    try:
        w, s = synth.block_quantize(rng.normal(0, 0.02, size=(O, I)).astype(np.float32))
        key = moe.Fp8Matrix.expert_key(74, S % 500, 1)
        moe.matrix_load(key, w, s)
        x = rng.normal(size=(S, I)).astype(np.float32)
        y = _run(x, [(w, s, key)], I)[0]
        odd = x.copy()
        odd[1, 3], odd[4, 300], odd[9], odd[S - 1, 130] = np.inf, np.nan, 3e38, -2e33
        z = _run(odd, [(w, s, key)], I)[0]
        same = np.setdiff1d(np.arange(S), [1, 4, 9, S - 1])
        assert np.array_equal(f32_bits(y[same]), f32_bits(z[same]))
    finally:
        moe.set_vram_budget(0)


@pytest.mark.parametrize("S", [16, 129, 513])
@pytest.mark.parametrize("I", [256, 384])
def test_largest_floats(gpu, S, I):
    """Rows whose products with the weights' bytes pass the largest float
    where those with the scaled weights, the result's terms, do not."""
    rng = np.random.default_rng(S + I)
    O = 130
    moe.set_vram_budget(1 << 30)
    try:
        w, s = synth.block_quantize(np.abs(rng.normal(0, 0.02, size=(O, I))).astype(np.float32) + 0.01)
        x = np.abs(rng.normal(size=(S, I))).astype(np.float32)
        x[0] = 3e37
        x[3] = 1e36 * (1 + x[3])
        x[S - 1, ::2] = 2e36
        x[5] = 3.4e38  # its result does pass it
        key = moe.Fp8Matrix.expert_key(72, S + I % 3, 1)
        moe.matrix_load(key, w, s)
        y = _run(x, [(w, s, key)], I)[0]
        with np.errstate(all="ignore"):
            ref = (x.astype(np.float64) @ _dequant(w, s).T).astype(np.float32)
        assert np.isfinite(ref[:5]).all() and np.isinf(ref[5]).any()
        near = np.abs(ref) > 3.3e38  # on either side of the limit
        assert np.array_equal(np.isinf(y) | near, np.isinf(ref) | near) and not np.isnan(y).any()
        fin = np.isfinite(ref) & ~near
        assert (np.abs(y[fin] - ref[fin]) <= 2e-6 * np.abs(ref[fin])).all()
    finally:
        moe.set_vram_budget(0)


@pytest.mark.parametrize("H,E,K,I,SI,S", [(256, 16, 8, 128, 0, 1025), (512, 24, 10, 256, 0, 900),
                                          (256, 64, 16, 384, 256, 600)])
def test_layer_past_8192_slots(gpu, H, E, K, I, SI, S):
    print(f"layer H={H} E={E} K={K} I={I} SI={SI} S={S}", flush=True)
    host = synth.make_layer(H, E, K, I, SI, True, seed=S)
    L = moe.register_layer(0, host)
    x = synth.hidden_states(S, H, seed=S)
    assert _lib.hip().colizig_hip_usage_reset() == 0
    out, idx, gates = L.forward(x)
    ro, ri, rg = orc.OracleLayer(host).forward(x)
    assert np.array_equal(idx, ri)
    assert np.array_equal(f32_bits(gates), f32_bits(rg))
    err = rel_l2(out, ro)
    print(f"  rel L2 {err:.2e}", flush=True)
    assert err < 1.5e-6  # three such products, silu, the oracle's own f32 sums
    counts = np.zeros((1, E), np.uint64)
    assert _lib.hip().colizig_hip_usage_read(0, 1, E, counts.ctypes.data) == 0
    assert np.array_equal(counts[0], np.bincount(ri.ravel(), minlength=E).astype(np.uint64))
