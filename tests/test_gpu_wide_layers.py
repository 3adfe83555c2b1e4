"""Layers past 8192 slots (tokens x top-k) through the grouped products at f32
accuracy, where the plain forward is not the caller: chains and their graphs
(RMS rows, residual, the combine that forms the next layer's rows), a chain
with a smaller layer between, BF16 routers and native shared experts, the
streaming tier, both prefill modes, and the slot counts at which the regime
begins and ends.

Bounds: 1.5e-6 for one layer (three products, silu, the oracle's own f32 sums),
1e-3 wherever a layer of at most 8192 slots takes part."""
from __future__ import annotations

import numpy as np
import pytest

from colizig_amd import _lib, moe, synth
from tests.helpers import f32_bits, rel_l2

pytestmark = pytest.mark.gpu

H, E, I, EPS = 256, 16, 128, 1e-6
RTOL = 1.5e-6


def _chain(base, n, x0, graph=False):
    hip = _lib.hip()
    S = x0.shape[0]
    xb = moe.DeviceBuffer(x0.nbytes)
    try:
        if not graph:
            xb.upload(x0)
            assert hip.colizig_hip_chain_decode(base, n, xb.ptr, S, EPS, None, None, None, None) == 0, _lib.last_error()
            assert hip.colizig_hip_sync() == 0
            return xb.download(np.empty_like(x0))
        g = hip.colizig_hip_chain_graph_create(base, n, xb.ptr, S, EPS)
        assert g > 0, _lib.last_error()
        outs = []
        for _ in range(3):
            xb.upload(x0)
            assert hip.colizig_hip_graph_launch(g, None) == 0, _lib.last_error()
            assert hip.colizig_hip_sync() == 0
            outs.append(xb.download(np.empty_like(x0)))
            _chain(base, n, x0[:20])  # eager work of another size between the replays
        hip.colizig_hip_graph_destroy(g)
        assert all(np.array_equal(f32_bits(o), f32_bits(outs[0])) for o in outs)
        return outs[0]
    finally:
        xb.free()


@pytest.mark.parametrize("ks,SI", [((8, 8, 8), 0), ((8, 8), 256), ((8, 4, 8), 0)])
def test_chains(gpu, oracle_lib, ks, SI):
    """1100 tokens: 8800 slots with top-8, 4400 with top-4."""
    S, base = 1100, 6000
    hosts = [synth.make_layer(H, E, K, I, SI, True, seed=31 + 7 * l) for l, K in enumerate(ks)]
    for l, h in enumerate(hosts):
        moe.register_layer(base + l, h)
    x0 = synth.hidden_states(S, H, seed=len(ks) + SI)
    want = x0.copy()
    for h in hosts:
        oracle_lib.OracleLayer(h).chain(want, EPS)
    for mode in (1, 0):
        prev = _lib.hip().colizig_hip_set_prefill_fp8(mode)
        try:
            got = _chain(base, len(ks), x0)
            # of what the layers add (the stream itself rounds to 2^-25 of x, about 20 times larger)
            err = rel_l2(got - x0, want - x0)
            print(f"chain {ks} SI={SI} mode {mode}: rel L2 {err:.2e}", flush=True)
            assert err < (1e-5 if min(ks) == 8 else 1e-3)
            assert np.array_equal(f32_bits(_chain(base, len(ks), x0, graph=True)), f32_bits(got))
        finally:
            _lib.hip().colizig_hip_set_prefill_fp8(prev)


@pytest.mark.parametrize("router_bf16,shared", [(True, None), (False, "bf16"), (True, "f32")])
def test_native_weights(gpu, oracle_lib, router_bf16, shared):
    S, K, SI = 1030, 8, 256 if shared else 0
    host = synth.with_native(synth.make_layer(H, E, K, I, SI, True, seed=41), seed=42, router_bf16=router_bf16,
                             shared=shared)
    L = moe.register_layer(6010, host)
    O = oracle_lib.OracleLayer(host)
    x = synth.hidden_states(S, H, seed=43)
    out, idx, gates = L.forward(x)
    ro, ri, rg = O.forward(x)
    assert np.array_equal(idx, ri) and np.array_equal(f32_bits(gates), f32_bits(rg))
    err = rel_l2(out, ro)
    print(f"native router {router_bf16} shared {shared}: rel L2 {err:.2e}", flush=True)
    assert err < RTOL
    want = x.copy()
    O.chain(want, EPS)
    assert rel_l2(_chain(6010, 1, x), want) < RTOL


def test_streamed_equals_resident(gpu):
    S, K = 1030, 8
    d = moe.dims(H, E, K, I)
    host = synth.make_layer(H, E, K, I, 0, True, seed=51)
    moe.stream_pool_init(d, E * (3 * I * H + 3 * moe.nblk(I) * moe.nblk(H) * 4 + 16))
    try:
        res, strm = moe.register_layer(6020, host), moe.register_layer(6021, host)
        wb, sb = moe.host_expert_slab(d, host["experts"])
        moe.stream_layer_from_host(6021, wb, sb)
        x = synth.hidden_states(S, H, seed=52)
        a, b = res.forward(x), strm.forward(x)
        for p, q in zip(a, b):
            assert np.array_equal(p.view(np.uint32), q.view(np.uint32))
    finally:
        moe.stream_pool_free()


def test_prefill_mode_has_no_effect(gpu):
    host = synth.make_layer(H, E, 8, I, 256, True, seed=61)
    L = moe.register_layer(6030, host)
    x = synth.hidden_states(1025, H, seed=62)
    outs = []
    for mode in (1, 0):
        prev = _lib.hip().colizig_hip_set_prefill_fp8(mode)
        try:
            outs.append(L.forward(x)[0])
        finally:
            _lib.hip().colizig_hip_set_prefill_fp8(prev)
    assert np.array_equal(f32_bits(outs[0]), f32_bits(outs[1]))


@pytest.mark.parametrize("K,S", [(1, 8192), (1, 8193), (16, 512), (16, 513), (1, 65535), (1, 65536), (1, 65537)])
def test_slot_limits(gpu, oracle_lib, K, S):
    """Up to 8192 slots the default mode's three E4M3 terms, then f32 accuracy;
    past 65,536 the per-token kernels.  64 rows of each against the oracle."""
    host = synth.make_layer(H, E if K > 1 else 4, K, I, 0, True, seed=71)
    L = moe.register_layer(6040, host)
    x = synth.hidden_states(S, H, seed=72)
    out, idx, gates = L.forward(x)
    rows = np.unique(np.concatenate([np.arange(16), S - 1 - np.arange(16), np.linspace(0, S - 1, 32).astype(int)]))
    ro, ri, rg = oracle_lib.OracleLayer(host).forward(x[rows])
    assert np.array_equal(idx[rows], ri) and np.array_equal(f32_bits(gates[rows]), f32_bits(rg))
    err = rel_l2(out[rows], ro)
    print(f"K={K} S={S}: rel L2 {err:.2e}", flush=True)
    assert err < (2e-4 if S * K <= 8192 else RTOL)


def test_small_elements_beside_large_ones(gpu, oracle_lib):
    """An element 1e4 to 1e10 times the rest whose weights are zero: the rest
    keep all of their bits."""
    S, K = 1030, 8
    host = synth.make_layer(H, E, K, I, 0, True, seed=81)
    cols = [9, 150]
    host["router"][:, cols] = 0.0
    for e in host["experts"]:
        e["gate_w"][:, cols] = 0
        e["up_w"][:, cols] = 0
    L = moe.register_layer(6050, host)
    x = synth.hidden_states(S, H, seed=82)
    x[:, cols] = (10.0 ** np.array([4, 6, 8, 10])[np.arange(S) % 4])[:, None]
    out, idx, _ = L.forward(x)
    ro, ri, _ = oracle_lib.OracleLayer(host).forward(x)
    assert np.array_equal(idx, ri)
    err = np.linalg.norm(out - ro, axis=1) / np.linalg.norm(ro, axis=1)
    print(f"small beside large: worst row {err.max():.2e}", flush=True)
    assert err.max() < 2 * RTOL
