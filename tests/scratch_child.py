"""Child process of tests/test_gpu_scratch_limit.py: in a fresh library state
whose scratch buffers are refused above a limit, a chain of a top-4 layer (at
1100 tokens under 8192 slots) and a top-8 layer (past them, its O rows
refused), eager and as a graph, and large and small calls in turn.  Prints one
JSON line."""
from __future__ import annotations

import ctypes
import json
import os
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

from colizig_amd import _lib, moe, synth  # noqa: E402
from oracle import oracle as orc  # noqa: E402
from tests.helpers import f32_bits, rel_l2  # noqa: E402

H, E, I, S, EPS = 256, 16, 128, 1100, 1e-6
LIMIT = 6 << 20  # top-4's O rows 4.5 MB, top-8's 9.0 MB (16.8 as a step)


def held(hip) -> int:
    b = ctypes.c_uint64(0)
    assert hip.colizig_hip_work_bytes(ctypes.byref(b)) == 0
    return b.value


def main() -> None:
    moe.init()
    hip = _lib.hip()
    assert hip.colizig_hip_set_scratch_limit(LIMIT) == 0
    hosts = [synth.make_layer(H, E, K, I, 0, True, seed=5 + K) for K in (4, 8)]
    layers = [moe.register_layer(l, h) for l, h in enumerate(hosts)]
    x0 = synth.hidden_states(S, H, seed=9)
    want = x0.copy()
    for h in hosts:
        orc.OracleLayer(h).chain(want, EPS)
    xb = moe.DeviceBuffer(x0.nbytes)
    res = {}

    def chain() -> np.ndarray:
        xb.upload(x0)
        assert hip.colizig_hip_chain_decode(0, 2, xb.ptr, S, EPS, None, None, None, None) == 0, _lib.last_error()
        assert hip.colizig_hip_sync() == 0
        return xb.download(np.empty_like(x0))

    def graph() -> np.ndarray:
        g = hip.colizig_hip_chain_graph_create(0, 2, xb.ptr, S, EPS)
        assert g > 0, _lib.last_error()
        for _ in range(3):
            xb.upload(x0)
            assert hip.colizig_hip_graph_launch(g, None) == 0, _lib.last_error()
            assert hip.colizig_hip_sync() == 0
        hip.colizig_hip_graph_destroy(g)
        return xb.download(np.empty_like(x0))

    eager = chain()
    res["limited"] = rel_l2(eager, want)
    res["limited_graph_same"] = bool(np.array_equal(f32_bits(graph()), f32_bits(eager)))
    # large and small calls in turn hold what they held
    xs = synth.hidden_states(S, H, seed=10)
    layers[1].forward(xs)
    layers[1].forward(xs[:500])
    before = held(hip)
    outs = []
    for _ in range(4):
        outs.append((layers[1].forward(xs)[0], layers[1].forward(xs[:500])[0]))
    res["held_grew"] = held(hip) - before
    res["repeat_same"] = all(np.array_equal(f32_bits(a), f32_bits(b)) for o in outs[1:] for a, b in zip(o, outs[0]))
    res["fallback"] = rel_l2(outs[0][0], orc.OracleLayer(hosts[1]).forward(xs)[0])
    # with room: the grouped products
    assert hip.colizig_hip_set_scratch_limit(0) == LIMIT
    eager = chain()
    res["full"] = rel_l2(eager, want)
    res["full_graph_same"] = bool(np.array_equal(f32_bits(graph()), f32_bits(eager)))
    res["grown"] = held(hip) - before
    wide = layers[1].forward(xs)[0]
    res["wide"] = rel_l2(wide, orc.OracleLayer(hosts[1]).forward(xs)[0])
    res["route_changed"] = bool(not np.array_equal(f32_bits(wide), f32_bits(outs[0][0])))
    xb.free()
    print(json.dumps(res), flush=True)


if __name__ == "__main__":
    main()
