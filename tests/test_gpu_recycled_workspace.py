"""A workspace whose words other memory users have rewritten between launches:
an exchange may take nothing from an earlier launch, whatever the header holds.

The eager operator's workspace comes from the caching allocator on each call,
and a captured one's is reused by other tensors of the graph, so the head of a
workspace may hold the same bytes before two launches while the records further
on are still those of the first."""
from __future__ import annotations

import os

import numpy as np
import pytest

from inputs import to_bits
from test_gpu_parity import _say, check, fetch, to_device

pytestmark = pytest.mark.gpu

HEADER = 256 + 4 * 2048  # bytes of the workspace in front of a path's own layout


def _setup(pkg, device, force, n, T, D):
    rng = np.random.default_rng(7000 + n + T + D)
    K, M = n * D, n * n + 2 * n
    xs = [to_bits(rng.standard_normal((T, n, D)).astype(np.float32) * (1 + 2 * i), True) for i in range(4)]
    phi = (rng.standard_normal((M, K)) / np.sqrt(K)).astype(np.float32)
    alpha = np.asarray([0.3, -0.2, 0.05], dtype=np.float32)
    bias = rng.uniform(-0.5, 0.5, M).astype(np.float32)
    gamma = (1 + 0.1 * rng.standard_normal(K)).astype(np.float32)
    args = to_device(pkg, device, xs[0], True, phi, alpha, bias, gamma)
    os.environ["MHCPRE_FORCE_PATH"] = force
    try:
        op = pkg.MhcPreOp(*args, h_pre=True)
    finally:
        os.environ.pop("MHCPRE_FORCE_PATH", None)
    return xs, (phi, alpha, bias, gamma), args[0], op


@pytest.mark.parametrize("captured", [False, True])
@pytest.mark.parametrize("force,n,T,D", [
    ("cell", 4, 128, 256), ("cell", 8, 40, 1024), ("slab", 6, 300, 1024), ("strip", 4, 300, 1200),
    ("strip", 4, 300, 2048), ("fused", 4, 300, 1024),
])
def test_header_restored_between_launches(pkg, orc, device, force, n, T, D, captured):
    """Every launch finds the header as the first one found it and the rest of
    the workspace as the launch before left it."""
    import torch

    xs, weights, xt, op = _setup(pkg, device, force, n, T, D)
    _say(f"[recycled] {force} n={n} T={T} D={D} captured={captured}")
    head = op.workspace[:HEADER]
    before = torch.zeros_like(head)
    before[64:68] = 7
    launch = op.launch
    if captured:
        op.launch()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            op.launch()
        launch = graph.replay
    exchanged = 0
    for r, x in enumerate(xs):
        xt.copy_(torch.from_numpy(x.view(np.int16)).to(device).view(torch.bfloat16))
        head.copy_(before)
        for t in op.outputs():
            t.fill_(float("nan"))
        torch.cuda.synchronize()
        launch()
        torch.cuda.synchronize()
        _say(f"  launch {r}")
        assert op.device_status() == 0 and op.kernel == force
        exchanged += not op.computed_waits()
        check(fetch(op), orc.mhc_pre(x, True, *weights), x, True, orc)
    assert exchanged >= len(xs) - 1  # (a device held up once may have had its waits computed)
    op.close()


def _nodes(graph):
    import ctypes

    hip = ctypes.CDLL("libamdhip64.so")
    count = ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(count)) == 0
    return count.value


def test_captured_launches_share_out_the_replay_words(pkg, orc, device):
    """A captured launch counts its replays in words that its graph owns; with
    none left (MHCPRE_REPLAY_WORDS, a test knob) a node sets words of the
    workspace instead, and a graph's end gives its words back."""
    import time

    import torch

    T, D = 100, 208  # 7 row tiles, 4 slices, 2 column tiles: no other test's grid
    xs, weights, xt, op = _setup(pkg, device, "cell", 4, T, D)

    def capture():
        graph = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(graph):
            op.launch()
        return graph

    def replay(graph):
        for r, x in enumerate(xs):
            xt.copy_(torch.from_numpy(x.view(np.int16)).to(device).view(torch.bfloat16))
            op.workspace[:HEADER] = 0
            for t in op.outputs():
                t.fill_(float("nan"))
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            check(fetch(op), orc.mhc_pre(x, True, *weights), x, True, orc)

    op.launch()
    torch.cuda.synchronize()
    os.environ["MHCPRE_REPLAY_WORDS"] = "0"
    try:
        none = capture()
        assert _nodes(none) == 2
        _say("[recycled] words of the workspace")
        replay(none)
    finally:
        os.environ.pop("MHCPRE_REPLAY_WORDS", None)
    own, other = capture(), capture()
    assert _nodes(own) == 1 and _nodes(other) == 1
    _say("[recycled] words of the library")
    replay(own)
    replay(other)
    replay(own)
    own.reset()
    del own
    time.sleep(2.5)  # blocks are handed out again two seconds after their return
    os.environ["MHCPRE_REPLAY_WORDS"] = "0"
    try:
        again, more = capture(), capture()
    finally:
        os.environ.pop("MHCPRE_REPLAY_WORDS", None)
    assert _nodes(again) == 1 and _nodes(more) == 2
    _say("[recycled] words given back")
    replay(again)
    replay(other)
    replay(more)
    op.close()
