"""The slab kernel (n = 6: one launch, x read once) at the sizes where it can go
wrong, against the CPU oracle at the tolerances of tests/helpers.py."""
from __future__ import annotations

import os

import numpy as np
import pytest

from inputs import to_bits
from test_gpu_parity import _say, check, fetch, run_gpu, to_device

pytestmark = pytest.mark.gpu

N = 6


def _inputs(T, D, is_bf16, has_gamma, seed=0):
    rng = np.random.default_rng(6000 + 17 * T + D + seed)
    K, M = N * D, N * N + 2 * N
    xf = rng.standard_normal((T, N, D)).astype(np.float32)
    xf[::7] *= 50.0  # large rows exercise the RMS scale
    phi = (rng.standard_normal((M, K)) / np.sqrt(K)).astype(np.float32)
    alpha = np.asarray([0.3, -0.2, 0.05], dtype=np.float32)
    bias = rng.uniform(-0.5, 0.5, M).astype(np.float32)
    gamma = (1 + 0.1 * rng.standard_normal(K)).astype(np.float32) if has_gamma else None
    return to_bits(xf, is_bf16), phi, alpha, bias, gamma


@pytest.mark.parametrize("T,D,is_bf16,has_gamma", [
    (1, 16, True, True),        # one row, one slice of 16 columns
    (16, 128, False, False),    # one whole tile of one whole slice
    (17, 144, True, False),     # a second slice of 16 columns, a second tile of one row
    (63, 1024, False, True),    # fewer tiles than teams
    (2065, 1040, True, True),   # several own steps, ragged rows and columns
    (1000, 2000, False, False), # teams across XCDs, D % 64 == 16
    (4100, 256, True, True),    # more tiles per team than ring slots
    (200, 8192, True, False),   # 64 slices
])
def test_slab_shapes(pkg, orc, device, T, D, is_bf16, has_gamma):
    x, phi, alpha, bias, gamma = _inputs(T, D, is_bf16, has_gamma)
    _say(f"[slab] T={T} D={D} bf16={is_bf16} gamma={has_gamma}")
    out = run_gpu(pkg, device, x, is_bf16, phi, alpha, bias, gamma, force_path="slab", kernel="slab")
    check(out, orc.mhc_pre(x, is_bf16, phi, alpha, bias, gamma), x, is_bf16, orc)


@pytest.mark.parametrize("geometry", ["8,3,1", "8,2,4", "1,25,2", "1,3,8"])
def test_slab_geometries_agree(pkg, orc, device, geometry):
    """Teams inside an XCD and across, one and several reducer workgroups: the
    sums over a team's slices have one order, so every division of the device
    gives the same bits."""
    T, D = 1500, 1024
    x, phi, alpha, bias, gamma = _inputs(T, D, True, True)
    want = run_gpu(pkg, device, x, True, phi, alpha, bias, gamma, force_path="slab", kernel="slab")
    os.environ["MHCPRE_SLAB"] = geometry
    try:
        got = run_gpu(pkg, device, x, True, phi, alpha, bias, gamma, force_path="slab", kernel="slab")
    finally:
        os.environ.pop("MHCPRE_SLAB", None)
    check(got, orc.mhc_pre(x, True, phi, alpha, bias, gamma), x, True, orc)
    for k in ("h_in", "h_post", "h_res", "h_pre"):
        assert np.array_equal(got[k], want[k]), k


@pytest.mark.parametrize("T,D,is_bf16", [(700, 1040, True), (1100, 1024, False)])
def test_slab_prepared_matches_plain(pkg, orc, device, T, D, is_bf16):
    x, phi, alpha, bias, gamma = _inputs(T, D, is_bf16, True)
    xt, pt, at, bt, gt = to_device(pkg, device, x, is_bf16, phi, alpha, bias, gamma)
    weights = pkg.MhcPreWeights(pt, gt, N)
    os.environ["MHCPRE_FORCE_PATH"] = "slab"
    try:
        plain = pkg.MhcPreOp(xt, pt, at, bt, gt, h_pre=True)
        prep = pkg.MhcPreOp(xt, None, at, bt, None, h_pre=True, weights=weights)
    finally:
        os.environ.pop("MHCPRE_FORCE_PATH", None)
    plain.launch(check=True)
    prep.launch(check=True)
    assert plain.kernel == "slab" and prep.kernel == "slab"
    a, b = fetch(plain), fetch(prep)
    check(a, orc.mhc_pre(x, is_bf16, phi, alpha, bias, gamma), x, is_bf16, orc)
    for k in a:
        assert np.array_equal(a[k], b[k]), k
    plain.close()
    prep.close()


@pytest.mark.parametrize("knob", ["MHCPRE_SPIN_LIMIT=0", "MHCPRE_SPIN_EVERY=5"])
@pytest.mark.parametrize("T,D,is_bf16,prepared", [(300, 528, True, False), (90, 1024, True, True),
                                                 (700, 1200, False, False), (170, 400, False, True)])
def test_slab_expired_waits_are_computed(pkg, orc, device, T, D, is_bf16, prepared, knob):
    """A spin limit of 0, in all or every fifth workgroup, makes every wait that
    does not find its data at once expire: the workgroups then compute what they
    waited for in the order of the exchange (the same bits), it is no error, and
    the next launch on the workspace is clean."""
    x, phi, alpha, bias, gamma = _inputs(T, D, is_bf16, True)
    xt, pt, at, bt, gt = to_device(pkg, device, x, is_bf16, phi, alpha, bias, gamma)
    weights = pkg.MhcPreWeights(pt, gt, N) if prepared else None
    args = (xt, None, at, bt, None) if prepared else (xt, pt, at, bt, gt)
    os.environ["MHCPRE_FORCE_PATH"] = "slab"
    name, value = knob.split("=")
    os.environ[name] = value
    try:
        hurried = pkg.MhcPreOp(*args, h_pre=True, weights=weights)
        os.environ.pop(name)
        calm = pkg.MhcPreOp(*args, h_pre=True, weights=weights, workspace=hurried.workspace)
    finally:
        os.environ.pop("MHCPRE_FORCE_PATH", None)
        os.environ.pop(name, None)
    calm.launch(check=True)
    want = fetch(calm)
    check(want, orc.mhc_pre(x, is_bf16, phi, alpha, bias, gamma), x, is_bf16, orc)
    for op in (hurried, calm, hurried):
        for t in op.outputs():
            t.fill_(float("nan"))
        _say(f"[slab] T={T} D={D} {'calm' if op is calm else knob}")
        op.launch(check=True)
        assert op.kernel == "slab" and (op.computed_waits() or op is calm)
        got = fetch(op)
        for k in got:
            assert np.array_equal(got[k], want[k]), k
    hurried.close()
    calm.close()


def test_slab_graph_replays(pkg, orc, device):
    """Replays of a captured launch with new x between them: each counts itself
    into the exchange's tags, so no replay takes an earlier one's words."""
    import torch

    T, D = 1200, 1024
    x, phi, alpha, bias, gamma = _inputs(T, D, True, True)
    xs = [_inputs(T, D, True, True, seed=i)[0] for i in range(3)]
    xt, pt, at, bt, gt = to_device(pkg, device, x, True, phi, alpha, bias, gamma)
    op = pkg.MhcPreOp(xt, pt, at, bt, gt, h_pre=True)
    op.launch(check=True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        op.launch()
    for i in (1, 2, 0, 1):
        xt.copy_(torch.from_numpy(xs[i].view(np.int16)).to(device).view(torch.bfloat16))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert op.kernel == "slab"
        replayed = fetch(op)
        check(replayed, orc.mhc_pre(xs[i], True, phi, alpha, bias, gamma), xs[i], True, orc)
        op.launch(check=True)
        eager = fetch(op)
        for k in replayed:
            assert np.array_equal(replayed[k], eager[k]), (i, k)
    del graph
    op.close()
