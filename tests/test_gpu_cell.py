"""The cell kernel (small batches of every n and path, in place of the path's
kernels), against the CPU oracle at the tolerances of tests/helpers.py."""
from __future__ import annotations

import os

import numpy as np
import pytest

from inputs import to_bits
from test_gpu_parity import _say, check, fetch, run_gpu, to_device

pytestmark = pytest.mark.gpu


def _inputs(n, T, D, is_bf16, has_gamma):
    rng = np.random.default_rng(5000 + 17 * T + D + n)
    K, M = n * D, n * n + 2 * n
    xf = rng.standard_normal((T, n, D)).astype(np.float32)
    xf[::7] *= 50.0  # large rows exercise the RMS scale
    phi = (rng.standard_normal((M, K)) / np.sqrt(K)).astype(np.float32)
    alpha = np.asarray([0.3, -0.2, 0.05], dtype=np.float32)
    bias = rng.uniform(-0.5, 0.5, M).astype(np.float32)
    gamma = (1 + 0.1 * rng.standard_normal(K)).astype(np.float32) if has_gamma else None
    return to_bits(xf, is_bf16), phi, alpha, bias, gamma


@pytest.mark.parametrize("n,T,D,is_bf16,has_gamma,path,kernel", [
    (4, 1, 16, True, True, "split", "cell"),       # one slice, a quarter of a strip
    (4, 33, 256, False, False, "rows", "cell"),    # 4 narrow slices, three row tiles
    (4, 512, 1024, True, True, "strip", "cell"),   # the largest grid: two workgroups per CU
    (4, 17, 8192, False, True, "rows", "cell"),    # 64 slices
    (4, 100, 1200, True, False, "split", "cell"),  # D % 64 == 48, wide slices
    (6, 5, 80, True, True, "split", "cell"),       # streams that start in mid k-step
    (6, 130, 2560, False, True, "rows", "rows"),   # more workgroups than are resident: the path's kernels
    (6, 112, 2560, True, True, "rows", "cell"),    # two workgroups per CU
    (6, 31, 7168, True, False, "rows", "cell"),
    (8, 16, 16, False, True, "rows", "cell"),
    (8, 250, 496, True, True, "rows", "cell"),
    (8, 9, 3056, True, False, "rows", "cell"),     # wide slices, the last 112 columns
])
def test_cell(pkg, orc, device, n, T, D, is_bf16, has_gamma, path, kernel):
    x, phi, alpha, bias, gamma = _inputs(n, T, D, is_bf16, has_gamma)
    _say(f"[cell] n={n} T={T} D={D} bf16={is_bf16} gamma={has_gamma}")
    ref = orc.mhc_pre(x, is_bf16, phi, alpha, bias, gamma)
    plain = run_gpu(pkg, device, x, is_bf16, phi, alpha, bias, gamma, force_path="cell",
                    kernel=kernel)
    os.environ["MHCPRE_FORCE_PATH"] = "cell"
    try:
        xt, pt, at, bt, gt = to_device(pkg, device, x, is_bf16, phi, alpha, bias, gamma)
        op = pkg.MhcPreOp(xt, None, at, bt, None, h_pre=True, weights=pkg.MhcPreWeights(pt, gt, n))
    finally:
        os.environ.pop("MHCPRE_FORCE_PATH", None)
    assert plain.pop("path") == path
    check(plain, ref, x, is_bf16, orc)
    op.launch(check=True)  # prepared weights: the same bits
    assert op.kernel == kernel
    got = fetch(op)
    for k in plain:
        assert np.array_equal(got[k], plain[k]), k
    op.close()


@pytest.mark.parametrize("knob", ["MHCPRE_SPIN_LIMIT=0", "MHCPRE_SPIN_EVERY=1", "MHCPRE_SPIN_EVERY=3"])
@pytest.mark.parametrize("n,T,D,prepared", [(4, 40, 256, False), (6, 20, 528, True), (8, 19, 304, False)])
def test_expired_waits_are_computed(pkg, orc, device, n, T, D, prepared, knob):
    """A spin limit of 0 makes every wait that does not find its data at once
    expire, the other knob every wait of all or every third workgroup: they then
    compute the sums themselves, in the order of the exchange (the same bits),
    and it is no error."""
    x, phi, alpha, bias, gamma = _inputs(n, T, D, True, True)
    xt, pt, at, bt, gt = to_device(pkg, device, x, True, phi, alpha, bias, gamma)
    weights = pkg.MhcPreWeights(pt, gt, n) if prepared else None
    args = (xt, None, at, bt, None) if prepared else (xt, pt, at, bt, gt)
    name, value = knob.split("=")
    os.environ[name] = value
    try:
        op = pkg.MhcPreOp(*args, h_pre=True, weights=weights)
    finally:
        os.environ.pop(name, None)
    want = run_gpu(pkg, device, x, True, phi, alpha, bias, gamma, kernel="cell")
    check(want, orc.mhc_pre(x, True, phi, alpha, bias, gamma), x, True, orc)
    for _ in range(2):
        for t in op.outputs():
            t.fill_(float("nan"))
        _say(f"[cell] n={n} T={T} D={D} {knob}")
        op.launch(check=True)
        assert op.kernel == "cell"
        assert op.computed_waits() or name == "MHCPRE_SPIN_LIMIT"
        got = fetch(op)
        for k in got:
            assert np.array_equal(got[k], want[k]), k
    op.close()


def test_graph_replays_on_new_inputs(pkg, orc, device):
    """Replays between eager launches on the same workspace, each with its own x."""
    import torch
    x, phi, alpha, bias, gamma = _inputs(4, 33, 512, True, True)
    xt, pt, at, bt, gt = to_device(pkg, device, x, True, phi, alpha, bias, gamma)
    op = pkg.MhcPreOp(xt, pt, at, bt, gt, h_pre=True)
    op.launch(check=True)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        op.launch()
    for r in range(4):
        xr = np.roll(x, r, axis=0)
        xt.copy_(to_device(pkg, device, xr, True, phi, alpha, bias, gamma)[0])
        for t in op.outputs():
            t.fill_(float("nan"))
        _say(f"[cell] graph replay {r}")
        g.replay()
        torch.cuda.synchronize()
        check(fetch(op), orc.mhc_pre(xr, True, phi, alpha, bias, gamma), xr, True, orc)
        op.launch(check=True)
        assert op.kernel == "cell"
    op.close()
