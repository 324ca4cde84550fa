"""The strip kernel at widths with D % 32 == 16 (n = 4; shapes of the split path,
which runs it in place of its own kernels), against the CPU oracle at the
tolerances of tests/helpers.py."""
from __future__ import annotations

import os

import numpy as np
import pytest

from inputs import to_bits
from test_gpu_parity import _say, check, fetch, run_gpu, to_device

pytestmark = pytest.mark.gpu

N = 4


def _inputs(T, D, is_bf16, has_gamma):
    rng = np.random.default_rng(4000 + 17 * T + D)
    K, M = N * D, N * N + 2 * N
    xf = rng.standard_normal((T, N, D)).astype(np.float32)
    xf[::7] *= 50.0  # large rows exercise the RMS scale
    phi = (rng.standard_normal((M, K)) / np.sqrt(K)).astype(np.float32)
    alpha = np.asarray([0.3, -0.2, 0.05], dtype=np.float32)
    bias = rng.uniform(-0.5, 0.5, M).astype(np.float32)
    gamma = (1 + 0.1 * rng.standard_normal(K)).astype(np.float32) if has_gamma else None
    return to_bits(xf, is_bf16), phi, alpha, bias, gamma


@pytest.mark.parametrize("T,D,is_bf16,has_gamma,prepared", [
    (1, 208, True, True, False),       # one row, one slice: 3 strips and 16 columns
    (17, 240, False, False, True),     # one slice, the last strip 48 columns
    (777, 1200, True, False, False),   # D % 64 == 48, ragged rows
    (300, 1040, False, True, True),    # the last slice 16 columns
    (2100, 2256, True, True, True),    # 9 slices, teams across XCDs
    (130, 16368, True, True, False),   # 64 slices
])
def test_strip_at_half_step_widths(pkg, orc, device, T, D, is_bf16, has_gamma, prepared):
    x, phi, alpha, bias, gamma = _inputs(T, D, is_bf16, has_gamma)
    _say(f"[strip half] T={T} D={D} bf16={is_bf16} gamma={has_gamma} prepared={prepared}")
    ref = orc.mhc_pre(x, is_bf16, phi, alpha, bias, gamma)
    plain = run_gpu(pkg, device, x, is_bf16, phi, alpha, bias, gamma, force_path="strip",
                    kernel="strip")
    os.environ["MHCPRE_FORCE_PATH"] = "strip"
    try:
        xt, pt, at, bt, gt = to_device(pkg, device, x, is_bf16, phi, alpha, bias, gamma)
        op = pkg.MhcPreOp(xt, None, at, bt, None, h_pre=True, weights=pkg.MhcPreWeights(pt, gt, N))
    finally:
        os.environ.pop("MHCPRE_FORCE_PATH", None)
    assert plain.pop("path") == "split"
    check(plain, ref, x, is_bf16, orc)
    if prepared:  # the same bits from prepared weights
        op.launch(check=True)
        assert op.kernel == "strip"
        got = fetch(op)
        for k in plain:
            assert np.array_equal(got[k], plain[k]), k
    op.close()


@pytest.mark.parametrize("knob", ["MHCPRE_SPIN_LIMIT=0", "MHCPRE_SPIN_EVERY=5"])
@pytest.mark.parametrize("T,D,is_bf16,prepared", [(300, 1200, True, False), (200, 720, True, True),
                                                 (500, 3600, False, False), (130, 240, False, True)])
def test_expired_waits_are_computed(pkg, orc, device, T, D, is_bf16, prepared, knob):
    """A spin limit of 0, in all or every fifth workgroup, makes every wait that
    does not find its data at once expire: the workgroups then compute what they
    waited for in the order of the exchange (the same bits) and it is no error."""
    x, phi, alpha, bias, gamma = _inputs(T, D, is_bf16, True)
    xt, pt, at, bt, gt = to_device(pkg, device, x, is_bf16, phi, alpha, bias, gamma)
    weights = pkg.MhcPreWeights(pt, gt, N) if prepared else None
    args = (xt, None, at, bt, None) if prepared else (xt, pt, at, bt, gt)
    name, value = knob.split("=")
    os.environ[name] = value
    os.environ["MHCPRE_FORCE_PATH"] = "strip"
    try:
        op = pkg.MhcPreOp(*args, h_pre=True, weights=weights)
    finally:
        os.environ.pop(name, None)
        os.environ.pop("MHCPRE_FORCE_PATH", None)
    want = run_gpu(pkg, device, x, is_bf16, phi, alpha, bias, gamma, force_path="strip", kernel="strip")
    want.pop("path")
    check(want, orc.mhc_pre(x, is_bf16, phi, alpha, bias, gamma), x, is_bf16, orc)
    for _ in range(2):
        for t in op.outputs():
            t.fill_(float("nan"))
        _say(f"[strip half] T={T} D={D} {knob}")
        op.launch(check=True)
        assert op.kernel == "strip" and op.computed_waits()
        got = fetch(op)
        for k in want:
            assert np.array_equal(got[k], want[k]), k
    op.close()
