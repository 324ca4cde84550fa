"""What the operator's speed is measured on.

Every case is one call of MhcPre, the pre-mixing step of a multi-stream
residual block, as a model calls it once per block:

  op        torch.ops.mhcpre.mhc_pre on new output tensors each call (a model
            run eagerly: plan, outputs and workspace are the operator's own);
  op_h_pre  the same with the optional hPre output;
  launch    one launch of an executor made beforehand over static buffers (a
            serving loop), from phi and gamma;
  prepared  the same from weights prepared once (static weights).

The path has one direction (the operator is forward-only).  Its range: 4, 6 or
8 streams, fp16 or bf16 activations, gamma on or off, any row count (1 token of
a decode step to several thousand of a prefill chunk) and any stream width that
is a multiple of 16, ragged ones included.
"""
from __future__ import annotations

import math

import torch

import __graft_entry__

_pkg = __graft_entry__.load_package()
_ops = _pkg.torch_ops() and torch.ops.mhcpre

NORM_EPS = 1e-6
HC_EPS = 1e-6
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _case(n, D, T, dtype, gamma, api, alpha=(0.01, 0.01, 0.01), outliers=False, lead=1):
    return dict(n=n, D=D, T=T, dtype=dtype, gamma=gamma, api=api, alpha_pre=alpha[0],
                alpha_post=alpha[1], alpha_res=alpha[2], outliers=outliers, lead=lead)


_MIXED = (0.5, 0.3, 0.2)  # trained-size mixing weights; 0.01 is the start of training


def listed():
    return [
        # A small model's block over a short prompt: launches and host time count.
        dict(_case(4, 256, 128, "fp16", False, "op"), name="n4_small"),
        # One decode step of 16 sequences at the width of a large model, static weights.
        dict(_case(4, 7168, 16, "bf16", True, "prepared", _MIXED), name="n4_decode"),
        # A decode batch with 8 streams: the weights are most of the bytes.
        dict(_case(8, 7168, 64, "fp16", False, "launch"), name="n8_decode"),
        # A decode batch of odd size, 6 streams, wide rows.
        dict(_case(6, 5120, 37, "bf16", True, "op", _MIXED), name="n6_decode_odd"),
        # Eager prefill chunks of small and mid-size models (one per stream count).
        dict(_case(4, 2560, 2048, "fp16", True, "op", _MIXED), name="n4_chunk"),
        dict(_case(6, 1024, 2048, "bf16", True, "op", _MIXED), name="n6_chunk"),
        dict(_case(8, 1024, 1024, "fp16", True, "op_h_pre", _MIXED), name="n8_chunk"),
        # A mid-size prefill chunk with hPre kept.
        dict(_case(4, 4096, 1024, "bf16", True, "op_h_pre"), name="n4_mid"),
        # Ragged everything: an odd row count and a width that is a multiple of 16 only.
        dict(_case(4, 1200, 777, "bf16", False, "op", _MIXED), name="n4_ragged"),
        # Prefill chunk of a large model with 6 streams, static weights.
        dict(_case(6, 4096, 4096, "bf16", True, "prepared", _MIXED), name="n6_prefill"),
        # Prefill of a large model, 4 streams, two sequences.
        dict(_case(4, 7168, 8192, "bf16", True, "launch", lead=2), name="n4_prefill"),
        # The largest: 8 streams over a ragged batch, some rows much larger than the rest.
        dict(_case(8, 8192, 5472, "bf16", True, "launch", outliers=True), name="n8_prefill"),
    ]


def draw(rng):
    most = max(work(c)["bytes"] for c in listed())
    while True:
        n = rng.choice((4, 4, 6, 8))
        D = 16 * round(math.exp(rng.uniform(math.log(256), math.log(8192))) / 16)
        if rng.random() < 0.5:  # widths of models are multiples of 128 more often than not
            D = max(256, 128 * round(D / 128))
        T = round(math.exp(rng.uniform(0.0, math.log(8192))))
        c = _case(n, D, T, rng.choice(("fp16", "bf16")), rng.random() < 0.7,
                  rng.choice(("op", "op", "op_h_pre", "launch", "prepared")),
                  rng.choice(((0.01, 0.01, 0.01), _MIXED)), rng.random() < 0.2)
        if work(c)["bytes"] <= most:
            return c


def _sizes(case):
    n, D = case["n"], case["D"]
    return n, D, n * D, n * n + 2 * n, case["T"]


def _inputs(case, seed):
    """x [lead, T / lead, n, D], phi (memory [M][K]), alpha, bias, gamma or None."""
    n, D, K, M, T = _sizes(case)
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda")

    x = torch.empty((T, n, D), dtype=DTYPES[case["dtype"]], device="cuda")
    for r in range(0, T, 1024):
        x[r:r + 1024] = normal(min(1024, T - r), n, D)
    if case["outliers"]:  # about one row in a hundred 50 times larger, the last one always
        big = torch.rand(T, generator=g, device="cuda") < 0.01
        big[-1] = True
        x[big] = x[big] * 50
    phi = normal(M, K) / math.sqrt(K)
    bias = torch.rand(M, generator=g, device="cuda") * 0.2 - 0.1
    gamma = 1 + 0.1 * normal(n, D) if case["gamma"] else None
    alpha = torch.tensor([case["alpha_pre"], case["alpha_post"], case["alpha_res"]], device="cuda")
    return x.view(case["lead"], T // case["lead"], n, D), phi, alpha, bias, gamma


def prepare(case, seed):
    _, _, K, M, _ = _sizes(case)
    x, phi, alpha, bias, gamma = _inputs(case, seed)
    if case["api"].startswith("op"):
        call = _ops.mhc_pre_with_h_pre if case["api"] == "op_h_pre" else _ops.mhc_pre
        return {"call": call, "args": (x, phi.view(K, M), alpha, bias, gamma, NORM_EPS, HC_EPS)}
    if case["api"] == "prepared":
        weights = _pkg.MhcPreWeights(phi, gamma, case["n"])
        op = _pkg.MhcPreOp(x, None, alpha, bias, None, NORM_EPS, HC_EPS, weights=weights)
    else:
        op = _pkg.MhcPreOp(x, phi.view(K, M), alpha, bias, gamma, NORM_EPS, HC_EPS)
    return {"op": op}


def run(state):
    """(hIn, hPost, hRes) and hPre where the call gives it."""
    if "call" in state:
        return state["call"](*state["args"])
    op = state["op"]
    op.launch()
    return op.h_in, op.h_post, op.h_res


def work(case):
    n, D, K, M, T = _sizes(case)
    size = T * K * 2 + K * M * 4 + M * 4 + 12  # x, phi (or its prepared form), bias, alpha
    if case["gamma"] and case["api"] != "prepared":
        size += K * 4
    size += T * D * 2 + T * n * 4 + T * n * n * 4  # hIn, hPost, hRes
    if case["api"] == "op_h_pre":
        size += T * n * 4
    # the mixing product, the sum of squares and the weighted sum of the streams
    return {"bytes": size, "flops": 2 * T * K * M + 2 * T * K + 2 * T * K}


def tolerance(case):
    # Four times the largest difference seen between the operator's own kernels
    # forced onto the same inputs (they add in other orders), over the listed
    # cases and some drawn ones: rel 2.1e-5 (hIn; the fp32 outputs 4e-7 to
    # 1.9e-6), max one unit in hIn's last place (7.6e-3 in bf16, 9.7e-4 in fp16).
    return {"rel": 8e-5, "max": 0.03 if case["dtype"] == "bf16" else 4e-3}


def exact(case, seed):
    n, D, K, M, T = _sizes(case)
    x, phi, alpha, bias, gamma = _inputs(case, seed)
    lead = tuple(x.shape[:2])
    x = x.view(T, K)
    b = phi.double()
    if gamma is not None:
        b = b * gamma.double().view(1, K)
    bias, alpha = bias.double(), alpha.double()
    h_in, h_pre, h_post, h_res = [], [], [], []
    for r in range(0, T, 1024):
        xr = x[r:r + 1024].double()
        scale = 1 / torch.sqrt((xr * xr).mean(1, keepdim=True) + NORM_EPS)
        mix = (xr @ b.t()) * scale
        pre = torch.sigmoid(mix[:, :n] * alpha[0] + bias[:n]) + HC_EPS
        h_pre.append(pre)
        h_post.append(2 * torch.sigmoid(mix[:, n:2 * n] * alpha[1] + bias[n:2 * n]))
        h_res.append(mix[:, 2 * n:] * alpha[2] + bias[2 * n:])
        h_in.append((xr.view(-1, n, D) * pre[:, :, None]).sum(1))
    out = [torch.cat(h_in).view(*lead, D), torch.cat(h_post).view(*lead, n),
           torch.cat(h_res).view(*lead, n, n)]
    if case["api"] == "op_h_pre":
        out.append(torch.cat(h_pre).view(*lead, n))
    return tuple(out)
