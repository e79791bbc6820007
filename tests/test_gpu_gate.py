"""The gate of a gated projection: as one kernel behind the product (csrc/cascmm_gate_kernel.h), and the fit that the gated stores and its
16-bit form evaluate (gelu_values, csrc/cascmm_common.h)."""
import os
import re

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from basedxl_amd import PreparedWeight, _lib, cascaded_lowp_matmul
from basedxl_amd.cascaded_lowp_matmul import gate_product


# inner: runs of 16 bytes, of 4, single elements; one run, the last run of a workgroup, several workgroups
@pytest.mark.gpu
@pytest.mark.parametrize("dtype,ulp", [(torch.float32, 2.0 ** -23), (torch.float16, 2.0 ** -10), (torch.bfloat16, 2.0 ** -7)])
@pytest.mark.parametrize("rows,inner", [(1, 1), (1, 4), (3, 8), (5, 1024), (7, 2050), (33, 331), (257, 640)])
def test_gate_product(gpu_device, dtype, ulp, rows, inner):
    print(dtype, rows, inner, flush=True)
    g = torch.Generator().manual_seed(rows + inner)
    h = (torch.randn(rows, 2 * inner, generator=g) * 3).to(dtype)
    h.view(-1)[0] = -30.0
    value, gate = h.double().chunk(2, dim=-1)
    want = value * F.gelu(gate)
    frame = torch.full((rows, 2 * inner + 3), float("nan"), dtype=dtype, device="cuda")     # rows that start anywhere
    frame[:, :2 * inner] = h
    for x in (h.cuda(), frame[:, :2 * inner]):
        got = gate_product(x)
        assert got.shape == want.shape and got.dtype == dtype
        # erf within two fp32 ulps of 1 + erf, four roundings of fp32, one of the result
        bound = value.abs() * gate.abs() * 2.0 ** -22 + want.abs() * (3 * 2.0 ** -23 + ulp / 2) + 2.0 ** -24
        err = (got.cpu().double() - want).abs()
        assert (err <= bound).all(), (err / bound).max().item()


def test_what_the_gate_refuses():
    l, ok = _lib.lib(), 1 << 20
    assert l.cascmm_gate(ok, ok, 4, 4, 8, 4, 7, None) == -3                       # dtype
    assert l.cascmm_gate(ok, ok, 4, 4, 7, 4, 0, None) == l.cascmm_gate(ok, ok, 4, 4, 8, 3, 0, None) == -2
    assert l.cascmm_gate(None, ok, 4, 4, 8, 4, 0, None) != 0 and l.cascmm_gate(ok + 2, ok, 4, 4, 8, 4, 0, None) != 0
    assert l.cascmm_gate(ok, ok, 1 << 20, 1 << 12, 1 << 13, 1 << 12, 0, None) != 0   # counts beyond 32 bits
    assert l.cascmm_gate(None, None, 0, 4, 8, 4, 0, None) == 0


def _fit():
    text = open(os.path.join(os.path.dirname(_lib.__file__), "csrc", "cascmm_common.h")).read()
    c = re.search(r"kGeluFit\[10\] = \{([^}]*)\}", text).group(1)
    return [float(np.float32(x.strip().rstrip("f"))) for x in c.split(",")] + [0.0]


def test_fit_behind_the_gated_stores():
    """The bound that stands beside the constants, and what lets nothing be clamped behind the fit's end."""
    c = np.poly1d(_fit())
    x = np.linspace(0.0, 5.66, 200001)
    want = torch.special.log_ndtr(torch.from_numpy(-x)).numpy() / np.log(2.0) + 1.0
    assert (np.abs(c(x) - want) <= 7.2e-8 * (1 + (x / 2) ** 4)).all()
    far = c(np.geomspace(5.66, 1e30, 100001))
    assert (np.diff(far) < 0).all()


# rms error against 64 bits over the result's rms, for gates of N(0, std): measured 3.7e-8, 3.5e-8, 2.7e-8, 2.2e-8, of which the result's own
# rounding is about 2.2e-8.  As g (1 - Phi(-g)), Phi from a fit with its constant in it, the first three were 5.6e-8, 5.1e-8, 3.5e-8; as
# (2 - erfc) g / 2 4.5e-8, 4.5e-8, 3.5e-8.
@pytest.mark.gpu
@pytest.mark.parametrize("std,bar", [(0.1, 4.2e-8), (0.3, 4.0e-8), (1.0, 3.2e-8), (3.0, 2.6e-8)])
def test_gate_error_of_the_gated_stores(gpu_device, std, bar):
    """A = I with three fp16 terms, which hold a weight to 33 bits, and value columns of ones: the result is gelu of the gate columns."""
    inner = 1024
    g = torch.Generator().manual_seed(int(10 * std))
    w = torch.ones(64, 2 * inner)
    w[:, inner:] = torch.randn(64, inner, generator=g) * std
    y = cascaded_lowp_matmul(torch.eye(64, device="cuda"), PreparedWeight(w.cuda(), lowp="fp16", terms=3, glu=True)).cpu().double()
    gate = w[:, inner:].double()
    want = gate * torch.special.ndtr(gate)
    rms = ((y - want).square().mean() / want.square().mean()).sqrt().item()
    positive = gate > 0
    largest = ((y - want).abs() / want.abs())[positive].max().item()
    print(f"gate error, gates of N(0, {std}): rms {rms:.3e}, positive gates at most {largest:.3e}", flush=True)
    assert rms <= bar and largest <= 1.6e-7


@pytest.mark.gpu
def test_gates_that_are_not_finite(gpu_device):
    """As 0.5 g (1 + erf(g / sqrt 2)) has them: inf, not a number, not a number; large ones are themselves or zero."""
    gates = torch.tensor([float("inf"), float("-inf"), float("nan"), 3.0e38, -3.0e38, 6.0e4, -6.0e4, -0.0])
    want = torch.tensor([float("inf"), float("nan"), float("nan"), 3.0e38, 0.0, 6.0e4, 0.0, 0.0])
    bias = torch.ones(128)
    bias[64:] = gates.repeat(8)
    for lowp, terms in (("bf16", 2), ("fp16", 3)):
        w = PreparedWeight(torch.zeros(64, 128, device="cuda"), lowp=lowp, terms=terms, glu=True)
        y = cascaded_lowp_matmul(torch.ones(40, 64, device="cuda"), w, bias=bias.cuda())
        torch.testing.assert_close(y.cpu(), want.repeat(40, 8), rtol=2e-7, atol=0, equal_nan=True)
    h = torch.ones(3, 16, dtype=torch.bfloat16)
    h[:, 8:] = gates
    torch.testing.assert_close(gate_product(h.cuda()).cpu(), want.to(torch.bfloat16).repeat(3, 1), rtol=0, atol=0, equal_nan=True)
