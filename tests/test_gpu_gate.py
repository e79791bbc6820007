"""The gate of a gated projection as one kernel behind the product (csrc/cascmm_gate_kernel.h)."""
import pytest
import torch
import torch.nn.functional as F

from basedxl_amd import _lib
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
