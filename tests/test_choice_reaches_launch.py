"""The automatic choice of a kernel and the kernels' own launch checks have to agree: a problem that the library selects a
kernel for must not be refused by that kernel's launcher.

The calls run in a child process that sees no GPU, on addresses that are never read: arguments are checked, a kernel is
selected, its launcher checks them again, and then the launch itself fails for want of a device.  That status (LAUNCH) is what
a call has to reach."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LAUNCH, BAD_FORMAT, ALIGNMENT, TOO_LARGE = -7, -4, -6, -9
F32_BF16X2, FP16, BF16 = (0, 0, 2), (1, 1, 1), (2, 0, 1)          # (dtype, format, terms)

CHILD = """
import ctypes, json, sys
from basedxl_amd import _lib
l = _lib.lib()
if l.cascmm_init() == 0:
    raise SystemExit("a GPU is visible")
A, B, C, WS = 1 << 40, 2 << 40, 3 << 40, 4 << 40
out = []
for c in json.load(sys.stdin):
    M, K, N, (dt, fmt, terms) = c["M"], c["K"], c["N"], c["cascade"]
    glu, n = c.get("glu", False), c.get("count", 1)
    lda, ldb, ldc = c.get("lda", K), c.get("ldb", N), c.get("ldc", N // 2 if glu else N)
    a = A + c.get("a_offset", 0)
    need = l.cascmm_workspace_bytes(M, N, K, dt, fmt, terms, 0) * n if c.get("workspace", True) else 0
    ws = (WS if need else None, need, None)
    arr = lambda p: (ctypes.c_void_p * n)(*[p] * n)
    if glu:
        st = l.cascmm_gemm_prepared_glu(n, arr(a), arr(B), arr(C), None, M, N, K, lda, ldc, dt, fmt, terms, 0, None, None, -1)
    elif c.get("prepared"):
        st = l.cascmm_gemm_prepared(n, arr(a), arr(B), arr(C), None, M, N, K, lda, ldc, dt, fmt, terms, 0, None, *ws, -1)
    elif n > 1:
        st = l.cascmm_gemm_grouped(n, arr(a), arr(B), arr(C), None, M, N, K, lda, ldb, ldc, dt, fmt, terms, 0, None, *ws, -1)
    else:
        st = l.cascmm_gemm(a, B, C, None, M, N, K, lda, ldb, ldc, dt, fmt, terms, 0, None, *ws)
    out.append(st)
json.dump(out, sys.stdout)
"""


def statuses(cases):
    env = dict(os.environ, PYTHONPATH=ROOT, HIP_VISIBLE_DEVICES="-1", ROCR_VISIBLE_DEVICES="")
    r = subprocess.run([sys.executable, "-c", CHILD], input=json.dumps(cases), cwd=ROOT, env=env, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    return json.loads(r.stdout)


def refused(cases):
    """The cases that do not reach the launch, with their statuses."""
    return [(c, st) for c, st in zip(cases, statuses(cases)) if st != LAUNCH]


@pytest.mark.parametrize("step", [1, 2, 3])
def test_prepared_widths_off_four(step):
    """Weights kept split, two bf16 terms: any width, from a few rows to those that the large tiles are chosen for."""
    cases = [dict(M=M, K=K, N=N + step, cascade=F32_BF16X2, prepared=True)
             for M in (1, 40, 64, 200, 333, 1000, 2466, 4096, 8192) for K in (64, 72, 336, 640, 1280, 3712)
             for N in (4, 256, 316, 320, 636, 1280, 2016, 3000, 5100, 10240)]
    assert not refused(cases)


@pytest.mark.parametrize("cascade", [FP16, BF16])
def test_sixteen_bit_activations_beyond_two_gib(cascade):
    """16-bit layers with prepared weights, plain and gated, one problem and several: activations of any size."""
    cases = [dict(M=M, K=K, N=N, cascade=cascade, prepared=True, glu=glu, count=count, lda=K + pad)
             for M, K in ((4194304, 320), (9105865, 384), (26000000, 64), (1100000, 1000)) for N in (64, 640, 10240) for glu in (False, True)
             for count in (1, 3) for pad in (0, 64)]
    assert not refused(cases)


def test_prepared_buffers_of_whole_32_k_stages():
    """A prepared weight whose K is a multiple of 32 holds its own slots and no more, so buffers kept from before any rounding fit, and
    one just below 2 GiB is taken."""
    from basedxl_amd import _lib
    for K in (32, 96, 1056, 1280):
        for fmt, terms, planes in ((0, 2, 2), (1, 3, 3), (0, 1, 1), (1, 1, 1)):
            assert _lib.lib().cascmm_prepared_bytes(K, 332, fmt, terms) == planes * K * 332 * 2
    assert not refused([dict(M=M, K=K, N=N, cascade=c, prepared=True) for M in (1, 300) for K, N, c in
                        ((1056, 500368, F32_BF16X2), (224, 2166220, F32_BF16X2), (160, 2217588, (0, 0, 3)), (352, 1414720, (0, 2, 3)), (1056, 500369, F32_BF16X2))])


def test_what_a_prepared_weight_says_it_takes_reaches_the_launch():
    """``usable_with`` decides between the prepared and the raw weight of a layer: it must say no to what no prepared kernel
    takes (fp32 activations of 2 GiB off the 64-k stages or of odd width, slots of 2 GiB), and go on saying yes to what one does."""
    import torch
    from basedxl_amd import PreparedWeight
    names = {F32_BF16X2: (torch.float32, "bf16", 2), FP16: (torch.float16, "fp16", 1), BF16: (torch.bfloat16, "bf16", 1)}
    taken, said_no = [], []
    for cascade, (dtype, lowp, terms) in names.items():
        for K, N in ((64, 64), (72, 64), (72, 63), (1280, 1282), (328, 640), (640, 640), (96, 3), (1056, 508402), (1048, 508402), (72, 7456540), (32, 16000000)):
            w = PreparedWeight.from_slots(torch.empty(1, dtype=torch.uint8, device="meta"), K, N, dtype, lowp, terms)
            for M in (1, 33, 4096, 500000, 1700000, 2000000, 9000000):
                if M * N > 2 ** 42:
                    continue                 # (more tiles than a launch has)
                for pad in (0, 4, 8, 1 << 20):
                    a = torch.empty_strided((M, K), (K + pad, 1), dtype=dtype, device="meta")
                    c = dict(M=M, K=K, N=N, cascade=cascade, prepared=True, lda=K + pad if M > 1 else K)
                    if (K + pad) % (4 if dtype == torch.float32 else 8) != 0:
                        c["lda"] = K             # (such rows are copied)
                    (taken if w.usable_with(a) else said_no).append(c)
    assert len(taken) > 300
    aligned = [c for c in taken if c["K"] % 64 == 0 and c["N"] % 4 == 0]      # (the rule of always; rows of a MiB apart had no kernel then either)
    assert not [r for r in refused([c for c in taken if c not in aligned])]
    assert not [r for r in refused(aligned) if r[0]["lda"] * 2048 < 2 ** 31 - 1]
    # and no kernel goes unused: what it says no to has none
    assert len(refused(said_no)) == len(said_no) > 20


def test_prepared_calls_say_what_is_wrong_with_the_rows():
    """Rows off 16-byte boundaries that no prepared kernel takes are an alignment error, whatever else would be wrong with K."""
    F32X3, FP16X3, FP8X3 = (0, 0, 3), (0, 1, 3), (0, 2, 3)
    off = [dict(M=M, K=K, N=64, cascade=c, prepared=True, glu=glu, **rows) for M in (1, 200) for glu in (False, True)
           for c, K in ((F32X3, 320), (F32X3, 24), (FP16X3, 64), (FP8X3, 44), (F32_BF16X2, 33))
           for rows in (dict(lda=K + 4 - K % 4 + 2), dict(a_offset=4, lda=K + 4 - K % 4))]
    off += [dict(M=200, K=K, N=64, cascade=c, prepared=True, **rows) for c in (FP16, BF16) for K in (64, 66) for rows in (dict(lda=71), dict(lda=72, a_offset=2))]
    assert {st for st in statuses(off)} == {ALIGNMENT}
    assert {st for st in statuses([dict(M=200, K=K, N=64, cascade=c, prepared=True, lda=64) for c in (F32X3, FP16X3, FP16) for K in (12, 60)])} == {BAD_FORMAT}
