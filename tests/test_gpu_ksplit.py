"""K split over workgroups (csrc/cascmm_ksplit.h): every kernel that has it, with ragged last tiles and last splits, odd N,
a bias and a result with gaps between its rows; the automatic choice; and the partial results behind copied operands."""
import ctypes

import pytest
import torch

from basedxl_amd import PreparedWeight, _lib, cascaded_lowp_matmul

pytestmark = pytest.mark.gpu
DTYPES = {torch.float32: (0, _lib.FMT_BF16, 2), torch.float16: (1, _lib.FMT_FP16, 1), torch.bfloat16: (2, _lib.FMT_BF16, 1)}


def _call(a, b, slots, bias, out, M, N, K, splits, vi, workspace):
    l = _lib.lib()
    dt, fmt, terms = DTYPES[a.dtype]
    stream = torch.cuda.current_stream().cuda_stream
    ws = (workspace.data_ptr(), workspace.numel(), stream, vi | splits << 16)
    if slots is None:
        return l.cascmm_gemm_variant(a.data_ptr(), b.data_ptr(), out.data_ptr(), bias.data_ptr(), M, N, K, a.stride(0), b.stride(0),
                                     out.stride(0), dt, fmt, terms, 0, None, *ws)
    one = lambda t: (ctypes.c_void_p * 1)(t.data_ptr())
    return l.cascmm_gemm_prepared(1, one(a), one(slots), one(out), one(bias), M, N, K, a.stride(0), out.stride(0), dt, fmt, terms, 0,
                                  None, *ws)


def _kernels():
    for vi, n in enumerate(_lib.variant_names()):
        if "_h16_" in n or n.startswith(("k64x160x16", "k64x80x32")):
            yield vi, n, torch.float32 if n.startswith("k64") else torch.bfloat16 if "bf16x1" in n else torch.float16


# (M, K, N, splits): one row; a last split of one 64-k stage, of a tail; ragged tiles; as many splits as there are
@pytest.mark.parametrize("M, K, N, splits", [(1, 128, 64, 2), (65, 328, 162, 3), (70, 1096, 330, 9), (40, 1024, 100, 16), (257, 640, 324, 5)])
def test_every_kernel_is_exact_on_integers_in_splits(gpu_device, M, K, N, splits):
    gen = torch.Generator().manual_seed(M + K)
    ints = lambda *s: torch.randint(-3, 4, s, generator=gen)
    A, B, bias = ints(M, K), ints(K, N), ints(N)
    want = A @ B + bias
    workspace = torch.empty(splits * M * ((N + 3) // 4 * 4) * 4, dtype=torch.uint8, device="cuda")
    for vi, name, dtype in _kernels():
        frame = torch.full((M, K + 8), float("nan"), dtype=dtype, device="cuda")
        frame[:, :K] = A.to(dtype)
        b, biasd = B.to(dtype).cuda(), bias.to(dtype).cuda()
        slots = PreparedWeight(b).slots if "_bpre" in name else None
        out = torch.full((M, N + 6), 777.0, dtype=dtype, device="cuda")
        workspace.fill_(255)                                  # (NaNs: nothing but what the launch wrote is read back)
        print(name, M, K, N, splits, flush=True)
        for again in range(2):
            assert _call(frame, b, slots, biasd, out, M, N, K, splits, vi, workspace) == 0, name
        got = out[:, :N].cpu().double()
        assert torch.equal(got, want.to(dtype).double()), name
        assert (out[:, N:] == 777.0).all(), name
        # without room for the partial results K stays whole; of a count that leaves splits empty the others run
        for short, count in ((1, splits), (0, min(16, K // 64 + 2))):
            out.fill_(777.0)
            assert _call(frame, b, slots, biasd, out, M, N, K, count, vi, workspace[:workspace.numel() - short]) == 0, name
            assert torch.equal(out[:, :N].cpu().double(), want.to(dtype).double()), name


# fp32: two bf16 terms drop lo.lo, 2^-18 relative; 16-bit: one rounding of the result
@pytest.mark.parametrize("dtype, tol", [(torch.float32, 2.0 ** -16), (torch.float16, 2.0 ** -11), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("M, K, N", [(7, 3264, 880), (64, 5120, 1280), (34, 2008, 2176), (30, 5117, 1281)])
def test_automatic_choice_on_few_rows_and_deep_k(gpu_device, M, K, N, dtype, tol):
    gen = torch.Generator(device="cuda").manual_seed(3)
    a = torch.randn(M, K, device="cuda", generator=gen).to(dtype)
    b = (torch.randn(K, N, device="cuda", generator=gen) * 0.02).to(dtype)
    bias = torch.randn(N, device="cuda", generator=gen).to(dtype)
    want = a.cpu().double() @ b.cpu().double() + bias.cpu().double()
    for w in (b, PreparedWeight(b)) if K % 8 == 0 else (b,):
        got = cascaded_lowp_matmul(a, w, bias=bias)
        assert torch.equal(got, cascaded_lowp_matmul(a, w, bias=bias))
        assert ((got.cpu().double() - want).norm() / want.norm()).item() < tol


def test_workspace_holds_what_the_choice_asks_for():
    """The size the library asks for is enough for the splits it then takes: the choice with just that much is the choice
    with any amount (the same sums in the same order)."""
    l = _lib.lib()
    for M, K, N in [(7, 3264, 880), (64, 5120, 1280), (30, 5117, 1281), (512, 5120, 1280)]:
        for dtype, (dt, fmt, terms) in DTYPES.items():
            a, b = torch.randn(M, K, device="cuda").to(dtype), (torch.randn(K, N, device="cuda") * 0.02).to(dtype)
            need = l.cascmm_workspace_bytes(M, N, K, dt, fmt, terms, 0)
            outs = []
            for size in (need, 1 << 28):
                ws, c = torch.empty(max(size, 16), dtype=torch.uint8, device="cuda"), torch.empty(M, N, dtype=dtype, device="cuda")
                assert l.cascmm_gemm(a.data_ptr(), b.data_ptr(), c.data_ptr(), None, M, N, K, K, N, N, dt, fmt, terms, 0, None,
                                     ws.data_ptr(), size, torch.cuda.current_stream().cuda_stream) == 0
                outs.append(c)
            assert torch.equal(*outs), (M, K, N, dtype)
