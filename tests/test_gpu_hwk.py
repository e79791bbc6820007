"""16-bit tensors on the kernels that split K over the eight waves of a workgroup (cascmm_hwk_kernel.h): every tile, at the edges of
its tile, of a 64-k step, of 16-byte chunks, of the straight code's numbers of steps and of the ring."""
import pytest
import torch

from basedxl_amd import PreparedWeight, _lib, cascaded_lowp_matmul, cascaded_lowp_matmul_grouped, cascaded_lowp_matmul_prepared

pytestmark = pytest.mark.gpu

_TILES = [n for n in _lib.variant_names() if "_hwk_" in n]


def _integers(g, *shape):
    return torch.randint(-1, 2, shape, generator=g)


def _dtype(name):
    return torch.float16 if "fp16" in name else torch.bfloat16


@pytest.mark.parametrize("name", _TILES)
@pytest.mark.parametrize("K", [8, 64, 72, 504, 520, 1016, 1088, 1544, 2056, 2568, 3592])
def test_every_number_of_steps_is_exact_on_integers(name, K):
    """Operands in {-1, 0, 1}, of A's columns one in 8 for deep K, and an integer bias: every sum is an integer below 2^8 (checked), exact in
    either format.  The rows of A have NaNs between them, the result gaps that stay as they are, and is written in quads and one by one."""
    bm, bn = (int(x) for x in name.split("_")[0][1:].split("x")[:2])
    g, dtype, variant = torch.Generator().manual_seed(K), _dtype(name), _lib.variant_names().index(name)
    for M, N, gap in ((bm, bn, 4), (7, 2 * bn + 2, 1), (bm + 9, bn - 3 if "bpre" in name else bn - 2, 3), (2 * bm + 1, 3 * bn + 4, 0)):
        a, b, bias = _integers(g, M, K), _integers(g, K, N), _integers(g, N)
        a[:, torch.arange(K) % 8 != 3] *= int(K <= 520)
        a[:, K - 1] = 1
        want = a @ b + bias
        assert int(want.abs().max()) < 256
        frame = torch.full((M, K + 8), float("nan"), dtype=dtype, device="cuda:0")
        frame[:, :K] = a.to(dtype).to("cuda:0")
        w = b.to(dtype).to("cuda:0")
        gap *= "bpre" not in name          # (a prepared call's result is contiguous)
        out = torch.full((M + 1, N + gap), -77.0, dtype=dtype, device="cuda:0")
        print("hwk", name, (M, K, N), flush=True)
        cascaded_lowp_matmul(frame[:, :K], PreparedWeight(w) if "bpre" in name else w, bias=bias.to(dtype).to("cuda:0"), out=out[:M, :N], variant=variant)
        assert torch.equal(out[:M, :N].cpu().long(), want), (M, N)
        assert bool((out[M] == -77.0).all()) and bool((out[:, N:] == -77.0).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,N", [(33, 72, 64), (16, 200, 192), (81, 520, 704)])
def test_the_gated_store(dtype, M, K, N):
    """value * gelu(gate) of integers: sums exact, the gate within an fp32 ulp of the exact one (4e-7, for values below 2^8), the result
    rounded once."""
    g = torch.Generator().manual_seed(M + K + N)
    a, b, bias = _integers(g, M, K), _integers(g, K, N), _integers(g, N)
    value, gate = (a @ b + bias).double().chunk(2, -1)
    want = value * torch.nn.functional.gelu(gate)
    w = PreparedWeight(b.to(dtype).to("cuda:0"), glu=True)
    half_ulp = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    names = [n for n in _TILES if "bpre" in n and _dtype(n) == dtype and n.split("x")[1] == "64"]
    assert len(names) == 3
    for name in names:
        print("hwk gated", name, (M, K, N), flush=True)
        got = cascaded_lowp_matmul(a.to(dtype).to("cuda:0"), w, bias=bias.to(dtype).to("cuda:0"), variant=_lib.variant_names().index(name)).cpu().double()
        assert bool(((got - want).abs() <= half_ulp * 1.001 * want.abs() + 256 * 4e-7).all()), name


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,N", [(2, 1280, 1280), (154, 2048, 640), (77, 256, 641), (1, 8, 2), (320, 328, 322), (3, 5120, 40)])
def test_the_library_s_own_choice(dtype, M, K, N):
    """Raw and prepared, alone and in groups, against 64 bits: one rounding of the result and the error of the sums (K eps32 at most for
    each of the terms, sqrt(K) of it expected: below 1e-5 here); infinities and NaNs stay in their row and column."""
    g = torch.Generator(device="cuda:0").manual_seed(M * K + N)
    a, b = torch.randn(M, K, device="cuda:0", generator=g).to(dtype), (torch.randn(K, N, device="cuda:0", generator=g) * 0.02).to(dtype)
    want = a.cpu().double() @ b.cpu().double()
    half_ulp = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    w = PreparedWeight(b)
    print("hwk chosen", dtype, (M, K, N), flush=True)
    outs = [cascaded_lowp_matmul(a, b), cascaded_lowp_matmul(a, w)] + cascaded_lowp_matmul_grouped([a, a], [b, b]) + cascaded_lowp_matmul_prepared([a, a], [w, w])
    scale = float(want.pow(2).mean().sqrt())
    for o in outs:
        assert bool(((o.cpu().double() - want).abs() <= half_ulp * 1.001 * want.abs() + 1e-5 * scale + 2.0 ** -25).all())
    a[M // 2, K - 1], b[0, N // 3] = float("inf"), float("nan")
    for o in (cascaded_lowp_matmul(a, b), cascaded_lowp_matmul(a, PreparedWeight(b))):
        bad = ~torch.isfinite(o)
        assert bool(bad[M // 2].all()) and bool(bad[:, N // 3].all()) and int(bad.sum()) == M + N - 1
