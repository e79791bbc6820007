"""The 16-bit kernels (fp16 / bf16 tensors as one term of their own format, cascmm_h16_kernel.h): every tile, with a
prepared and with a raw right operand, at the edges of its tiles, stages and 16-byte chunks."""
import pytest
import torch

from basedxl_amd import PreparedWeight, _lib, cascaded_lowp_matmul, cascaded_lowp_matmul_grouped, cascaded_lowp_matmul_prepared

pytestmark = pytest.mark.gpu

DTYPES = {torch.float16: ("_bpre_ioh", "_io16h"), torch.bfloat16: ("_bpre_iob", "_io16b")}


def _variants(tag):
    return [(i, n) for i, n in enumerate(_lib.variant_names()) if "_h16_" in n and tag in n]


def _integers(g, *shape):
    return torch.randint(-1, 2, shape, generator=g)


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("M,K,N", [(1, 8, 8), (31, 64, 16), (65, 72, 104), (130, 136, 84), (257, 328, 328), (300, 200, 641), (512, 64, 640)])
def test_every_tile_is_exact_on_integers(gpu_device, dtype, M, K, N):
    """Operands in {-1, 0, 1} and an integer bias: every sum is an integer below 2^8 (six standard deviations of the
    deepest K here: 6 sqrt(328 x 4 / 9) = 72), exact in either format, so the result must be the exact one.  The left
    operand has NaNs between its rows, and the result gaps that must stay as they are."""
    g = torch.Generator().manual_seed(M + K + N)
    a, b, bias = _integers(g, M, K), _integers(g, K, N), _integers(g, N)
    want = (a @ b + bias).to("cuda:0")
    assert int(want.abs().max()) < 256
    frame = torch.full((M, K + 8), float("nan"), dtype=dtype, device="cuda:0")
    frame[:, :K] = a.to(dtype).to("cuda:0")
    bd, biasd = b.to(dtype).to("cuda:0"), bias.to(dtype).to("cuda:0")
    w = PreparedWeight(bd)
    for vi, name in _variants(DTYPES[dtype][0]):
        print("16-bit prepared", (M, K, N), name, flush=True)
        assert torch.equal(cascaded_lowp_matmul(frame[:, :K], w, bias=biasd, variant=vi).long(), want), name
    if N % 8 == 0:
        for vi, name in _variants(DTYPES[dtype][1]):
            print("16-bit raw", (M, K, N), name, flush=True)
            out = torch.full((M + 1, N + 3), -77.0, dtype=dtype, device="cuda:0")      # (rows not 16-byte aligned: single stores)
            cascaded_lowp_matmul(frame[:, :K], bd, bias=biasd, out=out[:M, :N], variant=vi)
            assert torch.equal(out[:M, :N].long(), want), name
            assert bool((out[:M, N:] == -77.0).all()) and bool((out[M] == -77.0).all()), name
    assert torch.equal(cascaded_lowp_matmul(frame[:, :K], bd, bias=biasd).long(), want)      # the library's own choice
    for o in cascaded_lowp_matmul_grouped([frame[:, :K]] * 2, [bd, bd], biases=[biasd, biasd]) + \
            cascaded_lowp_matmul_prepared([frame[:, :K]] * 2, [w, w], biases=[biasd, biasd]):
        assert torch.equal(o.long(), want)


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("M,K,N", [(33, 72, 64), (257, 200, 704)])
def test_the_gated_store_of_every_tile(gpu_device, dtype, M, K, N):
    """value * gelu(gate) of the same integers: sums exact, the gate within an fp32 ulp of the exact one (4e-7, for values
    below 2^8), the result rounded once: half a unit in the last place of the 16-bit result."""
    g = torch.Generator().manual_seed(M + K + N)
    a, b, bias = _integers(g, M, K), _integers(g, K, N), _integers(g, N)
    value, gate = (a @ b + bias).double().chunk(2, -1)
    want = value * torch.nn.functional.gelu(gate)
    w = PreparedWeight(b.to(dtype).to("cuda:0"), glu=True)
    half_ulp = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    ran = 0
    for vi, name in _variants(DTYPES[dtype][0]):
        if name.split("x")[1] in ("64", "160"):
            continue          # (tiles whose waves own an odd number of column blocks have no gated store)
        print("16-bit gated", (M, K, N), name, flush=True)
        got = cascaded_lowp_matmul(a.to(dtype).to("cuda:0"), w, bias=bias.to(dtype).to("cuda:0"), variant=vi).cpu().double()
        assert bool(((got - want).abs() <= half_ulp * 1.001 * want.abs() + 256 * 4e-7).all()), name
        ran += 1
    assert ran >= 5


@pytest.mark.parametrize("ldc", [9000000, 17000008])
def test_rows_of_the_result_far_apart(gpu_device, ldc):
    """A result that is a view into something wide: 128 rows of 9 million elements, 64 rows of 17 million, span more than 2 GiB."""
    M, K, N, dtype = 257, 64, 72, torch.float16
    g = torch.Generator().manual_seed(ldc)
    a, b = _integers(g, M, K), _integers(g, K, N)
    ad, bd = a.to(dtype).to("cuda:0"), b.to(dtype).to("cuda:0")
    out = torch.empty(M * ldc, dtype=dtype, device="cuda:0").as_strided((M, N + 8), (ldc, 1))
    for vi, name in _variants("_fp16x1_io16h") + [(-1, "automatic")]:
        out.fill_(-77.0)
        print("far apart", ldc, name, flush=True)
        cascaded_lowp_matmul(ad, bd, out=out[:, :N], variant=vi)
        assert torch.equal(out[:, :N].cpu().long(), a @ b), name
        assert bool((out[:, N:] == -77.0).all()), name
    del out
    torch.cuda.empty_cache()
