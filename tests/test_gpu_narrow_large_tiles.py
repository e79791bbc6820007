"""The large-tile kernels on 256 x 192 and 256 x 128 (NTL 3 and 2 in csrc/cascmm_w512_kernel.h): plain and gated stores."""
import pytest
import torch

from basedxl_amd import PreparedWeight, _lib, cascaded_lowp_matmul

pytestmark = pytest.mark.gpu


def _kernels(suffix=""):
    names = [(vi, n) for vi, n in enumerate(_lib.variant_names()) if "_w512_narrow_" in n and n.endswith(suffix)]
    assert names
    return names


# (M, K, N): the fewest rows and one tile of each width, one row, one quad and one column more, a wave's half missing; K: one pair of stages,
# fewer pairs than are in flight, as many, one more, in the first and the second stage of a pair, one chunk into a stage
@pytest.mark.parametrize("M, K, N", [(64, 32, 192), (256, 64, 128), (257, 64, 196), (385, 96, 324), (128, 128, 448), (1000, 160, 388), (300, 72, 260),
                                     (64, 88, 192), (258, 1256, 388), (200, 36, 256), (270, 68, 452), (256, 64, 193), (513, 96, 321)])
def test_exact_on_integers(gpu_device, M, K, N):
    gen = torch.Generator().manual_seed(M + N)
    ints = lambda *s: torch.randint(-90, 91, s, generator=gen)
    A, B, bias = ints(M, K), ints(K, N), ints(N)
    want = A @ B + bias
    ran = 0
    for vi, name in _kernels():
        prepared = name.endswith("_bpre")
        if "x192x" in name and N < 192 or not prepared and N % 4 != 0 or prepared and (K % 8 != 0 or K % 32 != 0 and K < 64):
            continue                                    # (narrower than a tile; what the raw loads and prepared weights ask for)
        frame = torch.full((M + 4, max(K + 8, 32)), float("nan"), device="cuda")   # NaNs that no result may see, 777 that stay
        frame[:M, :K] = A
        b = B.float().cuda()
        out = torch.full((M + 4, N if prepared else N + 8), 777.0, device="cuda")
        print(name, M, K, N, flush=True)
        cascaded_lowp_matmul(frame[:M, :K], PreparedWeight(b) if prepared else b, bias=bias.float().cuda(), out=out[:M, :N], variant=vi)
        assert torch.equal(out[:M, :N].cpu().long(), want), name
        assert (out[M:] == 777.0).all() and (out[:, N:] == 777.0).all(), name
        ran += 1
    assert ran


# N: value and gate columns together, of one tile, a pair of blocks more, several tiles.  Sums of integers are exact; the gate is within an
# fp32 ulp of the exact one (4e-7 + 2e-7 |gate|), the product rounded once
@pytest.mark.parametrize("M, K, N", [(64, 64, 128), (300, 64, 192), (257, 128, 448), (1000, 192, 640)])
def test_gated_store(gpu_device, M, K, N):
    gen = torch.Generator().manual_seed(M + N)
    A, B, bias = torch.randint(-3, 4, (M, K), generator=gen), torch.randint(-3, 4, (K, N), generator=gen), torch.randint(-9, 10, (N,), generator=gen)
    B[:, N // 2:] = B[:, N // 2:].clamp(-1, 1) * (torch.rand(K, N // 2, generator=gen) < 0.1)    # (gates of a few units)
    value, gate = (A @ B + bias).double().chunk(2, dim=-1)
    want = value * torch.nn.functional.gelu(gate)
    w = PreparedWeight(B.float().cuda(), glu=True)
    (vi, name), = [(vi, n) for vi, n in _kernels("_bpre") if "x128x" in n]
    out = torch.full((M + 4, N // 2), 777.0, device="cuda")
    cascaded_lowp_matmul(A.float().cuda(), w, bias=bias.float().cuda(), out=out[:M], variant=vi)
    err, bound = (out[:M].cpu().double() - want).abs(), value.abs() * (4e-7 + 2e-7 * gate.abs()) + 1.2e-7 * want.abs()
    assert (err <= bound).all(), (name, (err - bound).max().item())
    assert (out[M:] == 777.0).all(), name
