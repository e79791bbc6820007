"""The large-tile kernels whose tiles may hang over the edges of C (EDGE in csrc/cascmm_w512_kernel.h): plain and gated stores."""
import pytest
import torch

from basedxl_amd import BasedXLLowPLinear, PreparedWeight, _lib, cascaded_lowp_matmul

pytestmark = pytest.mark.gpu


def _kernels(suffix=""):
    names = [(vi, n) for vi, n in enumerate(_lib.variant_names()) if "_w512_edge_" in n and n.endswith(suffix)]
    assert names
    return names


# (M, K, N): the fewest rows, one tile and a row or four columns more, a wave's half of the tile missing, several tiles;
# the gaps between the rows of both sides, the rows and columns past the ends: NaNs that no result may see, 777 that stay
@pytest.mark.parametrize("M, K, N", [(64, 32, 320), (256, 64, 320), (257, 64, 324), (385, 96, 460), (128, 32, 576), (1000, 160, 1284), (515, 64, 640),
                                     # K: in the first stage of a pair, in the second, one 16-byte chunk into a stage, one short of it
                                     (300, 72, 452), (64, 88, 320), (258, 1256, 388), (200, 36, 324), (270, 60, 644), (128, 4, 320)])
def test_exact_on_integers_over_the_edges(gpu_device, M, K, N):
    gen = torch.Generator().manual_seed(M + N)
    ints = lambda *s: torch.randint(-90, 91, s, generator=gen)
    A, B, bias = ints(M, K), ints(K, N), ints(N)
    want = A @ B + bias
    for vi, name in _kernels():
        if name.endswith("_bpre") and (K % 8 != 0 or (K % 32 != 0 and K < 64)):
            continue                                    # (a prepared weight of such a K is refused)
        frame = torch.full((M + 4, max(K + 8, 32)), float("nan"), device="cuda")
        frame[:M, :K] = A
        a, b, biasd = frame[:M, :K], B.float().cuda(), bias.float().cuda()
        prepared = name.endswith("_bpre")
        w = PreparedWeight(b) if prepared else b
        out = torch.full((M + 4, N if prepared else N + 8), 777.0, device="cuda")   # (a prepared weight's result is contiguous)
        print(name, M, K, N, flush=True)
        cascaded_lowp_matmul(a, w, bias=biasd, out=out[:M, :N], variant=vi)
        assert torch.equal(out[:M, :N].cpu().long(), want), name
        assert (out[M:] == 777.0).all() and (out[:, N:] == 777.0).all(), name


# a prepared weight's width is anything: one column more than whole tiles, than a wave's half, one short of a tile; rows whole and not
@pytest.mark.parametrize("M, K, N", [(256, 64, 641), (300, 72, 322), (64, 336, 1283), (513, 64, 481), (256, 96, 639)])
def test_prepared_widths_off_four_are_exact_on_integers(gpu_device, M, K, N):
    gen = torch.Generator().manual_seed(M + N)
    ints = lambda *s: torch.randint(-90, 91, s, generator=gen)
    A, B, bias = ints(M, K), ints(K, N), ints(N)
    want = A @ B + bias
    w = PreparedWeight(B.float().cuda())
    for vi, name in _kernels("_bpre"):
        out = torch.full((M + 4, N), 777.0, device="cuda")
        print(name, M, K, N, flush=True)
        cascaded_lowp_matmul(A.float().cuda(), w, bias=bias.float().cuda(), out=out[:M], variant=vi)
        assert torch.equal(out[:M].cpu().long(), want), name
        assert (out[M:] == 777.0).all(), name


@pytest.mark.parametrize("M, K, N", [(2466, 336, 2019), (1000, 640, 2562)])
def test_prepared_layer_of_odd_width(gpu_device, M, K, N):
    """The layer on the kernel that is chosen for it.  Two bf16 terms of each factor drop lo.lo: 2^-18 of a product, 2^-16 of the
    result at most."""
    lin = torch.nn.Linear(K, N).to("cuda")
    x = torch.randn(M, K, device="cuda")
    want = torch.nn.functional.linear(x.double(), lin.weight.double(), lin.bias.double())
    got = BasedXLLowPLinear(lin, prepared=True)(x)
    assert ((got.double() - want).norm() / want.norm()).item() < 2.0 ** -16


# N: value and gate columns together; the 256 x 320 tile has the gated store where its columns are whole
@pytest.mark.parametrize("M, K, N", [(64, 64, 320), (300, 64, 640), (257, 128, 448), (1000, 192, 1280)])
def test_gated_store_over_the_edges(gpu_device, M, K, N):
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    a = torch.randn(M, K, device="cuda", generator=gen)
    b, bias = torch.randn(K, N, device="cuda", generator=gen) * 0.2, torch.randn(N, device="cuda", generator=gen)
    value, gate = (a.cpu().double() @ b.cpu().double() + bias.cpu().double()).chunk(2, dim=-1)
    want = value * torch.nn.functional.gelu(gate)
    w = PreparedWeight(b, glu=True)
    ran = 0
    for vi, name in _kernels("_bpre"):
        if "320" in name and N % 320 != 0:
            continue
        out = torch.full((M + 4, N // 2), 777.0, device="cuda")
        print(name, M, K, N, flush=True)
        cascaded_lowp_matmul(a, w, bias=bias, out=out[:M], variant=vi)
        # two bf16 terms drop lo.lo, 2^-18 of a product; value and gate each: 2^-16 of the result at most
        assert ((out[:M].cpu().double() - want).norm() / want.norm()).item() < 2.0 ** -16, name
        assert (out[M:] == 777.0).all(), name
        ran += 1
    assert ran


def test_ragged_rows_of_a_wide_layer_take_the_large_tile():
    l, names = _lib.lib(), _lib.variant_names()
    pick = lambda M, K, N: names[l.cascmm_select_variant(M, N, K, K, N, N, 0, 0, 2, 0) & 0xFFFF]
    assert pick(1976, 1280, 10240) == "t256x320x32_w512_edge_bf16x2_tri" and pick(4096, 4096, 4096) == "t256x256x32_w512_edge_bf16x2_tri"
    assert pick(8192, 328, 2560) == "t256x320x32_w512_edge_bf16x2_tri" and "w512" not in pick(2496, 2504, 2500)
    assert pick(2048, 1280, 10240) == "t256x320x32_w512_bf16x2_tri" and "w512" not in pick(2048, 2048, 2048)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N", [(1330, 1768, 1856), (1775, 2408, 1088)])
def test_a_group_runs_problem_by_problem_where_that_is_faster(M, K, N):
    """K off 32: one launch has the eight-wave tiles only (138 and 155 us for three), three launches the kernels of single calls (89 and
    104), whose bits the results have."""
    from basedxl_amd import PreparedWeight, cascaded_lowp_matmul, cascaded_lowp_matmul_prepared
    g = torch.Generator(device="cuda:0").manual_seed(N)
    a = [torch.randn(M, K, device="cuda:0", generator=g) for _ in range(3)]
    w = [PreparedWeight(torch.randn(K, N, device="cuda:0", generator=g) * 0.02) for _ in range(3)]
    bias = [torch.randn(N, device="cuda:0", generator=g) for _ in range(3)]
    print("group", (M, K, N), flush=True)
    for got, x, p, b in zip(cascaded_lowp_matmul_prepared(a, w, biases=bias), a, w, bias):
        assert torch.equal(got, cascaded_lowp_matmul(x, p, bias=b))
