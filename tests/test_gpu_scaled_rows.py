"""Three fp16 terms of few rows whose K or N fits no whole stages: K over the eight waves, each tile scaled by its own workgroup where
its values need it, in the place of the slot kernels, which scale both operands in launches of their own."""
import pytest
import torch

from basedxl_amd import _lib, cascaded_lowp_matmul

NAMES = [n for n in _lib.variant_names() if n.endswith("_scaled")]
SHAPES = [(1, 33, 5), (17, 100, 47), (33, 1193, 70), (5, 2570, 129)]


def test_few_rows_take_the_kernel_that_scales_its_own_tiles():
    l, names = _lib.lib(), _lib.variant_names()

    def kernel(M, K, N, ws=None):
        return names[l.cascmm_call_variant(1 << 40, 2 << 40, M, N, K, K, N, N, 0, 1, 3, 0, l.cascmm_workspace_bytes(M, N, K, 0, 1, 3, 0) if ws is None else ws) & 0xFFFF]

    for shape in ((5, 3164, 3136), (6, 1193, 462), (33, 1612, 1374)):
        assert kernel(*shape).endswith("_scaled"), shape
        assert kernel(*shape, ws=0) == kernel(*shape), shape       # (it needs no room for slots)
    for shape in ((882, 899, 3968), (300, 576, 4480), (2048, 1281, 1280)):
        assert "_wavek_" not in kernel(*shape), shape


def _check(a, b, c, bias=None):
    """Each of a wave's sums over K / 256 steps is rounded once per MFMA and folded in blocks, the waves' eight are added: below 16 + K / 256
    roundings of 2^-24 of the sum of magnitudes; the terms hold an operand to 2^-39 of the largest element of its tile (half of 2^-46 where that
    is 2^-8, the least that is taken unscaled; tiles of 32 at most): twice that, for the products of two such roundings and the dropped ones."""
    ad, bd = a.double(), b.double()
    ref = ad @ bd + (0 if bias is None else bias.double())
    K = a.shape[1]
    mag = ad.abs() @ bd.abs()
    tile_a = torch.cat([r.abs().amax().expand(r.shape[0]) for r in ad.split(32)])[:, None]
    tile_b = torch.cat([r.abs().amax().expand(r.shape[1]) for r in bd.split(32, 1)])[None, :]
    bound = (16 + K / 256) * 2.0 ** -24 * mag + 2.0 ** -38 * (tile_a * bd.abs().sum(0)[None, :] + tile_b * ad.abs().sum(1)[:, None])
    bad = ~((c.double() - ref).abs() <= bound + ref.abs() * 2.0 ** -23)
    assert not bad.any(), float(((c.double() - ref).abs() / bound).max())


@pytest.mark.gpu
@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_scaled_rows(M, K, N, name):
    print(name, M, K, N, flush=True)
    v = _lib.variant_names().index(name)
    g = torch.Generator(device="cuda").manual_seed(M + N)
    a, b = (torch.randn(s, device="cuda", generator=g) for s in ((M, K), (K, N)))
    bias = torch.randn(N, device="cuda", generator=g)

    def run(x, y, **kw):
        return cascaded_lowp_matmul(x, y, lowp="fp16", terms=3, variant=v, **kw)

    # as they are; beyond fp16's range; below what its terms hold; both; rows of A that lie apart
    _check(a, b, run(a, b, bias=bias), bias)
    for ea, eb in ((40, -30), (0, 17), (-25, 0), (-50, 55)):
        _check(a * 2.0 ** ea, b * 2.0 ** eb, run(a * 2.0 ** ea, b * 2.0 ** eb))
    wide = torch.full((M, K + 3), 1.0e30, device="cuda")
    wide[:, :K] = a
    _check(a, b, run(wide[:, :K], b))
    # operands without a positive element, of zeros, of whole numbers
    _check(-a.abs(), -b.abs(), run(-a.abs(), -b.abs()))
    # waves whose first steps are small, zero, large or of another size than what follows
    k = torch.arange(K, device="cuda") // 32
    for first, rest in ((-30, 0), (0, -30), (-30, 30), (30, -12), (-9, 12)):
        x = a * 2.0 ** torch.where(k < 8, first, rest)
        _check(x, b, run(x, b))
        y = b * 2.0 ** torch.where(k < 8, first, rest)[:, None]
        _check(a, y, run(a, y))
    x, y = a * 2.0 ** (10.0 * (k % 5) - 20), b * (k % 3 != 0)[:, None] * 2.0 ** -14
    _check(x, y, run(x, y))
    # ... and computed once, with the unscaled kernel's bits (a second pass splits small elements into other terms and folds its sums elsewhere)
    once, low = _lib.variant_names().index(name[:-len("_scaled")]), a.clamp(max=0) * torch.logspace(-1.5, 0, K, device="cuda")
    for x, y in ((a, b), (low, b), (a, -b.abs())):
        assert torch.equal(run(x, y), cascaded_lowp_matmul(x, y, lowp="fp16", terms=3, variant=once))
    assert not run(torch.zeros_like(a), b).any() and not run(a, torch.zeros_like(b)).any()
    ia, ib = (a * 8).round(), (b * 8).round()
    assert torch.equal(run(ia, ib).double(), ia.double() @ ib.double())
    # one element out of range in a row of each 32, the last column of B not finite
    big, nan = a.clone(), b.clone()
    big[::32, K - 1] = 3.0e6
    _check(big, b, run(big, b))
    nan[0, N - 1] = float("nan")
    inf = a.clone()
    inf[M - 1, K // 2] = float("inf")
    c = run(inf, nan)
    assert not torch.isfinite(c[M - 1]).any() and torch.isnan(c[:, N - 1]).all()
    if M > 1:
        _check(inf[:M - 1], nan[:, :N - 1], c[:M - 1, :N - 1])


@pytest.mark.gpu
@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("top", [2.0 ** -8 * (1 + 2.0 ** -10), 2.0 ** -8 * (1 - 2.0 ** -10), 2.0 ** -10, 2.0 ** -13 * 1.01, 2.0 ** -13 * 0.99])
def test_scaled_rows_near_the_least_unscaled_tile(top, name):
    """Operands whose largest element meets zeros and whose other elements are 2^-20 of it: the results' errors are what the terms resolve
    (unscaled 2^-47 an element, against the bound 2^-38 of the largest), the roundings of the sums 2^-40 of that."""
    print(name, top, flush=True)
    v = _lib.variant_names().index(name)
    g = torch.Generator(device="cuda").manual_seed(7)
    M, K, N = 19, 41, 45
    a, b = torch.randn(M, K, device="cuda", generator=g), torch.randn(K, N, device="cuda", generator=g)
    a[:, 5:], b[5:] = 0, 0
    low_a, low_b, plain_a, plain_b = a * (top * 2.0 ** -20), b * (top * 2.0 ** -20), a.clone(), b.clone()
    low_a[:, 0], plain_b[0] = top, 0            # A's largest elements meet zeros
    low_b[0], plain_a[:, 0] = top, 0            # B's
    low_b2, low_a2 = low_b.clone(), low_a.clone()
    low_b2[0], low_b2[7], low_a2[:, 7] = 0, top, 0          # both
    for x, y in ((low_a, plain_b), (plain_a, low_b), (low_a2, low_b2)):
        _check(x, y, cascaded_lowp_matmul(x, y, lowp="fp16", terms=3, variant=v))


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N", [(5, 3164, 3136), (33, 1612, 1374)])
def test_few_rows_without_a_workspace_hold_values_beyond_the_format(M, K, N):
    print(M, K, N, flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    a, b = torch.randn(M, K, device="cuda", generator=g) * 2.0 ** 20, torch.randn(K, N, device="cuda", generator=g)
    c = torch.full((M, N), 7.0, device="cuda")
    st = _lib.lib().cascmm_gemm(a.data_ptr(), b.data_ptr(), c.data_ptr(), None, M, N, K, K, N, N, 0, 1, 3, 0, None, None, 0,
                                torch.cuda.current_stream().cuda_stream)
    assert st == 0
    _check(a, b, c)
    assert torch.equal(c, cascaded_lowp_matmul(a, b, lowp="fp16", terms=3))
