"""The kernels that split K over the eight waves of a workgroup (cascmm_wavek_kernel.h): every tile, at the edges of its tile, of a
32-k step, of the straight code's numbers of steps and of the ring."""
import pytest
import torch

from basedxl_amd import PreparedWeight, _lib, cascaded_lowp_matmul
from basedxl_amd.cascaded_lowp_matmul import cascaded_lowp_matmul_glu

pytestmark = pytest.mark.gpu

_TILES = [n for n in _lib.variant_names() if "_wavek_" in n]


@pytest.mark.parametrize("name", _TILES)
@pytest.mark.parametrize("K", [1, 3, 32, 33, 72, 255, 264, 511, 1016, 1280, 1310, 2081, 2568, 3333])
def test_every_number_of_steps_is_exact_on_integers(name, K):
    """One, two, ... steps per wave and the trips behind the straight code; K off the steps and off 16-byte chunks, NaNs between the rows
    of A and beside B's columns, columns and rows past the edge of C untouched."""
    bm, bn = (int(x) for x in name.split("_")[0][1:].split("x")[:2])
    lowp, terms = name.split("_")[2].split("x")
    g = torch.Generator().manual_seed(K)
    for M, N in ((bm, bn), (7, 2 * bn + 1), (bm + 9, bn - 3)):
        a, b = (torch.randint(-60, 61, s, generator=g) for s in ((M, K), (K, N)))
        frame = torch.full((M, K + 3), float("nan"), device="cuda:0")
        frame[:, :K] = a.float().to("cuda:0")
        out = torch.full((M + 1, N + 1), -77.0, device="cuda:0")
        print("wavek", name, (M, K, N), flush=True)
        got, w, variant = out[:M, :N], b.float().to("cuda:0"), _lib.variant_names().index(name)
        if name.endswith("_bpre"):
            if K % 8 != 0 or (K < 64 and K % 32 != 0):
                with pytest.raises(_lib.CascmmError):
                    cascaded_lowp_matmul(frame[:, :K], PreparedWeight(w, lowp=lowp, terms=int(terms)), variant=variant)
                continue
            assert torch.equal(cascaded_lowp_matmul(frame[:, :K], PreparedWeight(w, lowp=lowp, terms=int(terms)), variant=variant).cpu().long(), a @ b), (M, N)
            continue
        cascaded_lowp_matmul(frame[:, :K], w, out=got, lowp=lowp, terms=int(terms), variant=variant)
        assert torch.equal(got.cpu().long(), a @ b), (M, N)
        assert bool((out[M] == -77.0).all()) and bool((out[:, N] == -77.0).all())


@pytest.mark.parametrize("name", _TILES)
@pytest.mark.parametrize("side", ["A", "B"])
def test_every_term_of_either_operand_reaches_the_result(name, side):
    """The other operand picks one k for each row or column (one +-1, zeros): the result is the picked values with their signs, exact where
    the terms hold all their bits.  Two bf16 terms hold integers below 2^16, three fp8 terms below 2^12, three fp16 terms 23 bits."""
    bm, bn = (int(x) for x in name.split("_")[0][1:].split("x")[:2])
    lowp, terms = name.split("_")[2].split("x")
    bits, unit = {"bf16": (16, 1.0), "fp8": (12, 1.0), "fp16": (23, 2.0 ** -8)}[lowp]
    g = torch.Generator().manual_seed(bits)
    for M, K, N in ((7, 1304, 2 * bn + 1), (bm + 9, 264, bn), (2 * bm, 2568, bn + 8)):
        rows, cols = (M, K) if side == "A" else (K, N)
        values = torch.randint(-2 ** bits + 1, 2 ** bits, (rows, cols), generator=g).double() * unit
        count = N if side == "A" else M
        k, sign = torch.randint(0, K, (count,), generator=g), torch.randint(0, 2, (count,), generator=g) * 2.0 - 1
        k[0], k[-1] = K - 1, 0
        pick = torch.zeros(count, K, dtype=torch.double)
        pick[torch.arange(count), k] = sign.double()
        a, b = (values, pick.T.contiguous()) if side == "A" else (pick, values)
        want = values[:, k] * sign if side == "A" else values[k] * sign[:, None]
        w = b.float().to("cuda:0")
        print("wavek terms", name, side, (M, K, N), flush=True)
        options = {} if name.endswith("_bpre") else dict(lowp=lowp, terms=int(terms))
        got = cascaded_lowp_matmul(a.float().to("cuda:0"), PreparedWeight(w, lowp=lowp, terms=int(terms)) if name.endswith("_bpre") else w,
                                   variant=_lib.variant_names().index(name), **options)
        assert torch.equal(got.cpu().double(), want), (M, K, N)


@pytest.mark.parametrize("name", [n for n in _TILES if n.endswith("_bpre") and n.split("x")[1] == "64"])
@pytest.mark.parametrize("M,K,N", [(7, 72, 64), (8, 1280, 128), (9, 264, 192), (17, 520, 320), (81, 2568, 704)])
def test_the_gated_store(name, M, K, N):
    """value * gelu(gate) of integers below 2^18: sums exact, the gate within an fp32 ulp of the exact one (4e-7 + 2e-7 |gate|), the product
    rounded once (2^-24 of it)."""
    g = torch.Generator().manual_seed(M + K + N)
    a, b, bias = (torch.randint(-9, 10, s, generator=g) for s in ((M, K), (K, N), (N,)))
    value, gate = (a @ b + bias).double().chunk(2, -1)
    want = value * torch.nn.functional.gelu(gate)
    print("wavek gated", name, (M, K, N), flush=True)
    frame = torch.full((M, K + 4), float("nan"), device="cuda:0")
    frame[:, :K] = a.float().to("cuda:0")
    got = cascaded_lowp_matmul(frame[:, :K], PreparedWeight(b.float().to("cuda:0"), glu=True), bias=bias.float().to("cuda:0"),
                               variant=_lib.variant_names().index(name)).cpu().double()
    assert bool(((got - want).abs() <= value.abs() * (4e-7 + 2e-7 * gate.abs()) + 2.0 ** -24 * want.abs()).all())


def test_the_gated_store_is_on_prepared_weights_only():
    for name in _TILES:
        if not name.endswith("_bpre"):
            a, b = torch.randn(8, 64, device="cuda:0"), torch.randn(64, 64, device="cuda:0")
            with pytest.raises(_lib.CascmmError):
                cascaded_lowp_matmul_glu(a, b, variant=_lib.variant_names().index(name))


@pytest.mark.parametrize("name", [n for n in _TILES if n.startswith("t16x")])
@pytest.mark.parametrize("M", [1, 2, 8, 9])
def test_few_rows_on_either_side_of_the_half_filled_stage(name, M):
    """Up to eight rows are half a stage of a 16-row tile, which is all that is fetched and read: up to every stage of the ring and past it."""
    lowp, terms = name.split("_")[2].split("x")
    g = torch.Generator().manual_seed(M)
    for K in (256, 1280, 1536, 2816):
        a, b = (torch.randint(-60, 61, s, generator=g) for s in ((M, K), (K, 96)))
        w = b.float().to("cuda:0")
        print("wavek rows", name, M, K, flush=True)
        got = cascaded_lowp_matmul(a.float().to("cuda:0"), PreparedWeight(w, lowp=lowp, terms=int(terms)) if name.endswith("_bpre") else w,
                                   **({} if name.endswith("_bpre") else dict(lowp=lowp, terms=int(terms))), variant=_lib.variant_names().index(name))
        assert torch.equal(got.cpu().long(), a @ b), K


@pytest.mark.parametrize("M,K,N", [(2, 1280, 1280), (16, 2047, 477), (130, 1281, 448), (600, 600, 600), (1024, 1024, 1024), (3, 5120, 40)])
def test_a_call_repeats_its_bits_and_keeps_non_finite_values_to_their_rows(M, K, N):
    a, b = torch.randn(M, K, device="cuda:0"), torch.randn(K, N, device="cuda:0")
    a[M // 2, K - 1] = float("inf")
    b[0, N // 3] = float("nan")
    print("wavek", (M, K, N), flush=True)
    first = cascaded_lowp_matmul(a, b)
    for _ in range(3):
        assert torch.equal(cascaded_lowp_matmul(a, b).nan_to_num(7.0), first.nan_to_num(7.0))
    bad = ~torch.isfinite(first)
    assert bool(bad[M // 2].all()) and bool(bad[:, N // 3].all()) and int(bad.sum()) == M + N - 1
    want = a.double() @ b.double()
    ok = ~bad
    assert float((first.double() - want)[ok].norm() / want[ok].norm()) < 1.8e-5


@pytest.mark.parametrize("M,K,N", [(2, 1280, 1280), (64, 520, 640), (200, 2560, 640), (640, 1280, 1280)])
@pytest.mark.parametrize("glu", [False, True])
def test_the_kernel_that_a_prepared_call_is_said_to_launch(M, K, N, glu):
    """Its bits are those of that kernel by index."""
    g = torch.Generator(device="cuda:0").manual_seed(M)
    a, w = torch.randn(M, K, device="cuda:0", generator=g), PreparedWeight(torch.randn(K, N, device="cuda:0", generator=g), glu=glu)
    v = _lib.lib().cascmm_call_variant_prepared(a.data_ptr(), int(glu), M, N, K, K, N // 2 if glu else N, 0, 0, 2, 0,
                                                _lib.lib().cascmm_workspace_bytes(M, N, K, 0, 0, 2, 0))
    print("wavek call", (M, K, N), glu, _lib.variant_names()[v & 0xFFFF], flush=True)
    if "_wavek_" in _lib.variant_names()[v]:      # (the others may split K over workgroups, which the index alone does not)
        assert torch.equal(cascaded_lowp_matmul(a, w), cascaded_lowp_matmul(a, w, variant=v))
