"""Shapes whose rows are not whole 16-byte chunks, 32-k steps or column tiles, on the fast kernels: tails of K read as zeros,
rows on any dword, odd N, operands copied into the workspace first (cascmm_api.hip: row_fit, relay_of, rounded_up)."""
import pytest
import torch

from basedxl_amd import PreparedWeight, _lib, cascaded_lowp_matmul, cascaded_lowp_matmul_grouped

pytestmark = pytest.mark.gpu

# (M, K, N): K = 4 mod 8 and 8 mod 32, odd K and N, K below one stage, more than one tile each way, a K deep enough for
# every wave of the kernels that split it, one row
SHAPES = [(333, 456, 211), (44, 1124, 1728), (1, 33, 5), (257, 1061, 641), (300, 744, 744), (65, 100, 448), (129, 1001, 1003),
          (600, 72, 1002), (17, 20, 19)]
CASCADES = [(torch.float32, None, None), (torch.float32, "fp8", 3), (torch.float32, "fp16", 3), (torch.float16, None, None),
            (torch.bfloat16, None, None)]


@pytest.mark.parametrize("dtype,lowp,terms", CASCADES)
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_ragged_shapes_are_exact_on_integers(gpu_device, dtype, lowp, terms, M, K, N):
    """Integers that the first terms hold exactly (|x| <= 7; 16-bit tensors: |x| <= 1) whose sums stay below 2^24 (2^8 for
    the 16-bit results: 6 sqrt(1061 x 4 / 9) = 130): the result must be the exact one, the gaps between the rows of A (NaN)
    must never reach it, and the gaps of the result must stay as they were."""
    hi = 7 if dtype == torch.float32 else 1
    g = torch.Generator().manual_seed(M + K + N)
    a, b, bias = (torch.randint(-hi, hi + 1, s, generator=g) for s in ((M, K), (K, N), (N,)))
    want = (a @ b + bias).to("cuda:0")
    assert int(want.abs().max()) < (2 ** 24 if dtype == torch.float32 else 2 ** 8)
    kw = {} if lowp is None else dict(lowp=lowp, terms=terms)
    bd, biasd = b.to(dtype).to("cuda:0"), bias.to(dtype).to("cuda:0")
    weight = PreparedWeight(bd) if lowp is None and K % 8 == 0 and K >= 64 else None
    for pad in (0, 1, 2, 8):          # row strides of every alignment
        print("ragged", dtype, lowp, (M, K, N), "pad", pad, flush=True)
        frame = torch.full((M, K + pad), float("nan"), dtype=dtype, device="cuda:0")
        frame[:, :K] = a.to(dtype).to("cuda:0")
        out = torch.full((M + 1, N + 1), -77.0, dtype=dtype, device="cuda:0")
        cascaded_lowp_matmul(frame[:, :K], bd, bias=biasd, out=out[:M, :N], **kw)
        assert torch.equal(out[:M, :N].double(), want.double()), pad
        assert bool((out[:M, N] == -77.0).all()) and bool((out[M] == -77.0).all()), pad
        if lowp is None:
            for o in cascaded_lowp_matmul_grouped([frame[:, :K]] * 2, [bd, bd], biases=[biasd, biasd]):
                assert torch.equal(o.double(), want.double()), pad
        if weight is not None:
            assert torch.equal(cascaded_lowp_matmul(frame[:, :K], weight, bias=biasd).double(), want.double()), pad
    flat = torch.full((M * K + 1,), float("nan"), dtype=dtype, device="cuda:0")       # the first row off its alignment too
    flat[1:] = a.to(dtype).to("cuda:0").flatten()
    assert torch.equal(cascaded_lowp_matmul(flat[1:].view(M, K), bd, bias=biasd, **kw).double(), want.double())


@pytest.mark.parametrize("name", ["k64x160x16_wk4_bf16x2_tri", "t32x32x32_wavek_bf16x2_tri", "t32x64x32_wavek_bf16x2_tri",
                                  "k64x160x16_wk4_bf16x2_tri_bpre", "k64x80x32_wk4_bf16x2_tri_bpre"])
@pytest.mark.parametrize("M,K,N", [(70, 136, 163), (65, 72, 321), (33, 1064, 82)])
def test_each_kernel_with_a_tail_is_exact_on_integers(gpu_device, name, M, K, N):
    g = torch.Generator().manual_seed(K + N)
    a, b = (torch.randint(-100, 101, s, generator=g) for s in ((M, K), (K, N)))
    ad, bd = a.float().to("cuda:0"), b.float().to("cuda:0")
    print("tail", name, (M, K, N), flush=True)
    got = cascaded_lowp_matmul(ad, PreparedWeight(bd) if name.endswith("_bpre") else bd, variant=_lib.variant_names().index(name))
    assert torch.equal(got.cpu().long(), a @ b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,N", [(70, 96, 163), (300, 72, 644), (129, 360, 1003), (65, 104, 64)])
def test_nothing_past_a_prepared_buffer_is_read_into_the_result(gpu_device, dtype, M, K, N):
    """Slots in the middle of a buffer of NaNs, K off the 64-k stages: every kernel for such a weight, exact on integers (16-bit
    results: |x| <= 1, sums of at most 360 products below 2^8)."""
    hi = 100 if dtype == torch.float32 else 1
    g = torch.Generator().manual_seed(K + N)
    a, b = (torch.randint(-hi, hi + 1, s, generator=g) for s in ((M, K), (K, N)))
    w = PreparedWeight(b.to(dtype).to("cuda:0"))
    frame = torch.full((w.slots.numel() + 2 * 128 * N * 16,), 0xFF, dtype=torch.uint8, device="cuda:0")
    inner = frame[128 * N * 16:][:w.slots.numel()]
    inner.copy_(w.slots)
    moved = PreparedWeight.from_slots(inner, K, N, dtype, w.lowp, w.terms)
    frame_a = torch.full((M, K + 8), float("nan"), dtype=dtype, device="cuda:0")
    frame_a[:, :K] = a.to(dtype).to("cuda:0")
    tag = {torch.float32: ("bf16x2_tri_bpre",), torch.float16: ("_h16_fp16x1_bpre_ioh",), torch.bfloat16: ("_h16_bf16x1_bpre_iob",)}[dtype]
    ran = 0
    for vi, name in [(-1, "automatic")] + [(vi, n) for vi, n in enumerate(_lib.variant_names()) if n.endswith(tag)]:
        print("slots", dtype, (M, K, N), name, flush=True)
        try:
            got = cascaded_lowp_matmul(frame_a[:, :K], moved, variant=vi)
        except _lib.CascmmError as e:
            assert vi >= 0 and e.status == -8      # (that kernel takes whole stages or tiles only: refused on the host)
            continue
        assert torch.equal(got.cpu().double(), (a @ b).to(dtype).double()), name
        ran += 1
    assert ran >= 3                                # (of the fp32 ones the two K-over-waves kernels take any shape)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,N,lda", [(300, 64, 33, 1 << 21), (70, 72, 641, (1 << 21) + 2), (5, 100, 65, 1 << 22)])
def test_rows_far_apart_next_to_a_weight_of_odd_width(gpu_device, dtype, M, K, N, lda):
    """A raw 16-bit weight of odd width is copied into slots first, and slots have the kernels with 32-bit offsets only; rows of A
    2^21 elements apart are beyond those (exact on integers)."""
    g = torch.Generator().manual_seed(K + N)
    a, b = (torch.randint(-1, 2, s, generator=g) for s in ((M, K), (K, N)))
    wide = torch.empty(M * lda, dtype=dtype, device="cuda:0").as_strided((M, K), (lda, 1))
    wide.copy_(a.to(dtype))
    bd = b.to(dtype).to("cuda:0")
    print("far apart", dtype, (M, K, N, lda), flush=True)
    assert torch.equal(cascaded_lowp_matmul(wide, bd).cpu().long(), a @ b)
    for o in cascaded_lowp_matmul_grouped([wide, wide], [bd, bd]):
        assert torch.equal(o.cpu().long(), a @ b)
