"""The native short cut of ordinary eager calls (csrc/host/native.cpp): the same results as the Python wrapper it stands for,
and None for every call that is not the ordinary case."""
import pytest
import torch

from basedxl_amd import BasedXLFusedKV, BasedXLLowPGEGLU, BasedXLLowPLinear, PreparedWeight, _lib, cascaded_lowp_matmul
from basedxl_amd.cascaded_lowp_matmul import tensor_scale_exp

_native = _lib.native()


def test_the_package_imports_before_anything_is_built(tmp_path):
    """A fresh checkout holds neither library, and the build itself imports the package."""
    import os
    import shutil
    import subprocess
    import sys

    import basedxl_amd
    src = os.path.dirname(basedxl_amd.__file__)
    shutil.copytree(src, tmp_path / "basedxl_amd", ignore=shutil.ignore_patterns("*.so", "build", "__pycache__"))
    code = ("from basedxl_amd import build, _lib\nassert build.sources()\n"
            "for load in (_lib.lib, _lib.native):\n    try:\n        load()\n    except ImportError as e:\n"
            "        assert 'basedxl_amd.build' in str(e), e\n    else:\n        raise SystemExit('loaded what is not there')\n")
    r = subprocess.run([sys.executable, "-c", code], cwd=tmp_path, env={**os.environ, "PYTHONPATH": str(tmp_path)}, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr


@pytest.mark.parametrize("in_its_place", [("_native.so", ""), ("_native.py", "matmul = prepared = init = lambda *_: None\n"),
                                          ("_native.py", "matmul = prepared = init = init_scales = lambda *_: None\n")],
                         ids=["no extension", "of a build before the fp8 calls", "half of one"])
def test_without_the_extension_calls_take_the_python_path(tmp_path, in_its_place):
    """An extension that does not load (a changed torch: here an empty file in its place), or one that an earlier build left, costs
    host time and a warning, no call."""
    import os
    import shutil
    import subprocess
    import sys

    import basedxl_amd
    src = os.path.dirname(basedxl_amd.__file__)
    shutil.copytree(src, tmp_path / "basedxl_amd", ignore=shutil.ignore_patterns("_native.so", "build", "__pycache__"))
    (tmp_path / "basedxl_amd" / in_its_place[0]).write_text(in_its_place[1])
    code = """
import warnings, torch, basedxl_amd as b
from basedxl_amd import _lib
op = lambda: b.cascaded_lowp_matmul(torch.randn(2, 64), torch.randn(64, 8))
lin, glu = b.BasedXLLowPLinear(torch.nn.Linear(64, 8)), b.BasedXLLowPGEGLU(torch.nn.Linear(64, 64))
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    for call in (op, lambda: lin(torch.randn(2, 64)), lambda: glu(torch.randn(2, 64)), op):
        try:
            call()
        except RuntimeError as e:
            assert "no CPU fallback" in str(e), e       # (the wrapper's own words: it was reached)
        else:
            raise SystemExit("ran on the CPU")
assert [w.category for w in seen] == [RuntimeWarning], [str(w.message) for w in seen]
assert _lib.short_cut().prepared(1, 2, 3) is None and _lib.lib().cascmm_version() == 100
"""
    r = subprocess.run([sys.executable, "-c", code], cwd=tmp_path, env={**os.environ, "PYTHONPATH": str(tmp_path)}, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr


def test_what_is_not_ordinary_is_left_to_the_wrapper():
    a, b = torch.randn(4, 8), torch.randn(8, 4)
    assert _native.matmul(a, b, None, None, None, "tri") is None                       # no GPU tensors
    assert _native.matmul(a.numpy(), b, None, None, None, "tri") is None
    assert _native.matmul(a, b, None, "fp7", 2 ** 80, "tri") is None and _native.matmul(a, b) is None
    assert _native.prepared(a, b, None, 8, 4, 0, 2, "tri", 0, False, 0) is None
    with pytest.raises(TypeError):
        _native.init([])


def test_prepared_weights_pickled_before_the_short_cut_still_load():
    """A pickled model holds its layers' PreparedWeight objects as plain attributes: those of before have no dtype code."""
    import pickle
    w = PreparedWeight.from_slots(torch.zeros(2 * 8 * 16 * 16, dtype=torch.uint8), 64, 16, torch.float32, "bf16", 2)
    del w.__dict__["dt"]
    assert set(w.__dict__) == {"K", "N", "shape", "lowp", "terms", "fmt", "dtype", "device", "glu", "out_features", "exp", "slots"}
    again = pickle.loads(pickle.dumps(w))
    with pytest.raises(RuntimeError, match="no CPU fallback"):          # (as far as a CPU tensor comes: the short cut has read its arguments)
        cascaded_lowp_matmul(torch.randn(2, 64), again)
    assert pickle.loads(pickle.dumps(again)).dt == again.dt == _lib.DT_F32


@pytest.mark.parametrize("lowp,terms,products,rows,raw", [("fp16", 3, "tri", 2, True), ("fp16", 3, "tri", 31, True), ("fp16", 3, "tri", 32, False),
                                                         ("bf16", 3, "tri", 16, True), ("bf16", 2, "full", 2, True), ("bf16", 2, "tri", 2, False),
                                                         ("fp8", 3, "tri", 2, True), ("fp8", 3, "tri", 4100, False)])
def test_eager_and_traced_layers_choose_the_same_weight(monkeypatch, lowp, terms, products, rows, raw):
    """A prepared layer asks one rule whether few rows take the raw weight, whichever way it is called."""
    from basedxl_amd import compiled
    from basedxl_amd.modules import lowp_linear
    taken, exp = [], torch.zeros(1, dtype=torch.int32) if lowp == "fp8" else None

    class Recorder:
        def matmul(*args):
            taken.append("raw")
            return args[0]

        def prepared(*args):
            taken.append("slots")
            return args[0]

        def fp8(*args):
            taken.append("slots" if args[8] else "raw")
            return args[0]

    layer = BasedXLLowPLinear(torch.nn.Linear(128, 64), lowp=lowp, terms=terms, products=products, prepared=True)
    layer._prepared_weight = PreparedWeight.from_slots(torch.zeros(16, dtype=torch.uint8), 128, 64, torch.float32, lowp, terms, exp=exp)
    layer._weight_exp = exp
    monkeypatch.setattr(lowp_linear._lib, "short_cut", lambda: Recorder)
    x = torch.zeros(rows, 128)
    layer(x)
    monkeypatch.undo()
    monkeypatch.setattr(PreparedWeight, "usable_with", lambda self, a2, products: True)
    monkeypatch.setattr(compiled, "cascaded_lowp_matmul", lambda a, b, **_: taken.append("slots" if isinstance(b, PreparedWeight) else "raw") or a.new_empty(rows, 64))
    compiled.cascade_linear._init_fn(x, layer.weight, layer._prepared_weight.slots, None, lowp, terms, products, False, exp)
    assert taken == ["raw" if raw else "slots"] * 2


def test_slots_are_checked_against_the_layout():
    w = PreparedWeight.from_slots(torch.zeros(2 * 12 * 64 * 16, dtype=torch.uint8), 96, 64, torch.float32, "bf16", 2)
    w.check_slots()
    for n in (16, 2 * 12 * 64 * 16 - 16, 2 * 16 * 64 * 16):
        w.slots = torch.zeros(n, dtype=torch.uint8)
        with pytest.raises(ValueError, match="slots"):
            w.check_slots()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,N", [(2, 1280, 320), (154, 320, 200), (512, 640, 640)])
def test_same_bits_as_the_wrapper(gpu_device, dtype, M, K, N):
    """`out=` takes the Python path; the result must be the same kernel's, bit for bit, raw and prepared, with and without a
    bias, batch dimensions, row strides, and inside a device graph."""
    g = torch.Generator().manual_seed(K)
    rn = lambda *s: (torch.randn(*s, generator=g) * 0.1).to("cuda:0").to(dtype)
    a, w, bias, frame = rn(M, K), rn(K, N), rn(N), rn(M, K + 8)
    pw = PreparedWeight(w)
    for x in (a, frame[:, :K], a.view(M // 2, 2, K)):
        for b in (w, pw):
            for bb in (None, bias):
                out = torch.empty(M, N, dtype=dtype, device="cuda:0")
                want = cascaded_lowp_matmul(x, b, bias=bb, out=out)
                got = cascaded_lowp_matmul(x, b, bias=bb)
                assert got.shape == (*x.shape[:-1], N) and torch.equal(got, want)
    assert _native.matmul(a, w, None, None, None, "tri") is not None                     # (the short cut did run)
    assert _native.matmul(a.t(), w, None, None, None, "tri") is None and _native.matmul(a, w.t(), None, None, None, "tri") is None
    assert _native.matmul(a, w, bias[:-1], None, None, "tri") is None and _native.matmul(a, w, None, "fp8", 3, "tri") is None
    want = cascaded_lowp_matmul(a, w)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        got = cascaded_lowp_matmul(a, w)
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N", [(64, 128, 64), (300, 456, 212), (2, 1280, 640), (40, 1280, 1281)])
def test_fp8_calls_are_those_of_the_python_path(gpu_device, M, K, N):
    """Raw and prepared, scale of the weight kept or found, bit for bit against `out=`, and inside a device graph."""
    g = torch.Generator().manual_seed(K)
    rn = lambda *s: torch.randn(*s, generator=g).to("cuda:0")
    a, w, bias, frame = rn(M, K), rn(K, N) * 0.02, rn(N), rn(M, K + 8)
    weights = [w] + ([PreparedWeight(w, lowp="fp8", terms=3)] if K % 64 == 0 and N % 4 == 0 else [])
    exp = tensor_scale_exp(w)
    for x in (a, frame[:, :K], a.view(M // 2, 2, K)):
        for b in weights:
            for bb, e in ((None, None), (bias, None), (bias, exp)):
                kw = dict(bias=bb) if isinstance(b, PreparedWeight) else dict(bias=bb, lowp="fp8", terms=3, b_exp=e)
                want = cascaded_lowp_matmul(x, b, out=torch.empty(M, N, device="cuda:0"), **kw)
                got = cascaded_lowp_matmul(x, b, **kw)
                assert got.shape == (*x.shape[:-1], N) and torch.equal(got, want.view(got.shape))
    assert _native.fp8(a, w, bias, exp, 0, 0, 3, "tri", False) is not None and _native.fp8(a, w, None, None, 0, 0, 3, "tri", False) is not None
    for args in ((a.half(), w, None, exp, 0, 0, 3, "tri", False), (a, w.t(), None, exp, 0, 0, 3, "tri", False), (a, w, bias[:-1], exp, 0, 0, 3, "tri", False),
                 (a, w, None, exp.float(), 0, 0, 3, "tri", False), (a, w, None, exp, 0, 0, None, "tri", False), (a, w, None, exp, 0, 0, 3, "all", False),
                 (a, torch.zeros(64, dtype=torch.uint8, device="cuda:0"), None, exp, K, N, 3, "tri", True), (a, w, None)):
        assert _native.fp8(*args) is None
    want = cascaded_lowp_matmul(a, w, lowp="fp8", terms=3)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        assert _native.fp8(a, w, None, exp, 0, 0, 3, "tri", False) is None         # (a recorded call: its own scratch, kept by the Python path)
        got = cascaded_lowp_matmul(a, w, lowp="fp8", terms=3)
    for _ in range(3):
        got.zero_()
        graph.replay()
        assert torch.equal(cascaded_lowp_matmul(a, w, lowp="fp8", terms=3), want)
        torch.cuda.synchronize()
        assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,K,N", [(1, 640, 1280), (33, 640, 1280), (204, 1280, 1280), (205, 1280, 1312), (257, 4160, 320)])
def test_fp8_layers_on_either_side_of_the_raw_weight_s_rule(gpu_device, rows, K, N):
    """Prepared and not, before and after prepare(), few tiles and more: the same products, added in another order."""
    torch.manual_seed(rows)
    lin, x = torch.nn.Linear(K, N).to("cuda:0").requires_grad_(False), torch.randn(rows, K, device="cuda:0")
    want = x.double() @ lin.weight.double().t() + lin.bias.double()
    for prepared in (False, True):
        mod = BasedXLLowPLinear(lin, lowp="fp8", terms=3, prepared=prepared)
        first = mod(x)
        mod.prepare()
        assert torch.equal(mod(x), first)
        assert float((first.double() - want).norm() / want.norm()) < 1.4e-4       # (four times the cascade's own error, 3.5e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("lowp,terms,products", [("fp16", 3, "tri"), ("bf16", 3, "tri"), ("bf16", 2, "full"), ("bf16", 2, "tri")])
@pytest.mark.parametrize("rows", [2, 31, 33])
def test_first_later_and_traced_calls_of_a_prepared_layer_have_the_same_bits(gpu_device, lowp, terms, products, rows):
    from basedxl_amd.compiled import cascade_linear
    torch.manual_seed(rows)
    lin, x = torch.nn.Linear(1280, 640).to("cuda:0").requires_grad_(False), torch.randn(rows, 1280, device="cuda:0")
    mod = BasedXLLowPLinear(lin, lowp=lowp, terms=terms, products=products, prepared=True)
    first = mod(x)
    mod.prepare()
    assert torch.equal(mod(x), first)
    assert torch.equal(cascade_linear(x, mod.weight, mod._prepared_weight.slots, mod.bias, lowp, terms, products, False, None), first)
    if rows < 32 and (lowp, terms, products) != ("bf16", 2, "tri"):
        assert torch.equal(BasedXLLowPLinear(lin, lowp=lowp, terms=terms, products=products)(x), first)


@pytest.mark.gpu
def test_slots_of_another_layout_are_refused(gpu_device):
    """A buffer that is shorter or longer than the weight's slots, as one kept in a file from another layout would be."""
    w, x = PreparedWeight(torch.randn(96, 64, device="cuda:0")), torch.randn(40, 96, device="cuda:0")
    want = cascaded_lowp_matmul(x, w)
    for n in (-16, 16, 2 * 4 * 64 * 16):
        slots = torch.zeros(w.slots.numel() + n, dtype=torch.uint8, device="cuda:0")
        other = PreparedWeight.from_slots(slots, 96, 64, torch.float32, "bf16", 2)
        assert _native.prepared(x, slots, None, 96, 64, other.fmt, 2, "tri", other.dt, False, 0) is None
        with pytest.raises(ValueError, match="slots"):
            cascaded_lowp_matmul(x, other)
    assert torch.equal(cascaded_lowp_matmul(x, PreparedWeight.from_slots(w.slots, 96, 64, torch.float32, "bf16", 2)), want)


@pytest.mark.gpu
def test_gated_layer_refuses_activations_of_another_dtype(gpu_device):
    """A 16-bit weight kept as two bf16 terms has fp32 kernels, but the layer's input has its weight's dtype."""
    mod = BasedXLLowPGEGLU(torch.nn.Linear(64, 128).to("cuda:0", torch.bfloat16), lowp="bf16", terms=2)
    mod.prepare()
    with pytest.raises(TypeError):
        mod(torch.randn(40, 64, device="cuda:0"))


@pytest.mark.gpu
def test_modules_take_it_on_another_stream_and_after_a_move_of_shape(gpu_device):
    torch.manual_seed(3)
    lin = torch.nn.Linear(640, 320).to("cuda:0")
    mod, kv = BasedXLLowPLinear(lin, prepared=True), BasedXLFusedKV(lin, torch.nn.Linear(640, 320).to("cuda:0"))
    for rows in (2, 40, 300, 2):
        x = torch.randn(rows, 640, device="cuda:0")
        want = BasedXLLowPLinear(lin)(x)
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            y = mod(x)
            k, v = kv(x)
        s.synchronize()
        torch.testing.assert_close(y, want, rtol=1e-5, atol=1e-5)
        torch.testing.assert_close(k, want, rtol=1e-5, atol=1e-5)
        assert k.shape == v.shape == (rows, 320)
