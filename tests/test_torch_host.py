"""The native form of the tensor interface (fmha_amd/csrc/fmha_decode_torch.cpp):
what it takes gives the Python form's results, and what it leaves alone
raises the Python form's errors."""
import math
import sys
import warnings

import pytest
import torch

import fmha_amd
from fmha_amd import decode


class _Leaves:
    """Stands in for the native module: leaves every call to Python."""

    def __getattr__(self, name):
        return lambda *args: None


def _cpu_case():
    bf = torch.bfloat16
    return torch.zeros(2, 4, 64, dtype=bf), torch.zeros(2, 3, 4, 64, dtype=bf), torch.zeros(2, 3, 4, 64, dtype=bf)


def test_leaves_what_it_does_not_know():
    """CPU tensors, other types, subclasses and odd flags: None, never an
    error or a call."""
    n = decode._load_native()
    q, k, v = _cpu_case()

    class Sub(torch.Tensor):
        pass

    for args in [(q, k, v, None, None, None, None, False, False, False),
                 (1, k, v, None, None, None, None, False, False, False),
                 (q.as_subclass(Sub), k, v, None, None, None, None, False, False, False),
                 (q, None, v, None, 3, "x", None, 0, False, 1)]:
        assert n.decode(*args) is None
    assert n.splitkv(q, k, v, None, 3, None, None, None) is None
    assert n.strided(q, k, v, None, None, None, None) is None
    assert n.paged(q, k, v, q, q, None, None, None, None) is None
    with pytest.raises(TypeError):
        n.decode(q)
    with pytest.raises(TypeError):
        n.bind(1)
    with pytest.raises(ValueError):
        n.bind(*([0] * 12))


def test_works_without_the_module(monkeypatch):
    """Where the native module does not load, one warning, and every call is
    the Python form's, with its errors; the library itself still has to be
    there."""
    monkeypatch.setitem(sys.modules, "fmha_amd._host", None)
    monkeypatch.setattr(decode, "_native", None)
    q, k, v = _cpu_case()
    lens = torch.zeros(2, dtype=torch.int32)
    with pytest.warns(RuntimeWarning, match="native call path"):
        with pytest.raises(ValueError, match="q must be"):
            fmha_amd.fmha_decode(q, k, v)
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        with pytest.raises(ValueError):
            fmha_amd.fmha_decode_splitkv(q, k, v, lens, 3)
        with pytest.raises(ValueError):
            fmha_amd.fmha_decode_strided(q, k, v)
        with pytest.raises(ValueError):
            fmha_amd.fmha_decode_paged(q, k, v, lens.view(2, 1), lens)
    monkeypatch.setattr(decode, "_native", None)
    monkeypatch.setattr(decode._lib, "_lib", None)
    monkeypatch.setattr(decode._lib, "LIB_PATH", "/nonexistent/libfmha_decode.so")
    with pytest.raises(RuntimeError, match="not built"):
        fmha_amd.fmha_decode(q, k, v)


def _args(layout):
    g = torch.Generator(device="cuda").manual_seed(3)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda", dtype=torch.bfloat16)

    lens = torch.tensor([5, 16, 0, 9], dtype=torch.int32, device="cuda")
    cu = torch.tensor([0, 5, 21, 21, 30], dtype=torch.int32, device="cuda")
    q = normal(4, 8, 1, 64)
    if layout == "uniform":
        return fmha_amd.fmha_decode, (q, normal(4, 7, 4, 64), normal(4, 7, 4, 64)), {}
    if layout == "seqlen":
        return fmha_amd.fmha_decode, (q, normal(4 * 7, 4, 64), normal(4 * 7, 4, 64)), {"seqlen_kv": 7}
    if layout == "cu":
        return fmha_amd.fmha_decode, (q, normal(30, 4, 64), normal(30, 4, 64)), {"cu_seqlens_kv": cu}
    if layout in ("exact", "fast", "fp32_weights"):
        return fmha_amd.fmha_decode, (q, normal(30, 4, 64), normal(30, 4, 64)), {"cu_seqlens_kv": cu, layout: True}
    if layout == "splitkv":
        return fmha_amd.fmha_decode_splitkv, (q, normal(30, 4, 64), normal(30, 4, 64), cu, 40), {}
    if layout == "strided":
        return fmha_amd.fmha_decode_strided, (q, normal(4, 4, 16, 64).transpose(1, 2), normal(4, 4, 16, 64).transpose(1, 2),
                                              lens), {}
    if layout == "strided_long":
        return fmha_amd.fmha_decode_strided, (q, normal(4, 50, 4, 64), normal(4, 50, 4, 64)), {"softmax_scale": 0.25}
    table = torch.arange(8, dtype=torch.int32, device="cuda").view(4, 2)
    kv = (normal(8, 16, 4, 64), normal(8, 16, 4, 64))
    return fmha_amd.fmha_decode_paged, (q, *kv, table, lens), {} if layout == "paged" else {"max_seqlen_kv": 32}


LAYOUTS = ["uniform", "seqlen", "cu", "exact", "fast", "fp32_weights", "splitkv", "strided", "strided_long", "paged",
           "paged_long"]


@pytest.mark.gpu
@pytest.mark.parametrize("layout", LAYOUTS)
def test_same_as_python(monkeypatch, layout):
    """Bits, shape, a given output, another stream, a query that requires a
    gradient; the native form takes each of them."""
    fn, args, kw = _args(layout)
    taken = []
    real = decode._load_native()

    class Counts:
        def __getattr__(self, name):
            def call(*a):
                r = getattr(real, name)(*a)
                taken.append(r is not None)
                return r
            return call

    monkeypatch.setattr(decode, "_native", _Leaves())
    want = fn(*args, **kw)
    assert want.dtype == torch.float16 and not taken
    monkeypatch.setattr(decode, "_native", Counts())
    got = fn(*args, **kw)
    assert got.shape == want.shape and torch.equal(got.view(torch.int16), want.view(torch.int16))
    out = torch.empty_like(want)
    assert fn(*args, **kw, out=out) is out and torch.equal(out.view(torch.int16), want.view(torch.int16))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        other = fn(*args, **kw)
    side.synchronize()
    assert torch.equal(other.view(torch.int16), want.view(torch.int16))
    grad = fn(args[0].detach().requires_grad_(), *args[1:], **kw)
    assert not grad.requires_grad and torch.equal(grad.view(torch.int16), want.view(torch.int16))
    assert taken == [True] * 4


BAD = [
    ("uniform", lambda a: (a[0].float(), *a[1:]), {}),
    ("uniform", lambda a: (a[0].cpu(), *a[1:]), {}),
    ("uniform", lambda a: (a[0], a[1][:, :, :2], a[2]), {}),
    ("uniform", lambda a: a, {"out": torch.float32}),
    ("uniform", lambda a: a, {"fp32_weights": True}),
    ("uniform", lambda a: a, {"seqlen_kv": 9}),
    ("cu", lambda a: a, {"exact": True, "fast": True}),
    ("cu", lambda a: a, {"cu_seqlens_kv": "short"}),
    ("cu", lambda a: a, {"softmax_scale": float("nan")}),
    ("splitkv", lambda a: (*a[:4], -1), {}),
    ("splitkv", lambda a: a, {"workspace": "small"}),
    ("strided", lambda a: (a[0], a[1], a[2].contiguous(), a[3]), {}),
    ("strided", lambda a: (*a[:3], a[3].long()), {}),
    ("paged", lambda a: (*a[:3], a[3].t(), a[4]), {}),
    ("paged", lambda a: (*a[:4], None), {}),
    ("paged", lambda a: (a[0], a[1][:, :12].contiguous(), a[2][:, :12].contiguous(), *a[3:]), {}),
]


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(BAD)))
def test_same_errors(monkeypatch, i):
    """A refused call raises the same error through both forms."""
    layout, change, more = BAD[i]
    fn, args, kw = _args(layout)
    args = change(args)
    more = dict(more)
    if more.get("out") is torch.float32:
        more["out"] = torch.empty(args[0].shape, dtype=torch.float32, device="cuda")
    if isinstance(more.get("cu_seqlens_kv"), str):
        more["cu_seqlens_kv"] = torch.zeros(3, dtype=torch.int32, device="cuda")
    if isinstance(more.get("workspace"), str):
        more["workspace"] = torch.empty(16, dtype=torch.uint8, device="cuda")
    kw = {**kw, **more}
    seen = []
    for native in (_Leaves(), decode._load_native()):
        monkeypatch.setattr(decode, "_native", native)
        with pytest.raises(Exception) as e:
            fn(*args, **kw)
        seen.append((type(e.value), str(e.value)))
    assert seen[0] == seen[1]


@pytest.mark.gpu
def test_modes_and_default_scale(monkeypatch):
    """A dispatch mode sees the allocation, as through Python; the default
    scale is 1/sqrt(D)."""
    from torch.utils._python_dispatch import TorchDispatchMode
    fn, args, kw = _args("uniform")
    seen = []

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, a=(), k=None):
            seen.append(func)
            return func(*a, **(k or {}))

    with Mode():
        got = fn(*args, **kw)
    assert seen and torch.equal(got, fn(*args, **kw, softmax_scale=1.0 / math.sqrt(64)))
