"""The CPython binding's operators: what they leave to the Python layer (host code
only: CPU tensors are never launched on)."""
import pytest
import torch

BF16, FP8 = torch.bfloat16, torch.float8_e4m3fn


@pytest.fixture(scope="module")
def mod(pkg):
    from fagq_mi355x import _lib
    if _lib.fast_launch() is None:
        pytest.skip("binding not built")
    assert _lib._fast_mod.quant is not None
    return _lib


def test_cpu_tensors_and_odd_arguments_are_left_to_python(mod):
    b, err = mod._fast_mod, mod.FAST_ARG_ERROR
    x, w = torch.zeros(4, 128, dtype=BF16), torch.zeros(128, dtype=BF16)
    q = [x, x, w, 1e-6, 128, 1, 0, 0, 0, 0, 0]
    assert b.quant(*q) == err
    assert b.quant([x, x], *q[1:]) == err and b.quant([], *q[1:]) == err
    assert b.quant([x] * 9, *q[1:]) == err and b.quant([x, None], *q[1:]) == err
    for i, v in ((0, None), (3, 1), (4, 128.0), (4, True), (4, 1 << 70), (5, 2), (8, -2), (10, None)):
        assert b.quant(*q[:i], v, *q[i + 1:]) == err, (i, v)
    a = torch.zeros(4, 128, dtype=FP8)
    assert b.gemm(a, torch.zeros(4, 1), a, torch.zeros(1, 1), None, 0) == err
    i32 = torch.zeros(1, 4, dtype=torch.int32)
    assert b.dsa(torch.zeros(1, 1, 4, 4), i32, i32, i32[0, :1], i32, i32, 16, 4, 0) == err
    assert b.mla(x, x, x, x, x, x, x, 1.0, 0) == err and b.mla(x, x, x, x, x, x, x, "1", 0) == err
    for fn, n in ((b.quant, 11), (b.gemm, 6), (b.dsa, 9), (b.mla, 9), (b.bind_all, 5)):
        with pytest.raises(TypeError):
            fn(*[0] * (n - 1))
    with pytest.raises(ValueError):
        b.bind_all(0, 0, 0, 0, 0)


def test_fast_module_needs_a_plain_gpu_tensor(mod):
    for t in (torch.zeros(2), None, torch.nn.Parameter(torch.zeros(2)), torch.zeros(2, device="meta")):
        assert mod.fast_module(t) == (None, None)


def test_an_older_binding_leaves_every_call_to_ctypes(pkg, monkeypatch):
    """A _fagq_py built before an entry was added has bind() but not bind_all()."""
    import sys
    import types
    from fagq_mi355x import _lib
    old = types.ModuleType("fagq_mi355x._fagq_py")
    old.bind, old.launch = (lambda *a: None), (lambda *a: 0)
    monkeypatch.setitem(sys.modules, "fagq_mi355x._fagq_py", old)
    monkeypatch.setattr(pkg, "_fagq_py", old, raising=False)
    for name, v in (("_fast", None), ("_fast_mod", None), ("_fast_tried", False)):
        monkeypatch.setattr(_lib, name, v)
    assert _lib.fast_launch() is None
    assert _lib._fast is None and _lib._fast_mod is None and _lib._fast_tried
