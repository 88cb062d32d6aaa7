"""Every operator through the CPython binding and through the Python path: the same
outputs (bits, types, strides, identities), the same errors for the same calls."""
import pytest
import torch

from tests.gpu_util import note

pytestmark = pytest.mark.gpu

BF16, F16, F32, FP8, I8 = (torch.bfloat16, torch.float16, torch.float32, torch.float8_e4m3fn,
                           torch.int8)


def both(monkeypatch, fn):
    """fn() through the binding and, with the binding's operators out, in Python."""
    from fagq_mi355x import _lib
    assert _lib.fast_launch() is not None and _lib._fast_mod is not None

    def outcome():
        try:
            return fn()
        except Exception as e:                            # noqa: BLE001 (compared below)
            return type(e), str(e)
    a = outcome()
    with monkeypatch.context() as m:
        m.setattr(_lib, "_fast_mod", None)
        b = outcome()
    torch.cuda.synchronize()
    return a, b


def same(a, b):
    if isinstance(a, torch.Tensor):
        a, b = (a,), (b,)
    assert type(a) is type(b) and len(a) == len(b), (a, b)
    for x, y in zip(a, b):
        if not isinstance(x, torch.Tensor):
            assert x == y, (a, b)
            continue
        assert (x.dtype, x.shape, x.stride(), x.device, x.requires_grad) == \
               (y.dtype, y.shape, y.stride(), y.device, y.requires_grad)
        view = {1: torch.uint8, 2: torch.int16, 4: torch.int32}[x.element_size()]
        assert torch.equal(x.contiguous().view(view), y.contiguous().view(view))


QUANT = [dict(M=4, D=8192, out_dtype=I8), dict(M=1, D=128, scale_col_major=True),
         dict(M=300, D=128, scale_col_major=True), dict(M=33, D=1024, group_size=64, scale_ue8m0=True),
         dict(M=5, D=512, out_dtype=I8, rounding=None), dict(M=5, D=512, out_dtype=I8, rounding="trunc"),
         dict(M=7, D=768, rounding="trunc"), dict(M=9, D=512, act=F16, res=F16, scale_col_major=True),
         dict(M=9, D=512, res=F32), dict(M=9, D=512, act=F32, res=F32), dict(M=0, D=256),
         dict(M=0, D=256, scale_col_major=True), dict(M=0, D=0), dict(M=0, D=0, scale_col_major=True),
         dict(M=3, D=0), dict(M=0, D=192, group_size=96), dict(M=0, D=256, eps=-1.0),
         dict(M=0, D=256, act=F32, res=BF16),
         dict(M=6, D=512, inplace_residual=True),
         # what the Python layer refuses or the library does
         dict(M=4, D=512, act=F32, res=BF16), dict(M=4, D=512, group_size=96), dict(M=4, D=512, group_size=32),
         dict(M=4, D=512, out_dtype=I8, rounding="floor"), dict(M=4, D=512, eps=-1.0),
         dict(M=4, D=512, eps=1)]


@pytest.mark.parametrize("c", QUANT, ids=str)
@pytest.mark.parametrize("parts", [0, 1, 3])
def test_quantizer(pkg, gpu, monkeypatch, c, parts):
    c = dict(c)
    M, D = c.pop("M"), c.pop("D")
    act, res = c.pop("act", BF16), c.pop("res", BF16)
    note(f"binding quant M={M} D={D} {act} {res} {c} parts={parts}")
    g = torch.Generator().manual_seed(M + D)
    x = [torch.randn(M, D, generator=g).to(act).to(gpu) for _ in range(max(parts, 1))]
    r, w = torch.randn(M, D, generator=g).to(res).to(gpu), torch.randn(D, generator=g).to(act).to(gpu)

    def call():
        rr = r.clone()
        if parts:
            out = pkg.fused_reduce_add_rmsnorm_group_quant(x, rr, w, **c)
        else:
            out = pkg.fused_add_rmsnorm_group_quant_fn(x[0], rr, w, **c)
        assert (out[0] is rr) == c.get("inplace_residual", False)
        return out
    same(*both(monkeypatch, call))


def test_quantizer_rejects_alike(pkg, gpu, monkeypatch):
    note("binding quant, wrong tensors")
    x = torch.zeros(4, 256, dtype=BF16, device=gpu)
    w = torch.zeros(256, dtype=BF16, device=gpu)
    fn = pkg.fused_add_rmsnorm_group_quant_fn
    for args in ((x, x[:3], w), (x, x, w[:128]), (x[0], x, w), (x, x.cpu(), w), (x.t(), x.t(), w[:4]),
                 (torch.zeros(4, 512, dtype=BF16, device=gpu)[:, ::2], x, w)):
        same(*both(monkeypatch, lambda: fn(*args)))
    same(*both(monkeypatch, lambda: fn(x, x, w, out_dtype=torch.uint8)))
    p = torch.nn.Parameter(x, requires_grad=True)
    same(*both(monkeypatch, lambda: fn(p, p, w)))


def test_gemm(pkg, gpu, monkeypatch):
    note("binding gemm")
    g = torch.Generator().manual_seed(1)
    a = torch.randn(40, 512, generator=g).to(FP8).to(gpu)
    b = torch.randn(144, 512, generator=g).to(FP8).to(gpu)
    s = torch.rand(4, 40, generator=g).to(gpu)
    bs = torch.rand(2, 4, generator=g).to(gpu)
    u = torch.randint(120, 130, (40, 4), generator=g, dtype=torch.uint8).to(gpu)
    out = torch.empty(40, 144, dtype=BF16, device=gpu)
    fn = pkg.fp8_block_scaled_gemm
    assert fn(a, s.t(), b, bs, out) is out
    for args in ((a, s.t(), b, bs), (a, s.t().contiguous(), b, bs), (a, u, b, bs), (a, s.t(), b, bs, out),
                 (a[:0], s.t()[:0], b, bs), (a, s, b, bs), (a, s.t(), b, bs.half()), (a, s.t(), b[:, :256], bs),
                 (a, s.t(), b[:100], bs), (a, s.t(), b, bs, out.float()), (a, s.t(), b, bs, out[:, :128]),
                 (a.view(torch.uint8), s.t(), b, bs), (a, s.t(), b.cpu(), bs),
                 (a, s.t(), b, bs, a.view(torch.uint8).view(-1)[:0].view(BF16))):
        same(*both(monkeypatch, lambda: fn(*args)))


@pytest.mark.parametrize("idx", [torch.int32, torch.int64])
def test_dsa(pkg, gpu, monkeypatch, idx):
    note("binding dsa")
    g = torch.Generator().manual_seed(2)
    s = torch.randn(2, 3, 5, 200, generator=g).to(gpu)
    pt = torch.randint(0, 99, (2, 200), generator=g, dtype=torch.int32).to(gpu)
    pos = torch.randint(0, 3200, (2, 5), generator=g).to(idx).to(gpu)
    kv = torch.tensor([3200, 900], dtype=idx, device=gpu)
    ob = torch.empty(2, 3, 5, 16, dtype=torch.int32, device=gpu)
    op = torch.empty_like(ob)

    def call(*a):
        ob.fill_(-7), op.fill_(-7)
        r = pkg.dsa_topk_page_table_transform(*a)
        assert r[0] is ob and r[1] is op
        return r[0].clone(), r[1].clone()
    import numpy as np
    for a in ((s, pt, pos, kv, ob, op, 16, 16), (s.bfloat16(), pt, pos, kv, ob, op, np.int64(16), 16),
              (s, pt, pos, kv, ob, op, 0, 16), (s, pt, pos, kv, ob, op, 16, 8), (s[0], pt, pos, kv, ob, op, 16, 16),
              (s, pt, pos, kv.to(torch.int16), ob, op, 16, 16), (s, pt, pos, kv, ob, ob, 16, 16),
              (s.transpose(1, 2), pt, pos, kv, ob, op, 16, 16), (s.half(), pt, pos, kv, ob, op, 16, 16)):
        same(*both(monkeypatch, lambda: call(*a)))


def test_mla(pkg, gpu, monkeypatch):
    note("binding mla")
    from fagq_mi355x.workloads import MlaWorkload, make_mla_inputs
    q, c, out, do, lse = (t.to(gpu) for t in make_mla_inputs(MlaWorkload("t", 1, 3, 50, 128)))
    dq, dc = torch.empty_like(q), torch.empty(1, 50, 128, device=gpu)

    def call(*a):
        dq.zero_(), dc.zero_()
        r = pkg.mla_bwd_nope_dkdv(*a)
        assert r[0] is dq and r[1] is dc
        return r[0].clone(), r[1].clone()
    for a in ((q, c, out, do, lse, dq, dc, 0.1), (q, c, out, do, lse, dq, dc, 1),
              (q, c, out, do, lse, dq, dc, float("nan")), (q, c, out, do, lse.double(), dq, dc, 0.1),
              (q, c, out, do, lse, dq, dc.half(), 0.1), (q, c, out, do, lse, q, dc, 0.1),
              (q, c[:, :49], out, do, lse, dq, dc, 0.1), (q[..., :96].contiguous(), c, out, do, lse, dq, dc, 0.1)):
        same(*both(monkeypatch, lambda: call(*a)))


def test_other_streams_and_threads(pkg, gpu):
    """Allocations and launches follow the current stream, from several threads at once."""
    import threading
    note("binding on side streams")
    g = torch.Generator().manual_seed(4)
    x = torch.randn(64, 2048, generator=g).to(BF16).to(gpu)
    w = torch.ones(2048, dtype=BF16, device=gpu)
    want = pkg.fused_add_rmsnorm_group_quant_fn(x, x, w)
    torch.cuda.synchronize()
    bad = []

    def work():
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(50):
                got = pkg.fused_add_rmsnorm_group_quant_fn(x, x, w)
            s.synchronize()
            if not all(torch.equal(p.view(torch.uint8), q.view(torch.uint8)) for p, q in zip(got, want)):
                bad.append(1)
    ts = [threading.Thread(target=work) for _ in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad


HOLD_C = """
#include <unistd.h>
long long hold(void) { usleep(150000); return 0; }
"""


def test_launches_leave_the_gil_to_other_threads(pkg, gpu, tmp_path):
    """The library's entry points replaced by one that takes 150 ms on the host: a
    Python thread beside the call runs on (it would not get a turn under the GIL)."""
    import ctypes
    import shutil
    import subprocess
    import threading
    import time
    from fagq_mi355x import _lib
    from fagq_mi355x.workloads import MlaWorkload, make_mla_inputs
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None:
        pytest.skip("no C compiler")
    note("binding without the GIL")
    (tmp_path / "hold.c").write_text(HOLD_C)
    subprocess.run([cc, "-shared", "-fPIC", "-o", str(tmp_path / "hold.so"), str(tmp_path / "hold.c")],
                   check=True)
    addr = lambda f: ctypes.cast(f, ctypes.c_void_p).value
    hold = addr(ctypes.CDLL(str(tmp_path / "hold.so")).hold)
    assert _lib.fast_launch() is not None
    mod, lib = _lib._fast_mod, _lib.load()
    z = lambda *s, dt=BF16: torch.zeros(*s, dtype=dt, device=gpu)
    x, w = z(4, 256), z(256)
    i32 = lambda *s: z(*s, dt=torch.int32)
    q, c, out, do, lse = (t.to(gpu) for t in make_mla_inputs(MlaWorkload("t", 1, 2, 20, 64)))
    dq, dc = torch.empty_like(q), torch.empty_like(c)
    calls = {
        "quant": lambda: pkg.fused_add_rmsnorm_group_quant_fn(x, x, w),
        "typed": lambda: pkg.fused_add_rmsnorm_group_quant_fn(x.half(), x.half(), w.half()),
        "parts": lambda: pkg.fused_reduce_add_rmsnorm_group_quant([x, x], x, w),
        "gemm": lambda: pkg.fp8_block_scaled_gemm(z(4, 128, dt=FP8), z(4, 1, dt=F32),
                                                  z(16, 128, dt=FP8), z(1, 1, dt=F32)),
        "dsa": lambda: pkg.dsa_topk_page_table_transform(z(1, 1, 2, 64, dt=F32), i32(1, 64), i32(1, 2),
                                                         i32(1), i32(1, 1, 2, 8), i32(1, 1, 2, 8), 16, 8),
        "mla": lambda: pkg.mla_bwd_nope_dkdv(q, c, out, do, lse, dq, dc, 0.1),
    }
    for f in calls.values():                              # first calls, on the library itself
        f()
    torch.cuda.synchronize()
    ticks, stop = [0], threading.Event()

    def tick():
        while not stop.is_set():
            ticks[0] += 1
            time.sleep(0.001)
    t = threading.Thread(target=tick)
    t.start()
    got = {}
    try:
        mod.bind(hold, hold)
        mod.bind_all(hold, hold, hold, addr(lib.fagq_mla_bwd_workspace_bytes), hold)
        for name, f in calls.items():
            t0, n0 = time.perf_counter(), ticks[0]
            f()
            got[name] = (ticks[0] - n0, time.perf_counter() - t0)
    finally:
        mod.bind(addr(lib.fagq_launch), addr(lib.fagq_launch_typed))
        mod.bind_all(*[addr(f) for f in (lib.fagq_launch_parts, lib.fagq_gemm_launch,
                                         lib.fagq_dsa_topk_launch, lib.fagq_mla_bwd_workspace_bytes,
                                         lib.fagq_mla_bwd_launch)])
        stop.set()
        t.join()
    for name, (n, s) in got.items():
        # 150 sleeps of 1 ms fit; a thread kept out has its one turn at either end.
        assert s >= 0.15 and n >= 20, (name, got)
