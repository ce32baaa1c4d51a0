"""The native call front (csrc/iq_pyfast.cpp) against the general Python path over the forms it accepts and
the ones it passes on: the same kernels with the same arguments, so the same bits, the same errors and
the same state afterwards.  (Runs short enough that no wave order varies between calls.)"""
import ctypes

import pytest
import torch

from innerq_amd import _lib, ops
from innerq_amd.cache import InnerqDynamicLayer
from innerq_amd.presets import preset_config

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture
def general(monkeypatch):
    """Runs a function through the general path only."""
    def run(f):
        with monkeypatch.context() as m:
            m.setattr(ops, "_native", lambda t: None)
            return f()
    return run


def stores(dt, B=2, H=2, D=128, n=256, g=32):
    gen = torch.Generator(DEV).manual_seed(n)
    x = torch.randn(B, H, n + 40, D, device=DEV, generator=gen).to(dt)
    ks = ops.PackedStore("channel", B, H, D, g, 4, "asymmetric", DEV, dtype=dt)
    vs = ops.PackedStore("token", B, H, D, g, 3, "symmetric", DEV, dtype=dt)
    ks.append(x[:, :, :n])
    vs.append(x[:, :, :n])
    return x, ks, vs


def both(general, f):
    a = f()
    b = general(f)
    return torch.equal(a, b)


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("form", ["plain", "window", "norm", "strided q", "q column view", "out", "strided out", "offset",
                                  "dense only", "sink"])
def test_decode(general, dt, form):
    x, ks, vs = stores(dt)
    B, H, D = 2, 2, 128
    q = torch.randn(B, 8, D, device=DEV).to(dt)
    w = x[:, :, 256:]
    k = dict(k_sink=None, k_store=ks, k_recent=None, v_sink=None, v_store=vs, v_recent=None)
    more = {}
    if form == "window":
        k.update(k_recent=w, v_recent=w)
    if form == "norm":
        more["norm"] = torch.rand(B, H, 1, D, device=DEV).to(dt) + 0.5
    if form == "strided q":
        q = torch.randn(8, B, D, device=DEV).to(dt).transpose(0, 1)
    if form == "q column view":  # head_dim not contiguous: the general path copies
        q = torch.randn(B, 8, D, 2, device=DEV).to(dt)[..., 0]
    if form == "out":
        more["out"] = torch.empty(B, 8, D, device=DEV, dtype=dt)
    if form == "strided out":
        more["out"] = torch.empty(8, B, D, device=DEV, dtype=dt).transpose(0, 1)
    if form == "offset":
        more.update(k_t0=64, v_t0=64)
    if form == "dense only":
        k.update(k_store=None, v_store=None, k_recent=w, v_recent=w)
    if form == "sink":
        k.update(k_sink=w[:, :, :5], v_sink=w[:, :, :5])

    def call():
        r = ops.decode_attention(q, **k, scale=0.09, **more)
        return r.clone()

    assert both(general, call)
    if "out" in more:
        assert ops.decode_attention(q, **k, scale=0.09, **more) is more["out"]


def test_gemvs(general):
    x, ks, vs = stores(torch.float16)
    q = torch.randn(2, 8, 128, device=DEV).half()
    p = torch.softmax(torch.randn(2, 8, 300, device=DEV), -1).half()
    for kw in ({}, {"t0": 64}, {"t0": 64, "T": 100}, {"norm": torch.rand(2, 2, 128, device=DEV).half() + 0.5},
               {"out": torch.empty(2, 8, 256, device=DEV)}):
        assert both(general, lambda: ops.qk_gemv(q, ks, 0.1, **kw).clone())
    for kw in ({}, {"t0": 32}, {"t0": 64, "T": 96}, {"out32": torch.empty(2, 8, 128, device=DEV)},
               {"out": torch.zeros(2, 8, 128, device=DEV).half()}):
        assert both(general, lambda: ops.av_gemv(p, vs, **kw).clone())
    acc = torch.ones(2, 8, 128, device=DEV)
    one = ops.av_gemv(p, vs, out32=torch.zeros(2, 8, 128, device=DEV))
    assert torch.equal(ops.av_gemv(p, vs, out32=acc, accumulate=True), 1.0 + one)


@pytest.mark.parametrize("bad", ["q dims", "q 4-d", "heads", "T", "cpu q", "dtype", "range", "norm size", "out shape"])
def test_errors_are_the_general_paths(general, bad):
    x, ks, vs = stores(torch.float16)
    q = torch.randn(2, 8, 128, device=DEV).half()
    a, kw = [q, None, ks, None, None, vs, None, 0.1], {}
    if bad == "q dims": a[0] = q[0]
    if bad == "q 4-d": a[0] = q[:, :, None]
    if bad == "heads": a[0] = torch.randn(2, 7, 128, device=DEV).half()
    if bad == "T": a[3] = x[:, :, 256:]
    if bad == "cpu q": a[0] = q.cpu()
    if bad == "dtype": a[0] = q.float()
    if bad == "range": kw["k_t0"] = 300
    if bad == "norm size": kw["norm"] = torch.ones(5, device=DEV).half()
    if bad == "out shape": kw["out"] = torch.empty(2, 8, 64, device=DEV).half()
    with pytest.raises(Exception) as fast:
        ops.decode_attention(*a, **kw)
    with pytest.raises(Exception) as slow:
        general(lambda: ops.decode_attention(*a, **kw))
    assert type(fast.value) is type(slow.value) and str(fast.value) == str(slow.value)


@pytest.mark.parametrize("t0,T", [(0, -1), (0, -5), (64, -1), (0, 257), (64, 193), (-64, None), (320, None), (0, 0),
                                  (2 ** 62, 2 ** 62), (0, 10 ** 30), (0, 1.5)])
@pytest.mark.parametrize("role", ["qk", "av"])
def test_gemv_ranges_are_the_general_paths(general, role, t0, T):
    """A token range outside the store's, a negative count among them, is refused as the general path
    refuses it; an empty one gives what it gives."""
    x, ks, vs = stores(torch.float16)
    q = torch.randn(2, 8, 128, device=DEV).half()
    p = torch.rand(2, 8, 256, device=DEV).half()

    def call():
        try:
            return (ops.qk_gemv(q, ks, 0.1, t0=t0, T=T) if role == "qk" else ops.av_gemv(p, vs, t0=t0, T=T)).shape
        except Exception as e:
            return type(e), str(e)

    got = call()
    assert got == general(call)
    assert T == 0 or not isinstance(got, torch.Size)


@pytest.mark.parametrize("preset", ["innerq_base", "innerq_hybrid"])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_layer_steps(general, preset, dt):
    """A generation through both paths: outputs, windows and stores after window moves, V flushes and
    store growth."""
    def generate():
        gen = torch.Generator(DEV).manual_seed(3)
        layer = InnerqDynamicLayer(preset_config(preset), 0)
        layer.update(*(torch.randn(2, 2, 230, 128, device=DEV, generator=gen).to(dt) for _ in range(2)))
        outs = []
        for _ in range(150):
            kn, vn = (torch.randn(2, 2, 1, 128, device=DEV, generator=gen).to(dt) for _ in range(2))
            layer.append(kn, vn)
            q = torch.randn(2, 8, 1, 128, device=DEV, generator=gen).to(dt)
            outs.append(layer.attend(q, 0.09))
        return torch.stack(outs), *layer.get_deq_tensors()

    for a, b in zip(generate(), general(generate)):
        assert torch.equal(a, b)


def test_streams_and_capture(general):
    """A call on another stream uses that stream's workspace; a captured call replays."""
    x, ks, vs = stores(torch.float16)
    q = torch.randn(2, 8, 128, device=DEV).half()
    want = general(lambda: ops.decode_attention(q, None, ks, None, None, vs, None, 0.1))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = ops.decode_attention(q, None, ks, None, None, vs, None, 0.1)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(got, want)
    assert (0, side.cuda_stream) in ops._WS
    out = torch.empty_like(want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        ops.decode_attention(q, None, ks, None, None, vs, None, 0.1, out=out)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        ops.decode_attention(q, None, ks, None, None, vs, None, 0.1)


ENTRIES = ("iq_decode_workspace_bytes", "iq_decode_attention", "iq_qk_workspace_bytes", "iq_qk_gemv",
           "iq_av_workspace_bytes", "iq_av_gemv", "iq_window_append")
ENTRY = {"decode": ENTRIES[1], "qk": ENTRIES[3], "av": ENTRIES[5], "append": ENTRIES[6]}


def entered_as(entry, stand_in, call):
    """call() with the front's C entry point replaced by the Python function ``stand_in`` (its status)."""
    name = ENTRY[entry]
    fake = ctypes.CFUNCTYPE(ctypes.c_int, *[t if issubclass(t, ctypes._SimpleCData) else ctypes.c_void_p
                                            for t in _lib.SIGNATURES[name][1]])(stand_in)
    at = {n: ctypes.cast(getattr(_lib.lib(), n), ctypes.c_void_p).value for n in ENTRIES}
    at[name] = ctypes.cast(fake, ctypes.c_void_p).value
    try:
        ops._native(torch.empty(0, device=DEV)).bind(tuple(at[n] for n in ENTRIES), ops._WS,
                                                     torch._C._cuda_getCurrentRawStream)
        return call()
    finally:
        ops._fast = None  # bound to the library again by the next call


def four_calls():
    """The four entries' calls over one pair of stores and windows."""
    x, ks, vs = stores(torch.float16)
    q = torch.randn(2, 8, 128, device=DEV).half()
    p = torch.rand(2, 8, 256, device=DEV).half()
    kwin, vwin = (ops.RecentWindow(x[:, :, :40]) for _ in range(2))
    new = x[:, :, 40:41].contiguous()
    ks.reserve(512)
    vs.reserve(512)
    return ks, vs, kwin, vwin, {
        "decode": lambda: ops.decode_attention(q, None, ks, None, None, vs, None, 0.1),
        "qk": lambda: ops.qk_gemv(q, ks, 0.1), "av": lambda: ops.av_gemv(p, vs),
        "append": lambda: ops.window_append(kwin, new, 32, ks, None, vwin, new, 32, vs)}


@pytest.mark.parametrize("entry", ["decode", "qk", "av", "append"])
def test_tensors_are_held_while_other_threads_run(entry):
    """The front lets other threads run while it enqueues kernels.  What one of them may do meanwhile (a
    larger workspace for the stream, a store or a window that grows) frees none of the call's memory.  The
    entry point is stood in for by a function that drops every reference Python has; no kernel runs."""
    ks, vs, kwin, vwin, calls = four_calls()
    if entry != "append":
        calls[entry]()  # the stream's workspace
        kwin.buf = vwin.buf = None
    if entry in ("qk", "av"):  # the other role's store is not this call's
        other = vs if entry == "qk" else ks
        other.codes = other.meta = None
    freed = []

    def during(*_):
        before = torch.cuda.memory_allocated()
        if entry != "append":
            del ops._WS[(0, torch.cuda.current_stream().cuda_stream)]
        for t in (ks, vs):
            t.codes = t.meta = None
        kwin.buf = vwin.buf = None
        freed.append(before - torch.cuda.memory_allocated())
        return 0

    entered_as(entry, during, calls[entry])
    assert freed == [0]


@pytest.mark.parametrize("entry", ["decode", "qk", "av", "append"])
def test_a_failed_launch_is_raised_once(entry):
    """A launch that reports an error is not tried again (it may have run, and an append is no call to run
    twice); an argument that the entry point refuses is the general path's to refuse or to serve."""
    ks, vs, kwin, vwin, calls = four_calls()
    state = [t.clone() for t in (ks.codes, ks.meta, vs.codes, vs.meta, kwin.tensor, vwin.tensor)]
    with pytest.raises(_lib.IQError) as e:
        calls[entry]() if entry != "append" else None  # the stream's workspace
        entered_as(entry, lambda *_: -9, calls[entry])
    assert e.value.status == -9 and ENTRY[entry] in str(e.value)
    assert (ks.length, vs.length, kwin.start, kwin.n, vwin.start, vwin.n) == (256, 256, 0, 40, 0, 40)
    for a, b in zip(state, (ks.codes, ks.meta, vs.codes, vs.meta, kwin.tensor, vwin.tensor)):
        assert torch.equal(a, b)
    served = entered_as(entry, lambda *_: -5, calls[entry])
    if entry == "append":
        assert (ks.length, vs.length, kwin.start, kwin.n) == (288, 288, 32, 9)
    else:
        assert torch.equal(served, calls[entry]())
