"""Dense reads of packed stores at the sizes where the kernels' tiles end: single tokens and block
edges, ranges that start inside a block, head_dims whose rows do not divide a workgroup (K), odd
column counts (V), and outputs whose rows do or do not take vector stores.  The values are defined
bit for bit: fp32(c * s + z), times the factor in fp32, one rounding to the output type (oracle)."""
import numpy as np
import pytest
import torch
from torch.autograd import forward_ad

from innerq_amd import ops
from innerq_amd.cache import InnerqDynamicLayer
from innerq_amd.presets import preset_config
from oracle import quant_ref as Q

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TD = {"f16": torch.float16, "bf16": torch.bfloat16}
MODES = [("asymmetric", (1, 2, 3, 4)), ("symmetric", (2, 3, 4)), ("hybrid", (2, 3, 4))]
FN = {(m, ax): (getattr(Q, f"quantize_{ax}dim_{s}"), getattr(Q, f"dequantize_{ax}dim_{s}"))
      for m, s in (("asymmetric", "asym"), ("symmetric", "sym"), ("hybrid", "hybrid")) for ax in ("channel", "token")}


def view(B, H, T, D, dtype, layout):
    if layout == "plain":
        return torch.zeros(B, H, T, D, dtype=dtype, device=DEV)
    if layout == "inside":  # the slice that update() fills between sinks and window
        return torch.zeros(B, H, T + 5, D, dtype=dtype, device=DEV)[:, :, 2:T + 2]
    if layout == "heads last":
        return torch.zeros(B, T, H, D, dtype=dtype, device=DEV).transpose(1, 2)
    return torch.zeros(B, H, T, D + 1, dtype=dtype, device=DEV)[..., 1:]  # odd rows


@pytest.mark.parametrize("act", ["f16", "bf16"])
@pytest.mark.parametrize("mode,widths", MODES)
@pytest.mark.parametrize("axis,n,t0,D,G,layout,norm", [
    ("channel", 1, 0, 128, 32, "plain", False), ("channel", 65, 1, 64, 64, "inside", True),
    ("channel", 130, 63, 96, 32, "heads last", True), ("channel", 513, 0, 128, 128, "odd rows", False),
    ("channel", 33, 0, 384, 128, "inside", True), ("token", 32, 0, 128, 32, "plain", False),
    ("token", 320, 64, 64, 64, "inside", False), ("token", 256, 128, 130, 128, "heads last", False),
    ("token", 96, 32, 33, 32, "odd rows", False), ("token", 64, 0, 1, 64, "plain", False)])
def test_dequant(act, mode, widths, axis, n, t0, D, G, layout, norm):
    B, H = 2, 2
    rng = np.random.default_rng(n + D + G)
    x = torch.from_numpy(rng.standard_normal((B, H, n, D)).astype(np.float32)).to(TD[act])
    xh = x.float().numpy() if act == "bf16" else x.numpy()
    nf = torch.from_numpy(rng.uniform(0.2, 3.0, (B, H, 1, D)).astype(np.float32)).to(TD[act]) if norm else None
    quant, deq = FN[mode, axis]
    xq = xh
    if norm:
        xq = Q._div16(xh, nf.float().numpy() if act == "bf16" else nf.numpy(), act)
    for bits in widths:
        want = deq(*quant(xq, G, bits, act), G).astype(np.float32)
        if norm:
            want = want * nf.float().numpy()
        want = want[:, :, t0:]
        st = ops.PackedStore(axis, B, H, D, G, bits, mode, DEV, dtype=TD[act])
        st.append(x.to(DEV), norm=None if nf is None else nf.to(DEV))
        for dtype in (TD[act], torch.float32):
            out = view(B, H, n - t0, D, dtype, layout)
            st.dequant(t0, n - t0, out=out, norm=None if nf is None else nf.to(DEV))
            ref = torch.from_numpy(np.ascontiguousarray(want)).to(dtype)
            assert torch.equal(out.cpu(), ref)  # equal values: -0 == +0


@pytest.mark.parametrize("act", ["f16", "bf16"])
@pytest.mark.parametrize("axis,D,ns,n,nr,layout", [("channel", 128, 32, 70, 96, "plain"), ("token", 128, 0, 64, 7, "plain"),
                                                   ("token", 64, 3, 96, 0, "plain"), ("channel", 96, 1, 1, 1, "plain"),
                                                   ("channel", 64, 5, 129, 9, "heads last"),
                                                   ("token", 128, 33, 32, 40, "odd rows")])
def test_read_dense(act, axis, D, ns, n, nr, layout):
    """[sink | packed | recent] in one launch equals the parts, for sources whose rows do or do not take
    vector loads."""
    B, H = 2, 3
    dt = TD[act]

    def rows(m):
        t = view(B, H, m, D, dt, layout)
        return t.copy_(torch.randn(B, H, m, D, device=DEV).to(dt))

    sink, recent = rows(ns), rows(nr)
    st = ops.PackedStore(axis, B, H, D, 32, 3, "symmetric", DEV, dtype=dt)
    norm = torch.rand(B, H, 1, D, device=DEV).to(dt) + 0.5 if axis == "channel" else None
    st.append(torch.randn(B, H, n, D, device=DEV).to(dt), norm=norm)
    got = ops.read_dense(sink, st, recent, norm)
    assert torch.equal(got, torch.cat([sink, st.dequant(norm=norm), recent], dim=2))


@pytest.mark.parametrize("act", ["f16", "bf16"])
@pytest.mark.parametrize("bits,mode,G", [(1, "asymmetric", 32), (2, "hybrid", 64), (3, "symmetric", 32),
                                         (3, "hybrid", 128), (4, "asymmetric", 128)])
@pytest.mark.parametrize("D,n,layout", [(128, 24576, "plain"), (33, 87296, "odd rows"), (96, 32768, "heads last")])
def test_value_reads_past_the_few_thread_line(act, bits, mode, G, D, n, layout):
    """A read of values by more than 49,152 threads of 32 tokens (the line between the two kernels: 2 heads x
    n / 32 x ceil(D / 4)), and one at the line, equal the same tokens read in small pieces (which the
    tests above check against the oracle)."""
    st = ops.PackedStore("token", 1, 2, D, G, bits, mode, DEV, dtype=TD[act])
    st.append(torch.randn(1, 2, n + 256, D, device=DEV).to(TD[act]))
    for dtype in (TD[act], torch.float32):
        for T in (n, n + 256):
            out = view(1, 2, T, D, dtype, layout)
            st.dequant(0, T, out=out)
            for t0 in range(0, T, 8192):
                m = min(8192, T - t0)
                assert torch.equal(out[:, :, t0:t0 + m], st.dequant(t0, m, dtype=dtype))


@pytest.mark.parametrize("act", ["f16", "bf16"])
@pytest.mark.parametrize("axis", ["channel", "token"])
def test_large_reads_equal_small_ones(axis, act):
    """A read past 104 MB of output, where the stores stream (16-bit and fp32 outputs), equals the same
    tokens read in pieces below it."""
    B, H, T, D, step = 2, 8, 28672, 128, 7168
    assert 2 * B * H * T * D > 104 << 20 > 4 * B * H * step * D
    st = ops.PackedStore(axis, B, H, D, 32, 3, "symmetric", DEV, dtype=TD[act])
    norm = torch.rand(B, H, 1, D, device=DEV).to(TD[act]) + 0.5 if axis == "channel" else None
    st.append(torch.randn(B, H, T, D, device=DEV).to(TD[act]), norm=norm)
    for dtype in (TD[act], torch.float32):
        whole = st.dequant(dtype=dtype, norm=norm)
        for t0 in range(0, T, step):
            assert torch.equal(whole[:, :, t0:t0 + step], st.dequant(t0, step, dtype=dtype, norm=norm))
    sink, recent = (torch.randn(B, H, n, D, device=DEV).to(TD[act]) for n in (32, 95))
    got = ops.read_dense(sink, st, recent, norm)
    assert torch.equal(got[:, :, :32], sink) and torch.equal(got[:, :, 32 + T:], recent)
    for t0 in range(0, T, step):
        assert torch.equal(got[:, :, 32 + t0:32 + t0 + step], st.dequant(t0, step, norm=norm))


@pytest.mark.parametrize("preset", ["innerq_base", "innerq_hybrid"])
@pytest.mark.parametrize("act", ["f16", "bf16"])
def test_gradients_pass_through_dense_reads(preset, act):
    """A dense read of a layer whose prompt carries gradients: those of the rows that are the prompt's own
    (sinks and windows) are 1, backward and forward, and the quantized tokens' are 0; the values are the
    ones without gradients."""
    layer = InnerqDynamicLayer(preset_config(preset), 0)
    T = 300
    k, v = (torch.randn(2, 2, T, 128, device=DEV).to(TD[act]).requires_grad_() for _ in range(2))
    layer.update(k, v)
    read = layer.get_deq_tensors()
    (read[0].float().sum() + read[1].float().sum()).backward()
    with torch.no_grad():
        plain = layer.get_deq_tensors()
    for x, r, p, sink, q in zip((k, v), read, plain, (layer.keys_sink, layer.values_sink), (layer._kq, layer._vq)):
        assert torch.equal(r, p) and not p.requires_grad
        want = torch.ones_like(x)
        ns = sink.shape[2]
        want[:, :, ns:ns + q.length] = 0.0
        assert torch.equal(x.grad, want)
    with forward_ad.dual_level():
        layer = InnerqDynamicLayer(preset_config(preset), 0)
        layer.update(*(forward_ad.make_dual(x.detach(), torch.ones_like(x)) for x in (k, v)))
        for r, sink, q in zip(layer.get_deq_tensors(), (layer.keys_sink, layer.values_sink), (layer._kq, layer._vq)):
            t = forward_ad.unpack_dual(r).tangent
            ns = sink.shape[2]
            assert bool((t[:, :, :ns] == 1).all()) and bool((t[:, :, ns + q.length:] == 1).all())
