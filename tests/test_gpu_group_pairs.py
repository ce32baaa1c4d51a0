"""Decode attention over K and V of different group sizes: the fused kernel takes the smaller group and
reads the larger store's groups in pieces that share their scale and zero point.  Every pair of
sizes, both ways round, at the piece boundaries (a range that ends inside a 64-token block, one V
group, several runs per head), with windows, against the float64 oracle within the decode's
1e-3 of max|ref| (tests/test_gpu_kernels.py)."""
import pytest
import torch

from innerq_amd import _lib, ops
from tests.test_gpu_kernels import TOL, _decode_case

pytestmark = pytest.mark.gpu
PAIRS = [(32, 64), (32, 128), (64, 32), (64, 128), (128, 32), (128, 64)]


@pytest.mark.parametrize("kg,vg", PAIRS)
@pytest.mark.parametrize("kb,vb,kmode,vmode,nrep,norm", [(4, 2, "asymmetric", "asymmetric", 4, False),
                                                         (3, 4, "symmetric", "asymmetric", 8, True),
                                                         (2, 3, "asymmetric", "symmetric", 1, False),
                                                         (4, 3, "symmetric", "hybrid", 2, True)])
def test_group_pairs(kg, vg, kb, vb, kmode, vmode, nrep, norm):
    vq = 128 * 5 + (vg if vg < 128 else 0)  # ends inside a 64-token block (groups of 32) or not
    kseg = (16, vq + 10, 7)  # both stores start at token 16: a fused range needs a common K block and V group start
    vseg = (16, vq, 17)
    assert _decode_case(2, 2, nrep, 128, kseg, vseg, (kb, kg, kmode), (vb, vg, vmode), seed=kg + vg, norm=norm) < TOL


@pytest.mark.parametrize("kg,vg,D,n", [(32, 128, 64, 128), (64, 32, 64, 32), (32, 64, 128, 64 * 300),
                                       (128, 32, 128, 64 * 257)])
def test_group_pairs_short_and_many_runs(kg, vg, D, n):
    seg = (0, n, 5)
    assert _decode_case(1, 1, 4, D, seg, seg, (4, kg, "asymmetric"), (4, vg, "asymmetric"), seed=n) < TOL


def test_refusals_of_different_groups_stand():
    """bf16 layers and hybrid keys decode with one group size only, as before."""
    dev = "cuda:0"
    for dt, kmode in ((torch.bfloat16, "asymmetric"), (torch.float16, "hybrid")):
        x = torch.randn(1, 1, 256, 128, device=dev).to(dt)
        ks = ops.PackedStore("channel", 1, 1, 128, 32, 4, kmode, dev, dtype=dt)
        vs = ops.PackedStore("token", 1, 1, 128, 64, 4, "asymmetric", dev, dtype=dt)
        ks.append(x)
        vs.append(x)
        with pytest.raises(_lib.IQError):
            ops.decode_attention(torch.randn(1, 4, 128, device=dev).to(dt), None, ks, None, None, vs, None, 0.1)


@pytest.mark.parametrize("kg,vg,B,H,nrep,T,win", [(32, 64, 8, 8, 4, 8192, 128), (64, 32, 3, 5, 8, 9000, 0),
                                                  (128, 32, 2, 8, 1, 700, 60)])
def test_calls_repeat_bit_for_bit(kg, vg, B, H, nrep, T, win):
    """Runs of many blocks, of an odd number of splits and of less than one: every call sums in one order."""
    x = torch.randn(B, H, T, 128, device="cuda:0").half()
    n = (T - win) // vg * vg
    ks = ops.PackedStore("channel", B, H, 128, kg, 4, "asymmetric", "cuda:0")
    vs = ops.PackedStore("token", B, H, 128, vg, 2, "asymmetric", "cuda:0")
    ks.append(x[:, :, :n])
    vs.append(x[:, :, :n])
    q = torch.randn(B, H * nrep, 128, device="cuda:0").half()
    tail = x[:, :, n:] if n < T else None
    a = ops.decode_attention(q, None, ks, tail, None, vs, tail, 0.09)
    for _ in range(12):
        assert torch.equal(ops.decode_attention(q, None, ks, tail, None, vs, tail, 0.09), a)


def test_a_splits_largest_probability_is_exact():
    """The probabilities that meet V are fp16 against their 256-token split's own maximum, so two tokens that
    hold a head's whole weight in different splits count in fp32.  Token 5 has value 1 and token 519, of a
    somewhat higher logit, about minus the weights' quotient: the output is their small difference, which a
    probability rounded to fp16 (2^-12 of ~0.2) would move by up to ~5e-5.  Bound: logits below 34 rounded to
    2^-24 in about 4 steps each move the quotient by 34 * 8 * 6e-8 = 1.6e-5 of ~0.25, and the fp16 output
    (below 2^-9) adds 2^-21."""
    B, H, T, D = 8, 8, 4096, 128  # four splits per workgroup
    gen = torch.Generator().manual_seed(1)
    delta = 0.5 + 4.5 * torch.rand(B, H, generator=gen)
    q = torch.zeros(B, 4 * H, D)
    q[:, :, 0] = 8.0
    k = torch.zeros(B, H, T, D)
    k[:, :, 5, 0] = 28.0
    k[:, :, 519, 0] = 28.0 + delta
    ks = ops.PackedStore("channel", B, H, D, 32, 4, "asymmetric", "cuda:0")
    ks.append(k.half().to("cuda:0"))
    logit = (ks.dequant(dtype=torch.float32).cpu().double()[..., 0] * 8.0 * 0.125)[:, :, [5, 519]]
    w = torch.exp(logit[..., 1] - logit[..., 0])
    v = torch.zeros(B, H, T, D)
    v[:, :, 5] = 1.0
    v[:, :, 519] = -(1.0 / w).float()[..., None]
    vs = ops.PackedStore("token", B, H, D, 64, 2, "asymmetric", "cuda:0")
    vs.append(v.half().to("cuda:0"))
    vd = vs.dequant(dtype=torch.float32).cpu().double()[..., 0]
    want = (vd[..., 5] + w * vd[..., 519]) / (1.0 + w)
    assert float(want.abs().max()) < 2.0 ** -9
    got = ops.decode_attention(q.half().to("cuda:0"), None, ks, None, None, vs, None, 0.125).cpu().double()
    err = (got.view(B, H, 4, D) - want[..., None, None]).abs().max()
    assert float(err) < 0.25 * 1.6e-5 + 2.0 ** -21
