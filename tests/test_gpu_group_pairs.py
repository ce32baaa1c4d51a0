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
