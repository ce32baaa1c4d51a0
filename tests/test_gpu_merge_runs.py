"""Decode steps whose window is merged with 1 to 20 fused runs per KV head: the merging dense kernel takes
up to 12 (4 for eight query heads per KV head, bf16 layers, windows past 192 tokens (one head: 128) and
windows with packed rows), the slices and the combine the rest; counts around its rounds of four.  Against the float64 oracle within the decode's 1e-3 of max|ref|."""
import pytest
import torch

from innerq_amd import ops
from tests.test_gpu_kernels import TOL, _decode_case

pytestmark = pytest.mark.gpu


# splits of 256 tokens, one per run while there are fewer than workgroups
@pytest.mark.parametrize("runs", [1, 4, 5, 8, 9, 12, 13, 16, 17, 20])
@pytest.mark.parametrize("nrep,D", [(4, 128), (1, 64), (8, 128)])
def test_runs_per_head(runs, nrep, D):
    seg = (0, 256 * runs, 70)
    assert _decode_case(1, 2, nrep, D, seg, seg, (4, 32, "asymmetric"), (4, 32, "asymmetric"), seed=runs) < TOL


@pytest.mark.parametrize("runs", [4, 5, 12, 13])
@pytest.mark.parametrize("nrep,win", [(2, 1), (2, 192), (2, 193), (2, 256), (2, 257), (1, 128), (1, 129)])
def test_window_lengths(runs, nrep, win):
    """Windows of one chunk per section, of two, and past what is merged."""
    seg = (0, 256 * runs, win)
    assert _decode_case(1, 2, nrep, 128, seg, seg, (4, 32, "asymmetric"), (4, 32, "asymmetric"), seed=win) < TOL


@pytest.mark.parametrize("runs", [4, 5, 12])
def test_windows_with_packed_rows(runs):
    """K packed 32 tokens further than V: those rows are read packed in the window."""
    k, v = (0, 256 * runs + 32, 70), (0, 256 * runs, 102)
    assert _decode_case(1, 2, 4, 128, k, v, (4, 32, "asymmetric"), (4, 32, "asymmetric"), seed=runs) < TOL


@pytest.mark.parametrize("runs", [4, 5, 9])
def test_runs_per_head_bf16(runs):
    """bf16: the window's slices past four runs give what the merge gives (the same stores read
    as one batch of two and as single sequences), within the fp32 sums' order."""
    B, H, D, n = 2, 2, 128, 256 * runs
    x = torch.randn(B, H, n + 40, D, device="cuda:0", generator=torch.Generator("cuda:0").manual_seed(runs)).bfloat16()
    ks = ops.PackedStore("channel", B, H, D, 32, 4, "asymmetric", "cuda:0", dtype=x.dtype)
    vs = ops.PackedStore("token", B, H, D, 32, 4, "asymmetric", "cuda:0", dtype=x.dtype)
    ks.append(x[:, :, :n])
    vs.append(x[:, :, :n])
    q = torch.randn(B, 8, D, device="cuda:0").bfloat16()
    w = x[:, :, n:]
    both = ops.decode_attention(q, None, ks, w, None, vs, w, D ** -0.5)
    each = torch.cat([ops.decode_attention(q[b:b + 1], None, ks.batch_view(b, b + 1), w[b:b + 1], None,
                                           vs.batch_view(b, b + 1), w[b:b + 1], D ** -0.5) for b in range(B)])
    # one bf16 ulp where the fp32 results straddle a rounding boundary
    assert torch.allclose(both.float(), each.float(), rtol=2 ** -7, atol=1e-6)
