"""The K quantizers agree bit for bit: the prompt's (quant_k_kernel: a thread per eight values, packed
arithmetic, a reciprocal for the division) in one large call and in many small ones, and the window
append's (a lane per value, the reference's own arithmetic), on inputs with the groups where they could
part: signed zeros at the minimum, constant groups (scale 0, NaN codes), NaN and infinity, exact rounding
ties, fp16 subnormals.  Small calls are also checked against the oracle in test_gpu_kernels (random
data) and test_gpu_quantize_edges."""
import numpy as np
import pytest
import torch

from innerq_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
N_TOK = 4160  # the large call: 2080 workgroups of quant_k_kernel
CHUNK = 64    # the small ones: 32 workgroups, or a window append's flush


def adversarial(H, T, D, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((1, H, T, D)).astype(np.float32)
    x[0, 0, 0, :] = np.where(np.arange(D) % 2 == 0, 0.0, -0.0)       # zeros of both signs only
    x[0, 0, 1, :] = 1.5                                               # constant groups
    x[0, 0, 2, 5] = np.nan                                            # NaN in group 0
    x[0, 0, 2, 40] = np.inf                                           # infinity in group 1
    x[0, 0, 3, :32] = np.arange(32) % 16 + 0.5                        # ties at 4-bit scale 1
    x[0, 0, 3, 32:64] = (np.arange(32) % 4) - 2                       # the 2-bit tie pattern
    x[0, 0, 4, :] = np.abs(x[0, 0, 4, :])
    x[0, 0, 4, ::7] = -0.0                                            # minimum -0 among positives
    x[0, 0, 5, :] = -0.0                                              # negative zeros only
    x[0, 0, 6, :] = rng.standard_normal(D) * 1e-6                     # fp16 subnormals
    x[0, 1, 7, :] = np.where(np.arange(D) % 3 == 0, -0.0, 0.0) + (np.arange(D) % 5 == 0) * 2.0
    return x.astype(np.float16)


def store_bytes(st):
    n = st.length // 64
    bh = st.B * st.H
    return (st.codes.view(bh, st.t_cap // 64, -1)[:, :n].cpu().numpy(),
            st.meta.view(bh, st.t_cap // 64, -1)[:, :n].cpu().numpy())


@pytest.mark.parametrize("mode,bits", [("asymmetric", 1), ("asymmetric", 2), ("asymmetric", 3), ("asymmetric", 4),
                                       ("symmetric", 2), ("symmetric", 3), ("symmetric", 4)])
@pytest.mark.parametrize("G", [32, 64])
@pytest.mark.parametrize("norm", [False, True])
def test_lane_and_thread_quantizers_agree(mode, bits, G, norm):
    H, D = 8, 128
    x = torch.from_numpy(adversarial(H, N_TOK, D, seed=bits * G)).to(DEV)
    nf = ops.key_norm_factor(x[:, :, 8:200]) if norm else None
    big = ops.PackedStore("channel", 1, H, D, G, bits, mode, DEV)
    big.append(x, norm=nf)
    small = ops.PackedStore("channel", 1, H, D, G, bits, mode, DEV)
    for t in range(0, N_TOK, CHUNK):
        small.append(x[:, :, t:t + CHUNK], norm=nf)
    lanes = ops.PackedStore("channel", 1, H, D, G, bits, mode, DEV)
    win = ops.RecentWindow(x[:, :, :0])
    for t in range(0, N_TOK, CHUNK):
        ops.window_append(win, x[:, :, t:t + CHUNK], CHUNK, lanes, nf, None, None, 0, None)
    bc, bm = store_bytes(big)
    for other in (small, lanes):
        oc, om = store_bytes(other)
        np.testing.assert_array_equal(oc, bc)
        np.testing.assert_array_equal(om, bm)


@pytest.mark.parametrize("mode", ["asymmetric", "symmetric"])
@pytest.mark.parametrize("bits,G", [(2, 32), (3, 64), (4, 32)])
def test_lane_and_thread_reference_outputs_agree(mode, bits, G):
    # quant.py-format outputs (codes, scale, zero | signs) of a small call equal
    # the same rows of a large call
    x = torch.from_numpy(adversarial(8, N_TOK, 128, seed=7 * bits + G)).to(DEV)
    cb, sb, zb = ops.quantize_dense(x, G, bits, mode, "channel")
    cs, ss, zs = ops.quantize_dense(x[:, :, :CHUNK].contiguous(), G, bits, mode, "channel")
    assert torch.equal(cs, cb[:, :, :CHUNK])
    assert torch.equal(ss.view(torch.int16), sb[:, :, :CHUNK].contiguous().view(torch.int16))
    assert torch.equal(zs.view(torch.int16), zb[:, :, :CHUNK].contiguous().view(torch.int16))
