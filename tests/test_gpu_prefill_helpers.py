"""The prefill helpers of a layer return the tokens to quantize as a contiguous copy (cache.py:157-186), and a
subclass that overrides one of the prefill's steps is handed that copy; a layer without overrides reads
the prompt in place, with the same state."""
import pytest
import torch

from innerq_amd.cache import InnerqDynamicLayer
from innerq_amd.presets import preset_config

pytestmark = pytest.mark.gpu


def prompt(dt, T=230):
    """As a projection leaves it: [B, T, H, D] seen as [B, H, T, D]."""
    return [torch.randn(2, T, 3, 128, device="cuda:0").to(dt).transpose(1, 2) for _ in range(2)]


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_helpers_return_contiguous_copies(dt):
    k, v = prompt(dt)
    layer = InnerqDynamicLayer(preset_config("innerq_base"), 0)
    layer.dtype, layer.device = k.dtype, k.device
    ks, vs = layer.initialize_sinks(k, v)
    for x, r, win in zip((ks, vs), layer.initialize_recents(ks, vs), (layer._kwin, layer._vwin)):
        n = x.shape[2] - win.n
        assert r.is_contiguous() and torch.equal(r, x[:, :, :n]) and torch.equal(win.tensor, x[:, :, n:])
        r.zero_()  # the caller's own: the prompt stays
        assert bool((x[:, :, :n] != 0).any())


@pytest.mark.parametrize("step", ["initialize_keys_q", "initialize_keys_recent"])
def test_subclass_steps_own_their_tokens(step):
    class Doubled(InnerqDynamicLayer):
        pass

    def q(self, x):
        return InnerqDynamicLayer.initialize_keys_q(self, x.view(-1).mul_(2.0).view(x.shape))

    def recent(self, x):
        return InnerqDynamicLayer.initialize_keys_recent(self, x).mul_(2.0)

    setattr(Doubled, step, q if step == "initialize_keys_q" else recent)
    k, v = prompt(torch.float16)
    kept = k.clone()
    a, b = Doubled(preset_config("innerq_base"), 0), InnerqDynamicLayer(preset_config("innerq_base"), 0)
    a.update(k, v)
    assert torch.equal(k, kept)
    n, ns = a._kq.length, a.keys_sink.shape[2]
    twice = k.clone()
    twice[:, :, ns:ns + n] *= 2.0
    b.update(twice, v)
    for x, y in zip(a.get_deq_tensors(), b.get_deq_tensors()):
        assert torch.equal(x, y)
