"""Which dense reads of a layer go through the one launch (ops.read_dense) and which through the copies:
the rule alone, on tensors without memory, with the launch and the dequantization recorded."""
from types import SimpleNamespace

import pytest
import torch
from torch.autograd import forward_ad

from innerq_amd import ops
from innerq_amd.cache import InnerqDynamicLayer

H16 = torch.float16


def rows(n, B=1, H=1, D=128, dtype=H16, device="meta"):
    return torch.empty(B, H, n, D, dtype=dtype, device=device)


def route(monkeypatch, sink, recent, nq=64, dtype=H16, store_dtype=H16):
    layer = InnerqDynamicLayer(SimpleNamespace(), 0)
    layer.device = "meta"
    taken = []
    monkeypatch.setattr(ops, "read_dense", lambda *a: taken.append("launch"))
    q = SimpleNamespace(length=nq, store=SimpleNamespace(dtype=store_dtype, codes=rows(1)),
                        dequant_into=lambda out, norm: taken.append("copies"))
    out = layer._dense(sink, q, recent, None, dtype)
    return taken, out


def test_ordinary_reads_take_the_launch(monkeypatch):
    assert route(monkeypatch, rows(32), rows(96))[0] == ["launch"]
    x = rows(32).requires_grad_()
    with torch.no_grad():  # nothing is followed
        assert route(monkeypatch, x, rows(96))[0] == ["launch"]


def test_reads_that_autograd_follows_take_the_copies(monkeypatch):
    for which in (0, 1):
        x = [rows(32), rows(96)]
        x[which].requires_grad_()
        taken, out = route(monkeypatch, *x)
        assert taken == ["copies"] and out.requires_grad
    with forward_ad.dual_level():
        x = forward_ad.make_dual(rows(32), rows(32))
        assert route(monkeypatch, x, rows(96))[0] == ["copies"]


@pytest.mark.parametrize("ns,nr,nq,taken", [(0, 2 ** 27 - 1, 64, "launch"), (0, 2 ** 27, 64, "copies"),
                                            (2 ** 26, 2 ** 26, 64, "copies")])
def test_reads_past_the_launchs_counts_take_the_copies(monkeypatch, ns, nr, nq, taken):
    assert route(monkeypatch, rows(ns), rows(nr), nq)[0] == [taken]


def test_other_types_and_devices_take_the_copies(monkeypatch):
    assert route(monkeypatch, rows(32), rows(96), dtype=torch.float32)[0] == ["copies"]
    assert route(monkeypatch, rows(32, dtype=torch.bfloat16), rows(96))[0] == ["copies"]
    assert route(monkeypatch, rows(32, device="cpu"), rows(96))[0] == ["copies"]
