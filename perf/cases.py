"""The measured workloads: what a program that keeps its KV cache in this package has it do.

Every case is one of seven kinds of call (``kind``), each through a public entry point:

* ``decode``   ops.decode_attention: one new token per sequence attends over [packed | fp16 window] K and V;
* ``qk``       ops.qk_gemv: the logits of one query token per head over packed K;
* ``av``       ops.av_gemv: attention weights times packed V;
* ``append``   ops.PackedStore(...).append: a prompt's keys or values quantized into a new store;
* ``prefill``  cache.InnerqDynamicLayer(preset).update(prompt): sinks, recent windows, key normalization, both stores;
* ``steps``    a whole generation of one layer: prefill of a prompt, then append() + attend() token by token;
* ``read``     InnerqDynamicLayer.get_deq_tensors(): the dense K and V that update() hands to a model's own attention.

Keys and values are normal with a few outlier channels per head (what the key normalization and
the per-group scales are there for), queries normal: softmax rows neither flat nor one-hot.
"""
from __future__ import annotations

import math

import torch

from innerq_amd import ops
from innerq_amd.cache import InnerqDynamicLayer
from innerq_amd.presets import PRESETS, preset_config

DEV = "cuda:0"
DT = {"fp16": torch.float16, "bf16": torch.bfloat16}
# tokens x KV heads x head_dim of the largest listed case: no drawn case is larger
MOST_VALUES = 8 * 8 * 32768 * 128


def listed():
    return [
        # one user, a short chat: the smallest step, bound by launches and latency; the formats of innerq_base
        dict(name="decode_one_short", kind="decode", B=1, Hq=32, Hkv=8, D=128, T=1000, win=128, kb=3, vb=3,
             kmode="symmetric", vmode="symmetric", kg=32, vg=32, dtype="fp16", norm=True),
        # one user, a long document: a head is spread over many workgroups
        dict(name="decode_one_long", kind="decode", B=1, Hq=32, Hkv=8, D=128, T=131072, win=0, kb=4, vb=4,
             kmode="asymmetric", vmode="asymmetric", kg=32, vg=32, dtype="fp16", norm=False),
        # a serving batch at 32k context, 4-bit K and V, every token packed: the benchmark's step
        dict(name="decode_batch_4bit", kind="decode", B=8, Hq=32, Hkv=8, D=128, T=32768, win=0, kb=4, vb=4,
             kmode="asymmetric", vmode="asymmetric", kg=32, vg=32, dtype="fp16", norm=False),
        # the same batch with 2-bit K, 4-bit V and a 128-token fp16 window (one layer of the 32-layer benchmark)
        dict(name="decode_batch_window", kind="decode", B=8, Hq=32, Hkv=8, D=128, T=32768, win=128, kb=2, vb=4,
             kmode="asymmetric", vmode="asymmetric", kg=32, vg=32, dtype="fp16", norm=False),
        # a bf16 model with eight query heads per KV head; innerq_hybrid's formats, a ragged length
        dict(name="decode_gqa8_bf16", kind="decode", B=4, Hq=64, Hkv=8, D=128, T=8191, win=128, kb=3, vb=2,
             kmode="symmetric", vmode="hybrid", kg=32, vg=32, dtype="bf16", norm=True),
        # K and V configured with different group sizes (key_group_size, value_group_size)
        dict(name="decode_groups_differ", kind="decode", B=8, Hq=32, Hkv=8, D=128, T=16384, win=128, kb=4, vb=2,
             kmode="asymmetric", vmode="asymmetric", kg=32, vg=64, dtype="fp16", norm=False),
        # the two halves of a step on their own, as the benchmark's single-GEMV configurations call them
        dict(name="qk_one", kind="qk", B=1, Hq=32, Hkv=8, D=128, T=8192, kb=4, kmode="asymmetric", kg=32, norm=False),
        dict(name="av_batch", kind="av", B=8, Hq=32, Hkv=8, D=128, T=32768, vb=2, vmode="asymmetric", vg=64),
        # a 32k prompt's keys quantized into a store (a batch of 8)
        dict(name="append_keys", kind="append", role="K", B=8, H=8, D=128, T=32768, bits=4, mode="asymmetric", g=32,
             dtype="fp16", norm=False),
        # the prefill of one layer of a bf16 model, innerq_base, a ragged prompt length
        dict(name="prefill_layer", kind="prefill", preset="innerq_base", B=4, H=8, D=128, T=8190, dtype="bf16"),
        # a short generation of one layer, innerq_hybrid: prefill of 500 tokens, then 40 steps (a V flush among them)
        dict(name="steps_layer", kind="steps", preset="innerq_hybrid", B=4, Hq=32, Hkv=8, D=128, T=500, n=40,
             dtype="fp16"),
        # the dense K and V for a model that runs its own attention over the cache
        dict(name="read_layer", kind="read", preset="innerq_small", B=4, H=8, D=128, T=16384, dtype="fp16"),
    ]


def _logu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any kind, batch, GQA ratio, head_dim, length (ragged ones among them), format and dtype."""
    kind = rng.choice(["decode", "decode", "decode", "qk", "av", "append", "prefill", "steps", "read"])
    D = rng.choice([128, 128, 128, 64])
    H = rng.choice([1, 2, 4, 8, 8])
    nrep = rng.choice([1, 2, 4, 4, 8])
    B = _logu(rng, 1, 16)
    most = MOST_VALUES // (B * H * D)
    groups = [g for g in (32, 32, 64, 128) if g <= D]
    mode = lambda: rng.choice(["asymmetric", "symmetric"])  # noqa: E731
    if kind == "decode":
        T = _logu(rng, 400, min(most, 131072))
        kg = rng.choice(groups)
        vg = kg if rng.random() < 0.75 else rng.choice([32, 64, 128])
        dtype = "fp16" if kg != vg else rng.choice(["fp16", "fp16", "bf16"])
        vmode = "hybrid" if kg == vg and rng.random() < 0.25 else mode()
        return dict(kind=kind, B=B, Hq=H * nrep, Hkv=H, D=D, T=T, win=rng.choice([0, rng.randint(1, 160)]),
                    kb=rng.choice([2, 3, 4]), vb=rng.choice([2, 3, 4]), kmode=mode(), vmode=vmode, kg=kg, vg=vg,
                    dtype=dtype, norm=rng.random() < 0.4)
    if kind == "qk":
        return dict(kind=kind, B=B, Hq=H * nrep, Hkv=H, D=D, T=_logu(rng, 64, min(most, 131072) // max(1, nrep // 4)),
                    kb=rng.choice([2, 3, 4]), kmode=mode(), kg=rng.choice(groups), norm=rng.random() < 0.4)
    if kind == "av":
        g = rng.choice([32, 64, 128])
        T = _logu(rng, 256, min(most, 131072) // max(1, nrep // 4)) // g * g
        return dict(kind=kind, B=B, Hq=H * nrep, Hkv=H, D=D, T=T, vb=rng.choice([2, 3, 4]), vmode=mode(), vg=g)
    if kind == "append":
        role = rng.choice(["K", "V"])
        g = rng.choice(groups)
        T = _logu(rng, 256, min(most, 65536))
        m = rng.choice(["asymmetric", "symmetric", "hybrid"])
        return dict(kind=kind, role=role, B=B, H=H, D=D, T=T if role == "K" else T // g * g, bits=rng.choice([2, 3, 4]),
                    mode=m, g=g, dtype=rng.choice(["fp16", "fp16", "bf16"]), norm=role == "K" and rng.random() < 0.5)
    preset = rng.choice(["innerq_base", "innerq_small", "innerq_hybrid"])
    dtype = rng.choice(["fp16", "fp16", "bf16"])
    if kind == "steps":
        return dict(kind=kind, preset=preset, B=min(B, 8), Hq=H * nrep, Hkv=H, D=D, T=_logu(rng, 200, 4096),
                    n=rng.randint(8, 64), dtype=dtype)
    if kind == "read":
        preset = rng.choice([preset, "kivi", "kivi_sink"])
    return dict(kind=kind, preset=preset, B=B, H=H, D=D, T=_logu(rng, 400, min(most, 32768)), dtype=dtype)


# --- inputs -------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1000003 + 17)


def _kv(gen, B, H, T, D, dt, transposed=False):
    """K or V tokens [B,H,T,D]: normal, four channels of each head ten times as large.  transposed: the
    layout a projection leaves, [B,T,H,D] seen as [B,H,T,D]."""
    x = torch.randn((B, T, H, D) if transposed else (B, H, T, D), generator=gen, device=DEV)
    ch = torch.rand(H, D, generator=gen, device=DEV).argsort(-1)[:, :4]
    f = torch.ones(H, D, device=DEV).scatter_(1, ch, 10.0)
    if transposed:
        return (x * f).to(dt).transpose(1, 2)
    return (x * f[:, None]).to(dt)


def _factor(k):
    """A key normalization factor as the cache computes it from the keys it quantizes."""
    return k.abs().amax(2, keepdim=True).sqrt()


def _split(case):
    """(packed tokens, fp16 tokens after them): K and V packed up to V's last whole group before the window."""
    n = (case["T"] - case["win"]) // case["vg"] * case["vg"]
    return n, case["T"] - n


def _inputs(case, seed):
    gen, kind = _gen(seed), case["kind"]
    dt = DT[case.get("dtype", "fp16")]
    B, D, T = case["B"], case["D"], case["T"]
    if kind == "decode":
        k, v = _kv(gen, B, case["Hkv"], T, D, dt), _kv(gen, B, case["Hkv"], T, D, dt)
        q = torch.randn(B, case["Hq"], D, generator=gen, device=DEV)
        norm = _factor(k) if case["norm"] else None
        return dict(k=k, v=v, q=q.to(dt), norm=norm)
    if kind == "qk":
        k = _kv(gen, B, case["Hkv"], T, D, dt)
        q = torch.randn(B, case["Hq"], D, generator=gen, device=DEV).to(dt)
        return dict(k=k, q=q, norm=_factor(k) if case["norm"] else None)
    if kind == "av":
        v = _kv(gen, B, case["Hkv"], T, D, dt)
        p = torch.softmax(2.0 * torch.randn(B, case["Hq"], T, generator=gen, device=DEV), dim=-1).to(dt)
        return dict(v=v, p=p)
    if kind == "append":
        x = _kv(gen, B, case["H"], T, D, dt)
        return dict(x=x, norm=_factor(x) if case["norm"] else None)
    H = case["Hkv"] if kind == "steps" else case["H"]
    k, v = _kv(gen, B, H, T, D, dt, transposed=True), _kv(gen, B, H, T, D, dt, transposed=True)
    d = dict(k=k, v=v)
    if kind == "steps":
        n = case["n"]
        d["q"] = torch.randn(n, B, case["Hq"], 1, D, generator=gen, device=DEV).to(dt)
        new = torch.randn(2, n, B, H, 1, D, generator=gen, device=DEV)
        d["kn"], d["vn"] = new[0].to(dt), new[1].to(dt)
    return d


def prepare(case, seed):
    """What the program holds before the call: its stores (decode and read), windows, queries or prompt."""
    s, kind = _inputs(case, seed), case["kind"]
    s["case"] = case
    if kind == "decode":
        n, r = _split(case)
        k, v, dt = s.pop("k"), s.pop("v"), DT[case["dtype"]]
        B, H, D = case["B"], case["Hkv"], case["D"]
        s["ks"] = ops.PackedStore("channel", B, H, D, case["kg"], case["kb"], case["kmode"], DEV, dtype=dt)
        s["vs"] = ops.PackedStore("token", B, H, D, case["vg"], case["vb"], case["vmode"], DEV, dtype=dt)
        s["ks"].append(k[:, :, :n], norm=s["norm"])
        s["vs"].append(v[:, :, :n])
        s["kr"] = k[:, :, n:].contiguous() if r else None
        s["vr"] = v[:, :, n:].contiguous() if r else None
    elif kind == "qk":
        s["ks"] = ops.PackedStore("channel", case["B"], case["Hkv"], case["D"], case["kg"], case["kb"], case["kmode"],
                                  DEV)
        s["ks"].append(s.pop("k"), norm=s["norm"])
    elif kind == "av":
        s["vs"] = ops.PackedStore("token", case["B"], case["Hkv"], case["D"], case["vg"], case["vb"], case["vmode"],
                                  DEV)
        s["vs"].append(s.pop("v"))
    elif kind == "read":
        s["layer"] = InnerqDynamicLayer(preset_config(case["preset"]), 0)
        s["layer"].update(s.pop("k"), s.pop("v"))
    return s


def _layer_outputs(layer):
    """A layer's state after a prefill: codes and metadata of both stores, factor, sinks and windows."""
    ks, vs = layer._kq.store, layer._vq.store
    uk, uv = -(-ks.length // ks.unit), vs.length // vs.unit  # the units that hold tokens
    bh = ks.B * ks.H
    out = dict(kc=ks.codes.view(bh, ks.t_cap // ks.unit, -1)[:, :uk], km=ks.meta.view(bh, ks.t_cap // ks.unit, -1)[:, :uk],
               vc=vs.codes.view(bh, vs.t_cap // vs.unit, -1)[:, :uv], vm=vs.meta.view(bh, vs.t_cap // vs.unit, -1)[:, :uv],
               kr=layer.keys_recent, vr=layer.values_recent)
    if layer.key_normalization_factor is not None:
        out["factor"] = layer.key_normalization_factor
    return out


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        return ops.decode_attention(s["q"], None, s["ks"], s["kr"], None, s["vs"], s["vr"], case["D"] ** -0.5,
                                    norm=s["norm"])
    if kind == "qk":
        return ops.qk_gemv(s["q"], s["ks"], case["D"] ** -0.5, norm=s["norm"])
    if kind == "av":
        return ops.av_gemv(s["p"], s["vs"])
    if kind == "append":
        x = s["x"]
        st = ops.PackedStore("channel" if case["role"] == "K" else "token", case["B"], case["H"], case["D"], case["g"],
                             case["bits"], case["mode"], DEV, dtype=x.dtype)
        st.append(x, norm=s["norm"])
        u, bh = st.unit, case["B"] * case["H"]
        n = -(-st.length // u)
        return dict(codes=st.codes.view(bh, st.t_cap // u, -1)[:, :n], meta=st.meta.view(bh, st.t_cap // u, -1)[:, :n])
    if kind == "read":
        return s["layer"].get_deq_tensors()
    layer = InnerqDynamicLayer(preset_config(case["preset"]), 0)
    layer.update(s["k"], s["v"])
    if kind == "prefill":
        return _layer_outputs(layer)
    outs = []
    for i in range(case["n"]):
        layer.append(s["kn"][i], s["vn"][i])
        outs.append(layer.attend(s["q"][i], case["D"] ** -0.5))
    return torch.stack(outs)


# --- what the path cannot do without ---------------------------------------------
def _packed_bytes(B, H, T, D, bits, mode, g):
    return B * H * T * D * bits / 8 + B * H * T * D / g * (2 if mode == "symmetric" else 4)


def _layer_split(case, T):
    """(K packed, V packed) tokens of a preset's layer after a prefill of T tokens."""
    p = PRESETS[case["preset"]]

    def one(sink, recent, over_token, flush):
        n = max(T - sink, 0)
        r = min(recent, n)
        while over_token and (n - r) % flush:
            r -= 1
        return n - r

    return (one(p["key_w_sink"], p["key_w_recent"], p["key_quantize_over_token"], p["key_flush_size"]),
            one(p["value_w_sink"], p["value_w_recent"], p["value_quantize_over_token"], p["value_flush_size"]))


def work(case):
    kind, B, D, T = case["kind"], case["B"], case["D"], case["T"]
    if kind == "decode":
        H, n = case["Hkv"], _split(case)[0]
        b = _packed_bytes(B, H, n, D, case["kb"], case["kmode"], case["kg"])
        b += _packed_bytes(B, H, n, D, case["vb"], case["vmode"], case["vg"])
        return dict(bytes=b + 2 * B * H * (T - n) * D * 2 + 2 * B * case["Hq"] * D * 2, flops=4 * B * case["Hq"] * T * D)
    if kind == "qk":
        b = _packed_bytes(B, case["Hkv"], T, D, case["kb"], case["kmode"], case["kg"])
        return dict(bytes=b + B * case["Hq"] * (2 * D + 4 * T), flops=2 * B * case["Hq"] * T * D)
    if kind == "av":
        b = _packed_bytes(B, case["Hkv"], T, D, case["vb"], case["vmode"], case["vg"])
        return dict(bytes=b + B * case["Hq"] * (2 * D + 2 * T), flops=2 * B * case["Hq"] * T * D)
    if kind == "append":
        H = case["H"]
        return dict(bytes=2 * B * H * T * D + _packed_bytes(B, H, T, D, case["bits"], case["mode"], case["g"]),
                    flops=8 * B * H * T * D)
    p = PRESETS[case["preset"]]
    H = case["Hkv"] if kind == "steps" else case["H"]
    nk, nv = _layer_split(case, T)
    packed = _packed_bytes(B, H, nk, D, p["k_bits"], p["key_quantize_mode"], p["key_group_size"]) + \
        _packed_bytes(B, H, nv, D, p["v_bits"], p["value_quantize_mode"], p["value_group_size"])
    dense = 2 * B * H * (2 * T - nk - nv) * D  # fp16 sinks and windows
    if kind == "read":
        return dict(bytes=packed + dense + 2 * 2 * B * H * T * D, flops=4 * B * H * T * D)
    pre = 2 * 2 * B * H * T * D + packed + dense
    if kind == "prefill":
        return dict(bytes=pre, flops=16 * B * H * T * D)
    n, Hq = case["n"], case["Hq"]
    step = packed + dense + 4 * B * H * D + 4 * B * Hq * D
    return dict(bytes=pre + n * step, flops=n * 4 * B * Hq * (T + n // 2) * D)


def tolerance(case):
    """Stores and dense reads are defined bit for bit.  Logits are fp32 sums of 128 products (rel 1.4e-6 to 2.8e-6,
    max 5e-5 against 64 bits, measured).  Attention outputs carry fp16 probabilities and one rounding to the
    output's type (measured against 64 bits: rel 2.5e-4, max 2.6e-3 and, between two calls whose waves took the
    blocks in another order, 7.5e-3 in fp16; rel 1.7e-3, max 4e-3 in bf16).  About four times each."""
    kind = case["kind"]
    if kind in ("append", "prefill", "read"):
        return "exact"
    if kind == "qk":
        return {"rel": 1e-5, "max": 2e-4}
    if case.get("dtype") == "bf16":
        return {"rel": 7e-3, "max": 3e-2}
    return {"rel": 1e-3, "max": 3e-2}


# --- 64-bit values without this package's code --------------------------------------
def _div(a, b):
    """a / b rounded once to a's type."""
    return (a.float() / torch.as_tensor(b, device=a.device).float().expand_as(a)).to(a.dtype)


def _quantized(x, bits, mode, g, axis, norm=None):
    """The 64-bit values that the quantization of x [B,H,n,D] stands for (groups along D: axis 'channel';
    along tokens: 'token'); every step of the quantizer rounds to x's type."""
    if x.shape[2] == 0:
        return x.double()
    if norm is not None:
        x = _div(x, norm.expand_as(x))
    B, H, n, D = x.shape
    if axis == "channel":
        xr, dim = x.reshape(B, H, n, D // g, g), 4
    else:
        xr, dim = x.reshape(B, H, n // g, g, D), 3

    def asym(b):
        lo, hi, top = xr.amin(dim, keepdim=True), xr.amax(dim, keepdim=True), 2 ** b - 1
        s = _div(hi - lo, float(top))
        c = _div(xr - lo, s.expand_as(xr)).float().clamp(0, top).round().nan_to_num(0.0)
        return c.double() * s.double() + lo.double()

    def sym(b):
        top = 2 ** (b - 1) - 1
        s = _div(xr.abs().amax(dim, keepdim=True), float(top))
        c = _div(xr.abs(), s.expand_as(xr)).float().clamp(0, top).round().nan_to_num(0.0)
        return c.double() * s.double() * torch.sign(xr).double()

    if mode == "asymmetric":
        y = asym(bits)
    elif mode == "symmetric":
        y = sym(bits)
    else:  # per group the 1-bit-narrower asym or the sym values, whichever is nearer in L1
        a, b = asym(bits - 1), sym(bits)
        ea, eb = ((t - xr.double()).abs().sum(dim, keepdim=True) for t in (a, b))
        y = torch.where(ea > eb, b, a)
    y = y.reshape(B, H, n, D)
    return y if norm is None else y * norm.double()


def _attend(q, k, v, scale):
    """softmax(q k^T scale) v in 64 bits: q [Hq,D], k and v [Hkv,T,D]."""
    Hkv, T, D = k.shape
    nrep = q.shape[0] // Hkv
    s = (q.double().view(Hkv, nrep, D) @ k.transpose(1, 2).contiguous()) * scale
    return (torch.softmax(s, -1) @ v).reshape(-1, D)


def exact(case, seed):
    kind, d = case["kind"], _inputs(case, seed)
    if kind == "decode":
        n, outs = _split(case)[0], []
        for b in range(case["B"]):  # one sequence at a time: 64-bit copies of K and V
            k, v, f = d["k"][b:b + 1], d["v"][b:b + 1], None if d["norm"] is None else d["norm"][b:b + 1]
            kd = torch.cat([_quantized(k[:, :, :n], case["kb"], case["kmode"], case["kg"], "channel", f),
                            k[:, :, n:].double()], 2)
            vd = torch.cat([_quantized(v[:, :, :n], case["vb"], case["vmode"], case["vg"], "token"),
                            v[:, :, n:].double()], 2)
            outs.append(_attend(d["q"][b], kd[0], vd[0], case["D"] ** -0.5))
        return torch.stack(outs)
    if kind in ("qk", "av"):
        outs, H = [], case["Hkv"]
        for b in range(case["B"]):
            if kind == "qk":
                f = None if d["norm"] is None else d["norm"][b:b + 1]
                kd = _quantized(d["k"][b:b + 1], case["kb"], case["kmode"], case["kg"], "channel", f)[0]
                s = d["q"][b].double().view(H, -1, case["D"]) @ kd.transpose(1, 2).contiguous() * case["D"] ** -0.5
                outs.append(s.reshape(-1, case["T"]))
            else:
                vd = _quantized(d["v"][b:b + 1], case["vb"], case["vmode"], case["vg"], "token")[0]
                outs.append((d["p"][b].double().view(H, -1, case["T"]) @ vd).reshape(-1, case["D"]))
        return torch.stack(outs)
    if kind in ("append", "prefill"):
        return None  # packed bytes: no 64-bit value
    p = PRESETS[case["preset"]]
    nk, nv = _layer_split(case, case["T"])
    sk, sv = p["key_w_sink"], p["value_w_sink"]
    axes = {True: "token", False: "channel"}
    f = _factor(d["k"][:, :, sk:sk + nk]) if p["key_normalize"] and nk else None

    def dense(x, sink, n, bits, mode, g, over_token, factor):
        y = _quantized(x[:, :, sink:sink + n], bits, mode, g, axes[over_token], factor)
        return torch.cat([x[:, :, :sink].double(), y, x[:, :, sink + n:].double()], 2)

    def both(k, v, mk, mv):
        return (dense(k, sk, mk, p["k_bits"], p["key_quantize_mode"], p["key_group_size"],
                      p["key_quantize_over_token"], f),
                dense(v, sv, mv, p["v_bits"], p["value_quantize_mode"], p["value_group_size"],
                      p["value_quantize_over_token"], None))

    if kind == "read":
        return both(d["k"], d["v"], nk, nv)
    outs = []
    for i in range(case["n"]):
        k = torch.cat([d["k"]] + [t for t in d["kn"][:i + 1]], 2)
        v = torch.cat([d["v"]] + [t for t in d["vn"][:i + 1]], 2)
        nk += p["key_flush_size"] if k.shape[2] - sk - nk >= p["key_flush_size"] else 0
        nv += p["value_flush_size"] if v.shape[2] - sv - nv >= p["value_flush_size"] else 0
        kd, vd = both(k, v, nk, nv)
        outs.append(torch.stack([_attend(d["q"][i, b, :, 0], kd[b], vd[b], case["D"] ** -0.5)
                                 for b in range(case["B"])])[:, :, None])
    return torch.stack(outs)
