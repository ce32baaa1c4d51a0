"""Prompt quantization at the sizes where the kernels' tiles and lanes end:
one token, block edges, offsets inside a block, head_dims whose rows do not
divide a workgroup (K) and odd or misaligned columns (V), strided inputs, every
mode, width, group and activation type.  Bit-exact against the oracle: the
quantizers are defined bit for bit (codes, scales, zero points)."""
import numpy as np
import pytest
import torch

from innerq_amd import ops
from oracle import quant_ref as Q

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TD = {"f16": torch.float16, "bf16": torch.bfloat16}
MODES = [("asymmetric", (1, 2, 3, 4)), ("symmetric", (2, 3, 4)), ("hybrid", (2, 3, 4))]


def planted(B, H, n, D, seed, act):
    """Normal data with the groups that leave the fast arithmetic: zeros of both signs, constant
    rows, exact ties, subnormals, NaN, infinities, a range that overflows fp16."""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((B, H, n, D)).astype(np.float32)
    flat = x.reshape(B * H, n, D)
    flat[-1, ::5] = 0.0
    flat[-1, ::5, 1::2] = -0.0
    flat[0, n // 2] = 1.5
    flat[0, n // 3] = np.arange(D) % 16 + 0.5
    flat[-1, n - 1] *= 1e-6
    flat[-1, 0, D // 2] = np.nan
    flat[0, n - 1, 0] = np.inf
    flat[0, 0, :2] = [60000.0, -60000.0][:D]
    return torch.from_numpy(x).to(TD[act])


def host(t):
    return t.float().numpy() if t.dtype == torch.bfloat16 else t.numpy()


def act_bits(a, act):
    return Q.f16_bits(a) if act == "f16" else Q.bf16_bits(a)


def expected(x, G, bits, mode, axis, act):
    """(fields, meta halves [.., M]) of the packed groups, from the oracle."""
    ch = axis == "channel"
    with np.errstate(all="ignore"):
        if mode == "hybrid":
            c, s, z = (Q.quantize_channeldim_hybrid if ch else Q.quantize_tokendim_hybrid)(x, G, bits, act)
            mask = s["mask"]
            el = np.repeat(mask, G, axis=-1 if ch else 2)
            za = np.where(c["zp"] == Q.INT32_MIN, 0, c["zp"])
            sy = np.where(c["nozp"] == Q.INT32_MIN, 0, c["nozp"]) * z["nozp"].astype(np.int32) + (1 << (bits - 1))
            half = np.where(mask, act_bits(s["nozp"], act) | 0x8000, act_bits(s["zp"], act) & 0x7FFF)
            zero = np.where(mask, 0, act_bits(z["zp"], act))
            return np.where(el, sy, za), np.stack([half, zero], -1).astype(np.uint16)
        f = {("symmetric", True): Q.quantize_channeldim_sym, ("symmetric", False): Q.quantize_tokendim_sym,
             ("asymmetric", True): Q.quantize_channeldim_asym, ("asymmetric", False): Q.quantize_tokendim_asym}
        c, s, z = f[mode, ch](x, G, bits, act)
    c = np.where(c == Q.INT32_MIN, 0, c)
    if mode == "symmetric":
        return c * z.astype(np.int32) + (1 << (bits - 1)), act_bits(s, act)[..., None]
    return c & ((1 << bits) - 1), np.stack([act_bits(s, act), act_bits(z, act)], -1)


def same_meta(got, want, act):
    """Equal bits, any NaN pattern standing for NaN and a zero of either sign for zero (torch's amin
    and numpy's min may keep either of two zeros)."""
    exp = 0x7C00 if act == "f16" else 0x7F80
    nan = ((got & 0x7FFF) > exp) & ((want & 0x7FFF) > exp)
    zero = ((got & 0x7FFF) == 0) & ((want & 0x7FFF) == 0)
    return bool(np.all((got == want) | nan | zero))


# the sign of an all-NaN hybrid group's flag and the like stay out of the comparison: the planted
# NaN sits in one group, compared by its fields
@pytest.mark.parametrize("act", ["f16", "bf16"])
@pytest.mark.parametrize("mode,widths", MODES)
@pytest.mark.parametrize("n,D,G,off,strided", [(1, 128, 32, 0, False), (63, 64, 32, 0, True), (65, 128, 64, 63, False),
                                               (64, 128, 128, 1, True), (130, 96, 32, 5, False),
                                               (17, 384, 128, 0, False), (1027, 64, 64, 0, True)])
def test_keys(act, mode, widths, n, D, G, off, strided):
    B, H = 2, 2
    x = planted(B, H, n, D, n + D, act)
    xd = x.to(DEV)
    if strided:
        xd = xd.transpose(1, 2).contiguous().transpose(1, 2)
    for bits in widths:
        st = ops.PackedStore("channel", B, H, D, G, bits, mode, DEV, dtype=TD[act])
        if off:
            st.append(torch.ones(B, H, off, D, device=DEV, dtype=TD[act]))
        st.append(xd)
        fields, meta = expected(host(x), G, bits, mode, "channel", act)
        W, M, ng = G * bits // 32, meta.shape[-1], D // G
        T = off + n
        words = st.codes.cpu().numpy().view(np.uint32).reshape(B, H, -1, ng, 64, W)
        got = words.transpose(0, 1, 2, 4, 3, 5).reshape(B, H, -1, ng, W)[:, :, off:T]
        np.testing.assert_array_equal(Q.unpack_groups(got, bits, G).reshape(B, H, n, D), fields)
        gm = st.meta.cpu().numpy().view(np.uint16).reshape(B, H, -1, ng, 64, M)
        gm = gm.transpose(0, 1, 2, 4, 3, 5).reshape(B, H, -1, ng, M)[:, :, off:T]
        assert same_meta(gm, meta, act)


@pytest.mark.parametrize("act", ["f16", "bf16"])
@pytest.mark.parametrize("mode,widths", MODES)
@pytest.mark.parametrize("groups,D,G,off,layout", [(1, 128, 32, 0, "plain"), (3, 64, 64, 1, "heads last"),
                                                   (2, 128, 128, 0, "heads last"), (5, 33, 32, 1, "plain"),
                                                   (2, 1, 64, 0, "plain"), (2, 130, 32, 0, "odd rows")])
def test_values(act, mode, widths, groups, D, G, off, layout):
    B, H, n = 2, 2, groups * G
    x = planted(B, H, n, D, n + D, act)
    xd = x.to(DEV)
    if layout == "heads last":
        xd = xd.transpose(1, 2).contiguous().transpose(1, 2)
    if layout == "odd rows":  # rows that start at odd elements
        y = torch.empty(B, H, n, D + 1, dtype=TD[act], device=DEV)
        y[..., 1:] = xd
        xd = y[..., 1:]
    for bits in widths:
        st = ops.PackedStore("token", B, H, D, G, bits, mode, DEV, dtype=TD[act])
        if off:
            st.append(torch.ones(B, H, off * G, D, device=DEV, dtype=TD[act]))
        st.append(xd)
        fields, meta = expected(host(x), G, bits, mode, "token", act)
        W, M = G * bits // 32, meta.shape[-1]
        words = st.codes.cpu().numpy().view(np.uint32).reshape(B, H, -1, D, W)[:, :, off:off + groups]
        got = Q.unpack_groups(words, bits, G).transpose(0, 1, 2, 4, 3).reshape(B, H, n, D)
        np.testing.assert_array_equal(got, fields)
        gm = st.meta.cpu().numpy().view(np.uint16).reshape(B, H, -1, D, M)[:, :, off:off + groups]
        assert same_meta(gm, meta, act)


def same_bits(a, b):
    return torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


@pytest.mark.parametrize("act", ["f16", "bf16"])
@pytest.mark.parametrize("bits,mode,D,G,norm", [(4, "asymmetric", 128, 32, False), (3, "symmetric", 96, 32, True),
                                                (2, "hybrid", 64, 64, True), (1, "asymmetric", 384, 128, False)])
@pytest.mark.parametrize("rows", [0, 37])
def test_long_key_calls_equal_short_ones(act, bits, mode, D, G, norm, rows):
    """A call of at most 2^19 lanes of 8 values takes one row per lane, a longer one four: calls at the line
    and a ragged number of rows past it hold the bytes of calls of 100 tokens."""
    B, H = 2, 4
    n = (1 << 19) // (B * H * D // 8) + rows
    x = torch.cat([planted(B, H, 64, D, bits, act), torch.randn(B, H, n - 64, D).to(TD[act])], dim=2).to(DEV)
    nf = (torch.rand(B, H, 1, D, device=DEV) + 0.5).to(TD[act]) if norm else None
    whole, parts = (ops.PackedStore("channel", B, H, D, G, bits, mode, DEV, dtype=TD[act]) for _ in range(2))
    whole.append(x, norm=nf)
    for t in range(0, n, 100):
        parts.append(x[:, :, t:t + 100], norm=nf)
    for a, b in zip(token_rows(whole), token_rows(parts)):
        assert torch.equal(a[:, :n], b[:, :n]) and int((a[:, n:] != 0).sum()) == 0


@pytest.mark.parametrize("act", ["f16", "bf16"])
@pytest.mark.parametrize("bits,mode", [(4, "asymmetric"), (2, "asymmetric"), (3, "symmetric")])
@pytest.mark.parametrize("D,G,groups", [(130, 32, 12), (33, 32, 42), (128, 64, 6), (33, 64, 21), (128, 32, 6), (128, 64, 3),
                                        (128, 32, 11)])
def test_long_value_calls_equal_short_ones(act, bits, mode, D, G, groups):
    """Short calls go by a lane per value (up to 2^17 or 2^18 values), longer ones by a thread per token group
    and column pair: calls on either side of the lines hold the bytes of calls of one group, stores and
    quant.py's outputs."""
    B, H, n = 2, 3, groups * G
    x = planted(B, H, n, D, bits, act).to(DEV)
    whole, parts = (ops.PackedStore("token", B, H, D, G, bits, mode, DEV, dtype=TD[act]) for _ in range(2))
    whole.append(x)
    dense = []
    for t in range(0, n, G):
        parts.append(x[:, :, t:t + G])
        dense.append(ops.quantize_dense(x[:, :, t:t + G].contiguous(), G, bits, mode, "token"))
    for a, b in ((whole.codes, parts.codes), (whole.meta, parts.meta)):
        m = whole.t_cap // G, parts.t_cap // G
        assert torch.equal(a.view(B * H, m[0], -1)[:, :groups], b.view(B * H, m[1], -1)[:, :groups])
    for a, b in zip(ops.quantize_dense(x, G, bits, mode, "token"), zip(*dense)):
        assert same_bits(a, torch.cat(b, dim=2))


@pytest.fixture
def stale(monkeypatch):
    """torch.empty as memory that held other values gives it: every byte of the stores' integers set."""
    empty = torch.empty

    def poisoned(*a, **k):
        t = empty(*a, **k)
        return t.fill_(-1) if t.dtype in (torch.int32, torch.int16) else t

    monkeypatch.setattr(torch, "empty", poisoned)


def token_rows(st):
    """(codes, meta) of a K store as [B H, token, ...]."""
    bh, nb, ng = st.B * st.H, st.t_cap // 64, st.D // st.group
    return [t.view(bh, nb, ng, 64, -1).transpose(2, 3).reshape(bh, nb * 64, -1) for t in (st.codes, st.meta)]


@pytest.mark.parametrize("n,t0", [(1, 0), (65, 0), (30, 50), (64, 0), (192, 64), (57, 200), (7, 250), (120, 250),
                                  (300, 255), (64, 256), (400, 200)])
@pytest.mark.parametrize("mode", ["asymmetric", "symmetric", "hybrid"])
def test_appended_store_clears_its_last_block(stale, mode, n, t0):
    """A store that an append made or grew (past 256 tokens here) is not cleared as a whole: the append
    clears the rows of its last 64-token block past the tokens and the blocks after it, over memory that
    held other values; the tokens of before stay."""
    B, H, D = 2, 3, 128
    st = ops.PackedStore("channel", B, H, D, 32, 3, mode, DEV)
    x = torch.randn(B, H, t0 + n, D, device=DEV).half()
    before = None
    if t0:
        st.append(x[:, :, :t0])
        before = [t[:, :t0].clone() for t in token_rows(st)]
    st.append(x[:, :, t0:])
    T, rows = t0 + n, token_rows(st)
    assert all(int((t[:, T:] != 0).sum()) == 0 for t in rows)
    if t0:
        assert all(torch.equal(t[:, :t0], b) for t, b in zip(rows, before))
    whole = ops.PackedStore("channel", B, H, D, 32, 3, mode, DEV)
    whole.reserve(T)
    whole.append(x)
    assert all(torch.equal(t[:, :T], w[:, :T]) for t, w in zip(rows, token_rows(whole)))


@pytest.mark.parametrize("axis,t0,n", [("channel", 0, 70), ("channel", 250, 70), ("token", 0, 64), ("token", 128, 32)])
def test_a_failed_append_leaves_cleared_units(stale, monkeypatch, axis, t0, n):
    """An append that grew the store and then raised leaves the new units as a cleared store has them."""
    st = ops.PackedStore(axis, 2, 3, 128, 32, 2, "asymmetric", DEV)
    x = torch.randn(2, 3, t0 + n, 128, device=DEV).half()
    if t0:
        st.append(x[:, :, :t0])
    cap = st.t_cap
    cut = -(-t0 // st.unit)
    old = [t.view(6, cap // st.unit, -1)[:, :cut].clone() for t in (st.codes, st.meta)] if t0 else []

    def fail(*a):
        raise RuntimeError("launch")

    monkeypatch.setattr(st, "_quantize", fail)
    with pytest.raises(RuntimeError, match="launch"):
        st.append(x[:, :, t0:])
    assert st.t_cap > cap and st.length == t0
    now = [t.view(6, st.t_cap // st.unit, -1) for t in (st.codes, st.meta)]
    assert all(int((t[:, cut:] != 0).sum()) == 0 for t in now)
    assert all(torch.equal(t[:, :cut], b) for t, b in zip(now, old))


@pytest.mark.parametrize("act", ["f16", "bf16"])
@pytest.mark.parametrize("D,T,strided", [(128, 1, False), (128, 255, True), (128, 257, False), (64, 513, True),
                                         (64, 4099, False), (128, 2049, True)])
def test_key_norm_slices(act, D, T, strided):
    """The factor over one slice, whole slices and ragged ones, against numpy (exact: one square root)."""
    k = torch.randn(2, 3, T, D, device=DEV).to(TD[act])
    k[0, 0, T - 1, 3] = 40.0
    k[1, 2, T // 2, 5] = -50.0
    k[1, 1, 0, 7] = float("nan")
    top = k.cpu().abs().max(dim=-2, keepdim=True).values.float().numpy()
    root = np.sqrt(top)  # correctly rounded in fp32, then to the type
    want = torch.from_numpy(root.astype(np.float16) if act == "f16" else Q.round_bf16(root)).to(TD[act])
    x = k.transpose(1, 2).contiguous().transpose(1, 2) if strided else k
    got = ops.key_norm_factor(x).cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got.nan_to_num(0.0), want.nan_to_num(0.0))
