"""fp32 forward passes that nobody differentiates, up to 64 channels on the dense kernels: their contractions run on parts of
3 x 8 bits (fastmax_amd/csrc/fm_cut.h).  Against the fp64 closed form, and against the training forward pass, which stays on
the fp32 instruction."""
import pytest
import torch

from oracle import fastmax_oracle as O

from helpers import assert_close

KERNEL_PATH = "dense"
gpu = pytest.mark.gpu
UNIT = 2.0 ** -24


def forwards(q, k, v, mask, normalize=True, a0=1.0, a1=1.0, a2=0.5, p=2):
    """(o, den) of a pass that no backward pass follows, and of one that may be differentiated"""
    from fastmax_amd import _ext

    ext = _ext.load()
    args = [t.cuda() for t in (q, k, v)] + [bool(mask), normalize, 1.0, a0, a1, a2, 1.0, p, False]
    return ext.forward_ex(*args, False)[:2], ext.forward_ex(*args)[:2]


@gpu
@pytest.mark.parametrize("d", [4, 24, 32, 40, 64])
@pytest.mark.parametrize("bh,bhkv,nq,nk", [(3, 3, 1, 1), (4, 2, 31, 31), (2, 2, 33, 160), (2, 1, 256, 256), (2, 2, 257, 257), (3, 3, 300, 1000), (2, 2, 100, 900),
                                           (132, 66, 289, 289), (260, 260, 70, 70)])   # (the last two: blocks of eight waves)
@pytest.mark.parametrize("mask", [True, False])
def test_against_the_closed_form(built, d, bh, bhkv, nq, nk, mask):
    q, _, _, go = O.seeded_inputs((bh, nq, d), seed=nq + d)
    _, k, v, _ = O.seeded_inputs((bhkv, nk, d), seed=nk + d + 1)
    print("forward only", d, bh, bhkv, nq, nk, mask, flush=True)
    (o, den), (ot, dent) = forwards(q, k, v, mask)
    rep = [t.double().repeat_interleave(bh // bhkv, 0) for t in (k, v)]
    want = O.dense_truth(q.double(), rep[0], rep[1], go.double(), mask=mask, normalize=True, p=2)[0]
    # (sums of up to 1000 terms of about equal size: sqrt(1000) roundings of 2^-24 each, and a few in the weights)
    assert_close("o", o, want, 40 * UNIT)
    assert_close("den", den, dent, 40 * UNIT)
    if mask and nq == nk:   # a query with few keys in sight: the bits of the training pass
        assert torch.equal(o[:, :32], ot[:, :32]) and torch.equal(den[:, :32], dent[:, :32])


@gpu
@pytest.mark.parametrize("mask", [True, False])
def test_the_module_keeps_the_two_apart(built, mask):
    """With gradients the module's output has the training pass's bits; without, it comes from the other kernel."""
    from fastmax_amd import FASTMultiHeadAttention

    q, k, v, _ = (t.cuda() for t in O.seeded_inputs((1, 8, 300, 64), seed=5))
    att = FASTMultiHeadAttention()
    args = (None, mask, 0.0, True, 1.0, 1.0, 1.0, 0.5, 1.0, 2)
    (o, _), (ot, _) = forwards(q[0].cpu(), k[0].cpu(), v[0].cpu(), mask)
    assert torch.equal(att(q.requires_grad_(True), k, v, *args)[0].detach(), ot)
    assert torch.equal(att(q.detach(), k, v, *args)[0], o) and not torch.equal(o, ot)


@gpu
@pytest.mark.parametrize("d", [24, 64])
@pytest.mark.parametrize("mask", [True, False])
def test_strided_views_have_the_same_bits(built, d, mask):
    """Slices of a fused projection, grouped heads, token-major output: the contiguous call's bits."""
    from fastmax_amd import _ext

    ext = _ext.load()
    b, t, groups, r = 2, 290, 2, 3
    x = torch.randn(b, t, groups, r + 2, d, generator=torch.Generator().manual_seed(d)).cuda()
    q5, k4, v4 = x[:, :, :, :r].permute(0, 2, 3, 1, 4), x[:, :, :, r].permute(0, 2, 1, 3), x[:, :, :, r + 1].permute(0, 2, 1, 3)
    tail = (mask, True, 1.0, 1.0, 1.0, 0.5, 1.0, 2, False, False)
    o5, den = ext.forward_strided(q5, k4, v4, *tail)[:2]
    o, den3 = ext.forward_ex(q5.reshape(-1, t, d), k4.reshape(-1, t, d), v4.reshape(-1, t, d), *tail)[:2]
    assert torch.equal(o5.reshape(-1, t, d), o) and torch.equal(den, den3)


@gpu
def test_packed_projection_without_gradients(built):
    """qkv_attention under no gradients against the same call with them (which has the training pass's bits)."""
    from fastmax_amd import qkv_attention

    qkv = torch.randn(2, 400, 4 * 3 * 64, generator=torch.Generator().manual_seed(3)).cuda()
    y = qkv_attention(qkv, None, None, 4, 1, 64, rope_n=0)
    yt = qkv_attention(qkv.clone().requires_grad_(True), None, None, 4, 1, 64, rope_n=0).detach()
    assert not torch.equal(y, yt)
    assert_close("y", y, yt, 40 * UNIT)


@gpu
def test_replays_of_a_captured_call(built):
    """Inference loops capture the call: every replay has the eager call's bits, with eager work in between."""
    from fastmax_amd import _ext

    ext = _ext.load()
    q, k, v = (t.cuda() for t in O.seeded_inputs((6, 300, 64), seed=11)[:3])
    args = (q, k, v, True, True, 1.0, 1.0, 1.0, 0.5, 1.0, 2, False, False)
    want = ext.forward_ex(*args)[0]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        o = ext.forward_ex(*args)[0]
    for _ in range(4):
        o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, want)
        assert torch.equal(ext.forward_ex(*args)[0], want)


@gpu
@pytest.mark.parametrize("bh,nq,nk,d,mask", [(256, 100, 1000, 32, True), (300, 100, 100, 64, False), (300, 100, 100, 64, True)])
def test_half_empty_blocks_are_not_slower(built, bh, nq, nk, d, mask):
    """Blocks that hold few queries (a short sequence, or a few queries behind a key prefix) are made small: with eight waves
    each, these took 1.04, 1.19 and 1.44 times as long as on the fp32 instruction; they take at most as long now (5 % of
    noise; each the best of interleaved batches)."""
    from fastmax_amd import _ext

    ext = _ext.load()
    q, k, v = torch.randn(bh, nq, d, device="cuda"), torch.randn(bh, nk, d, device="cuda"), torch.randn(bh, nk, d, device="cuda")
    args = (q, k, v, mask, True, 1.0, 1.0, 1.0, 0.5, 1.0, 2, False)
    best = {}
    for rep in range(12):
        for follows in (False, True):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            for _ in range(20):
                ext.forward_ex(*args, follows)
            end.record()
            torch.cuda.synchronize()
            if rep > 1:
                best[follows] = min(best.get(follows, 1e9), start.elapsed_time(end))
    assert best[False] <= 1.05 * best[True], f"{50 * best[False]:.1f} us against {50 * best[True]:.1f}"


# 1 + 2^-8 - 2^-17 and the like: the second and the third part of each are near their largest and of one sign, so that a
# product of parts left out adds up instead of averaging out
X, Y = 1.003883361816406, 1.003883242607117


def cut_parts(x):
    out = []
    x = torch.tensor(x, dtype=torch.float32)
    for _ in range(3):
        out.append(x.bfloat16().double())
        x = (x.double() - out[-1]).float()
    return out


def test_any_lost_product_of_parts_would_show():
    """Six products of parts give X Y to 2 units of 2^-24; without any one of them it is off by more than 100."""
    a, b = cut_parts(X), cut_parts(Y)
    exact = float(torch.tensor(X, dtype=torch.float32).double() * torch.tensor(Y, dtype=torch.float32).double())
    six = [(0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0)]
    off = lambda pairs: abs(float(sum(a[i] * b[j] for i, j in pairs)) / exact - 1) / UNIT
    assert off(six) < 2.0
    for lost in six:
        assert off([p for p in six if p != lost]) > 100, lost


@gpu
@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("bh", [3, 300])   # (blocks of four and of eight waves)
def test_fp32_contractions_keep_24_bits(built, d, bh):
    """The scores show in the denominators (f = s), the weighted sum in the output (f = a constant).  64 keys: 4 steps of 6
    roundings of at most half a unit each, 2 units left out, a few roundings at the end: 16 units in all."""
    n = 64
    q, k = torch.full((bh, n, d), X), torch.full((bh, n, d), Y)
    v = Y * (2.0 ** (torch.arange(d) % 5 - 2.0)).expand(bh, n, d).contiguous()
    x, y = torch.tensor(X).double(), torch.tensor(Y).double()
    (_, den), _ = forwards(q, k, v, False, normalize=False, a0=0.0, a1=1.0, a2=0.0)
    err = ((den.double().cpu() / (n * d * x * y) - 1).abs().max() / UNIT).item()
    assert err < 16, f"denominators off by {err:.1f} units"
    (o, _), _ = forwards(q, k, v, False, normalize=False, a0=X, a1=0.0, a2=0.0)
    err = ((o.double().cpu() / v.double() - 1).abs().max() / UNIT).item()
    assert err < 16, f"outputs off by {err:.1f} units"


def ranged(kind, d, n):
    """q, k, v with values that three bf16 parts do not hold, and the coefficients"""
    q, k, v, _ = O.seeded_inputs((2, n, d), seed=n + d)
    kw = dict(normalize=True, a0=0.5, a1=0.1, a2=0.1)
    j, c = n // 2, d - 3
    if kind == "infinite value":
        v[0, j, c] = float("inf")
    elif kind == "minus infinity in two rows":
        v[0, j, c] = v[1, n - 1, 0] = -float("inf")
    elif kind == "not a number":
        v[0, j, c] = k[1, j, 1] = float("nan")
    elif kind == "infinite key":
        k[0, j, c] = float("inf")
        kw.update(normalize=False)
    elif kind == "largest value":   # (rounds to infinity in bf16)
        v[0, j, c] = torch.finfo(torch.float32).max
        v[1, 0, 1] = torch.finfo(torch.float32).min
    elif kind == "tiny values":
        v *= 2.0 ** -115
    elif kind == "one tiny channel":
        v[..., c] *= 2.0 ** -112
    elif kind == "tiny and zero channels":
        v[..., c] = 0.0
        v[..., 1] *= 2.0 ** -112
    elif kind == "tiny keys and large queries":
        q, k = q * 2.0 ** 113, k * 2.0 ** -117
        kw.update(normalize=False)
    elif kind == "tiny scores":
        q, k = q.abs() * 2.0 ** -60, k.abs() * 2.0 ** -57
        kw.update(normalize=False, a0=0.0, a1=1.0, a2=0.0)
    elif kind == "tiny weights":
        kw.update(a0=2.0 ** -116, a1=2.0 ** -118, a2=0.0)
    elif kind == "tiny values under large weights":
        v *= 2.0 ** -118
        kw.update(a0=2.0 ** 100, a1=2.0 ** 97, a2=0.0)
    elif kind == "subnormal values":
        v *= 2.0 ** -137
        kw.update(a0=2.0 ** 100, a1=2.0 ** 97, a2=0.0)
    return q, k, v, kw


KINDS = ["infinite value", "minus infinity in two rows", "not a number", "infinite key", "largest value", "tiny values", "one tiny channel",
         "tiny and zero channels", "tiny keys and large queries", "tiny scores", "tiny weights", "tiny values under large weights",
         "subnormal values"]


@gpu
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("d,n", [(24, 270), (64, 300)])   # (causal: from 257 keys on)
@pytest.mark.parametrize("mask", [True, False])
def test_values_that_the_parts_do_not_hold(built, kind, d, n, mask):
    """What the training pass's kernel gives for them: not-a-number and infinities in the same places, and each channel as
    close as elsewhere.  Both are sums of n terms w v over the sum of w, so their rounding goes with the mean of the finite
    |v| of a channel (not with the result, which may come out near zero): sqrt(300) roundings each, 40 units in all."""
    q, k, v, kw = ranged(kind, d, n)
    print("range", kind, d, n, mask, flush=True)
    (o, den), (ot, dent) = forwards(q, k, v, mask, **kw)
    o, den, ot, dent = (t.double().cpu() for t in (o, den, ot, dent))
    size = torch.where(v.isfinite(), v.double().abs(), 0.0).mean(dim=(0, 1))
    for name, a, b, ref in (("o", o, ot, size), ("den", den[..., None], dent[..., None], None)):
        assert torch.equal(a.isnan(), b.isnan()), f"{name}: not-a-number in other places"
        assert torch.equal(a.isinf(), b.isinf()) and torch.equal(a[a.isinf()], b[b.isinf()]), f"{name}: infinities in other places"
        fin = b.isfinite()
        a, b = torch.where(fin, a, 0.0), torch.where(fin, b, 0.0)
        ref = b.abs().amax(dim=(0, 1)) if ref is None else ref
        err = ((a - b).abs().amax(dim=(0, 1)) / ref.clamp_min(1e-300)).max().item()
        assert err < 40 * UNIT, f"{name}: {err / UNIT:.0f} units of 2^-24 of a channel's size"
