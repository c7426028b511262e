"""The fp32 moment kernels at d = 64, p = 2 with enough heads to fill the chip (heads x 256-position blocks >= 256).  Against
the fp64 closed form on the CPU, and against the dense kernels for what the closed form would be slow at.

Limits: sums of n terms of about equal size round about sqrt(n) times 2^-24 of their size at most, n <= 1100 here, so 33 units =
2e-6; normwise the roundings average out.  Measured against 64 bits: l2 up to 4.0e-7 in o and dv, 5.9e-7 in dq and dk, the
largest element 1.5e-6 of the largest.  (Operands of 16 bits would show: 2.3e-6 to 4.5e-6 in l2.)"""
import pytest
import torch

from oracle import fastmax_oracle as O

from helpers import assert_close

pytestmark = pytest.mark.gpu
KERNEL_PATH = "moments"
L2 = {"o": 1e-6, "dq": 2e-6, "dk": 2e-6, "dv": 1e-6}
LARGEST = 4e-6


@pytest.fixture(scope="module")
def ops(built):
    from fastmax_amd import ops as _ops

    return _ops


def run(ops, q, k, v, go, **kw):
    qd, kd, vd, god = (t.cuda() for t in (q, k, v, go))
    o, den, sc, arg = ops.forward(qd, kd, vd, **kw)
    return (o,) + tuple(ops.backward(qd, kd, vd, o, den, god, qk_scale=sc, qk_argmax=arg, **kw))


def check(got, want):
    for name, g, w in zip(("o", "dq", "dk", "dv"), got, want):
        diff, w = (g.double() - w.double().to(g.device)), w.double().to(g.device)
        l2, largest = float(diff.norm() / w.norm()), float(diff.abs().max() / w.abs().max())
        assert l2 <= L2[name] and largest <= LARGEST, f"{name}: l2 rel {l2:.3e}, max-abs rel {largest:.3e}"


# (256 heads: one block each, no states at all; 128: two; 86: three; 52: five)
@pytest.mark.parametrize("bh,n", [(256, 40), (128, 257), (128, 512), (86, 513), (86, 769), (52, 1100)])
@pytest.mark.parametrize("mask", [True, False])
@pytest.mark.parametrize("normalize", [True, False])
def test_against_the_closed_form(ops, bh, n, mask, normalize):
    q, k, v, go = O.seeded_inputs((bh, n, 64), seed=bh + n)
    kw = dict(mask=mask, normalize=normalize, p=2, a0=0.7, a1=0.9, a2=0.4)
    if not normalize:
        q, k = 0.05 * q, 0.05 * k
    print("many heads", bh, n, mask, normalize, flush=True)
    check(run(ops, q, k, v, go, **kw), O.dense_truth(*(t.double() for t in (q, k, v, go)), **kw))


@pytest.mark.parametrize("bh,bhkv,nq,nk", [(172, 86, 600, 600), (128, 128, 1, 300), (96, 96, 300, 700), (128, 32, 255, 1025),
                                           (90, 90, 700, 700)])
@pytest.mark.parametrize("mask", [True, False])
def test_grouped_heads_and_key_prefix(ops, bh, bhkv, nq, nk, mask):
    q, _, _, go = O.seeded_inputs((bh, nq, 64), seed=nq)
    _, k, v, _ = O.seeded_inputs((bhkv, nk, 64), seed=nk + 1)
    kw = dict(mask=mask, normalize=True, p=2)
    print("many heads, groups", bh, bhkv, nq, nk, mask, flush=True)
    ratio = bh // bhkv
    o, dq, dk, dv = O.dense_truth(q.double(), k.double().repeat_interleave(ratio, 0), v.double().repeat_interleave(ratio, 0), go.double(), **kw)
    fold = lambda t: t.reshape(bhkv, ratio, nk, 64).sum(1)
    got = run(ops, q, k, v, go, **kw)
    check(got, (o, dq, fold(dk), fold(dv)))


@pytest.mark.parametrize("mask", [True, False])
def test_long_sequences_match_the_dense_kernels(ops, mask, monkeypatch):
    q, k, v, go = O.seeded_inputs((90, 2500, 64), seed=9)
    kw = dict(mask=mask, normalize=True, p=2)
    print("many heads, long", mask, flush=True)
    got = run(ops, q, k, v, go, **kw)
    monkeypatch.setenv("FASTMAX_PATH", "dense")
    for name, a, b in zip(("o", "dq", "dk", "dv"), got, run(ops, q, k, v, go, **kw)):   # (2500 terms: sqrt(2500) units on either side)
        assert_close(name, a, b, 100 * 2.0 ** -24)
